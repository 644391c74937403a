"""Packing of a right-padded batch (engine.py:705-751) on the CPU: the host-side lengths path
and the one-read path agree, the supervised count equals the packed targets', and a left-padded
mask is refused (engine.py:709-717)."""

import importlib

import pytest
import torch

pkg = importlib.import_module("hack-fe30cb28-opus-5-5-ultracode_amd")
E = pkg.engine


def _batch(lengths, T, seed):
    g = torch.Generator().manual_seed(seed)
    B = len(lengths)
    ids = torch.randint(0, 1000, (B, T), generator=g)
    mask = (torch.arange(T)[None, :] < torch.tensor(lengths)[:, None]).long()
    labels = torch.where(torch.rand(B, T, generator=g) < 0.7, ids, torch.full_like(ids, -100))
    labels[:, 0] = -100
    return ids, mask, labels


def _packed(ids, mask, labels, **kw):
    rope = E.RopeTable(1e6, 128, torch.device("cpu"))
    return E.Packed(ids, mask, labels, rope, None, 0.0, **kw)


@pytest.mark.parametrize("lengths,T", [([5, 9, 1, 9], 9), ([3, 0, 7], 8), ([16], 16)])
def test_one_read_matches_host_lengths(lengths, T):
    ids, mask, labels = _batch(lengths, T, sum(lengths))
    a = _packed(ids, mask, labels)
    b = _packed(ids, mask, labels, lengths=lengths)
    assert a.lengths == lengths and a.n == sum(lengths) and a.max_len == max(lengths)
    assert torch.equal(a.tok, b.tok) and torch.equal(a.targets, b.targets)
    assert a.n_supervised == b.n_supervised == int((a.targets >= 0).sum())
    assert a.cu_seqlens_host == b.cu_seqlens_host
    # the target of a row's last token is the label after it (the padding's), as the reference
    want = []
    for r, n in enumerate(lengths):
        for p in range(n):
            want.append(int(labels[r, p + 1]) if p + 1 < T else -100)
    assert a.targets.tolist() == want


def test_left_padding_is_refused():
    ids, mask, labels = _batch([4, 6], 6, 1)
    mask = mask.flip(1)
    with pytest.raises(E.UnsupportedBatch):
        _packed(ids, mask, labels)


def test_host_metadata_is_checked_on_the_device():
    """Caller-given lengths and supervised count are checked without a read: metadata_ok is a
    device bool that turns False for a mask not right-padded to the lengths or a wrong count."""
    lengths, T = [5, 9, 1, 9], 9
    ids, mask, labels = _batch(lengths, T, 3)
    right = _packed(ids, mask, labels)
    n_sup = right.n_supervised
    assert right.metadata_ok is None  # read from the device: nothing to check
    assert bool(_packed(ids, mask, labels, lengths=lengths, n_supervised=n_sup).metadata_ok)
    assert not bool(_packed(ids, mask, labels, lengths=lengths,
                            n_supervised=n_sup - 1).metadata_ok)
    assert not bool(_packed(ids, mask, labels, lengths=[5, 8, 1, 9],
                            n_supervised=n_sup).metadata_ok)


def test_next_token_labels_and_positions():
    """targets[i] is the label one column right of token i (-100 past the last column), pos
    restarts at 0 for every row, cu_seqlens are the running sums of the lengths."""
    lengths, T = [3, 0, 4], 4
    ids, mask, labels = _batch(lengths, T, 7)
    p = _packed(ids, mask, labels, lengths=lengths)
    assert p.pos.tolist() == [0, 1, 2, 0, 1, 2, 3]
    assert p.cu_seqlens.tolist() == [0, 3, 3, 7]
    assert p.tok.tolist() == [0, 1, 2, 8, 9, 10, 11]
    want = [int(labels[0, 1]), int(labels[0, 2]), int(labels[0, 3]),
            int(labels[2, 1]), int(labels[2, 2]), int(labels[2, 3]), -100]
    assert p.targets.tolist() == want
    sup = [i for i, t in enumerate(want) if t >= 0]
    assert p.head_order.tolist()[:len(sup)] == sup


@pytest.mark.parametrize("scaling", [{"rope_type": "yarn", "factor": 4.0},
                                     {"type": "linear", "factor": 2.0}])
def test_scaled_rotary_embedding_is_refused(scaling):
    """A checkpoint whose rotary embedding is scaled is refused, not trained with the plain
    tables."""
    from types import SimpleNamespace as NS
    q = NS(lora_A={"default": NS(weight=torch.zeros(16, 64))}, lora_B={}, scaling={"default": 2.0},
           active_adapter=["default"])
    v = NS(lora_A={"default": NS(weight=torch.zeros(16, 64))}, lora_B={}, scaling={"default": 2.0},
           active_adapter=["default"])
    plain = NS()
    layer = NS(self_attn=NS(q_proj=q, k_proj=plain, v_proj=v, o_proj=plain),
               mlp=NS(gate_proj=plain, up_proj=plain, down_proj=plain))
    cfg = NS(hidden_size=64, num_attention_heads=4, num_key_value_heads=2, head_dim=16,
             rope_theta=1e6, rope_scaling=scaling, intermediate_size=128, vocab_size=100)
    causal = NS(model=NS(layers=[layer]), config=cfg)
    with pytest.raises(E.UnsupportedModel, match="rotary"):
        E.from_peft(NS(get_base_model=lambda: causal))


@pytest.mark.parametrize("lengths,T", [([5, 9, 1, 9], 9), ([3, 0, 7], 8), ([16], 16)])
def test_padded_packing_keeps_the_real_tokens(lengths, T):
    """Device-only packing (padded=True): every row is a sequence of T tokens; at each real
    token the ids, position and next-token target equal the unpadded packing's, the padding
    tokens take no target, the supervised rows come first in the same order, and nothing in it
    depends on a read of the device (n, max_len and cu_seqlens follow from [B, T])."""
    ids, mask, labels = _batch(lengths, T, 7 + sum(lengths))
    a = _packed(ids, mask, labels)
    p = _packed(ids, mask, labels, padded=True)
    B = len(lengths)
    assert p.n == B * T and p.max_len == T and p.lengths == [T] * B
    assert p.cu_seqlens.tolist() == p.cu_seqlens_host == [T * r for r in range(B + 1)]
    assert torch.equal(p.tok, torch.arange(B * T)) and torch.equal(p.ids, ids.reshape(-1))
    assert torch.equal(p.pos.long(), torch.arange(B * T) % T)
    # the real tokens: same target as the unpadded packing; padding: none
    assert torch.equal(p.targets.index_select(0, a.tok), a.targets)
    real = mask.reshape(-1).bool()
    assert bool((p.targets[~real] == -100).all())
    # supervised first, in packed order: the same rows as the unpadded head order
    n_sup = a.n_supervised
    assert torch.equal(p.tok[p.head_order[:n_sup]], a.tok[a.head_order[:n_sup]])
    assert bool((p.targets[p.head_order[n_sup:]] < 0).all())
    assert p.n_supervised == B * T and bool(p.metadata_ok)
    assert p.ctr_base is None and p.drawn == 0


def test_padded_packing_flags_left_padding_without_a_read():
    ids, mask, labels = _batch([4, 6], 6, 1)
    p = _packed(ids, mask.flip(1), labels, padded=True)  # no exception: nothing is read
    assert not bool(p.metadata_ok)


def test_device_counter_base_needs_padding():
    ids, mask, labels = _batch([4, 6], 6, 2)
    with pytest.raises(ValueError):
        _packed(ids, mask, labels, ctr_base=torch.zeros(1, dtype=torch.int64))
    p = _packed(ids, mask, labels, padded=True, ctr_base=torch.zeros(1, dtype=torch.int64))
    assert p.ctr_base is not None
    with pytest.raises(ValueError):
        _packed(ids, mask, labels, padded=True, ctr_base=torch.zeros(2, dtype=torch.int64))


def test_gemm_shape_check():
    """The step refuses a model whose products the package GEMM cannot tile (a reduction or
    width off the multiples of 128) before any weight is built; every Qwen2 size passes."""
    for kw in ({}, dict(hidden_size=896, intermediate_size=4864, num_attention_heads=14,
                        num_key_value_heads=2, head_dim=64),
               dict(hidden_size=3584, intermediate_size=18944, num_attention_heads=28,
                    num_key_value_heads=4, vocab_size=152064)):
        E.check_gemm_shapes(E.Qwen2Config(**kw))
    for kw in (dict(vocab_size=151937), dict(vocab_size=3000), dict(intermediate_size=8900),
               dict(hidden_size=1500)):
        with pytest.raises(E.UnsupportedModel, match="multiples of 128"):
            E.check_gemm_shapes(E.Qwen2Config(**kw))


def test_attention_split_counts_the_launched_workgroups():
    """Key ranges are cut only where the forward's (dQ's) workgroups, four (query tile, q head) pairs
    of a kv head each, are few and long: the q heads of a kv head count too. Chunks are whole blocks
    of 64 keys, at most 16."""
    chunk = pkg.ops.attn_chunk
    assert chunk([], 12, 2, 128, "fwd") == 0 and chunk([0, 0], 2, 2, 64, "dq") == 0
    # the same tiles and kv heads, 96 and 16 workgroups
    assert chunk([2048], 2, 2, 128, "fwd") == 512 and chunk([2048], 12, 2, 128, "fwd") == 0
    assert chunk([2048], 8, 8, 128, "fwd") == 704 and chunk([2080], 8, 8, 128, "fwd") == 0
    assert chunk([1535], 1, 1, 64, "fwd") == 0 and chunk([1536], 1, 1, 64, "fwd") == 512
    assert chunk([1023], 4, 4, 128, "fwd") == 0 and chunk([1024], 4, 4, 128, "fwd") == 256
    assert chunk([1024], 12, 2, 128, "fwd") == 0 and chunk([611, 997, 283, 744], 12, 2, 128, "fwd") == 0
    assert chunk([4096], 1, 1, 128, "dq") == 0  # long with heads of 128: dK/dV beside dQ instead
    assert chunk([1024], 4, 4, 128, "dq") == 256
    assert chunk([1024], 2, 2, 64, "dq") == 256 and chunk([1024], 14, 2, 64, "dq") == 0
    for n in range(1, 20000, 317):
        for kind in ("fwd", "dq"):
            c = chunk([n, 5], 2, 1, 64 + n % 2 * 64, kind)
            assert c % 64 == 0 and (c == 0 or 2 <= -(-n // c) <= 16)
