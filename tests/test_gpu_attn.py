"""The HIP varlen causal attention (qlora_attn_fwd/bwd) against fp32 autograd of
scaled_dot_product_attention per sequence on the CPU, at the reference's tolerances
(test_kernels.py:244-281: out 2e-3, dq/dk/dv 1e-2), including the reference's own case
(lengths 7, 130, 1, 64; 12 q heads over 2 kv heads; D 128), the config-3/5 shapes (lengths up to
1024), k/v in grouped and in repeated layout, head_dim 64, and the split of long key ranges over
several workgroups (qlora_attn_fwd_split / qlora_attn_bwd_split) at forced chunk sizes."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


class _Packed:
    def __init__(self, lengths):
        self.cu_seqlens_host = [0, *torch.tensor(lengths).cumsum(0).tolist()]
        self.cu_seqlens = torch.tensor(self.cu_seqlens_host, device=DEV, dtype=torch.int32)
        self.max_len = max(lengths)


def _expand(x, group):
    n, kh, d = x.shape
    return x[:, :, None, :].expand(n, kh, group, d).reshape(n, kh * group, d)


def close(a, b, tol):
    torch.testing.assert_close(a.detach().cpu().float(), b.detach().cpu().float(), rtol=tol,
                               atol=tol)


def _reference(q, k, v, dout, lengths):
    """fp32 CPU autograd per sequence; k/v repeated to the q heads; dk/dv per q head."""
    group = q.shape[1] // k.shape[1]
    ke, ve = _expand(k.cpu().float(), group), _expand(v.cpu().float(), group)
    outs, lses, dqs, dks, dvs = [], [], [], [], []
    start = 0
    scale = q.shape[2] ** -0.5
    for length in lengths:
        sl = slice(start, start + length)
        qr = q[sl].cpu().float().transpose(0, 1).requires_grad_()
        kr = ke[sl].transpose(0, 1).requires_grad_()
        vr = ve[sl].transpose(0, 1).requires_grad_()
        ref = torch.nn.functional.scaled_dot_product_attention(qr, kr, vr, is_causal=True)
        g = torch.autograd.grad(ref, (qr, kr, vr), dout[sl].cpu().float().transpose(0, 1))
        s = (qr.detach() @ kr.detach().transpose(1, 2)) * scale
        s = s.masked_fill(torch.ones(length, length, dtype=torch.bool).triu(1), float("-inf"))
        lses.append(torch.logsumexp(s, dim=-1))  # [HQ, L]
        outs.append(ref.detach().transpose(0, 1))
        dqs.append(g[0].transpose(0, 1))
        dks.append(g[1].transpose(0, 1))
        dvs.append(g[2].transpose(0, 1))
        start += length
    return (torch.cat(outs), torch.cat(lses, dim=1), torch.cat(dqs), torch.cat(dks),
            torch.cat(dvs))


def _run(pkg, lengths, HQ, KH, D, seed=0, expand=False, chunk=None):
    torch.manual_seed(seed)
    n = sum(lengths)
    q = torch.randn(n, HQ, D, device=DEV, dtype=torch.float16)
    k = torch.randn(n, KH, D, device=DEV, dtype=torch.float16)
    v = torch.randn(n, KH, D, device=DEV, dtype=torch.float16)
    dout = torch.randn(n, HQ, D, device=DEV, dtype=torch.float16)
    packed = _Packed(lengths)
    if chunk is not None:  # force the split (0: none) instead of the cost model's choice
        packed._attn_plans = {("fwd", HQ, KH): chunk, ("dq", HQ, KH): chunk}
    kk, vv = (_expand(k, HQ // KH).contiguous(), _expand(v, HQ // KH).contiguous()) if expand \
        else (k, v)
    print(f"attn lengths={lengths} HQ={HQ} KH={KH} D={D} expand={expand} chunk={chunk}",
          flush=True)
    out, lse, _, _ = pkg.ops._attn_fwd(q, kk, vv, packed, D ** -0.5)
    dq, dk, dv = pkg.ops._attn_bwd(dout, q, kk, vv, out, lse, None, None, packed, D ** -0.5)
    torch.cuda.synchronize()
    ro, rl, rdq, rdk, rdv = _reference(q, k, v, dout, lengths)
    close(out, ro, 2e-3)
    close(lse, rl, 1e-4)
    close(dq, rdq, 1e-2)
    close(dk, rdk, 1e-2)
    close(dv, rdv, 1e-2)
    return out, lse, dq, dk, dv


def test_reference_case(pkg):
    """test_kernels.py:244-281: lengths 7, 130, 1, 64; 12/2 heads; D 128."""
    _run(pkg, [7, 130, 1, 64], 12, 2, 128)


@pytest.mark.parametrize("lengths", [[1], [32], [33], [64, 65], [63, 1, 97], [200, 5, 129]])
def test_block_edges(pkg, lengths):
    _run(pkg, lengths, 12, 2, 128, seed=len(lengths))


def test_repeated_kv_layout(pkg):
    """k/v already repeated to the q heads ([n, HQ, D], the reference's _expand_kv layout)."""
    _run(pkg, [7, 130, 1, 64], 12, 2, 128, expand=True)


def test_head_dim_64(pkg):
    _run(pkg, [17, 60, 33, 5], 4, 2, 64)


def test_config_shapes(pkg):
    """Config 3/5 shapes: 4 sequences, lengths in [128, 1024] (incl. the maximum)."""
    _run(pkg, [1024, 301, 777, 128], 12, 2, 128, seed=5)


def test_empty_sequences(pkg):
    """Zero-length rows inside cu_seqlens are skipped; n == 0 launches nothing."""
    _run(pkg, [5, 0, 40], 12, 2, 128, seed=7)
    packed = _Packed([0])
    q = torch.empty(0, 12, 128, device=DEV, dtype=torch.float16)
    k = torch.empty(0, 2, 128, device=DEV, dtype=torch.float16)
    out, lse, _, _ = pkg.ops._attn_fwd(q, k, k, packed, 128 ** -0.5)
    assert out.shape == (0, 12, 128) and lse.shape == (12, 0)


@pytest.mark.parametrize("chunk", [64, 128, 192, 512])
def test_split_key_ranges(pkg, chunk):
    """Key ranges cut into chunks of `chunk` keys (several workgroups per query tile and a merge
    kernel), incl. tiles of one chunk, a sequence of 1 and the longest row."""
    _run(pkg, [1024, 301, 777, 1, 128, 65], 12, 2, 128, seed=chunk, chunk=chunk)


def test_split_head_dim_64(pkg):
    _run(pkg, [300, 17, 129], 4, 2, 64, seed=3, chunk=64)


def test_split_is_deterministic_and_matches_unsplit(pkg):
    """The merge order is fixed: two split runs agree bit for bit, and with the unsplit kernels
    to fp32 summation order."""
    a = _run(pkg, [700, 300, 40], 12, 2, 128, seed=11, chunk=128)
    b = _run(pkg, [700, 300, 40], 12, 2, 128, seed=11, chunk=128)
    c = _run(pkg, [700, 300, 40], 12, 2, 128, seed=11, chunk=0)
    for x, y, z in zip(a, b, c):
        assert torch.equal(x, y)
        close(x, z, 2e-3)


def test_concurrent_backward_matches_sequential(pkg):
    """A batch of few long sequences runs dK/dV on a second stream beside dQ (delta from its own
    kernel); a full batch runs them one after the other (delta formed by dQ). Sequences are
    independent, so the rows of the shared sequences agree bit for bit."""
    HQ, KH, D = 12, 2, 128
    few, extra = [1024, 600], [1024] * 10
    n_few, n = sum(few), sum(few) + sum(extra)
    g = torch.Generator(device=DEV).manual_seed(21)
    q, dout = (torch.randn(n, HQ, D, device=DEV, generator=g).half() for _ in range(2))
    k, v = (torch.randn(n, KH, D, device=DEV, generator=g).half() for _ in range(2))
    res = []
    for lengths, rows in ((few, n_few), (few + extra, n)):
        print(f"attn concurrent/sequential lengths={lengths}", flush=True)
        packed = _Packed(lengths)
        packed._attn_plans = {("fwd", HQ, KH): 0, ("dq", HQ, KH): 0}  # no key-range split
        qq, kk, vv, dd = q[:rows], k[:rows], v[:rows], dout[:rows]
        out, lse, _, _ = pkg.ops._attn_fwd(qq, kk, vv, packed, D ** -0.5)
        dq, dk, dv = pkg.ops._attn_bwd(dd, qq, kk, vv, out, lse, None, None, packed, D ** -0.5)
        torch.cuda.synchronize()
        res.append((out[:n_few], lse[:, :n_few], dq[:n_few], dk[:n_few], dv[:n_few]))
    for x, y in zip(*res):
        assert torch.equal(x, y)


@pytest.mark.parametrize("HQ,KH,D", [(14, 2, 64), (16, 2, 128), (28, 4, 128), (8, 8, 64)])
def test_concurrent_backward_other_shapes(pkg, HQ, KH, D):
    """The backward of few sequences at other head sizes and group counts (Qwen2 0.5B 14/2 x 64, 3B
    16/2, 7B 28/4, and one q head per kv head) against fp32 SDPA, key ranges unsplit. (dQ and dK/dV
    in turn: test_backward_rules runs them side by side.)"""
    _run(pkg, [600, 300], HQ, KH, D, seed=HQ + D, chunk=0)


@pytest.mark.parametrize("HQ,KH,D,lengths,split", [
    (16, 2, 128, [1024, 70], False), (28, 4, 128, [1050], False), (8, 8, 128, [1100, 1, 333], False),
    (5, 5, 64, [2600], False), (14, 2, 64, [2560], False),  # dQ beside dK/dV, delta from its own kernel
    (2, 2, 64, [1024, 33], True), (1, 1, 64, [1500, 1100], True), (4, 2, 64, [1030], True),
    (4, 4, 128, [1024, 9], True)])
def test_backward_rules(pkg, HQ, KH, D, lengths, split):
    """The package's own choices on either side of their lines: dQ beside dK/dV (long sequences, few
    dK/dV workgroups), dQ's and the forward's key ranges cut (fewer still); against fp32 SDPA."""
    assert (pkg.ops.attn_chunk(lengths, HQ, KH, D, "dq") > 0) == split
    groups = -(-max(lengths) // 128) * len(lengths) * HQ
    assert split or (groups <= 300 and max(lengths) >= (1024 if D == 128 else 2560))
    _run(pkg, lengths, HQ, KH, D, seed=HQ + D)


@pytest.mark.parametrize("HQ,KH,D,lengths", [(12, 2, 128, [700, 33]), (14, 2, 64, [700, 33]),
                                             (12, 2, 128, [2500, 1700, 1600, 1500, 1000])])
def test_forward_rescales_as_scores_grow(pkg, HQ, KH, D, lengths):
    """Scores that grow along the keys by far more than 2^8 move the forward's reference maximum
    (and rescale O) in block after block; four and eight wavefronts a workgroup (3,072 tiles and
    more). Against fp32 SDPA on the GPU; out is a convex combination of v (|v| <= 1 here), p and
    out are rounded to fp16 once each: 2 x 2^-11 of it."""
    g = torch.Generator(device=DEV).manual_seed(5)
    n = sum(lengths)
    q = torch.rand(n, HQ, D, device=DEV, generator=g).half()
    v = (torch.rand(n, KH, D, device=DEV, generator=g) * 2 - 1).half()
    grow = torch.cat([torch.linspace(0, 8, x, device=DEV) for x in lengths])
    k = (torch.rand(n, KH, D, device=DEV, generator=g) * grow[:, None, None]).half()
    packed = _Packed(lengths)
    print(f"attn growing scores lengths={lengths} HQ={HQ} D={D}", flush=True)
    out, lse, _, _ = pkg.ops._attn_fwd(q, k, v, packed, D ** -0.5)
    torch.cuda.synchronize()
    start = 0
    for x in lengths:
        sl = slice(start, start + x)
        qf, kf, vf = (t[sl].float().transpose(0, 1) for t in (q, _expand(k, HQ // KH),
                                                              _expand(v, HQ // KH)))
        s = torch.bmm(qf, kf.transpose(1, 2).contiguous()) * D ** -0.5
        s = s.masked_fill(torch.ones(x, x, device=DEV, dtype=torch.bool).triu(1), float("-inf"))
        assert s.amax() - s[:, -1, 0].amin() > 12  # several rescales (8 in log2 units each)
        ref = torch.bmm(torch.softmax(s, -1), vf).transpose(0, 1)
        assert (out[sl].float() - ref).abs().amax() < 2 * 2 ** -11
        torch.testing.assert_close(lse[:, sl], torch.logsumexp(s, -1), rtol=1e-5, atol=1e-4)
        start += x


@pytest.mark.parametrize("HQ,KH,D", [(12, 2, 128), (14, 2, 64), (3, 3, 128)])
@pytest.mark.parametrize("chunk", [0, 64])
def test_backward_pipeline_block_counts(pkg, HQ, KH, D, chunk):
    """One to eight 32-token blocks, whole and ragged: the backward kernels' first block, pairs,
    left-over and last block, on and past the diagonal of a 128-key workgroup, and workgroups
    whose last (query tile, q head) pairs lie past the sequence; key ranges whole and cut."""
    _run(pkg, [32, 64, 95, 96, 97, 128, 129, 160, 161, 192, 224, 255, 256], HQ, KH, D, seed=chunk,
         chunk=chunk)


@pytest.mark.parametrize("HQ,KH,D", [(12, 2, 128), (14, 2, 64)])
@pytest.mark.parametrize("chunk", [0, 128])
def test_largest_probability_is_exact(pkg, HQ, KH, D, chunk):
    """A query's largest probability is 1 whichever block of keys holds it. Key 64 (the second
    block's first) is the maximum of every later query by 0.4 to 8 log2 units and alone has a
    non-zero v, so O = v / l is rounded by the fp16 store only: half an ulp, and 2^-18 of it for
    fp32's sums and reciprocal. A maximum that lags behind key 64 would round that probability to
    fp16 too."""
    n, top = 320, 64
    scale = D ** -0.5
    q, k, v = (torch.zeros(n, h, D, device=DEV, dtype=torch.float16) for h in (HQ, KH, KH))
    lead = torch.linspace(0.4, 8.0, HQ, device=DEV)  # log2 units by which key 64 leads, per head
    q[:, :, 0] = lead.half()
    k[top, :, 0] = 1.0 / (scale * 1.4426950408889634)
    g = torch.Generator(device=DEV).manual_seed(9)
    v[top] = (1 + torch.rand(KH, D, device=DEV, generator=g)).half()
    packed = _Packed([n])
    packed._attn_plans = {("fwd", HQ, KH): chunk}
    print(f"attn largest probability HQ={HQ} D={D} chunk={chunk}", flush=True)
    out, _, _, _ = pkg.ops._attn_fwd(q, k, v, packed, scale)
    s = q[0, :, 0].double() * k[top, 0, 0].double() * scale  # [HQ]: key 64's score; the others 0
    rows = torch.arange(top, n, device=DEV, dtype=torch.float64)
    weight = 1 / (1 + rows[:, None] * torch.exp(-s))  # [rows, HQ]; `rows` keys of score 0
    exact = weight[:, :, None] * _expand(v[top:top + 1], HQ // KH).double()
    ulp = torch.exp2(torch.floor(torch.log2(exact)) - 10)
    assert ((out[top:].double() - exact).abs() <= ulp / 2 + exact * 2 ** -18).all()


@pytest.mark.parametrize("HQ,KH,D,lengths,chunk",
                         [(1, 1, 128, [700], 0), (14, 2, 64, [500, 333], 0),
                          (12, 2, 128, [700, 300], 128), (8, 8, 64, [601], 64),
                          (8, 8, 64, [4096, 4000, 4300], 0), (8, 8, 128, [4096, 4000, 4300], 320)])
def test_values_that_are_not_finite_stay_causal(pkg, HQ, KH, D, lengths, chunk):
    """A token's infinities and NaNs reach other tokens' rows only where the sums over its own block
    multiply them by a probability of 0: queries before its key block (64 keys forward, 32 dQ) and
    keys after its query block (32) keep their bits, whatever else their workgroup holds (four and
    eight wavefronts, 1 to 7 q heads a kv head, whole and cut key ranges). A score of -inf masks its
    key: that key's dK and dV are 0, also in a ragged last block."""
    g = torch.Generator(device=DEV).manual_seed(3)
    n, last = sum(lengths), lengths[0] - 1
    q = torch.rand(n, HQ, D, device=DEV, generator=g).half()
    k, v = (torch.randn(n, KH, D, device=DEV, generator=g).half() for _ in range(2))
    dout = torch.randn(n, HQ, D, device=DEV, generator=g).half()

    def run(**changed):
        t = dict(dict(q=q, k=k, v=v, dout=dout), **changed)
        packed = _Packed(lengths)
        packed._attn_plans = {("fwd", HQ, KH): chunk, ("dq", HQ, KH): chunk}
        out, lse, _, _ = pkg.ops._attn_fwd(t["q"], t["k"], t["v"], packed, D ** -0.5)
        dq, dk, dv = pkg.ops._attn_bwd(t["dout"], t["q"], t["k"], t["v"], out, lse, None, None,
                                       packed, D ** -0.5)
        torch.cuda.synchronize()
        return out, lse, dq, dk, dv

    def with_(x, at, value):
        y = x.clone()
        y[at, :, 3] = value
        return y

    inf, nan = float("inf"), float("nan")
    out, lse, dq, dk, dv = run()
    for at in (130, 160, 255, last):
        print(f"attn not finite HQ={HQ} KH={KH} D={D} lengths={lengths} chunk={chunk} at={at}",
              flush=True)
        before64, before32 = at // 64 * 64, at // 32 * 32
        for value in (inf, nan):
            o, l, q_, _, _ = run(v=with_(v, at, value))
            assert torch.equal(o[:before64], out[:before64]), ("V", value)
            assert torch.equal(l, lse)
            assert torch.equal(q_[:before64], dq[:before64])  # delta is formed from out
            _, _, _, k_, v_ = run(dout=with_(dout, at, value))
            assert torch.equal(k_[at // 32 * 32 + 32:], dk[at // 32 * 32 + 32:]), ("dO", value)
            assert torch.equal(v_[at // 32 * 32 + 32:], dv[at // 32 * 32 + 32:]), ("dO", value)
            _, _, _, k_, v_ = run(q=with_(q, at, value))
            assert torch.equal(k_[at // 32 * 32 + 32:], dk[at // 32 * 32 + 32:]), ("Q", value)
            assert torch.equal(v_[at + 1:], dv[at + 1:]), ("Q", value)
        o, _, q_, k_, v_ = run(k=with_(k, at, -inf))  # q > 0: the key's scores are -inf
        assert torch.isfinite(o).all() and torch.equal(o[:at], out[:at])
        assert torch.equal(q_[:before32], dq[:before32])
        assert not k_[at].any() and not v_[at].any()
        assert torch.isfinite(k_).all() and torch.isfinite(v_).all()


@pytest.mark.parametrize("HQ,KH,D,lengths", [(14, 2, 64, [2600, 1, 33, 2100, 65, 2400, 7]),
                                             (8, 8, 128, [3300, 64, 1, 5000, 31, 4000, 130]),
                                             (28, 4, 128, [1900, 1, 65, 1600, 33, 97])])
def test_eight_wavefronts_match_four(pkg, HQ, KH, D, lengths):
    """3,072 (query tile, head) pairs and more take workgroups of eight wavefronts; each sequence on
    its own takes four, with the same bits: long sequences beside very short and ragged ones, so that
    workgroups end in wavefronts without a tile and hold tiles of different lengths. The longest
    sequence against fp32 SDPA."""
    assert -(-sum(lengths) // 32) * HQ >= 3072 > -(-max(lengths) // 32) * HQ
    g = torch.Generator(device=DEV).manual_seed(HQ)
    n = sum(lengths)
    q = torch.randn(n, HQ, D, device=DEV, generator=g).half()
    k, v = (torch.randn(n, KH, D, device=DEV, generator=g).half() for _ in range(2))

    def run(lengths, sl):
        packed = _Packed(lengths)
        packed._attn_plans = {("fwd", HQ, KH): 0}
        return pkg.ops._attn_fwd(q[sl], k[sl], v[sl], packed, D ** -0.5)[:2]

    print(f"attn eight wavefronts HQ={HQ} KH={KH} D={D} lengths={lengths}", flush=True)
    out, lse = run(lengths, slice(0, n))
    start = 0
    for x in lengths:
        sl = slice(start, start + x)
        o, l = run([x], sl)
        assert torch.equal(out[sl], o) and torch.equal(lse[:, sl], l), x
        if x == max(lengths):
            qf, kf, vf = (t[sl].float().transpose(0, 1) for t in (q, _expand(k, HQ // KH),
                                                                  _expand(v, HQ // KH)))
            s = torch.bmm(qf, kf.transpose(1, 2).contiguous()) * D ** -0.5
            s = s.masked_fill(torch.ones(x, x, device=DEV, dtype=torch.bool).triu(1),
                              float("-inf"))
            close(o, torch.bmm(torch.softmax(s, -1), vf).transpose(0, 1), 2e-3)
            close(l, torch.logsumexp(s, -1), 1e-4)
        start += x
