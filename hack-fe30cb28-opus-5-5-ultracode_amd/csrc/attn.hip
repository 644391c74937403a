// Causal attention over the packed variable-length sequences of a step (flash attention: online
// softmax, no [L, L] matrix in memory), grouped-query heads, forward and backward, on gfx950
// MFMA (v_mfma_f32_32x32x16_f16: fp16 operands, fp32 accumulation).
// Reference: _attn_fwd / _attn_bwd engine.py:857-869 (PyTorch's memory-efficient attention in
// its cu_seqlens form, causal, dropout 0, scale = D^-1/2) fed with k/v repeated to the q heads by
// _expand_kv engine.py:655-660. Here k/v are read in their grouped layout [n, KH, D]: q head h
// uses kv head h / (HQ / KH).
//
// Layout of the work. A wavefront owns 32 queries of one q head (forward, dQ) or 32 keys of one
// q head (dK/dV). MFMA register layout for C[32x32] = A[32x16] B[16x32]: lane l supplies
// A[l % 32][8(l / 32) .. +7] and B[8(l / 32) .. +7][l % 32]; register r of lane l receives
// C[8(r / 4) + 4(l / 32) + r % 4][l % 32].
//  * forward / dQ compute S^T = K Q^T, so lane l holds one query (l % 32) and 16 of the keys of
//    each 32-key tile; the online-softmax state (running max, sum) is a per-lane scalar (lanes l
//    and l ^ 32 share a query and combine their maxima with one shuffle), and O^T = V^T P^T
//    keeps the lane <-> query ownership, so rescaling O is a per-lane multiply.
//  * dK/dV compute S = Q K^T (lane <-> key), dV^T = dO^T P and dK^T = Q^T dS.
// A product that contracts over tokens needs a token-contiguous operand (V^T forward, K^T dQ,
// Q^T and dO^T dK/dV): the tiles are staged row-major with 16-byte stores and read transposed
// with ds_read_b64_tr_b16 (TrFrags). The P/dS operand comes straight from the accumulator
// registers, whose rows within each 16-row group are in the order 0-3, 8-11, 4-7, 12-15 for the
// lower/upper half-wave; TrFrags hands out the tokens in that same order, so no register
// shuffles are needed.
// LDS tiles are XOR-swizzled by 16-byte chunk so that the operand reads (32 rows, same chunk)
// and the staging writes are spread over the banks.
//
// One workgroup = consecutive (query tile, q head) pairs of one kv head (forward, dQ), which share
// the staged K/V tiles; dK/dV: four wavefronts on 128 consecutive keys of one q head, sharing the
// staged Q/dO. The next tiles arrive by LDS DMA during the current tile's MFMAs. dK/dV come out
// per q head ([n, HQ, D]); the caller sums each group (the RoPE backward does, as the reference
// sums the repeated kv heads). The log-sum-exp of the forward (natural log, fp32 [HQ, n]) and
// delta = rowsum(dO * O) (fp32 [HQ, n], written by attn_delta_kernel or the dQ kernel) feed the dQ
// and the dK/dV kernels, which run in turn or side by side on two streams (bwd_concurrent).
#include "common.h"

#include <mutex>

namespace qlora {
namespace attn {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kTok = 32;   // queries (forward, dQ) or keys (dK/dV) per wavefront
constexpr int kKB = 64;    // keys per staged block (forward, dQ)
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

struct Args {
  const uint16_t* q;     // fp16 [n, HQ, D]
  const uint16_t* k;     // fp16 [n, KH, D]
  const uint16_t* v;     // fp16 [n, KH, D]
  const uint16_t* o;     // fp16 [n, HQ, D] (forward output; read by the backward)
  const uint16_t* dout;  // fp16 [n, HQ, D]
  uint16_t* out;         // forward: o; dQ: dq [n, HQ, D]
  uint16_t* dk;          // fp16 [n, HQ, D]
  uint16_t* dv;          // fp16 [n, HQ, D]
  float* lse;            // fp32 [HQ, n] natural-log log-sum-exp of each query's scores
  float* delta;          // fp32 [HQ, n]
  const int32_t* cu;     // int32 [nseq + 1]
  float* part;           // split key range: fp32 partial O / dQ [nch][n][HQ][D]
  float2* part_ml;       // forward split: (running max (log2 units), sum) [nch][HQ][n]
  int64_t n;
  int HQ, KH;
  int chunk;             // key blocks per workgroup (0: the whole range in one workgroup)
  int ntiles;            // workgroups per sequence and kv head (forward, dQ), per sequence and q
                         // head (dK/dV); query tiles per sequence (merge)
  float scale;
};

// The key range of a query tile with nkb key blocks may be cut into chunks of a.chunk blocks, one
// workgroup each (blockIdx.z = chunk), when a batch of few long sequences would otherwise leave
// most of the GPU idle while its longest tiles walk their keys. With one chunk the workgroup
// writes the result itself; otherwise each writes fp32 partials and attn_merge_kernel merges them
// in chunk order.
__device__ __forceinline__ int num_chunks(int nkb, int chunk) {
  return chunk > 0 ? (nkb + chunk - 1) / chunk : 1;
}

// 2^x by the hardware instruction (v_exp_f32): no denormal-range fix-up (results below 2^-126
// flush to zero, which a probability that small does not miss).
__device__ __forceinline__ float ex2(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ f32x16 mfma(half8_t a, half8_t b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// [rows][D] tile, 16-byte chunk c of row r at chunk c ^ (r mod D/8).
template <int D>
__host__ __device__ constexpr int rm_off(int row, int chunk) {
  return row * D + ((chunk ^ (row & (D / 8 - 1))) << 3);
}

// [rows][D] tile read transposed by ds_read_b64_tr_b16 (TrFrags): a half-wave reads 4
// consecutive rows (the first a multiple of 4) x 4 aligned chunks, which this swizzle spreads
// over distinct banks; 16-byte row stores (16 threads a row) stay conflict-free too.
template <int D>
__host__ __device__ constexpr int tt_off(int row, int chunk) {
  const int j = D == 128 ? row : row >> 1;  // rows sharing the 64 banks: 1 (D = 128) or 2
  const int sw = D == 128 ? (((j & 3) << 2) | ((j >> 2) & 3)) : (((j & 1) << 2) | ((j >> 1) & 3));
  return row * D + ((chunk ^ sw) << 3);
}

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4_t lds_short4_t;

__device__ __forceinline__ uint32_t word_of(const uint4& x, int i) {
  return i < 2 ? (i == 0 ? x.x : x.y) : (i == 2 ? x.z : x.w);
}

// A resource over rows [0, L) of one head of a token-major [*, stride] fp16 matrix starting at
// `base` (the sequence's first row, this head's first column).
__device__ __forceinline__ rsrc_t rows_rsrc(const uint16_t* base, int L, int64_t stride, int D) {
  return make_rsrc(base, L > 0 ? (uint32_t)(((int64_t)(L - 1) * stride + D) * 2) : 0u);
}

// One token's D/16 MFMA operands (chunks 2 kk + l/32 of row `row`) from a row resource.
template <int D>
__device__ __forceinline__ void load_token(rsrc_t src, int row, int stride_b, int lane,
                                           half8_t (&out)[D / 16]) {
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk)
    out[kk] = __builtin_bit_cast(
        half8_t, buf_load16(src, (uint32_t)(row * stride_b + (2 * kk + (lane >> 5)) * 16)));
}

// Row (query or key) index within the 32 x 32 tile of register r for this lane.
__device__ __forceinline__ int acc_row(int r, int lane) {
  return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
}

// Stores 32 x D values of one token (lane & 31) held as D/32 accumulators (d in the rows).
template <int D>
__device__ __forceinline__ void store_token_row(uint16_t* row, const f32x16 (&acc)[D / 32],
                                                float mul, int lane) {
#pragma unroll
  for (int u = 0; u < D / 32; ++u)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d = 32 * u + 8 * j + 4 * (lane >> 5);
      *reinterpret_cast<uint2*>(row + d) =
          make_uint2(pack2h(acc[u][4 * j] * mul, acc[u][4 * j + 1] * mul),
                     pack2h(acc[u][4 * j + 2] * mul, acc[u][4 * j + 3] * mul));
    }
}

// Stores 32 x D fp32 values of one token (lane & 31) held as D/32 accumulators (d in the rows).
template <int D>
__device__ __forceinline__ void store_token_row_f32(float* row, const f32x16 (&acc)[D / 32],
                                                    int lane) {
#pragma unroll
  for (int u = 0; u < D / 32; ++u)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d = 32 * u + 8 * j + 4 * (lane >> 5);
      *reinterpret_cast<float4*>(row + d) =
          make_float4(acc[u][4 * j], acc[u][4 * j + 1], acc[u][4 * j + 2], acc[u][4 * j + 3]);
    }
}

// ------------------------------------------------------------------------------------------------
// Forward: O = softmax(scale Q K^T + causal mask) V per sequence, and the log-sum-exp.
//
// A workgroup is NW wavefronts, one query tile each: NW consecutive (query tile, q head) pairs of
// one kv head, the heads fastest, which share the staged K/V blocks of 64 keys. Two wavefronts run
// per SIMD. The kernel is bound by what the SIMDs issue (per block and wavefront 32 MFMAs, 1,024
// cycles of the matrix core, beside 130 VALU instructions, 32 of them exponentials), so a block's
// softmax is formed two values at a time behind the MFMAs of the next block's S and of P V (every
// instruction pinned behind an MFMA by sched_barrier), no address is formed per fragment
// (RowFrags, TrFrags), and masks are applied from the diagonal on only. The maximum is the running
// one of all scores so far, so a query's largest probability is 1, which fp16 holds exactly: with a
// maximum that may lag (O rescaled only once a score exceeds it by 2^8) the forward is 3-5 % faster,
// but every probability is rounded and the output's error against 64 bits 2-3 % larger. K and V
// arrive by LDS DMA, two stages each, one barrier a block. MI355X, against one q head group per
// workgroup with the blocks staged through registers and two barriers a block, kernel averages: four
// sequences of 283-997 tokens, 12/2 heads of 128, 37.0 -> 25.5 us, 14/2 of 64 24.9 -> 17.0; two of
// 4,096 and 3,001 151 -> 113 and 103 -> 80.
// NW 4 or 8 (wide_groups): four wavefronts spread a small batch over the CUs, eight read K and V half
// as often.
// grid (ceil(ceil(max_len / 32) G / NW) nseq KH, 1, chunks), block 64 NW.
// ------------------------------------------------------------------------------------------------
// max(a, b, c) without the quieting of signalling NaNs that fmaxf adds per operand.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
// max (sum) of lanes l and l ^ 32
__device__ __forceinline__ float pair_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ uint32_t cvt2h(float a, float b) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){a, b}, h2));
}

// LDS byte addresses of the fragments of a [rows][D] stage. A swizzle acts on chunk bits that the
// fragment's column offset only flips, so a few lane addresses (one per column offset, formed once
// a block: N of them) and immediate row offsets reach all of a stage's fragments.
typedef __attribute__((address_space(3))) const half8_t lds_half8_t;
// rm_off stage (TT: tt_off): fragment (kk, half): row lane % 32 + 32 half, chunk 2 kk + lane / 32.
template <int D, bool TT = false>
struct RowFrags {
  uint32_t at[D / 16];
  __device__ __forceinline__ void set(uint32_t stage, int lane) {
    const int row = lane & 31, chunk = lane >> 5;
    const uint32_t l0 = (uint32_t)(2 * (TT ? tt_off<D>(row, chunk) : rm_off<D>(row, chunk)));
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) at[kk] = l0 ^ (uint32_t)(32 * kk);
    move(stage);
  }
  __device__ __forceinline__ void move(uint32_t by) {
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) {
      at[kk] += by;
      asm volatile("" : "+v"(at[kk]));  // the row offsets stay immediates
    }
  }
  __device__ __forceinline__ half8_t get(int kk, int half) const {
    return *(lds_half8_t*)(uintptr_t)(at[kk] + (uint32_t)(half * 32 * D * 2));
  }
};
// tt_off stage read transposed: fragment (kk, u) is the A operand T[d][8 token slots] (T = the
// stage transposed) of tokens k0 = 16 kk .., columns d0 = 32 u ..
// Lane l supplies d = d0 + l % 32 and tokens k0 + 4 (l / 32) + {0..3, 8..11}, the slot order of an
// accumulator's rows (acc_row). ds_read_b64_tr_b16 gives lane i of each 16-lane group element
// i % 4 of the 4 halves read by lane 4 j + i / 4 of the group, as its element j; so lane p of the
// group reads row (first token) + p / 4, columns (group's first d) + 4 (p % 4) .. + 3.
template <int D>
struct TrFrags {
  uint32_t lo[D / 32], hi[D / 32];
  __device__ __forceinline__ void set(uint32_t stage, int lane) {
    const int p = lane & 15, col = 16 * ((lane >> 4) & 1) + 4 * (p & 3);
    const uint32_t l0 =
        (uint32_t)(2 * (tt_off<D>(4 * (lane >> 5) + (p >> 2), col >> 3) + (col & 7)));
#pragma unroll
    for (int u = 0; u < D / 32; ++u) {
      lo[u] = l0 ^ (uint32_t)(64 * u);
      hi[u] = l0 ^ (uint32_t)(64 * u + 32);  // eight rows on: two chunks flipped
    }
    move(stage);
  }
  __device__ __forceinline__ void move(uint32_t by) {
#pragma unroll
    for (int u = 0; u < D / 32; ++u) {
      lo[u] += by;
      hi[u] += by;
      asm volatile("" : "+v"(lo[u]), "+v"(hi[u]));
    }
  }
  __device__ __forceinline__ half8_t get(int kk, int u) const {
    const uint32_t a0 = lo[u] + (uint32_t)(16 * kk * D * 2);
    const uint32_t a1 = hi[u] + (uint32_t)((16 * kk + 8) * D * 2);
    const short4_t x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(uintptr_t)a0);
    const short4_t y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(uintptr_t)a1);
    return __builtin_bit_cast(half8_t, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
  }
};

// The DMA of ROWS-row blocks of a token-major matrix by NW wavefronts (ROWS / NW rows each) into a
// swizzled [ROWS][D] stage (rm_off, or TT: tt_off).
template <int D, int ROWS, int NW, bool TT>
struct BlockDma {
  static constexpr int CPR = D / 8, RPI = 64 / CPR, RW = ROWS / NW;
  static constexpr int N = RW / RPI;  // instructions a wavefront
  static_assert(RW % RPI == 0 && RW <= 16, "whole instructions, rows of one swizzle period");
  uint32_t off;    // lane byte offset of instruction 0's rows of the block in the sequence
  uint32_t row_b;  // bytes of one instruction's rows
  __device__ __forceinline__ void init(int row0, int stride_b, int lane, int wave) {
    const int r = RW * wave + lane / CPR;
    const int o = TT ? tt_off<D>(r, lane % CPR) : rm_off<D>(r, lane % CPR);  // XOR: an involution
    off = (uint32_t)((row0 + r) * stride_b + (o - r * D) * 2);
    row_b = (uint32_t)(RPI * stride_b);
  }
  // Instruction J's rows swizzle as instruction 0's with some chunk bits flipped (an XOR of the
  // byte offset: the rows themselves are whole multiples of CPR chunks apart).
  template <int J>
  static constexpr uint32_t flip() {
    const int r = RPI * J;  // (RW wave: the flip does not depend on it, RW J' < 16 rows apart)
    return (uint32_t)(2 * (TT ? tt_off<D>(r, 0) - r * D : rm_off<D>(r, 0) - r * D));
  }
  template <int J>
  __device__ __forceinline__ void issue(rsrc_t src, uint32_t lds, int wave) const {
    dma16<J>(src, (off ^ flip<J>()) + J * row_b, lds + (uint32_t)(RW * wave * D * 2));
  }
  __device__ __forceinline__ void step(uint32_t bytes) {
    off += bytes;
    asm volatile("" : "+v"(off));  // the other offsets are formed when they are used
  }
};

// Steps of the probabilities done before product q of the ns that form the next block's scores.
constexpr int p_of(int q, int ns) {
  return q < ns / 2 ? q * 8 / (ns / 2) : 8 + (q - ns / 2) * 4 / (ns / 2);
}

template <int D, int NW>
__global__ __launch_bounds__(64 * NW, 2) void attn_fwd_kernel(Args a) {
  constexpr int KC = D / 16, DT = D / 32, kStage = kKB * D;
  typedef BlockDma<D, kKB, NW, false> KDma;
  typedef BlockDma<D, kKB, NW, true> VDma;
  constexpr int NI = KDma::N;
  constexpr int kAhead = 3;  // fragment reads issued ahead of their MFMAs
  __shared__ __align__(1024) uint16_t smem[4 * kStage];  // two K stages, two V stages
  const int G = a.HQ / a.KH;
  // blockIdx.x = rank pairs + (seq KH + kvh - rank) mod pairs: the longest rows of every sequence
  // first (a late long one would end last), and since the dispatcher deals consecutive workgroups
  // to the 8 XCDs in turn, a sequence's groups move on by one XCD a rank
  const int pairs = gridDim.x / a.ntiles, rank = blockIdx.x / pairs;
  const int sh = ((int)blockIdx.x - rank * pairs + rank) % pairs, grp = a.ntiles - 1 - rank;
  const int seq = sh / a.KH, kvh = sh % a.KH;
  const int start = a.cu[seq], L = a.cu[seq + 1] - start;
  const int total = (L + kTok - 1) / kTok * G;
  if (grp * NW >= total) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto blocks_of = [&](int f) { return (min(f / G * kTok + kTok, L) + kKB - 1) / kKB; };
  const int nkb = blocks_of(min(grp * NW + NW - 1, total - 1));  // of the longest tile
  const int ch = blockIdx.z;
  if (ch >= num_chunks(nkb, a.chunk)) return;
  const int kb0 = ch * a.chunk, kb1 = num_chunks(nkb, a.chunk) == 1 ? nkb : min(nkb, kb0 + a.chunk);

  const int64_t qs = (int64_t)a.HQ * D, kvs = (int64_t)a.KH * D;
  const int kvs_b = (int)(kvs * 2);
  const rsrc_t ksrc = rows_rsrc(a.k + (int64_t)start * kvs + kvh * D, L, kvs, D);
  const rsrc_t vsrc = rows_rsrc(a.v + (int64_t)start * kvs + kvh * D, L, kvs, D);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem;
  KDma kd;
  VDma vd;
  kd.init(kb0 * kKB, kvs_b, lane, wave);
  vd.init(kb0 * kKB, kvs_b, lane, wave);
  const uint32_t blk_b = (uint32_t)(kKB * kvs_b);
  // stage s (0, 1) of K and V
  auto k_lds = [&](int s) { return lds0 + (uint32_t)(s * kStage * 2); };
  auto v_lds = [&](int s) { return lds0 + (uint32_t)((2 + s) * kStage * 2); };
  auto dma_k = [&](int s) {
    static_for<NI>([&](auto j) { kd.template issue<j.value>(ksrc, k_lds(s), wave); });
    kd.step(blk_b);
  };
  dma_k(0);
  if (kb0 + 1 < kb1) dma_k(1);
  static_for<NI>([&](auto j) { vd.template issue<j.value>(vsrc, v_lds(0), wave); });
  vd.step(blk_b);

  // the wavefront's tile: q head, first query, this lane's query and the last key it attends to;
  // past the last tile: the last one again, not stored
  const int f = grp * NW + wave, fc = min(f, total - 1);
  const int h = kvh * G + __builtin_amdgcn_readfirstlane(fc % G);
  const int q0 = __builtin_amdgcn_readfirstlane(fc / G) * kTok;
  const int qi = q0 + (lane & 31), lim = min(qi, L - 1);
  const int nch = num_chunks(blocks_of(fc), a.chunk);
  const bool live = f < total && ch < nch;
  // the wavefront's blocks end here
  const int kbw = __builtin_amdgcn_readfirstlane(live ? min(blocks_of(fc), kb1) : kb0);
  half8_t qr[KC];  // queries past the sequence read zeros (their rows are not stored)
  if (live)
    load_token<D>(rows_rsrc(a.q + (int64_t)start * qs + h * D, L, qs, D), qi, (int)(qs * 2), lane,
                  qr);
  f32x16 o[DT], s[2], sn[2];
  half8_t pb[4];
  float m = 0.f, mx = 0.f, alpha = 1.f, lsum = 0.f, ps = 0.f;
  const float c = a.scale * kLog2e;
#pragma unroll
  for (int u = 0; u < DT; ++u) o[u] = f32x16{};

  // K fragment f = half KC + kk (half: of the 64 keys) and V fragment f = kk DT + u of a stage
  half8_t kf[2 * KC], vf[4 * DT];
  RowFrags<D> kat;
  TrFrags<D> vat;
  kat.set(k_lds(0), lane);
  vat.set(v_lds(0), lane);
  auto read_k = [&](auto i) { kf[i.value] = kat.get(i.value % KC, i.value / KC); };
  auto read_v = [&](auto i) { vf[i.value] = vat.get(i.value / DT, i.value % DT); };
  // MFMA q of S = K Q^T: fragment q
  auto s_mfma = [&](auto qc, f32x16 (&x)[2]) {
    constexpr int kk = qc.value % KC, hf = qc.value / KC;
    x[hf] = mfma(kf[qc.value], qr[kk], kk == 0 ? f32x16{} : x[hf]);
  };
  // a block on the diagonal: keys past the query are masked
  auto mask = [&](f32x16 (&x)[2], int k0) {
    const int d = lim - k0 - 4 * (lane >> 5);  // acc_row(r, lane) is acc_row(r, 0) past that
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        x[hf][r] = 32 * hf + acc_row(r, 0) > d ? -__builtin_inff() : x[hf][r];
  };
  // Step i (0 .. 15) of the block's maximum: two values.
  auto max_step = [&](auto ic, const f32x16 (&x)[2]) {
    constexpr int hf = ic.value >> 3, r = 2 * (ic.value & 7);
    mx = max3(ic.value == 0 ? -__builtin_inff() : mx, x[hf][r], x[hf][r + 1]);
  };
  // Step i (0 .. 15) of the block's probabilities: two values of P fragment i / 4. The state is in
  // log2 units of the scaled scores.
  auto p_step = [&](auto ic, const f32x16 (&x)[2]) {
    constexpr int kk = ic.value >> 2, e = 2 * (ic.value & 3);
    const float p0 = ex2(fmaf(x[kk >> 1][8 * (kk & 1) + e], c, -m));
    const float p1 = ex2(fmaf(x[kk >> 1][8 * (kk & 1) + e + 1], c, -m));
    ps += p0;
    ps += p1;
    uint4 w = __builtin_bit_cast(uint4, pb[kk]);
    (e == 0 ? w.x : e == 2 ? w.y : e == 4 ? w.z : w.w) = cvt2h(p0, p1);
    pb[kk] = __builtin_bit_cast(half8_t, w);
  };

  int cur = 0;                                // the stage of K(b) and V(b); b + 1's is the other
  uint32_t k_at = k_lds(0), v_at = v_lds(0);  // the stages kat and vat address
  // The loads of K(b + 2) and V(b + 1), when every wavefront is done with b - 1.
  auto load = [&]() {
    static_for<NI>([&](auto j) {
      kd.template issue<j.value>(ksrc, k_lds(cur), wave);
      vd.template issue<j.value>(vsrc, v_lds(cur ^ 1), wave);
    });
    kd.step(blk_b);
    vd.step(blk_b);
  };
  // Block b: its scores (masked) in x and their maximum in mx; the next block's go to xn and mx.
  // last: there is none for this wavefront; masked: the next block reaches past the first query.
  auto block = [&](auto last, auto masked, int b, f32x16 (&x)[2], f32x16 (&xn)[2]) {
    constexpr bool kLast = last.value;
    const int next = cur ^ 1;
    constexpr int NS = 2 * KC, NV = 4 * DT;  // MFMAs of S and of P V
    sync_tile<0>();  // K(b + 1) and V(b) landed, every wavefront is done with b - 1
    if (!kLast) kat.move(k_lds(next) - k_at);
    k_at = k_lds(next);
    vat.move(v_lds(cur) - v_at);
    v_at = v_lds(cur);
    if (!kLast) static_for<kAhead>([&](auto i) { read_k(i); });
    else static_for<kAhead>([&](auto i) { read_v(i); });
    const float mn = fmaxf(m, mx * c);
    alpha = ex2(m - mn);
    m = mn;
    if (__any(alpha != 1.f)) {  // once the running maxima settle, many blocks skip this
#pragma unroll
      for (int u = 0; u < DT; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[u][r] *= alpha;
    }
    if constexpr (!kLast) {
      __builtin_amdgcn_sched_barrier(0);
      static_for<NS>([&](auto qc) {
        constexpr int q = qc.value;
        s_mfma(qc, xn);
        if constexpr (q + kAhead < 2 * KC) read_k(std::integral_constant<int, q + kAhead>{});
        else read_v(std::integral_constant<int, q + kAhead - 2 * KC>{});
        // the probabilities of the first half's keys behind the first half's products (their
        // scores' registers are then free for the second half's), half of the others' behind the
        // second half's; the loads of K(b + 2), V(b + 1)
        static_for<p_of(q + 1, NS) - p_of(q, NS)>([&](auto i) {
          p_step(std::integral_constant<int, p_of(q, NS) + i.value>{}, x);
        });
        if constexpr (q % 4 == 3 && q / 4 < NI)
          kd.template issue<q / 4 < NI ? q / 4 : 0>(ksrc, k_lds(cur), wave);
        if constexpr (q % 4 == 1 && q / 4 < NI)
          vd.template issue<q / 4 < NI ? q / 4 : 0>(vsrc, v_lds(next), wave);
        __builtin_amdgcn_sched_barrier(0);
      });
      kd.step(blk_b);
      vd.step(blk_b);
    } else {
      if (b + 1 < kb1) load();
      static_for<12>([&](auto i) { p_step(i, x); });
    }
    // P V: behind the first half of its products the rest of the probabilities, behind the second
    // the next block's maximum
    __builtin_amdgcn_sched_barrier(0);
    static_for<NV>([&](auto qc) {
      constexpr int q = qc.value, kk = q / DT, u = q % DT, half = NV / 2;
      o[u] = mfma(vf[q], pb[kk], o[u]);
      if constexpr (q + kAhead < NV) read_v(std::integral_constant<int, q + kAhead>{});
      if constexpr (q < half) {
        static_for<(q + 1) * 4 / half - q * 4 / half>([&](auto i) {
          p_step(std::integral_constant<int, 12 + q * 4 / half + i.value>{}, x);
        });
      } else if constexpr (!kLast) {
        if constexpr (q == half) {
          // max3 is assembly, whose operands the compiler does not wait for: read no earlier than
          // here, half of P V after the last product of S
          asm volatile("" : "+v"(xn[0]), "+v"(xn[1]));
          if constexpr (masked.value) mask(xn, (b + 1) * kKB);
        }
        static_for<(q + 1 - half) * 16 / half - (q - half) * 16 / half>([&](auto i) {
          max_step(std::integral_constant<int, (q - half) * 16 / half + i.value>{}, xn);
        });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    lsum = lsum * alpha + ps;
    ps = 0.f;
    if constexpr (!kLast) mx = pair_max(mx);
    cur = next;
  };

  if (kb0 + 1 < kb1) sync_tile<2 * NI>();  // K(kb0) landed
  else sync_tile<NI>();
  int b = kb0;
  if (b < kbw) {
    // the first block's scores and maximum
    static_for<2 * KC>([&](auto i) { read_k(i); });
    static_for<2 * KC>([&](auto q) { s_mfma(q, s); });
    // max3 is assembly: the products' latency is waited for here
    asm volatile("s_nop 15\n\ts_nop 15" : "+v"(s[0]), "+v"(s[1]));
    mask(s, kb0 * kKB);
    static_for<16>([&](auto i) { max_step(i, s); });
    mx = pair_max(mx);
    m = mx * c;
    // masked from the first block that reaches past the first query on
    const int edge = min(q0 / kKB, kbw - 1);
    const std::false_type no;
    const std::true_type yes;
    for (; b + 2 < edge; b += 2) {  // in pairs: no score changes its registers
      block(no, no, b, s, sn);
      block(no, no, b + 1, sn, s);
    }
    for (; b + 1 < kbw; ++b) {
      block(no, yes, b, s, sn);
      s[0] = sn[0];
      s[1] = sn[1];
    }
    block(yes, no, b, s, sn);
    ++b;
  }
  // Blocks past the wavefront's own: loaded for the others. (Their P would be 0, but 0 times a
  // value that is not finite is NaN: it may not reach queries before its key's block.)
  for (; b < kb1; ++b) {
    sync_tile<0>();
    if (b + 1 < kb1) load();
    cur ^= 1;
  }
  __builtin_amdgcn_s_waitcnt(0);  // loads past the range: none in flight when the wavefront ends
  const float ltot = lsum + __shfl_xor(lsum, 32, 64);
  if (!live || qi >= L) return;
  if (nch == 1) {
    store_token_row<D>(a.out + (int64_t)(start + qi) * qs + h * D, o, 1.0f / ltot, lane);
    if (lane < 32) a.lse[(int64_t)h * a.n + start + qi] = (m + log2f(ltot)) * kLn2;
    return;
  }
  // Several chunks: this one's unnormalised partial and (m, l). Every chunk of a tile holds at
  // least one unmasked key of each query (the last one starts at or before the tile's first query:
  // q0 is a multiple of 32, blocks are 64 keys; the others precede it), so m is finite.
  store_token_row_f32<D>(a.part + (((int64_t)ch * a.n + start + qi) * a.HQ + h) * D, o, lane);
  if (lane < 32) a.part_ml[((int64_t)ch * a.HQ + h) * a.n + start + qi] = make_float2(m, ltot);
}

// ------------------------------------------------------------------------------------------------
// Backward, delta = rowsum(dO * O) per (q head, token), fp32 [HQ, n], read by both the dQ and the
// dK/dV kernel (which may then run at the same time). Two threads per row: thread `half` sums
// the products of the 16-byte chunks 2 kk + half (kk = 0 .. D/16 - 1) in order, then the pair's
// two sums are added.
// ------------------------------------------------------------------------------------------------
template <int D>
__global__ __launch_bounds__(256) void attn_delta_kernel(const uint16_t* dout, const uint16_t* o,
                                                         float* delta, int64_t n, int HQ) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t p = t >> 1;  // h n + token
  const int half = (int)(t & 1);
  const bool ok = p < n * HQ;
  float s = 0.f;
  if (ok) {
    const int64_t h = p / n, tok = p - h * n;
    const uint4* dr = reinterpret_cast<const uint4*>(dout + (tok * HQ + h) * D);
    const uint4* orow = reinterpret_cast<const uint4*>(o + (tok * HQ + h) * D);
    uint4 x[D / 16], y[D / 16];
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) {
      x[kk] = dr[2 * kk + half];
      y[kk] = orow[2 * kk + half];
    }
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const uint32_t xa = word_of(x[kk], w), ya = word_of(y[kk], w);
        s += lo_h(xa) * lo_h(ya);
        s += hi_h(xa) * hi_h(ya);
      }
  }
  const float tot = s + __shfl_xor(s, 1, 64);
  if (ok && half == 0) delta[p] = tot;
}

// ------------------------------------------------------------------------------------------------
// Staging of the backward kernels: blocks of 32 rows of two token-major matrices with the same
// rows and stride (K and V for dQ, Q and dO for dK/dV), as one [64][D] tt_off stage of LDS: rows
// 0-31 the first matrix, 32-63 the second, so that one set of fragment addresses reaches both
// (RowFrags: (kk, matrix), TrFrags: (kk + 2 matrix, u)).
// ------------------------------------------------------------------------------------------------
template <int D, int NW>
struct PairDma {
  typedef BlockDma<D, kTok, NW, true> Dma;
  static constexpr int N = 2 * Dma::N;           // instructions a wavefront and block
  static constexpr uint32_t kHalf = kTok * D * 2, kStage = 2 * kHalf;  // bytes
  Dma d;
  __device__ __forceinline__ void init(int row0, int stride_b, int lane, int wave) {
    d.init(row0, stride_b, lane, wave);
  }
  template <int J>
  __device__ __forceinline__ void issue(rsrc_t first, rsrc_t second, uint32_t stage,
                                        int wave) const {
    if constexpr (J < Dma::N) d.template issue<J>(first, stage, wave);
    else d.template issue<J - Dma::N>(second, stage + kHalf, wave);
  }
};

// The wait for the first of `blocks` blocks, up to three of them in flight (NL loads each): a block
// that is not there is not loaded, and its loads do not count.
template <int NL>
__device__ __forceinline__ void first_block(int blocks) {
  if (blocks >= 3) sync_tile<2 * NL>();
  else sync_tile<0>();
}

// Halves 2 i and 2 i + 1 of a fragment.
__device__ __forceinline__ void set_pair(half8_t& f, int i, uint32_t pair) {
  uint4 w = __builtin_bit_cast(uint4, f);
  (i == 0 ? w.x : i == 1 ? w.y : i == 2 ? w.z : w.w) = pair;
  f = __builtin_bit_cast(half8_t, w);
}

// Steps of a block's dS (of 8) formed before MFMA q of the 3 D / 16 they hide behind: the second
// half of the dQ products of the block before, the next block's S and dP, the first half of its own
// dQ.
template <int D>
constexpr int ds_before(int q) {
  return q * 8 / (3 * D / 16);
}

// ------------------------------------------------------------------------------------------------
// Backward, dQ: per 32 queries of a q head, over 32-key blocks up to the diagonal: S^T = K Q^T,
// P = exp(S - lse), dP^T = V dO^T, dS = P (dP - delta), dQ^T += K^T dS^T. Workgroups, their order
// and the chunks as the forward. Block b's dS is formed a few instructions at a time (ds_step)
// behind the MFMAs of block b + 1's S and dP and of block b's dQ, as in attn_dkdv_kernel; K and V
// arrive by LDS DMA, four stages, one barrier a block, and masks start at the diagonal.
// MI355X, against one q head group per workgroup, staging through registers and two barriers a block,
// kernel averages: sequences of 4,096 and 3,001 tokens, 12/2 heads of 128, 194 -> 140 us, 14/2 of 64
// 126 -> 91; four of 283-997 (beside dK/dV before, in turn now) 44 -> 31 and 27 -> 19.
// OWN_DELTA: the kernel forms delta itself (lanes l and l ^ 32 sum the chunks of
// attn_delta_kernel's two threads, in its order) and the first chunk writes it for the dK/dV
// kernel that follows; else it reads attn_delta_kernel's.
// ------------------------------------------------------------------------------------------------
template <int D, int NW, bool OWN_DELTA>
__global__ __launch_bounds__(64 * NW, 2) void attn_dq_kernel(Args a) {
  constexpr int KC = D / 16, DT = D / 32, kStages = 4;
  typedef PairDma<D, NW> Dma;
  constexpr int NL = Dma::N;  // loads a wavefront and block
  __shared__ __align__(1024) uint8_t smem[kStages * Dma::kStage];
  const int G = a.HQ / a.KH;
  const int pairs = gridDim.x / a.ntiles, rank = blockIdx.x / pairs;  // as the forward
  const int sh = ((int)blockIdx.x - rank * pairs + rank) % pairs, grp = a.ntiles - 1 - rank;
  const int seq = sh / a.KH, kvh = sh % a.KH;
  const int start = a.cu[seq], L = a.cu[seq + 1] - start;
  const int total = (L + kTok - 1) / kTok * G;
  if (grp * NW >= total) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto blocks_of = [&](int f) { return f / G + 1; };  // key blocks are as long as query tiles
  const int nkb = blocks_of(min(grp * NW + NW - 1, total - 1));  // of the longest tile
  const int ch = blockIdx.z;
  if (ch >= num_chunks(nkb, a.chunk)) return;
  const int kb0 = ch * a.chunk, kb1 = num_chunks(nkb, a.chunk) == 1 ? nkb : min(nkb, kb0 + a.chunk);

  const int64_t qs = (int64_t)a.HQ * D, kvs = (int64_t)a.KH * D;
  const int qs_b = (int)(qs * 2), kvs_b = (int)(kvs * 2);
  const rsrc_t ksrc = rows_rsrc(a.k + (int64_t)start * kvs + kvh * D, L, kvs, D);
  const rsrc_t vsrc = rows_rsrc(a.v + (int64_t)start * kvs + kvh * D, L, kvs, D);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem;
  Dma dma;
  dma.init(kb0 * kTok, kvs_b, lane, wave);
  auto stage_at = [&](int b) { return lds0 + (uint32_t)(b & (kStages - 1)) * Dma::kStage; };
  auto load = [&](auto j, int b) {  // load j of block b; the last moves to the next block
    dma.template issue<j.value>(ksrc, vsrc, stage_at(b), wave);
    if constexpr (j.value == NL - 1) dma.d.step((uint32_t)(kTok * kvs_b));
  };
  for (int b = kb0; b < min(kb0 + 3, kb1); ++b) static_for<NL>([&](auto j) { load(j, b); });

  // the wavefront's tile, as the forward: past the last tile the last one again, not stored
  const int f = grp * NW + wave, fc = min(f, total - 1);
  const int h = kvh * G + __builtin_amdgcn_readfirstlane(fc % G);
  const int q0 = __builtin_amdgcn_readfirstlane(fc / G) * kTok;
  const int qi = q0 + (lane & 31), lim = min(qi, L - 1);
  const int nch = num_chunks(blocks_of(fc), a.chunk);
  const bool live = f < total && ch < nch;
  // the wavefront's blocks end here
  const int kbw = __builtin_amdgcn_readfirstlane(live ? min(blocks_of(fc), kb1) : kb0);

  // this query's q and dO (queries past the sequence read zeros; their dq is not stored), its
  // log-sum-exp and delta (attn_delta_kernel)
  const int64_t hoff = (int64_t)start * qs + h * D;
  half8_t qr[KC], dr[KC];
  float lse2 = 0.f, delta = 0.f;
  if (live) {
    load_token<D>(rows_rsrc(a.q + hoff, L, qs, D), qi, qs_b, lane, qr);
    load_token<D>(rows_rsrc(a.dout + hoff, L, qs, D), qi, qs_b, lane, dr);
    lse2 = buf_load_f32(make_rsrc(a.lse + (int64_t)h * a.n + start, (uint32_t)L * 4), qi * 4) *
           kLog2e;
    if constexpr (OWN_DELTA) {
      half8_t orow[KC];
      load_token<D>(rows_rsrc(a.o + hoff, L, qs, D), qi, qs_b, lane, orow);
      float dpart = 0.f;
#pragma unroll
      for (int kk = 0; kk < KC; ++kk)
#pragma unroll
        for (int i = 0; i < 8; ++i) dpart += (float)dr[kk][i] * (float)orow[kk][i];
      delta = dpart + __shfl_xor(dpart, 32, 64);
      if (ch == 0 && qi < L && lane < 32) a.delta[(int64_t)h * a.n + start + qi] = delta;
    } else {
      delta = buf_load_f32(make_rsrc(a.delta + (int64_t)h * a.n + start, (uint32_t)L * 4), qi * 4);
    }
  }

  f32x16 dq[DT], s[2], sn[2];  // s: S and dP
#pragma unroll
  for (int u = 0; u < DT; ++u) dq[u] = f32x16{};
  const float c = a.scale * kLog2e;
  half8_t sb[2];  // dS fragments
  RowFrags<D, true> rat;
  TrFrags<D> tat;
  uint32_t r_at = stage_at(kb0), t_at = r_at;  // the stages rat and tat address
  rat.set(r_at, lane);
  tat.set(t_at, lane);
  half8_t rf[2 * KC], tf[2 * DT];
  // MFMA q of S, dP: row fragment q (even: K, odd: V); of dQ: transposed fragment q (first the
  // first 16 keys)
  auto read_r = [&](auto i) { rf[i.value] = rat.get(i.value >> 1, i.value & 1); };
  auto read_t = [&](auto i) { tf[i.value] = tat.get(i.value / DT, i.value % DT); };
  auto s_mfma = [&](auto qc, f32x16 (&x)[2]) {
    constexpr int kk = qc.value >> 1, t = qc.value & 1;
    x[t] = mfma(rf[qc.value], t ? dr[kk] : qr[kk], kk == 0 ? f32x16{} : x[t]);
  };
  // dS of keys acc_row(2 k) and the next (k = 0 .. 7)
  auto ds_step = [&](auto kc, f32x16 (&x)[2]) {
    constexpr int r = 2 * kc.value;
    const float p0 = ex2(fmaf(x[0][r], c, -lse2)), p1 = ex2(fmaf(x[0][r + 1], c, -lse2));
    set_pair(sb[r >> 3], (r & 7) >> 1, cvt2h(p0 * (x[1][r] - delta), p1 * (x[1][r + 1] - delta)));
  };
  // keys past the query: P = dS = 0
  auto mask = [&](int b, f32x16 (&x)[2]) {
    const int d = lim - b * kTok - 4 * (lane >> 5);
#pragma unroll
    for (int r = 0; r < 16; ++r) x[0][r] = acc_row(r, 0) > d ? -__builtin_inff() : x[0][r];
  };
  constexpr int NS = 2 * KC, NV = 2 * DT, half = NV / 2;  // MFMAs of S and dP, of dQ
  constexpr int kAhead = 3;  // fragment reads issued ahead of their MFMAs

  // Block b, its S and dP in x and the first steps of its dS done: the next block's go to xn.
  // last: there is none for this wavefront; masked: it reaches past the first query.
  auto block = [&](auto last, auto masked, int b, f32x16 (&x)[2], f32x16 (&xn)[2]) {
    constexpr bool kLast = last.value;
    sync_tile<NL>();  // block b + 1 landed, every wavefront is done with b - 1
    if (!kLast) {
      rat.move(stage_at(b + 1) - r_at);
      r_at = stage_at(b + 1);
    }
    tat.move(stage_at(b) - t_at);
    t_at = stage_at(b);
    if constexpr (!kLast) {
      static_for<kAhead>([&](auto i) { read_r(i); });
      __builtin_amdgcn_sched_barrier(0);
      static_for<NS>([&](auto qc) {
        constexpr int q = qc.value, p = ds_before<D>(half + q);
        s_mfma(qc, xn);
        if constexpr (q + kAhead < NS) read_r(std::integral_constant<int, q + kAhead>{});
        else read_t(std::integral_constant<int, q + kAhead - NS>{});
        static_for<ds_before<D>(half + q + 1) - p>([&](auto i) {
          ds_step(std::integral_constant<int, p + i.value>{}, x);
        });
        if constexpr (q % 3 == 1 && q / 3 < NL) load(std::integral_constant<int, q / 3>{}, b + 3);
        __builtin_amdgcn_sched_barrier(0);
      });
    } else {
      if (b + 1 < kb1) static_for<NL>([&](auto j) { load(j, b + 3); });
      static_for<kAhead>([&](auto i) { read_t(i); });
      static_for<ds_before<D>(half + NS) - ds_before<D>(half)>([&](auto i) {
        ds_step(std::integral_constant<int, ds_before<D>(half) + i.value>{}, x);
      });
      __builtin_amdgcn_sched_barrier(0);
    }
    static_for<NV>([&](auto qc) {
      constexpr int q = qc.value, kk = q / DT, u = q % DT;
      dq[u] = mfma(tf[q], sb[kk], dq[u]);
      if constexpr (q + kAhead < NV) read_t(std::integral_constant<int, q + kAhead>{});
      if constexpr (q < half) {
        constexpr int p = ds_before<D>(half + NS + q);
        static_for<ds_before<D>(half + NS + q + 1) - p>([&](auto i) {
          ds_step(std::integral_constant<int, p + i.value>{}, x);
        });
        if constexpr (!kLast && masked.value && q == half - 1) mask(b + 1, xn);
      } else if constexpr (!kLast) {
        constexpr int p = ds_before<D>(q - half);
        static_for<ds_before<D>(q - half + 1) - p>([&](auto i) {
          ds_step(std::integral_constant<int, p + i.value>{}, xn);
        });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  static_assert(3 * (NL - 1) + 1 < NS, "a block's loads are issued behind S and dP");
  static_assert(ds_before<D>(half + NS) >= 4, "the first 16 keys' dS is whole before dQ");

  first_block<NL>(kb1 - kb0);
  int b = kb0;
  if (b < kbw) {
    static_for<NS>([&](auto i) { read_r(i); });
    static_for<NS>([&](auto q) { s_mfma(q, s); });
    mask(kb0, s);
    static_for<ds_before<D>(half)>([&](auto i) { ds_step(i, s); });
    const std::false_type no;
    const std::true_type yes;
    const int edge = min(q0 / kTok, kbw - 1);
    for (; b + 2 < edge; b += 2) {  // in pairs: no product changes its registers
      block(no, no, b, s, sn);
      block(no, no, b + 1, sn, s);
    }
    for (; b + 1 < kbw; ++b) {
      block(no, yes, b, s, sn);
      s[0] = sn[0];
      s[1] = sn[1];
    }
    block(yes, no, b, s, sn);
    ++b;
  }
  // blocks past the wavefront's own: loaded for the others (as the forward)
  for (; b < kb1; ++b) {
    sync_tile<NL>();
    static_for<NL>([&](auto j) { load(j, b + 3); });
  }
  __builtin_amdgcn_s_waitcnt(0);  // loads past the range: none in flight when the wavefront ends
  if (!live || qi >= L) return;
  if (nch == 1) {
    store_token_row<D>(a.out + (int64_t)(start + qi) * qs + h * D, dq, a.scale, lane);
    return;
  }
  // several chunks: this one's unscaled partial
  store_token_row_f32<D>(a.part + (((int64_t)ch * a.n + start + qi) * a.HQ + h) * D, dq, lane);
}

// ------------------------------------------------------------------------------------------------
// Merge of the chunks' partials, in chunk order. Forward: M = max m_c, l = sum l_c 2^(m_c - M),
// O = sum o_c 2^(m_c - M) / l, lse = (M + log2 l) ln 2; dQ: dq = scale sum dq_c. One thread per
// 4 columns of a query row: all C chunk loads are issued before any use (chunks past the tile's
// count read the last one again and weigh 0). blockIdx.x = tile + ntiles (q head of the group +
// G (seq KH + kvh)), block 32 D/4; tiles of one chunk were written directly and are skipped.
// ------------------------------------------------------------------------------------------------
template <int D, int C, bool FWD>
__global__ __launch_bounds__(32 * D / 4) void attn_merge_kernel(Args a) {
  constexpr int D4 = D / 4, KBLK = FWD ? kKB : kTok;
  const int G = a.HQ / a.KH;
  const int rest = blockIdx.x / a.ntiles;
  const int tile = (int)(blockIdx.x - rest * a.ntiles);
  const int g = rest % G, sh = rest / G;
  const int seq = sh / a.KH, h = (sh % a.KH) * G + g;
  const int q0 = tile * kTok;
  const int start = a.cu[seq], L = a.cu[seq + 1] - start;
  if (q0 >= L) return;
  const int kend = min(q0 + kTok, L);
  const int nch = num_chunks((kend + KBLK - 1) / KBLK, a.chunk);
  const int qi = q0 + (int)(threadIdx.x / D4), d4 = (int)(threadIdx.x % D4);
  if (nch == 1 || qi >= L) return;
  const int64_t cstride = a.n * a.HQ * D, mstride = (int64_t)a.HQ * a.n;
  const float* src = a.part + ((int64_t)(start + qi) * a.HQ + h) * D + 4 * d4;
  float4 x[C];
  float w[C];
#pragma unroll
  for (int c = 0; c < C; ++c) x[c] = *reinterpret_cast<const float4*>(src + min(c, nch - 1) * cstride);
  float M = 0.f, l = 0.f;
  if constexpr (FWD) {
    const float2* ml = a.part_ml + (int64_t)h * a.n + start + qi;
    float2 y[C];
#pragma unroll
    for (int c = 0; c < C; ++c) y[c] = ml[min(c, nch - 1) * mstride];
    M = -__builtin_inff();
#pragma unroll
    for (int c = 0; c < C; ++c) M = fmaxf(M, y[c].x);  // repeats of the last chunk change nothing
#pragma unroll
    for (int c = 0; c < C; ++c) {
      w[c] = c < nch ? ex2(y[c].x - M) : 0.f;
      l += y[c].y * w[c];
    }
    const float inv = 1.0f / l;
#pragma unroll
    for (int c = 0; c < C; ++c) w[c] *= inv;
  } else {
#pragma unroll
    for (int c = 0; c < C; ++c) w[c] = c < nch ? a.scale : 0.f;
  }
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int c = 0; c < C; ++c) {
    acc.x += w[c] * x[c].x;
    acc.y += w[c] * x[c].y;
    acc.z += w[c] * x[c].z;
    acc.w += w[c] * x[c].w;
  }
  *reinterpret_cast<uint2*>(a.out + ((int64_t)(start + qi) * a.HQ + h) * D + 4 * d4) =
      make_uint2(pack2h(acc.x, acc.y), pack2h(acc.z, acc.w));
  if (FWD && d4 == 0) a.lse[(int64_t)h * a.n + start + qi] = (M + log2f(l)) * kLn2;
}

// ------------------------------------------------------------------------------------------------
// Backward, dK and dV of one q head: a workgroup of 4 wavefronts owns 128 consecutive keys (32
// per wavefront) and walks the 32-query blocks from its first key to the end of the sequence:
// S = Q K^T, P = exp(S - lse), dP = dO V^T, dS = P (dP - delta), dV^T += dO^T P, dK^T += Q^T dS.
//
// dK, dV, K and V take 192 registers a lane (D = 128), so one wavefront runs per SIMD and a block's
// own products cannot hide its exponentials: block b's P and dS are formed a few instructions at a
// time (p_sub) behind the MFMAs of block b + 1's S and dP and of block b's dV and dK, every
// instruction pinned behind an MFMA by sched_barrier. Per block and wavefront 32 MFMAs (D = 128;
// 1,024 cycles of the matrix core) stand beside about 150 VALU instructions. Q and dO arrive by LDS
// DMA, four stages (two blocks' time to land), one barrier a block. A wavefront skips the query
// blocks before its keys; its first block (the diagonal) and its last (rows past the sequence, which
// read zeros) are masked, the others run without.
// MI355X, against two barriers a block, staging through registers and a block's products,
// exponentials and products one after the other, kernel averages: two sequences of 4,096 and 3,001
// tokens, 12/2 heads of 128, 279 -> 212 us, 14/2 of 64 166 -> 129; four of 283-997 (beside dQ before,
// in turn now) 66 -> 41 and 50 -> 29.
// grid (nseq * HQ * ceil(max_len / 128)), block 256.
// ------------------------------------------------------------------------------------------------
constexpr int kKeyWaves = 4;

template <int D>
__global__ __launch_bounds__(64 * kKeyWaves, 1) void attn_dkdv_kernel(Args a) {
  constexpr int KC = D / 16, DT = D / 32, kStages = 4;
  typedef PairDma<D, kKeyWaves> Dma;
  constexpr uint32_t kRowBytes = kStages * Dma::kStage;  // then per stage lse and delta, 64 floats each
  __shared__ __align__(1024) uint8_t smem[kRowBytes + kStages * 512];
  // blockIdx.x = (seq HQ + h) + pairs key tile: the first key tiles of every sequence and head,
  // which walk the most queries, are dispatched first (with more workgroups than CUs, the
  // heaviest then do not wait for a free CU)
  const int pairs = (int)(gridDim.x / a.ntiles);
  const int kt = blockIdx.x / pairs, sh = (int)(blockIdx.x - kt * pairs);
  const int seq = sh / a.HQ, h = sh % a.HQ;
  const int kvh = h / (a.HQ / a.KH);
  const int kw0 = kt * kTok * kKeyWaves;
  const int start = a.cu[seq], L = a.cu[seq + 1] - start;
  if (kw0 >= L) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kj = kw0 + kTok * wave + (lane & 31);
  const int nb = (L - kw0 + kTok - 1) / kTok;  // query blocks
  const int64_t qs = (int64_t)a.HQ * D, kvs = (int64_t)a.KH * D;
  const int qs_b = (int)(qs * 2), kvs_b = (int)(kvs * 2);
  const int64_t hoff = (int64_t)start * qs + h * D;
  const rsrc_t qsrc = rows_rsrc(a.q + hoff, L, qs, D);
  const rsrc_t dsrc = rows_rsrc(a.dout + hoff, L, qs, D);
  // even wavefronts fetch a block's lse, odd ones its delta (64 values, the first 32 are used)
  const rsrc_t rsrc = make_rsrc(((wave & 1) ? a.delta : a.lse) + (int64_t)h * a.n + start,
                                (uint32_t)L * 4);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem;
  const uint32_t row_lds = lds0 + kRowBytes + (uint32_t)(wave & 1) * 256;

  Dma dma;
  dma.init(kw0, qs_b, lane, wave);
  uint32_t row_off = (uint32_t)(kw0 + lane) * 4;
  constexpr int NL = Dma::N + 1;  // loads a wavefront and block
  auto stage_at = [&](int b) { return lds0 + (uint32_t)(b & (kStages - 1)) * Dma::kStage; };
  auto load = [&](auto j, int b) {  // load j of block b (j = NL - 1, the last, moves to the next)
    if constexpr (j.value < Dma::N) {
      dma.template issue<j.value>(qsrc, dsrc, stage_at(b), wave);
    } else {
      dma4(rsrc, row_off, row_lds + (uint32_t)(b & (kStages - 1)) * 512);
      dma.d.step((uint32_t)(kTok * qs_b));
      row_off += kTok * 4;
    }
  };
  // with fewer than three blocks only those there are (first_block)
  for (int b = 0; b < min(3, nb); ++b) static_for<NL>([&](auto j) { load(j, b); });

  half8_t kr[KC], vr[KC];  // keys past the sequence read zeros (their rows are not stored)
  if (wave < nb) {         // (a wavefront of such keys only multiplies nothing)
    const int64_t koff = (int64_t)start * kvs + kvh * D;
    load_token<D>(rows_rsrc(a.k + koff, L, kvs, D), kj, kvs_b, lane, kr);
    load_token<D>(rows_rsrc(a.v + koff, L, kvs, D), kj, kvs_b, lane, vr);
  }
  f32x16 dk[DT], dv[DT], s[2], sn[2];  // s: S and dP
#pragma unroll
  for (int u = 0; u < DT; ++u) dk[u] = dv[u] = f32x16{};
  const float c = a.scale * kLog2e;
  half8_t pb[2], sb[2];  // P and dS fragments
  float4 l4[4], d4[4];   // lse and delta of queries 8 j + 4 (lane / 32) ..
  RowFrags<D, true> rat;
  TrFrags<D> tat;
  rat.set(lds0, lane);
  tat.set(lds0, lane);
  uint32_t r_at = lds0, t_at = lds0;  // the stages rat and tat address
  half8_t rf[2 * KC], tf[4 * DT];
  // MFMA q of S, dP: row fragment q (even: Q, odd: dO); q of dV, dK: transposed fragment q (first
  // the first 16 queries; even: dO, odd: Q)
  auto read_r = [&](auto i) { rf[i.value] = rat.get(i.value >> 1, i.value & 1); };
  auto read_t = [&](auto i) {
    constexpr int kk = i.value / (2 * DT), u = i.value % (2 * DT) >> 1;
    tf[i.value] = tat.get(kk + 2 * (1 - (i.value & 1)), u);
  };
  auto s_mfma = [&](auto qc, f32x16 (&x)[2]) {
    constexpr int kk = qc.value >> 1, t = qc.value & 1;
    x[t] = mfma(rf[qc.value], t ? vr[kk] : kr[kk], kk == 0 ? f32x16{} : x[t]);
  };
  auto g_mfma = [&](auto qc) {
    constexpr int kk = qc.value / (2 * DT), u = qc.value % (2 * DT) >> 1;
    if constexpr (qc.value & 1) dk[u] = mfma(tf[qc.value], sb[kk], dk[u]);
    else dv[u] = mfma(tf[qc.value], pb[kk], dv[u]);
  };
  auto move_rows = [&](int b) {
    rat.move(stage_at(b) - r_at);
    r_at = stage_at(b);
  };
  // the address of block b's lse and delta for this half of the lanes
  auto row_at = [&](int b) {
    uint32_t at = lds0 + kRowBytes + (uint32_t)(b & (kStages - 1)) * 512 + 16 * (lane >> 5);
    asm volatile("" : "+v"(at));  // not read before here
    return at;
  };
  auto read_rows = [&](auto j, uint32_t at) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) const f4 lds_f4_t;
    l4[j.value] = __builtin_bit_cast(float4, *(lds_f4_t*)(uintptr_t)(at + 32 * j.value));
    d4[j.value] = __builtin_bit_cast(float4, *(lds_f4_t*)(uintptr_t)(at + 256 + 32 * j.value));
  };
  // Part k % 4 of the P and dS of queries acc_row(2 (k / 4)) and the next (k = 0 .. 31) of block b.
  // masked: P = 0 where the query precedes the key or lies past the sequence, also where its score or
  // log-sum-exp is not finite.
  auto p_sub = [&](auto masked, auto kc, int b, f32x16 (&x)[2]) {
    constexpr int r = 2 * (kc.value >> 2), part = kc.value & 3;
    const float4 lj = l4[r >> 2], dj = d4[r >> 2];
    auto p_of = [&](int i, float lse) {
      const float p = ex2(fmaf(x[0][i], c, -(lse * kLog2e)));
      if constexpr (!masked.value) return p;
      const int first = kj - kw0 - kTok * b - 4 * (lane >> 5);  // the key's own query
      return acc_row(i, 0) >= first && acc_row(i, 0) - first < L - kj ? p : 0.f;
    };
    if constexpr (part == 0) x[0][r] = p_of(r, r & 2 ? lj.z : lj.x);
    if constexpr (part == 1) x[0][r + 1] = p_of(r + 1, r & 2 ? lj.w : lj.y);
    if constexpr (part == 2) {
      x[1][r] = x[0][r] * (x[1][r] - (r & 2 ? dj.z : dj.x));
      x[1][r + 1] = x[0][r + 1] * (x[1][r + 1] - (r & 2 ? dj.w : dj.y));
    }
    if constexpr (part == 3) {
      set_pair(pb[r >> 3], (r & 7) >> 1, cvt2h(x[0][r], x[0][r + 1]));
      set_pair(sb[r >> 3], (r & 7) >> 1, cvt2h(x[1][r], x[1][r + 1]));
    }
  };
  constexpr int NS = 2 * KC, NV = 4 * DT, half = NV / 2;  // MFMAs of S and dP, of dV and dK
  constexpr int kPer = 32 / (NS + NV);                    // parts of P and dS per MFMA
  constexpr int kHead = half * kPer;  // parts done in the block before (the last in this one's end)
  constexpr int kAhead = 3;           // fragment reads issued ahead of their MFMAs

  // Block b, its S and dP in x and the first kHead parts of its P and dS done: the next block's S
  // and dP go to xn. last: there is none; masked: one of the two may need masks.
  auto block = [&](auto last, auto masked, int b, f32x16 (&x)[2], f32x16 (&xn)[2]) {
    constexpr bool kLast = last.value;
    sync_tile<NL>();  // block b + 1 landed, every wavefront is done with b - 1
    if (!kLast) move_rows(b + 1);
    tat.move(stage_at(b) - t_at);
    t_at = stage_at(b);
    const uint32_t at = row_at(b), atn = row_at(b + 1);
    static_for<3>([&](auto j) { read_rows(std::integral_constant<int, j.value + 1>{}, at); });
    if constexpr (!kLast) {
      static_for<kAhead>([&](auto i) { read_r(i); });
      __builtin_amdgcn_sched_barrier(0);
      static_for<NS>([&](auto qc) {
        constexpr int q = qc.value;
        s_mfma(qc, xn);
        if constexpr (q + kAhead < NS) read_r(std::integral_constant<int, q + kAhead>{});
        else read_t(std::integral_constant<int, q + kAhead - NS>{});
        static_for<kPer>([&](auto i) {
          p_sub(masked, std::integral_constant<int, kHead + q * kPer + i.value>{}, b, x);
        });
        if constexpr (q % 3 == 1 && q / 3 < NL) load(std::integral_constant<int, q / 3>{}, b + 3);
        __builtin_amdgcn_sched_barrier(0);
      });
    } else {
      static_for<kAhead>([&](auto i) { read_t(i); });
      static_for<NS * kPer>([&](auto i) {
        p_sub(masked, std::integral_constant<int, kHead + i.value>{}, b, x);
      });
      __builtin_amdgcn_sched_barrier(0);
    }
    static_for<NV>([&](auto qc) {
      constexpr int q = qc.value;
      g_mfma(qc);
      if constexpr (q + kAhead < NV) read_t(std::integral_constant<int, q + kAhead>{});
      if constexpr (q < half) {
        static_for<kPer>([&](auto i) {
          p_sub(masked, std::integral_constant<int, kHead + NS * kPer + q * kPer + i.value>{}, b, x);
        });
        if constexpr (!kLast && q == half - 1) read_rows(std::integral_constant<int, 0>{}, atn);
      } else if constexpr (!kLast) {
        static_for<kPer>([&](auto i) {
          p_sub(masked, std::integral_constant<int, (q - half) * kPer + i.value>{}, b + 1, xn);
        });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  static_assert(3 * (NL - 1) + 1 < NS, "a block's loads are issued behind S and dP");
  static_assert(kHead <= 8, "the parts done ahead need the first four queries' lse only");
  static_assert(kPer * (NS + NV) == 32, "every part of P and dS has its place");

  first_block<NL>(nb);
  // blocks wholly before the wavefront's keys: loaded for the others (their P would be 0, but 0
  // times a value that is not finite is NaN: it may not reach later keys)
  int b = 0;
  for (; b < min(wave, nb); ++b) {
    sync_tile<NL>();
    static_for<NL>([&](auto j) { load(j, b + 3); });
  }
  if (b < nb) {
    const std::false_type no;
    const std::true_type yes;
    move_rows(b);
    static_for<NS>([&](auto i) { read_r(i); });
    static_for<NS>([&](auto q) { s_mfma(q, s); });
    read_rows(std::integral_constant<int, 0>{}, row_at(b));
    static_for<kHead>([&](auto i) { p_sub(yes, i, b, s); });
    // the diagonal's block, the blocks without masks in pairs (no product changes its registers),
    // those that are left over and the last
    if (b + 1 < nb) {
      block(no, yes, b, s, sn);
      s[0] = sn[0];
      s[1] = sn[1];
      ++b;
    }
    for (; b + 3 < nb; b += 2) {
      block(no, no, b, s, sn);
      block(no, no, b + 1, sn, s);
    }
    for (; b + 1 < nb; ++b) {
      block(no, yes, b, s, sn);
      s[0] = sn[0];
      s[1] = sn[1];
    }
    block(yes, yes, b, s, sn);
  }
  __builtin_amdgcn_s_waitcnt(0);  // loads past the sequence: none in flight when the wavefront ends
  if (kj < L) {
    const int64_t off = (int64_t)(start + kj) * qs + h * D;
    store_token_row<D>(a.dk + off, dk, a.scale, lane);
    store_token_row<D>(a.dv + off, dv, 1.0f, lane);
  }
}

}  // namespace attn
}  // namespace qlora

using namespace qlora::attn;

namespace {

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

int check_common(int32_t nseq, int32_t max_len, int64_t n, int32_t HQ, int32_t KH, int32_t D) {
  QLORA_CHECK_ARG(nseq >= 0 && max_len >= 0 && n >= 0);
  QLORA_CHECK_ARG(D == 64 || D == 128);
  QLORA_CHECK_ARG(HQ > 0 && KH > 0 && HQ % KH == 0);
  const int G = HQ / KH;
  QLORA_CHECK_ARG(G >= 1 && G <= 8);  // every Qwen2 size: 14/2, 12/2, 16/2, 28/4, 40/8, 64/8
  QLORA_CHECK_ARG((int64_t)nseq * HQ < (1ll << 31));
  // buffer offsets within one sequence's rows (plus the prefetch past its end) fit 32 bits
  QLORA_CHECK_ARG(((int64_t)max_len + 4 * kKB) * HQ * D * 2 < (1ll << 31));
  return 0;
}

// Chunks of the split forms: chunk_keys a positive multiple of 64, at most kMaxChunks chunks.
constexpr int kMaxChunks = 16;
int split_chunks(int32_t max_len, int32_t chunk_keys, int64_t* nch) {
  QLORA_CHECK_ARG(chunk_keys >= kKB && chunk_keys % kKB == 0);
  *nch = qlora_cdiv(max_len, chunk_keys);
  QLORA_CHECK_ARG(*nch >= 1 && *nch <= kMaxChunks);
  return 0;
}

// Workgroups of one launch: tiles x (sequence, head) pairs, within the 32-bit grid.
int grid_of(int64_t tiles, int64_t pairs, unsigned* x) {
  QLORA_CHECK_ARG(tiles * pairs < (1ll << 31));
  *x = (unsigned)(tiles * pairs);
  return 0;
}

// The merge kernel for nch chunks (C: the next supported count at or above it).
template <bool FWD>
int launch_merge(const Args& a, int D, int64_t nseq, int64_t nch, hipStream_t s) {
  unsigned gx;
  if (int rc = grid_of(a.ntiles, nseq * a.HQ, &gx)) return rc;
#define QLORA_MERGE(DD, CC) \
  hipLaunchKernelGGL((attn_merge_kernel<DD, CC, FWD>), dim3(gx), dim3(32 * DD / 4), 0, s, a)
  if (D == 128) {
    if (nch <= 2) QLORA_MERGE(128, 2);
    else if (nch <= 4) QLORA_MERGE(128, 4);
    else if (nch <= 8) QLORA_MERGE(128, 8);
    else QLORA_MERGE(128, 16);
  } else {
    if (nch <= 2) QLORA_MERGE(64, 2);
    else if (nch <= 4) QLORA_MERGE(64, 4);
    else if (nch <= 8) QLORA_MERGE(64, 8);
    else QLORA_MERGE(64, 16);
  }
#undef QLORA_MERGE
  return qlora_launch_status();
}

template <int D, int NW>
int launch_fwd(Args a, int32_t nseq, int64_t tiles, int64_t nch, hipStream_t s) {
  a.ntiles = (int)qlora_cdiv(tiles * (a.HQ / a.KH), NW);
  unsigned gx;
  if (int rc = grid_of(a.ntiles, (int64_t)nseq * a.KH, &gx)) return rc;
  hipLaunchKernelGGL((attn_fwd_kernel<D, NW>), dim3(gx, 1, (unsigned)nch), dim3(64 * NW), 0, s, a);
  return qlora_launch_status();
}

// Whether the forward takes workgroups of eight wavefronts: from 3,072 (query tile, head) pairs on,
// 1.5 of such workgroups a CU. Four against eight, MI355X, head counts 8/8 to 64/8, us: below, four
// are faster by 0-20 % (12/2 heads of 128, six sequences of 1,024, 2,304 pairs: 32 against 35; 8/8,
// 8,192 tokens, 2,048: 166 against 194); above, within 5 % either way for most (12/2, two of 4,096:
// 121.5 against 122.7; 14/2 heads of 64, 4,096 + 3,001, 3,108: 76 against 70; 32/32, 4,096, 4,096:
// 163 against 148; 64/8 heads of 64, 4,096, 8,192: 171 against 176). Also where four would need more
// workgroups than a grid holds.
bool wide_groups(const Args& a, int32_t nseq, int64_t tiles) {
  return qlora_cdiv(a.n, kTok) * a.HQ >= 3072 ||
         qlora_cdiv(tiles * (a.HQ / a.KH), 4) * nseq * a.KH >= (1ll << 31);
}

int run_fwd(Args a, int32_t nseq, int32_t max_len, int D, int64_t nch, hipStream_t s) {
  const int64_t tiles = qlora_cdiv(max_len, kTok);
  const bool wide = wide_groups(a, nseq, tiles);
  int rc;
  if (D == 128)
    rc = wide ? launch_fwd<128, 8>(a, nseq, tiles, nch, s)
              : launch_fwd<128, 4>(a, nseq, tiles, nch, s);
  else
    rc = wide ? launch_fwd<64, 8>(a, nseq, tiles, nch, s)
              : launch_fwd<64, 4>(a, nseq, tiles, nch, s);
  a.ntiles = (int)tiles;
  if (rc == 0 && nch > 1) rc = launch_merge<true>(a, D, nseq, nch, s);
  return rc;
}

// The second stream of each device on which the dK/dV kernel runs while the dQ kernel runs on
// the caller's stream (both only read what the delta kernel and the forward wrote): neither
// launch alone fills the GPU when the batch holds few sequences. Fork and join are event
// waits, so the caller's stream orders everything after the backward as before. Created on
// first use (default priority), kept for the process.
struct SideStream {
  hipStream_t stream = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
};
std::mutex g_side_mu;
SideStream g_side[64];

int side_stream(SideStream** out) {
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev)) return (int)e;
  if (dev < 0 || dev >= 64) return (int)hipErrorInvalidDevice;
  SideStream& ss = g_side[dev];
  if (ss.stream == nullptr) {
    if (hipError_t e = hipStreamCreateWithFlags(&ss.stream, hipStreamNonBlocking)) return (int)e;
    if (hipError_t e = hipEventCreateWithFlags(&ss.fork, hipEventDisableTiming)) return (int)e;
    if (hipError_t e = hipEventCreateWithFlags(&ss.join, hipEventDisableTiming)) return (int)e;
  }
  *out = &ss;
  return 0;
}

// dQ and dK/dV side by side pay when one of them leaves room for the other (at most 300 dK/dV
// workgroups, one a CU at D = 128) and both are long enough for the delta kernel, the fork and the
// join. Side by side against in turn on MI355X, us a call: 12/2 heads of 128, 1,024 tokens (96
// workgroups) 59 against 61, 512 (48) 48 against 41, 2,048 (192) 87 against 106, 3,072 (288) 141
// against 160, four of 283-997 (384) 70 against 66, two of 2,048 (384) 139 against 125, 28/4, 1,536
// (336) 104 against 95; 8/8 heads of 64, 2,048 (128) 71 against 74, 3,072 (192) 94 against 104, 14/2,
// 2,048 (224) 77 against 75, 1,024 (112) 52 against 43. A cut dQ (nch chunks) runs in turn: it fills
// the GPU itself.
bool bwd_concurrent(int32_t max_len, int D, int64_t nch, unsigned dkdv_groups) {
  return nch == 1 && max_len >= (D == 128 ? 1024 : 2560) && dkdv_groups <= 300;
}

// The dQ kernel, OWN: forming delta itself.
template <bool OWN>
int launch_dq(Args a, int D, int32_t nseq, int64_t tiles, int64_t nch, hipStream_t s) {
  constexpr int NW = 4;
  a.ntiles = (int)qlora_cdiv(tiles * (a.HQ / a.KH), NW);
  unsigned gx;
  if (int rc = grid_of(a.ntiles, (int64_t)nseq * a.KH, &gx)) return rc;
  const dim3 grid(gx, 1, (unsigned)nch), block(64 * NW);
  if (D == 128) hipLaunchKernelGGL((attn_dq_kernel<128, NW, OWN>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((attn_dq_kernel<64, NW, OWN>), grid, block, 0, s, a);
  return qlora_launch_status();
}

void launch_dkdv(const Args& b, int D, unsigned gkv, hipStream_t s) {
  if (D == 128)
    hipLaunchKernelGGL(attn_dkdv_kernel<128>, dim3(gkv), dim3(64 * kKeyWaves), 0, s, b);
  else
    hipLaunchKernelGGL(attn_dkdv_kernel<64>, dim3(gkv), dim3(64 * kKeyWaves), 0, s, b);
}

int run_bwd(Args a, int32_t nseq, int32_t max_len, int D, int64_t nch, hipStream_t s) {
  Args b = a;  // dK/dV
  b.ntiles = (int)qlora_cdiv(max_len, kTok * kKeyWaves);
  unsigned gkv;
  if (int rc = grid_of(b.ntiles, (int64_t)nseq * a.HQ, &gkv)) return rc;
  a.ntiles = (int)qlora_cdiv(max_len, kTok);  // of dQ and the merge
  if (!bwd_concurrent(max_len, D, nch, gkv)) {  // dQ (writing delta), then dK/dV
    if (int rc = launch_dq<true>(a, D, nseq, a.ntiles, nch, s)) return rc;
    if (nch > 1) {
      if (int rc = launch_merge<false>(a, D, nseq, nch, s)) return rc;
    }
    launch_dkdv(b, D, gkv, s);
    return qlora_launch_status();
  }
  const int64_t rows = a.n * a.HQ;
  QLORA_CHECK_ARG(qlora_cdiv(2 * rows, 256) < (1ll << 31));
  const dim3 dgrid((unsigned)qlora_cdiv(2 * rows, 256));
  if (D == 128)
    hipLaunchKernelGGL(attn_delta_kernel<128>, dgrid, dim3(256), 0, s, a.dout, a.o, a.delta,
                       a.n, a.HQ);
  else
    hipLaunchKernelGGL(attn_delta_kernel<64>, dgrid, dim3(256), 0, s, a.dout, a.o, a.delta, a.n,
                       a.HQ);
  if (int rc = qlora_launch_status()) return rc;

  std::lock_guard<std::mutex> lock(g_side_mu);
  SideStream* ss;
  if (int rc = side_stream(&ss)) return rc;
  if (hipError_t e = hipEventRecord(ss->fork, s)) return (int)e;
  if (hipError_t e = hipStreamWaitEvent(ss->stream, ss->fork, 0)) return (int)e;
  launch_dkdv(b, D, gkv, ss->stream);
  int rc = qlora_launch_status();
  if (rc == 0) rc = launch_dq<false>(a, D, nseq, a.ntiles, nch, s);
  if (rc == 0 && nch > 1) rc = launch_merge<false>(a, D, nseq, nch, s);
  // join whatever was launched, also after an error
  if (hipError_t e = hipEventRecord(ss->join, ss->stream)) return rc ? rc : (int)e;
  if (hipError_t e = hipStreamWaitEvent(s, ss->join, 0)) return rc ? rc : (int)e;
  return rc;
}

Args make_args(const void* q, const void* k, const void* v, int64_t n, int32_t HQ, int32_t KH,
               float scale, const int32_t* cu) {
  Args a{};
  a.q = static_cast<const uint16_t*>(q);
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint16_t*>(v);
  a.cu = cu;
  a.n = n;
  a.HQ = HQ;
  a.KH = KH;
  a.scale = scale;
  return a;
}

// The split's chunk count and fp32 workspace for these sizes (none when max_len fits one chunk).
int split_sizes(int32_t max_len, int64_t n, int32_t HQ, int32_t D, int32_t chunk_keys,
                int64_t* nch, int64_t* work) {
  if (int rc = split_chunks(max_len, chunk_keys, nch)) return rc;
  *work = *nch == 1 ? 0 : *nch * n * HQ * (int64_t)(D + 2);
  return 0;
}

}  // namespace

// fp32 workspace elements of qlora_attn_fwd_split / qlora_attn_bwd_split for these sizes and
// chunk_keys (keys per workgroup: a positive multiple of 64 with ceil(max_len / chunk_keys)
// <= 16); 0 when max_len fits one chunk. No reference counterpart: a work split of the same
// attention.
QLORA_API int qlora_attn_split_workspace(int32_t max_len, int64_t n, int32_t HQ, int32_t D,
                                         int32_t chunk_keys, int64_t* work_elems) {
  QLORA_CHECK_ARG(work_elems && max_len >= 0 && n >= 0 && HQ > 0 && (D == 64 || D == 128));
  *work_elems = 0;
  if (max_len == 0 || n == 0) return 0;
  int64_t nch;
  return split_sizes(max_len, n, HQ, D, chunk_keys, &nch, work_elems);
}

// qlora_attn_fwd with each query tile's key range cut into chunks of chunk_keys keys (0: not
// cut), one workgroup each, and a second kernel that merges the fp32 partials in chunk order.
// work: fp32, 16-byte aligned, of qlora_attn_split_workspace elements. Same reference call site
// as qlora_attn_fwd (engine.py:857-862).
QLORA_API int qlora_attn_fwd_split(const void* q, const void* k, const void* v, void* out,
                                   float* lse, const int32_t* cu_seqlens, int32_t nseq,
                                   int32_t max_len, int64_t n, int32_t HQ, int32_t KH, int32_t D,
                                   float scale, int32_t chunk_keys, float* work,
                                   int64_t work_elems, void* stream) {
  if (int rc = check_common(nseq, max_len, n, HQ, KH, D)) return rc;
  if (n == 0 || nseq == 0 || max_len == 0) return 0;
  int64_t nch = 1, need = 0;
  if (chunk_keys != 0) {
    if (int rc = split_sizes(max_len, n, HQ, D, chunk_keys, &nch, &need)) return rc;
  }
  QLORA_CHECK_ARG(q && k && v && out && lse && cu_seqlens);
  QLORA_CHECK_ARG(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out));
  QLORA_CHECK_ARG(work_elems >= need && (nch == 1 || (work && aligned16(work))));
  Args a = make_args(q, k, v, n, HQ, KH, scale, cu_seqlens);
  a.out = static_cast<uint16_t*>(out);
  a.lse = lse;
  if (nch > 1) {
    a.chunk = chunk_keys / kKB;
    a.part = work;
    a.part_ml = reinterpret_cast<float2*>(work + nch * n * HQ * D);
  }
  return run_fwd(a, nseq, max_len, D, nch, (hipStream_t)stream);
}

// Forward. q [n, HQ, D], k/v [n, KH, D], out [n, HQ, D] fp16 contiguous; lse fp32 [HQ, n];
// cu_seqlens int32 [nseq + 1] on the device, non-decreasing from 0 to n, every length
// <= max_len (the kernel reads no token outside [cu[s], cu[s + 1]) for sequence s).
QLORA_API int qlora_attn_fwd(const void* q, const void* k, const void* v, void* out, float* lse,
                             const int32_t* cu_seqlens, int32_t nseq, int32_t max_len, int64_t n,
                             int32_t HQ, int32_t KH, int32_t D, float scale, void* stream) {
  return qlora_attn_fwd_split(q, k, v, out, lse, cu_seqlens, nseq, max_len, n, HQ, KH, D, scale,
                              0, nullptr, 0, stream);
}

// qlora_attn_bwd with the dQ kernel's key range cut into chunks of chunk_keys keys (0: not cut),
// one workgroup each, summed in chunk order by a second kernel; dK/dV as in qlora_attn_bwd. work
// as for qlora_attn_fwd_split. Same reference call site (engine.py:865-869).
QLORA_API int qlora_attn_bwd_split(const void* dout, const void* q, const void* k, const void* v,
                                   const void* out, const float* lse, float* delta, void* dq,
                                   void* dk, void* dv, const int32_t* cu_seqlens, int32_t nseq,
                                   int32_t max_len, int64_t n, int32_t HQ, int32_t KH, int32_t D,
                                   float scale, int32_t chunk_keys, float* work,
                                   int64_t work_elems, void* stream) {
  if (int rc = check_common(nseq, max_len, n, HQ, KH, D)) return rc;
  if (n == 0 || nseq == 0 || max_len == 0) return 0;
  int64_t nch = 1, need = 0;
  if (chunk_keys != 0) {
    if (int rc = split_sizes(max_len, n, HQ, D, chunk_keys, &nch, &need)) return rc;
  }
  QLORA_CHECK_ARG(dout && q && k && v && out && lse && delta && dq && dk && dv && cu_seqlens);
  QLORA_CHECK_ARG(aligned16(dout) && aligned16(q) && aligned16(k) && aligned16(v) &&
                  aligned16(out) && aligned16(dq) && aligned16(dk) && aligned16(dv));
  QLORA_CHECK_ARG(work_elems >= need && (nch == 1 || (work && aligned16(work))));
  Args a = make_args(q, k, v, n, HQ, KH, scale, cu_seqlens);
  a.o = static_cast<const uint16_t*>(out);
  a.dout = static_cast<const uint16_t*>(dout);
  a.out = static_cast<uint16_t*>(dq);
  a.dk = static_cast<uint16_t*>(dk);
  a.dv = static_cast<uint16_t*>(dv);
  a.lse = const_cast<float*>(lse);
  a.delta = delta;
  if (nch > 1) {
    a.chunk = chunk_keys / kTok;
    a.part = work;
  }
  return run_bwd(a, nseq, max_len, D, nch, (hipStream_t)stream);
}

// Backward. dout/out/q [n, HQ, D], k/v [n, KH, D] as in the forward, lse from it; delta: fp32
// workspace [HQ, n]; dq, dk, dv fp16 [n, HQ, D] (dk/dv per q head, not yet summed over the
// q heads of a kv head).
QLORA_API int qlora_attn_bwd(const void* dout, const void* q, const void* k, const void* v,
                             const void* out, const float* lse, float* delta, void* dq, void* dk,
                             void* dv, const int32_t* cu_seqlens, int32_t nseq, int32_t max_len,
                             int64_t n, int32_t HQ, int32_t KH, int32_t D, float scale,
                             void* stream) {
  return qlora_attn_bwd_split(dout, q, k, v, out, lse, delta, dq, dk, dv, cu_seqlens, nseq,
                              max_len, n, HQ, KH, D, scale, 0, nullptr, 0, stream);
}
