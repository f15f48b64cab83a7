// Matrix-core forward passes on one MI355X (gfx950) over M token rows at once:
//   * prefill  — the M tokens of one prompt at positions 0..M-1 (model.py:194-231,
//                prefill_with_kv, as called by generate.py:70-90)
//   * batched decode — one token of each of M independent sequences, each at its own
//                position, over a paged KV cache (the reference's described batched paged
//                decode; kernels/multi_sm_decode.py:77-357 semantics per sequence)
// writing the KV cache rows of every layer and the logits, with every projection on the
// matrix cores.
//
// Numerics: model.py:94-191 in f32.  Each activation entering a projection (RMSNorm outputs,
// attention output, SwiGLU output, final norm) is stored as two bf16 parts, hi = bf16(x) and
// lo = bf16(x - hi), and both are multiplied with the bf16 weights on the matrix cores
// (v_mfma_f32_16x16x32_bf16) into one f32 accumulator: the projection sees x to about 2^-17
// relative, where the reference kernel rounds it to bf16 (multi_sm_decode.py:143,229,268,289,
// 320).  The residual stream, RoPE, softmax attention and SwiGLU are f32, K/V are stored to the
// cache as bf16 after RoPE (model.py:212-215).  In batched decode the current position attends
// with its un-rounded K/V (multi_sm_decode.py:197,205).
//
// KV cache: [layer][K, V][kv_head][pool positions][64] bf16 with pool positions = 16 * pages.
// A row's position p lives at page table[p / 16] * 16 + p % 16; without a table the page is
// p / 16 (the contiguous cache of one sequence is the pool with the identity table).
//
// With the tile copy of the weights (msd_pack_tiles) a layer is five kernels on the caller's stream: mx_gemm_rows
// for QKV, O, gate/up and down, with the norms, RoPE, SwiGLU and the residual in its epilogues, and the
// attention (run_layers).  Without it:
//   mx_norm        residual += split-K partials of the previous projection (in split order),
//                  then RMSNorm -> bf16 activations in the weights' permuted input order
//   mx_gemm        q/k/v projection, split-K partials
//   mx_qkv_fin     sum of the partials, RoPE on q/k, f32 q/k/v (a prefill: K and V as operand planes),
//                  bf16 K/V cache rows
//   attention      prefill: causal GQA over the prompt; batched decode: each sequence over
//                  its cached rows plus its current K/V
//   mx_gemm        O projection, split-K partials
//   mx_norm        (as above) -> ln2 activations
//   mx_gemm        gate/up projection, split-K partials
//   mx_swiglu_fin  silu(gate) * up -> bf16 in the down projection's input order
//   mx_gemm        down projection, split-K partials
// Either way then mx_norm with the final scale, the tied logits (mx_gemm for one row, mx_logits for more) and
// mx_argmax per row.
//
// mx_gemm: C[M x N] = A[M x K] * W[N x K]^T with A (activations) and W (packed weight rows)
// both K-contiguous.  A workgroup of four waves covers 64 columns and BM rows; each wave
// holds RB x CB 16 x 16 MFMA tiles, every operand fragment one 16-byte run along K loaded
// straight from memory (W streamed once per row tile, A from L2).  K is split across grid.z
// into enough workgroups to keep every compute unit streaming; partials are summed in split
// order by the consuming kernel.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <vector>

#include "../../include/msdecode.h"
#include "arith.h"
#include "batched.h"
#include "internal.h"

namespace mpf {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kDh = 64;
constexpr int kPage = 16;     // positions per KV page
constexpr int kBN = 64;       // GEMM tile columns
constexpr int kBK = 32;       // K per MFMA step
constexpr int kNormThreads = 256;
constexpr int kMaxSplitK = 16;  // largest K split (partials summed by the consumers)
constexpr int kMaxRows = 1024;

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float(uint32_t(b) << 16); }
__device__ __forceinline__ uint16_t f2bf(float f) {   // round to nearest even
  const uint32_t u = __float_as_uint(f);
  return uint16_t((u + (((u >> 16) & 1u) + 0x7fffu)) >> 16);
}

// An activation entering a projection as two bf16 parts, hi = bf16(x) and lo = bf16(x - hi): the
// matrix cores multiply both with the bf16 weight and add in f32, so the product carries x to
// about 2^-17 relative instead of bf16's 2^-9 (the f32 activations of model.py, not the
// reference kernel's bf16 rounding points).  The lo part lives in a second plane of the buffer.
__device__ __forceinline__ void put_split(uint16_t* hi, int64_t plane, float x) {
  const uint16_t h = f2bf(x);
  hi[0] = h;
  hi[plane] = f2bf(x - bf2f(h));
}

// Wave64 reductions with DPP row shifts and row broadcasts (fixed order, no LDS traffic);
// the result is read from lane 63 as a wave-uniform value.
template <int CTRL, int ROWMASK>
__device__ __forceinline__ float dpp(float v, float fill) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(fill), __float_as_int(v), CTRL, ROWMASK, 0xf, false));
}
// The sum over each row of 16 lanes, in every lane of the row: the butterfly lane ^ 1, ^ 2, ^ 4,
// ^ 8 with DPP (quad permutes, then the half-row and row mirrors: after each step the lanes of a
// group hold the same value, so a mirror adds the other group's sum exactly as the xor would)
// instead of LDS permutes
__device__ __forceinline__ float sum16_lanes(float v) {
  v += dpp<0xB1, 0xf>(v, 0.f);    // quad_perm [1, 0, 3, 2]: lane ^ 1
  v += dpp<0x4E, 0xf>(v, 0.f);    // quad_perm [2, 3, 0, 1]: lane ^ 2
  v += dpp<0x141, 0xf>(v, 0.f);   // row_half_mirror: the other quad of the 8
  v += dpp<0x140, 0xf>(v, 0.f);   // row_mirror: the other 8 of the row
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp<0x111, 0xf>(v, 0.f);
  v += dpp<0x112, 0xf>(v, 0.f);
  v += dpp<0x114, 0xf>(v, 0.f);
  v += dpp<0x118, 0xf>(v, 0.f);
  v += dpp<0x142, 0xa>(v, 0.f);
  v += dpp<0x143, 0xc>(v, 0.f);
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp<0x111, 0xf>(v, -INFINITY));
  v = fmaxf(v, dpp<0x112, 0xf>(v, -INFINITY));
  v = fmaxf(v, dpp<0x114, 0xf>(v, -INFINITY));
  v = fmaxf(v, dpp<0x118, 0xf>(v, -INFINITY));
  v = fmaxf(v, dpp<0x142, 0xa>(v, -INFINITY));
  v = fmaxf(v, dpp<0x143, 0xc>(v, -INFINITY));
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// Position of input element i in a row of K under the packed row layout: blocks of 512
// (the last one S = 8m long); element b*512 + k*m + l sits at b*512 + 8*l + k.
__device__ __forceinline__ int perm_pos(int i, int K) {
  const int b = i >> 9, r = i & 511;
  const int S = min(512, K - (b << 9));
  const int m = S >> 3;
  const int k = r / m, l = r - k * m;
  return (b << 9) + 8 * l + k;
}
// Input element stored at position j (inverse of perm_pos).
__device__ __forceinline__ int perm_elem(int j, int K) {
  const int b = j >> 9, o = j & 511;
  const int S = min(512, K - (b << 9));
  const int m = S >> 3;
  return (b << 9) + (o & 7) * m + (o >> 3);
}

// Element (m, j) of an activation plane with rows of K (j a packed position).  ldx > 0: rows
// ldx apart.  ldx == 0: matrix-core tile order, the layout the projections read: 16 rows x 32
// positions form a tile of 64 lanes x 16 bytes in MFMA operand order (row m % 16 and positions
// 8 ((j % 32) / 8) .. + 8 in lane (m % 16) + 16 ((j % 32) / 8)), tile (m / 16, j / 32) at
// ((m / 16) (K / 32) + j / 32) 512 elements, so a wave's operand load reads 1 KB in one piece.
__device__ __forceinline__ int64_t act_index(int m, int j, int K, int ldx) {
  if (ldx > 0) return int64_t(m) * ldx + j;
  return ((int64_t(m >> 4) * (K >> 5) + (j >> 5)) * 64 + (m & 15) + 16 * ((j & 31) >> 3)) * 8 + (j & 7);
}

// Rows of a pass: row m is sequence seq(m) at position pos(m).
struct Rows {
  int M;
  const int32_t* pos;     // NULL: pos(m) = pos0 + m (prefill from pos0)
  int batched;            // seq(m) = m; else every row is sequence 0
  const int32_t* pages;   // [seq][max_pages] page table, NULL = identity
  int max_pages;
  int pool;               // pool positions (16 * pages)
  int pos0;               // position of row 0 when pos is NULL
};
__device__ __forceinline__ int row_pos(const Rows& r, int m) { return r.pos ? r.pos[m] : r.pos0 + m; }
__device__ __forceinline__ int64_t cache_row(const Rows& r, int m, int p) {
  const int seq = r.batched ? m : 0;
  const int page = r.pages ? r.pages[int64_t(seq) * r.max_pages + p / kPage] : p / kPage;
  return int64_t(page) * kPage + p % kPage;
}

// What mx_gemm_rows does with its final outputs.
enum Epi { kEpiStore = 0, kEpiSwiglu = 1, kEpiQkv = 2, kEpiResid = 3 };
// Operands of the fused epilogues.
struct EpiArgs {
  uint16_t* act;       // SwiGLU: the down projection's input planes; Resid: the next RMSNorm's (or NULL)
  int64_t act_plane;   // input planes (scale * h); tile order, the lo plane act_plane further
  const uint16_t* xscale;   // Resid: the next RMSNorm's scales in packed order
  float* ssq;               // Resid: each row's partial sum of h^2 per column group, [M][N / (16 CT)]
  const float* rope;   // QKV: RoPE table, rows, cache and the f32 q/k/v rows (as mx_qkv_fin)
  Rows rows;
  uint16_t* kc;
  uint16_t* vc;
  float* qkv;
  int H, KV;
  uint16_t* kvp;   // QKV of a prefill: the attention's K/V operand planes (below), else NULL
  int MP;
};

// A prefill's K and V for its own attention, as bf16 hi/lo planes [K hi | K lo | V hi | V lo] of KV * MP *
// 64 values (MP: rows padded to 32), each K/V head in the tile order of the matrix-core operand
// that reads it: K as rows of 64 dims (16 keys x 32 dims per tile), V as the transpose (16 dims x 32
// keys per tile).
__device__ __forceinline__ int64_t k_plane_index(int g, int key, int dim, int MP) {
  return int64_t(g) * MP * kDh + act_index(key, dim, kDh, 0);
}
__device__ __forceinline__ int64_t v_plane_index(int g, int key, int dim, int MP) {
  return int64_t(g) * MP * kDh + act_index(dim, key, MP, 0);
}

struct GemmArgs {
  const uint16_t* A;   // [M][lda] bf16 (or tile order, see act_index): the hi parts; the lo
  int64_t a_plane;     // parts follow at A + a_plane
  const uint16_t* W;   // [N][K] bf16 (or tile order: tile (n / 16, k / 32) at ((n / 16) (K / 32) + k / 32) 512)
  float* out;          // partials [splits][M][N] f32, or [M][ldo] (single split)
  int M, N, K, lda, ldo, splits;
  EpiArgs e;
  const float* ssq;   // mx_gemm_rows with the norm folded in (AM 2): each row's partial sums of h^2,
  int nssq;           // [M][nssq], summed in a fixed order for the rms that divides the outputs
};

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 u) { return __builtin_bit_cast(bf16x8, u); }

// Two f32 values as hi/lo parts, packed (a in the low halves; v_cvt_pk_bf16_f32 rounds to nearest even).
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
}
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  hi = pack2(a, b);
  lo = pack2(a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xffff0000u));
}

// Eight f32 values as hi/lo bf16 parts (hi = bf16(x), lo = bf16(x - hi)), packed as MFMA operands.
__device__ __forceinline__ void split8(const float (&x)[8], uint4& hi, uint4& lo) {
  split2(x[0], x[1], hi.x, lo.x);
  split2(x[2], x[3], hi.y, lo.y);
  split2(x[4], x[5], hi.z, lo.z);
  split2(x[6], x[7], hi.w, lo.w);
}

// f32 operands as hi/lo parts on the matrix cores: a b ~ ah bh + ah bl + al bh (the lo lo term,
// ~2^-16 of the product, is left out).
__device__ __forceinline__ f32x4 mfma3(uint4 ah, uint4 al, uint4 bh, uint4 bl, f32x4 c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(ah), as_bf16x8(bh), c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(ah), as_bf16x8(bl), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(al), as_bf16x8(bh), c, 0, 0, 0);
}


// Four waves as WM x (4 / WM); a wave covers RB 16-row blocks and (WM) 16-column blocks.  TA:
// the activations in tile order (one 1 KB piece per operand load); the weights are in row order.
template <int RB, int WM, bool TA>
__global__ __launch_bounds__(256) void mx_gemm(GemmArgs g) {
  constexpr int WN = 4 / WM, CB = 4 / WN, BM = 16 * RB * WM;
  constexpr int U = RB * CB <= 2 ? 8 : 4;   // K steps with loads in flight
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int wm = wv / WN, wn = wv % WN;
  const int m0 = blockIdx.y * BM + 16 * RB * wm, n0 = blockIdx.x * kBN + 16 * CB * wn;
  const int nchunks = g.K / kBK;
  const int c0 = (nchunks * int(blockIdx.z)) / g.splits, c1 = (nchunks * (int(blockIdx.z) + 1)) / g.splits;
  const int kq = 8 * (lane >> 4);   // this lane's 8-element K run within a 32 chunk
  const int r16 = lane & 15;
  // operand pointers of chunk 0
  const uint16_t* arow[RB];   // hi parts (the lo parts a_plane elements further)
  bool aval[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int m = m0 + 16 * rb + r16;
    aval[rb] = m < g.M;
    if constexpr (TA)   // tiles past the last one read the last (those rows are zeroed)
      arow[rb] = g.A + (int64_t(min(m0 + 16 * rb, g.M - 1) >> 4) * nchunks * 64 + lane) * 8;
    else
      arow[rb] = g.A + int64_t(aval[rb] ? m : 0) * g.lda + kq;
  }
  const uint16_t* wrow[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
    wrow[cb] = g.W + int64_t(n0 + 16 * cb + r16) * g.K + kq;
  f32x4 acc[RB][CB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](const uint4* a, const uint4* al, const uint4* w) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        acc[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[rb]), as_bf16x8(w[cb]), acc[rb][cb], 0, 0, 0);
        acc[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(al[rb]), as_bf16x8(w[cb]), acc[rb][cb], 0, 0, 0);
      }
  };
  // U chunks per round, all loads issued before the first MMA; the last round's chunks past c1
  // reload chunk c1 - 1 and are skipped (loads stay unconditional: a load under a branch is
  // waited for at the join)
  for (int c = c0; c < c1; c += U) {
    uint4 a[U][RB], al[U][RB], w[U][CB];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int ch = min(c + u, c1 - 1);
      const int64_t ka = int64_t(ch) * (TA ? 512 : kBK), kw = int64_t(ch) * kBK;
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const uint4 v = *reinterpret_cast<const uint4*>(arow[rb] + ka);
        const uint4 vl = *reinterpret_cast<const uint4*>(arow[rb] + g.a_plane + ka);
        a[u][rb] = aval[rb] ? v : make_uint4(0, 0, 0, 0);
        al[u][rb] = aval[rb] ? vl : make_uint4(0, 0, 0, 0);
      }
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) w[u][cb] = *reinterpret_cast<const uint4*>(wrow[cb] + kw);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c + u < c1) step(a[u], al[u], w[u]);
  }
  // D layout of a 16 x 16 tile: lane holds rows 4*(lane/16) + r (r < 4) of column lane % 16
  float* out = g.splits > 1 ? g.out + int64_t(blockIdx.z) * g.M * g.N : g.out;
  const int ldo = g.splits > 1 ? g.N : g.ldo;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + 16 * rb + 4 * (lane >> 4) + r;
        if (row < g.M) out[int64_t(row) * ldo + n0 + 16 * cb + r16] = acc[rb][cb][r];
      }
}

using msdc::quotient;
using msdc::swiglu;   // of a gate/up pair: packed rows 2f, 2f + 1

// Four outputs of the packed q/k/v rows col .. col + 3 (col a multiple of 4) of row `row`, whose position
// has the RoPE row rp: q and k pairs are rotated (dims i, i + 32; model.py:110-117), v is stored
// as projected; f32 q/k/v in natural head-dim order to the row's q (with ea.kvp k and v go to the
// operand planes instead, row = key), bf16 K/V to the cache row crow (multi_sm_decode.py:179-180).
__device__ __forceinline__ void qkv_quad(f32x4 v, const float* rp, int col, int row, const EpiArgs& ea, float* q,
                                         int64_t crow) {
  const int H = ea.H, KV = ea.KV, head = col / kDh, rr = col % kDh;
  const int64_t pl = int64_t(KV) * ea.MP * kDh;
  q += head * kDh;
  if (head >= H + KV) {   // v: four consecutive dims
    const int g = head - H - KV;
    if (ea.kvp) {
      uint32_t hi[2], lo[2];
      split2(v[0], v[1], hi[0], lo[0]);
      split2(v[2], v[3], hi[1], lo[1]);
      uint16_t* vp = ea.kvp + 2 * pl;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t at = v_plane_index(g, row, rr + e, ea.MP);
        vp[at] = uint16_t(hi[e >> 1] >> (16 * (e & 1)));
        vp[pl + at] = uint16_t(lo[e >> 1] >> (16 * (e & 1)));
      }
    } else {
      *reinterpret_cast<f32x4*>(q + rr) = v;
    }
    *reinterpret_cast<uint2*>(ea.vc + (int64_t(g) * ea.rows.pool + crow) * kDh + rr) =
        make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
    return;
  }
  const int ri = rr >> 1;   // pairs: dims ri, ri + 32 and ri + 1, ri + 33
  const f32x2 c = *reinterpret_cast<const f32x2*>(rp + ri), s = *reinterpret_cast<const f32x2*>(rp + kDh / 2 + ri);
  const f32x2 x = {v[0] * c[0] - v[1] * s[0], v[2] * c[1] - v[3] * s[1]};
  const f32x2 y = {v[0] * s[0] + v[1] * c[0], v[2] * s[1] + v[3] * c[1]};
  if (head < H || !ea.kvp) {
    *reinterpret_cast<f32x2*>(q + ri) = x;
    *reinterpret_cast<f32x2*>(q + ri + kDh / 2) = y;
  }
  if (head >= H) {
    const int g = head - H;
    if (ea.kvp) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        uint32_t hi, lo;
        split2(half ? y[0] : x[0], half ? y[1] : x[1], hi, lo);
        uint16_t* kp = ea.kvp + k_plane_index(g, row, ri + half * kDh / 2, ea.MP);
        *reinterpret_cast<uint32_t*>(kp) = hi;
        *reinterpret_cast<uint32_t*>(kp + pl) = lo;
      }
    }
    uint16_t* cp = ea.kc + (int64_t(g) * ea.rows.pool + crow) * kDh;
    *reinterpret_cast<uint32_t*>(cp + ri) = pack2(x[0], x[1]);
    *reinterpret_cast<uint32_t*>(cp + ri + kDh / 2) = pack2(y[0], y[1]);
  }
}

typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
template <bool NT>
__device__ __forceinline__ uint4 load_w(const uint16_t* p) {
  const u32x4v* q = reinterpret_cast<const u32x4v*>(p);
  return __builtin_bit_cast(uint4, NT ? __builtin_nontemporal_load(q) : *q);
}

// C = A W^T for many rows: a workgroup owns 16 RT rows x 16 CT columns over the whole of K, so it
// streams 16 CT complete weight rows (contiguous in memory), every weight tile it loads serves
// 16 RT rows, and it writes final outputs (no split-K partials).  The last column group may be
// short (N / 16 need not be a multiple of CT).  Its NW waves each hold the whole output tile and
// take interleaved 32-wide K steps (wave w: steps w, w + NW, ...) with P steps of loads in
// flight; the waves' tiles are added through LDS in wave order, row tile by row tile, so the result
// is deterministic.  Tiles are dealt XCD-aware: each XCD (workgroup b runs on XCD b mod 8) takes a
// contiguous range of the tiles, row tiles innermost, so a column group's weights reach its L2 once.
// AM: the A operand as bf16 hi/lo tiles (1), or (2) RMSNorm folded in (model.py:94-98): A = the hi/lo tiles of scale * h that the previous projection's
// epilogue wrote (kEpiResid), and every output divided by sqrt(mean(h^2) + 1e-5), the sum of
// h^2 of each row added up from that epilogue's per-column-group partials.  TW: the weights in tile
// order (else in row order).
// EPI: store the outputs, add them to the residual out (tile order; with an act plane also the
// hi/lo tiles of scale * h and the row's partial sum of h^2 for the next RMSNorm), or finish them
// in place of mx_swiglu_fin / mx_qkv_fin (the same arithmetic).
// Measured at 306M in the pass (one 16-row tile per workgroup and scalar epilogues before): gate/up of
// 511 rows 31.8 -> 20.6 us, of 128 11.8 -> 10.7, of 5 7.2 -> 5.5; what bounds it is in rows_tile.
// NT: the weights are read non-temporal (layers past kKeepBytes).
template <int RT, int CT, int P, int NW, int AM, bool TW, int EPI, bool NT = false>
__global__ __launch_bounds__(64 * NW) void mx_gemm_rows(GemmArgs g) {
  static_assert(RT == 1 || TW, "several row tiles per workgroup: tile-order weights");
  // the waves' partial tiles of one row tile, a lane's four outputs as one 16-byte piece (written and
  // read across lanes contiguously); two buffers, so one barrier per row tile suffices
  __shared__ f32x4 red[RT > 1 ? 2 : 1][NW][CT][64];
  __shared__ float rms[2][16 * RT];     // AM 2: each row's rms and its reciprocal
  __shared__ float hs[RT][NW][16];      // kEpiResid: each wave's part of the rows' sums of h^2
  // wave-uniform wave index: the step count and its loop stay scalar (a per-lane loop would copy
  // the accumulators out of and back into the AGPRs around every step)
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n16 = g.N / 16, T = (g.M + 15) / 16, TG = (T + RT - 1) / RT, C = (n16 + CT - 1) / CT;
  const int xcd = blockIdx.x & 7, per = gridDim.x >> 3, rest = gridDim.x & 7;
  const int id = xcd * per + min(xcd, rest) + (blockIdx.x >> 3);
  const int t = id % TG, c = id / TG;
  const int m0 = 16 * RT * t, n0 = 16 * CT * c;
  const int ctn = min(CT, n16 - CT * c);   // column tiles of this group (the last group may be short)
  const int r16 = lane & 15, kq = 8 * (lane >> 4);
  const int S = g.K / kBK;
  // rows past M read row M - 1 (a row tile past the last reads the last): an MFMA row only feeds its
  // own output row, which is not stored, and a short tile costs only its rows' cache lines
  const uint16_t* ar[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int tile = min(RT * t + rt, T - 1);
    ar[rt] = g.A + (int64_t(tile) * S * 64 + min(r16, g.M - 1 - 16 * tile) + 16 * (lane >> 4)) * 8;
  }
  const uint16_t* wr = TW ? g.W + (int64_t(n0 >> 4) * S * 64 + lane) * 8 : g.W + int64_t(n0 + r16) * g.K + kq;
  // element offsets of step ks and of column tile ct
  const int64_t astep = 512, wstep = TW ? 512 : kBK;
  const int64_t wtile = TW ? int64_t(S) * 512 : int64_t(16) * g.K;
  const int ns = (S - wv + NW - 1) / NW;   // K steps of this wave (possibly none)
  f32x4 acc[RT][CT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  // A thread's outputs are, per column tile ct = wave, wave + NW, ..., row lane % 16 and columns 16 ct
  // + 4 (lane / 16) .. + 4 (the MFMA's A operand is the weights).  The residual elements it updates
  // are requested before the K loop (one row tile) or before the row tile's barrier, so that the
  // epilogue does not wait a memory round trip for them (rows past M read row M - 1)
  constexpr bool kResid = EPI == kEpiResid;
  constexpr int NI = (CT + NW - 1) / NW;
  const int orow = lane & 15, ocol = 4 * (lane >> 4);
  f32x4 hold[NI];
  auto load_hold = [&](int rt) {
    if constexpr (kResid) {
      const int row = min(m0 + 16 * rt + orow, g.M - 1);
#pragma unroll
      for (int i = 0; i < NI; ++i)
        hold[i] = *reinterpret_cast<const f32x4*>(
            g.out + act_index(row, n0 + 16 * min(wv + NW * i, ctn - 1) + ocol, g.N, 0));
    }
  };
  if constexpr (RT == 1) load_hold(0);
  uint4 a[P][RT], al[P][RT], w[P][CT];
  // step i of this wave, clamped to its last: loads stay unconditional, so no wait lands at a
  // branch join (a column tile past a short group's end reads its last tile; a wave without steps
  // reads the first)
  auto load = [&](int p, int i) {
    const int ks = min(wv + NW * min(i, ns - 1), S - 1);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
      w[p][ct] = load_w<NT>(wr + min(ct, ctn - 1) * wtile + max(ks, 0) * wstep);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      a[p][rt] = *reinterpret_cast<const uint4*>(ar[rt] + max(ks, 0) * astep);
      al[p][rt] = *reinterpret_cast<const uint4*>(ar[rt] + g.a_plane + max(ks, 0) * astep);
    }
  };
  auto mma = [&](int p, bool live) {   // (a step past the end multiplies a zero A fragment)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      uint4 x = a[p][rt], xl = al[p][rt];
      if (!live) x = xl = make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(w[p][ct]), as_bf16x8(x), acc[rt][ct], 0, 0, 0);
        acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(w[p][ct]), as_bf16x8(xl), acc[rt][ct], 0, 0, 0);
      }
    }
  };
#pragma unroll
  for (int p = 0; p < P; ++p) load(p, p);
  // AM 2: the sums of h^2 of row 16 rt + tid / 16 (column groups tid % 16 + 16 j), requested
  // behind the first steps and added up after the K loop
  constexpr int kSq = 4, NR = (16 * RT * 16 + 64 * NW - 1) / (64 * NW);   // rows per thread
  float sq[NR][kSq];
  if constexpr (AM == 2) {
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      const int64_t rrow = min(m0 + int(threadIdx.x >> 4) + 4 * NW * q, g.M - 1);
#pragma unroll
      for (int j = 0; j < kSq; ++j) {
        const int cg = int(threadIdx.x & 15) + 16 * j;
        sq[q][j] = g.ssq[rrow * g.nssq + min(cg, g.nssq - 1)];
      }
    }
  }
  // whole rounds of P steps with the next round's loads behind each step, then the last steps
  // (a load past the end would cost as much traffic as a step)
  int i0 = 0;
  for (; i0 + 2 * P <= ns; i0 += P) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      mma(p, true);
      load(p, i0 + p + P);
    }
  }
#pragma unroll
  for (int p = 0; p < P; ++p) {
    mma(p, i0 + p < ns);
    if (i0 + p + P < ns) load(p, i0 + p + P);
  }
  if (i0 + P < ns) {
#pragma unroll
    for (int p = 0; p < P - 1; ++p) mma(p, i0 + P + p < ns);
  }
  if constexpr (AM == 2) {   // the rows' sums of h^2 over their nssq <= 64 partials, in a fixed order
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < kSq; ++j) sum += int(threadIdx.x & 15) + 16 * j < g.nssq ? sq[q][j] : 0.f;
      sum = sum16_lanes(sum);
      const int row = int(threadIdx.x >> 4) + 4 * NW * q;
      if ((threadIdx.x & 15) == 0 && row < 16 * RT) {
        const float r = sqrtf(sum / float(g.K) + 1e-5f);
        rms[0][row] = r;
        rms[1][row] = 1.f / r;
      }
    }
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    f32x4(*rd)[CT][64] = red[rt & 1 & (RT - 1)];
    if constexpr (RT > 1) load_hold(rt);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) rd[wv][ct][lane] = acc[rt][ct];
    __syncthreads();
    const int row = m0 + 16 * rt + orow;
    const bool live = row < g.M;
    const EpiArgs& ea = g.e;
    int64_t crow = 0;
    const float* rp = nullptr;
    if constexpr (EPI == kEpiQkv) {   // the row's position: cache row and RoPE factors
      const int p = row_pos(ea.rows, min(row, g.M - 1));
      crow = cache_row(ea.rows, min(row, g.M - 1), p);
      rp = ea.rope + int64_t(p) * kDh;
    }
    float hsq = 0.f;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int ct = wv + NW * i;
      if (ct >= ctn) break;
      f32x4 v = rd[0][ct][lane];
#pragma unroll
      for (int w2 = 1; w2 < NW; ++w2) v += rd[w2][ct][lane];
      if constexpr (AM == 2) {
        const float r = rms[0][16 * rt + orow], rr = rms[1][16 * rt + orow];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = quotient(v[e], r, rr);
      }
      const int col = n0 + 16 * ct + ocol;
      if (!live) continue;
      if constexpr (EPI == kEpiStore) {
        *reinterpret_cast<f32x4*>(g.out + int64_t(row) * g.ldo + col) = v;
      } else if constexpr (kResid) {
        v += hold[i];
        const int64_t at = act_index(row, col, g.N, 0);
        *reinterpret_cast<f32x4*>(g.out + at) = v;
        if (ea.act) {
          const uint2 sc = *reinterpret_cast<const uint2*>(ea.xscale + col);
          const f32x4 x = {__uint_as_float(sc.x << 16) * v[0], __uint_as_float(sc.x & 0xffff0000u) * v[1],
                           __uint_as_float(sc.y << 16) * v[2], __uint_as_float(sc.y & 0xffff0000u) * v[3]};
          uint2 hi, lo;
          split2(x[0], x[1], hi.x, lo.x);
          split2(x[2], x[3], hi.y, lo.y);
          *reinterpret_cast<uint2*>(ea.act + at) = hi;
          *reinterpret_cast<uint2*>(ea.act + ea.act_plane + at) = lo;
          hsq += ((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2]) + v[3] * v[3];
        }
      } else if constexpr (EPI == kEpiSwiglu) {
        // (the tile copy orders the gate/up pairs by the down projection's input positions)
        const int64_t at = act_index(row, col >> 1, g.N / 2, 0);
        uint32_t hi, lo;
        split2(swiglu(v[0], v[1]), swiglu(v[2], v[3]), hi, lo);
        *reinterpret_cast<uint32_t*>(ea.act + at) = hi;
        *reinterpret_cast<uint32_t*>(ea.act + ea.act_plane + at) = lo;
      } else {
        qkv_quad(v, rp, col, row, ea, ea.qkv + int64_t(row) * g.N, crow);
      }
    }
    if constexpr (kResid) {   // the wave's columns of the row: four lanes, in a fixed order
      hsq += __shfl_xor(hsq, 16);
      hsq += __shfl_xor(hsq, 32);
      if (lane < 16) hs[rt][wv][lane] = hsq;
    }
  }
  if (kResid && g.e.act) {   // the waves' parts of each row's sum, in wave order
    __syncthreads();
    const int row = m0 + int(threadIdx.x);
    if (threadIdx.x < 16 * RT && row < g.M) {
      float sum = hs[threadIdx.x >> 4][0][threadIdx.x & 15];
#pragma unroll
      for (int w2 = 1; w2 < NW; ++w2) sum += hs[threadIdx.x >> 4][w2][threadIdx.x & 15];
      g.e.ssq[int64_t(row) * C + c] = sum;
    }
  }
}

__device__ __forceinline__ float block_sum256(float v, float* red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  const float s = (red[0] + red[1]) + (red[2] + red[3]);
  __syncthreads();
  return s;
}

// Row blockIdx.x + row0: h += sum_z part[z] (z in order), then
// xn[j] = scale[i] * (h[i] / sqrt(mean(h^2) + 1e-5)) as hi/lo bf16 parts (planes `plane` apart),
// with i the input element at position j of the packed row layout (model.py:94-98).  Every partial is requested before
// the first is added, so the sum costs one memory round trip.  With packed, h holds the row in
// packed order (element i at position perm_pos(i)) in tile order (act_index), and no partials are
// added.
__global__ __launch_bounds__(kNormThreads) void mx_norm(float* h, const float* part, int splits, int M, int d,
                                                        const uint16_t* scale, uint16_t* xn, int64_t plane,
                                                        int row0, int ldx, int packed) {
  constexpr int NE = kMaxRows / kNormThreads;
  __shared__ float red[4];
  __shared__ __align__(16) float hs[kMaxRows];
  const int m = blockIdx.x + row0;
  float* hr = h + int64_t(m) * d;
  // every load (residual, partials, the scales of this thread's outputs) is issued up front from
  // clamped indices: a load under a branch is waited for at the join.  Thread t sums elements
  // 4t..4t+3 (16-byte loads; d is a multiple of 32) and writes outputs t, t + 256, ...
  static_assert(kMaxRows == 4 * kNormThreads, "one float4 of the row per thread");
  const int n4 = 4 * threadIdx.x, n4c = min(n4, d - 4);
  const bool own = n4 < d;
  uint16_t sc[NE];
#pragma unroll
  for (int i = 0; i < NE; ++i) sc[i] = scale[perm_elem(min(int(threadIdx.x) + kNormThreads * i, d - 1), d)];
  float4 v = *reinterpret_cast<const float4*>(packed ? h + act_index(m, n4c, d, 0) : hr + n4c);
  {   // partials (none when splits == 0: then split 0 is read and ignored)
    float4 pv[kMaxSplitK];
#pragma unroll
    for (int z = 0; z < kMaxSplitK; ++z)
      pv[z] = *reinterpret_cast<const float4*>(part + (int64_t(min(z, max(splits, 1) - 1)) * M + m) * d + n4c);
#pragma unroll
    for (int z = 0; z < kMaxSplitK; ++z)
      if (z < splits) {
        v.x += pv[z].x;
        v.y += pv[z].y;
        v.z += pv[z].z;
        v.w += pv[z].w;
      }
  }
  float ss = 0.f;
  if (own) {
    if (splits) *reinterpret_cast<float4*>(hr + n4) = v;
    *reinterpret_cast<float4*>(hs + n4) = v;
    ss = ((v.x * v.x + v.y * v.y) + v.z * v.z) + v.w * v.w;
  }
  ss = block_sum256(ss, red);
  const float r = sqrtf(ss / float(d) + 1e-5f);
#pragma unroll
  for (int q = 0; q < NE; ++q) {
    const int j = threadIdx.x + kNormThreads * q;
    if (j < d)
      put_split(xn + act_index(blockIdx.x, j, d, ldx), plane, bf2f(sc[q]) * (hs[packed ? j : perm_elem(j, d)] / r));
  }
}

// Row m of the residual stream: the embedding of tokens[m] (element n at n, or with packed at its
// packed position perm_pos(n) in tile order, act_index).  With xscale (packed only) also the first
// RMSNorm's input planes, scale * h as hi/lo tiles (xn, lo plane `plane` further), and the row's
// sum of h^2 in ssq[m].
__global__ __launch_bounds__(256) void mx_embed(const uint16_t* emb, const int32_t* tokens, int d, float* h,
                                                int32_t* status, int V, int packed, const uint16_t* xscale,
                                                uint16_t* xn, int64_t plane, float* ssq) {
  __shared__ float red[4];
  const int m = blockIdx.x;
  int t = tokens[m];
  const bool bad = t < 0 || t >= V;
  if (threadIdx.x == 0) status[m] = bad ? 2 : 0;
  if (bad) t = 0;
  constexpr int NE = kMaxRows / 256;   // every load issued before the first store
  uint16_t e[NE];
#pragma unroll
  for (int i = 0; i < NE; ++i) e[i] = emb[int64_t(t) * d + min(int(threadIdx.x) + 256 * i, d - 1)];
  float hsq = 0.f;
#pragma unroll
  for (int i = 0; i < NE; ++i) {
    const int n = threadIdx.x + 256 * i;
    if (n < d) {
      const float hv = bf2f(e[i]);
      if (packed) {
        const int j = perm_pos(n, d);
        h[act_index(m, j, d, 0)] = hv;
        if (xscale) put_split(xn + act_index(m, j, d, 0), plane, bf2f(xscale[j]) * hv);
      } else {
        h[int64_t(m) * d + n] = hv;
      }
      hsq += hv * hv;
    }
  }
  if (xscale) {
    hsq = block_sum256(hsq, red);
    if (threadIdx.x == 0) ssq[m] = hsq;
  }
}

// Row blockIdx.x: q/k/v = sum_z part[z] (z in order) over the packed q/k/v rows; RoPE on the
// q and k pairs (packed rows 2i, 2i+1 = dims i, i+32; model.py:110-117) at the row's
// position; f32 q/k/v in natural head-dim order to qkv; bf16 K/V to the cache.
__global__ __launch_bounds__(256) void mx_qkv_fin(const float* part, int splits, int M, EpiArgs ea) {
  const int m = blockIdx.x, nq = (ea.H + 2 * ea.KV) * kDh;
  const int t = blockIdx.y * 256 + threadIdx.x;
  if (t >= nq / 4) return;
  const int col = 4 * t;   // column pairs (col, col + 1) and (col + 2, col + 3), one head
  float4 pv[kMaxSplitK];
#pragma unroll
  for (int z = 0; z < kMaxSplitK; ++z)
    pv[z] = *reinterpret_cast<const float4*>(part + (int64_t(min(z, splits - 1)) * M + m) * nq + col);
  const int p = row_pos(ea.rows, m);
  const int64_t crow = cache_row(ea.rows, m, p);
  float4 sv = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int z = 0; z < kMaxSplitK; ++z)
    if (z < splits) {
      sv.x += pv[z].x;
      sv.y += pv[z].y;
      sv.z += pv[z].z;
      sv.w += pv[z].w;
    }
  qkv_quad(f32x4{sv.x, sv.y, sv.z, sv.w}, ea.rope + int64_t(p) * kDh, col, m, ea, ea.qkv + int64_t(m) * nq, crow);
}

// Row blockIdx.x: act_f = silu(gate_f) * up_f over the summed partials (gate/up are the packed
// rows 2f, 2f+1; model.py:159), as hi/lo bf16 parts at the down projection's input position of f.
__global__ __launch_bounds__(256) void mx_swiglu_fin(const float* part, int splits, int M, int F, uint16_t* act,
                                                     int64_t plane) {
  const int m = blockIdx.x, f = 2 * (blockIdx.y * 256 + threadIdx.x);   // outputs f and f + 1 (F is even)
  if (f >= F) return;
  float4 pv[kMaxSplitK];
#pragma unroll
  for (int z = 0; z < kMaxSplitK; ++z)
    pv[z] = *reinterpret_cast<const float4*>(part + (int64_t(min(z, splits - 1)) * M + m) * (2 * F) + 2 * f);
  float g0 = 0.f, u0 = 0.f, g1 = 0.f, u1 = 0.f;
#pragma unroll
  for (int z = 0; z < kMaxSplitK; ++z)
    if (z < splits) {
      g0 += pv[z].x;
      u0 += pv[z].y;
      g1 += pv[z].z;
      u1 += pv[z].w;
    }
  put_split(act + act_index(m, perm_pos(f, F), F, 0), plane, swiglu(g0, u0));
  put_split(act + act_index(m, perm_pos(f + 1, F), F, 0), plane, swiglu(g1, u1));
}

// Reductions over the 16 lanes of a DPP row, every lane receiving the result (rotations by 1, 2,
// 4, 8).  The sum's rounding may differ between the lanes of a row; callers read one lane.
template <int CTRL>
__device__ __forceinline__ float dpp_ror(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, dpp_ror<0x121>(v));
  v = fmaxf(v, dpp_ror<0x122>(v));
  v = fmaxf(v, dpp_ror<0x124>(v));
  return fmaxf(v, dpp_ror<0x128>(v));
}
__device__ __forceinline__ float row16_sum(float v) {
  v += dpp_ror<0x121>(v);
  v += dpp_ror<0x122>(v);
  v += dpp_ror<0x124>(v);
  return v + dpp_ror<0x128>(v);
}

// Prefill: causal GQA attention of query block blockIdx.y (16 rows) for head blockIdx.x on the
// matrix cores.  The key range 0..q0+15 is cut into 32-key chunks, wave w taking chunks w, w + NW,
// ...: S = Q K^T (16 x 32) and O += P V (16 x 64) run on v_mfma_f32_16x16x32_bf16 with every f32
// operand as hi/lo bf16 parts (mfma3), the softmax is online per query row in f32, and the NW
// waves' (max, sum, O) are merged by log-sum-exp at the end.  Scale 1/sqrt(64) (model.py:98).
// MFMA operand lanes: A[i][8 (l / 16) ..] = row i = l % 16; B[8 (l / 16) ..][n] with n = l % 16;
// D: rows 4 (l / 16) + r of column l % 16.
// The head outputs go to the O projection's input planes at their packed positions, or with
// natural at their element index (the tile copy's O columns are in natural order).  K and V come as
// operand planes from the QKV epilogue, so a chunk is 16 loads of 1 KB and no conversion (reading f32
// rows took 40 loads of 64-byte segments and eight splits per chunk in every head and query block:
// 511 rows 17.2 us, now 8.8; 200 rows 8.5, now 5.7; 128 rows 6.6, now 4.9).  Eight waves past 128 rows
// (mean of 24 layers, eight / four: 200 rows 5.6 / 5.9 us, 511 9.0 / 8.9), four where no wave of eight
// would have a second chunk.
template <int NW>
__global__ __launch_bounds__(64 * NW) void mx_attention_prefill(const float* qkv, const uint16_t* kvp, int MP, int M, int H,
                                                                int KV, uint16_t* att, int64_t plane, int natural) {
  constexpr int PS = 36;   // row stride (floats) of a wave's P tile in LDS: 16-byte reads of 16 rows spread over banks
  __shared__ __align__(16) float sp[NW][16 * PS];
  __shared__ float sm[NW][16], sl[NW][16];
  __shared__ float so[NW][16][kDh + 4];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kq = lane >> 4;
  const int h = blockIdx.x, g = h / (H / KV);
  const int nqkv = (H + 2 * KV) * kDh, d = H * kDh;
  // the first half of the grid takes the later query blocks, latest first, the second half the earlier
  // ones, earliest first: two workgroups half a grid apart, which tend to share a CU, then have
  // about the same number of chunks together on every CU (511 rows: 10.2 -> 8.8 us, 200: 5.8 -> 5.7)
  const int half = gridDim.y / 2;
  const int q0 = 16 * (int(blockIdx.y) < half ? int(gridDim.y) - 1 - int(blockIdx.y) : int(blockIdx.y) - half);
  const int nk = min(q0 + 16, M), nch = (nk + 31) / 32;
  // Q fragments (rows past M read row M - 1: their outputs are not stored)
  uint4 qh[2], ql[2];
  {
    const float* qr = qkv + int64_t(min(q0 + r16, M - 1)) * nqkv + h * kDh + 8 * kq;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const float4 a = *reinterpret_cast<const float4*>(qr + 32 * ks);
      const float4 b = *reinterpret_cast<const float4*>(qr + 32 * ks + 4);
      const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      split8(x, qh[ks], ql[ks]);
    }
  }
  float m[4], l[4];   // rows 4 kq + r: running max and sum (alike in the 16 lanes of the row)
  f32x4 o[4];         // O columns 16 dt + r16
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    m[r] = -INFINITY;
    l[r] = 0.f;
    o[r] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float* P = sp[wv];
  const int64_t pl = int64_t(KV) * MP * kDh;
  const uint16_t* kp = kvp + int64_t(g) * MP * kDh + lane * 8;
  const uint16_t* vp = kp + 2 * pl;
  for (int c = wv; c < nch; c += NW) {
    const int kb = 32 * c;
    // K (B of S: key kb + 16 t + r16, dims 32 ks + 8 kq ..) and V (B of P V: keys kb + 8 kq .., dim 16
    // dt + r16), all requested before the first MFMA, each load one 1 KB piece; keys past M hold
    // anything: their scores are masked and their V is cleared below
    uint4 kh[2][2], kl[2][2], vh[4], vl[4];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const uint16_t* kr = kp + ((kb >> 4) + t) * 1024 + ks * 512;
        kh[t][ks] = *reinterpret_cast<const uint4*>(kr);
        kl[t][ks] = *reinterpret_cast<const uint4*>(kr + pl);
      }
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      const uint16_t* vr = vp + (dt * (MP >> 5) + (kb >> 5)) * 512;
      vh[dt] = *reinterpret_cast<const uint4*>(vr);
      vl[dt] = *reinterpret_cast<const uint4*>(vr + pl);
    }
    f32x4 s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) s[t] = mfma3(qh[ks], ql[ks], kh[t][ks], kl[t][ks], s[t]);
    }
    if (kb + 32 > M) {   // (uniform) V of keys past M: 0 (0 times what the padding holds could be NaN)
      const int nv = M - kb - 8 * kq;
      auto clear = [&](uint4& u) {
        uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = 2 * j + 1 < nv ? w[j] : (2 * j < nv ? w[j] & 0xffffu : 0u);
        u = make_uint4(w[0], w[1], w[2], w[3]);
      };
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        clear(vh[dt]);
        clear(vl[dt]);
      }
    }
    // scale, causal mask, online softmax of rows 4 kq + r over keys kb + 16 t + r16
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = q0 + 4 * kq + r;
      const int j0 = kb + r16, j1 = kb + 16 + r16;
      const float v0 = (j0 <= i && j0 < M) ? s[0][r] * 0.125f : -INFINITY;
      const float v1 = (j1 <= i && j1 < M) ? s[1][r] * 0.125f : -INFINITY;
      const float mn = fmaxf(m[r], row16_max(fmaxf(v0, v1)));
      const float p0 = mn == -INFINITY ? 0.f : expf(v0 - mn), p1 = mn == -INFINITY ? 0.f : expf(v1 - mn);
      const float alpha = m[r] == -INFINITY ? 0.f : expf(m[r] - mn);
      l[r] = l[r] * alpha + row16_sum(p0 + p1);
      m[r] = mn;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) o[dt][r] *= alpha;
      P[(4 * kq + r) * PS + r16] = p0;
      P[(4 * kq + r) * PS + 16 + r16] = p1;
    }
    __builtin_amdgcn_wave_barrier();
    uint4 ph, plo;
    {
      const float4 a = *reinterpret_cast<const float4*>(P + r16 * PS + 8 * kq);
      const float4 b = *reinterpret_cast<const float4*>(P + r16 * PS + 8 * kq + 4);
      const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      split8(x, ph, plo);
    }
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) o[dt] = mfma3(ph, plo, vh[dt], vl[dt], o[dt]);
    __builtin_amdgcn_wave_barrier();
  }
  // merge the waves by log-sum-exp
  if (r16 == 0)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      sm[wv][4 * kq + r] = m[r];
      sl[wv][4 * kq + r] = l[r];
    }
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) so[wv][4 * kq + r][16 * dt + r16] = o[dt][r];
  __syncthreads();
  if (threadIdx.x >= 256) return;
  const int qi = threadIdx.x >> 4, d4 = 4 * (threadIdx.x & 15);
  float mx = -INFINITY;
#pragma unroll
  for (int w = 0; w < NW; ++w) mx = fmaxf(mx, sm[w][qi]);
  float L = 0.f, O[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float wt = sm[w][qi] == -INFINITY ? 0.f : expf(sm[w][qi] - mx);
    L += sl[w][qi] * wt;
#pragma unroll
    for (int e = 0; e < 4; ++e) O[e] += so[w][qi][d4 + e] * wt;
  }
  const int i = q0 + qi, el = h * kDh + d4;
  if (i >= M) return;
  if (natural) {   // four consecutive positions
    uint2 hi, lo;
    split2(O[0] / L, O[1] / L, hi.x, lo.x);
    split2(O[2] / L, O[3] / L, hi.y, lo.y);
    const int64_t at = act_index(i, el, d, 0);
    *reinterpret_cast<uint2*>(att + at) = hi;
    *reinterpret_cast<uint2*>(att + plane + at) = lo;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) put_split(att + act_index(i, perm_pos(el + e, d), d, 0), plane, O[e] / L);
  }
}

static void launch_attention_prefill(int M, int H, int KV, hipStream_t s, const float* qkv, const uint16_t* kvp, int MP,
                                     uint16_t* att, int64_t plane, int natural) {
  const dim3 grid(H, (M + 15) / 16);
  if (M > 128)
    hipLaunchKernelGGL(mx_attention_prefill<8>, grid, dim3(512), 0, s, qkv, kvp, MP, M, H, KV, att, plane, natural);
  else
    hipLaunchKernelGGL(mx_attention_prefill<4>, grid, dim3(256), 0, s, qkv, kvp, MP, M, H, KV, att, plane, natural);
}

// Batched decode: row m = blockIdx.x (one sequence at position p = pos(m)) and the GH query heads
// GH blockIdx.y .. (of one K/V head) attend over the cached rows 0..p-1 of the sequence (bf16, through
// its page table) and the row's current, un-rounded K/V (multi_sm_decode.py:182-221).  What bounds it
// is latency and load instructions, not bytes (24 rows of up to 384 positions: 21 MB when every head
// reads its K/V): wave w takes the 32-position blocks w, w + 8, ..., the next block's rows requested
// before the current one's arithmetic.  Lane l reads dims 8 (l % 8) .. + 8 of position 8 i + l / 8, i = 0..3,
// of K and of V: whole rows, 1 KB per instruction (a lane per position for K and per dim for V took
// 72 instructions per 64 positions and 64 cache lines per K instruction: 13.9 us for the 24 rows, now
// 8.4; 5 rows at position 211: 7.4, now 5.4).  The
// 8 lanes of a position add their partial scores with DPP, so every lane ends up with the weights of
// exactly the V rows it holds; only (max, sum, output) partials go through LDS at the end.
constexpr int kAttnWaves = 8;
// The longest context of verification and batched decode: that of the decode step whose rows they stand for
// (msdecode.hip).  The kernel itself streams blocks and has no bound of its own.
constexpr int kDecodeMaxCtx = 2048;
__device__ __forceinline__ float sum8_lanes(float v) {   // over each 8 consecutive lanes, as sum16_lanes
  v += dpp<0xB1, 0xf>(v, 0.f);
  v += dpp<0x4E, 0xf>(v, 0.f);
  return v + dpp<0x141, 0xf>(v, 0.f);
}
template <int GH>
__global__ __launch_bounds__(64 * kAttnWaves) void mx_attention_decode(const float* qkv, Rows rows, int H, int KV,
                                                                       const uint16_t* kc, const uint16_t* vc,
                                                                       uint16_t* att, int64_t plane, int natural) {
  // per wave and row of 16 lanes: the output's partial sums and the softmax denominator's
  __shared__ float so[kAttnWaves][4][GH][kDh];
  __shared__ float sl[kAttnWaves][4][GH];
  __shared__ float sm[kAttnWaves][GH];
  constexpr int kPos = 32, kLd = kPos / 8;   // positions per block, loads of K and of V per lane
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = lane >> 3, d8 = 8 * (lane & 7);
  const int m = blockIdx.x, h0 = GH * blockIdx.y, g = h0 / (H / KV);
  const int nqkv = (H + 2 * KV) * kDh, d = H * kDh;
  const float* qr = qkv + int64_t(m) * nqkv;
  // the page-table loads do not wait for p (every entry of a row is a sanitized page; p only selects
  // which rows are cached positions); positions past the table or past p read the row of position 0
  auto page_of = [&](int page) {   // wave-uniform
    return rows.pages ? rows.pages[int64_t(rows.batched ? m : 0) * rows.max_pages + min(page, rows.max_pages - 1)] : page;
  };
  int pg0 = page_of(2 * wv), pg1 = page_of(2 * wv + 1);
  const int first = page_of(0);
  const int p = row_pos(rows, m);
  float q[GH][8], kcur[8], vcur[8];
  auto load8 = [&](const float* src, float (&x)[8]) {
    const float4 a = *reinterpret_cast<const float4*>(src), b = *reinterpret_cast<const float4*>(src + 4);
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
    x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
  };
#pragma unroll
  for (int h = 0; h < GH; ++h) load8(qr + (h0 + h) * kDh + d8, q[h]);
  load8(qr + (H + g) * kDh + d8, kcur);
  load8(qr + (H + KV + g) * kDh + d8, vcur);
  const uint16_t* kg = kc + int64_t(g) * rows.pool * kDh + d8;
  const uint16_t* vg = vc + int64_t(g) * rows.pool * kDh + d8;
  uint4 kb[2][kLd], vb[2][kLd];
  auto load = [&](uint4 (&k)[kLd], uint4 (&v)[kLd], int blk, int p0, int p1) {
#pragma unroll
    for (int i = 0; i < kLd; ++i) {
      const bool in = kPos * blk + 8 * i + sub < p;
      const int64_t r = in ? int64_t(i < 2 ? p0 : p1) * kPage + (8 * i + sub) % kPage : int64_t(first) * kPage;
      k[i] = *reinterpret_cast<const uint4*>(kg + r * kDh);
      v[i] = *reinterpret_cast<const uint4*>(vg + r * kDh);
    }
  };
  const int nb = (p + kPos - 1) / kPos;
  load(kb[0], vb[0], wv, pg0, pg1);
  // the last wave starts from the current position (its first 8 lanes), the others from nothing
  float mx[GH], ls[GH], o[GH][8];
#pragma unroll
  for (int h = 0; h < GH; ++h) {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) s += q[h][e] * kcur[e];
    s = sum8_lanes(s) * 0.125f;
    const bool cur = wv == kAttnWaves - 1;
    mx[h] = cur ? s : -INFINITY;
    ls[h] = cur && sub == 0 ? 1.f : 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[h][e] = cur && sub == 0 ? vcur[e] : 0.f;
  }
  auto unpack = [](uint4 u, float (&x)[8]) {
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[2 * e] = __uint_as_float(w[e] << 16);
      x[2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
    }
  };
  auto block = [&](const uint4 (&k)[kLd], const uint4 (&v)[kLd], int blk) {
    float s[GH][kLd], old[GH];
#pragma unroll
    for (int h = 0; h < GH; ++h) old[h] = mx[h];
#pragma unroll
    for (int i = 0; i < kLd; ++i) {
      float x[8];
      unpack(k[i], x);
      const bool in = kPos * blk + 8 * i + sub < p;
#pragma unroll
      for (int h = 0; h < GH; ++h) {
        float a = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) a += q[h][e] * x[e];
        s[h][i] = in ? sum8_lanes(a) * 0.125f : -INFINITY;
      }
    }
#pragma unroll
    for (int h = 0; h < GH; ++h) {
      const float bm = wave_max(fmaxf(fmaxf(s[h][0], s[h][1]), fmaxf(s[h][2], s[h][3])));
      mx[h] = fmaxf(mx[h], bm);
      const float nm = mx[h] == -INFINITY ? 0.f : mx[h];   // (only scores of -inf so far: weights 0)
      const float al = expf(old[h] - nm);
#pragma unroll
      for (int i = 0; i < kLd; ++i) s[h][i] = expf(s[h][i] - nm);
      ls[h] = ls[h] * al + ((s[h][0] + s[h][1]) + (s[h][2] + s[h][3]));
#pragma unroll
      for (int e = 0; e < 8; ++e) o[h][e] *= al;
    }
#pragma unroll
    for (int i = 0; i < kLd; ++i) {
      float x[8];
      unpack(v[i], x);
#pragma unroll
      for (int h = 0; h < GH; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e) o[h][e] += s[h][i] * x[e];
    }
  };
  for (int blk = wv; blk < nb; blk += 2 * kAttnWaves) {
    const int b1 = blk + kAttnWaves, b2 = b1 + kAttnWaves;
    if (b1 < nb) load(kb[1], vb[1], b1, page_of(2 * b1), page_of(2 * b1 + 1));
    block(kb[0], vb[0], blk);
    if (b2 < nb) load(kb[0], vb[0], b2, page_of(2 * b2), page_of(2 * b2 + 1));
    if (b1 < nb) block(kb[1], vb[1], b1);
  }
  // the two positions of each row of 16 lanes are added here, the rest by the merge below
#pragma unroll
  for (int h = 0; h < GH; ++h) {
    const float l2 = ls[h] + dpp<0x128, 0xf>(ls[h], 0.f);   // row_ror 8: lane ^ 8
    if ((lane & 15) == 0) sl[wv][lane >> 4][h] = l2;
    if (lane == 0) sm[wv][h] = mx[h];
    float r[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = o[h][e] + dpp<0x128, 0xf>(o[h][e], 0.f);
    if ((lane & 8) == 0) {
      float* dst = so[wv][lane >> 4][h] + d8;
      *reinterpret_cast<float4*>(dst) = make_float4(r[0], r[1], r[2], r[3]);
      *reinterpret_cast<float4*>(dst + 4) = make_float4(r[4], r[5], r[6], r[7]);
    }
  }
  __syncthreads();
  // dims 2 t, 2 t + 1 of a head: the waves' states merged by log-sum-exp (waves without a position
  // carry weight 0)
  if (threadIdx.x < GH * kDh / 2) {
    const int h = threadIdx.x / (kDh / 2), e = 2 * (threadIdx.x % (kDh / 2));
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) M = fmaxf(M, sm[w][h]);
    float num0 = 0.f, num1 = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) {
      const float a = expf(sm[w][h] - M);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float2 v = *reinterpret_cast<const float2*>(so[w][r][h] + e);
        num0 += a * v.x;
        num1 += a * v.y;
        den += a * sl[w][r][h];
      }
    }
    num0 /= den;
    num1 /= den;
    const int el = (h0 + h) * kDh + e;
    if (natural) {
      uint32_t hi, lo;
      split2(num0, num1, hi, lo);
      const int64_t at = act_index(m, el, d, 0);
      *reinterpret_cast<uint32_t*>(att + at) = hi;
      *reinterpret_cast<uint32_t*>(att + plane + at) = lo;
    } else {
      put_split(att + act_index(m, perm_pos(el, d), d, 0), plane, num0);
      put_split(att + act_index(m, perm_pos(el + 1, d), d, 0), plane, num1);
    }
  }
}

// Four heads of a K/V head per workgroup read its K/V rows once, but their workgroups take four times as
// long, so the last pass over the CUs has to be nearly full (7/8): measured per step at 12..100 / 48..384
// positions, four heads against one: 306M 64 rows (256 workgroups) 0.950 / 0.937, 56 (224) 0.966 / 0.973,
// 128 (512) 0.941 / 0.956, 40 (160) 0.983 / 1.013, 96 (384) 1.013 / 1.027, 72 (288) 1.044 / 1.051;
// 512 wide with 8 heads, 128 rows (256) 0.980 / 0.963, 96 (192) 1.003 / 1.019, 160 (320) 1.042 / 1.069.
// (Two heads, 24 rows of the 306M: 806 us against 803 with one and 859 with four.)
static void launch_attention_decode(int M, int H, int KV, hipStream_t s, const float* qkv, const Rows& rows,
                                    const uint16_t* kc, const uint16_t* vc, uint16_t* att, int64_t plane,
                                    int natural) {
  const int G = H / KV;
  auto go = [&](auto k, int gh) {
    hipLaunchKernelGGL(k, dim3(M, H / gh), dim3(64 * kAttnWaves), 0, s, qkv, rows, H, KV, kc, vc, att, plane, natural);
  };
  const int last = (M * H / 4 + 255) % 256 + 1;   // workgroups of the last pass
  if (G % 4 == 0 && last >= 224) go(mx_attention_decode<4>, 4);
  else go(mx_attention_decode<1>, 1);
}

// Tied logits of several rows: out[m][v] = sum_k x[m][k] W[v][k] with x the final norm's hi/lo planes
// (rows of K) and W the embedding rows.  A workgroup of four waves owns 128 vocabulary rows x TOK rows;
// K advances 32 at a time through a ring of S LDS stages filled by direct DMA (W rows, hi rows, lo
// rows of 64 bytes; piece c of row r at position c ^ ((r >> 2) & 3), which makes the fragment reads
// conflict-free).  Each output sums K steps in order, hi then lo, on 16 x 16 x 32 MFMAs as mx_gemm
// does, so the last row's logits are bitwise the same whether one row or every row is requested.
// mx_gemm's fragment loads of the row layout are 64 requests of 16 bytes each and bound it: 203 rows
// of d 768 93 us, here 32.5; 24 rows of d 1024 33 us, here 15.8 (65 MB: 13 us at the card's
// copy rate).  TOK: 32 and 64 where the rows fit, else 128 (LDS reads per MFMA fall with TOK).
template <int RB, int CB>
struct LogitFrags {
  u32x4v w[RB], x[2][CB];
};
// the fragment reads of a stage and their wait in one block
__device__ __forceinline__ void logit_reads(LogitFrags<2, 2>& f, uint32_t a, uint32_t b, uint32_t bl) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile(
      "ds_read_b128 %0, %6\nds_read_b128 %1, %6 offset:1024\n"
      "ds_read_b128 %2, %7\nds_read_b128 %3, %7 offset:1024\n"
      "ds_read_b128 %4, %8\nds_read_b128 %5, %8 offset:1024\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(f.w[0]), "=&v"(f.w[1]), "=&v"(f.x[0][0]), "=&v"(f.x[0][1]), "=&v"(f.x[1][0]), "=&v"(f.x[1][1])
      : "v"(a), "v"(b), "v"(bl));
#endif
}
__device__ __forceinline__ void logit_reads(LogitFrags<4, 2>& f, uint32_t a, uint32_t b, uint32_t bl) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile(
      "ds_read_b128 %0, %8\nds_read_b128 %1, %8 offset:1024\n"
      "ds_read_b128 %2, %8 offset:2048\nds_read_b128 %3, %8 offset:3072\n"
      "ds_read_b128 %4, %9\nds_read_b128 %5, %9 offset:1024\n"
      "ds_read_b128 %6, %10\nds_read_b128 %7, %10 offset:1024\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(f.w[0]), "=&v"(f.w[1]), "=&v"(f.w[2]), "=&v"(f.w[3]), "=&v"(f.x[0][0]), "=&v"(f.x[0][1]),
        "=&v"(f.x[1][0]), "=&v"(f.x[1][1])
      : "v"(a), "v"(b), "v"(bl));
#endif
}
__device__ __forceinline__ void logit_reads(LogitFrags<4, 4>& f, uint32_t a, uint32_t b, uint32_t bl) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile(
      "ds_read_b128 %0, %12\nds_read_b128 %1, %12 offset:1024\n"
      "ds_read_b128 %2, %12 offset:2048\nds_read_b128 %3, %12 offset:3072\n"
      "ds_read_b128 %4, %13\nds_read_b128 %5, %13 offset:1024\n"
      "ds_read_b128 %6, %13 offset:2048\nds_read_b128 %7, %13 offset:3072\n"
      "ds_read_b128 %8, %14\nds_read_b128 %9, %14 offset:1024\n"
      "ds_read_b128 %10, %14 offset:2048\nds_read_b128 %11, %14 offset:3072\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(f.w[0]), "=&v"(f.w[1]), "=&v"(f.w[2]), "=&v"(f.w[3]), "=&v"(f.x[0][0]), "=&v"(f.x[0][1]),
        "=&v"(f.x[0][2]), "=&v"(f.x[0][3]), "=&v"(f.x[1][0]), "=&v"(f.x[1][1]), "=&v"(f.x[1][2]), "=&v"(f.x[1][3])
      : "v"(a), "v"(b), "v"(bl));
#endif
}
// at most n (< D) stages of NI DMA instructions outstanding, then the workgroup's barrier (a bare one:
// __syncthreads would wait for every outstanding DMA)
template <int NI, int D>
__device__ __forceinline__ void wait_stage_barrier(int n) {
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (D > 1) {
    if (n < D - 1) return wait_stage_barrier<NI, D - 1>(n);
  }
  asm volatile("s_waitcnt vmcnt(%0)\ns_barrier" ::"n"((D - 1) * NI) : "memory");
#endif
}
constexpr int kLogitRows = 128;   // vocabulary rows per workgroup
template <int TOK>
__global__ __launch_bounds__(256) void mx_logits(const uint16_t* X, int64_t plane, const uint16_t* W, int M, int V, int K,
                                                 float* out) {
  constexpr int GM = TOK == 32 ? 4 : 2, GN = 4 / GM;              // waves over vocabulary x rows
  constexpr int RB = kLogitRows / GM / 16, CB = TOK / GN / 16;    // 16-row fragments per wave
  constexpr int SD = (kLogitRows + 2 * TOK) * 64, NI = SD / 1024 / 4, S = TOK == 128 ? 3 : (TOK == 64 ? 4 : 6), D = S - 1;
  __shared__ __align__(1024) uint8_t ring[S * SD];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wv / GN, wn = wv % GN;
  // (each XCD takes a contiguous range of the tiles, row tiles innermost, so W reaches its L2 once)
  const int MT = (M + TOK - 1) / TOK, xcd = blockIdx.x & 7, per = gridDim.x >> 3, rest = gridDim.x & 7;
  const int id = xcd * per + min(xcd, rest) + (blockIdx.x >> 3);
  const int v0 = kLogitRows * (id / MT), m0 = TOK * (id % MT);
  // instruction u of this wave fills the 1 KB piece wv + 4 u of a stage: 16 rows of W, hi or lo (rows
  // past the last read the last)
  const uint16_t* src[NI];
#pragma unroll
  for (int u = 0; u < NI; ++u) {
    const int q = wv + 4 * u, x = q - kLogitRows / 16;
    const int r = 16 * (x < 0 ? q : x % (TOK / 16)) + (lane >> 2);
    const int piece = (lane & 3) ^ ((r >> 2) & 3);
    src[u] = (x < 0 ? W + int64_t(min(v0 + r, V - 1)) * K
                    : X + (x < TOK / 16 ? 0 : plane) + int64_t(min(m0 + r, M - 1)) * K) + 8 * piece;
  }
  auto dma = [&](int kt) {
#if defined(__HIP_DEVICE_COMPILE__)
    uint8_t* st = ring + (kt % S) * SD;
#pragma unroll
    for (int u = 0; u < NI; ++u)
      __builtin_amdgcn_global_load_lds(src[u] + kt * kBK,
                                       (__attribute__((address_space(3))) void*)(st + 1024 * (wv + 4 * u)), 16, 0, 0);
#endif
  };
  const int KT = K / kBK;
  for (int s = 0; s < D && s < KT; ++s) dma(s);
  f32x4 acc[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int r16 = lane & 15, kq = lane >> 4;
  const uint32_t base = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)ring));
  const uint32_t fr = base + r16 * 64 + ((kq ^ ((r16 >> 2) & 3)) << 4);
  for (int kt = 0; kt < KT; ++kt) {
    // stage kt landed for every wave, and stage kt - 1's reads done: its slot takes stage kt + D
    wait_stage_barrier<NI, D>(min(KT, kt + D) - kt - 1);
    if (kt + D < KT) dma(kt + D);
    const uint32_t st = fr + (kt % S) * SD;
    LogitFrags<RB, CB> f;
    const uint32_t b = st + (kLogitRows + wn * 16 * CB) * 64;
    logit_reads(f, st + wm * RB * 1024, b, b + TOK * 64);
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        const bf16x8 w = __builtin_bit_cast(bf16x8, f.w[i]);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, __builtin_bit_cast(bf16x8, f.x[0][j]), acc[i][j], 0, 0, 0);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, __builtin_bit_cast(bf16x8, f.x[1][j]), acc[i][j], 0, 0, 0);
      }
  }
  // a lane holds four consecutive vocabulary ids of one row (V is a multiple of 16)
#pragma unroll
  for (int j = 0; j < CB; ++j) {
    const int m = m0 + 16 * (wn * CB + j) + r16;
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      const int v = v0 + 16 * (wm * RB + i) + 4 * kq;
      if (m < M && v < V) *reinterpret_cast<f32x4*>(out + int64_t(m) * V + v) = acc[i][j];
    }
  }
}

// argmax of each row of logits (lowest index on ties): out[2*row] = index, out[2*row+1] = the pass's
// status, i.e. every row's flags (status[0..nflags): tokens by mx_embed, then positions by
// mx_sanitize_rows) together.  copy (optional, one row): the row's logits again.
__global__ __launch_bounds__(1024) void mx_argmax(const float* logits, int V, int ld, int32_t* out,
                                                  const int32_t* status, int nflags, float* copy) {
  __shared__ uint64_t red[16];
  __shared__ int rflags[16];
  int flags = 0;
  for (int i = threadIdx.x; i < nflags; i += 1024) flags |= status[i];
  const float* lr = logits + int64_t(blockIdx.x) * ld;
  uint64_t best = 0;
  constexpr int kBatch = 16;   // loads in flight per thread (clamped, so none sits under a branch)
  for (int j0 = threadIdx.x; j0 < V; j0 += kBatch * 1024) {
    float x[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) x[u] = lr[min(j0 + 1024 * u, V - 1)];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int j = j0 + 1024 * u;
      if (copy && j < V) copy[j] = x[u];
      uint32_t b = __float_as_uint(x[u]);
      b = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
      const uint64_t key = (uint64_t(b) << 32) | uint64_t(0xffffffffu - uint32_t(j));
      best = j < V && key > best ? key : best;
    }
  }
  for (int o = 32; o; o >>= 1) {
    const uint64_t w = __shfl_xor(best, o);
    best = w > best ? w : best;
  }
  flags = (__any(flags & 2) ? 2 : 0) | (__any(flags & 4) ? 4 : 0);
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6] = best;
    rflags[threadIdx.x >> 6] = flags;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t b = red[0];
    for (int i = 1; i < 16; ++i) {
      b = red[i] > b ? red[i] : b;
      flags |= rflags[i];
    }
    out[2 * blockIdx.x] = int32_t(0xffffffffu - uint32_t(b & 0xffffffffu));
    out[2 * blockIdx.x + 1] = flags;
  }
}

// Copies the rows' positions and page tables into the workspace, which is what every later
// kernel addresses the cache with: a position outside [0, ctx) or past the table, and a table
// entry outside the pool, is replaced by 0 (status bit 2), so no access leaves the pool.
// pos == NULL: every row is at fixed_pos (the last position of a prefill).
__global__ void mx_sanitize_rows(const int32_t* pos, int fixed_pos, const int32_t* pages, int M, int max_pages,
                                 int ctx, int pool_pages, int32_t* pos_out, int32_t* pages_out, int32_t* status) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  int p = pos ? pos[m] : fixed_pos;
  bool bad = p < 0 || p >= ctx || p / kPage >= max_pages;
  if (bad) p = 0;
  constexpr int kBatch = 8;   // page-table loads in flight (clamped indices, stores after)
  for (int i0 = 0; i0 < max_pages; i0 += kBatch) {
    int pv[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) pv[u] = pages[int64_t(m) * max_pages + min(i0 + u, max_pages - 1)];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int i = i0 + u;
      int pg = pv[u];
      if (pg < 0 || pg >= pool_pages) {
        if (i < max_pages && i <= p / kPage) bad = true;
        pg = 0;
      }
      if (i < max_pages) pages_out[int64_t(m) * max_pages + i] = pg;
    }
  }
  if (pos_out) pos_out[m] = p;
  status[m] = bad ? 4 : 0;
}

// One 16-byte piece per thread of the tile copy of an N x K matrix W (rows in packed order): piece
// p is lane p % 64 of tile p / 64 = (n / 16) (K / 32) + k / 32, i.e. row n = 16 (tile / (K / 32)) +
// lane % 16 at positions 32 (tile % (K / 32)) + 8 (lane / 16) .. + 8.  Row orders (rowperm): 1 = row
// n of the copy is row perm_elem(n, N) of W, so output column n is element perm_elem(n) of an
// N-long vector, i.e. its packed position n (the O and down projections, whose outputs add to the
// residual); 2 = row pair n / 2 is pair perm_elem(n / 2, N / 2) (gate/up: output pair f is then the
// down projection's input at its packed position f).  With natk, column k of the copy is input
// element k (W's column perm_pos(k)): the O projection, whose input the attention writes in
// natural order.  Either way an epilogue's consecutive outputs land on consecutive positions.
__global__ __launch_bounds__(256) void mx_pack_tiles(const uint16_t* W, int N, int K, int rowperm, int natk,
                                                     uint16_t* T) {
  const int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const int S = K / kBK;
  if (p >= int64_t(N) * S * 64) return;
  const int lane = int(p & 63);
  const int64_t tile = p >> 6;
  const int n = int(16 * (tile / S)) + (lane & 15);
  const int64_t src = rowperm == 1 ? perm_elem(n, N) : (rowperm == 2 ? 2 * perm_elem(n >> 1, N / 2) + (n & 1) : n);
  const int k = kBK * int(tile % S) + 8 * (lane >> 4);
  if (natk) {
    uint16_t v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = W[src * K + perm_pos(k + e, K)];
#pragma unroll
    for (int e = 0; e < 8; ++e) T[p * 8 + e] = v[e];
  } else {
    *reinterpret_cast<uint4*>(T + p * 8) = *reinterpret_cast<const uint4*>(W + src * K + k);
  }
}

// A layer's two RMSNorm scales in packed order: out[j] = scale[perm_elem(j, d)] for [ln1 | ln2].
__global__ __launch_bounds__(256) void mx_pack_scales(const uint16_t* ln, int d, uint16_t* out) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= 2 * d) return;
  const int half = j >= d ? d : 0;
  out[j] = ln[half + perm_elem(j - half, d)];
}

// ---------------------------------------------------------------- host side
struct Layout {
  size_t h, xn, ssq, qkv, kvp, att, act, part, status, rowpos, pages, bytes;
};

static size_t al256(size_t x) { return (x + 255) & ~size_t(255); }


// Widest projection mx_gemm_rows takes with weights in row order: wider ones (the 306M gate/up,
// 5632 outputs) run faster on the split-K kernel (measured: 128-token prefill 1.95 -> 1.79 ms).
constexpr int kRowsMaxN = 4096;

// Column tiles (of 16) per workgroup of mx_gemm_rows with weights in row order: the widest that still
// gives about one workgroup per compute unit; 0 when the projection has too few output tiles for it
// (few rows), or too short a K for every wave to take a step, and the split-K kernel runs instead.
static int rows_ct(int M, int N, int K) {
  const int T = (M + 15) / 16, n16 = N / 16;
  if (K / kBK < 4 || M < 48 || N > kRowsMaxN) return 0;
  for (int ct : {8, 6, 4, 3, 2, 1})
    if (n16 % ct == 0 && T * (n16 / ct) >= 224) return ct;
  return 0;
}

// Output tile of a workgroup of mx_gemm_rows with weights in tile order: RT x CT tiles of 16.
struct RowsTile {
  int rt, ct, nw;   // row tiles, column tiles, waves
};
constexpr RowsTile kRowsTiles[] = {{1, 1, 8}, {1, 1, 4}, {1, 2, 4}, {1, 3, 4}, {1, 4, 4}, {1, 6, 4},
                                   {2, 3, 4}, {2, 4, 4}, {2, 6, 4}, {4, 4, 4}, {4, 6, 4}, {4, 11, 4}};

// The tile of a projection, from a model of its time (us) fitted to cold-weight runs of the 306M
// projections at 5..511 rows (within ~10 % of each; e.g. 511-row gate/up: 4 x 11 19.0 us, 2 x 6
// 20.5, 4 x 6 25.2, 1 x 8 27.4; 128-row gate/up 2 x 6 8.9, 1 x 3 11.2; 24-row 1 x 3 5.7, 1 x 2 6.9).
// The widest entry is 11 column tiles because the 306M's gate/up has 352: from 449 rows (8 row groups of
// 4) on, 11 make one workgroup per CU, 12 leave 16 CUs idle (passes of 383 and 511 rows 1568 / 1569 us
// with 11, 1576 / 1584 with 12; the other models' passes within 1 % either way) and 10 take a second
// pass over the CUs.  The model: launch, first loads and drain 2.6; every K step moves 2 RT + CT operand
// fragments into the CU (13 ns each); the epilogue takes 0.19 per tile; workgroups past one per
// CU cost a share of both where two fit a CU's registers (up to 12 tiles), whole passes where not.
// max_groups: an upper limit on column groups (0: none).
static RowsTile rows_tile(int M, int N, int K, int max_groups = 0) {
  const int T = (M + 15) / 16, n16 = N / 16, S = K / kBK;
  RowsTile best = kRowsTiles[0];
  double best_cost = 1e30;
  for (const RowsTile& t : kRowsTiles) {
    const int C = (n16 + t.ct - 1) / t.ct;
    if (max_groups && C > max_groups) continue;
    // single tiles: 8 waves for one row tile, and for a long K until the grid fills the chip (down
    // projection, 8 / 4 waves: 5 rows 5.3 / 5.7 us, 24 rows 5.4 / 5.5, 64 rows 6.8 / 5.8)
    if (t.rt * t.ct == 1 && (t.nw == 8) != (T == 1 || (S >= 64 && T < 4))) continue;
    const int wg = ((T + t.rt - 1) / t.rt) * C;
    const double step = 0.013 * (2 * t.rt + t.ct) * S, epi = 0.19 * t.rt * t.ct;
    const double cost = t.rt * t.ct <= 12 ? std::max(1.0, wg / 256.0) * step + epi + (wg > 256 ? 0.4 : 0.0)
                                          : ((wg + 255) / 256) * (step + epi);
    if (cost < best_cost) {
      best_cost = cost;
      best = t;
    }
  }
  return best;
}

// Column groups of the O and down projections, which leave one partial sum of h^2 each per row (the
// consumer takes up to 64).
constexpr int kMaxGroups = 64;
static int resid_groups(int M, int N, int K) {
  const int ct = rows_tile(M, N, K, kMaxGroups).ct;
  return (N / 16 + ct - 1) / ct;
}

// K splits of a projection: 1 for mx_gemm_rows, else enough split-K workgroups to occupy every
// compute unit, at least 4 K steps each
static int splits_for(int M, int N, int K, int bm, bool tw) {
  if (tw || rows_ct(M, N, K) > 0) return 1;
  const int tiles = (N / kBN) * ((M + bm - 1) / bm);
  int s = 1;
  while (tiles * s < 256 && (K / kBK) / (2 * s) >= 4 && 2 * s <= kMaxSplitK) s *= 2;
  return s;
}

static int bm_for(int M) { return M <= 16 ? 16 : (M <= 64 ? 64 : 128); }

static size_t part_floats(const msd_config* c, int M) {
  const int d = c->d_model, ff = c->d_ff, nqkv = (c->n_heads + 2 * c->n_kv_heads) * kDh;
  const int bm = bm_for(M);
  size_t mx = 0;
  for (bool tw : {false, true}) {
    mx = std::max(mx, size_t(splits_for(M, nqkv, d, bm, tw)) * nqkv);
    mx = std::max(mx, size_t(splits_for(M, d, d, bm, tw)) * d);
    mx = std::max(mx, size_t(splits_for(M, 2 * ff, d, bm, tw)) * 2 * ff);
    mx = std::max(mx, size_t(splits_for(M, d, ff, bm, tw)) * d);
  }
  return mx * M;
}

// The largest part_floats over passes of 1..M rows: a pass of fewer rows may split K more and need more
// (306M: 128 rows 9.4 MB of partials, 129 rows 4.2).  The split counts change with the number of
// 16-row tiles and at 48 rows only, and are 1 for every N past kRowsPerPass rows, so the last two row
// counts of each 16 cover them all.
static size_t part_floats_upto(const msd_config* c, int M) {
  constexpr int kRowsPerPass = 128 * 256;   // a 128-row tile per CU
  size_t mx = part_floats(c, M);
  for (int m = 16; m < M + 16 && m <= kRowsPerPass; m += 16)
    for (int q : {m - 1, m}) mx = std::max(mx, part_floats(c, std::min(q, M)));
  return mx;
}

static int pad16(int M) { return (M + 15) & ~15; }
static int pad32(int M) { return (M + 31) & ~31; }

// part: floats of the split-K partials
static Layout layout(const msd_config* c, int M, size_t part) {
  const int d = c->d_model, ff = c->d_ff, nqkv = (c->n_heads + 2 * c->n_kv_heads) * kDh;
  Layout L;
  size_t o = 0;
  L.h = o;      o += al256(size_t(pad16(M)) * d * 4);   // rows padded to whole tiles (tile order)
  // activation planes (hi and lo) in tile order, rows padded to whole tiles
  L.xn = o;     o += al256(size_t(pad16(M)) * d * 2 * 2);
  L.ssq = o;    o += al256(size_t(M) * (d / 16) * 4);   // partial sums of h^2: at most d / 16 per row
  L.qkv = o;    o += al256(size_t(M) * nqkv * 4);
  L.kvp = o;    o += al256(size_t(pad32(M)) * c->n_kv_heads * kDh * 2 * 4);   // prefill: K/V operand planes
  L.att = o;    o += al256(size_t(pad16(M)) * d * 2 * 2);
  L.act = o;    o += al256(size_t(pad16(M)) * ff * 2 * 2);
  L.part = o;   o += al256(part * 4);
  L.status = o; o += al256(size_t(M) * 2 * 4);   // flags: each row's token, then each row's position
  L.rowpos = o; o += al256(size_t(M) * 4);
  L.pages = o;  o += al256(size_t(M) * ((c->context_len + kPage - 1) / kPage) * 4);
  L.bytes = o;
  return L;
}
static Layout layout(const msd_config* c, int M) { return layout(c, M, part_floats(c, M)); }

// Bytes that hold any pass of 1..M rows (every other region grows with the rows).
static int64_t workspace_bytes(const msd_config* c, int M) {
  return int64_t(layout(c, M, part_floats_upto(c, M)).bytes);
}

static bool mx_config_ok(const msd_config* c) {
  if (!c || c->d_head != kDh || c->n_heads <= 0 || c->n_kv_heads <= 0 || c->n_layers <= 0) return false;
  if (c->n_heads * kDh != c->d_model || c->n_heads % c->n_kv_heads) return false;
  if (c->d_model % kBN || (2 * c->d_ff) % kBN || c->vocab_size % kBN || c->d_ff % 8) return false;
  if (c->d_model % kBK || c->d_ff % kBK || c->context_len <= 0 || c->d_model > kMaxRows) return false;
  return true;
}

static void launch_rows_packed(int ct, int grid, hipStream_t s, const GemmArgs& g) {
  switch (ct) {
    case 8: hipLaunchKernelGGL((mx_gemm_rows<1, 8, 3, 4, 1, false, kEpiStore>), dim3(grid), dim3(256), 0, s, g); break;
    case 6: hipLaunchKernelGGL((mx_gemm_rows<1, 6, 3, 4, 1, false, kEpiStore>), dim3(grid), dim3(256), 0, s, g); break;
    case 4: hipLaunchKernelGGL((mx_gemm_rows<1, 4, 4, 4, 1, false, kEpiStore>), dim3(grid), dim3(256), 0, s, g); break;
    case 3: hipLaunchKernelGGL((mx_gemm_rows<1, 3, 4, 4, 1, false, kEpiStore>), dim3(grid), dim3(256), 0, s, g); break;
    case 2: hipLaunchKernelGGL((mx_gemm_rows<1, 2, 4, 4, 1, false, kEpiStore>), dim3(grid), dim3(256), 0, s, g); break;
    default: hipLaunchKernelGGL((mx_gemm_rows<1, 1, 4, 4, 1, false, kEpiStore>), dim3(grid), dim3(256), 0, s, g); break;
  }
}

// K steps in flight per wave: 4 while the tile leaves the registers for it (single residual tiles of 4
// waves: 8, all of a 1024-wide projection; more gained nothing elsewhere)
template <int AM, int EPI, int I = 0>
static void launch_rows_tiles(const RowsTile& t, int grid, hipStream_t s, const GemmArgs& g, bool nt) {
  constexpr RowsTile k = kRowsTiles[I];
  if (t.rt == k.rt && t.ct == k.ct && t.nw == k.nw) {
    constexpr int P = k.rt * k.ct == 1 && k.nw == 4 && EPI == kEpiResid ? 8 : k.rt == 1 && k.ct <= 4 ? 4 : (k.rt * k.ct <= 6 ? 3 : 2);
    // (the tiles that passes of up to kStreamRows rows take have a non-temporal form)
    constexpr bool kNt = EPI == kEpiSwiglu ? k.rt <= 2 : k.rt == 1 && k.ct <= (EPI == kEpiQkv ? 3 : 1);
    if constexpr (kNt) {
      if (nt) {
        hipLaunchKernelGGL((mx_gemm_rows<k.rt, k.ct, P, k.nw, AM, true, EPI, true>), dim3(grid), dim3(64 * k.nw), 0, s, g);
        return;
      }
    }
    hipLaunchKernelGGL((mx_gemm_rows<k.rt, k.ct, P, k.nw, AM, true, EPI>), dim3(grid), dim3(64 * k.nw), 0, s, g);
  } else if constexpr (I + 1 < int(sizeof(kRowsTiles) / sizeof(kRowsTiles[0]))) {
    launch_rows_tiles<AM, EPI, I + 1>(t, grid, s, g, nt);
  }
}

template <bool TA>
static void launch_splitk(int bm, dim3 grid, hipStream_t s, const GemmArgs& g) {
  if (bm == 16) hipLaunchKernelGGL((mx_gemm<1, 1, TA>), grid, dim3(256), 0, s, g);
  else if (bm == 64) hipLaunchKernelGGL((mx_gemm<2, 2, TA>), grid, dim3(256), 0, s, g);
  else hipLaunchKernelGGL((mx_gemm<4, 2, TA>), grid, dim3(256), 0, s, g);
}

// C = A W^T split over K: partials [splits][M][N] (pass ldo = N), or with splits == 1 rows
// of stride ldo.  lda == 0: A in tile order (act_index); tw: W in tile order (msd_pack_tiles).
// ssq: A is the scale * h planes of an RMSNorm folded into mx_gemm_rows, whose rms comes from the
// nssq partial sums of h^2 per row in ssq.  epi / ea: the epilogue of mx_gemm_rows (tile-order
// weights only).
// rows_ok: mx_gemm_rows may run (single split only).  The tied logits pass false: one row and
// every row then come from the same kernel and summation order, so the last row's logits are
// bitwise the same either way.
static hipError_t gemm(const uint16_t* A, int64_t a_plane, int lda, const uint16_t* W, bool tw, int M, int N, int K,
                       float* out, int ldo, int splits, hipStream_t s, bool rows_ok = true, int epi = kEpiStore,
                       const EpiArgs* ea = nullptr, const float* ssq = nullptr, int nssq = 0,
                       bool nt = false) {
  GemmArgs g{A, a_plane, W, out, M, N, K, lda, ldo, splits, ea ? *ea : EpiArgs{}, ssq, nssq};
  const int am = ssq ? 2 : (lda == 0 ? 1 : 0);
  if ((epi != kEpiStore) != tw || (epi != kEpiStore && (!ea || am == 0 || splits != 1)))
    return hipErrorInvalidValue;
  if (am == 2 && (lda != 0 || nssq < 1 || nssq > kMaxGroups || !tw)) return hipErrorInvalidValue;
  const int T = (M + 15) / 16;
  if (tw) {
    const RowsTile t = rows_tile(M, N, K, epi == kEpiResid ? kMaxGroups : 0);
    const int grid = ((T + t.rt - 1) / t.rt) * ((N / 16 + t.ct - 1) / t.ct);
    if (am == 2 && epi == kEpiQkv) launch_rows_tiles<2, kEpiQkv>(t, grid, s, g, nt);
    else if (am == 2 && epi == kEpiSwiglu) launch_rows_tiles<2, kEpiSwiglu>(t, grid, s, g, nt);
    else if (am == 1 && epi == kEpiResid) launch_rows_tiles<1, kEpiResid>(t, grid, s, g, nt);
    else return hipErrorInvalidValue;
    return hipGetLastError();
  }
  if (const int ct = splits == 1 && rows_ok && am == 1 ? rows_ct(M, N, K) : 0; ct > 0) {
    launch_rows_packed(ct, T * (N / (16 * ct)), s, g);
    return hipGetLastError();
  }
  const int bm = bm_for(M);
  const dim3 grid(N / kBN, (M + bm - 1) / bm, splits);
  if (am == 1) launch_splitk<true>(bm, grid, s, g);
  else launch_splitk<false>(bm, grid, s, g);
  return hipGetLastError();
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Tied logits of M rows (planes [M][K], the lo plane M K further).  One row: mx_gemm (15.4 us for the
// 306M's; its weight rows come straight to the registers), which 5 rows already make slower (17.8).
static hipError_t launch_logits(const uint16_t* x, const uint16_t* W, int M, int V, int K, float* out, hipStream_t s) {
  const int64_t plane = int64_t(M) * K;
  const int nv = (V + kLogitRows - 1) / kLogitRows;
  if (M == 1 || !aligned16(out)) return gemm(x, plane, K, W, false, M, V, K, out, V, 1, s, false);
  if (M <= 32) hipLaunchKernelGGL(mx_logits<32>, dim3(nv), dim3(256), 0, s, x, plane, W, M, V, K, out);
  else if (M <= 64) hipLaunchKernelGGL(mx_logits<64>, dim3(nv), dim3(256), 0, s, x, plane, W, M, V, K, out);
  else hipLaunchKernelGGL(mx_logits<128>, dim3(nv * ((M + 127) / 128)), dim3(256), 0, s, x, plane, W, M, V, K, out);
  return hipGetLastError();
}

struct Weights {
  const uint16_t* emb;
  const uint16_t* outp;
  const uint16_t* w;
  const uint16_t* lnf;
  const float* rope;
  const uint16_t* tiles;   // the projections in tile order (msd_pack_tiles), or NULL
};

// Elements of one layer in the tile copy: QKV, O, gate/up, down, each N x K in tile order (the
// O and down rows permuted so that their outputs come in packed order), then the two RMSNorm
// scales in packed order; layer after layer.
static int64_t tile_layer_elems(const msd_config* c) {
  const int64_t d = c->d_model, ff = c->d_ff, nqkv = int64_t(c->n_heads + 2 * c->n_kv_heads) * kDh;
  return nqkv * d + d * d + 2 * ff * d + d * ff + 2 * d;
}

// Element offset of the first layer's packed RMSNorm1 scales in the tile copy.
static int64_t first_norm_scales(const msd_config* c) {
  const int64_t d = c->d_model, ff = c->d_ff, nqkv = int64_t(c->n_heads + 2 * c->n_kv_heads) * kDh;
  return nqkv * d + d * d + 2 * ff * d + d * ff;
}

// Weights that do not fit the 256 MB last-level cache (tile copies past kCacheBytes) are split: the first
// layers, up to kKeepBytes, are read with the default policy and stay there until the next pass, the
// others non-temporal, so they stream past.  That gains between passes that follow each other (chunks
// of a prompt, drafts and their verification) and nothing after a decode step, which streams its own
// copy of the weights.  Measured at 306M (541 MB; default policy / split, passes in a row and each after
// a decode step): verification of 5 tokens 664 / 603 and 670 / 668 us, prefill of 16 691 / 641 and
// 706 / 705, of 64 739 / 695 and 754 / 758, but of 128 870 / 841 and 879 / 908: at more rows a weight tile
// serves more row tiles' workgroups, and its lines leave the L2 before the last has read them (200 rows
// in a row 1124 / 1182).  So kStreamRows is the largest that loses nothing in either order.
// A batched step keeps the default policy: its own K/V rows want the cache, and the host does not know the
// positions (9 sequences of up to 40 positions 709 / 653 us, but 24 of up to 384 751 / 756, 48 926 / 952).
constexpr int64_t kKeepBytes = int64_t(150) << 20, kCacheBytes = int64_t(224) << 20;
constexpr int kStreamRows = 64;

// The layer stack over M rows whose residual stream is already in h; leaves the last
// projection's partials pending (returned split count).
static int run_layers(const msd_config* cfg, const Weights& wt, const Rows& rows, uint16_t* kv, const Layout& L,
                      char* ws, bool prefill, hipStream_t s, hipError_t& err) {
  const int M = rows.M, d = cfg->d_model, ff = cfg->d_ff, H = cfg->n_heads, KV = cfg->n_kv_heads;
  const int nqkv = (H + 2 * KV) * kDh;
  float* h = reinterpret_cast<float*>(ws + L.h);
  uint16_t* xn = reinterpret_cast<uint16_t*>(ws + L.xn);
  float* qkv = reinterpret_cast<float*>(ws + L.qkv);
  uint16_t* kvp = reinterpret_cast<uint16_t*>(ws + L.kvp);
  const int MP = pad32(M);
  uint16_t* att = reinterpret_cast<uint16_t*>(ws + L.att);
  uint16_t* act = reinterpret_cast<uint16_t*>(ws + L.act);
  float* part = reinterpret_cast<float*>(ws + L.part);
  float* ssq = reinterpret_cast<float*>(ws + L.ssq);
  const int64_t off_ln2 = d, off_qkv = 2 * int64_t(d), off_o = off_qkv + int64_t(nqkv) * d,
                off_gu = off_o + int64_t(d) * d, off_dn = off_gu + 2 * int64_t(ff) * d,
                layer = off_dn + int64_t(d) * ff;
  const int bm = bm_for(M);
  const bool tw = wt.tiles != nullptr;
  const int sq = splits_for(M, nqkv, d, bm, tw), so = splits_for(M, d, d, bm, tw),
            sg = splits_for(M, 2 * ff, d, bm, tw), sd = splits_for(M, d, ff, bm, tw);
  // the tile copy's per-layer offsets
  const int64_t toff_o = int64_t(nqkv) * d, toff_gu = toff_o + int64_t(d) * d, toff_dn = toff_gu + 2 * int64_t(ff) * d,
                toff_sc = toff_dn + int64_t(d) * ff;
  // partial sums of h^2 per row that the O and down epilogues leave (one per column group); the
  // first layer's come from mx_embed (one per row)
  const int cg_o = tw ? resid_groups(M, d, d) : 0, cg_d = tw ? resid_groups(M, d, ff) : 0;
  int pending = 0;
  err = hipSuccess;
  for (int l = 0; l < cfg->n_layers && err == hipSuccess; ++l) {
    const uint16_t* Wl = wt.w + int64_t(l) * layer;
    uint16_t* kc = kv + int64_t(l) * 2 * KV * rows.pool * kDh;
    uint16_t* vc = kc + int64_t(KV) * rows.pool * kDh;
    // activation planes in tile order (ldx 0), the lo planes after the hi planes
    const int64_t pd = int64_t(pad16(M)) * d, pf = int64_t(pad16(M)) * ff;
    EpiArgs eq{};
    eq.rope = wt.rope;
    eq.rows = rows;
    eq.kc = kc;
    eq.vc = vc;
    eq.qkv = qkv;
    eq.H = H;
    eq.KV = KV;
    eq.kvp = prefill ? kvp : nullptr;
    eq.MP = MP;
    if (tw) {
      // Five kernels per layer over the tile copy, h in packed order: QKV with RMSNorm1 folded in
      // and q/k/v, RoPE and the cache rows in its epilogue; attention; O adding to h and writing
      // RMSNorm2's input planes; gate/up with RMSNorm2 folded in and SwiGLU in its epilogue; down
      // adding to h and writing the next layer's RMSNorm1 input planes.
      const uint16_t* Tl = wt.tiles + int64_t(l) * tile_layer_elems(cfg);
      const bool last = l + 1 == cfg->n_layers;
      const int64_t bytes = 2 * tile_layer_elems(cfg);
      const bool nt = M <= kStreamRows && !rows.batched && cfg->n_layers * bytes > kCacheBytes && (l + 1) * bytes > kKeepBytes;
      if ((err = gemm(xn, pd, 0, Tl, true, M, nqkv, d, nullptr, 0, 1, s, true, kEpiQkv, &eq, ssq, l == 0 ? 1 : cg_d,
                      nt)) !=
          hipSuccess)
        break;
      if (prefill)
        launch_attention_prefill(M, H, KV, s, qkv, kvp, MP, att, pd, 1);
      else
        launch_attention_decode(M, H, KV, s, qkv, rows, kc, vc, att, pd, 1);
      EpiArgs en{};   // the next RMSNorm's input planes and partial sums of h^2
      en.act = xn;
      en.act_plane = pd;
      en.ssq = ssq;
      en.xscale = Tl + toff_sc + d;
      if ((err = gemm(att, pd, 0, Tl + toff_o, true, M, d, d, h, d, 1, s, true, kEpiResid, &en, nullptr, 0,
                      nt)) != hipSuccess)
        break;
      EpiArgs eg{};
      eg.act = act;
      eg.act_plane = pf;
      if ((err = gemm(xn, pd, 0, Tl + toff_gu, true, M, 2 * ff, d, nullptr, 0, 1, s, true, kEpiSwiglu, &eg, ssq, cg_o,
                      nt)) !=
          hipSuccess)
        break;
      if (last) en.act = nullptr;   // (the final norm reads h)
      else en.xscale = Tl + tile_layer_elems(cfg) + toff_sc;   // the next layer's RMSNorm1
      if ((err = gemm(act, pf, 0, Tl + toff_dn, true, M, d, ff, h, d, 1, s, true, kEpiResid, &en, nullptr, 0,
                      nt)) != hipSuccess)
        break;
      continue;
    }
    hipLaunchKernelGGL(mx_norm, dim3(M), dim3(kNormThreads), 0, s, h, part, pending, M, d, Wl, xn, pd, 0, 0, 0);
    if ((err = gemm(xn, pd, 0, Wl + off_qkv, false, M, nqkv, d, part, nqkv, sq, s)) != hipSuccess) break;
    hipLaunchKernelGGL(mx_qkv_fin, dim3(M, (nqkv / 4 + 255) / 256), dim3(256), 0, s, part, sq, M, eq);
    if (prefill)
      launch_attention_prefill(M, H, KV, s, qkv, kvp, MP, att, pd, 0);
    else
      launch_attention_decode(M, H, KV, s, qkv, rows, kc, vc, att, pd, 0);
    if ((err = gemm(att, pd, 0, Wl + off_o, false, M, d, d, part, d, so, s)) != hipSuccess) break;
    hipLaunchKernelGGL(mx_norm, dim3(M), dim3(kNormThreads), 0, s, h, part, so, M, d, Wl + off_ln2, xn, pd, 0, 0, 0);
    if ((err = gemm(xn, pd, 0, Wl + off_gu, false, M, 2 * ff, d, part, 2 * ff, sg, s)) != hipSuccess) break;
    hipLaunchKernelGGL(mx_swiglu_fin, dim3(M, (ff / 2 + 255) / 256), dim3(256), 0, s, part, sg, M, ff, act, pf);
    if ((err = gemm(act, pf, 0, Wl + off_dn, false, M, d, ff, part, d, sd, s)) != hipSuccess) break;
    pending = sd;
  }
  if (err == hipSuccess) err = hipGetLastError();
  return pending;
}

// ---- Replaying a pass's launches from a graph (opt-in) ----
// A pass is ~125 dependent launches; enqueueing them costs the host ~0.32 ms per pass (306M),
// replaying them from a graph ~0.09 ms.  The device runs the replay ~1 % slower (128-token
// prefill 0.872 vs 0.863 ms; 64 tokens 0.703 vs 0.694, 16 0.651 vs 0.642), so graphs are for callers
// whose host thread is the bottleneck and are off unless asked for (msd_set_launch_graphs, or
// MSD_LAUNCH_GRAPHS=1 in the environment).  The key holds every value a launch bakes in (shape, device pointers, sizes); buffer
// contents are read when the kernels run, so a replay with new tokens or weights in the same
// buffers is exact.  Captured on a private stream of the device (capture runs nothing) and launched
// on the caller's stream; a stream that is itself being captured gets the launches directly.
constexpr size_t kGraphCache = 16;   // graphs kept per process (least recently used is dropped)

struct GraphEntry {
  std::vector<char> key;
  int dev;
  hipGraphExec_t exec;
  hipEvent_t done;   // recorded after the latest replay: waited for before the graph is dropped
  uint64_t used;
};

static std::atomic<int> g_use_graphs{-1};   // -1: not read yet (MSD_LAUNCH_GRAPHS=1 switches them on)

static bool graphs_on() {
  int v = g_use_graphs.load();
  if (v < 0) {
    const char* e = std::getenv("MSD_LAUNCH_GRAPHS");
    int want = e && e[0] == '1' ? 1 : 0;
    g_use_graphs.compare_exchange_strong(v, want);
    v = g_use_graphs.load();
  }
  return v != 0;
}

struct KeyBuf {
  std::vector<char> b;
  template <class T>
  KeyBuf& add(const T& v) {
    const char* p = reinterpret_cast<const char*>(&v);
    b.insert(b.end(), p, p + sizeof(T));
    return *this;
  }
  KeyBuf& cfg(const msd_config* c) {
    return add(c->vocab_size).add(c->d_model).add(c->n_heads).add(c->n_kv_heads).add(c->n_layers).add(c->d_head)
        .add(c->d_ff).add(c->context_len);
  }
};

template <class F>
static int32_t launch_graphed(const std::vector<char>& key, hipStream_t s, F&& body) {
  if (!graphs_on()) return body(s);
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &cs) != hipSuccess) return MSD_E_HIP;
  if (cs != hipStreamCaptureStatusNone) return body(s);
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return MSD_E_HIP;
  static std::mutex mu;
  static std::vector<GraphEntry> cache;
  static std::vector<hipStream_t> capture_streams;
  static uint64_t tick = 0;
  std::lock_guard<std::mutex> lock(mu);
  GraphEntry* e = nullptr;
  for (GraphEntry& c : cache)
    if (c.dev == dev && c.key == key) e = &c;
  if (!e) {
    if (int(capture_streams.size()) <= dev) capture_streams.resize(dev + 1, nullptr);
    if (!capture_streams[dev] && hipStreamCreateWithFlags(&capture_streams[dev], hipStreamNonBlocking) != hipSuccess)
      return MSD_E_HIP;
    hipStream_t cap = capture_streams[dev];
    if (hipStreamBeginCapture(cap, hipStreamCaptureModeRelaxed) != hipSuccess) return MSD_E_HIP;
    const int32_t rc = body(cap);
    hipGraph_t g = nullptr;
    const hipError_t ec = hipStreamEndCapture(cap, &g);
    if (rc != MSD_OK || ec != hipSuccess) {
      if (g) (void)hipGraphDestroy(g);
      (void)hipGetLastError();
      return rc != MSD_OK ? rc : MSD_E_HIP;
    }
    hipGraphExec_t ex = nullptr;
    const hipError_t ei = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (ei != hipSuccess) return MSD_E_HIP;
    hipEvent_t ev = nullptr;
    if (hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) {
      (void)hipGraphExecDestroy(ex);
      return MSD_E_HIP;
    }
    if (cache.size() >= kGraphCache) {
      auto lru = std::min_element(cache.begin(), cache.end(),
                                  [](const GraphEntry& a, const GraphEntry& b) { return a.used < b.used; });
      // cleanup of an evicted entry: its failures leave nothing to undo
      (void)hipEventSynchronize(lru->done);
      (void)hipGraphExecDestroy(lru->exec);
      (void)hipEventDestroy(lru->done);
      cache.erase(lru);
    }
    cache.push_back(GraphEntry{key, dev, ex, ev, 0});
    e = &cache.back();
  }
  e->used = ++tick;
  if (hipGraphLaunch(e->exec, s) != hipSuccess || hipEventRecord(e->done, s) != hipSuccess) return MSD_E_HIP;
  return MSD_OK;
}

}  // namespace mpf

using namespace mpf;

extern "C" int64_t msd_prefill_workspace_bytes(const msd_config* cfg, int32_t n_tokens) {
  if (!mx_config_ok(cfg)) return MSD_E_CONFIG;
  if (n_tokens <= 0 || n_tokens > cfg->context_len) return MSD_E_ARG;
  return workspace_bytes(cfg, n_tokens);
}

// The forward pass over tokens[0..n_tokens) at positions start..start+n_tokens-1.  With
// start == 0 this is the prompt prefill (causal attention within the pass, f32 keys and values
// of the pass, model.py:194-231).  With start > 0 it is the verification of draft tokens over an
// existing cache: every row attends like a decode step at its position (cached rows 0..p-1 as
// stored bf16, including the draft rows this pass has just written, and its own un-rounded K/V,
// multi_sm_decode.py:182-221), so row i's logits are those the sequential decode steps would
// give after accepting rows 0..i-1.  argmax_all (optional) receives every row's
// (argmax, status) pair.
static int32_t prefill_impl(const msd_config* cfg, const Weights& wt, const int32_t* tokens, int32_t n_tokens,
                            int32_t start, const int32_t* page_table, int32_t max_pages, int32_t pool_pages,
                            void* kv, void* workspace, float* logits_last, float* logits_all, int32_t* next_token,
                            int32_t* argmax_all, hipStream_t s) {
  if (!mx_config_ok(cfg)) return MSD_E_CONFIG;
  const int M = n_tokens;
  if (M <= 0 || start < 0 || start + M > cfg->context_len) return MSD_E_ARG;
  if (start > 0 && cfg->context_len > kDecodeMaxCtx) return MSD_E_CONFIG;
  if (argmax_all && !logits_all) return MSD_E_ARG;
  if (!wt.emb || !wt.outp || !wt.w || !wt.lnf || !wt.rope || !tokens || !kv || !workspace || !logits_last ||
      !next_token)
    return MSD_E_ARG;
  if (!aligned16(wt.emb) || !aligned16(wt.outp) || !aligned16(wt.w) || !aligned16(kv) || !aligned16(workspace) ||
      !aligned16(wt.tiles))
    return MSD_E_ARG;
  if (page_table && (max_pages * kPage < start + M || max_pages > (cfg->context_len + kPage - 1) / kPage ||
                     pool_pages <= 0))
    return MSD_E_ARG;
  KeyBuf key;
  key.add('p').cfg(cfg).add(wt).add(tokens).add(M).add(start).add(page_table).add(max_pages).add(pool_pages).add(kv)
      .add(workspace).add(logits_last).add(logits_all).add(next_token).add(argmax_all);
  return launch_graphed(key.b, s, [&](hipStream_t s) -> int32_t {
  const int d = cfg->d_model, V = cfg->vocab_size;
  const Layout L = layout(cfg, M);
  char* ws = static_cast<char*>(workspace);
  float* h = reinterpret_cast<float*>(ws + L.h);
  uint16_t* xn = reinterpret_cast<uint16_t*>(ws + L.xn);
  float* part = reinterpret_cast<float*>(ws + L.part);
  int32_t* status = reinterpret_cast<int32_t*>(ws + L.status);
  int32_t* pages = reinterpret_cast<int32_t*>(ws + L.pages);
  if (page_table)
    hipLaunchKernelGGL(mx_sanitize_rows, dim3(1), dim3(64), 0, s, nullptr, start + M - 1, page_table, 1, max_pages,
                       cfg->context_len, pool_pages, nullptr, pages, status + M);
  Rows rows{M, nullptr, 0, page_table ? pages : nullptr, max_pages, page_table ? pool_pages * kPage : cfg->context_len,
            start};
  const int packed = wt.tiles != nullptr;   // the tile path keeps h in packed order
  // with the tile copy also the first layer's RMSNorm1 input planes and sums of h^2
  hipLaunchKernelGGL(mx_embed, dim3(M), dim3(256), 0, s, wt.emb, tokens, d, h, status, V, packed,
                     packed ? wt.tiles + first_norm_scales(cfg) : nullptr, xn, int64_t(pad16(M)) * d,
                     reinterpret_cast<float*>(ws + L.ssq));
  hipError_t err;
  const int pending = run_layers(cfg, wt, rows, static_cast<uint16_t*>(kv), L, ws, start == 0, s, err);
  if (err != hipSuccess) return MSD_E_HIP;
  // final norm of the rows whose logits are wanted, then the tied output projection
  const int r0 = logits_all ? 0 : M - 1, nr = M - r0;
  hipLaunchKernelGGL(mx_norm, dim3(nr), dim3(kNormThreads), 0, s, h, part, pending, M, d, wt.lnf, xn,
                     int64_t(nr) * d, r0, d, packed);
  if (launch_logits(xn, wt.outp, nr, V, d, logits_all ? logits_all : logits_last, s) != hipSuccess) return MSD_E_HIP;
  const float* last = logits_all ? logits_all + int64_t(M - 1) * V : logits_last;
  const int nflags = M + (page_table ? 1 : 0);
  if (argmax_all)   // every row (next_token points at the last row's pair)
    hipLaunchKernelGGL(mx_argmax, dim3(M), dim3(1024), 0, s, logits_all, V, V, argmax_all, status, nflags, nullptr);
  if (!argmax_all || last != logits_last)
    hipLaunchKernelGGL(mx_argmax, dim3(1), dim3(1024), 0, s, last, V, V, next_token, status, nflags,
                       last != logits_last ? logits_last : nullptr);
  return hipGetLastError() == hipSuccess ? MSD_OK : MSD_E_HIP;
  });
}

extern "C" int64_t msd_tiles_bytes(const msd_config* cfg) {
  if (!mx_config_ok(cfg)) return MSD_E_CONFIG;
  return tile_layer_elems(cfg) * cfg->n_layers * 2;
}

extern "C" int32_t msd_pack_tiles(const msd_config* cfg, const void* packed_w, void* tiles, void* stream) {
  if (!mx_config_ok(cfg)) return MSD_E_CONFIG;
  if (!packed_w || !tiles || !aligned16(packed_w) || !aligned16(tiles)) return MSD_E_ARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int d = cfg->d_model, ff = cfg->d_ff, nqkv = (cfg->n_heads + 2 * cfg->n_kv_heads) * kDh;
  const int64_t off_qkv = 2 * int64_t(d), off_o = off_qkv + int64_t(nqkv) * d, off_gu = off_o + int64_t(d) * d,
                off_dn = off_gu + 2 * int64_t(ff) * d, layer = off_dn + int64_t(d) * ff;
  const int64_t dst_o = int64_t(nqkv) * d, dst_gu = dst_o + int64_t(d) * d, dst_dn = dst_gu + 2 * int64_t(ff) * d,
                dst_sc = dst_dn + int64_t(d) * ff;
  const struct { int64_t src, dst; int N, K, rowperm, natk; } mats[4] = {
      {off_qkv, 0, nqkv, d, 0, 0}, {off_o, dst_o, d, d, 1, 1}, {off_gu, dst_gu, 2 * ff, d, 2, 0},
      {off_dn, dst_dn, d, ff, 1, 0}};
  const uint16_t* w = static_cast<const uint16_t*>(packed_w);
  uint16_t* t = static_cast<uint16_t*>(tiles);
  for (int l = 0; l < cfg->n_layers; ++l) {
    uint16_t* tl = t + l * tile_layer_elems(cfg);
    for (const auto& m : mats) {
      const int64_t pieces = int64_t(m.N) * m.K / 8;
      hipLaunchKernelGGL(mx_pack_tiles, dim3(unsigned((pieces + 255) / 256)), dim3(256), 0, s, w + l * layer + m.src,
                         m.N, m.K, m.rowperm, m.natk, tl + m.dst);
    }
    hipLaunchKernelGGL(mx_pack_scales, dim3((2 * d + 255) / 256), dim3(256), 0, s, w + l * layer, d, tl + dst_sc);
  }
  return hipGetLastError() == hipSuccess ? MSD_OK : MSD_E_HIP;
}

extern "C" int32_t msd_prefill(const msd_config* cfg, const void* token_emb, const void* output_proj,
                               const void* packed_w, const void* tiles, const void* lnf_s, const float* rope,
                               const int32_t* tokens, int32_t n_tokens, void* kv, void* workspace, float* logits_last,
                               float* logits_all, int32_t* next_token, void* stream) {
  const Weights wt{static_cast<const uint16_t*>(token_emb), static_cast<const uint16_t*>(output_proj),
                   static_cast<const uint16_t*>(packed_w), static_cast<const uint16_t*>(lnf_s), rope,
                   static_cast<const uint16_t*>(tiles)};
  return prefill_impl(cfg, wt, tokens, n_tokens, 0, nullptr, 0, 0, kv, workspace, logits_last, logits_all, next_token,
                      nullptr, static_cast<hipStream_t>(stream));
}

extern "C" int32_t msd_prefill_paged(const msd_config* cfg, const void* token_emb, const void* output_proj,
                                     const void* packed_w, const void* tiles, const void* lnf_s, const float* rope,
                                     const int32_t* tokens, int32_t n_tokens, const int32_t* page_table,
                                     int32_t max_pages, void* kv_pool, int32_t pool_pages, void* workspace,
                                     float* logits_last, int32_t* next_token, void* stream) {
  if (!page_table) return MSD_E_ARG;
  const Weights wt{static_cast<const uint16_t*>(token_emb), static_cast<const uint16_t*>(output_proj),
                   static_cast<const uint16_t*>(packed_w), static_cast<const uint16_t*>(lnf_s), rope,
                   static_cast<const uint16_t*>(tiles)};
  return prefill_impl(cfg, wt, tokens, n_tokens, 0, page_table, max_pages, pool_pages, kv_pool, workspace, logits_last,
                      nullptr, next_token, nullptr, static_cast<hipStream_t>(stream));
}

extern "C" int64_t msd_verify_workspace_bytes(const msd_config* cfg, int32_t n_tokens) {
  return msd_prefill_workspace_bytes(cfg, n_tokens);
}

extern "C" int32_t msd_verify(const msd_config* cfg, const void* token_emb, const void* output_proj,
                              const void* packed_w, const void* tiles, const void* lnf_s, const float* rope,
                              const int32_t* tokens, int32_t n_tokens, int32_t start_pos, void* kv, void* workspace,
                              float* logits, int32_t* argmax, void* stream) {
  if (!cfg || !logits || !argmax || n_tokens <= 0 || start_pos < 1) return MSD_E_ARG;
  const Weights wt{static_cast<const uint16_t*>(token_emb), static_cast<const uint16_t*>(output_proj),
                   static_cast<const uint16_t*>(packed_w), static_cast<const uint16_t*>(lnf_s), rope,
                   static_cast<const uint16_t*>(tiles)};
  // the last row's logits land in logits (as part of logits_all); its argmax again in argmax[2(n-1)]
  return prefill_impl(cfg, wt, tokens, n_tokens, start_pos, nullptr, 0, 0, kv, workspace,
                      logits + int64_t(n_tokens - 1) * cfg->vocab_size, logits, argmax + 2 * (n_tokens - 1), argmax,
                      static_cast<hipStream_t>(stream));
}

// The batched workspace: the persistent step's region (fixed size per shape, first, so that
// its epoch and flags stay put whatever the batch), then the multi-kernel step's buffers.
static int64_t batch_region(const msd_config* cfg) { return (mbd::region_bytes(cfg) + 255) & ~int64_t(255); }

extern "C" int64_t msd_batch_workspace_bytes(const msd_config* cfg, int32_t batch) {
  if (!mx_config_ok(cfg)) return MSD_E_CONFIG;
  if (batch <= 0 || batch > kMaxRows) return MSD_E_ARG;
  return batch_region(cfg) + workspace_bytes(cfg, batch);
}

extern "C" int32_t msd_batch_decode_step(const msd_config* cfg, const void* token_emb, const void* output_proj,
                                         const void* packed_w, const void* tiles, const void* lnf_s, const float* rope,
                                         const int32_t* tokens, const int32_t* positions, int32_t batch,
                                         const int32_t* page_tables, int32_t max_pages, void* kv_pool,
                                         int32_t pool_pages, void* workspace, float* logits,
                                         int32_t* next_tokens, void* stream) {
  if (!mx_config_ok(cfg)) return MSD_E_CONFIG;
  const int M = batch;
  if (M <= 0 || M > kMaxRows) return MSD_E_ARG;
  if (!token_emb || !output_proj || !packed_w || !lnf_s || !rope || !tokens || !positions || !page_tables ||
      !kv_pool || !workspace || !logits || !next_tokens)
    return MSD_E_ARG;
  if (!aligned16(token_emb) || !aligned16(output_proj) || !aligned16(packed_w) || !aligned16(kv_pool) ||
      !aligned16(workspace) || !aligned16(tiles))
    return MSD_E_ARG;
  if (max_pages <= 0 || max_pages > (cfg->context_len + kPage - 1) / kPage || pool_pages <= 0) return MSD_E_ARG;
  if (cfg->context_len > kDecodeMaxCtx) return MSD_E_CONFIG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  {   // up to 8 sequences: one persistent launch when the shape and the device allow it
    const mbd::StepArgs sa{cfg, static_cast<const uint16_t*>(token_emb), static_cast<const uint16_t*>(output_proj),
                           static_cast<const uint16_t*>(packed_w), static_cast<const uint16_t*>(lnf_s), rope, tokens,
                           positions, batch, page_tables, max_pages, static_cast<uint16_t*>(kv_pool), pool_pages,
                           workspace, logits, next_tokens, s};
    const int32_t rc = mbd::try_step(sa);
    if (rc != 1) return rc;
  }
  const Weights wt{static_cast<const uint16_t*>(token_emb), static_cast<const uint16_t*>(output_proj),
                   static_cast<const uint16_t*>(packed_w), static_cast<const uint16_t*>(lnf_s), rope,
                   static_cast<const uint16_t*>(tiles)};
  KeyBuf key;
  key.add('b').cfg(cfg).add(wt).add(tokens).add(positions).add(M).add(page_tables).add(max_pages).add(kv_pool)
      .add(pool_pages).add(workspace).add(logits).add(next_tokens);
  return launch_graphed(key.b, s, [&](hipStream_t s) -> int32_t {
  const int d = cfg->d_model, V = cfg->vocab_size;
  const Layout L = layout(cfg, M);
  char* ws = static_cast<char*>(workspace) + batch_region(cfg);
  float* h = reinterpret_cast<float*>(ws + L.h);
  uint16_t* xn = reinterpret_cast<uint16_t*>(ws + L.xn);
  float* part = reinterpret_cast<float*>(ws + L.part);
  int32_t* status = reinterpret_cast<int32_t*>(ws + L.status);
  int32_t* rowpos = reinterpret_cast<int32_t*>(ws + L.rowpos);
  int32_t* pages = reinterpret_cast<int32_t*>(ws + L.pages);
  hipLaunchKernelGGL(mx_sanitize_rows, dim3((M + 255) / 256), dim3(256), 0, s, positions, 0, page_tables, M, max_pages,
                     cfg->context_len, pool_pages, rowpos, pages, status + M);
  Rows rows{M, rowpos, 1, pages, max_pages, pool_pages * kPage, 0};
  const int packed = wt.tiles != nullptr;
  // with the tile copy also the first layer's RMSNorm1 input planes and sums of h^2
  hipLaunchKernelGGL(mx_embed, dim3(M), dim3(256), 0, s, wt.emb, tokens, d, h, status, V, packed,
                     packed ? wt.tiles + first_norm_scales(cfg) : nullptr, xn, int64_t(pad16(M)) * d,
                     reinterpret_cast<float*>(ws + L.ssq));
  hipError_t err;
  const int pending = run_layers(cfg, wt, rows, static_cast<uint16_t*>(kv_pool), L, ws, false, s, err);
  if (err != hipSuccess) return MSD_E_HIP;
  hipLaunchKernelGGL(mx_norm, dim3(M), dim3(kNormThreads), 0, s, h, part, pending, M, d, wt.lnf, xn, int64_t(M) * d, 0,
                     d, packed);
  if (launch_logits(xn, wt.outp, M, V, d, logits, s) != hipSuccess) return MSD_E_HIP;
  hipLaunchKernelGGL(mx_argmax, dim3(M), dim3(1024), 0, s, logits, V, V, next_tokens, status, 2 * M, nullptr);
  return hipGetLastError() == hipSuccess ? MSD_OK : MSD_E_HIP;
  });
}

extern "C" int32_t msd_config_support(const msd_config* cfg, int32_t n_workgroups) {
  if (!cfg) return MSD_E_ARG;
  const int G = n_workgroups > 0 ? n_workgroups : 256;
  int32_t paths = 0;
  if (msdc::decode_supported(cfg, G)) paths |= MSD_PATH_DECODE;
  if (mx_config_ok(cfg)) {
    paths |= MSD_PATH_PREFILL;
    if (cfg->context_len <= kDecodeMaxCtx) paths |= MSD_PATH_VERIFY | MSD_PATH_BATCHED;
    if ((paths & MSD_PATH_BATCHED) && mbd::region_bytes(cfg) > 0) paths |= MSD_PATH_BATCHED_STEP;
  }
  if (msdc::sample_supported(cfg->vocab_size)) paths |= MSD_PATH_SAMPLE;
  return paths;
}

extern "C" int32_t msd_set_launch_graphs(int32_t enabled) {
  graphs_on();
  return g_use_graphs.exchange(enabled ? 1 : 0);
}
