// Fused output projection + cross-entropy, forward and backward, on the matrix cores (gfx950).
//
// Reference: model.py:279-379 -- _chunked_ce_fwd (chunked online logsumexp, :281-302),
// fused_cross_entropy (jax.custom_vjp, :305-312), _fused_ce_bwd (:320-361) and
// fused_output_and_loss (:367-379).  h (N, d) and weight (V, d) are bf16 (train.py:113 casts the
// parameters to bf16), targets int32 (N).  Every logit is a bf16 x bf16 dot product accumulated
// in f32 (v_mfma_f32_32x32x16_bf16); softmax statistics are f32.
//
// Forward (msd_xent_forward): one GEMM S^T = W h^T over the whole vocabulary whose epilogue never
// stores it: each 256 x 256 tile (256 vocabulary ids x 256 tokens) reduces its token columns to a
// partial (max, sum of exp(s - max)) and captures the target logits (the transposed product puts
// one token's 64 values per tile in each lane's registers, so the reduction stays in registers);
// xent_lse merges a token's partials in a fixed order (lse = max + log sum, the online logsumexp
// of :293-301), xent_mean takes the mean of lse - target logit in a fixed order (float64 sum).
// The logits never exist in memory, as in the reference, whose chunk loop materialises only one
// (N, chunk) block at a time.
//
// Backward (msd_xent_backward), per vocabulary chunk (the reference's chunk loop, :344-353; the
// chunk bounds the probability block, see plan()):
//   1. xent_gemm<kEpiProb>: S^T = W_c h^T, then P' = (exp(S - lse) - onehot(target)) * g / N as
//      bf16, stored token-major as P (N x C) through LDS staging;
//   2. xent_gemm<kEpiStoreBf16>: grad_W[c]^T = h^T P'  (the whole reduction over N rows, so
//      the chunk's rows of grad_W are final; stored transposed through LDS staging);
//   3. xent_gemm<kEpiPartF32>: grad_h += P' W_c, the chunk's K range split over enough workgroups to
//      fill the chip; each split adds to its own f32 partial across chunks, and xent_sum_parts adds
//      the partials in split order and rounds to bf16.
// The target terms (:356-358) ride in P' (its -1 at the target column), so grad_h = (softmax -
// onehot) W g/N and grad_W = (softmax - onehot)^T h g/N as in the reference.  The forward's lse
// is reused instead of recomputing the logsumexp (:331-340).  P, h and W are read as they lie:
// an operand whose rows run along K's other dimension (both of 2, W of 3) is staged K-major and
// transposed on the way from LDS to the registers (ds_read_b64_tr_b16), so no transposed copy of
// P, h or W is ever written.
//
// GEMM (xent_gemm<T, TRA, TRB, EPI>): C = A B^T.  A workgroup of 2 x 2 waves owns a T x T tile, T =
// 256 (128 x 128 per wave: 256 accumulators per lane, one wave per SIMD) or 128 (64 x 64 per wave,
// two workgroups per CU) where 256-tiles would leave CUs idle; each wave a block of 32 x 32 MFMA
// tiles.  What bounds it is LDS: per K = 32 stage a 256 tile costs 1,024 MFMA cycles per SIMD and,
// at 128 bytes a cycle, 512 cycles of fragment reads plus 256 of DMA writes (eight waves of
// 128 x 64 read 96 KB instead of 64 and just saturate it; a 128 tile needs 384 LDS cycles for 256
// of MFMA).  K advances 32 at a time through a ring of 4 LDS stages filled by direct DMA
// (global_load_lds, 16 bytes per lane); a wave reads the fragments of stage k + 1 while the matrix
// cores work on stage k, one barrier per stage.
// Measured (N 4096, V 32000, d 1024, one chunk; 268 GFLOP per product): forward 306 us (8 waves of 128 x 64,
// fragments read stage by stage: 329), probabilities 328 (8 chunks: 450 with P and P^T), grad_W
// 253 (128-tiles 304), grad_h 259 + 12 for the partials' sum (128-tiles 340); W^T and h^T are not
// copied.  Timing-only copies without the operand DMA or without
// the fragment reads take 207 us per gradient: what is left is the matrix cores at their
// sustained rate (a large library product: 1.21 PFLOP/s = 221 us) and the epilogues, which one
// workgroup per CU does not overlap.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <math.h>

#include <algorithm>

#include "../../include/msxent.h"
#include "internal.h"

namespace mxe {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));   // a native vector (HIP's uint4 is a struct)
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kStatusTarget = 4;  // a target id outside [0, V) (replaced by 0)

// round to nearest even (finite inputs; NaN stays NaN)
__device__ __forceinline__ uint16_t f2bf(float x) {
  const uint32_t u = __float_as_uint(x);
  if ((u & 0x7fffffffu) > 0x7f800000u) return uint16_t((u >> 16) | 0x40);
  return uint16_t((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

// two values as bf16 (round to nearest even, v_cvt_pk_bf16_f32), a in the low half
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
}

// exp(x) for x <= 0 (x = -inf gives 0): the hardware base-2 exponential of x log2(e)
__device__ __forceinline__ float exp_neg(float x) { return __builtin_amdgcn_exp2f(x * kLog2e); }

enum Epi { kEpiLse = 0, kEpiProb = 1, kEpiPartF32 = 2, kEpiStoreBf16 = 3 };

struct GemmArgs {
  const uint16_t* A;   // M x K, row stride lda (transposed: K x M, row stride lda)
  int64_t lda;
  int a_valid;         // rows of A in memory: a row past the last reads the last
  const uint16_t* B;   // Nn x K, row stride ldb (transposed: K x Nn)
  int64_t ldb;
  int b_valid;
  int a_cols, b_cols;       // transposed operands: elements per row in memory (multiples of 8)
  int K, k_split;           // multiples of 64: split z covers K range [z k_split, (z + 1) k_split)
  int tiles_m, tiles_n;     // output tiles; the grid is tiles_m * tiles_n * splits
  int m_valid, n_valid;     // output rows / columns that exist (the rest are padding)
  const int32_t* targets;   // kEpiLse, kEpiProb: target per token (output column)
  int vocab;                // kEpiLse, kEpiProb: targets outside [0, vocab) are taken as 0 and reported
  int32_t* status;
  int vcol0;                // kEpiProb: vocabulary index of output column 0
  const float* lse;         // kEpiProb: per token
  const float* grad;        // kEpiProb: the loss gradient g (device scalar)
  float inv_n;              // kEpiProb: 1 / N
  float* part;              // kEpiLse: (max, sum) per (vocabulary tile, token): [tiles_m][ldp][2]
  int64_t ldp;
  float* tgt;               // kEpiLse: target logit per token
  uint16_t* P;              // kEpiProb: tokens x ldP
  int64_t ldP;
  float* acc;               // kEpiPartF32: [splits][rows][ldacc] f32, splits acc_split apart
  int64_t ldacc, acc_split;
  int accumulate;           // kEpiPartF32: add to acc (else overwrite)
  uint16_t* out;            // kEpiStoreBf16: columns x ldout (the transpose of the tile)
  int64_t ldout;
};

constexpr int kKD = 32;       // K per LDS stage
constexpr int kStages = 4;    // LDS ring
constexpr int kWaves = 4;     // 2 x 2 waves per workgroup
template <int T>
constexpr int stage_bytes() { return 2 * T * kKD * 2; }
template <int T>
constexpr int staging_pitch() { return T + 8; }   // bf16 per row of the epilogue's LDS tile
template <int T, int EPI>
constexpr size_t lds_bytes() {
  constexpr size_t ring = size_t(kStages) * stage_bytes<T>();
  return EPI == kEpiProb || EPI == kEpiStoreBf16 ? std::max<size_t>(ring, size_t(T) * staging_pitch<T>() * 2 + T * 8) : ring;
}

// Tile (tm, tn) and split z of workgroup b.  Workgroup b runs on XCD b % 8, which takes a
// contiguous range of the tile ids (the ranges differ by at most one id); ids walk, split by split,
// blocks of 8 column tiles, row tile by row tile, so the 32 workgroups an XCD holds at a time
// cover 4 row tiles x 8 column tiles and share their operand rows in its L2.
__device__ __forceinline__ void tile_of(int b, int total, int tiles_m, int tiles_n, int& tm, int& tn, int& z) {
  const int x = b & 7, q = total >> 3, r = total & 7;
  int t = x * q + min(x, r) + (b >> 3);
  const int tiles = tiles_m * tiles_n;
  z = t / tiles;
  t -= z * tiles;
  const int blk = t / (8 * tiles_m), w = min(8, tiles_n - 8 * blk), rem = t - blk * 8 * tiles_m;
  tm = rem / w;
  tn = 8 * blk + rem % w;
}

// ---- LDS stages ----
// Plain operand (rows contiguous along K): a stage is T rows of 64 bytes (4 pieces of 8 K values);
// row r holds piece c at position c ^ ((r >> 2) & 3).  Measured with a probe of ds_read_b128
// address patterns (SQ_LDS_BANK_CONFLICT): the fragment read of 32 rows x one piece is
// conflict-free with this swizzle and takes twice the LDS cycles with c ^ ((r >> 1) & 3) or with
// no swizzle.
// Transposed operand (rows along K, contiguous in the tile's T columns): a stage is 32 rows of 2T
// bytes; row k holds the 32-byte unit u (16 columns) at position u ^ (2 (k & 3)), so the 8 units a
// half-wave's transposing read touches (4 rows x 2 units) lie in distinct banks.
// The fragment reads are inline assembly with explicit waits: the compiler would otherwise wait for
// every outstanding DMA (vmcnt(0)) before each LDS read, and __syncthreads' fence would too, so
// the stage barrier is a bare s_barrier after this wave's own DMAs of the stage have landed.
typedef __attribute__((address_space(3))) uint8_t lds_u8;
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return uint32_t(reinterpret_cast<uintptr_t>((const lds_u8*)p));
}
// (the host pass instantiates these templates along with the kernels but never emits them, and
// an x86 compile rejects the vector-register constraints and the LDS builtin, so their bodies
// are in the device pass only)
template <int N>
__device__ __forceinline__ void wait_vm() {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
#endif
}
// Wait until at most n (< D, wave-uniform) stages of NIW DMA instructions are outstanding.
template <int NIW, int D>
__device__ __forceinline__ void wait_stages(int n) {
  if constexpr (D > 1) {
    if (n >= D - 1) {
      wait_vm<(D - 1) * NIW>();
      return;
    }
    wait_stages<NIW, D - 1>(n);
  } else {
    wait_vm<0>();
  }
}

// One operand of a wave: NB fragments (32 rows each) per K step of 16, two steps per stage.  The
// MFMA operand of lane l is row l % 32, K values 8 (l / 32) .. + 8.
template <int T, int NB, bool TR>
struct Operand;

// reads issued here are waited for by wait_reads, whose "+v" operands tie the registers to the wait:
// no use or copy of a fragment can be placed before it
template <int T, int NB>
struct Operand<T, NB, false> {
  struct Frags {
    u32x4 f[2][NB];
  };
  uint32_t a[2];   // LDS byte offset of fragment 0 per K step
  __device__ __forceinline__ void init(uint32_t base, int row0, int lane) {
    const int fr = lane & 31, fh = lane >> 5;
    for (int ks = 0; ks < 2; ++ks) a[ks] = base + (row0 + fr) * 64 + (((2 * ks + fh) ^ ((fr >> 2) & 3)) << 4);
  }
  template <int KS>
  __device__ __forceinline__ void read(Frags& F, uint32_t st) const {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint32_t p = a[KS] + st;
    if constexpr (NB == 4)
      asm volatile(
          "ds_read_b128 %0, %4\n"
          "ds_read_b128 %1, %4 offset:2048\n"
          "ds_read_b128 %2, %4 offset:4096\n"
          "ds_read_b128 %3, %4 offset:6144"
          : "=&v"(F.f[KS][0]), "=&v"(F.f[KS][1]), "=&v"(F.f[KS][2]), "=&v"(F.f[KS][3])
          : "v"(p));
    else
      asm volatile(
          "ds_read_b128 %0, %2\n"
          "ds_read_b128 %1, %2 offset:2048"
          : "=&v"(F.f[KS][0]), "=&v"(F.f[KS][1])
          : "v"(p));
#endif
  }
  __device__ __forceinline__ static void wait(Frags& F) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (NB == 4)
      asm volatile("s_waitcnt lgkmcnt(0)"
                   : "+v"(F.f[0][0]), "+v"(F.f[0][1]), "+v"(F.f[0][2]), "+v"(F.f[0][3]), "+v"(F.f[1][0]),
                     "+v"(F.f[1][1]), "+v"(F.f[1][2]), "+v"(F.f[1][3]));
    else
      asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(F.f[0][0]), "+v"(F.f[0][1]), "+v"(F.f[1][0]), "+v"(F.f[1][1]));
#endif
  }
  template <int KS>
  __device__ __forceinline__ static bf16x8 get(const Frags& F, int i) {
    return __builtin_bit_cast(bf16x8, F.f[KS][i]);
  }
};

// ds_read_b64_tr_b16: the 16 lanes of a group read 4 K rows x 4 lanes x 4 columns (lane t: row
// t / 4, columns 4 (t % 4) ..), and lane t receives column t of the 4 rows.
template <int T, int NB>
struct Operand<T, NB, true> {
  struct Frags {
    u32x2 f[2][NB][2];   // K values 0..3 and 4..7 of the lane's eight
  };
  static constexpr int kRow = 2 * T;   // bytes per K row
  uint32_t a[NB];
  __device__ __forceinline__ void init(uint32_t base, int col0, int lane) {
    const int t = lane & 15, k = 8 * (lane >> 5) + (t >> 2);   // K row of the first read (k & 3 = t >> 2)
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int unit = (col0 >> 4) + 2 * i + ((lane >> 4) & 1);
      a[i] = base + k * kRow + ((unit ^ (2 * (t >> 2))) << 5) + 8 * (t & 3);
    }
  }
  template <int KS>
  __device__ __forceinline__ void read(Frags& F, uint32_t st) const {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int i = 0; i < NB; ++i)
      asm volatile(
          "ds_read_b64_tr_b16 %0, %2 offset:%3\n"
          "ds_read_b64_tr_b16 %1, %2 offset:%4"
          : "=&v"(F.f[KS][i][0]), "=&v"(F.f[KS][i][1])
          : "v"(a[i] + st), "n"(16 * KS * kRow), "n"(16 * KS * kRow + 4 * kRow));
#endif
  }
  __device__ __forceinline__ static void wait(Frags& F) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (NB == 4)
      asm volatile("s_waitcnt lgkmcnt(0)"
                   : "+v"(F.f[0][0][0]), "+v"(F.f[0][0][1]), "+v"(F.f[0][1][0]), "+v"(F.f[0][1][1]), "+v"(F.f[0][2][0]),
                     "+v"(F.f[0][2][1]), "+v"(F.f[0][3][0]), "+v"(F.f[0][3][1]), "+v"(F.f[1][0][0]), "+v"(F.f[1][0][1]),
                     "+v"(F.f[1][1][0]), "+v"(F.f[1][1][1]), "+v"(F.f[1][2][0]), "+v"(F.f[1][2][1]), "+v"(F.f[1][3][0]),
                     "+v"(F.f[1][3][1]));
    else
      asm volatile("s_waitcnt lgkmcnt(0)"
                   : "+v"(F.f[0][0][0]), "+v"(F.f[0][0][1]), "+v"(F.f[0][1][0]), "+v"(F.f[0][1][1]), "+v"(F.f[1][0][0]),
                     "+v"(F.f[1][0][1]), "+v"(F.f[1][1][0]), "+v"(F.f[1][1][1]));
#endif
  }
  template <int KS>
  __device__ __forceinline__ static bf16x8 get(const Frags& F, int i) {
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(F.f[KS][i][0], F.f[KS][i][1], 0, 1, 2, 3));
  }
};

// This wave's DMAs of one operand's stage: instruction u fills the 1 KB at dst + 1024 (wv + 4 u).
template <int T, bool TR>
struct Loader {
  static constexpr int NI = T * kKD * 2 / 1024 / kWaves;   // instructions per wave and stage
  const uint16_t* src;
  uint32_t off[NI];   // plain: element offset of stage 0; transposed: column of the piece
  uint32_t ld;
  int kr[NI], kmax;   // transposed: K row within the stage, last K row in memory
  __device__ __forceinline__ void init(const uint16_t* p, int64_t ldp, int valid, int cols, int row0, int k0, int lane,
                                       int wv) {
    ld = uint32_t(ldp);
    if constexpr (TR) {
      constexpr int LPR = T / 8;   // lanes (16-byte pieces) per K row
      src = p + int64_t(k0) * ldp;
      kmax = valid - 1 - k0;
#pragma unroll
      for (int u = 0; u < NI; ++u) {
        const int piece = 64 * (wv + kWaves * u) + lane;
        kr[u] = piece / LPR;
        const int pos = piece % LPR;
        const int c = 16 * ((pos >> 1) ^ (2 * (kr[u] & 3))) + 8 * (pos & 1);
        off[u] = uint32_t(min(row0 + c, cols - 8));   // columns past the last are padding outputs
      }
    } else {
      src = p + k0;
#pragma unroll
      for (int u = 0; u < NI; ++u) {
        const int r = 16 * (wv + kWaves * u) + (lane >> 2);
        off[u] = uint32_t(min(row0 + r, valid - 1)) * ld + 8 * ((lane & 3) ^ ((r >> 2) & 3));
      }
    }
  }
  __device__ __forceinline__ void stage(int kt, uint8_t* dst, int wv) const {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (TR) {
#pragma unroll
      for (int u = 0; u < NI; ++u) {
        const uint32_t o = uint32_t(min(kt * kKD + kr[u], kmax)) * ld + off[u];
        __builtin_amdgcn_global_load_lds(src + o, (__attribute__((address_space(3))) void*)(dst + 1024 * (wv + kWaves * u)),
                                         16, 0, 0);
      }
    } else {
#pragma unroll
      for (int u = 0; u < NI; ++u)
        __builtin_amdgcn_global_load_lds(src + (off[u] + kt * kKD),
                                         (__attribute__((address_space(3))) void*)(dst + 1024 * (wv + kWaves * u)), 16, 0,
                                         0);
    }
#endif
  }
};

// target of a token, an id outside the vocabulary replaced by 0 (and reported by one row of tiles)
__device__ __forceinline__ int target_of(const GemmArgs& g, int tok, bool report) {
  const int t = g.targets[tok];
  if (t >= 0 && t < g.vocab) return t;
  if (report) atomicOr(g.status, kStatusTarget);
  return 0;
}

// MFMAs of row blocks [I0, I1) for one K step
template <int KS, int I0, int I1, class OA, class OB, int RB, int CB>
__device__ __forceinline__ void mma_rows(f32x16 (&acc)[RB][CB], const typename OA::Frags& fa, const typename OB::Frags& fb) {
#pragma unroll
  for (int i = I0; i < I1; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j)
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(OA::template get<KS>(fa, i), OB::template get<KS>(fb, j),
                                                          acc[i][j], 0, 0, 0);
}

// The MFMAs of one stage on the fragments fa, fb, with the next stage's fragment reads (LDS offset
// st) issued in four groups between them, so that reads and matrix work overlap and at most a
// few reads queue at a time.  The scheduling barriers keep each group in its place.
template <class OA, class OB, int RB, int CB>
__device__ __forceinline__ void mma_stage(f32x16 (&acc)[RB][CB], const typename OA::Frags& fa,
                                          const typename OB::Frags& fb, const OA& oa, const OB& ob,
                                          typename OA::Frags& na, typename OB::Frags& nb, uint32_t st) {
  oa.template read<0>(na, st);
  __builtin_amdgcn_sched_barrier(0);
  mma_rows<0, 0, RB / 2, OA, OB>(acc, fa, fb);
  __builtin_amdgcn_sched_barrier(0);
  ob.template read<0>(nb, st);
  __builtin_amdgcn_sched_barrier(0);
  mma_rows<0, RB / 2, RB, OA, OB>(acc, fa, fb);
  __builtin_amdgcn_sched_barrier(0);
  oa.template read<1>(na, st);
  __builtin_amdgcn_sched_barrier(0);
  mma_rows<1, 0, RB / 2, OA, OB>(acc, fa, fb);
  __builtin_amdgcn_sched_barrier(0);
  ob.template read<1>(nb, st);
  __builtin_amdgcn_sched_barrier(0);
  mma_rows<1, RB / 2, RB, OA, OB>(acc, fa, fb);
  __builtin_amdgcn_sched_barrier(0);
  OA::wait(na);
  OB::wait(nb);
}

template <int T, bool TRA, bool TRB, int EPI>
__global__ __launch_bounds__(64 * kWaves) void xent_gemm(GemmArgs g) {
  extern __shared__ __align__(16) uint8_t smem[];
  constexpr int kThreads = 64 * kWaves;
  constexpr int TM = T, TN = T, GM = 2, GN = 2;
  constexpr int WM = TM / GM, WN = TN / GN;   // wave tile
  constexpr int RB = WM / 32, CB = WN / 32;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wv / GN, wn = wv % GN;
  int tm, tn, z;
  tile_of(blockIdx.x, gridDim.x, g.tiles_m, g.tiles_n, tm, tn, z);
  const int row0 = tm * TM, col0 = tn * TN;

  f32x16 acc[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) acc[i][j] = f32x16{};
  const int fr = lane & 31, fh = lane >> 5;
  {
    constexpr int SD = stage_bytes<T>(), SA = SD / 2, S = kStages;
    using OA = Operand<T, RB, TRA>;
    using OB = Operand<T, CB, TRB>;
    using LA = Loader<T, TRA>;
    using LB = Loader<T, TRB>;
    constexpr int NIW = LA::NI + LB::NI;
    const int k0 = z * g.k_split, KT = min(g.k_split, g.K - k0) / kKD;   // an even number of stages
    LA la;
    LB lb;
    la.init(g.A, g.lda, g.a_valid, g.a_cols, row0, k0, lane, wv);
    lb.init(g.B, g.ldb, g.b_valid, g.b_cols, col0, k0, lane, wv);
    OA oa;
    OB ob;
    const uint32_t base = lds_addr(smem);
    oa.init(base, wm * WM, lane);
    ob.init(base + SA, wn * WN, lane);
    auto dma = [&](int kt) {
      uint8_t* st = smem + (kt % S) * SD;
      la.stage(kt, st, wv);
      lb.stage(kt, st + SA, wv);
    };
    for (int s = 0; s < S && s < KT; ++s) dma(s);
    typename OA::Frags fa, na;
    typename OB::Frags fb, nb;
    wait_stages<NIW, S>(min(S, KT) - 1);
    __builtin_amdgcn_s_barrier();
    oa.template read<0>(fa, 0);
    ob.template read<0>(fb, 0);
    oa.template read<1>(fa, 0);
    ob.template read<1>(fb, 0);
    OA::wait(fa);
    OB::wait(fb);
    // Stage kt's fragments are in registers when its iteration starts, so after the barrier (every
    // wave has them, and stage kt + 1 has landed for every wave) its slot takes stage kt + S.  The
    // last iteration reads a slot that holds an old stage; those fragments are not used.
    auto step = [&](int kt, typename OA::Frags& ca, typename OB::Frags& cb, typename OA::Frags& xa,
                    typename OB::Frags& xb) {
      wait_stages<NIW, S - 1>(max(min(KT, kt + S) - kt - 2, 0));
      __builtin_amdgcn_s_barrier();
      if (kt + S < KT) dma(kt + S);
      mma_stage<OA, OB>(acc, ca, cb, oa, ob, xa, xb, uint32_t(((kt + 1) % S) * SD));
    };
    for (int kt = 0; kt < KT; kt += 2) {
      step(kt, fa, fb, na, nb);
      step(kt + 1, na, nb, fa, fb);
    }
    __builtin_amdgcn_s_barrier();   // the epilogue reuses the ring
  }

  // Output element e of acc[i][j] (32 x 32 MFMA layout): row 8 (e / 4) + 4 (lane / 32) + e % 4,
  // column lane % 32 of the block.
  auto trow = [&](int i, int e) { return wm * WM + i * 32 + 8 * (e >> 2) + 4 * fh + (e & 3); };
  auto tcol = [&](int j) { return wn * WN + j * 32 + fr; };

  if constexpr (EPI == kEpiLse) {
    // rows are vocabulary ids, columns tokens: a lane holds one token per 32-column block and 16
    // vocabulary rows per 32-row block, so a token's (max, sum) is a reduction in registers, one
    // exchange with the other half-wave and a merge of the GM waves that share the column
    float* smax = reinterpret_cast<float*>(smem);   // [GM][TN]
    float* ssum = smax + GM * TN;                    // [GM][TN]
    int* stg = reinterpret_cast<int*>(ssum + GM * TN);  // [TN] target of each token
    for (int c = tid; c < TN; c += kThreads) stg[c] = target_of(g, min(col0 + c, g.n_valid - 1), tm == 0);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < CB; ++j) {
      const int ct = tcol(j), t = stg[ct] - row0;
      if (row0 + TM > g.m_valid) {   // rows past the vocabulary do not count
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            if (row0 + trow(i, e) >= g.m_valid) acc[i][j][e] = -INFINITY;
      }
      float mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < RB; ++i) {
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = fmaxf(mx, acc[i][j][e]);
        // few 32-row blocks hold a target of one of the wave's 32 tokens
        if (__any(uint32_t(t - (wm * WM + i * 32)) < 32u)) {
#pragma unroll
          for (int e = 0; e < 16; ++e)
            if (trow(i, e) == t && col0 + ct < g.n_valid) g.tgt[col0 + ct] = acc[i][j][e];
        }
      }
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      float s = 0.f;
      if (mx != -INFINITY) {
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e) s += exp_neg(acc[i][j][e] - mx);
      }
      s += __shfl_xor(s, 32);
      if (fh == 0) {
        smax[wm * TN + ct] = mx;
        ssum[wm * TN + ct] = s;
      }
    }
    __syncthreads();
    for (int c = tid; c < TN; c += kThreads) {
      float m = -INFINITY;
#pragma unroll
      for (int w = 0; w < GM; ++w) m = fmaxf(m, smax[w * TN + c]);
      float s = 0.f;
#pragma unroll
      for (int w = 0; w < GM; ++w)
        if (smax[w * TN + c] != -INFINITY) s += ssum[w * TN + c] * exp_neg(smax[w * TN + c] - m);
      float2* p = reinterpret_cast<float2*>(g.part) + int64_t(tm) * g.ldp + col0 + c;
      *p = make_float2(m, s);
    }
  } else if constexpr (EPI == kEpiProb) {
    // rows are the chunk's vocabulary ids, columns tokens: staged token-major (the 4 consecutive
    // vocabulary rows of a lane in one 8-byte write), then P rows as 16-byte pieces
    constexpr int PITCH = staging_pitch<T>();
    uint16_t* st = reinterpret_cast<uint16_t*>(smem);   // the stage buffers are free now
    float* slse = reinterpret_cast<float*>(smem + size_t(TN) * PITCH * 2);
    int* stg = reinterpret_cast<int*>(slse + TN);
    for (int c = tid; c < TN; c += kThreads) {
      const int tok = min(col0 + c, g.n_valid - 1);
      slse[c] = g.lse[tok];
      stg[c] = target_of(g, tok, tm == 0) - g.vcol0;
    }
    __syncthreads();
    const float scale = g.grad[0] * g.inv_n;
#pragma unroll
    for (int j = 0; j < CB; ++j) {
      const int ct = tcol(j), t = stg[ct];
      const float ls = slse[ct];
      // padding outputs are 0 (tiles past the tokens or the chunk's ids), the target's -1 is found in
      // few 32-row blocks
      const int rows = col0 + ct < g.n_valid ? g.m_valid - row0 : 0;
      const bool ragged = row0 + TM > g.m_valid || col0 + TN > g.n_valid;
#pragma unroll
      for (int i = 0; i < RB; ++i) {
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = exp_neg(acc[i][j][e] - ls);
        if (__any(uint32_t(t - row0 - (wm * WM + i * 32)) < 32u)) {
#pragma unroll
          for (int e = 0; e < 16; ++e)
            if (row0 + trow(i, e) == t) acc[i][j][e] -= 1.f;
        }
        if (ragged) {
#pragma unroll
          for (int e = 0; e < 16; ++e)
            if (trow(i, e) >= rows) acc[i][j][e] = 0.f;
        }
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
          uint32_t h[2];
#pragma unroll
          for (int u = 0; u < 2; ++u)
            h[u] = pack2(acc[i][j][4 * e4 + 2 * u] * scale, acc[i][j][4 * e4 + 2 * u + 1] * scale);
          *reinterpret_cast<uint2*>(st + ct * PITCH + trow(i, 4 * e4)) = make_uint2(h[0], h[1]);
        }
      }
    }
    __syncthreads();
    for (int q = tid; q < TN * TM / 8; q += kThreads) {
      const int c = q / (TM / 8), r8 = q % (TM / 8);
      *reinterpret_cast<u32x4*>(g.P + int64_t(col0 + c) * g.ldP + row0 + 8 * r8) =
          *reinterpret_cast<const u32x4*>(st + c * PITCH + 8 * r8);
    }
  } else if constexpr (EPI == kEpiPartF32) {
    float* part = g.acc + z * g.acc_split;
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int r = row0 + trow(i, e);
        if (r >= g.m_valid) continue;
#pragma unroll
        for (int j = 0; j < CB; ++j) {
          const int c = col0 + tcol(j);
          if (c >= g.n_valid) continue;
          float* p = part + int64_t(r) * g.ldacc + c;
          *p = g.accumulate ? *p + acc[i][j][e] : acc[i][j][e];
        }
      }
  } else {   // kEpiStoreBf16: the transpose, staged like kEpiProb (output row = tile column)
    constexpr int PITCH = staging_pitch<T>();
    uint16_t* st = reinterpret_cast<uint16_t*>(smem);
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4)
          *reinterpret_cast<uint2*>(st + tcol(j) * PITCH + trow(i, 4 * e4)) =
              make_uint2(pack2(acc[i][j][4 * e4], acc[i][j][4 * e4 + 1]), pack2(acc[i][j][4 * e4 + 2], acc[i][j][4 * e4 + 3]));
    __syncthreads();
    for (int q = tid; q < TN * TM / 8; q += kThreads) {
      const int c = q / (TM / 8), r = 8 * (q % (TM / 8));
      if (col0 + c < g.n_valid && row0 + r < g.m_valid)   // (m_valid is a multiple of 8)
        *reinterpret_cast<u32x4*>(g.out + int64_t(col0 + c) * g.ldout + row0 + r) =
            *reinterpret_cast<const u32x4*>(st + c * PITCH + r);
    }
  }
}

// out = bf16 of the sum of the splits' partials, in split order; 4 values per thread
__global__ __launch_bounds__(256) void xent_sum_parts(const float* part, int splits, int64_t stride, int64_t n4,
                                                      uint16_t* out) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n4) return;
  float4 s = reinterpret_cast<const float4*>(part)[i];
  for (int z = 1; z < splits; ++z) {
    const float4 v = reinterpret_cast<const float4*>(part + z * stride)[i];
    s.x += v.x;
    s.y += v.y;
    s.z += v.z;
    s.w += v.w;
  }
  reinterpret_cast<uint2*>(out)[i] =
      make_uint2(f2bf(s.x) | (uint32_t(f2bf(s.y)) << 16), f2bf(s.z) | (uint32_t(f2bf(s.w)) << 16));
}

// Targets as int32 and, in status[0], whether any is outside [0, V): such an id, compared at its own width,
// becomes -1, which the other kernels take as 0.  One workgroup: it needs no cleared status word and is done long before the logits GEMM,
// so a caller that checks waits for this kernel only.
template <typename I>
__global__ __launch_bounds__(1024) void xent_targets(const I* targets, int n, int V, int32_t* out, int32_t* status) {
  bool bad = false;
  for (int i = threadIdx.x; i < n; i += 1024) {
    const I t = targets[i];
    const bool in = t >= 0 && t < V;
    out[i] = in ? int32_t(t) : -1;
    bad |= !in;
  }
  bad = __syncthreads_or(bad);
  if (threadIdx.x == 0) status[0] = bad ? kStatusTarget : 0;
}

// lse of each token from its vocabulary tiles' (max, sum); loss term lse - target logit.  16 lanes
// per token (a block of 256 threads takes 16 tokens): lane u merges tiles u, u + 16, ... in order,
// then the 16 partials are merged pairwise in a fixed tree (lanes u, u ^ 1, u ^ 2, u ^ 4, u ^ 8)
__device__ __forceinline__ void merge_ms(float& m, float& s, float m2, float s2) {
  if (m2 == -INFINITY) return;
  if (m == -INFINITY) {
    m = m2;
    s = s2;
    return;
  }
  const float nm = fmaxf(m, m2);
  s = s * exp_neg(m - nm) + s2 * exp_neg(m2 - nm);
  m = nm;
}
__global__ __launch_bounds__(256) void xent_lse(const float2* part, int tiles, int64_t ldp, const float* tgt, int n,
                                                float* lse, float* lrow) {
  const int u = threadIdx.x & 15;
  const int r = blockIdx.x * 16 + (threadIdx.x >> 4);
  const int rr = min(r, n - 1);
  float m = -INFINITY, s = 0.f;
  for (int t = u; t < tiles; t += 16) {
    const float2 p = part[int64_t(t) * ldp + rr];
    merge_ms(m, s, p.x, p.y);
  }
#pragma unroll
  for (int x = 1; x < 16; x <<= 1) {
    const float m2 = __shfl_xor(m, x, 16), s2 = __shfl_xor(s, x, 16);
    // both lanes of a pair merge in the same order (lower lane's partial first)
    if (u & x) {
      float mm = m2, ss = s2;
      merge_ms(mm, ss, m, s);
      m = mm;
      s = ss;
    } else {
      merge_ms(m, s, m2, s2);
    }
  }
  if (u == 0 && r < n) {
    const float l = m + logf(s);
    lse[r] = l;
    lrow[r] = l - tgt[r];
  }
}

// mean of lrow[0..n) in a fixed order: float64 partial sums per thread, then a tree
__global__ __launch_bounds__(1024) void xent_mean(const float* lrow, int n, float* loss) {
  __shared__ double s[1024];
  double a = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) a += double(lrow[i]);
  s[threadIdx.x] = a;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if (int(threadIdx.x) < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss[0] = float(s[0] / double(n));
}

int64_t al256(int64_t b) { return (b + 255) / 256 * 256; }
int rup(int x, int m) { return (x + m - 1) / m * m; }

// How a call's work is split.  256-tiles where they use the chip: the outputs they cover take at
// least kFill of the 256 CUs' whole passes (a tile per CU and pass), ragged edges and a last pass
// that is partly empty counted as lost; else 128-tiles, whose two workgroups per CU hide each
// other's epilogues.  Measured per product (fill: 256 / 128 us), S^T of the forward: 0.49: 33.6 / 28.4, 0.54: 34.6 /
// 31.8, 0.73: 57.5 / 51.0, 0.75: 68.3 / 71.1, 0.89: 59.1 / 66.9, 0.97: 33.5 / 37.1, 0.98 (N 4096, V 32000,
// d 1024): 306 / 336; grad_W: 0.42: 50.8 / 32.2, 0.73: 42.8 / 35.0, 54.6 / 46.3 and (N 4096) 107 / 115, 0.80: 26.6
// / 28.2, 0.98: 45.4 / 44.3 (N 512) and 253 / 304 (N 4096).  grad_h, whose tiles are split over K, by
// its tiles of 256: 8: 47.8 / 43.5, 16: 77.6 / 77.3, 24: 106 / 116 and 42.6 / 36.3, 32: 133 / 147, 64: 259 / 340.
struct Plan {
  int Np;          // tokens padded to 256
  int C;           // vocabulary ids per chunk (a multiple of 256)
  bool big_f;      // 256-tiles for the forward's S^T (the whole vocabulary)
  bool big_s, big_w, big_h;   // 256-tiles for S^T, grad_W, grad_h
  int splits, k_split;        // grad_h: K splits of a chunk, K per split (a multiple of 64)
};
constexpr double kFill = 0.8, kSplits = 0.75;
constexpr int64_t kBlockBytes = int64_t(256) << 20, kRoomBytes = int64_t(64) << 20;

int cdiv(int x, int m) { return (x + m - 1) / m; }

Plan plan(int n, int V, int d, int chunk) {
  Plan p;
  p.Np = rup(n, 256);
  const int Vp = rup(V, 256), c0 = std::min(rup(std::max(chunk, 1), 256), Vp);
  auto fills = [](int m, int n, int tiles) {   // 256-tiles of m x n outputs on a multiple of 256 CUs
    return double(m) * n >= kFill * 65536.0 * 256 * cdiv(tiles, 256);
  };
  const int t256 = cdiv(n, 256) * cdiv(d, 256);
  // (grad_h's tiles are split over K until they fill the chip)
  p.big_h = t256 >= 32 && double(n) * d >= kFill * 65536.0 * t256;
  const int tiles = p.big_h ? t256 : cdiv(n, 128) * (d / 128);
  p.big_f = fills(Vp, n, Vp / 256 * cdiv(n, 256));
  // Few chunks are what fills the chip (N 509, V 32000: eight chunks 1027 us, one 249), but the chunk is
  // how a caller bounds the memory.  So the vocabulary is cut into as few equal chunks as keep the block
  // within kBlockBytes (or the caller's own block), and the block with grad_h's partials within `room`:
  // eight of the caller's blocks (fewer under 1024 ids, two at 256, the smallest) and the size of W, h
  // and an f32 grad_h, of which W^T, h^T and one grad_h were once held; kRoomBytes in any case.
  // kSplits of the splits that fill the chip are enough.
  const int64_t block = 2 * int64_t(p.Np), part = 4 * int64_t(n) * d;
  const int64_t room =
      std::max(kRoomBytes, std::min(8, c0 / 128) * block * c0 + 2 * (int64_t(Vp) + p.Np) * d + 4 * int64_t(p.Np) * d -
                               (p.big_f ? 0 : 8 * int64_t(Vp / 256) * p.Np));   // (more partials of the forward)
  const int most = std::max<int>(c0, int(std::min<int64_t>(kBlockBytes / block / 256 * 256, Vp)));
  int want = 1;
  for (int k = cdiv(Vp, most);; ++k) {
    p.C = rup(cdiv(Vp, k), 256);
    want = std::max(1, std::min((p.big_h ? 256 : 512) / tiles, p.C / 512));
    const int64_t got = std::max<int64_t>((room - block * p.C) / part, 0);
    const bool enough = double(got) >= kSplits * want;
    want = int(std::max<int64_t>(std::min<int64_t>(want, got), 1));
    if (enough || p.C <= c0) break;
  }
  p.big_s = fills(p.C, n, p.C / 256 * cdiv(n, 256));
  p.big_w = fills(p.C, d, p.C / 256 * cdiv(d, 256));
  p.k_split = rup(cdiv(p.C, want), 64);
  p.splits = cdiv(p.C, p.k_split);
  return p;
}

struct Layout {
  int64_t part, tgt, lrow, P, dh, bytes;
};

Layout layout(int n, int V, int d, const Plan& p) {
  Layout L;
  int64_t o = 0;
  L.part = o;    o += al256(int64_t(rup(V, 256) / (p.big_f ? 256 : 128)) * p.Np * 8);
  L.tgt = o;     o += al256(int64_t(p.Np) * 4);
  L.lrow = o;    o += al256(int64_t(p.Np) * 4);
  L.P = o;       o += al256(int64_t(p.Np) * p.C * 2);
  L.dh = o;      o += al256(int64_t(p.splits) * n * d * 4);
  L.bytes = o;
  return L;
}

// d_model a multiple of 128 (the K step of the logits GEMM, the 128-column tiles of the gradients)
// and every operand small enough for the GEMM's 32-bit element offsets (rows x row stride < 2^31)
bool shape_ok(int n, int V, int d) {
  if (n < 1 || V < 1 || d < 128 || d % 128 || d > 65536) return false;
  const int64_t Np = rup(n, 256), Vp = rup(V, 256);
  return Np * d < (int64_t(1) << 31) && Vp * d < (int64_t(1) << 31) && Np * Vp < (int64_t(1) << 31);
}
template <int T, bool TRA, bool TRB, int EPI>
hipError_t launch_gemm(GemmArgs g, int splits, hipStream_t s) {
  const void* fn = reinterpret_cast<const void*>(&xent_gemm<T, TRA, TRB, EPI>);
  const size_t lds = lds_bytes<T, EPI>();
  if (hipError_t e = msdc::ensure_dynamic_lds(fn, lds); e != hipSuccess) return e;
  g.tiles_m = cdiv(g.m_valid, T);
  g.tiles_n = cdiv(g.n_valid, T);
  hipLaunchKernelGGL((xent_gemm<T, TRA, TRB, EPI>), dim3(g.tiles_m * g.tiles_n * splits), dim3(64 * kWaves), lds, s, g);
  return hipGetLastError();
}
template <bool TRA, bool TRB, int EPI>
hipError_t launch_gemm(bool big, const GemmArgs& g, int splits, hipStream_t s) {
  return big ? launch_gemm<256, TRA, TRB, EPI>(g, splits, s) : launch_gemm<128, TRA, TRB, EPI>(g, splits, s);
}

}  // namespace mxe

using namespace mxe;

extern "C" int64_t msd_xent_workspace_bytes(int32_t n_rows, int32_t vocab, int32_t d_model, int32_t chunk) {
  if (!shape_ok(n_rows, vocab, d_model)) return MSD_E_CONFIG;
  return layout(n_rows, vocab, d_model, plan(n_rows, vocab, d_model, chunk)).bytes;
}

extern "C" int32_t msd_xent_plan(int32_t n_rows, int32_t vocab, int32_t d_model, int32_t chunk, int32_t* out) {
  if (!out) return MSD_E_ARG;
  if (!shape_ok(n_rows, vocab, d_model)) return MSD_E_CONFIG;
  const Plan p = plan(n_rows, vocab, d_model, chunk);
  const int chunks = cdiv(vocab, p.C), last = vocab - (chunks - 1) * p.C;
  const int32_t v[8] = {p.C, chunks, p.big_f ? 256 : 128, p.big_s ? 256 : 128, p.big_w ? 256 : 128, p.big_h ? 256 : 128,
                        cdiv(rup(std::min(p.C, vocab), 64), p.k_split), cdiv(rup(last, 64), p.k_split)};
  std::copy(v, v + 8, out);
  return MSD_OK;
}

extern "C" int32_t msd_xent_targets(const void* targets, int32_t bytes_each, int32_t n_rows, int32_t vocab, int32_t* out,
                                    int32_t* status, void* stream) {
  if (n_rows < 1 || vocab < 1) return MSD_E_CONFIG;
  if (!targets || !out || !status || (bytes_each != 4 && bytes_each != 8)) return MSD_E_ARG;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (bytes_each == 8)
    hipLaunchKernelGGL(xent_targets<int64_t>, dim3(1), dim3(1024), 0, s, static_cast<const int64_t*>(targets), n_rows, vocab,
                       out, status);
  else
    hipLaunchKernelGGL(xent_targets<int32_t>, dim3(1), dim3(1024), 0, s, static_cast<const int32_t*>(targets), n_rows, vocab,
                       out, status);
  return hipGetLastError() == hipSuccess ? MSD_OK : MSD_E_HIP;
}

extern "C" int32_t msd_xent_forward(const void* h, const void* weight, const int32_t* targets, int32_t n_rows,
                                    int32_t vocab, int32_t d_model, void* workspace, float* loss, float* lse,
                                    int32_t* status, void* stream) {
  if (!shape_ok(n_rows, vocab, d_model)) return MSD_E_CONFIG;
  if (!h || !weight || !targets || !workspace || !loss || !lse || !status) return MSD_E_ARG;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const Plan p = plan(n_rows, vocab, d_model, vocab);   // (what it takes of it is the same for every chunk)
  const Layout L = layout(n_rows, vocab, d_model, p);
  char* ws = static_cast<char*>(workspace);
  GemmArgs g{};
  // S^T = W h^T: tile rows are vocabulary ids, columns tokens
  g.A = static_cast<const uint16_t*>(weight);
  g.lda = d_model;
  g.a_valid = vocab;
  g.B = static_cast<const uint16_t*>(h);
  g.ldb = d_model;
  g.b_valid = n_rows;
  g.K = g.k_split = d_model;
  g.m_valid = vocab;
  g.n_valid = n_rows;
  g.targets = targets;
  g.vocab = vocab;
  g.status = status;
  g.part = reinterpret_cast<float*>(ws + L.part);
  g.ldp = p.Np;
  g.tgt = reinterpret_cast<float*>(ws + L.tgt);
  if (launch_gemm<false, false, kEpiLse>(p.big_f, g, 1, s) != hipSuccess) return MSD_E_HIP;
  float* lrow = reinterpret_cast<float*>(ws + L.lrow);
  hipLaunchKernelGGL(xent_lse, dim3((n_rows + 15) / 16), dim3(256), 0, s, reinterpret_cast<const float2*>(g.part),
                     cdiv(vocab, p.big_f ? 256 : 128), int64_t(p.Np), g.tgt, n_rows, lse, lrow);
  hipLaunchKernelGGL(xent_mean, dim3(1), dim3(1024), 0, s, lrow, n_rows, loss);
  return hipGetLastError() == hipSuccess ? MSD_OK : MSD_E_HIP;
}

extern "C" int32_t msd_xent_backward(const void* h, const void* weight, const int32_t* targets, const float* lse,
                                     const float* grad_loss, int32_t n_rows, int32_t vocab, int32_t d_model,
                                     int32_t chunk, void* workspace, void* grad_h, void* grad_weight,
                                     int32_t* status, void* stream) {
  if (!shape_ok(n_rows, vocab, d_model)) return MSD_E_CONFIG;
  if (!h || !weight || !targets || !lse || !grad_loss || !workspace || !grad_h || !grad_weight || !status)
    return MSD_E_ARG;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const Plan pl = plan(n_rows, vocab, d_model, chunk);
  const Layout L = layout(n_rows, vocab, d_model, pl);
  char* ws = static_cast<char*>(workspace);
  uint16_t* P = reinterpret_cast<uint16_t*>(ws + L.P);
  float* dh = reinterpret_cast<float*>(ws + L.dh);
  const uint16_t* W = static_cast<const uint16_t*>(weight);
  const uint16_t* H = static_cast<const uint16_t*>(h);
  int splits = 1;
  for (int v0 = 0; v0 < vocab; v0 += pl.C) {
    const int cv = std::min(pl.C, vocab - v0);   // valid columns of this chunk
    GemmArgs p{};
    p.A = W + int64_t(v0) * d_model;   // S^T of the chunk: rows vocabulary ids, columns tokens
    p.lda = d_model;
    p.a_valid = cv;
    p.B = H;
    p.ldb = d_model;
    p.b_valid = n_rows;
    p.K = p.k_split = d_model;
    p.m_valid = cv;
    p.n_valid = n_rows;
    p.targets = targets;
    p.vocab = vocab;
    p.status = status;
    p.vcol0 = v0;
    p.lse = lse;
    p.grad = grad_loss;
    p.inv_n = 1.0f / float(n_rows);
    p.P = P;
    p.ldP = pl.C;
    if (launch_gemm<false, false, kEpiProb>(pl.big_s, p, 1, s) != hipSuccess) return MSD_E_HIP;
    // grad_W^T of the chunk = h^T P over the tokens, whose padding (to 64, inside P's tiles) is 0 in
    // P; the rows of h past the last read the last
    GemmArgs w{};
    w.A = H;
    w.lda = d_model;
    w.a_valid = n_rows;
    w.a_cols = d_model;
    w.B = P;
    w.ldb = pl.C;
    w.b_valid = pl.Np;
    w.b_cols = pl.C;
    w.K = w.k_split = rup(n_rows, 64);
    w.m_valid = d_model;
    w.n_valid = cv;
    w.out = static_cast<uint16_t*>(grad_weight) + int64_t(v0) * d_model;
    w.ldout = d_model;
    if (launch_gemm<true, true, kEpiStoreBf16>(pl.big_w, w, 1, s) != hipSuccess) return MSD_E_HIP;
    // grad_h partials (+)= P W_c over the chunk's ids, padded with P's zeros likewise
    GemmArgs a{};
    a.A = P;
    a.lda = pl.C;
    a.a_valid = n_rows;
    a.B = W + int64_t(v0) * d_model;
    a.ldb = d_model;
    a.b_valid = cv;
    a.b_cols = d_model;
    a.K = rup(cv, 64);
    a.k_split = pl.k_split;
    a.m_valid = n_rows;
    a.n_valid = d_model;
    a.acc = dh;
    a.ldacc = d_model;
    a.acc_split = int64_t(n_rows) * d_model;
    a.accumulate = v0 > 0;
    const int sp = cdiv(a.K, a.k_split);   // (a short last chunk may have fewer)
    splits = std::max(splits, sp);
    if (launch_gemm<false, true, kEpiPartF32>(pl.big_h, a, sp, s) != hipSuccess) return MSD_E_HIP;
  }
  const int64_t n4 = int64_t(n_rows) * d_model / 4;
  hipLaunchKernelGGL(xent_sum_parts, dim3(unsigned((n4 + 255) / 256)), dim3(256), 0, s, dh, splits,
                     int64_t(n_rows) * d_model, n4, static_cast<uint16_t*>(grad_h));
  return hipGetLastError() == hipSuccess ? MSD_OK : MSD_E_HIP;
}
