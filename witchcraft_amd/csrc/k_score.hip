// k_score.hip -- query-side scoring next to the encoder: C = A . B^T in f32 and its per-row
// argmax (k-means assignment).
//
// Reference: fast_ops::matmul_t (src/fast_ops.rs:98-116) and PackedRight::matmul
// (:65-95), used for query x centroid / residual scores (src/lib.rs:637,735,759,1646), and
// matmul_argmax_batched (src/lib.rs:187-208, called at :235,1330).  The default build
// multiplies f32 x f32 (candle); the fbgemm build first truncates B to bf16
// (PackedMatrixBf16, fbgemm-rs/src/bf16.rs:21-31) and accumulates in f32 -- bf16_b selects it.
//
// f32 MFMA (v_mfma_f32_16x16x4_f32): products are exact f32 as on the CPU.  A lane holds 4
// consecutive K values of one row (one float4 load from global) and feeds them to 4
// consecutive MFMAs, each of which sums its K-lane group g = lane / 16 over k = 16 kb + 4 g + j;
// A and B use the same assignment, so every product a[k] b[k] is summed once.
//   * matmul_t: wave tile = 16 MB rows x 64 columns, MB = ceil(M / 16) up to 4, so query-sized
//     M (32 query tokens against many residuals, HBM-bound on B) pads to 16 rows at most.
//     Workgroup = 4 waves side by side along N (or along M when N <= 64).
//   * argmax:   workgroup = 4 waves on 64 rows, looping over N in 256-column chunks; the
//     running (max, index) per row lives in registers, the 4 waves' results meet in LDS.
//     Ties resolve to the smallest column index (candle's argmax keeps the first maximum).
//     128-d rows run on f16 MFMAs with split operands (matmul_argmax_split_kernel).
#include "common.hpp"

#include <algorithm>
#include <atomic>

namespace {

typedef float f4v __attribute__((ext_vector_type(4)));

// Word 3 of a raw (stride 0) buffer descriptor on gfx9-family GPUs: 32-bit data format, so
// an access beyond num_records returns zero (loads) or is dropped (stores).
constexpr int kBufDword3 = 0x00020000;
constexpr int kBufNt = 2;  // buffer access policy bit: non-temporal

__device__ __forceinline__ float4 ldg4(const float* p) { return *reinterpret_cast<const float4*>(p); }

__device__ __forceinline__ float4 trunc_bf16(float4 v) {
  auto t = [](float x) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x) & 0xffff0000u;
    return __builtin_bit_cast(float, u);
  };
  return make_float4(t(v.x), t(v.y), t(v.z), t(v.w));
}

// p[0..3] of one row (zero if !ok).  VEC: rows are 16-byte aligned (D % 4 == 0 and aligned
// bases), so one float4 load; otherwise 4 scalar loads.
template <bool VEC>
__device__ __forceinline__ float4 ld4(const float* p, bool ok) {
  if (VEC) return ok ? ldg4(p) : make_float4(0.f, 0.f, 0.f, 0.f);
  return ok ? make_float4(p[0], p[1], p[2], p[3]) : make_float4(0.f, 0.f, 0.f, 0.f);
}

// p[j] for j < n (zero past it, or everywhere if !ok): the last, partial K block.
__device__ __forceinline__ float4 ld4_tail(const float* p, int n, bool ok) {
  float v[4];
#pragma unroll
  for (int j = 0; j < 4; j++) v[j] = (ok && j < n) ? p[j] : 0.f;
  return make_float4(v[0], v[1], v[2], v[3]);
}

template <int MB>
__device__ __forceinline__ void mfma_4x4(const float4 (&a)[4], const float4 (&b)[4], f4v (&acc)[4][4]) {
#pragma unroll
  for (int mb = 0; mb < MB; mb++)
#pragma unroll
    for (int nb = 0; nb < 4; nb++) {
      // B as the MFMA A operand: lane ends with 4 consecutive columns of one row
      acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[nb].x, a[mb].x, acc[mb][nb], 0, 0, 0);
      acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[nb].y, a[mb].y, acc[mb][nb], 0, 0, 0);
      acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[nb].z, a[mb].z, acc[mb][nb], 0, 0, 0);
      acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[nb].w, a[mb].w, acc[mb][nb], 0, 0, 0);
    }
}

// acc[mb][nb] += A[rows 16mb..] . B[cols 16nb..]^T over all of K for a 16 MB x 64 wave tile;
// rows / columns outside the matrices and K past D read as zero.  Full 16-wide K blocks run
// unguarded; the last partial block (D % 16 != 0) masks per element.
template <int MB, bool BF16B, bool VEC>
__device__ __forceinline__ void wave_tile(const float* __restrict__ A, const float* __restrict__ B, int M,
                                           int N, int D, int r0, int c0, int lane, f4v (&acc)[4][4]) {
  const int lr = lane & 15, lg = lane >> 4;
  const float* ar[4];
  const float* br[4];
  bool av[4], bv[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int r = r0 + 16 * i + lr, c = c0 + 16 * i + lr;
    av[i] = r < M;
    bv[i] = c < N;
    ar[i] = A + (size_t)(av[i] ? r : 0) * D + 4 * lg;
    br[i] = B + (size_t)(bv[i] ? c : 0) * D + 4 * lg;
  }
  const int dfull = D & ~15;
  for (int kb = 0; kb < dfull; kb += 16) {
    float4 a[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      a[i] = i < MB ? ld4<VEC>(ar[i] + kb, av[i]) : make_float4(0.f, 0.f, 0.f, 0.f);
      b[i] = ld4<VEC>(br[i] + kb, bv[i]);
      if (BF16B) b[i] = trunc_bf16(b[i]);
    }
    mfma_4x4<MB>(a, b, acc);
  }
  if (dfull < D) {
    // this lane's 4 values are k = dfull + 4 lg + j, of which the first D - dfull - 4 lg exist
    const int n = D - dfull - 4 * lg;
    float4 a[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      a[i] = i < MB ? ld4_tail(ar[i] + dfull, n, av[i]) : make_float4(0.f, 0.f, 0.f, 0.f);
      b[i] = ld4_tail(br[i] + dfull, n, bv[i]);
      if (BF16B) b[i] = trunc_bf16(b[i]);
    }
    mfma_4x4<MB>(a, b, acc);
  }
}

// With B as the MFMA A operand (16 columns) and A as the B operand (16 rows), lane l holds
// C[row 16mb + (l % 16)][cols 16nb + 4(l / 16) + 0..3].  wn = waves of the workgroup along N
// (4, or 1 when N <= 64, then the 4 waves stack along M).
template <int MB, bool BF16B, bool VEC>
__global__ __launch_bounds__(256) void matmul_t_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                       float* __restrict__ C, int M, int N, int D, int wn,
                                                       int tiles_n) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wm = 4 / wn;
  // 1-D grid, column tiles fastest: workgroups in flight share rows of A and walk B in order
  const int bm = blockIdx.x / tiles_n, bn = blockIdx.x - bm * tiles_n;
  const int r0 = (bm * wm + wave / wn) * 16 * MB, c0 = (bn * wn + wave % wn) * 64;
  if (r0 >= M || c0 >= N) return;  // wave-uniform; no workgroup barrier follows
  f4v acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = f4v{0.f, 0.f, 0.f, 0.f};
  wave_tile<MB, BF16B, VEC>(A, B, M, N, D, r0, c0, lane, acc);
  const int lr = lane & 15, lg = lane >> 4;
  const bool vec_out = (N & 3) == 0 && VEC;
#pragma unroll
  for (int mb = 0; mb < MB; mb++) {
    const int r = r0 + 16 * mb + lr;
    if (r >= M) continue;
#pragma unroll
    for (int nb = 0; nb < 4; nb++) {
      const int c = c0 + 16 * nb + 4 * lg;
      float* out = C + (size_t)r * N + c;
      if (vec_out && c + 3 < N) {
        *reinterpret_cast<float4*>(out) = make_float4(acc[mb][nb][0], acc[mb][nb][1], acc[mb][nb][2], acc[mb][nb][3]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (c + i < N) out[i] = acc[mb][nb][i];
      }
    }
  }
}

// Query-sized A (16 MB <= 32 rows per grid row) against a long B of 128-d rows
// (src/lib.rs:734-735): a stream over B.  Persistent waves; wave w takes 32-column tiles
// w, w + W, w + 2W, ... (W = all waves of the grid, so the waves in flight cover one
// contiguous stretch of B).  A sits in LDS for the whole run, and the next tile's B loads
// are issued before the current tile's MFMAs and stores, so HBM streams while the f32
// MFMAs run.
template <int MB, bool BF16B, bool NT>
__global__ __launch_bounds__(256, 2) void matmul_t_stream_kernel(const float* __restrict__ A,
                                                                 const float* __restrict__ B,
                                                                 float* __restrict__ C, int M, int N) {
  constexpr int D = 128, KB = D / 16, AS = D / 4 + 1;  // A row stride in LDS: 33 float4
  __shared__ float4 As[16 * MB * AS];
  A += (size_t)blockIdx.y * 16 * MB * D;  // this grid row's pass of query rows
  C += (size_t)blockIdx.y * 16 * MB * N;
  M = min(M - (int)blockIdx.y * 16 * MB, 16 * MB);
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  // wave index made visibly uniform, so tile bases and descriptors live in scalar registers
  const int w0 = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = gridDim.x * 4;
  const int ntiles = (N + 31) / 32, nfull = N / 32, tail_bytes = (N % 32) * D * 4;
  // A (16 MB rows, rows past M repeat row M - 1) into LDS once; no barrier after this one
  for (int e = threadIdx.x; e < 16 * MB * (D / 4); e += 256) {
    const int r = e / (D / 4), q = e - r * (D / 4);
    As[r * AS + q] = ldg4(A + (size_t)min(r, M - 1) * D + 4 * q);
  }
  __syncthreads();
  // B tile t through a buffer descriptor whose range ends at column N: columns past N (the
  // last tile's tail, and the prefetch past the last tile) read as zero without touching
  // memory.  Lane offsets are loop-invariant, so no address registers live across the loop.
  const int voff[2] = {(lr * D + 4 * lg) * 4, ((16 + lr) * D + 4 * lg) * 4};
  auto load = [&](int t, float4 (&b)[KB][2]) {
    // (selected on the tile index rather than clamped: a clamp becomes a vector med3, whose
    // result register the allocator may take from a load still in flight)
    const int bytes = t < nfull ? 32 * D * 4 : (t == nfull ? tail_bytes : 0);
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)(B + (size_t)t * 32 * D), (short)0, bytes, kBufDword3);
#pragma unroll
    for (int nb = 0; nb < 2; nb++)
#pragma unroll
      for (int kb = 0; kb < KB; kb++) {
        const f4v v = __builtin_amdgcn_raw_buffer_load_b128(rs, voff[nb] + 64 * kb, 0, 0);
        b[kb][nb] = make_float4(v[0], v[1], v[2], v[3]);
      }
  };
  auto compute = [&](const float4 (&b)[KB][2], f4v (&acc)[MB][2]) {
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
      for (int nb = 0; nb < 2; nb++) acc[i][nb] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < KB; kb++)
#pragma unroll
      for (int nb = 0; nb < 2; nb++) {
        const float4 bb = BF16B ? trunc_bf16(b[kb][nb]) : b[kb][nb];
#pragma unroll
        for (int i = 0; i < MB; i++) {
          const float4 a = As[(16 * i + lr) * AS + 4 * kb + lg];
          acc[i][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(bb.x, a.x, acc[i][nb], 0, 0, 0);
          acc[i][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(bb.y, a.y, acc[i][nb], 0, 0, 0);
          acc[i][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(bb.z, a.z, acc[i][nb], 0, 0, 0);
          acc[i][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(bb.w, a.w, acc[i][nb], 0, 0, 0);
        }
      }
  };
  // lane holds C[16 i + lr][32 t + 16 nb + 4 lg + 0..3] (stores through a descriptor based at
  // column 32 t; row offsets r N 4 < 2^31 is a launch condition)
  int soff[MB];
#pragma unroll
  for (int i = 0; i < MB; i++) soff[i] = ((16 * i + lr) * N + 4 * lg) * 4;
  auto store = [&](int t, const f4v (&acc)[MB][2]) {
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)(C + (size_t)t * 32), (short)0, 0x7fffffff, kBufDword3);
#pragma unroll
    for (int i = 0; i < MB; i++) {
      const bool row_ok = 16 * i + lr < M;
#pragma unroll
      for (int nb = 0; nb < 2; nb++)
        if (row_ok && 32 * t + 16 * nb + 4 * lg + 3 < N)
          __builtin_amdgcn_raw_buffer_store_b128(acc[i][nb], rs, soff[i] + 64 * nb, 0, NT ? kBufNt : 0);
      if (t >= nfull && row_ok)
#pragma unroll
        for (int nb = 0; nb < 2; nb++) {  // the last tile: N may end inside a lane's four columns
          const int left = N - (32 * t + 16 * nb + 4 * lg);
#pragma unroll
          for (int j = 0; j < 3; j++)
            if (left < 4 && j < left)
              __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[i][nb][j]), rs, soff[i] + 64 * nb + 4 * j, 0, 0);
        }
    }
  };
  // Per tile: issue the next tile's loads, then the previous tile's stores, then this tile's
  // MFMAs.  Loads and stores share one in-order counter, so stores issued after the next
  // loads never hold up the wait for this tile's data.  Two tiles per trip let the B and
  // accumulator buffers alternate without copies; every bound is wave-uniform.  (The
  // scheduling barriers keep that issue order.)
  float4 b0[KB][2], b1[KB][2];
  f4v acc0[MB][2], acc1[MB][2];
  int t = w0, t1 = -1;  // t1: tile whose results wait in acc1
  load(t, b0);
  while (t < ntiles) {
    load(t + nw, b1);
    __builtin_amdgcn_sched_barrier(0);
    if (t1 >= 0) store(t1, acc1);
    __builtin_amdgcn_sched_barrier(0);
    compute(b0, acc0);
    const int t0 = t;
    t += nw;
    t1 = -1;
    if (t >= ntiles) {
      store(t0, acc0);
      break;
    }
    load(t + nw, b0);
    __builtin_amdgcn_sched_barrier(0);
    store(t0, acc0);
    __builtin_amdgcn_sched_barrier(0);
    compute(b1, acc1);
    t1 = t;
    t += nw;
  }
  if (t1 >= 0) store(t1, acc1);
}

// (v, i) beats (w, j) if v > w, or v == w and i < j (first maximum wins).
__device__ __forceinline__ void amax_merge(float& v, int& i, float w, int j) {
  if (w > v || (w == v && j < i)) {
    v = w;
    i = j;
  }
}

template <bool BF16B, bool VEC>
__global__ __launch_bounds__(256) void matmul_argmax_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                            uint32_t* __restrict__ out, int M, int N, int D) {
  __shared__ float sv[4][64];
  __shared__ int si[4][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int lr = lane & 15, lg = lane >> 4;
  const int r0 = blockIdx.x * 64;
  // running maximum of row 16mb + lr (identical in the 4 lanes of that row); starting from
  // (-inf, 0) keeps the result in range when no score exceeds -inf (NaN or -inf rows give 0)
  float bv[4];
  int bi[4];
#pragma unroll
  for (int mb = 0; mb < 4; mb++) {
    bv[mb] = -INFINITY;
    bi[mb] = 0;
  }
  for (int n0 = 0; n0 < N; n0 += 256) {
    const int c0 = n0 + wave * 64;
    if (c0 >= N) break;  // wave-uniform
    f4v acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) acc[i][j] = f4v{0.f, 0.f, 0.f, 0.f};
    wave_tile<4, BF16B, VEC>(A, B, M, N, D, r0, c0, lane, acc);
#pragma unroll
    for (int mb = 0; mb < 4; mb++) {
      float v = -INFINITY;
      int ix = 0x7fffffff;
#pragma unroll
      for (int nb = 0; nb < 4; nb++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int c = c0 + 16 * nb + 4 * lg + i;
          if (c < N) amax_merge(v, ix, acc[mb][nb][i], c);
        }
      // combine the 4 lanes (lg = 0..3) holding this row: lanes l ^ 16, l ^ 32
#pragma unroll
      for (int o = 16; o <= 32; o <<= 1) {
        const float w = __shfl_xor(v, o);
        const int j = __shfl_xor(ix, o);
        amax_merge(v, ix, w, j);
      }
      amax_merge(bv[mb], bi[mb], v, ix);
    }
  }
  if (lg == 0)
#pragma unroll
    for (int mb = 0; mb < 4; mb++) {
      sv[wave][16 * mb + lr] = bv[mb];
      si[wave][16 * mb + lr] = bi[mb];
    }
  __syncthreads();
  if (threadIdx.x < 64) {
    const int t = threadIdx.x, r = r0 + t;
    float v = sv[0][t];
    int ix = si[0][t];
    for (int w = 1; w < 4; w++) amax_merge(v, ix, sv[w][t], si[w][t]);
    if (r < M) out[r] = (uint32_t)ix;
  }
}

// k-means assignment (src/lib.rs:233-236, 1330) at D = 128: argmax of the f32 products, bound by
// the matrix cores.  An f32 MFMA runs at 1/16 of the f16 rate, so both operands are split into two
// f16 parts of a power-of-two multiple (x s = hi + lo + r, |r| <= 2^-23 of x's binade) and a
// product is hi hi + hi lo + lo hi, each exact in the f32 accumulator: 3 f16 MFMAs for 16 f32
// ones.  What is dropped (lo lo and the r terms) is at most 2^-21 |a b| per product, without a
// common sign over the 128 products; the f32 accumulation takes 24 steps where the f32 MFMAs take
// 32.  So the scores compared are nearer to 64 bits than on f32 MFMAs: winning scores 1.0e-7 off (2-norm;
// largest 4 to 7e-7) against 1.7e-7 (7 to 11e-7), over normal, clustered and all-positive rows and columns
// of one size or spread over 50 and 10,000 times; 1.1 to 1.3e-7 against 1.4 to 1.6e-7 on heavy tails.
//  * Rows of A: each scaled by its own power of two (an argmax over the row does not change) and
//    held in registers for the whole run, 32 RBL rows per wave on 32x32x16 MFMAs.
//  * Columns of B: 64 or 128 at a time through double-buffered LDS, split once per workgroup on
//    the way in, by one power of two set from the first columns, whose largest value comes to the
//    middle of f16's precise range.  A column whose largest |b s| lies outside [2^3, 2^15] takes a
//    power of two of its own, which is taken out of its products again, exactly, before they are
//    compared (cscale).  4,096 x 16,384: 275 us, one column at the end 16 times larger 275, empty
//    columns in front 275, sizes over three decades 495; 2,460 to 2,740 when such columns sent all
//    rows to the f32 MFMAs.
//  * A column 2^60 off the first ones, a row beyond 2^-87 .. 2^123, an infinity or a NaN makes the
//    workgroup redo its rows on f32 MFMAs (argmax_rows_f32), so such inputs give what they gave there.
// The 8 waves of a workgroup hold 8 / WN row groups; the WN waves of a group take 1 / WN of a
// chunk's columns each, for inputs with too few rows to fill the chip.
// 131,072 x 16,384: 5.03 ms on f32 MFMAs (109 TFLOP/s) -> 1.28-1.40 ms (390-430); 4,096 x 4,096:
// 228 -> 76 us.  Counters on an earlier form of the loop: MFMA busy 56% at a 1.7 GHz clock, the
// rest vector work (splitting B, the running maxima).
typedef float f16v __attribute__((ext_vector_type(16)));

__device__ __forceinline__ uint32_t float_exp(float v) { return (__float_as_uint(v) >> 23) & 0xffu; }
__device__ __forceinline__ float pow2_bits(uint32_t biased) { return __uint_as_float(biased << 23); }
__device__ __forceinline__ float max4abs(float4 v) {
  return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
}
// Not finite (fmaxf drops NaNs, so the largest magnitude alone does not tell).
__device__ __forceinline__ bool odd4(float4 v) {
  const float z = (v.x - v.x) + (v.y - v.y) + (v.z - v.z) + (v.w - v.w);
  return !(z == 0.f);
}
// Largest of the 32 lanes of a wave half.
__device__ __forceinline__ float max32(float v) {
#define T5K_ROR(n) v = fmaxf(v, __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x120 + (n), 0xf, 0xf, false)))
  T5K_ROR(8);
  T5K_ROR(4);
  T5K_ROR(2);
  T5K_ROR(1);
#undef T5K_ROR
  return max_xor16(v);
}
// s x = hi + lo, each rounded to nearest f16
__device__ __forceinline__ void split_f16(float x, float s, _Float16& hi, _Float16& lo) {
  hi = (_Float16)(x * s);
  lo = (_Float16)__builtin_fmaf(x, s, -(float)hi);
}

// 256 rows from wg_r0 (8 waves of 32) on f32 MFMAs: A in registers, 64-column chunks of B through
// double-buffered LDS (Bs, 2 x 64 x 33 float4).
constexpr int ARG_F32_LDS = 2 * 64 * 33;
template <bool BF16B>
__device__ __forceinline__ void argmax_rows_f32(const float* __restrict__ A, const float* __restrict__ B,
                                             uint32_t* __restrict__ out, int M, int N, int wg_r0, float4* Bs) {
  constexpr int D = 128, KB = D / 16, BS = D / 4 + 1, RB = 2;  // LDS row stride: 33 float4
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int r0 = wg_r0 + wave * (16 * RB);
  // A fragments: row r0 + 16 mb + lr, K slice 16 kb + 4 lg; rows past M repeat row M - 1
  // (their results are not stored)
  float4 a[KB][4];
#pragma unroll
  for (int mb = 0; mb < RB; mb++) {
    const float* p = A + (size_t)min(r0 + 16 * mb + lr, M - 1) * D + 4 * lg;
#pragma unroll
    for (int kb = 0; kb < KB; kb++) a[kb][mb] = ldg4(p + 16 * kb);
  }
  // chunk loader: thread tid moves float4 q = tid + 512 j (j < 4) of the 64 x 32 float4 chunk;
  // columns past N repeat column N - 1 (masked out of the argmax)
  float4 st[4];
  auto gload = [&](int n0) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int q = tid + 512 * j, c = q >> 5, k4 = q & 31;
      st[j] = ldg4(B + (size_t)min(n0 + c, N - 1) * D + 4 * k4);
    }
  };
  auto lstore = [&](int buf) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int q = tid + 512 * j, c = q >> 5, k4 = q & 31;
      Bs[buf * 64 * BS + c * BS + k4] = BF16B ? trunc_bf16(st[j]) : st[j];
    }
  };
  float bv[RB];
  int bi[RB];
#pragma unroll
  for (int mb = 0; mb < RB; mb++) {
    bv[mb] = -INFINITY;
    bi[mb] = 0;
  }
  const int nchunks = (N + 63) / 64;
  gload(0);
  lstore(0);
  __syncthreads();
  for (int ch = 0; ch < nchunks; ch++) {
    const int buf = ch & 1, n0 = ch * 64;
    if (ch + 1 < nchunks) gload(n0 + 64);
    f4v acc[4][4];
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) acc[i][j] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < KB; kb++) {
      float4 b[4];
#pragma unroll
      for (int nb = 0; nb < 4; nb++) b[nb] = Bs[buf * 64 * BS + (16 * nb + lr) * BS + 4 * kb + lg];
      mfma_4x4<RB>(a[kb], b, acc);
    }
#pragma unroll
    for (int mb = 0; mb < RB; mb++) {
      float v = -INFINITY;
      int ix = 0x7fffffff;
#pragma unroll
      for (int nb = 0; nb < 4; nb++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int c = n0 + 16 * nb + 4 * lg + i;
          if (c < N) amax_merge(v, ix, acc[mb][nb][i], c);
        }
#pragma unroll
      for (int o = 16; o <= 32; o <<= 1) {
        const float w = __shfl_xor(v, o);
        const int j = __shfl_xor(ix, o);
        amax_merge(v, ix, w, j);
      }
      amax_merge(bv[mb], bi[mb], v, ix);
    }
    if (ch + 1 < nchunks) {
      lstore(buf ^ 1);
      __syncthreads();
    }
  }
  if (lg == 0)
#pragma unroll
    for (int mb = 0; mb < RB; mb++) {
      const int r = r0 + 16 * mb + lr;
      if (r < M) out[r] = (uint32_t)bi[mb];
    }
}

template <bool BF16B, int RBL, int WN>
__global__ __launch_bounds__(512, 2) void matmul_argmax_split_kernel(const float* __restrict__ A,
                                                                     const float* __restrict__ B,
                                                                     uint32_t* __restrict__ out, int M, int N) {
  constexpr int D = 128, KS = D / 16, PARTS = BF16B ? 1 : 2;  // a truncated b s is one f16
  constexpr int COLS = WN == 4 ? 128 : 64, CB = COLS / 32 / WN, NL = COLS / 16;
  constexpr int PART = COLS * 16;  // h8 per part of a chunk: COLS columns x 16 chunks of 8 k
  constexpr int LDS4 = 2 * PARTS * PART > ARG_F32_LDS ? 2 * PARTS * PART : ARG_F32_LDS;
  __shared__ float4 lds[LDS4];  // chunks [2][PARTS][PART] h8, or argmax_rows_f32's
  __shared__ float red[8];
  __shared__ int redo[2];  // by barrier parity: a flag is rewritten only after every thread has read it
  // what each column's products are multiplied by, and whether any factor of a buffer has ever been
  // other than 1, so that the products need a look at them
  __shared__ __attribute__((aligned(16))) float cscale[2][COLS];
  __shared__ int scaled[2];
  h8* Bs = reinterpret_cast<h8*>(lds);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, lr = lane & 31, lg = lane >> 5;
  constexpr int wg_rows = 32 * RBL * (8 / WN);
  const int wg_r0 = blockIdx.x * wg_rows, r0 = wg_r0 + (wave / WN) * 32 * RBL, cb0 = (wave % WN) * CB;
  bool bad = false;
  // thread tid moves the float4 k4 of columns c0 + 16 j (j < NL) of a chunk, 32 lanes to a column;
  // columns past N repeat column N - 1, which then ties with itself at a larger index
  const int c0 = tid >> 5, k4 = tid & 31;
  float4 st[NL];
  auto gload = [&](int n0) {  // also past the last chunk: unconditional, so nothing waits for it early
    const int first = min(n0, N - 1);  // 64-bit on the scalar unit, 32-bit offsets inside the chunk
    const char* base = reinterpret_cast<const char*>(B) + (size_t)first * (4 * D);
#pragma unroll
    for (int j = 0; j < NL; j++)
      st[j] = *reinterpret_cast<const float4*>(base + ((uint32_t)min(c0 + 16 * j, N - 1 - first) * (4u * D) + 16u * k4));
  };
  gload(0);
  for (int i = tid; i < 2 * COLS; i += 512) (&cscale[0][0])[i] = 1.f;
  {  // one power of two for every column: the first chunk's largest magnitude comes to [2^9, 2^10)
    float m = 0.f;
#pragma unroll
    for (int j = 0; j < NL; j++) m = fmaxf(m, max4abs(BF16B ? trunc_bf16(st[j]) : st[j]));
    m = max_xor32(max32(m));
    if (lane == 0) red[wave] = m;
    if (tid == 0) redo[0] = redo[1] = scaled[0] = scaled[1] = 0;
  }
  __syncthreads();
  float bmax = red[0];
#pragma unroll
  for (int i = 1; i < 8; i++) bmax = fmaxf(bmax, red[i]);
  const bool empty = bmax == 0.f;  // all columns of the first chunk: then as for values of size 1
  const uint32_t be = empty ? 127 : float_exp(bmax);
  if (be < 40 || be > 250) bad = true;  // tiny, huge, infinite
  const uint32_t bse = bad ? 127 : 127 + 9 + 127 - be;  // exponent of the common power of two
  const float bs = pow2_bits(bse);
  int own = 0;  // bit buf: this wave has factors other than 1 in cscale[buf]
  // 16-byte chunk k / 8 of column c sits at chunk (k / 8) ^ (c % 16): the operand reads below (32
  // columns x one chunk) and these stores (one column, 16 chunks) hit every bank once
  const int at0 = (c0 * 16 + ((k4 >> 1) ^ c0)) * 2 + (k4 & 1);
  auto lstore = [&](int buf) {
    uint32_t u[NL];   // largest magnitude of the thread's values: infinities and NaNs compare above every finite one
    bool odd = false;  // wave-uniform: some column outside the range of the common power of two
#pragma unroll
    for (int j = 0; j < NL; j++) {
      const float4 v = BF16B ? trunc_bf16(st[j]) : st[j];
      u[j] = max(max(__float_as_uint(v.x) & 0x7fffffffu, __float_as_uint(v.y) & 0x7fffffffu),
                 max(__float_as_uint(v.z) & 0x7fffffffu, __float_as_uint(v.w) & 0x7fffffffu));
      const float m = __uint_as_float(u[j]) * bs;
      // a column is a wave half: some lane reaches 2^3 or every lane is zero
      const unsigned long long big = __builtin_amdgcn_ballot_w64(m >= 8.f), any = __builtin_amdgcn_ballot_w64(u[j] != 0);
      odd |= __builtin_amdgcn_ballot_w64(!(m <= 32768.f)) != 0 || ((uint32_t)big == 0 && (uint32_t)any != 0) ||
             (big >> 32 == 0 && any >> 32 != 0);
    }
    if (__builtin_expect(odd || (own >> buf & 1), 0)) {
#pragma unroll
      for (int j = 0; j < NL; j++) {
        const float top = max32(__uint_as_float(min(u[j], 0x7f800000u)));  // the column's largest; NaN as infinity
        const int e = (int)float_exp(top), k = (int)be - e;  // by 2^k it comes to the first chunk's size
        const bool out = top != 0.f && !(top * bs >= 8.f && top * bs <= 32768.f);
        const bool far = out && (e < 1 || e == 255 || k < -60 || k > 60);
        bad |= far;
        const int by = out && !far ? k : 0;
        const float f = pow2_bits(127 + by);
        st[j] = make_float4(st[j].x * f, st[j].y * f, st[j].z * f, st[j].w * f);
        if (k4 == 0) cscale[buf][c0 + 16 * j] = pow2_bits(127 - by);
      }
      own = odd ? own | 1 << buf : own & ~(1 << buf);
      if (lane == 0) scaled[buf] = 1;
    }
#pragma unroll
    for (int j = 0; j < NL; j++) {
      const float4 v = BF16B ? trunc_bf16(st[j]) : st[j];
      h4 hi, lo;
      _Float16 h, l;
      split_f16(v.x, bs, h, l); hi[0] = h; lo[0] = l;
      split_f16(v.y, bs, h, l); hi[1] = h; lo[1] = l;
      split_f16(v.z, bs, h, l); hi[2] = h; lo[2] = l;
      split_f16(v.w, bs, h, l); hi[3] = h; lo[3] = l;
      h4* dst = reinterpret_cast<h4*>(Bs + buf * PARTS * PART) + at0 + j * (16 * 16 * 2);
      dst[0] = hi;
      if (PARTS == 2) dst[PART * 2] = lo;
    }
  };
  lstore(0);
  gload(COLS);
  // A operand of K step ks: row r0 + 32 rb + lr, k = 16 ks + 8 lg .. +7; rows past M repeat row M - 1
  h8 ah[RBL][KS], al[RBL][KS];
#pragma unroll
  for (int rb = 0; rb < RBL; rb++) {
    const float* p = A + (size_t)min(r0 + 32 * rb + lr, M - 1) * D + 8 * lg;
    float4 v[2 * KS];
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < 2 * KS; i++) {
      v[i] = ldg4(p + 16 * (i >> 1) + 4 * (i & 1));
      m = fmaxf(m, max4abs(v[i]));
      bad |= odd4(v[i]);
    }
    m = max_xor32(m);
    const uint32_t e = float_exp(m);
    bad |= e > 250 || (e < 40 && m != 0.f);
    const float as = pow2_bits(e > 250 || e < 40 ? 127 : 127 + 12 + 127 - e);
#pragma unroll
    for (int i = 0; i < 2 * KS; i++) {
      const float x[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
      for (int j = 0; j < 4; j++) {
        _Float16 h, l;
        split_f16(x[j], as, h, l);
        ah[rb][i >> 1][4 * (i & 1) + j] = h;
        al[rb][i >> 1][4 * (i & 1) + j] = l;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  float bv[RBL];
  int bi[RBL];
#pragma unroll
  for (int rb = 0; rb < RBL; rb++) {
    bv[rb] = -INFINITY;
    bi[rb] = 0;
  }
  if (bad) redo[0] = 1;
  __syncthreads();
  auto multiply = [&](int buf, int n0, int factors) {
#pragma unroll
    for (int cb = 0; cb < CB; cb++) {
      f16v acc[RBL];
#pragma unroll
      for (int rb = 0; rb < RBL; rb++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[rb][i] = 0.f;
      const h8* bp = Bs + buf * PARTS * PART + (32 * (cb0 + cb) + lr) * 16;
      // each step's operands are read from LDS one step (3 RBL MFMAs) ahead
      h8 bh[2], bl[2];
      auto read = [&](int ks) {
        const int at = (2 * ks + lg) ^ (lr & 15);
        bh[ks & 1] = bp[at];
        if (PARTS == 2) bl[ks & 1] = bp[PART + at];
      };
      read(0);
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        if (ks + 1 < KS) read(ks + 1);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (PARTS == 2)
#pragma unroll
          for (int rb = 0; rb < RBL; rb++)
            acc[rb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bl[ks & 1], ah[rb][ks], acc[rb], 0, 0, 0);
#pragma unroll
        for (int rb = 0; rb < RBL; rb++)
          acc[rb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bh[ks & 1], al[rb][ks], acc[rb], 0, 0, 0);
#pragma unroll
        for (int rb = 0; rb < RBL; rb++)
          acc[rb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bh[ks & 1], ah[rb][ks], acc[rb], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (__builtin_expect(factors, 0)) {
#pragma unroll
        for (int i = 0; i < 16; i += 4) {
          const float4 c = *reinterpret_cast<const float4*>(&cscale[buf][32 * (cb0 + cb) + 2 * i + 4 * lg]);
#pragma unroll
          for (int rb = 0; rb < RBL; rb++) {
            acc[rb][i] *= c.x;
            acc[rb][i + 1] *= c.y;
            acc[rb][i + 2] *= c.z;
            acc[rb][i + 3] *= c.w;
          }
        }
      }
      // lane: row lr of the block, columns 8 (i / 4) + 4 lg + i % 4 of the 32, ascending in i, so
      // the first of equal scores is kept by "greater" over chunks and a descending search inside
#pragma unroll
      for (int rb = 0; rb < RBL; rb++) {
        float m = acc[rb][0];
#pragma unroll
        for (int i = 1; i < 16; i++) m = fmaxf(m, acc[rb][i]);
        if (m > bv[rb]) {
          int ix = 15;
#pragma unroll
          for (int i = 14; i >= 0; i--) ix = acc[rb][i] == m ? i : ix;
          bi[rb] = n0 + 32 * (cb0 + cb) + 8 * (ix >> 2) + 4 * lg + (ix & 3);
          bv[rb] = m;
        }
      }
    }
  };
  // Chunk ch + 1 is split into the other buffer while chunk ch is multiplied, by the first wave of
  // each SIMD (waves 0-3) before its products and by the second after, so one wave's vector work
  // runs beside the other's MFMAs.
  const int nchunks = (N + COLS - 1) / COLS;
  bool f32 = redo[0];  // workgroup-uniform
  int factors = __builtin_amdgcn_readfirstlane(scaled[0]);
  for (int ch = 0; ch < nchunks && !f32; ch++) {
    const int buf = ch & 1;
    if (wave < 4) {
      lstore(buf ^ 1);
      gload((ch + 2) * COLS);
      __builtin_amdgcn_sched_barrier(0);
    }
    multiply(buf, ch * COLS, factors);
    if (wave >= 4) {
      lstore(buf ^ 1);
      gload((ch + 2) * COLS);
    }
    if (bad) redo[(ch + 1) & 1] = 1;
    __syncthreads();
    f32 = redo[(ch + 1) & 1];
    factors = __builtin_amdgcn_readfirstlane(scaled[(ch + 1) & 1]);
  }
  if (f32) {
    for (int r = wg_r0; r < min(wg_r0 + wg_rows, M); r += 256) {
      __syncthreads();
      argmax_rows_f32<BF16B>(A, B, out, min(M, wg_r0 + wg_rows), N, r, lds);
    }
    return;
  }
  // the two lanes, and the WN waves, that hold parts of a row
#pragma unroll
  for (int rb = 0; rb < RBL; rb++) {
    const float w = __shfl_xor(bv[rb], 32);
    const int j = __shfl_xor(bi[rb], 32);
    amax_merge(bv[rb], bi[rb], w, j);
  }
  if constexpr (WN > 1) {  // the loop ended with a barrier: the chunks are no longer read
    float* sv = reinterpret_cast<float*>(lds);
    int* si = reinterpret_cast<int*>(sv + 8 * 32 * RBL);
#pragma unroll
    for (int rb = 0; rb < RBL; rb++)
      if (lg == 0) {
        sv[(wave * RBL + rb) * 32 + lr] = bv[rb];
        si[(wave * RBL + rb) * 32 + lr] = bi[rb];
      }
    __syncthreads();
    if (wave % WN) return;
#pragma unroll
    for (int rb = 0; rb < RBL; rb++)
      for (int w = 1; w < WN; w++)
        amax_merge(bv[rb], bi[rb], sv[((wave + w) * RBL + rb) * 32 + lr], si[((wave + w) * RBL + rb) * 32 + lr]);
  }
  if (lg == 0)
#pragma unroll
    for (int rb = 0; rb < RBL; rb++) {
      const int r = r0 + 32 * rb + lr;
      if (r < M) out[r] = (uint32_t)bi[rb];
    }
}

}  // namespace

namespace t5k {
namespace {
bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// compute units of the current device (cached per device; 256 if the query fails)
int num_cus() {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int v = cache[dev].load(std::memory_order_relaxed);
  if (v <= 0) {
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
    cache[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}
}  // namespace

hipError_t launch_matmul_t(const float* A, const float* B, float* C, int M, int N, int D, bool bf16_b,
                           hipStream_t s) {
  if (M <= 0 || N <= 0) return hipSuccess;
  if (D < 0) return hipErrorInvalidValue;
  const int mb = M >= 64 ? 4 : (M + 15) / 16;
  const int wn = N <= 64 ? 1 : 4, wm = 4 / wn;
  const long tiles_n = (N + 64L * wn - 1) / (64L * wn), tiles_m = (M + 16L * mb * wm - 1) / (16L * mb * wm);
  if (tiles_n * tiles_m > 0x7fffffffL) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(tiles_n * tiles_m));
  const bool vec = D % 4 == 0 && aligned16(A) && aligned16(B) && aligned16(C);
  // Few rows of A against a long B: the persistent streaming kernel in passes of 32 rows.  The passes
  // share two workgroups per CU, in whole groups of 8, so that the same columns meet in one XCD's L2 in
  // every pass; with two per CU for each pass they ran one after the other and read B again (33 x 50,000
  // 18.8 -> 15.0 us, 80 x 200,000 67 -> 54, 112 x 1,048,576 519 -> 382).  Streaming kernel / tiled
  // kernel: 32 x 1,000 5.9 / 8.9 us, 48 x 16,384 6.5 / 12.2, 64 x 65,536 15.7 / 18.6, 64 x 200,000 47 / 59,
  // 128 x 4,096 6.1 / 15.3; from 256 rows on the tiled kernel (256 x 16,384 19.5 / 19.1, 1,000 x 50,000
  // 215 / 182 before the passes shared).
  const bool rows16 = D % 4 == 0 && aligned16(A) && aligned16(B);
  bool stream = rows16 && D == 128 && M <= 128 && N >= 512 && 32L * N * 4 < (1L << 31);
  // 33 to 48 rows are three of the tiled kernel's row blocks but two passes: it takes them where its
  // rounds of 256 columns per CU, 13 us each, cost less than the streaming kernel's of 128, 6.1 us each
  // behind 3 us (40,000 columns 13.4 / 15.2 us, 80,000 25 / 20), and where B outgrows the last-level cache,
  // which the two passes then drift apart in (40 x 1,048,576 214 / 224).
  if (stream && mb == 3 && vec && N % 4 == 0) {
    const long cus = num_cus(), wide = (N + 256 * cus - 1) / (256 * cus), narrow = (N + 128 * cus - 1) / (128 * cus);
    stream = 13.0 * wide > 3 + 6.1 * narrow && (size_t)N * D * 4 < (size_t)384 << 20;
  }
  if (stream) {
    const int passes = mb == 1 ? 1 : (M + 31) / 32;
    const long per = passes == 1 ? 2L * num_cus() : std::max(8L, 2L * num_cus() / passes / 8 * 8);
    const dim3 g((unsigned)std::min<long>(per, (N + 127) / 128), (unsigned)passes);
    // scores past the caches as they are written: a store of whole 128-byte lines, and more of them than
    // the L2s would hold for a reader (16 x 262,144 34.9 -> 33.4 us, 32 x 1,048,576 140.5 -> 137; a row
    // that starts inside a line loses: see matmul_t_q4's rule)
    const bool nt = N % 32 == 0 && ((uintptr_t)C & 127) == 0 && (size_t)M * N * 4 >= (size_t)8 << 20;
#define T5K_STREAM(MBV, BF, NT) \
  hipLaunchKernelGGL((matmul_t_stream_kernel<MBV, BF, NT>), g, dim3(256), 0, s, A, B, C, M, N)
#define T5K_STREAM_NT(MBV, BF) \
  if (nt) T5K_STREAM(MBV, BF, true); \
  else T5K_STREAM(MBV, BF, false)
    if (mb == 1) {
      if (bf16_b) { T5K_STREAM_NT(1, true); } else { T5K_STREAM_NT(1, false); }
    } else {
      if (bf16_b) { T5K_STREAM_NT(2, true); } else { T5K_STREAM_NT(2, false); }
    }
#undef T5K_STREAM_NT
#undef T5K_STREAM
    return hipGetLastError();
  }
#define T5K_MMT(MBV, BF, VEC) \
  hipLaunchKernelGGL((matmul_t_kernel<MBV, BF, VEC>), grid, dim3(256), 0, s, A, B, C, M, N, D, wn, (int)tiles_n)
#define T5K_MMT_MB(BF, VEC)      \
  switch (mb) {                  \
    case 1: T5K_MMT(1, BF, VEC); break; \
    case 2: T5K_MMT(2, BF, VEC); break; \
    case 3: T5K_MMT(3, BF, VEC); break; \
    default: T5K_MMT(4, BF, VEC); break; \
  }
  if (bf16_b) {
    if (vec) { T5K_MMT_MB(true, true) } else { T5K_MMT_MB(true, false) }
  } else {
    if (vec) { T5K_MMT_MB(false, true) } else { T5K_MMT_MB(false, false) }
  }
#undef T5K_MMT_MB
#undef T5K_MMT
  return hipGetLastError();
}

hipError_t launch_matmul_argmax(const float* A, const float* B, uint32_t* out, int M, int N, int D, bool bf16_b,
                                hipStream_t s) {
  if (M <= 0) return hipSuccess;
  if (N <= 0 || D < 0) return hipErrorInvalidValue;
  const bool vec = D % 4 == 0 && aligned16(A) && aligned16(B);
  if (vec && D == 128) {
    // Rows per workgroup (one workgroup per CU at a time): a shorter tile re-splits B more often per
    // row but fills the chip with fewer rows.  Times of one round over 4,096 columns: 512 rows 279
    // us, 256 rows 190, 128 rows 110, 64 rows 80; the least rounds x time is taken (16,384 x 4,096:
    // 80 us on 64 rows, 97 on 128, 166 on 256, 258 on 512, 233 on the f32 kernel below).  256 rows are
    // eight waves of 32, each on all columns: four pairs of 64 rows that halve the columns read every row
    // of A twice, which bounds few columns (65,536 rows x 64 columns 11.4 us, by pairs 15.8, the f32
    // kernel 13.9; x 1,024 55 and 59; x 16,384 702 and 694).
    const long cus = num_cus();
    const double cost[4] = {279, 190, 110, 80};
    int v = 0;
    double best = 1e30;
    for (int i = 0; i < 4; i++) {
      const long rows = 512 >> i, wgs = (M + rows - 1) / rows;
      const double t = (double)((wgs + cus - 1) / cus) * cost[i];
      if (t < best) {
        best = t;
        v = i;
      }
    }
#define T5K_AMS(RBL, WN)                                                                                          \
  do {                                                                                                            \
    const dim3 g((M + 256 * RBL / WN - 1) / (256 * RBL / WN));                                                    \
    if (bf16_b)                                                                                                   \
      hipLaunchKernelGGL((matmul_argmax_split_kernel<true, RBL, WN>), g, dim3(512), 0, s, A, B, out, M, N);         \
    else                                                                                                          \
      hipLaunchKernelGGL((matmul_argmax_split_kernel<false, RBL, WN>), g, dim3(512), 0, s, A, B, out, M, N);        \
  } while (0)
    switch (v) {
      case 0: T5K_AMS(2, 1); break;
      case 1: T5K_AMS(1, 1); break;
      case 2: T5K_AMS(1, 2); break;
      default: T5K_AMS(1, 4); break;
    }
#undef T5K_AMS
    return hipGetLastError();
  }
  const dim3 grid((M + 63) / 64);
  if (bf16_b) {
    if (vec)
      hipLaunchKernelGGL((matmul_argmax_kernel<true, true>), grid, dim3(256), 0, s, A, B, out, M, N, D);
    else
      hipLaunchKernelGGL((matmul_argmax_kernel<true, false>), grid, dim3(256), 0, s, A, B, out, M, N, D);
  } else {
    if (vec)
      hipLaunchKernelGGL((matmul_argmax_kernel<false, true>), grid, dim3(256), 0, s, A, B, out, M, N, D);
    else
      hipLaunchKernelGGL((matmul_argmax_kernel<false, false>), grid, dim3(256), 0, s, A, B, out, M, N, D);
  }
  return hipGetLastError();
}
}  // namespace t5k
