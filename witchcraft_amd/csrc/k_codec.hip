// k_codec.hip -- the residual codec of the XTR-WARP index next to the encoder, and scoring
// straight from its 4-bit codes.
//
// Reference (src/packops.rs, src/lib.rs):
//   * index build: residual = embedding - assigned centre, compand() (mu-law, :136-142),
//     quantize(4) (:156-162), to_q4_bytes (:440-462) -- src/lib.rs:1375-1376;
//   * search: from_companded_q4_bytes (:491-513) through make_q4_dequant_table (:14-25), then
//     matmul_t(query, residuals) -- src/lib.rs:626,676-680,734-735.
//
// Encoding never evaluates the mu-law on the GPU: compand().quantize(4) is a non-decreasing
// step function of the f32 input, so the host finds its 15 thresholds once (bisection over
// the ordered f32 values, evaluating the reference's own op sequence) and a code is the count
// of thresholds at or below the value -- exact by construction, NaN -> 0 as the clamp gives.
// Decoding is the reference's 16-entry table lookup.
//
// Scoring reads the codes, not decoded f32: a 128-d residual row is 64 bytes instead of 512,
// so the stream over residuals moves 8x fewer input bytes.  Products run on
// v_mfma_f32_16x16x4_f32 (exact f32 products, as the f32 path).
#include "common.hpp"

#include <algorithm>
#include <cstdlib>

namespace t5k {
struct Q4Table {
  float v[16];
};
struct Q4Ladder {
  float t[15];
};
}  // namespace t5k

namespace {

using t5k::Q4Ladder;
using t5k::Q4Table;

typedef float f4v __attribute__((ext_vector_type(4)));
constexpr int kBufDword3 = 0x00020000;  // raw buffer descriptor word 3: 32-bit data, OOB -> 0
constexpr int kBufNt = 2;               // buffer access policy bit: non-temporal

// The code of r: the number of thresholds t[0..14] (strictly increasing) at or below r, found
// by bisection -- 4 compares instead of 15.  code >= 8 iff r >= t[7]; then, from base i,
// code >= i + 4 iff r >= t[i + 3], and so on.  NaN compares false everywhere: code 0.
__device__ __forceinline__ uint32_t q4_code(float r, const float* t, float t7) {
  uint32_t i = r >= t7 ? 8u : 0u;
  i += r >= t[i + 3] ? 4u : 0u;
  i += r >= t[i + 1] ? 2u : 0u;
  i += r >= t[i] ? 1u : 0u;
  return i;
}

// One thread per 8 values (4 code bytes) of a row; D % 8 == 0.  Rows whose assignment is out
// of range get zero bytes and raise *bad.
__global__ __launch_bounds__(256) void residual_encode_kernel(const float* __restrict__ emb,
                                                              const float* __restrict__ centers,
                                                              const uint32_t* __restrict__ assign, int N, int D,
                                                              int K, Q4Ladder lad, uint8_t* __restrict__ out,
                                                              unsigned* __restrict__ bad) {
  __shared__ float tl[16];
  if (threadIdx.x < 15) tl[threadIdx.x] = lad.t[threadIdx.x];
  __syncthreads();
  const int groups = D / 8;
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (size_t)N * groups) return;
  const int row = (int)(idx / groups), g = (int)(idx % groups);
  const uint32_t a = assign[row];
  uint32_t word = 0;
  if (a < (uint32_t)K) {
    const float* e = emb + (size_t)row * D + 8 * g;
    const float* c = centers + (size_t)a * D + 8 * g;
    const float t7 = lad.t[7];
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      const uint32_t hi = q4_code(e[j] - c[j], tl, t7), lo = q4_code(e[j + 1] - c[j + 1], tl, t7);
      word |= ((hi << 4) | lo) << (4 * j);  // byte j/2: value j in the high nibble
    }
  } else if (g == 0) {
    atomicOr(bad, 1u);
  }
  *reinterpret_cast<uint32_t*>(out + (size_t)row * (D / 2) + 4 * g) = word;
}

// Byte offset into the heap of thresholds (T[1] = t[7], children of T[i] at 2 i and 2 i + 1, so
// T[8 .. 15] = t[0], t[2], ..) after one comparison: 4 (2 i + (r >= T[i])).  NaN compares false.
__device__ __forceinline__ uint32_t q4_step(uint32_t at, float r, float t) { return 2 * at + (r >= t ? 4u : 0u); }

// 4 x the code of r.  t1, t2, t3: the heap's first three entries, from registers.
__device__ __forceinline__ uint32_t q4_code4(float r, const float* heap, float t1, float t2, float t3) {
  const bool up = r >= t1;
  uint32_t at = q4_step(up ? 12u : 8u, r, up ? t3 : t2);
  at = q4_step(at, r, *reinterpret_cast<const float*>(reinterpret_cast<const char*>(heap) + at));
  at = q4_step(at, r, *reinterpret_cast<const float*>(reinterpret_cast<const char*>(heap) + at));
  return at - 64;
}

// 128-d rows by the hundred thousand, bound by the embeddings' one pass through memory: 32 lanes a
// row, four values a lane, so a wave's loads are contiguous, and two rows a thread, both rows' loads
// in flight before the first is used.  Codes are non-temporal, and so are the embeddings (NT) where
// that pays: rows that outgrow the 256 MB last-level cache, or centres that fill an XCD's 4 MB L2 and
// are kept there.  Otherwise rows that a caller has just written come faster from that cache: 400,000
// rows, 64 centres 33 us plain, 44 non-temporal (45 both when not cached), 300,000 rows, 8,192 centres
// 35.7 and 34.4, 16,384 centres 40.6 and 37.0.  1,000,003 rows, 16,384 centres: 134 us with a thread
// per eight values -> 116 us (5.0 TB/s; a large copy reaches 5.06 on the same card); one row a thread
// 172, three 124, four 123, plain code stores 119.
constexpr int kEncU = 2;  // rows per thread; a workgroup takes 8 kEncU rows
constexpr size_t kEncNtBytes = (size_t)256 << 20, kEncNtCentres = (size_t)4 << 20;
// From here on it is the faster one whether or not the rows are in the caches: 131,072 rows 19.6 us
// warm and 21.2 from memory against 18.8 and 18.9, 100,000 rows 13.1 and 16.1 against 13.5 and 14.1.
constexpr size_t kEncStreamRows = 131072;
template <bool NT>
__global__ __launch_bounds__(256) void residual_encode_stream_kernel(const float* __restrict__ emb,
                                                                     const float* __restrict__ centers,
                                                                     const uint32_t* __restrict__ assign, int N,
                                                                     int K, Q4Ladder lad, uint8_t* __restrict__ out,
                                                                     unsigned* __restrict__ bad) {
  constexpr int D = 128;
  typedef f4v f4u __attribute__((aligned(4)));
  __shared__ float heap[16];
  if (threadIdx.x >= 1 && threadIdx.x < 16) {
    const int i = threadIdx.x, level = 31 - __clz(i);
    heap[i] = lad.t[((2 * (i - (1 << level)) + 1) << (3 - level)) - 1];
  }
  __syncthreads();
  const int c = threadIdx.x & 31;
  const size_t first = (size_t)blockIdx.x * (8 * kEncU) + (threadIdx.x >> 5);
  const float t1 = lad.t[7], t2 = lad.t[3], t3 = lad.t[11];
  uint32_t a[kEncU];
  f4v e[kEncU], m[kEncU];
#pragma unroll
  for (int u = 0; u < kEncU; u++) a[u] = assign[min(first + 8 * u, (size_t)N - 1)];
#pragma unroll
  for (int u = 0; u < kEncU; u++) {
    const f4u* p = reinterpret_cast<const f4u*>(emb + min(first + 8 * u, (size_t)N - 1) * D + 4 * c);
    e[u] = NT ? __builtin_nontemporal_load(p) : *p;
  }
#pragma unroll
  for (int u = 0; u < kEncU; u++)
    m[u] = *reinterpret_cast<const f4u*>(centers + (size_t)(a[u] < (uint32_t)K ? a[u] : 0u) * D + 4 * c);
#pragma unroll
  for (int u = 0; u < kEncU; u++) {
    const size_t row = first + 8 * u;
    if (row >= (size_t)N) break;
    uint32_t q[4];
#pragma unroll
    for (int j = 0; j < 4; j++) q[j] = q4_code4(e[u][j] - m[u][j], heap, t1, t2, t3);
    uint32_t w = (q[0] << 2) | (q[1] >> 2) | (q[2] << 10) | (q[3] << 6);  // byte j / 2: value j in the high nibble
    if (a[u] >= (uint32_t)K) {
      w = 0;
      if (c == 0) atomicOr(bad, 1u);
    }
    __builtin_nontemporal_store((uint16_t)w, reinterpret_cast<uint16_t*>(out + row * (D / 2) + 2 * c));
  }
}

// from_companded_q4_bytes: one thread per 4 code bytes -> 8 floats.
__global__ __launch_bounds__(256) void residual_decode_kernel(const uint8_t* __restrict__ codes, size_t nbytes,
                                                              Q4Table tab, float* __restrict__ out) {
  __shared__ float lut[16];
  if (threadIdx.x < 16) lut[threadIdx.x] = tab.v[threadIdx.x];
  __syncthreads();
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= nbytes) return;
  float v[8];
  const int n = nbytes - i < 4 ? (int)(nbytes - i) : 4;
  for (int b = 0; b < n; b++) {
    const uint32_t x = codes[i + b];
    v[2 * b] = lut[x >> 4];
    v[2 * b + 1] = lut[x & 15];
  }
  for (int j = 0; j < 2 * n; j++) out[2 * i + j] = v[j];
}

// Query-sized A (16 MB <= 32 rows per grid row, D = 128) against N coded residual rows: the stream of
// matmul_t_stream_kernel (k_score.hip) over 64-byte code rows.  Wave w takes 32-row tiles
// w, w + W, ...; lane (lr, lg) owns rows lr and 16 + lr of a tile and their values
// k = 32 lg .. 32 lg + 31 (16 contiguous code bytes), which it feeds to the MFMAs as
// k = 32 lg + 4 s + j in step s; A is read from LDS with the same assignment, so every product
// appears once.  C[m][n] for rows n >= N is computed from zero bytes and never stored.
template <int MB>
struct Q4StreamLds {
  float4 As[16 * MB * (128 / 4 + 1)];
  float lut[16];
};

template <int MB>
__device__ __forceinline__ void q4_stream_f32(const float* __restrict__ A, const uint8_t* __restrict__ codes,
                                              const Q4Table& tab, float* __restrict__ C, int M, int N,
                                              Q4StreamLds<MB>& sh) {
  constexpr int D = 128, AS = D / 4 + 1;
  float4* As = sh.As;
  float* lut = sh.lut;
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int w0 = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = gridDim.x * 4;
  const int ntiles = (N + 31) / 32, nfull = N / 32, tail_bytes = (N % 32) * (D / 2);
  for (int e = threadIdx.x; e < 16 * MB * (D / 4); e += 256) {
    const int r = e / (D / 4), q = e - r * (D / 4);
    As[r * AS + q] = *reinterpret_cast<const float4*>(A + (size_t)min(r, M - 1) * D + 4 * q);
  }
  if (threadIdx.x < 16) lut[threadIdx.x] = tab.v[threadIdx.x];
  __syncthreads();
  const int voff[2] = {lr * (D / 2) + 16 * lg, (16 + lr) * (D / 2) + 16 * lg};
  auto load = [&](int t, uint4 (&b)[2]) {
    const int bytes = t < nfull ? 32 * (D / 2) : (t == nfull ? tail_bytes : 0);
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)(codes + (size_t)t * 32 * (D / 2)), (short)0, bytes, kBufDword3);
#pragma unroll
    for (int nb = 0; nb < 2; nb++) {
      const f4v v = __builtin_amdgcn_raw_buffer_load_b128(rs, voff[nb], 0, 0);
      b[nb] = __builtin_bit_cast(uint4, v);
    }
  };
  auto compute = [&](const uint4 (&b)[2], f4v (&acc)[MB][2]) {
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
      for (int nb = 0; nb < 2; nb++) acc[i][nb] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 8; s++)
#pragma unroll
      for (int nb = 0; nb < 2; nb++) {
        const uint32_t w = (s < 2 ? b[nb].x : s < 4 ? b[nb].y : s < 6 ? b[nb].z : b[nb].w) >> (16 * (s & 1));
        // bytes 2s (values 4s, 4s+1) and 2s+1 (values 4s+2, 4s+3): high nibble first
        const float v0 = lut[(w >> 4) & 15], v1 = lut[w & 15], v2 = lut[(w >> 12) & 15], v3 = lut[(w >> 8) & 15];
#pragma unroll
        for (int i = 0; i < MB; i++) {
          const float4 a = As[(16 * i + lr) * AS + 8 * lg + s];
          acc[i][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0, a.x, acc[i][nb], 0, 0, 0);
          acc[i][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1, a.y, acc[i][nb], 0, 0, 0);
          acc[i][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(v2, a.z, acc[i][nb], 0, 0, 0);
          acc[i][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(v3, a.w, acc[i][nb], 0, 0, 0);
        }
      }
  };
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
          __builtin_amdgcn_raw_buffer_store_b128(acc[i][nb], rs, soff[i] + 64 * nb, 0, 0);
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
  // Same issue order as matmul_t_stream_kernel: next tile's loads, previous tile's stores,
  // this tile's MFMAs, two tiles per trip.
  uint4 b0[2], b1[2];
  f4v acc0[MB][2], acc1[MB][2];
  int t = w0, t1 = -1;
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

template <int MB>
__global__ __launch_bounds__(256, 2) void matmul_t_q4_stream_kernel(const float* __restrict__ A,
                                                                    const uint8_t* __restrict__ codes, Q4Table tab,
                                                                    float* __restrict__ C, int M, int N) {
  __shared__ Q4StreamLds<MB> sh;
  A += (size_t)blockIdx.y * 16 * MB * 128;
  C += (size_t)blockIdx.y * 16 * MB * N;
  q4_stream_f32<MB>(A, codes, tab, C, min(M - (int)blockIdx.y * 16 * MB, 16 * MB), N, sh);
}

// The same stream on bf16 MFMAs.  v_mfma_f32_16x16x32_bf16 runs 8x the FLOPs of
// v_mfma_f32_16x16x4_f32 in half the cycles, so each f32 operand is split into three bf16
// parts, x = x_hi + x_mid + x_lo (round to nearest each; the parts hold 24 significant bits,
// |x - sum| <= 2^-27 |x|), and a product is taken as the six part products with i + j <= 2 --
// the three dropped ones are below 2^-25 |a t|.  Each part product is exact in f32, so the
// result stays within the f32 summation bound of the f32 kernel, at 6 x 16 = 96 cycles of
// matrix core per 16 x 16 x 32 block instead of 8 x 32 = 256.
//  * Residual side (A operand): a 256-entry LDS table maps a code byte to the split parts of
//    its two values, (t[hi nibble], t[lo nibble]) packed as bf16 pairs -- hi pair, mid pair,
//    lo pair -- so a lane's 8 values of a 32-wide K slice (4 code bytes) are 4 table reads and
//    no packing.  Lane (lr, lg) keeps the f32 kernel's rows lr and 16 + lr and bytes
//    16 lg .. 16 lg + 15 (k = 32 lg .. 32 lg + 31); K slice s uses bytes 16 lg + 4 s .. + 3,
//    i.e. k = 32 lg + 8 s + 0 .. 7 in MFMA slots 8 lg .. 8 lg + 7.
//  * Query side (B operand): the same k for query row lr, split once at kernel start and held
//    in registers (48 per 16 query rows).
//  * A query block with a non-finite value takes the f32 kernel instead: inf times a split
//    table value can meet parts of both signs and turn into NaN where f32 gives inf.
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint32_t bf16_rne_bits(float x) {
  const uint32_t u = __float_as_uint(x);
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;  // finite x
}
// x = hi + mid + lo as bf16 bit patterns
__device__ __forceinline__ void split3(float x, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  hi = bf16_rne_bits(x);
  const float r1 = x - __uint_as_float(hi << 16);
  mid = bf16_rne_bits(r1);
  const float r2 = r1 - __uint_as_float(mid << 16);
  lo = bf16_rne_bits(r2);
}

template <int MB, bool NT>
__global__ __launch_bounds__(256, 2) void matmul_t_q4_split_kernel(const float* __restrict__ A,
                                                                   const uint8_t* __restrict__ codes, Q4Table tab,
                                                                   float* __restrict__ C, int M, int N) {
  constexpr int D = 128;
  // 16 MB query rows per grid row
  A += (size_t)blockIdx.y * 16 * MB * D;
  C += (size_t)blockIdx.y * 16 * MB * N;
  M = min(M - (int)blockIdx.y * 16 * MB, 16 * MB);
  __shared__ uint4 pt[256];
  __shared__ Q4StreamLds<MB> sh;
  __shared__ int bad;
  if (threadIdx.x == 0) bad = 0;
  __syncthreads();
  {
    // byte x -> parts of (t[x >> 4], t[x & 15]); the first value takes the low half (lower k)
    const int x = threadIdx.x;
    uint32_t h0, m0, l0, h1, m1, l1;
    split3(tab.v[x >> 4], h0, m0, l0);
    split3(tab.v[x & 15], h1, m1, l1);
    pt[x] = make_uint4(h0 | (h1 << 16), m0 | (m1 << 16), l0 | (l1 << 16), 0u);
    // Non-finite values, and finite ones of magnitude >= 0x7f7f8000 (which round to a bf16
    // infinity in split3, so x - inf would give NaN), take the f32 kernel.
    // 16 bytes a load, all unconditional (row M - 1 stands for rows past it) and so all in flight at
    // once: one value a load under a row test took a trip to memory each, 32 x 4,096 8.1 -> 6.3 us.
    int nf = 0;
#pragma unroll
    for (int j = 0; j < 2 * MB; j++) {
      const int e = threadIdx.x + 256 * j;
      const float4 v = *reinterpret_cast<const float4*>(A + (size_t)min(e / (D / 4), M - 1) * D + 4 * (e % (D / 4)));
      const float big = __uint_as_float(0x7f7f8000u);
      if (!(fabsf(v.x) < big) || !(fabsf(v.y) < big) || !(fabsf(v.z) < big) || !(fabsf(v.w) < big)) nf = 1;
    }
    if (nf) bad = 1;  // every writer stores 1
  }
  __syncthreads();
  if (bad) {
    q4_stream_f32<MB>(A, codes, tab, C, M, N, sh);
    return;
  }
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int w0 = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = gridDim.x * 4;
  const int ntiles = (N + 31) / 32, nfull = N / 32, tail_bytes = (N % 32) * (D / 2);

  // query parts: q[i][s][p] = part p of query row 16 i + lr, k = 32 lg + 8 s .. + 7
  uint4 q[MB][4][3];
#pragma unroll
  for (int i = 0; i < MB; i++) {
    const float* row = A + (size_t)min(16 * i + lr, M - 1) * D + 32 * lg;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const float4 u = *reinterpret_cast<const float4*>(row + 8 * s);
      const float4 v = *reinterpret_cast<const float4*>(row + 8 * s + 4);
      const float x[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
      uint32_t hp[8], mp[8], lp[8];
#pragma unroll
      for (int j = 0; j < 8; j++) split3(x[j], hp[j], mp[j], lp[j]);
      q[i][s][0] = make_uint4(hp[0] | (hp[1] << 16), hp[2] | (hp[3] << 16), hp[4] | (hp[5] << 16), hp[6] | (hp[7] << 16));
      q[i][s][1] = make_uint4(mp[0] | (mp[1] << 16), mp[2] | (mp[3] << 16), mp[4] | (mp[5] << 16), mp[6] | (mp[7] << 16));
      q[i][s][2] = make_uint4(lp[0] | (lp[1] << 16), lp[2] | (lp[3] << 16), lp[4] | (lp[5] << 16), lp[6] | (lp[7] << 16));
    }
  }

  const int voff[2] = {lr * (D / 2) + 16 * lg, (16 + lr) * (D / 2) + 16 * lg};
  auto load = [&](int t, uint4 (&b)[2]) {
    const int bytes = t < nfull ? 32 * (D / 2) : (t == nfull ? tail_bytes : 0);
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)(codes + (size_t)t * 32 * (D / 2)), (short)0, bytes, kBufDword3);
#pragma unroll
    for (int nb = 0; nb < 2; nb++) {
      const f4v v = __builtin_amdgcn_raw_buffer_load_b128(rs, voff[nb], 0, 0);
      b[nb] = __builtin_bit_cast(uint4, v);
    }
  };
  auto mm = [](const uint4& a, const uint4& b, f4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8v, a), __builtin_bit_cast(bf8v, b), c, 0, 0, 0);
  };
  auto compute = [&](const uint4 (&b)[2], f4v (&acc)[MB][2]) {
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
      for (int nb = 0; nb < 2; nb++) acc[i][nb] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nb = 0; nb < 2; nb++)
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const uint32_t w = s == 0 ? b[nb].x : s == 1 ? b[nb].y : s == 2 ? b[nb].z : b[nb].w;
        const uint4 e0 = pt[w & 255], e1 = pt[(w >> 8) & 255], e2 = pt[(w >> 16) & 255], e3 = pt[w >> 24];
        const uint4 rh = make_uint4(e0.x, e1.x, e2.x, e3.x);
        const uint4 rm = make_uint4(e0.y, e1.y, e2.y, e3.y);
        const uint4 rl = make_uint4(e0.z, e1.z, e2.z, e3.z);
#pragma unroll
        for (int i = 0; i < MB; i++) {
          f4v c = acc[i][nb];
          c = mm(rh, q[i][s][0], c);
          c = mm(rh, q[i][s][1], c);
          c = mm(rm, q[i][s][0], c);
          c = mm(rh, q[i][s][2], c);
          c = mm(rm, q[i][s][1], c);
          c = mm(rl, q[i][s][0], c);
          acc[i][nb] = c;
        }
      }
  };
  // Whole tiles only when non-temporal (N % 32 == 0): lanes lr and lr ^ 8 trade a half tile, so that a
  // store instruction writes 8 rows of 128 bytes instead of 16 of 64.  Medians of alternating runs
  // when this came in: 32 x 65,536 11.2 -> 10.7 us, 50 x 200,000 33.6 -> 32.4, 32 x 1,048,576 60.5 -> 58.9;
  // 16 x 1,048,576 42.4 -> 42.8, 8 x 1,048,576 40.6 -> 40.4.  With the query check above: 32 x 1,048,576
  // 53 us on cached codes, 59 on new ones.
  const bool upper = lr >= 8;
  int soff[MB];
#pragma unroll
  for (int i = 0; i < MB; i++)
    soff[i] = NT ? ((16 * i + (lr & 7)) * N + (upper ? 16 : 0) + 4 * lg) * 4 : ((16 * i + lr) * N + 4 * lg) * 4;
  auto store = [&](int t, const f4v (&acc)[MB][2]) {
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)(C + (size_t)t * 32), (short)0, 0x7fffffff, kBufDword3);
    if constexpr (NT) {
#pragma unroll
      for (int i = 0; i < MB; i++) {
        f4v c0, c1;  // rows 16 i + lr % 8 and + 8, columns 16 .. 31 on the upper lanes
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const float x = upper ? acc[i][0][j] : acc[i][1][j];
          const float y = __int_as_float(
              __builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128 /* row_ror:8 */, 0xf, 0xf, false));
          c0[j] = upper ? y : acc[i][0][j];
          c1[j] = upper ? acc[i][1][j] : y;
        }
        if (16 * i + (lr & 7) < M) __builtin_amdgcn_raw_buffer_store_b128(c0, rs, soff[i], 0, kBufNt);
        if (16 * i + 8 + (lr & 7) < M) __builtin_amdgcn_raw_buffer_store_b128(c1, rs, soff[i] + 32 * N, 0, kBufNt);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < MB; i++) {
      const bool row_ok = 16 * i + lr < M;
#pragma unroll
      for (int nb = 0; nb < 2; nb++)
        if (row_ok && 32 * t + 16 * nb + 4 * lg + 3 < N)
          __builtin_amdgcn_raw_buffer_store_b128(acc[i][nb], rs, soff[i] + 64 * nb, 0, 0);
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
  // the f32 kernel's issue order: next tile's loads, previous tile's stores, this tile's MFMAs
  uint4 b0[2], b1[2];
  f4v acc0[MB][2], acc1[MB][2];
  int t = w0, t1 = -1;
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

// Any M, D % 4 == 0: 64 x 64 workgroup tiles (4 waves of 16 rows x 64 columns), each lane
// owning k = kb + 4 lg .. +3 of one A row and one code row per 16-block of K.
__global__ __launch_bounds__(256) void matmul_t_q4_kernel(const float* __restrict__ A,
                                                          const uint8_t* __restrict__ codes, Q4Table tab,
                                                          float* __restrict__ C, int M, int N, int D) {
  __shared__ float lut[16];
  if (threadIdx.x < 16) lut[threadIdx.x] = tab.v[threadIdx.x];
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int r0 = blockIdx.y * 64 + wave * 16, c0 = blockIdx.x * 64;
  if (r0 >= M) return;  // no barrier follows
  const int r = r0 + lr;
  const bool rok = r < M;
  const float* ar = A + (size_t)(rok ? r : 0) * D;
  const uint8_t* br[4];
  bool bok[4];
#pragma unroll
  for (int nb = 0; nb < 4; nb++) {
    const int c = c0 + 16 * nb + lr;
    bok[nb] = c < N;
    br[nb] = codes + (size_t)(bok[nb] ? c : 0) * (D / 2);
  }
  f4v acc[4];
#pragma unroll
  for (int nb = 0; nb < 4; nb++) acc[nb] = f4v{0.f, 0.f, 0.f, 0.f};
  for (int kb = 0; kb < D; kb += 16) {
    const int k = kb + 4 * lg;
    const bool kok = k < D;  // D % 4 == 0: a lane's 4 values are all in or all out
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    if (rok && kok) a = make_float4(ar[k], ar[k + 1], ar[k + 2], ar[k + 3]);  // any alignment
#pragma unroll
    for (int nb = 0; nb < 4; nb++) {
      float v[4] = {0.f, 0.f, 0.f, 0.f};
      if (bok[nb] && kok) {
        const uint32_t x0 = br[nb][k / 2], x1 = br[nb][k / 2 + 1];
        v[0] = lut[x0 >> 4];
        v[1] = lut[x0 & 15];
        v[2] = lut[x1 >> 4];
        v[3] = lut[x1 & 15];
      }
      acc[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[0], a.x, acc[nb], 0, 0, 0);
      acc[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[1], a.y, acc[nb], 0, 0, 0);
      acc[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[2], a.z, acc[nb], 0, 0, 0);
      acc[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[3], a.w, acc[nb], 0, 0, 0);
    }
  }
  // lane holds C[r0 + lr][c0 + 16 nb + 4 lg + 0..3]
  if (!rok) return;
#pragma unroll
  for (int nb = 0; nb < 4; nb++) {
    const int c = c0 + 16 * nb + 4 * lg;
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (c + i < N) C[(size_t)r * N + c + i] = acc[nb][i];
  }
}

int num_cus_codec() {
  static int cus = 0;
  if (!cus) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      cus = 256;
  }
  return cus;
}

}  // namespace

namespace t5k {

hipError_t launch_residual_encode(const float* emb, const float* centers, const uint32_t* assign, int N, int D,
                                  int K, const Q4Ladder& lad, uint8_t* out, unsigned* bad, hipStream_t s) {
  if (N <= 0) return hipSuccess;
  // Non-temporal code stores want whole 128-byte lines: a wave's two rows.
  if (D == 128 && (size_t)N >= kEncStreamRows && ((uintptr_t)out & 127) == 0) {
    const dim3 grid((unsigned)(((size_t)N + 8 * kEncU - 1) / (8 * kEncU)));
    const bool nt = (size_t)N * D * 4 >= kEncNtBytes || (size_t)K * D * 4 >= kEncNtCentres;
    if (nt) hipLaunchKernelGGL((residual_encode_stream_kernel<true>), grid, dim3(256), 0, s, emb, centers, assign, N, K,
                               lad, out, bad);
    else hipLaunchKernelGGL((residual_encode_stream_kernel<false>), grid, dim3(256), 0, s, emb, centers, assign, N, K,
                            lad, out, bad);
    return hipGetLastError();
  }
  const size_t threads = (size_t)N * (D / 8);
  hipLaunchKernelGGL(residual_encode_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, emb, centers,
                     assign, N, D, K, lad, out, bad);
  return hipGetLastError();
}

hipError_t launch_residual_decode(const uint8_t* codes, size_t nbytes, const Q4Table& tab, float* out,
                                  hipStream_t s) {
  if (nbytes == 0) return hipSuccess;
  const size_t threads = (nbytes + 3) / 4;
  hipLaunchKernelGGL(residual_decode_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, codes, nbytes,
                     tab, out);
  return hipGetLastError();
}

// C[M][N] = A[M][D] . decode(codes[N][D/2])^T.  D % 4 == 0.
hipError_t launch_matmul_t_q4(const float* A, const uint8_t* codes, const Q4Table& tab, float* C, int M, int N,
                              int D, hipStream_t s) {
  if (M <= 0 || N <= 0) return hipSuccess;
  // A long stream of 128-d codes takes the streaming kernels in passes of 32 query rows, at any N:
  // split kernel / tiled kernel below: 32 x 1,000 6.2 / 9.4 us, 48 x 16,384 6.7 / 10.4, 48 x 200,000
  // 26 / 64, 32 x 1,048,575 59 / 204, 1,000 x 16,384 69 / 97.  (Scores may start on any f32: 16-byte
  // buffer stores need 4-byte alignment only.)
  const bool aligned = ((uintptr_t)A & 15) == 0 && ((uintptr_t)codes & 15) == 0;
  const int mb = M <= 16 ? 1 : 2, passes = M <= 16 ? 1 : (M + 31) / 32;
  if (D == 128 && N >= 512 && passes <= 65535 && aligned && (size_t)N * 4 * 32 < 0x7fffffffu) {
    const int wgs = std::min(2 * num_cus_codec(), (N + 127) / 128);
    // Scores as non-temporal stores where every store fills whole 128-byte lines and the scores outgrow
    // what the L2s would keep for a reader anyway: twice the bytes of the codes at 32 rows, they otherwise
    // evict the codes of the next tiles (with 64-byte stores 32 x 1,048,576 76 -> 63 us, 16 x 262,144
    // 17.9 -> 16.3, 32 x 65,536 12.4 -> 11.7).  Rows that start inside a line lose, each half line going
    // out by itself (32 x 1,048,575 78 -> 131 us).
    const bool nt = N % 32 == 0 && ((uintptr_t)C & 127) == 0 && (size_t)M * N * 4 >= (size_t)8 << 20;
    // T5H_Q4_SCORE_F32=1 keeps the f32-MFMA stream (measurement and tests)
    static const bool f32_only = [] {
      const char* e = getenv("T5H_Q4_SCORE_F32");
      return e && atoi(e) == 1;
    }();
    const dim3 grid(wgs, passes);
#define T5K_Q4(...) hipLaunchKernelGGL((__VA_ARGS__), grid, dim3(256), 0, s, A, codes, tab, C, M, N)
    if (f32_only) {
      if (mb == 1) T5K_Q4(matmul_t_q4_stream_kernel<1>);
      else T5K_Q4(matmul_t_q4_stream_kernel<2>);
    } else if (mb == 1) {
      if (nt) T5K_Q4(matmul_t_q4_split_kernel<1, true>);
      else T5K_Q4(matmul_t_q4_split_kernel<1, false>);
    } else {
      if (nt) T5K_Q4(matmul_t_q4_split_kernel<2, true>);
      else T5K_Q4(matmul_t_q4_split_kernel<2, false>);
    }
#undef T5K_Q4
    return hipGetLastError();
  }
  const dim3 grid((N + 63) / 64, (M + 63) / 64);
  hipLaunchKernelGGL(matmul_t_q4_kernel, grid, dim3(256), 0, s, A, codes, tab, C, M, N, D);
  return hipGetLastError();
}

}  // namespace t5k
