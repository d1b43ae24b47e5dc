// k_pack.hip -- Witchcraft's packed chunk-embedding codec on the GPU, byte-exact with the
// reference: embeddings_to_packed / embeddings_from_packed (src/packops.rs:172-301, :303-438),
// haar_forward/inverse_mirror_edge (src/haarops.rs:4-70), rANS64 (src/rans64.rs, ryg_rans).
//
// A batch holds many matrices ([rows][cols] f32, cols <= 255); each is cut into windows of at
// most 1024 rows.  The host builds one PkWin per window (offsets only); every transform, the
// entropy coder and the assembly of the output bytes run here:
//   encode: pk_colsort (column sums in row order, stable rank sort, inverse permutation bytes)
//           -> pk_haar_rows (permute + row transform, one wave per row)
//           -> pk_haar_cols (column transform in LDS, 8 columns per workgroup)
//           -> pk_quant (max |x| < 1, symbols round(29 x) folded to unsigned, histogram over
//              the used symbol range in 8192-bin LDS passes, scale_histogram)
//           -> pk_rans_enc (one workgroup per window: one wave runs the state loop, the state as
//              two f64 integers, and writes 32-bit words backwards; the others stage its
//              per-position parameters in LDS)
//           -> pk_assemble (header pieces and stream copied to host-computed offsets).
//   decode: pk_rans_dec (slot table in LDS, one wave runs the state loop, values in reverse)
//           -> pk_haar_rows<inverse> -> pk_haar_cols<inverse> -> pk_unpermute_norm.
// rANS64 has one state per window and the format fixes one stream per window, so the coder
// runs one stream per workgroup; windows run in parallel.
//
// Float arithmetic follows the reference operation by operation (two roundings for a*b + c,
// sequential sums in the reference's order, correctly rounded division and square root), so
// the bytes match exactly.
#include "common.hpp"

#pragma clang fp contract(off)

namespace t5k {
// One window of one matrix.  Host-filled: row0 (first row in the batch's row space), rows,
// cols (all windows share it), hdr (byte offset of the window's header scratch slot), data
// (byte offset of its rANS scratch, capacity 2 * rows * cols + 16), plus the decoder's input
// offsets.  Kernel-filled: m (histogram size), dlen (stream bytes), err.
struct PkWin {
  int row0, rows;
  long long hdr, data;    // scratch offsets (encode) / input offsets of perm+pairs, stream (decode)
  int m, dlen, err, pad;  // filled by pk_quant / pk_rans_enc; decode: m and dlen are inputs
};
}  // namespace t5k

namespace {

using t5k::PkWin;

constexpr float INV_SQRT2 = 0.7071067811865475f;
constexpr int RANS_BITS = 12, RANS_TOTAL = 1 << RANS_BITS;
constexpr unsigned long long RANS_L = 1ull << 31;

enum PkErr : int { PK_OK = 0, PK_NAN = 1, PK_HIST = 2, PK_OVERFLOW = 3, PK_CORRUPT = 4 };

// ---- encode 1: column sums (each column summed in row order, as the reference's r-outer
// loop does), stable rank by sum, inverse permutation bytes.  One workgroup per window. ----
__global__ __launch_bounds__(256) void pk_colsort(const float* __restrict__ x, PkWin* __restrict__ win, int cols,
                                                   uint8_t* __restrict__ hdr_scratch, int* __restrict__ perm_out) {
  __shared__ float sums[256];
  PkWin& w = win[blockIdx.x];
  const int c = threadIdx.x;
  // identity first: with a NaN sum the ranks below may collide (the window then fails), and
  // every slot must still hold a valid column for the row pass
  perm_out[(size_t)blockIdx.x * 256 + c] = c < cols ? c : 0;
  if (c < cols) {
    const float* p = x + (size_t)w.row0 * cols + c;
    // The sum is a chain of adds in row order, and the loads were too, one round trip to memory per
    // row (192 us for windows of 512 rows): 32 rows are now read at once, the next 32 while these are added.
    constexpr int U = 32;
    float s = 0.f, v[U];
    const int full = w.rows / U * U;
    for (int r = 0; r < full; r += U) {
#pragma unroll
      for (int j = 0; j < U; j++) v[j] = p[(size_t)(r + j) * cols];
#pragma unroll
      for (int j = 0; j < U; j++) s += v[j];
    }
    for (int r = full; r < w.rows; r++) s += p[(size_t)r * cols];
    sums[c] = s;
  }
  __syncthreads();  // also orders the identity fill before the ranked writes
  if (c < cols) {
    const float s = sums[c];
    if (s != s) atomicMax(&w.err, (int)PK_NAN);  // partial_cmp().unwrap() panics on NaN
    int rank = 0;
    for (int j = 0; j < cols; j++) {
      const float t = sums[j];
      rank += (t < s || (t == s && j < c)) ? 1 : 0;
    }
    hdr_scratch[w.hdr + c] = (uint8_t)rank;          // inv_perm[c] = new position of column c
    perm_out[(size_t)blockIdx.x * 256 + rank] = c;   // perm[new] = original column
  }
}

// Haar forward / inverse of one length-n vector held in LDS (v, scratch t), by one wave.
template <bool INV>
__device__ void haar_wave(float* v, float* t, int n, int lane) {
  if (!INV) {
    int m = n;
    while (m > 1) {
      const int pairs = m / 2, odd = m & 1, nc = pairs + odd;
      for (int i = lane; i < pairs; i += 64) {
        const float a = v[2 * i], b = v[2 * i + 1];
        t[i] = (a + b) * INV_SQRT2;
        t[nc + i] = (a - b) * INV_SQRT2;
      }
      if (odd && lane == 0) {
        const float a = v[m - 1];
        t[pairs] = (a + a) * INV_SQRT2;
      }
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      for (int i = lane; i < m; i += 64) v[i] = t[i];
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      m = nc;
    }
  } else {
    int levels[12], nl = 0, m = n;
    levels[nl++] = m;
    while (m > 1) {
      m = m / 2 + (m & 1);
      levels[nl++] = m;
    }
    for (int l = nl - 1; l >= 1; l--) {
      const int np = levels[l - 1], odd = np & 1, pairs = np / 2, nc = pairs + odd;
      for (int i = lane; i < pairs; i += 64) {
        const float sum = v[i], diff = v[nc + i];
        t[2 * i] = (sum + diff) * INV_SQRT2;
        t[2 * i + 1] = (sum - diff) * INV_SQRT2;
      }
      if (odd && lane == 0) t[np - 1] = v[nc - 1] * INV_SQRT2;
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      for (int i = lane; i < np; i += 64) v[i] = t[i];
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// ---- encode 2 / decode 3: rows.  One wave per row (4 rows per workgroup).  Encode gathers
// the row through the column permutation first. ----
template <bool INV>
__global__ __launch_bounds__(256) void pk_haar_rows(const float* __restrict__ src, float* __restrict__ dst,
                                                     int total_rows, int cols, const int* __restrict__ row_win,
                                                     const int* __restrict__ perm) {
  __shared__ float buf[4][2][256];
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + wv;
  if (row >= total_rows) return;  // wave-uniform; only wave barriers follow
  float* v = buf[wv][0];
  float* t = buf[wv][1];
  const float* s = src + (size_t)row * cols;
  const int* pm = INV ? nullptr : perm + (size_t)row_win[row] * 256;
  for (int c = lane; c < cols; c += 64) {
    int sc = c;
    if (!INV) {
      sc = pm[c];
      sc = (unsigned)sc < (unsigned)cols ? sc : 0;
    }
    v[c] = s[sc];
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  haar_wave<INV>(v, t, cols, lane);
  for (int c = lane; c < cols; c += 64) dst[(size_t)row * cols + c] = v[c];
}

// ---- encode 3 / decode 4: columns, in place.  Workgroup = (window, 8 columns); one wave per
// column pair; columns of up to 1024 rows in LDS. ----
template <bool INV>
__global__ __launch_bounds__(256) void pk_haar_cols(float* __restrict__ x, const PkWin* __restrict__ win, int cols) {
  __shared__ float buf[8][2][1024];
  const PkWin& w = win[blockIdx.x];
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n = w.rows;
  for (int k = 0; k < 2; k++) {
    const int c = blockIdx.y * 8 + wv * 2 + k;
    if (c >= cols) break;  // wave-uniform
    float* v = buf[wv * 2 + k][0];
    float* t = buf[wv * 2 + k][1];
    float* col = x + (size_t)w.row0 * cols + c;
    for (int r = lane; r < n; r += 64) v[r] = col[(size_t)r * cols];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    haar_wave<INV>(v, t, n, lane);
    for (int r = lane; r < n; r += 64) col[(size_t)r * cols] = v[r];
  }
}

// f32 -> unsigned symbol exactly as packops.rs does it (round(29 x) folded; Rust's saturating
// float -> usize cast, then the wrapping cast to u16).
__device__ __forceinline__ uint32_t pk_symbol(float v) {
  const float q = roundf(29.0f * v);
  const float sf = 2.0f * fabsf(q) + (q < 0.0f ? 1.0f : 0.0f);
  unsigned long long s;
  if (!(sf >= 1.0f)) s = 0;
  else if (sf >= 18446744073709551616.0f) s = ~0ull;
  else s = (unsigned long long)sf;
  return (uint32_t)(uint16_t)(s > 0 ? s - 1 : 0);
}

// ---- encode 4: scaling, symbols, histogram, scale_histogram.  One 1024-thread workgroup per
// window, so the latency of its loads and of LDS atomics bounds it.  Values are read eight at a time per
// thread.  The counts of the QLOW lowest symbols, which nearly all values have, are kept per lane number
// (a wave adds to 64 different banks; on one counter its atomics serialise) and summed at the end; the
// rest, and every symbol past the first HBINS, are counted one counter per symbol. ----
constexpr int HBINS = 8192, QLOW = 64, QU = 8;
__global__ __launch_bounds__(1024) void pk_quant(const float* __restrict__ x, PkWin* __restrict__ win, int cols,
                                                  uint16_t* __restrict__ syms, uint8_t* __restrict__ hdr_scratch,
                                                  uint32_t* __restrict__ pairs_scratch) {
  __shared__ uint32_t hist[HBINS];
  __shared__ uint32_t low[QLOW * 64];
  __shared__ float red[32];
  __shared__ uint32_t ured[32];
  __shared__ uint32_t cnt_m;
  PkWin& w = win[blockIdx.x];
  const int n = w.rows * cols, tid = threadIdx.x, wid = tid >> 6, lane = tid & 63;
  const float* v = x + (size_t)w.row0 * cols;
  uint16_t* sy = syms + (size_t)w.row0 * cols;
  // max over |x| < 1 (exact in any order), floor 1e-5
  float am = 0.00001f;
  for (int i0 = tid; i0 < n; i0 += 1024 * QU) {
    float a[QU];
#pragma unroll
    for (int j = 0; j < QU; j++) a[j] = i0 + 1024 * j < n ? fabsf(v[i0 + 1024 * j]) : 0.f;
#pragma unroll
    for (int j = 0; j < QU; j++)
      if (a[j] < 1.0f && a[j] > am) am = a[j];
  }
  for (int i = tid; i < HBINS; i += 1024) hist[i] = 0;
  for (int i = tid; i < QLOW * 64; i += 1024) low[i] = 0;
  for (int o = 32; o > 0; o >>= 1) am = fmaxf(am, __shfl_xor(am, o));
  if (lane == 0) red[wid] = am;
  __syncthreads();
  if (tid == 0) {
    float m = red[0];
    for (int i = 1; i < 16; i++) m = fmaxf(m, red[i]);
    red[16] = __fdiv_rn(1.0f, m);
  }
  __syncthreads();
  const float inv = red[16];
  uint32_t ms = 0;
  for (int i0 = tid; i0 < n; i0 += 1024 * QU) {
    float a[QU];
#pragma unroll
    for (int j = 0; j < QU; j++) a[j] = i0 + 1024 * j < n ? v[i0 + 1024 * j] : 0.f;
#pragma unroll
    for (int j = 0; j < QU; j++)
      if (i0 + 1024 * j < n) {
        const uint32_t s = pk_symbol(a[j] * inv);
        sy[i0 + 1024 * j] = (uint16_t)s;
        ms = ms > s ? ms : s;
        if (s < QLOW) atomicAdd(&low[s * 64 + lane], 1u);
        else if (s < HBINS) atomicAdd(&hist[s], 1u);
      }
  }
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t t = __shfl_xor(ms, o);
    ms = ms > t ? ms : t;
  }
  if (lane == 0) ured[wid] = ms;
  if (tid == 0) cnt_m = 0;
  __syncthreads();
  for (int s = wid; s < QLOW; s += 16) {
    uint32_t c = low[s * 64 + lane];
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
    if (lane == 0) hist[s] = c;
  }
  uint32_t max_sym = ured[0];
  for (int i = 1; i < 16; i++) max_sym = max_sym > ured[i] ? max_sym : ured[i];
  __syncthreads();
  // histogram in passes of HBINS symbols (the first is there); the used symbols, in increasing
  // order, with counts
  uint32_t* pairs = pairs_scratch + (size_t)blockIdx.x * 4096 * 2;  // (symbol, count) then freq
  for (uint32_t base = 0; base <= max_sym; base += HBINS) {
    if (base > 0) {
      for (int i = tid; i < HBINS; i += 1024) hist[i] = 0;
      __syncthreads();
      for (int i = tid; i < n; i += 1024) {
        const uint32_t s = sy[i];
        if (s >= base && s < base + HBINS) atomicAdd(&hist[s - base], 1u);
      }
      __syncthreads();
    }
    // compact the non-zero bins in order: per-thread chunks of 8 bins, exclusive scan of counts
    const int b0 = tid * 8;
    int nz = 0;
    for (int b = b0; b < b0 + 8; b++) nz += hist[b] != 0;
    // block-wide exclusive scan of nz
    int incl = nz;
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(incl, o);
      if (lane >= o) incl += t;
    }
    if (lane == 63) ured[wid] = incl;
    __syncthreads();
    int before = cnt_m;
    for (int i = 0; i < wid; i++) before += ured[i];
    int pos = before + incl - nz;
    for (int b = b0; b < b0 + 8; b++)
      if (hist[b] && pos < 4096) {
        pairs[2 * pos] = base + b;
        pairs[2 * pos + 1] = hist[b];
        pos++;
      }
    __syncthreads();
    if (tid == 0) {
      int tot = 0;
      for (int i = 0; i < 16; i++) tot += ured[i];
      cnt_m += tot;
    }
    __syncthreads();
  }
  const int m = cnt_m;
  if (tid == 0) w.m = m;
  if (m > RANS_TOTAL) {  // scale_histogram asserts: more symbols than frequency slots
    if (tid == 0) atomicMax(&w.err, (int)PK_HIST);
    return;
  }
  // scale_histogram (packops.rs:31-103): 1 + floor(count * (4096 - m) / n) each, the deficit to
  // the largest remainders (stable: lower index first on ties), residue to the last maximum.
  const uint64_t total = (uint64_t)n, rest = (uint64_t)(RANS_TOTAL - m);
  __syncthreads();
  // Each remainder (below n, so 32 bits) is taken once, not by every symbol that ranks itself
  // against it: a 64-bit modulus is about 150 instructions.
  uint32_t *rem = hist, *freq = hist + 4096;  // reuse
  if (tid == 0) ured[0] = 0;
  __syncthreads();
  for (int i = tid; i < m; i += 1024) {
    const uint64_t a = (uint64_t)pairs[2 * i + 1] * rest;
    const uint32_t q = (uint32_t)(a / total);
    rem[i] = (uint32_t)(a - q * total);
    freq[i] = 1 + q;
    atomicAdd(&ured[0], q);
  }
  __syncthreads();
  const uint32_t deficit = (uint32_t)rest - ured[0];
  for (int i = tid; i < m; i += 1024) {
    const uint32_t ri = rem[i];
    uint32_t rank = 0;
    for (int j = 0; j < m; j++) {
      const uint32_t rj = rem[j];
      rank += (rj > ri || (rj == ri && j < i)) ? 1 : 0;
    }
    freq[i] += rank < deficit ? 1u : 0u;
  }
  __syncthreads();
  uint8_t* hdr = hdr_scratch + w.hdr;
  if (tid == 0) {
    int64_t tot = 0;
    int mi = 0;
    for (int i = 0; i < m; i++) {
      tot += freq[i];
      if (freq[i] >= freq[mi]) mi = i;
    }
    while (tot < RANS_TOTAL) {
      freq[mi]++;
      tot++;
    }
    while (tot > RANS_TOTAL && freq[mi] > 1) {
      freq[mi]--;
      tot--;
    }
  }
  __syncthreads();
  // header bytes after the permutation: u16 m, then (u16 symbol, u16 freq) pairs
  if (tid == 0) {
    hdr[256] = (uint8_t)m;
    hdr[257] = (uint8_t)(m >> 8);
  }
  for (int i = tid; i < m; i += 1024) {
    const uint32_t s = pairs[2 * i], f = freq[i];
    uint8_t* p = hdr + 258 + 4 * i;
    p[0] = (uint8_t)s;
    p[1] = (uint8_t)(s >> 8);
    p[2] = (uint8_t)f;
    p[3] = (uint8_t)(f >> 8);
    pairs[2 * i + 1] = f;  // now (symbol, freq)
  }
}

// ---- encode 5: rANS64, one workgroup per window.  The state x is a serial chain over the
// window's symbols, so what bounds the launch is the latency of one step of one wave, not a
// unit: 65,536 steps for 512 rows of 128.  The step, with f = freq and g = 4096 - f, is
//   q = floor(x / f),  x' = x + start + q g
// (the reference multiplies by a 64-bit reciprocal, rans64.rs:41-87; both divide exactly).  In
// integers the 64 x 64-bit high product alone is seven multiplies and their carries on the
// scalar unit.  f64 is full rate here, so x lives as two f64 integers, x = A 2^32 + B (A < 2^31,
// B < 2^32), and a step is 12 f64 instructions, each exact:
//   qA = floor(A / f), rA = A - qA f, t = rA 2^32 + B < 2^44, qB = floor(t / f) < 2^32,
//   u = t + start + qB g < 2^44, c = floor(u / 2^32), B' = u - c 2^32, A' = 4096 qA + c.
// floor(v / f) = floor(v * rf) with rf = 1 / f rounded up: a multiple of f cannot fall below its
// quotient, and any other v / f lies at least 1 / f >= 2^-12 under the next integer, against an
// error of at most 2^32 * 2^-51.  The renormalisation test x >= f 2^51 is A / f >= 2^19, i.e.
// A * rf >= 2^19 by the same argument.  Wave 0 runs the chain (all lanes alike); the other
// waves gather the next chunk's per-position parameters into LDS meanwhile.
// 48 windows of up to 512 rows: 8.07 -> 3.25 ms. ----
constexpr int ENC_CHUNK = 1024;
struct EncPos {
  double rf, f, g, start;
};

// Exclusive prefix sums of the window's m frequencies (freq(i), i < m <= 4096) by 256 threads, 16
// consecutive entries each, written as start | freq << 16; returns the total.
template <class Freq>
__device__ __forceinline__ uint32_t pk_starts(int m, Freq freq, uint32_t* out, uint32_t* red) {
  const int tid = threadIdx.x, wid = tid >> 6, lane = tid & 63;
  uint32_t f[16], sum = 0;
#pragma unroll
  for (int j = 0; j < 16; j++) {
    f[j] = 16 * tid + j < m ? freq(16 * tid + j) : 0;
    sum += f[j];
  }
  uint32_t incl = sum;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(incl, o);
    if (lane >= o) incl += t;
  }
  if (lane == 63) red[wid] = incl;
  __syncthreads();
  uint32_t at = incl - sum, total = 0;
  for (int i = 0; i < 4; i++) {
    if (i < wid) at += red[i];
    total += red[i];
  }
#pragma unroll
  for (int j = 0; j < 16; j++) {
    if (16 * tid + j < m) out[16 * tid + j] = (at & 0xffffu) | (f[j] << 16);
    at += f[j];
  }
  __syncthreads();
  return total;
}

__global__ __launch_bounds__(256) void pk_rans_enc(const uint16_t* __restrict__ syms, PkWin* __restrict__ win,
                                                    int cols, const uint32_t* __restrict__ pairs_scratch,
                                                    uint8_t* __restrict__ data_scratch) {
  __shared__ uint32_t table[RANS_TOTAL];  // start | freq << 16
  __shared__ uint16_t sym2idx[HBINS];
  __shared__ __attribute__((aligned(16))) EncPos stage[2][ENC_CHUNK + 8];
  __shared__ uint32_t red[4];
  PkWin& w = win[blockIdx.x];
  if (w.err) return;  // uniform
  const int m = w.m, n = w.rows * cols, tid = threadIdx.x;
  const uint32_t* pairs = pairs_scratch + (size_t)blockIdx.x * 4096 * 2;
  const uint16_t* sy = syms + (size_t)w.row0 * cols;
  pk_starts(m, [&](int i) { return pairs[2 * i + 1]; }, table, red);
  for (int i = tid; i < m; i += 256)
    if (pairs[2 * i] < HBINS) sym2idx[pairs[2 * i]] = (uint16_t)i;
  __syncthreads();
  auto fill = [&](int c0, int t0, int nt) {  // positions [c0, c0 + ENC_CHUNK) by threads t0 .. t0 + nt
    EncPos* st = stage[(c0 / ENC_CHUNK) & 1];
    for (int i = t0; i < min(ENC_CHUNK, n - c0); i += nt) {
      const uint32_t s = sy[c0 + i];
      int kk;
      if (s < HBINS) {
        kk = sym2idx[s];
      } else {  // rare large symbols: binary search in the sorted symbol list
        int lo = 0, hi = m - 1;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (pairs[2 * mid] < s) lo = mid + 1;
          else hi = mid;
        }
        kk = lo;
      }
      const uint32_t sf = table[kk];
      const double f = (double)(sf >> 16);
      double r = 1.0 / f;
      if (__builtin_fma(r, f, -1.0) < 0.0) r = __longlong_as_double(__double_as_longlong(r) + 1);
      st[i] = EncPos{r, f, 4096.0 - f, (double)(sf & 0xffffu)};
    }
  };
  fill(0, tid, 256);
  __syncthreads();
  // The encoder pushes symbols 0..n-1 in order.  The reference writes them backwards into a
  // buffer of 2n bytes (renormalisation needs 4 free bytes, the final flush 8, else it
  // panics); here word j (the j-th emitted) goes to out_words[cap_w - 1 - j] and the state
  // just before the last word, so the stream is contiguous: state, words k-1 .. 0.
  uint32_t* out_words = reinterpret_cast<uint32_t*>(data_scratch + w.data);
  const int cap_w = n / 2 + 4, cap_k = (2 * n) / 4;  // the reference's buffer holds cap_k whole words
  int k = 0;                                         // words emitted; past cap_k: the window fails
  double A = 0.0, B = (double)RANS_L;
  // One step of (a, b) given z = a * rf.
  auto push = [](const EncPos& e, double a, double b, double z, double& an, double& bn) {
    const double qa = __builtin_floor(z);
    const double ra = __builtin_fma(-qa, e.f, a);
    const double bs = b + e.start;
    const double t = __builtin_fma(ra, 4294967296.0, b), ts = __builtin_fma(ra, 4294967296.0, bs);
    const double qb = __builtin_floor(t * e.rf);
    const double u = __builtin_fma(qb, e.g, ts);
    const double c = __builtin_floor(u * 0x1p-32);
    bn = __builtin_fma(c, -4294967296.0, u);
    an = __builtin_fma(qa, 4096.0, c);
  };
  // The step is taken before the renormalisation test is known (a vector compare takes ~16 clk to
  // reach the scalar branch) and taken again in the 5% of positions that emit a word.
  auto step = [&](const EncPos& e) {
    double an, bn;
    const double z = A * e.rf;
    const unsigned long long full = __builtin_amdgcn_ballot_w64(z >= 524288.0);  // all lanes alike
    push(e, A, B, z, an, bn);
    asm volatile("" : "+v"(an), "+v"(bn));  // taken here, not behind the branch
    if (__builtin_expect(full != 0, 0)) {
      out_words[cap_w - 1 - min(k, cap_k)] = (uint32_t)B;  // a full buffer fails the window below
      k++;
      push(e, 0.0, A, 0.0, an, bn);
    }
    A = an;
    B = bn;
  };
  for (int c0 = 0; c0 < n; c0 += ENC_CHUNK) {
    if (__builtin_amdgcn_readfirstlane(tid >> 6) == 0) {
      const EncPos* st = stage[(c0 / ENC_CHUNK) & 1];
      const int cn = min(ENC_CHUNK, n - c0), full = cn & ~7;
      EncPos nx[8];  // the next 8 positions, read from LDS while 8 are coded
#pragma unroll
      for (int j = 0; j < 8; j++) nx[j] = st[j];
      for (int i = 0; i < full && k <= cap_k; i += 8) {
        EncPos cu[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
          cu[j] = nx[j];
          nx[j] = st[i + 8 + j];  // up to 8 past the chunk: inside the array, not used
        }
#pragma unroll
        for (int j = 0; j < 8; j++) step(cu[j]);
      }
      for (int i = full; i < cn; i++) step(st[i]);
    } else if (c0 + ENC_CHUNK < n) {
      fill(c0 + ENC_CHUNK, tid - 64, 192);
    }
    __syncthreads();
  }
  if (tid == 0) {
    if (2LL * n - 4LL * k < 8) {
      atomicMax(&w.err, (int)PK_OVERFLOW);
    } else {
      out_words[cap_w - 2 - k] = (uint32_t)B;
      out_words[cap_w - 1 - k] = (uint32_t)A;
      w.dlen = 8 + 4 * k;
      w.pad = (cap_w - 2 - k) * 4;  // stream start within the slot
    }
  }
}

// ---- encode 6: assemble.  out_off[window] = output byte offset of the window's pieces:
// perm bytes, u16 m + pairs, u16 dlen, stream.  One workgroup per window. ----
__global__ __launch_bounds__(256) void pk_assemble(const PkWin* __restrict__ win, int cols,
                                                    const uint8_t* __restrict__ hdr_scratch,
                                                    const uint8_t* __restrict__ data_scratch,
                                                    const long long* __restrict__ out_off, uint8_t* __restrict__ out) {
  const PkWin& w = win[blockIdx.x];
  uint8_t* o = out + out_off[blockIdx.x];
  const uint8_t* h = hdr_scratch + w.hdr;
  const int tid = threadIdx.x;
  for (int i = tid; i < cols; i += 256) o[i] = h[i];
  const int hb = 2 + 4 * w.m;
  for (int i = tid; i < hb; i += 256) o[cols + i] = h[256 + i];
  if (tid == 0) {
    o[cols + hb] = (uint8_t)w.dlen;  // `data.len() as u16`, as the reference writes it
    o[cols + hb + 1] = (uint8_t)(w.dlen >> 8);
  }
  const uint8_t* d = data_scratch + w.data + w.pad;
  for (int i = tid; i < w.dlen; i += 256) o[cols + hb + 2 + i] = d[i];
}

// The u32 row count that opens each packed matrix (native-endian, as `to_ne_bytes`).
__global__ void pk_headers(const long long* __restrict__ off, const int* __restrict__ rows, int B,
                           uint8_t* __restrict__ out) {
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b >= B) return;
  const uint32_t r = (uint32_t)rows[b];
  uint8_t* o = out + off[b];
  o[0] = (uint8_t)r;
  o[1] = (uint8_t)(r >> 8);
  o[2] = (uint8_t)(r >> 16);
  o[3] = (uint8_t)(r >> 24);
}

// ---- decode 2: rANS64, one workgroup per window.  As in the encoder the launch lasts as long as
// one wave's serial chain: slot c = x % 4096 names the symbol, x' = freq (x / 4096) + c - start.
// Every slot's freq and c - start sit in LDS, and the wave-uniform state stays on the vector unit:
// each trip of a value from the vector to the scalar unit costs ~16 clk and one back into an
// instruction's lane select or branch as much again, against ~5 clk for a dependent vector
// instruction and ~48 for the LDS read.  Slots are collected one lane per symbol and turned into
// values 64 at a time; the stream's words are held 64 at a time in a register as well.
// 48 windows of up to 512 rows (65,536 steps): 8.14 -> 3.26 ms. ----
__global__ __launch_bounds__(256) void pk_rans_dec(const uint8_t* __restrict__ in, PkWin* __restrict__ win, int cols,
                                                    float* __restrict__ out) {
  __shared__ uint2 slot[RANS_TOTAL];     // 8 freq, 8 (c - start)
  __shared__ float cum_v[RANS_TOTAL];
  __shared__ uint32_t runs[RANS_TOTAL];  // start | freq << 16 of each symbol
  __shared__ uint32_t red[4];
  PkWin& w = win[blockIdx.x];
  const int tid = threadIdx.x, n = w.rows * cols, m = w.m;
  // freq 4096 (a single symbol) needs 13 bits next to the 16-bit start: start | freq << 16
  const uint8_t* pairs = in + w.hdr + cols + 2;  // after perm bytes and u16 m
  auto freq = [&](int i) -> uint32_t { return pairs[4 * i + 2] | (pairs[4 * i + 3] << 8); };
  uint32_t* first = reinterpret_cast<uint32_t*>(cum_v);  // 1 + the symbol whose slots start here, or 0
  for (int c = tid; c < RANS_TOTAL; c += 256) first[c] = 0;
  // more symbols or a larger total than slots: the reference indexes past its tables
  const uint32_t total = m > RANS_TOTAL ? RANS_TOTAL + 1u : pk_starts(m, freq, runs, red);
  if (total > (uint32_t)RANS_TOTAL) {
    if (tid == 0) atomicMax(&w.err, (int)PK_CORRUPT);
    return;  // uniform
  }
  for (int i = tid; i < m; i += 256)
    if (runs[i] >> 16) first[runs[i] & 0xffffu] = i + 1;
  __syncthreads();
  // Each thread names the symbols of 16 slots: the last one that starts at or before a slot, from a
  // running maximum over the starts.  (One thread writing all slots of its symbol took 4,096 steps for
  // a window of one symbol: 5 rows of one value 338 -> 160 us a call.)
  uint32_t own[16], last = 0;
#pragma unroll
  for (int j = 0; j < 16; j++) {
    own[j] = first[16 * tid + j];
    last = max(last, own[j]);
  }
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(last, o);
    if ((tid & 63) >= o) last = max(last, t);
  }
  if ((tid & 63) == 63) red[tid >> 6] = last;
  last = __shfl_up(last, 1);
  if ((tid & 63) == 0) last = 0;
  __syncthreads();  // also: every thread has read its starts, which cum_v overwrites
  for (int i = 0; i < (tid >> 6); i++) last = max(last, red[i]);
#pragma unroll
  for (int j = 0; j < 16; j++) {
    const uint32_t c = 16 * tid + j;
    last = max(last, own[j]);
    uint32_t f = 1, start = 0, sym = 0;  // slots no symbol covers keep RansDecSymbol::new(0, 1) and 0.0
    if (c < total) {
      f = runs[last - 1] >> 16;
      start = runs[last - 1] & 0xffffu;
      sym = pairs[4 * (last - 1)] | (pairs[4 * (last - 1) + 1] << 8);
    }
    const uint32_t q = sym + 1;
    slot[c] = make_uint2(8 * f, 8 * (c - start));
    cum_v[c] = sym != 0 ? (1.0f / 29.0f) * ((q & 1) ? -1.0f : 1.0f) * (float)(q >> 1) : 0.f;
  }
  __syncthreads();
  if (tid >= 64) return;  // wave 0 alone from here: no barrier follows
  const int lane = tid;
  // The stream, read 4 bytes at a time from any byte offset: two aligned dwords funnel-
  // shifted (the input buffer carries 16 bytes of padding).
  const uint8_t* d = in + w.data;
  const int clen = w.dlen;
  auto word_at = [&](int p) -> uint32_t {
    const uintptr_t a = (uintptr_t)(d + p);
    const uint32_t* q = reinterpret_cast<const uint32_t*>(a & ~(uintptr_t)3);
    const unsigned long long two = ((unsigned long long)q[1] << 32) | q[0];
    return (uint32_t)(two >> (8 * (a & 3)));
  };
  // words 64 b .. 64 b + 63 after the state, one per lane; lanes past the stream re-read its end
  auto words = [&](int b) { return word_at(min(8 + 4 * (64 * b + lane), clen - 4)); };
  float* dst = out + (size_t)w.row0 * cols;
  unsigned long long x = (unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane(word_at(4)) << 32 |
                         (uint32_t)__builtin_amdgcn_readfirstlane(word_at(0));
  asm volatile("" : "+v"(x));  // wave-uniform, but kept on the vector unit: scalar crossings cost more
  uint32_t wcur = words(0), wnext = words(1);
  const int avail = (clen - 8) / 4;  // whole words after the state
  int used = 0;
  bool bad = false;
  // e: the entry of x's slot, already requested.  Only two instructions stand between an entry
  // and the request for the next one: the byte offset of x' % 4096 needs just the low bits of
  // q = x / 4096 (a 24-bit multiply-add of the entry's factors of 8) and a mask.  x' itself, the
  // renormalisation test and its branch run while the entry is on its way.
  auto lookup = [&](uint32_t v8) {
    return *reinterpret_cast<const uint2*>(reinterpret_cast<const char*>(slot) + (v8 & (8 * RANS_TOTAL - 8)));
  };
  uint2 e = lookup((uint32_t)x << 3);
  auto step = [&]() -> uint32_t {
    const uint32_t c = (uint32_t)x & (RANS_TOTAL - 1);
    const unsigned long long q = x >> RANS_BITS;
    const uint2 next = lookup((uint32_t)__umul24(e.x, (uint32_t)q) + e.y);
    const uint32_t f = e.x >> 3;
    const unsigned long long y = (unsigned long long)f * (uint32_t)q + (e.y >> 3);
    // q < 2^52 and freq < 2^13: the high product fits 24-bit operands
    typedef uint32_t u2v __attribute__((ext_vector_type(2)));
    x = __builtin_bit_cast(unsigned long long,
                           u2v{(uint32_t)y, (uint32_t)(y >> 32) + (uint32_t)__umul24(f, (uint32_t)(q >> 32))});
    e = next;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(x < RANS_L) != 0, 0)) {  // all lanes alike
      asm volatile("" : "+v"(e.x), "+v"(e.y));  // used on both sides, so requested before the branch
      if (used >= avail) bad = true;
      x = x << 32 | (uint32_t)__builtin_amdgcn_readlane(wcur, used & 63);
      if ((++used & 63) == 0) {
        wcur = wnext;
        wnext = words(used / 64 + 1);
      }
      if (__builtin_amdgcn_ballot_w64(x < RANS_L)) bad = true;
      e = lookup((uint32_t)x << 3);
    }
    return c;
  };
  // the j-th symbol decoded is position n - 1 - j
  int j0 = 0;
  // where the loop starts in a line of instructions moves its time by 3%: 512 rows 3.96 ms at 16 bytes
  // past a multiple of 32, 3.98 at such a multiple, up to 4.07 elsewhere
  asm volatile(".p2align 5\n\ts_nop 0\n\ts_nop 0\n\ts_nop 0\n\ts_nop 0");
  for (; j0 + 64 <= n && !bad; j0 += 64) {
    uint32_t slots = 0;
#pragma unroll
    for (int j = 0; j < 64; j++) {
      const uint32_t c = step();
      slots = lane == j ? c : slots;
    }
    dst[n - 1 - j0 - lane] = cum_v[slots];
  }
  if (j0 < n && !bad) {
    uint32_t slots = 0;
    for (int j = 0; j < n - j0; j++) {
      const uint32_t c = step();
      if (lane == j) slots = c;
    }
    if (lane < n - j0) dst[n - 1 - j0 - lane] = cum_v[slots];
  }
  if (tid == 0) {
    if (bad) atomicMax(&w.err, (int)PK_CORRUPT);
    w.pad = 8 + 4 * used;  // bytes consumed
  }
}

// Correctly rounded f32 square root (Rust's f32::sqrt): the hardware estimate (within 1 ulp)
// moved to the neighbour on the right side of the true root, decided by the exact residual
// x - s' s of each neighbour s' (one fused multiply-add each).  Inputs below 2^-96 are scaled
// by 2^32 first (the root by 2^-16 after; both exact) so the residuals stay normal.
__device__ __forceinline__ float sqrt_rn(float x) {
  if (!(x > 0.f) || x == __builtin_inff()) return __builtin_sqrtf(x);  // 0, inf, NaN, < 0
  const bool small = x < 0x1p-96f;
  const float xs = small ? x * 0x1p32f : x;
  float s = __builtin_amdgcn_sqrtf(xs);
  const float sd = __uint_as_float(__float_as_uint(s) - 1u), su = __uint_as_float(__float_as_uint(s) + 1u);
  const float rd = __builtin_fmaf(-sd, s, xs), ru = __builtin_fmaf(-su, s, xs);
  s = rd <= 0.f ? sd : s;
  s = ru > 0.f ? su : s;
  return small ? s * 0x1p-16f : s;
}

// ---- decode 5: undo the column permutation and L2-normalise each row (row norms summed
// sequentially in column order, as the reference's iterator sum).  One wave per row. ----
__global__ __launch_bounds__(256) void pk_unpermute_norm(float* __restrict__ x, int total_rows, int cols,
                                                          const int* __restrict__ row_win,
                                                          const uint8_t* __restrict__ in,
                                                          const PkWin* __restrict__ win) {
  __shared__ float buf[4][256];
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + wv;
  if (row >= total_rows) return;  // wave-uniform
  const uint8_t* idxs = in + win[row_win[row]].hdr;
  float* r = x + (size_t)row * cols;
  float* v = buf[wv];
  for (int c = lane; c < cols; c += 64) v[c] = r[idxs[c]];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  float ss = 0.f;
  if (lane == 0)
    for (int c = 0; c < cols; c++) ss += v[c] * v[c];
  ss = __shfl(ss, 0);
  const float inv = __fdiv_rn(1.0f, sqrt_rn(ss));
  for (int c = lane; c < cols; c += 64) r[c] = v[c] * inv;
}

}  // namespace

namespace t5k {

hipError_t pk_encode(const float* x, int total_rows, int cols, PkWin* win, int nwin, const int* row_win,
                     float* work, uint16_t* syms, int* perm, uint8_t* hdr, uint32_t* pairs, uint8_t* data,
                     hipStream_t s) {
  if (nwin == 0) return hipSuccess;
  hipLaunchKernelGGL(pk_colsort, dim3(nwin), dim3(256), 0, s, x, win, cols, hdr, perm);
  hipLaunchKernelGGL((pk_haar_rows<false>), dim3((total_rows + 3) / 4), dim3(256), 0, s, x, work, total_rows, cols,
                     row_win, perm);
  hipLaunchKernelGGL((pk_haar_cols<false>), dim3(nwin, (cols + 7) / 8), dim3(256), 0, s, work, win, cols);
  hipLaunchKernelGGL(pk_quant, dim3(nwin), dim3(1024), 0, s, work, win, cols, syms, hdr, pairs);
  hipLaunchKernelGGL(pk_rans_enc, dim3(nwin), dim3(256), 0, s, syms, win, cols, pairs, data);
  return hipGetLastError();
}

hipError_t pk_assemble_out(const PkWin* win, int nwin, int cols, const uint8_t* hdr, const uint8_t* data,
                           const long long* out_off, const long long* mat_off, const int* mat_rows, int B,
                           uint8_t* out, hipStream_t s) {
  if (B > 0) hipLaunchKernelGGL(pk_headers, dim3((B + 255) / 256), dim3(256), 0, s, mat_off, mat_rows, B, out);
  if (nwin > 0) hipLaunchKernelGGL(pk_assemble, dim3(nwin), dim3(256), 0, s, win, cols, hdr, data, out_off, out);
  return hipGetLastError();
}

hipError_t pk_decode(const uint8_t* in, int total_rows, int cols, PkWin* win, int nwin, const int* row_win,
                     float* out, float* work, hipStream_t s) {
  if (nwin == 0) return hipSuccess;
  hipLaunchKernelGGL(pk_rans_dec, dim3(nwin), dim3(256), 0, s, in, win, cols, work);
  hipLaunchKernelGGL((pk_haar_rows<true>), dim3((total_rows + 3) / 4), dim3(256), 0, s, work, out, total_rows, cols,
                     row_win, nullptr);
  hipLaunchKernelGGL((pk_haar_cols<true>), dim3(nwin, (cols + 7) / 8), dim3(256), 0, s, out, win, cols);
  hipLaunchKernelGGL(pk_unpermute_norm, dim3((total_rows + 3) / 4), dim3(256), 0, s, out, total_rows, cols, row_win,
                     in, win);
  return hipGetLastError();
}

}  // namespace t5k
