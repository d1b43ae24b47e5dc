// k_gemm.hip -- the batched dense GEMMs on CDNA4 MFMA (v_mfma_f32_16x16x32_f16).
//
// C[M,N] = A[M,K] . W[N,K]^T, A = f16 activations (tokens x features).  Reference: every linear of
// the encoder, candle QMatMul / f32 matmul (src/quantized_t5.rs:383-424 QKV, :501 O, :231-252 FFN,
// :700 projection).
//
// Weights.  The matrix cores take f16(w) of the exact f32 weight, so launch_tile_weights forms that
// operand once, when the handle is made, from the Q4_K blocks (or f16 weights) and stores it, like
// the activations, in MFMA operand order (tiled_index): 2 bytes per weight next to the Q4_K blocks
// that the query path reads.  Unpacking inside the GEMM, by producer waves beside the math waves,
// left one math wave per SIMD: 590 us for gate|up at 74,640 tokens, 335 us for QKV.  Without it two
// or three workgroups share a CU: 451 and 263 us (1.04 and 1.00 PFLOP/s; the same products as a
// library f16 GEMM without epilogue run at 0.92 and 1.02).  All forms below take K in the same
// order, so every output has the same bits under any plan.
//
// Direct form (gemm_kernel): workgroup of 4 waves, each 16 MB tokens x all BN weight rows, K in
// steps of 64.  A goes from global memory straight to the wave's registers (no other wave needs it),
// one contiguous 1 KiB load per operand, one step ahead; the weight step, which all four waves
// read, goes global -> LDS without registers into the other half of a double buffer.  Bound at
// large M (gate|up, MB = 3, counters): MFMA busy 57% at the 1.7 GHz that power leaves, three waves
// per SIMD waiting to issue 57% of their cycles, vector-memory return path busy 93%.
//
// Ring form (ring_gemm_kernel): both operands through an LDS ring several steps deep, for launches
// with so few tiles that a step waits on memory: tiles of 32 x 64 to 128 x 128 tokens x rows.  A
// compute unit streams ~50 GB/s from the MALL whatever is in flight, so what bounds these launches
// is the bytes per tile (wo at 181 tokens, 32 x 64 tiles: 384 KB, 10.7 us; was 17 us).
#include "common.hpp"
#include "epilogue.hpp"

namespace {

constexpr int BK = 64;
constexpr int VMCNT0 = 0x0f70;  // s_waitcnt operand: vmcnt(0), the other counters unconstrained

// Global -> LDS loads as inline asm, invisible to the compiler's wait counts: it cannot tell the
// buffers apart and would wait for the copy just issued before each read.  The kernels order them:
// every copy of a step has landed (s_waitcnt vmcnt) before the barrier that publishes it, and every
// read of a buffer is complete before the barrier after which it is refilled; the "memory" clobbers
// keep each LDS access on its side.  M0 holds the wave's LDS destination; lane l's 16 bytes land at
// M0 + 16 l.  The source is a wave-uniform base (an SGPR pair) plus the lane's 32-bit offset.
__device__ __forceinline__ uint32_t lds_offset(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
__device__ __forceinline__ void lds_load16(const void* base, uint32_t voff, uint32_t m0) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(m0)
               : "memory", "m0");
}

// Byte address of block (row block i of a tile at n0, k 0 .. 31) of the weights.  Gated: blocks
// [0, NB / 2) are gate rows n0 .., blocks [NB / 2, NB) the up rows of the same columns.
template <int EPI, int NB>
__device__ __forceinline__ const char* wblock(const GemmArgs& p, int n0, int i) {
  const void* W = p.W0;
  int n = n0 / 16 + i;
  if (EPI == EPI_GATED) {
    W = i < NB / 2 ? p.W0 : p.W1;
    n = n0 / 16 + i % (NB / 2);
  }
  return reinterpret_cast<const char*>(W) + (size_t)n * (p.K / 32) * 1024;
}

template <int EPI, int BN, int MB>
__device__ __forceinline__ void gemm_tile(const GemmArgs& p, int m0, int n0, _Float16 (*Bs)[BN * BK]) {
  constexpr int NB = BN / 16, ND = 2 * NB / 4;  // 1 KiB copies per wave and step
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane & 15, lg = lane >> 4, nkt = p.K / BK;
  const uint32_t lane16 = 16u * lane;
  // copy j of this wave: stage block i = wave ND + j, i.e. row block i / 2, k half i % 2
  const char* wsrc[ND];
#pragma unroll
  for (int j = 0; j < ND; j++) wsrc[j] = wblock<EPI, NB>(p, n0, (wave * ND + j) >> 1) + ((wave * ND + j) & 1) * 1024;
  const uint32_t ldst = lds_offset(&Bs[0][0]) + wave * ND * 1024;
#define DMA(kt, slot)                                                                     \
  _Pragma("unroll") for (int j = 0; j < ND; j++)                                           \
      lds_load16(wsrc[j] + (size_t)(kt) * 2048, lane16, ldst + (slot) * (BN * BK * 2) + j * 1024);
  DMA(0, 0);
  // operand blocks of this wave's MB row groups; wave-uniform bases plus the lane's 16 bytes
  const size_t kblk = p.K / 32;
  const _Float16* ablk[MB];
  const int mrow0 = m0 + wave * 16 * MB;
#pragma unroll
  for (int mb = 0; mb < MB; mb++) ablk[mb] = p.A + ((size_t)(mrow0 / 16 + mb) * kblk) * 512;
  uint32_t alane = 16u * lane;
  f4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int j = 0; j < NB; j++) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
  // folded T5LayerNorm: the records are requested ahead of the first A loads
  const bool fold = EPI != EPI_RESID && p.rec != nullptr;
  float4 nrec[4];
  if (fold) norm_rec_load<MB>(p, mrow0, nrec);
  uint4 a[2][MB][2];  // steps kt and kt + 1
#define LOAD_A(st, kt)                                                                      \
  asm volatile("" : "+v"(alane));                                                            \
  _Pragma("unroll") for (int mb = 0; mb < MB; mb++) {                                        \
    a[st][mb][0] = *reinterpret_cast<const uint4*>(                                          \
        reinterpret_cast<const char*>(ablk[mb] + (size_t)(2 * (kt)) * 512) + alane);           \
    a[st][mb][1] = *reinterpret_cast<const uint4*>(                                          \
        reinterpret_cast<const char*>(ablk[mb] + (size_t)(2 * (kt) + 1) * 512) + alane);       \
  }
  LOAD_A(0, 0);
  const float fs = fold ? norm_factor<MB>(p, mrow0, n0, nrec) : 1.f;
  // vmcnt(0) through the builtin, so that the compiler knows its operand loads are complete too and
  // adds no wait of its own behind the next step's copies
  __builtin_amdgcn_s_waitcnt(VMCNT0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  const _Float16* bbase = &Bs[0][0] + lane * 8;
  for (int kt0 = 0; kt0 < nkt; kt0 += 2) {
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int kt = kt0 + u;
      const int kn = min(kt + 1, nkt - 1);
      DMA(kn, u ^ 1);
      LOAD_A(u ^ 1, kn);
      __builtin_amdgcn_sched_barrier(0);  // requested before this step's MFMAs
      const _Float16* bsrc = bbase + u * (BN * BK);
      // Weight fragments j = s * NB + nb in order, each read FD fragments ahead of its MFMAs so that
      // the LDS latency hides behind the MFMAs of the fragments before it
      constexpr int NF = 2 * NB, FD = 2;
      h8 wf[FD + 1];
#pragma unroll
      for (int j = 0; j < FD; j++)
        wf[j] = *reinterpret_cast<const h8*>(bsrc + ((j % NB) * 2 + j / NB) * 512);
#pragma unroll
      for (int j = 0; j < NF; j++) {
        if (j + FD < NF)
          wf[(j + FD) % (FD + 1)] =
              *reinterpret_cast<const h8*>(bsrc + (((j + FD) % NB) * 2 + (j + FD) / NB) * 512);
        const int s = j / NB, nb = j % NB;
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
          acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[j % (FD + 1)], __builtin_bit_cast(h8, a[u][mb][s]),
                                                                acc[mb][nb], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(VMCNT0);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
  }
#undef LOAD_A
#undef DMA

  // ---- epilogue: lane holds C[token mrow0 + 16 mb + lr][columns n0 + 16 nb + 4 lg + 0..3] ----
  if constexpr (EPI == EPI_RESID) {
    resid_store_tile<BN, MB>(p, mrow0, n0, acc);
    return;
  } else if (fold) {
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
      const float f = __shfl(fs, mb * 16 + lr);
#pragma unroll
      for (int nb = 0; nb < NB; nb++) acc[mb][nb] *= f;
    }
  }
  if constexpr (EPI == EPI_QKV) {
    if (p.dkv == 64) {  // every 64-column group of the tile is one head: full-row stores
      qkv_store_staged<BN, MB>(p, mrow0, n0, acc, &Bs[0][0] + wave * (16 * (BN + 8)));
      return;
    }
  }
#pragma unroll
  for (int mb = 0; mb < MB; mb++) {
    const int m = mrow0 + mb * 16 + lr;
    if (m >= p.M) continue;
    if constexpr (EPI == EPI_GATED) {
#pragma unroll
      for (int nb = 0; nb < NB / 2; nb++)
        store_quad_gated(p, m, n0 + nb * 16 + 4 * lg, acc[mb][nb], acc[mb][nb + NB / 2]);
    } else {
#pragma unroll
      for (int nb = 0; nb < NB; nb++) store_quad<EPI>(p, m, n0 + nb * 16 + 4 * lg, acc[mb][nb]);
    }
  }
}

// Tiles are ordered so that each XCD (8 per device, workgroups dealt round-robin) works on a
// contiguous band of them: its L2 holds the A rows it streams plus the weights.
__device__ __forceinline__ int xcd_tile() { return (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8; }

template <int EPI, int BN, int MB>
__global__ __launch_bounds__(256, 2) void gemm_kernel(GemmArgs p, int tiles_n, int tiles) {
  __shared__ __attribute__((aligned(16))) _Float16 Bs[2][BN * BK];
  constexpr int cols = EPI == EPI_GATED ? BN / 2 : BN;  // output columns per tile
  const int tile = xcd_tile();
  if (tile >= tiles) return;
  gemm_tile<EPI, BN, MB>(p, (tile / tiles_n) * 64 * MB, (tile % tiles_n) * cols, Bs);
}

// Ring form: WR x WC waves, each 16 MB tokens x 16 NB rows (NB = 4: a wave's columns are one
// 64-column group of the norm records and one head); S steps of H 32-wide K slices in flight.  A
// slice's operands are read from LDS while the slice before is multiplied; the wait and barrier for
// the next step come before the last slice's MFMAs, and the slot just read is refilled at once.
template <int EPI, int MB, int NB, int WR, int WC, int S, int H>
__global__ __launch_bounds__(64 * WR * WC) void ring_gemm_kernel(GemmArgs p, int tiles_n, int tiles) {
  constexpr int NW = WR * WC, AB = H * MB * WR, BB = H * NB * WC, NBLK = AB + BB, ND = NBLK / NW;
  static_assert(NBLK % NW == 0 && H % 2 == 0, "whole copies per wave, an even number of slices");
  __shared__ __attribute__((aligned(1024))) _Float16 Rs[S][NBLK * 512];
  constexpr int cols = EPI == EPI_GATED ? 8 * NB * WC : 16 * NB * WC;
  const int tile = xcd_tile();
  if (tile >= tiles) return;
  const int m0 = (tile / tiles_n) * 16 * MB * WR, n0 = (tile % tiles_n) * cols;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane & 15, lg = lane >> 4, wr = wave / WC, wc = wave % WC;
  const int nkt = p.K / (32 * H), mrow0 = m0 + wr * 16 * MB, nw0 = n0 + wc * (cols / WC);
  const bool fold = EPI != EPI_RESID && p.rec != nullptr;
  float4 nrec[4];
  if (fold) norm_rec_load<MB>(p, mrow0, nrec);
  const uint32_t lane16 = 16u * lane;
  const char* src[ND];
#pragma unroll
  for (int j = 0; j < ND; j++) {
    const int i = wave * ND + j, w = i - AB;
    src[j] = (i < AB ? reinterpret_cast<const char*>(p.A) + (size_t)(m0 / 16 + i / H) * (p.K / 32) * 1024
                     : wblock<EPI, NB>(p, n0 + (w / (H * NB)) * (cols / WC), (w / H) % NB)) +
             (i % H) * 1024;
  }
  const uint32_t ldst = lds_offset(&Rs[0][0]) + wave * ND * 1024;
  auto copy = [&](int kt, int slot) {
#pragma unroll
    for (int j = 0; j < ND; j++)
      lds_load16(src[j] + (size_t)kt * (1024 * H), lane16, ldst + slot * (NBLK * 1024) + j * 1024);
  };
#pragma unroll
  for (int i = 0; i < S; i++)
    if (i < nkt) copy(i, i);
  f4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int j = 0; j < NB; j++) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
  h8 af[2][MB], wf[2][NB];
  const _Float16* abase = &Rs[0][0] + wr * MB * H * 512 + lane * 8;
  const _Float16* bbase = &Rs[0][AB * 512] + wc * NB * H * 512 + lane * 8;
  auto read = [&](int slot, int h, int st) {
    const int o = slot * (NBLK * 512);
#pragma unroll
    for (int i = 0; i < MB; i++) af[st][i] = *reinterpret_cast<const h8*>(abase + o + (H * i + h) * 512);
#pragma unroll
    for (int i = 0; i < NB; i++) wf[st][i] = *reinterpret_cast<const h8*>(bbase + o + (H * i + h) * 512);
  };
  // Step kt of the `ahead` steps kt, kt + 1, .. requested so far has landed, and this wave's reads
  // are complete; after the barrier every wave's are.
  auto arrive = [&](int kt, int ahead) {
    if (kt + ahead <= nkt) {
      if (ahead == S) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S - 1) * ND) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S - 2) * ND) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    }
    if (NW > 1) asm volatile("s_barrier" ::: "memory");
  };
  arrive(0, S);
  read(0, 0, 0);
  int slot = 0;
  for (int kt = 0; kt < nkt; kt++) {
#pragma unroll
    for (int h = 0; h < H; h++) {
      if (h < H - 1) {
        read(slot, h + 1, (h + 1) & 1);
      } else if (kt + 1 < nkt) {
        arrive(kt + 1, S - 1);
        if (kt + S < nkt) copy(kt + S, slot);
        slot = slot + 1 == S ? 0 : slot + 1;
        read(slot, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int nb = 0; nb < NB; nb++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
          acc[mb][nb] =
              __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[h & 1][nb], af[h & 1][mb], acc[mb][nb], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if constexpr (EPI == EPI_RESID) {
    resid_store_tile<16 * NB, MB>(p, mrow0, nw0, acc);
    return;
  } else if (fold) {
    const float fs = norm_factor<MB>(p, mrow0, nw0, nrec);
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
      const float f = __shfl(fs, mb * 16 + lr);
#pragma unroll
      for (int nb = 0; nb < NB; nb++) acc[mb][nb] *= f;
    }
  }
  if constexpr (EPI == EPI_QKV) {
    if (p.dkv == 64 && NB % 4 == 0) {
      if (NW > 1) asm volatile("s_barrier" ::: "memory");  // the ring is no longer read
      qkv_store_staged<16 * NB, MB>(p, mrow0, nw0, acc, &Rs[0][0] + wave * (16 * (16 * NB + 8)));
      return;
    }
  }
#pragma unroll
  for (int mb = 0; mb < MB; mb++) {
    const int m = mrow0 + mb * 16 + lr;
    if (m >= p.M) continue;
    if constexpr (EPI == EPI_GATED) {
#pragma unroll
      for (int nb = 0; nb < NB / 2; nb++)
        store_quad_gated(p, m, nw0 + nb * 16 + 4 * lg, acc[mb][nb], acc[mb][nb + NB / 2]);
    } else {
#pragma unroll
      for (int nb = 0; nb < NB; nb++) store_quad<EPI>(p, m, nw0 + nb * 16 + 4 * lg, acc[mb][nb]);
    }
  }
}

template <int EPI, int BN, int MB>
hipError_t launch_direct(const GemmArgs& a, hipStream_t s) {
  constexpr int cols = EPI == EPI_GATED ? BN / 2 : BN;
  const int tiles_n = a.N / cols, tiles = (a.M + 64 * MB - 1) / (64 * MB) * tiles_n;
  T5K_LAUNCH((gemm_kernel<EPI, BN, MB>), dim3((tiles + 7) / 8 * 8), dim3(256), 0, s, a, tiles_n, tiles);
  return hipGetLastError();
}

template <int EPI, int MB, int NB, int WR, int WC, int S, int H>
hipError_t launch_ring(const GemmArgs& a, hipStream_t s) {
  constexpr int cols = EPI == EPI_GATED ? 8 * NB * WC : 16 * NB * WC, bm = 16 * MB * WR;
  const int tiles_n = a.N / cols, tiles = (a.M + bm - 1) / bm * tiles_n;
  T5K_LAUNCH((ring_gemm_kernel<EPI, MB, NB, WR, WC, S, H>), dim3((tiles + 7) / 8 * 8), dim3(64 * WR * WC), 0, s, a,
             tiles_n, tiles);
  return hipGetLastError();
}

template <int EPI>
hipError_t launch_epi(int variant, const GemmArgs& a, hipStream_t s) {
  using namespace t5k;
  switch (variant) {
    case GEMM_RING_32X64: return launch_ring<EPI, 1, 4, 2, 1, 4, 4>(a, s);
    case GEMM_RING_64X64: return launch_ring<EPI, 1, 4, 4, 1, 3, 4>(a, s);
    case GEMM_RING_128X64: return launch_ring<EPI, 2, 4, 4, 1, 3, 4>(a, s);
    case GEMM_RING_128X128: return launch_ring<EPI, 2, 4, 4, 2, 4, 2>(a, s);
    case GEMM_RING_128X128_2: return launch_ring<EPI, 2, 4, 4, 2, 2, 2>(a, s);
    case GEMM_128X128: return launch_direct<EPI, 128, 2>(a, s);
    case GEMM_192X128: return launch_direct<EPI, 128, 3>(a, s);
    case GEMM_256X128: return launch_direct<EPI, 128, 4>(a, s);
    case GEMM_64X128: return launch_direct<EPI, 128, 1>(a, s);
    case GEMM_256X64: return launch_direct<EPI, 64, 4>(a, s);
  }
  return hipErrorInvalidValue;
}

// W (Q4_K blocks or f16 [N][K]) -> the f16 operand in operand order; a thread forms 8 consecutive
// values of one row.  Q4_K: (d sc) q - dmin m, both products exact in f32, rounded once to f16.
template <bool Q4K>
__global__ __launch_bounds__(256) void tile_weights_kernel(const void* __restrict__ w, int N, int K,
                                                           _Float16* __restrict__ out) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;  // 8 consecutive values of one row
  if (i >= (size_t)N * K / 8) return;
  const int n = (int)(i / (K / 8)), k = (int)(i % (K / 8)) * 8;
  h8 v;
  if constexpr (Q4K) {
    const uint8_t* b = (const uint8_t*)w + ((size_t)n * (K / QK_K) + k / QK_K) * Q4K_BYTES;
    const uint16_t dh = (uint16_t)b[0] | ((uint16_t)b[1] << 8), mh = (uint16_t)b[2] | ((uint16_t)b[3] << 8);
    const int j = (k % QK_K) / 32, q0 = k % 32;
    int sc, m;
    const uint8_t* s = b + 4;
    if (j < 4) {
      sc = s[j] & 63;
      m = s[j + 4] & 63;
    } else {
      sc = (s[j + 4] & 15) | ((s[j - 4] >> 6) << 4);
      m = (s[j + 4] >> 4) | ((s[j] >> 6) << 4);
    }
    const float d = f16_bits_to_f32(dh) * (float)sc, o = f16_bits_to_f32(mh) * (float)m;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const uint8_t q = b[16 + 32 * (j >> 1) + q0 + e];
      v[e] = (_Float16)__builtin_fmaf(d, (float)((j & 1) ? q >> 4 : q & 15), -o);
    }
  } else {
    v = *reinterpret_cast<const h8*>((const _Float16*)w + (size_t)n * K + k);
  }
  *reinterpret_cast<h8*>(out + tiled_index(n, k, K)) = v;
}

}  // namespace

namespace t5k {
namespace {
// Microseconds of a launch's first tile on a CU and of each further tile of that CU, measured at
// 256 to 32,768 tokens: residual launches at K = 768 (O) and K = 2048 (wo), the others at K = 768
// (QKV, gate|up, projection); linear in K between and beyond.
struct GemmCost {
  int rows, cols;  // tokens x weight rows of a tile
  double rl, rw, rl2, rw2, l, w;
};
const GemmCost kGemmCost[GEMM_AUTO_VARIANTS] = {
    {32, 64, 6.6, 4.6, 10.7, 8.6, 7.0, 6.8},          // GEMM_RING_32X64
    {64, 64, 7.3, 5.4, 11.7, 10.0, 7.0, 6.0},         // GEMM_RING_64X64
    {128, 64, 10.8, 9.5, 17.7, 17.0, 8.8, 8.6},       // GEMM_RING_128X64
    {128, 128, 13.2, 16.0, 22.8, 27.0, 10.0, 10.0},   // GEMM_RING_128X128
    {128, 128, 15.0, 13.0, 27.5, 20.0, 10.6, 7.5},    // GEMM_RING_128X128_2
    {128, 128, 15.5, 14.0, 27.0, 22.0, 10.7, 6.6},    // GEMM_128X128
    {192, 128, 17.5, 21.0, 29.0, 34.0, 12.2, 8.75},   // GEMM_192X128
    {256, 128, 21.5, 27.0, 36.0, 45.0, 15.5, 12.1},   // GEMM_256X128
};
}  // namespace

// The variant with the least estimated time: ceil(tiles / CUs) tiles on the fullest CU, the first
// one a little slower when the chip is full (its loads share the fabric).  n_rows = weight rows of
// the launch (both matrices for the gated FFN).  Against the best variant measured per shape the
// estimate's choice is within 5% at most sizes (13% at the worst, O at 8,192 tokens).
GemmPlan gemm_plan(int epi, int M, int n_rows, int K, int cus) {
  GemmPlan pl;
  double best = 1e30;
  const double k = (K - 768) / 1280.0;
  for (int v = 0; v < GEMM_AUTO_VARIANTS; v++) {
    const GemmCost& c = kGemmCost[v];
    if (n_rows % c.cols) continue;
    const double dl = k * (c.rl2 - c.rl), dw = k * (c.rw2 - c.rw);
    const double l = (epi == EPI_RESID ? c.rl : c.l) + dl, w = (epi == EPI_RESID ? c.rw : c.w) + dw;
    const double tiles = (double)((M + c.rows - 1) / c.rows) * (n_rows / c.cols);
    const double n = (double)(((long)tiles + cus - 1) / cus);
    const double t = n <= 1 ? l + 0.2 * w * (tiles / cus) : l + (n - 1) * w;
    if (t < best) {
      best = t;
      pl.variant = v;
    }
  }
  return pl;
}

hipError_t launch_tile_weights(const void* w, int wfmt, int N, int K, _Float16* out, hipStream_t s) {
  if (N % 16 || K % 32 || (wfmt == WF_Q4K && K % QK_K)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(((size_t)N * K / 8 + 255) / 256));
  if (wfmt == WF_Q4K) hipLaunchKernelGGL((tile_weights_kernel<true>), grid, dim3(256), 0, s, w, N, K, out);
  else hipLaunchKernelGGL((tile_weights_kernel<false>), grid, dim3(256), 0, s, w, N, K, out);
  return hipGetLastError();
}

hipError_t launch_gemm(int epi, const GemmPlan& pl, const GemmArgs& a, hipStream_t s) {
  if (a.M <= 0) return hipSuccess;
  if (!a.W0 || (epi == EPI_GATED && !a.W1)) return hipErrorInvalidValue;
  // whole tiles along N (128 weight rows at most: 64 columns of each matrix when gated) and whole
  // 128-wide K steps
  if (a.N % (epi == EPI_GATED ? 64 : 128) || a.K % 128) return hipErrorInvalidValue;
  // folded T5LayerNorm: the normalised row must fit one norm record
  if (epi == EPI_RESID && a.nx && (!a.rec || !a.ngamma || a.N != a.ldo || a.N > NORM_REC_MAX_D))
    return hipErrorInvalidValue;
  if (epi != EPI_RESID && a.rec && a.K > NORM_REC_MAX_D) return hipErrorInvalidValue;
  switch (epi) {
    case EPI_RESID: return launch_epi<EPI_RESID>(pl.variant, a, s);
    case EPI_GATED: return launch_epi<EPI_GATED>(pl.variant, a, s);
    case EPI_F32: return launch_epi<EPI_F32>(pl.variant, a, s);
    case EPI_QKV: return launch_epi<EPI_QKV>(pl.variant, a, s);
    case EPI_RELU: return launch_epi<EPI_RELU>(pl.variant, a, s);
  }
  return hipErrorInvalidValue;
}
}  // namespace t5k
