// k_hybrid.hip -- Q4_K weights x Q8_K activations on the matrix cores (launch_gemm_hybrid).
//
// The hybrid-dequant numerics' gate|up and projection (src/fused_matmul.rs:27-59, 138-177): GGML's
// integer vec_dot per 256-value block, its integer sums exact.
//
// Warp-specialised workgroup: MW "math" wave64s + MW "producer" wave64s, one of each per SIMD, so
// the producers' global loads, nibble unpacking and block folds (VALU) issue while the math waves'
// MFMAs occupy the matrix core.
//  * Tile: 16 HYB_MB MW tokens x BN weight rows, K stepped by 64 (one Q4_K chunk).
//  * Producers: per K step, read each weight row's 16-byte Q4_K header and 32 bytes of nibbles and
//    write the int8 planes of the BN x 64 stage into LDS (double-buffered); the raw bytes of the
//    next steps are in flight meanwhile.  They also hold the f32 outputs and run the epilogue.
//  * Math waves: each owns 16 HYB_MB token rows, streamed from global memory in MFMA operand order.
//  * Tiles are ordered so that each XCD (8 per device, workgroups dealt round-robin) works on a
//    contiguous band of tiles.
#include "common.hpp"
#include "epilogue.hpp"
#include "q4k.hpp"

namespace {

constexpr int BK = 64, LDSK = BK;

// B-tile row r -> (weight matrix, output column).  Gated: rows [0, BN/2) are W0 columns
// n0.., rows [BN/2, BN) the same W1 columns, so a math wave's N blocks nb < NB/2 (gate)
// and nb + NB/2 (up) hold the same output columns in the same lanes.
template <int EPI, int BN>
__device__ __forceinline__ void brow(int r, int n0, const GemmArgs& p, const void*& W, int& n) {
  if (EPI == EPI_GATED) {
    W = r < BN / 2 ? p.W0 : p.W1;
    n = n0 + (r & (BN / 2 - 1));
  } else {
    W = p.W0;
    n = n0 + r;
  }
}

// Raw Q4_K weights of one K step held by a producer thread between load and unpack.
template <int NP, int BN>
struct BRaw {
  static constexpr int TPR = NP / BN;   // producer threads per weight row
  static constexpr int BPT = 32 / TPR;  // nibble bytes per thread: 32, 16 or 8
  static constexpr int NQ = BPT / 4;
  uint4 hd;
  uint32_t q[NQ];
};

template <int EPI, int NP, int BN>
__device__ __forceinline__ void load_b(BRaw<NP, BN>& br, const GemmArgs& p, int n0, int kt, int pt) {
  using R = BRaw<NP, BN>;
  const int r = pt / R::TPR, part = pt % R::TPR;
  const void* W;
  int n;
  brow<EPI, BN>(r, n0, p, W, n);
  const int kb = (kt * BK) / QK_K, c = ((kt * BK) % QK_K) / 64;
  const uint8_t* blk = (const uint8_t*)W + ((size_t)n * (p.K / QK_K) + kb) * Q4K_BYTES;
  br.hd = *reinterpret_cast<const uint4*>(blk);
  const uint8_t* qs = blk + 16 + 32 * c + part * R::BPT;
  if constexpr (R::BPT == 32) {
    const uint4 a = *reinterpret_cast<const uint4*>(qs), b = *reinterpret_cast<const uint4*>(qs + 16);
    br.q[0] = a.x; br.q[1] = a.y; br.q[2] = a.z; br.q[3] = a.w;
    br.q[4] = b.x; br.q[5] = b.y; br.q[6] = b.z; br.q[7] = b.w;
  } else if constexpr (R::BPT == 16) {
    const uint4 a = *reinterpret_cast<const uint4*>(qs);
    br.q[0] = a.x; br.q[1] = a.y; br.q[2] = a.z; br.q[3] = a.w;
  } else {
    const uint2 a = *reinterpret_cast<const uint2*>(qs);
    br.q[0] = a.x; br.q[1] = a.y;
  }
}

// Hybrid numerics (launch_gemm_hybrid): the stage holds the nibbles times their sub-block scale
// as two int8 planes.  A 6-bit scale splits as sc = 8 sh + sl (sh, sl <= 7), so sh q and sl q are
// at most 105 and fit int8: the hi plane holds sh q, the lo plane sl q, and a K block's integer
// sum is 8 (hi . q8) + (lo . q8), exact in int32.  Four nibbles masked into the bytes of a word
// times a scale <= 7 give all four products with one multiply (no byte carries into the next).
// Plane rows are 64 bytes (one K step); 16-byte chunk j of row r sits at chunk j ^ ((r >> 2) & 3),
// so the math waves' fragment reads (16 rows x one chunk) hit every bank once.  At the first K
// step of a 256-wide block the row's first producer thread also writes the block's d and dmin
// (Md) and its eight 6-bit mins as the A operand of the min-term MFMA (Mm: m0 m0 m1 m1 .. m7 m7,
// one per bsum).
// 16-token row blocks per math wave in a full hybrid tile (the tile is 16 HYB_MB MW tokens).
constexpr int HYB_MB = 3;
__device__ __forceinline__ int hyb_off(int r, int k) {  // byte offset of (row r, K index k) in a plane
  return r * 64 + ((((k >> 4) ^ (r >> 2)) & 3) << 4) + (k & 15);
}
template <int NP, int BN>
__device__ __forceinline__ void store_b_hybrid(const BRaw<NP, BN>& br, _Float16* Bs, float2* Md, h8* Mm,
                                               int kt, int pt) {
  using R = BRaw<NP, BN>;
  static_assert(R::BPT == 8 || R::BPT == 16 || R::BPT == 32, "nibble bytes per thread");
  const int r = pt / R::TPR, part = pt % R::TPR;
  const int c = ((kt * BK) % QK_K) / 64;
  const uint4 hd = br.hd;
  // get_scale_min_k4 on the 12 scale bytes (header words y, z, w); sub-blocks 2c, 2c + 1
  auto byte = [&](int i) -> int {
    const uint32_t w = i < 4 ? hd.y : (i < 8 ? hd.z : hd.w);
    return (int)((w >> (8 * (i & 3))) & 0xff);
  };
  auto scale_min = [&](int j, int& sc, int& m) {
    if (j < 4) {
      sc = byte(j) & 63;
      m = byte(j + 4) & 63;
    } else {
      sc = (byte(j + 4) & 15) | ((byte(j - 4) >> 6) << 4);
      m = (byte(j + 4) >> 4) | ((byte(j) >> 6) << 4);
    }
  };
  int sc0, m0, sc1, m1;
  scale_min(2 * c, sc0, m0);
  scale_min(2 * c + 1, sc1, m1);
  uint8_t* hi = reinterpret_cast<uint8_t*>(Bs);
  uint8_t* lo = hi + BN * 64;
  // nibble word w holds values k0 + 4w .. +3 of sub-block 2c (low nibbles) and of 2c + 1 (high)
  const int k0 = part * R::BPT;
#pragma unroll
  for (int w = 0; w < R::NQ; w += 2) {
    const uint32_t l0 = br.q[w] & 0x0f0f0f0fu, l1 = br.q[w + 1] & 0x0f0f0f0fu;
    const uint32_t h0 = (br.q[w] >> 4) & 0x0f0f0f0fu, h1 = (br.q[w + 1] >> 4) & 0x0f0f0f0fu;
    const int k = k0 + 4 * w;
    *reinterpret_cast<uint2*>(hi + hyb_off(r, k)) = make_uint2(l0 * (uint32_t)(sc0 >> 3), l1 * (uint32_t)(sc0 >> 3));
    *reinterpret_cast<uint2*>(lo + hyb_off(r, k)) = make_uint2(l0 * (uint32_t)(sc0 & 7), l1 * (uint32_t)(sc0 & 7));
    *reinterpret_cast<uint2*>(hi + hyb_off(r, 32 + k)) =
        make_uint2(h0 * (uint32_t)(sc1 >> 3), h1 * (uint32_t)(sc1 >> 3));
    *reinterpret_cast<uint2*>(lo + hyb_off(r, 32 + k)) =
        make_uint2(h0 * (uint32_t)(sc1 & 7), h1 * (uint32_t)(sc1 & 7));
  }
  if (c == 0 && part == 0) {
    Md[r] = make_float2(f16_bits_to_f32(hd.x & 0xffff), f16_bits_to_f32(hd.x >> 16));
    _Float16 mh[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      int sc, m;
      scale_min(j, sc, m);
      mh[j] = (_Float16)m;
    }
    Mm[2 * r] = h8{mh[0], mh[0], mh[1], mh[1], mh[2], mh[2], mh[3], mh[3]};
    Mm[2 * r + 1] = h8{mh[4], mh[4], mh[5], mh[5], mh[6], mh[6], mh[7], mh[7]};
  }
}

// Hybrid-numerics tile (launch_gemm_hybrid).  The stage holds sc q4 as the int8 planes
// hi = (sc >> 3) q4 and lo = (sc & 7) q4 (store_b_hybrid) and the A operand the Q8_K integers q8
// as int8, so v_mfma_i32_16x16x64_i8 sums each plane against q8 exactly in int32, and a 256-wide
// K block's integer sum is S = 8 hi + lo.  The block is then folded into the f32 output:
//   out += d8 * (d4 * float(S) - dmin4 * (mins . bsums)),
// the min term from one f16 MFMA of the row's mins (Mm) against the tokens' bsums (bsop, exact:
// <= 16 * 63 * 2048).  This is vec_dot's d * d8 * sum_j sc_j (q4 . q8)_j - dmin * d8 *
// sum_j m_j (bsum_2j + bsum_2j+1) per block (src/fused_matmul.rs:36-41,147-172): the integer
// sum is exact and converted to f32 once, as there.
// The math waves only run the integer MFMAs: at a block's last K step each writes its S tiles to
// the exchange buffer Sx, and producer wave MW + w folds math wave w's block during the next
// block's first K step (HybFold), so the fold's VALU work overlaps the next block's MFMAs on the
// same SIMD instead of stalling them.  Sx is read three barriers before it is written again.
// A operand (p.A as bytes): blocks of 16 tokens x 64 K (1 KiB) [Mpad/16][K/64], lane l holding
// token l % 16, K 16 (l / 16) .. +15; the weight fragment of lane l is row l % 16 of its row
// block, the same 16 K values.  Sx: [MW][MB][NB][64 lanes] int4, the lane's four outputs.
typedef int v4i __attribute__((ext_vector_type(4)));
template <int EPI, int MW, int BN, int S, int MB>
__device__ __forceinline__ void math_hybrid(const GemmArgs& p, int m0, _Float16 (*Bs)[BN * LDSK], int4* Sx) {
  constexpr int NB = BN / 16;
  static_assert(S == 2, "the hybrid loop unrolls a K block as two A stages");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15, lg = lane >> 4;
  const int nkt = p.K / BK, nblk = p.K / QK_K;
  const int mrow0 = m0 + wave * 16 * MB;
  const size_t kch = p.K / 64;  // 1 KiB operand blocks per 16-token row block
  const uint8_t* ablk[MB];
#pragma unroll
  for (int mb = 0; mb < MB; mb++)
    ablk[mb] = reinterpret_cast<const uint8_t*>(p.A) + (size_t)(mrow0 / 16 + mb) * kch * 1024 + lane * 16;
  int4* sx = Sx + (size_t)wave * MB * NB * 64 + lane;

  v4i acc_hi[MB][NB], acc_lo[MB][NB];
  uint4 a[S][MB];
#define LOAD_A(st, kt) \
  _Pragma("unroll") for (int mb = 0; mb < MB; mb++) a[st][mb] = *reinterpret_cast<const uint4*>(ablk[mb] + (size_t)(kt) * 1024);
  LOAD_A(0, 0);
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();

  // this lane's fragment of row block nb: row 16 nb + lr, K chunk lg
  int foff[NB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++) foff[nb] = hyb_off(16 * nb + lr, 16 * lg);
  const v4i izero = {0, 0, 0, 0};
  for (int b = 0; b < nblk; b++) {
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int kt = 4 * b + u;
      LOAD_A((u + 1) % S, min(kt + 1, nkt - 1));
      __builtin_amdgcn_sched_barrier(0);
      const uint8_t* hi = reinterpret_cast<const uint8_t*>(Bs[kt & 1]);
      const uint8_t* lo = hi + BN * 64;
      // every fragment of the step is requested before the first MFMA, so the LDS latency is
      // paid once per step rather than once per row block
      v4i wh[NB], wl[NB];
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        wh[nb] = *reinterpret_cast<const v4i*>(hi + foff[nb]);
        wl[nb] = *reinterpret_cast<const v4i*>(lo + foff[nb]);
      }
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
          const v4i x = __builtin_bit_cast(v4i, a[u % S][mb]);
          acc_hi[mb][nb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wh[nb], x, u == 0 ? izero : acc_hi[mb][nb], 0, 0, 0);
          acc_lo[mb][nb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wl[nb], x, u == 0 ? izero : acc_lo[mb][nb], 0, 0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (u == 3) {
        // block b's sums for the fold waves: lane holds rows 16nb + 4lg + i of token 16mb + lr
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
          for (int nb = 0; nb < NB; nb++) {
            const v4i sum = (acc_hi[mb][nb] << 3) + acc_lo[mb][nb];
            sx[(mb * NB + nb) * 64] = make_int4(sum[0], sum[1], sum[2], sum[3]);
          }
      }
      __syncthreads();
    }
  }
#undef LOAD_A
}

// Producer wave MW + w's share of a hybrid tile: the f32 outputs of math wave w, folded block by
// block from Sx, and the epilogue.
template <int EPI, int MW, int BN, int MB>
struct HybFold {
  static constexpr int NB = BN / 16;
  f4 out[MB][NB];
  float d8v[MB];  // the next block's d8 and bsum operand, requested a block ahead
  uint4 bsf[MB];
  int mrow0, lane, lr, lg, nblk;
  const int4* sx;

  __device__ __forceinline__ void load_meta(const GemmArgs& p, int b) {
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
      d8v[mb] = p.d8[(size_t)(mrow0 + 16 * mb + lr) * nblk + b];
      bsf[mb] = *reinterpret_cast<const uint4*>(p.bsop + ((size_t)(mrow0 / 16 + mb) * nblk + b) * 512 + lane * 8);
    }
  }
  __device__ __forceinline__ void init(const GemmArgs& p, int m0, const int4* Sx) {
    const int w = (threadIdx.x >> 6) - MW;
    lane = threadIdx.x & 63;
    lr = lane & 15;
    lg = lane >> 4;
    nblk = p.K / QK_K;
    mrow0 = m0 + w * 16 * MB;
    sx = Sx + (size_t)w * MB * NB * 64 + lane;
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
      for (int j = 0; j < NB; j++) out[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    load_meta(p, 0);
  }
  // block b: its sums in Sx, its row metadata in Md / Mm [b % 2], its d8 / bsums in d8v / bsf
  __device__ __forceinline__ void fold(const GemmArgs& p, int b, const float2 (*Md)[BN], const h8 (*Mm)[2 * BN]) {
    const int bp = b & 1;
    const f4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
      const float4 q0 = *reinterpret_cast<const float4*>(&Md[bp][16 * nb + 4 * lg]);
      const float4 q1 = *reinterpret_cast<const float4*>(&Md[bp][16 * nb + 4 * lg + 2]);
      const float dd[4] = {q0.x, q0.z, q1.x, q1.z}, dm[4] = {q0.y, q0.w, q1.y, q1.w};
      const h8 mf = lg < 2 ? Mm[bp][2 * (16 * nb + lr) + lg] : h8{};
#pragma unroll
      for (int mb = 0; mb < MB; mb++) {
        const f4 cm = __builtin_amdgcn_mfma_f32_16x16x32_f16(mf, __builtin_bit_cast(h8, bsf[mb]), zero, 0, 0, 0);
        const int4 sv = sx[(mb * NB + nb) * 64];
        const int si[4] = {sv.x, sv.y, sv.z, sv.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
          // d8 (d S - dmin M): the block's row scales first, the token's scale once
          const float t = __builtin_fmaf(-dm[i], cm[i], dd[i] * (float)si[i]);
          out[mb][nb][i] = __builtin_fmaf(d8v[mb], t, out[mb][nb][i]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // one row block at a time: bounded live registers
    }
    if (b + 1 < nblk) load_meta(p, b + 1);
  }
  __device__ __forceinline__ void epilogue(const GemmArgs& p, int n0) {
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
      const int m = mrow0 + mb * 16 + lr;
      if (m >= p.M) continue;
      if constexpr (EPI == EPI_GATED) {
#pragma unroll
        for (int nb = 0; nb < NB / 2; nb++) {
          const f4 g = out[mb][nb], v = out[mb][nb + NB / 2];
          *reinterpret_cast<h4*>((_Float16*)p.out + tiled_index(m, n0 + nb * 16 + 4 * lg, p.ldo)) =
              h4{(_Float16)(gelu_pade(g[0]) * v[0]), (_Float16)(gelu_pade(g[1]) * v[1]),
                 (_Float16)(gelu_pade(g[2]) * v[2]), (_Float16)(gelu_pade(g[3]) * v[3])};
        }
      } else {
#pragma unroll
        for (int nb = 0; nb < NB; nb++) store_quad<EPI_F32>(p, m, n0 + nb * 16 + 4 * lg, out[mb][nb]);
      }
    }
  }
};

// One output tile: tokens [m0, m0 + 16*MB*MW) x weight rows from n0.  MB = 16-row operand blocks
// per math wave: HYB_MB for full tiles, 1 for the thin tiles that spread the last, partial round
// of a launch over every CU.
template <int EPI, int MW, int BN, int S, int MB>
__device__ __forceinline__ void hybrid_tile(const GemmArgs& p, int m0, int n0, _Float16 (*Bs)[BN * LDSK],
                                            float2 (*Md)[BN], h8 (*Mm)[2 * BN], int4* Sx) {
  constexpr int NP = 64 * MW, PB = 4;
  using R = BRaw<NP, BN>;
  const int nkt = p.K / BK;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // waves [0, MW) compute, waves [MW, 2MW) produce; wave w runs on SIMD w % 4
  if (wave < MW) {
    math_hybrid<EPI, MW, BN, S, MB>(p, m0, Bs, Sx);
    return;
  }
  // Raw bytes of step j live in ring slot j % PB; step kt+1 is unpacked into LDS while steps
  // kt+2 .. kt+PB are in flight.  One barrier per step, as in the math waves.
  const int pt = tid - NP;
  R br[PB];
  // step kt's weights into stage kt % 2, the block's metadata into kt / 4 % 2
  auto store = [&](const R& r, int kt) {
    store_b_hybrid<NP, BN>(r, Bs[kt & 1], Md[(kt >> 2) & 1], Mm[(kt >> 2) & 1], kt, pt);
  };
  load_b<EPI, NP, BN>(br[0], p, n0, 0, pt);
  store(br[0], 0);
#pragma unroll
  for (int i = 1; i < PB; i++) load_b<EPI, NP, BN>(br[i], p, n0, i, pt);
  // these waves also fold the math waves' block sums (PB steps = one block)
  HybFold<EPI, MW, BN, MB> hf;
  static_assert(PB * BK == QK_K, "one producer ring turn per Q4_K block");
  hf.init(p, m0, Sx);
  __syncthreads();
  // nkt % PB == 0 (K % 256 == 0); loads past the last step re-read it (in bounds, unused)
  // so that every load is unconditional and the compiler's wait counts stay exact.
  for (int kt0 = 0; kt0 < nkt; kt0 += PB) {
#pragma unroll
    for (int u = 0; u < PB; u++) {
      const int kt = kt0 + u;
      if (kt + 1 < nkt) store(br[(u + 1) % PB], kt + 1);
      load_b<EPI, NP, BN>(br[u], p, n0, min(kt + PB, nkt - 1), pt);
      if (u == 0 && kt0 > 0) hf.fold(p, kt0 / PB - 1, Md, Mm);
      __syncthreads();
    }
  }
  hf.fold(p, nkt / PB - 1, Md, Mm);
  hf.epilogue(p, n0);
}

// Grid of one launch: blocks [0, main_blocks) run the full tiles of rows [0, m_main), the
// rest the thin tiles (TMB row blocks per math wave) of rows [m_main, M).  Within each part,
// block b runs on XCD b % 8 (workgroups are dealt round-robin), and each XCD gets a
// contiguous range of tiles, so its L2 holds the A rows it streams plus the weights.
struct HybGrid {
  int tiles_n, main_tiles, main_blocks, m_main, tail_tiles;
};

template <int EPI, int MW, int BN, int S, int TMB>
__global__ __launch_bounds__(128 * MW) __attribute__((amdgpu_waves_per_eu(2)))
void hybrid_gemm_kernel(GemmArgs p, HybGrid g) {
  __shared__ __attribute__((aligned(16))) _Float16 Bs[2][BN * LDSK];
  // per-row block metadata (d, dmin; mins as an MFMA operand), two blocks deep
  __shared__ __attribute__((aligned(16))) float2 Md[2][BN];
  __shared__ __attribute__((aligned(16))) h8 Mm[2][2 * BN];
  // the math waves' block sums for the fold waves
  __shared__ int4 Sx[MW * HYB_MB * (BN / 16) * 64];
  constexpr int cols = EPI == EPI_GATED ? BN / 2 : BN;  // output columns per tile
  int b = blockIdx.x;
  if (TMB == 0 || b < g.main_blocks) {
    const int tile = (b % 8) * (g.main_blocks / 8) + b / 8;
    if (tile >= g.main_tiles) return;
    hybrid_tile<EPI, MW, BN, S, HYB_MB>(p, (tile / g.tiles_n) * 16 * HYB_MB * MW, (tile % g.tiles_n) * cols, Bs, Md,
                                        Mm, Sx);
  } else {
    constexpr int MBT = TMB == 0 ? 1 : TMB;
    b -= g.main_blocks;
    const int tile = (b % 8) * (((int)gridDim.x - g.main_blocks) / 8) + b / 8;
    if (tile >= g.tail_tiles) return;
    hybrid_tile<EPI, MW, BN, S, MBT>(p, g.m_main + (tile / g.tiles_n) * 16 * MBT * MW, (tile % g.tiles_n) * cols, Bs,
                                     Md, Mm, Sx);
  }
}

template <int EPI, int BN, int S, int MW, int TMB>
hipError_t launch_plan(const t5k::HybridPlan& pl, const GemmArgs& a, hipStream_t s) {
  constexpr int cols = EPI == EPI_GATED ? BN / 2 : BN, bm = 16 * HYB_MB * MW;
  HybGrid g;
  g.tiles_n = a.N / cols;
  g.m_main = TMB ? pl.m_main : a.M;
  g.main_tiles = (g.m_main + bm - 1) / bm * g.tiles_n;
  g.main_blocks = (g.main_tiles + 7) / 8 * 8;
  const int bmt = 16 * (TMB ? TMB : 1) * MW;
  g.tail_tiles = TMB ? (a.M - g.m_main + bmt - 1) / bmt * g.tiles_n : 0;
  const int grid = g.main_blocks + (g.tail_tiles + 7) / 8 * 8;
  if (grid == 0) return hipSuccess;
  T5K_LAUNCH((hybrid_gemm_kernel<EPI, MW, BN, S, TMB>), dim3(grid), dim3(128 * MW), 0, s, a, g);
  return hipGetLastError();
}

// Run time of the last tile when `tail` tiles of cost c follow `main` tiles of cost 1 on
// `slots` workgroup slots, each tile taking the earliest free slot (the dispatcher's order).
// After the main tiles, slots free up at r (slots - k of them) and r + 1 (k of them); the
// tail tiles start at r + i*c and r + 1 + j*c, earliest first.
double list_makespan(int main, int tail, double c, int slots) {
  const int r = main / slots, k = main % slots;
  double end = k ? r + 1 : r;
  if (tail <= 0) return end;
  const int n1 = slots - k, n2 = k;
  int i = 0, j = 0, left = tail;
  double start = r;
  while (left > 0) {
    const double t1 = r + i * c, t2 = n2 ? r + 1 + j * c : 1e30;
    if (t1 <= t2) {
      start = t1;
      left -= n1;
      i++;
    } else {
      start = t2;
      left -= n2;
      j++;
    }
  }
  return start + c > end ? start + c : end;
}

}  // namespace

namespace t5k {
int gemm_hybrid_rows(int M) { return (M + 64 * HYB_MB - 1) / (64 * HYB_MB) * (64 * HYB_MB); }

// Full tiles of 64 HYB_MB tokens x 64 weight rows, or with a tail thin tiles of one row block per
// math wave for rows [m_main, M): with one workgroup per CU a launch of T full tiles takes
// ceil(T / CUs) rounds, and a last round that is mostly empty costs as much as a full one.  A thin
// tile costs 0.6 of a full one (measured as one round against one round).
HybridPlan gemm_plan_hybrid(int M, int n_rows, int cus) {
  HybridPlan pl;
  pl.m_main = M;
  pl.tail_mb = 0;
  const int bm = 64 * HYB_MB, tiles_n = n_rows / 64, full = (M + bm - 1) / bm;
  double best = list_makespan(full * tiles_n, 0, 1.0, cus);
  for (int j = full - 1; j >= 0; j--) {
    const int tail = (M - j * bm + 63) / 64 * tiles_n;
    const double t = list_makespan(j * tiles_n, tail, 0.6, cus);
    if (t < best - 1e-9) {
      best = t;
      pl.m_main = j * bm;
      pl.tail_mb = 1;
    }
  }
  return pl;
}

hipError_t launch_gemm_hybrid(int epi, const HybridPlan& pl, const GemmArgs& a, hipStream_t s) {
  if (a.M <= 0) return hipSuccess;
  if (a.K % 256 || !a.A || !a.d8 || !a.bsop) return hipErrorInvalidValue;
  if (pl.tail_mb && (pl.tail_mb != 1 || pl.m_main < 0 || pl.m_main % (64 * HYB_MB) || pl.m_main >= a.M))
    return hipErrorInvalidValue;
  if (epi == EPI_GATED) {
    if (a.N % 32 || !a.W1) return hipErrorInvalidValue;
    return pl.tail_mb ? launch_plan<EPI_GATED, 64, 2, 4, 1>(pl, a, s) : launch_plan<EPI_GATED, 64, 2, 4, 0>(pl, a, s);
  }
  if (epi != EPI_F32 || a.N % 64) return hipErrorInvalidValue;
  return pl.tail_mb ? launch_plan<EPI_F32, 64, 2, 4, 1>(pl, a, s) : launch_plan<EPI_F32, 64, 2, 4, 0>(pl, a, s);
}
}  // namespace t5k
