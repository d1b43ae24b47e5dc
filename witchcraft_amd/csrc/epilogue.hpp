// epilogue.hpp -- output stores shared by the GEMM and GEMV kernels.
//
// Both kernels run v_mfma_f32_16x16x32_f16 with the weight fragment as the A operand
// (D^T = W . X^T), so a lane ends with 4 consecutive output columns n..n+3 of one token m.
// These helpers write such a quad for every epilogue kind (Epilogue in common.hpp).
#pragma once
#include "common.hpp"

template <int EPI>
__device__ __forceinline__ void store_quad(const GemmArgs& p, int m, int n, f4 v) {
  if constexpr (EPI == EPI_RESID) {  // residual stream x += acc (f32)
    float4* x = reinterpret_cast<float4*>((float*)p.out + (size_t)m * p.ldo + n);
    float4 r = *x;
    r.x += v[0];
    r.y += v[1];
    r.z += v[2];
    r.w += v[3];
    *x = r;
  } else if constexpr (EPI == EPI_F32) {
    *reinterpret_cast<float4*>((float*)p.out + (size_t)m * p.ldo + n) = make_float4(v[0], v[1], v[2], v[3]);
  } else if constexpr (EPI == EPI_F16 || EPI == EPI_RELU) {  // operand order for the next GEMM
    if (EPI == EPI_RELU) v = f4{fmaxf(v[0], 0.f), fmaxf(v[1], 0.f), fmaxf(v[2], 0.f), fmaxf(v[3], 0.f)};
    *reinterpret_cast<h4*>((_Float16*)p.out + tiled_index(m, n, p.ldo)) =
        h4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
  } else if constexpr (EPI == EPI_QKV) {  // 4 consecutive columns stay inside one head (dkv % 4 == 0)
    const int inner = p.heads * p.dkv;
    const int nn = n + p.n_off;
    const int which = nn / inner, rem = nn % inner;
    const int h = rem / p.dkv, d = rem % p.dkv;
    _Float16* dst = (_Float16*)p.out + (((size_t)which * p.heads + h) * p.tpad + m) * p.dkv + d;
    *reinterpret_cast<h4*>(dst) = h4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
  }
}

// Gated FFN hidden state gelu_tanh(x W0^T) * (x W1^T), in operand order for the wo GEMM.
__device__ __forceinline__ void store_quad_gated(const GemmArgs& p, int m, int n, f4 g, f4 u) {
  *reinterpret_cast<h4*>((_Float16*)p.out + tiled_index(m, n, p.ldo)) =
      h4{(_Float16)(gelu_tanh_dev(g[0]) * u[0]), (_Float16)(gelu_tanh_dev(g[1]) * u[1]),
         (_Float16)(gelu_tanh_dev(g[2]) * u[2]), (_Float16)(gelu_tanh_dev(g[3]) * u[3])};
}

// Consumer side of a folded T5LayerNorm (GemmArgs::rec).  Lane l serves token
// mrow0 + 16 * (l / 16) + l % 16 (lanes whose row block lies past MB read block 0 instead):
// norm_rec_load fetches its record before the K loop's first loads, norm_factor turns it
// into rsqrt(mean(x^2) + eps) / s once those have landed.  The sums run in a fixed order, so
// every tile of every launch (and the one-launch FFN of k_ffn.hip) gets the same bits.  Tiles
// at n0 = 0 also store the next producer's operand scale.
template <int MB>
__device__ __forceinline__ int norm_row(int mrow0) {
  const int lane = threadIdx.x & 63, mb = lane >> 4;
  return mrow0 + 16 * (mb < MB ? mb : 0) + (lane & 15);
}
template <int MB>
__device__ __forceinline__ void norm_rec_load(const GemmArgs& p, int mrow0, float4 (&r)[4]) {
  const float4* src = reinterpret_cast<const float4*>(p.rec + (size_t)norm_row<MB>(mrow0) * 16);
#pragma unroll
  for (int i = 0; i < 4; i++) r[i] = src[i];
}
// rsqrt(mean(x^2) + eps) of a token of K features from its norm record r (slot 15 unused here).
__device__ __forceinline__ float norm_inv(const float4 (&r)[4], int K, float eps) {
  // slots past K / 64 are masked: the record array may hold another layout's data there
  const int ns = K / 64;
  float v[15];
#pragma unroll
  for (int i = 0; i < 15; i++) {
    const float4 q = r[i / 4];
    const float x = (i & 3) == 0 ? q.x : (i & 3) == 1 ? q.y : (i & 3) == 2 ? q.z : q.w;
    v[i] = i < ns ? x : 0.f;
  }
  const float tot = (((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]))) +
                    (((v[8] + v[9]) + (v[10] + v[11])) + ((v[12] + v[13]) + v[14]));
  return 1.0f / sqrtf(tot / (float)K + eps);
}
template <int MB>
__device__ __forceinline__ float norm_factor(const GemmArgs& p, int mrow0, int n0, const float4 (&r)[4]) {
  const float inv = norm_inv(r, p.K, p.eps);
  const int m = norm_row<MB>(mrow0);
  if (p.rec_next && n0 == 0 && (threadIdx.x & 63) < 16 * MB && m < p.M)
    p.rec_next[(size_t)m * 16 + 15] = norm_operand_scale(inv);
  return inv / r[3].w;
}

// A quad's sum of squares, as the residual epilogues add it into a norm record slot.
__device__ __forceinline__ float quad_sq(float4 r) { return (r.x * r.x + r.y * r.y) + (r.z * r.z + r.w * r.w); }

// QKV epilogue through LDS (d_kv = 64).  The accumulators give each lane 4 columns of one
// token, so direct stores into the head-major [3][H][tpad][64] layout write 16 x 32-byte
// pieces per instruction.  Instead each 16-token block is staged in this wave's LDS region
// (the weight stage, idle once the K loop has ended) and copied out as whole 128-byte head
// rows, 16 bytes per lane.  `stage` holds 16 rows of BN + 8 halves.  No wait is needed between
// the staging writes and reads: a wave's LDS instructions execute in order, and the compiler
// keeps the order of these possibly aliasing accesses.
template <int BN, int MB>
__device__ __forceinline__ void qkv_store_staged(const GemmArgs& p, int mrow0, int n0, const f4 (&acc)[MB][BN / 16],
                                                 _Float16* stage) {
  constexpr int NB = BN / 16, RS = BN + 8;
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int inner = p.heads * 64;
#pragma unroll
  for (int mb = 0; mb < MB; mb++) {
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
      *reinterpret_cast<h4*>(stage + lr * RS + 16 * nb + 4 * lg) =
          h4{(_Float16)acc[mb][nb][0], (_Float16)acc[mb][nb][1], (_Float16)acc[mb][nb][2], (_Float16)acc[mb][nb][3]};
#pragma unroll
    for (int g = 0; g < BN / 64; g++) {
      const int nn = n0 + 64 * g + p.n_off, which = nn / inner, h = (nn % inner) / 64;
      _Float16* dst = (_Float16*)p.out + ((size_t)which * p.heads + h) * p.tpad * 64;
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int c = lane + 64 * j, tok = c >> 3, part = c & 7;
        const int m = mrow0 + 16 * mb + tok;
        const uint4 v = *reinterpret_cast<const uint4*>(stage + tok * RS + 64 * g + 8 * part);
        if (m < p.M) *reinterpret_cast<uint4*>(dst + (size_t)m * 64 + 8 * part) = v;
      }
    }
  }
}

// Residual epilogue x += acc; with GemmArgs::nx set it also prepares the next T5LayerNorm:
// the f16 operand f16(x * gamma * s) in operand order and the tile's sums of x^2 per 64-column
// group in the token's norm record.  Lane (lr, lg) holds columns n0 + 16nb + 4lg .. +3 of token
// mrow0 + 16mb + lr, so a group's sum is the lane's 16 squares plus those of the lanes lr + 16,
// lr + 32, lr + 48 (xor 16, xor 32).  Every load is unconditional -- x and the records have
// Mpad rows, so rows past M read padding -- and the x reads of CH row blocks are issued
// together: a guarded load per quad would cost one memory round trip each.  Only the stores
// are guarded; rows past M take part in the sums but store nothing.
template <int BN, int MB>
__device__ __forceinline__ void resid_store_tile(const GemmArgs& p, int mrow0, int n0, const f4 (&acc)[MB][BN / 16]) {
  constexpr int NB = BN / 16, G = BN / 64;
  constexpr int CH = BN == 64 ? MB : (MB % 2 == 0 ? 2 : 1);  // row blocks whose x is read at once
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const bool fold = p.nx != nullptr;
  float* x = (float*)p.out;
  float4 g[NB];
  float s[MB], ss[MB][G];
#pragma unroll
  for (int mb = 0; mb < MB; mb++) {
#pragma unroll
    for (int j = 0; j < G; j++) ss[mb][j] = 0.f;
    s[mb] = 0.f;
  }
  if (fold) {
#pragma unroll
    for (int nb = 0; nb < NB; nb++) g[nb] = *reinterpret_cast<const float4*>(p.ngamma + n0 + 16 * nb + 4 * lg);
#pragma unroll
    for (int mb = 0; mb < MB; mb++) s[mb] = p.rec[(size_t)(mrow0 + 16 * mb + lr) * 16 + 15];
  }
#pragma unroll
  for (int c0 = 0; c0 < MB; c0 += CH) {
    float4 xv[CH][NB];
#pragma unroll
    for (int j = 0; j < CH; j++)
#pragma unroll
      for (int nb = 0; nb < NB; nb++)
        xv[j][nb] = *reinterpret_cast<const float4*>(x + (size_t)(mrow0 + 16 * (c0 + j) + lr) * p.ldo + n0 +
                                                     16 * nb + 4 * lg);
#pragma unroll
    for (int j = 0; j < CH; j++) {
      const int mb = c0 + j, m = mrow0 + 16 * mb + lr;
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        float4& r = xv[j][nb];
        r.x += acc[mb][nb][0];
        r.y += acc[mb][nb][1];
        r.z += acc[mb][nb][2];
        r.w += acc[mb][nb][3];
        ss[mb][nb / 4] += quad_sq(r);
      }
      if (m < p.M) {
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
          const int n = n0 + 16 * nb + 4 * lg;
          const float4 r = xv[j][nb];
          *reinterpret_cast<float4*>(x + (size_t)m * p.ldo + n) = r;
          if (fold)
            *reinterpret_cast<h4*>(p.nx + tiled_index(m, n, p.ldo)) =
                h4{(_Float16)((r.x * g[nb].x) * s[mb]), (_Float16)((r.y * g[nb].y) * s[mb]),
                   (_Float16)((r.z * g[nb].z) * s[mb]), (_Float16)((r.w * g[nb].w) * s[mb])};
        }
      }
    }
  }
  if (fold) {
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
      const int m = mrow0 + 16 * mb + lr;
#pragma unroll
      for (int j = 0; j < G; j++) {
        const float t = sum_xor32(sum_xor16(ss[mb][j]));
        if (m < p.M && lg == 0) p.rec[(size_t)m * 16 + n0 / 64 + j] = t;
      }
    }
  }
}
