// Kernels of the packed prefill's trunk around the MoE block: the mHC residual stream
// (modeling_qwen3_8_moe.py:994-1031). As torch operations it is a chain of passes over a large fp32
// tensor (268 MB at 4 x 4096 tokens and hidden 1024); here each pass is one kernel. fp32 is computed in
// fp32, and values are rounded to the parameters' dtype where the torch code rounds.
#include "q38moe_common.h"
#include "q38moe_kernels.h"

namespace q38 {
namespace {

template <bool BF16>
__device__ __forceinline__ float ld_dt(const void* p, int64_t i) {
  if constexpr (BF16) return bf16_to_f32(static_cast<const uint16_t*>(p)[i]);
  else return static_cast<const float*>(p)[i];
}
// Four consecutive elements (i a multiple of 4) as floats.
template <bool BF16>
__device__ __forceinline__ f32x4_t ld4_dt(const void* p, int64_t i) {
  if constexpr (BF16) {
    const uint2 v = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(p) + i);
    float a, b, c, d;
    unpack_bf16x2(v.x, a, b);
    unpack_bf16x2(v.y, c, d);
    return f32x4_t{a, b, c, d};
  } else {
    return *reinterpret_cast<const f32x4_t*>(static_cast<const float*>(p) + i);
  }
}
template <bool BF16>
__device__ __forceinline__ void st4_dt(void* p, int64_t i, f32x4_t v) {
  if constexpr (BF16)
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p) + i) =
        make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
  else
    *reinterpret_cast<f32x4_t*>(static_cast<float*>(p) + i) = v;
}
template <bool BF16>
__device__ __forceinline__ float round_dt(float v) {
  return BF16 ? round_bf16(v) : v;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// ---- mHC: the four-branch residual stream X [T, 4, h] fp32 --------------------------------------
//
// Every kernel that writes X also writes ssq[t] = sum of X[t]^2, which the next sublayer's coefficients
// need, so the stream is read once for its product with A (outside, z0 = X . A^T), once by mhc_pre and
// once by mhc_post. HBM-bound: 16 h bytes per token and pass. At 16384 tokens and h = 1024 mhc_pre takes
// 61 us (302 MB, 4.9 TB/s) and the update 82 us (570 MB, 6.9 TB/s); with torch's operations a sublayer's
// stream took 2.9 ms (a batched 4 x 4 product of 1.0 ms, 80 small launches for Sinkhorn, some ten passes).

constexpr int MHC_N = 4;
constexpr int MHC_COEF = 2 * MHC_N + MHC_N * MHC_N;  // pre, post, residual logits

// Sum of v over the block's four waves, in wave order, on every thread.
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return ((red[0] + red[1]) + red[2]) + red[3];
}

enum { MHC_INIT = 0, MHC_ADD = 1, MHC_POST = 2 };

// One block per token. MHC_INIT: X[t][b] = y[t] for every branch. MHC_ADD: X[t][b] += y[t]. MHC_POST:
// X[t][i] = sum_j P[t][i][j] X[t][j] + post[t][i] y[t] (modeling:1014-1018), in place: a thread owns
// its columns of all four branches. ssq as above.
template <int MODE, bool BF16>
__global__ __launch_bounds__(256) void mhc_update_kernel(float* X, const void* __restrict__ y,
                                                         const float* __restrict__ post,
                                                         const float* __restrict__ P, float* __restrict__ ssq,
                                                         int h) {
  __shared__ float red[4];
  const int64_t t = blockIdx.x;
  float* const xt = X + t * MHC_N * h;
  float p[MHC_N][MHC_N], w[MHC_N];
  if (MODE == MHC_POST) {
#pragma unroll
    for (int i = 0; i < MHC_N; ++i) {
      w[i] = load_uniform(post + t * MHC_N + i);
#pragma unroll
      for (int j = 0; j < MHC_N; ++j) p[i][j] = load_uniform(P + (t * MHC_N + i) * MHC_N + j);
    }
  }
  float s = 0.0f;
  for (int c = 4 * threadIdx.x; c < h; c += 1024) {
    const f32x4_t v = ld4_dt<BF16>(y, t * h + c);
    f32x4_t x[MHC_N];
    if (MODE != MHC_INIT) {
#pragma unroll
      for (int b = 0; b < MHC_N; ++b) x[b] = *reinterpret_cast<const f32x4_t*>(xt + b * h + c);
    }
#pragma unroll
    for (int i = 0; i < MHC_N; ++i) {
      f32x4_t o = v;
      if (MODE == MHC_ADD) o = x[i] + v;
      if (MODE == MHC_POST) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float a = p[i][0] * x[0][e];
#pragma unroll
          for (int j = 1; j < MHC_N; ++j) a = fmaf(p[i][j], x[j][e], a);
          o[e] = fmaf(w[i], v[e], a);
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) s = fmaf(o[e], o[e], s);
      *reinterpret_cast<f32x4_t*>(xt + i * h + c) = o;
    }
  }
  s = block_sum(s, red);
  if (threadIdx.x == 0) ssq[t] = s;
}

// Sublayer input and mixing coefficients (modeling:994-1031 and the zero-centred norm, :839-853) of TPB
// tokens per block: z = tanh((z0 r) B^T) with r the RMS factor of the token's 4 h values; pre =
// sigmoid(b_pre + a0 z), post = 2 sigmoid(b_post + a1 z); the 4 x 4 residual mix is Sinkhorn-normalised,
// sixteen lanes per token, one element each (row sums over lanes ^ 1, ^ 2, column sums over ^ 4, ^ 8).
// Then, one wave per token: xin = sum_b pre_b X_b, x = dt(xin / rms(xin) (1 + w)). 16 tokens per block
// keep every lane of the coefficient phase busy; 4 spread short prompts over the chip.
template <int TPB, int NCH, bool BF16>
__global__ __launch_bounds__(256) void mhc_pre_kernel(const float* __restrict__ X, const float* __restrict__ ssq,
                                                      const float* __restrict__ z0, const void* __restrict__ Bw,
                                                      const void* __restrict__ b_pre, const void* __restrict__ b_post,
                                                      const void* __restrict__ b_res,
                                                      const void* __restrict__ alphas,
                                                      const void* __restrict__ norm_w, void* __restrict__ x_out,
                                                      float* __restrict__ post, float* __restrict__ P, int64_t T,
                                                      int h, int rank, int iters, float eps) {
  constexpr int LD = 128 + 4;
  __shared__ __attribute__((aligned(16))) float zs[TPB][LD];
  __shared__ __attribute__((aligned(16))) float bs[MHC_COEF][LD];
  __shared__ float pre_s[TPB][MHC_N];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t t0 = (int64_t)blockIdx.x * TPB;
  for (int i = tid; i < MHC_COEF * rank; i += 256) bs[i / rank][i % rank] = ld_dt<BF16>(Bw, i);
  for (int i = tid; i < TPB * rank; i += 256) {
    const int64_t t = min(t0 + i / rank, T - 1);
    const float r = rsqrtf(ssq[t] / (float)(MHC_N * h) + 1e-6f);
    zs[i / rank][i % rank] = z0[t * rank + i % rank] * r;
  }
  __syncthreads();
  if (tid < TPB * 16) {
    const int u = tid >> 4, j = tid & 15;
    const int64_t t = t0 + u;
    float zr = 0.0f, zc = 0.0f;  // residual logit j, coefficient j % 8 (pre, post)
    for (int k = 0; k < rank; k += 4) {
      const f32x4_t z = *reinterpret_cast<const f32x4_t*>(&zs[u][k]);
      const f32x4_t br = *reinterpret_cast<const f32x4_t*>(&bs[8 + j][k]);
      const f32x4_t bc = *reinterpret_cast<const f32x4_t*>(&bs[j & 7][k]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        zr = fmaf(z[e], br[e], zr);
        zc = fmaf(z[e], bc[e], zc);
      }
    }
    zr = tanhf(zr);
    zc = tanhf(zc);
    if (j < MHC_N) {
      pre_s[u][j] = sigmoid_f32(ld_dt<BF16>(b_pre, j) + ld_dt<BF16>(alphas, 0) * zc);
    } else if (j < 2 * MHC_N && t < T) {
      post[t * MHC_N + j - MHC_N] = 2.0f * sigmoid_f32(ld_dt<BF16>(b_post, j - MHC_N) + ld_dt<BF16>(alphas, 1) * zc);
    }
    float l = ld_dt<BF16>(b_res, j) + ld_dt<BF16>(alphas, 2) * zr;
    float m = l;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) m = fmaxf(m, __shfl_xor(m, o));
    float v = expf(l - m);
    for (int it = 0; it < iters; ++it) {
      float s = v + __shfl_xor(v, 1);
      s += __shfl_xor(s, 2);
      v = v / fmaxf(s, 1e-9f);
      s = v + __shfl_xor(v, 4);
      s += __shfl_xor(s, 8);
      v = v / fmaxf(s, 1e-9f);
    }
    if (t < T) P[t * 16 + j] = v;
  }
  __syncthreads();
  f32x4_t wn[NCH];
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = 4 * lane + 256 * i;
    wn[i] = c < h ? ld4_dt<BF16>(norm_w, c) : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }
  for (int u = wave; u < TPB; u += 4) {
    const int64_t t = t0 + u;
    if (t >= T) break;
    const float* xt = X + t * MHC_N * h;
    f32x4_t x[MHC_N][NCH];
#pragma unroll
    for (int b = 0; b < MHC_N; ++b)
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        const int c = 4 * lane + 256 * i;
        x[b][i] = c < h ? *reinterpret_cast<const f32x4_t*>(xt + b * h + c) : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
      }
    f32x4_t o[NCH];
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < NCH; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float a = pre_s[u][0] * x[0][i][e];
#pragma unroll
        for (int b = 1; b < MHC_N; ++b) a = fmaf(pre_s[u][b], x[b][i][e], a);
        o[i][e] = a;
        s = fmaf(a, a, s);
      }
    const float r = rsqrtf(wave_sum(s) / (float)h + eps);
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = 4 * lane + 256 * i;
      if (c >= h) continue;
      f32x4_t y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = (o[i][e] * r) * (1.0f + wn[i][e]);
      st4_dt<BF16>(x_out, t * h + c, y);
    }
  }
}

}  // namespace

hipError_t launch_mhc_update(int mode, float* X, const void* y, const float* post, const float* P, float* ssq,
                             int64_t T, int h, bool bf16, hipStream_t stream) {
  if (T == 0) return hipSuccess;
#define Q38_MHC(M, B)                                                                                        \
  hipLaunchKernelGGL((mhc_update_kernel<M, B>), dim3((unsigned)T), dim3(256), 0, stream, X, y, post, P, ssq, h)
  if (mode == MHC_INIT) {
    if (bf16) Q38_MHC(MHC_INIT, true);
    else Q38_MHC(MHC_INIT, false);
  } else if (mode == MHC_ADD) {
    if (bf16) Q38_MHC(MHC_ADD, true);
    else Q38_MHC(MHC_ADD, false);
  } else {
    if (bf16) Q38_MHC(MHC_POST, true);
    else Q38_MHC(MHC_POST, false);
  }
#undef Q38_MHC
  return hipGetLastError();
}

template <int TPB, bool BF16>
static void launch_mhc_pre_t(const float* X, const float* ssq, const float* z0, const void* Bw, const void* b_pre,
                             const void* b_post, const void* b_res, const void* alphas, const void* norm_w,
                             void* x_out, float* post, float* P, int64_t T, int h, int rank, int iters, float eps,
                             hipStream_t stream) {
#define Q38_PRE(NCH)                                                                                             \
  case NCH:                                                                                                      \
    hipLaunchKernelGGL((mhc_pre_kernel<TPB, NCH, BF16>), dim3((unsigned)((T + TPB - 1) / TPB)), dim3(256), 0,    \
                       stream, X, ssq, z0, Bw, b_pre, b_post, b_res, alphas, norm_w, x_out, post, P, T, h, rank, \
                       iters, eps);                                                                              \
    break;
  switch ((h + 255) / 256) {
    Q38_PRE(1) Q38_PRE(2) Q38_PRE(3) Q38_PRE(4) Q38_PRE(5) Q38_PRE(6) Q38_PRE(7) Q38_PRE(8)
  }
#undef Q38_PRE
}

hipError_t launch_mhc_pre(const float* X, const float* ssq, const float* z0, const void* Bw, const void* b_pre,
                          const void* b_post, const void* b_res, const void* alphas, const void* norm_w,
                          void* x_out, float* post, float* P, int64_t T, int h, int rank, int iters, float eps,
                          bool bf16, hipStream_t stream) {
  if (T == 0) return hipSuccess;
  if (h > 2048 || h % 4 != 0 || rank > 128 || rank % 4 != 0) return hipErrorInvalidValue;
  // 16 tokens per block where that still makes two blocks per CU.
  const bool wide = T >= 32 * (int64_t)device_cus();
#define Q38_PRE_T(TPB, B)                                                                                        \
  launch_mhc_pre_t<TPB, B>(X, ssq, z0, Bw, b_pre, b_post, b_res, alphas, norm_w, x_out, post, P, T, h, rank, iters, \
                           eps, stream)
  if (wide) {
    if (bf16) Q38_PRE_T(16, true);
    else Q38_PRE_T(16, false);
  } else {
    if (bf16) Q38_PRE_T(4, true);
    else Q38_PRE_T(4, false);
  }
#undef Q38_PRE_T
  return hipGetLastError();
}

}  // namespace q38
