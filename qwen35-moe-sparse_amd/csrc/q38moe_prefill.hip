// Kernels of the packed prefill's trunk around the MoE block: the mHC residual stream
// (modeling_qwen3_8_moe.py:994-1031), the Gated DeltaNet token mixer (132-349, 464-577) and the QSA
// attention (1117-1165). As torch operations these are chains of passes over large fp32 tensors (the
// four-branch stream alone is 268 MB at 4 x 4096 tokens and hidden 1024) and, for the delta rule's chunk
// loop, some 400 launches per layer. Here each pass over the stream is one kernel, the delta rule with its
// gated norm three, and the attention one. fp32 is computed in fp32 (MFMA forms with fp32 operands), and
// values are rounded to the parameters' dtype where the torch code rounds.
#include <type_traits>

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
// sixteen lanes per token, one element each (row sums over lanes ^ 1, ^ 2, column sums over ^ 4, ^ 8). Its
// maximum and clamped sums keep a NaN, as torch's amax and clamp do (v_maximum3_f32; fmaxf would drop it).
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
    for (int o = 1; o < 16; o <<= 1) m = __builtin_elementwise_maximum(m, __shfl_xor(m, o));
    float v = expf(l - m);
    for (int it = 0; it < iters; ++it) {
      float s = v + __shfl_xor(v, 1);
      s += __shfl_xor(s, 2);
      v = v / __builtin_elementwise_maximum(s, 1e-9f);
      s = v + __shfl_xor(v, 4);
      s += __shfl_xor(s, 8);
      v = v / __builtin_elementwise_maximum(s, 1e-9f);
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

// ---- Gated DeltaNet ---------------------------------------------------------------------------

// Causal depthwise convolution of 4 taps in fp32, rounded to dt, then SiLU rounded to dt
// (modeling:184-205): qkv, out [B, S, C]. A thread owns 4 channels and GDN_TS consecutive steps (a
// sliding window of rows in registers); products and sums are rounded one by one. 273 MB at 16384 x 4160 in
// bf16 take 101 us in a prefill and 88-92 us alone (3 TB/s, below the copy rate; as torch operations on
// transposed fp32 copies some 1.2 ms): arithmetic next to the loads, so that 32-bit thread ids and one
// conversion per two roundings gained (107 -> 101 us, 1024 x 4160 alone 10.6 -> 10.0, 64 x 192 5.7 -> 5.2).
// 8 channels per thread by 16-byte loads: 81 us at the first of these, but 12.5 and 7.2 us at the others
// (too few threads) and fp32 103 -> 122 us.
constexpr int GDN_TS = 8;

template <bool BF16>
__global__ __launch_bounds__(256) void gdn_conv_kernel(const void* __restrict__ qkv, const void* __restrict__ w,
                                                       void* __restrict__ out, uint32_t runs, int S, int C) {
  const uint32_t id = blockIdx.x * 256u + threadIdx.x;
  const uint32_t cq = (uint32_t)C / 4;
  const uint32_t run = id / cq;  // (sequence, run of GDN_TS steps)
  if (run >= runs) return;
  const int c = 4 * (int)(id - run * cq);
  const uint32_t per_seq = (uint32_t)(S + GDN_TS - 1) / GDN_TS;
  const uint32_t b = run / per_seq;
  const int s0 = (int)(run - b * per_seq) * GDN_TS;
  f32x4_t taps[4];  // taps[i]: the four taps of channel c + i
#pragma unroll
  for (int i = 0; i < 4; ++i) taps[i] = ld4_dt<BF16>(w, 4 * (int64_t)(c + i));
  const int64_t base = (int64_t)b * S * C + c;
  f32x4_t x[3 + GDN_TS];
#pragma unroll
  for (int j = 0; j < 3 + GDN_TS; ++j) {
    const int s = s0 - 3 + j;
    x[j] = s >= 0 && s < S ? ld4_dt<BF16>(qkv, base + (int64_t)s * C) : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }
#pragma unroll
  for (int j = 0; j < GDN_TS; ++j) {
    if (s0 + j >= S) break;
    f32x4_t y;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      y[i] = __fmul_rn(x[j][i], taps[i][0]);
#pragma unroll
      for (int k = 1; k < 4; ++k) y[i] = __fadd_rn(y[i], __fmul_rn(x[j + k][i], taps[i][k]));
    }
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
      float lo = y[i], hi = y[i + 1];
      if (BF16) unpack_bf16x2(pack_bf16x2(lo, hi), lo, hi);  // both rounded by one instruction
      y[i] = silu_f32(lo);
      y[i + 1] = silu_f32(hi);
    }
    st4_dt<BF16>(out, base + (int64_t)(s0 + j) * C, y);
  }
}

__device__ __forceinline__ f32x4_t mfma16x16x4(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The gated delta rule (modeling:215-349, per token 352-413) in chunks of 64 tokens, head width 64,
// as q38.prefill.gated_delta_rule evaluates it: with c the cumulative log-decays of a chunk,
//   A[t, s] = beta_t e^{c_t - c_s} k_t.k_s (s < t),  (I + A) [Dv | Dk] = [beta V | beta e^c K]
// (gdn_chunk_kernel, all chunks at once), then from chunk to chunk (gdn_scan_kernel)
//   D = Dv - Dk S,  O = (q e^c) S + (q k^T e^{c_t - c_s})_{s <= t} D,  S <- e^{c_63} S + (k e^{c_63 - c})^T D.
//
// v_mfma_f32_16x16x4_f32: operand lane l holds row (or column) l % 16 at k = l / 16, result lane l rows
// 4 (l / 16) + i of column l % 16. Products take K in the order k = 16 j + 4 (l / 16) + e, so an operand
// is a 16-byte run per lane and j ("fragment"), and a result tile of rows 16 j .. is, register for
// register, the right-hand fragment j of the next product. Matrices that the scan reads are kept in
// scratch in fragment order: [.][64 lanes][4], one coalesced 16-byte access per lane.
//
// At 4 x 4096 tokens and 39 value heads (9984 chunks) the chunk kernel takes 320 us, the scan 290 us and
// the norm below 62 us, where the torch operations of one layer took about 8 ms (some 400 launches; the
// scan alone 64 x 5 small products). The chunk kernel is bound by its MFMA and LDS latency chains (two
// workgroups per CU by LDS) and 598 MB of scratch written, the scan by its serial chain of 64 chunks x (two
// dependent products, two barriers): 624 workgroups, 2.4 per CU.
//
// Fragments per chunk and head, each 64 lanes x 4 floats: Dv 16, Dk 16, K' = (k e^{c_63 - c})^T 16, the
// lower triangle of q k^T 10; then rows' q factors and e^c.
constexpr int GDN_C = 64;
constexpr int GDN_FRAG = 256;  // floats per fragment
constexpr int GDN_OFF_DK = 16 * GDN_FRAG, GDN_OFF_KW = 32 * GDN_FRAG, GDN_OFF_QK = 48 * GDN_FRAG,
              GDN_OFF_META = 58 * GDN_FRAG;
constexpr int GDN_CHUNK_FLOATS = GDN_OFF_META + 2 * GDN_C;
// Tile (b, a), a <= b, of a lower triangle of 4 x 4 tiles: index b (b + 1) / 2 + a.
__device__ __forceinline__ int tri(int b, int a) { return b * (b + 1) / 2 + a; }

// One workgroup per (sequence, chunk, value head). The triangular solve is blocked by 16: the four
// diagonal blocks are inverted by forward substitution (a column per lane), everything else is MFMA;
// a wave owns 32 of the 128 right-hand columns, whose block solutions stay in its registers as the
// operands of the later blocks.
template <bool BF16>
__global__ __launch_bounds__(256) void gdn_chunk_kernel(const void* __restrict__ qkv, const void* __restrict__ b_lin,
                                                        const void* __restrict__ a_lin,
                                                        const void* __restrict__ A_log,
                                                        const void* __restrict__ dt_bias, float* __restrict__ ws,
                                                        int S, int nk, int nv) {
  constexpr int LD = 68;
  __shared__ __attribute__((aligned(16))) float Ks[GDN_C * LD];
  __shared__ __attribute__((aligned(16))) float Qs[GDN_C * LD];  // after the products: Dk, row-major
  __shared__ __attribute__((aligned(16))) float Vs[GDN_C * LD];
  __shared__ __attribute__((aligned(16))) float Af[10][GDN_FRAG];  // -A, fragments of tile rows
  __shared__ __attribute__((aligned(16))) float If[4][GDN_FRAG];   // inverses of I + A's diagonal blocks
  __shared__ float cs[GDN_C], ec[GDN_C], beta[GDN_C];
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = S / GDN_C;
  const int hv = (int)(blockIdx.x % nv), ci = (int)(blockIdx.x / nv) % n, bb = (int)(blockIdx.x / nv) / n;
  const int hk = hv / (nv / nk);
  const int C = (2 * nk + nv) * 64;
  const int64_t tok0 = (int64_t)bb * S + (int64_t)ci * GDN_C;
  float* const out = ws + ((int64_t)(bb * nv + hv) * n + ci) * GDN_CHUNK_FLOATS;

  {
    // Rows of q, k, v: thread = row tid / 4, 16 columns; q and k L2-normalised, q scaled by 64^-1/2.
    const int row = tid >> 2, c0 = 16 * (tid & 3);
    const int64_t at = (tok0 + row) * C;
    f32x4_t q[4], k[4];
    float sq = 0.0f, sk = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      q[i] = ld4_dt<BF16>(qkv, at + 64 * hk + c0 + 4 * i);
      k[i] = ld4_dt<BF16>(qkv, at + 64 * (nk + hk) + c0 + 4 * i);
      *reinterpret_cast<f32x4_t*>(&Vs[row * LD + c0 + 4 * i]) = ld4_dt<BF16>(qkv, at + 64 * (2 * nk + hv) + c0 + 4 * i);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sq = fmaf(q[i][e], q[i][e], sq);
        sk = fmaf(k[i][e], k[i][e], sk);
      }
    }
    sq += __shfl_xor(sq, 1);
    sk += __shfl_xor(sk, 1);
    sq += __shfl_xor(sq, 2);
    sk += __shfl_xor(sk, 2);
    const float rq = rsqrtf(sq + 1e-6f), rk = rsqrtf(sk + 1e-6f);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *reinterpret_cast<f32x4_t*>(&Qs[row * LD + c0 + 4 * i]) = q[i] * rq * 0.125f;
      *reinterpret_cast<f32x4_t*>(&Ks[row * LD + c0 + 4 * i]) = k[i] * rk;
    }
    if ((tid & 3) == 0) out[GDN_OFF_META + row] = rq;
  }
  if (wave == 0) {
    // Log-decays, their prefix sums in float64 (log-step doubling, rounded once), and beta.
    const float x = ld_dt<BF16>(a_lin, (tok0 + lane) * nv + hv) + ld_dt<BF16>(dt_bias, hv);
    const float sp = x > 20.0f ? x : log1pf(expf(x));
    double c = (double)(-expf(ld_dt<BF16>(A_log, hv)) * sp);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const double v = __shfl_up(c, o);
      if (lane >= o) c += v;
    }
    cs[lane] = (float)c;
    const float e = expf((float)c);
    ec[lane] = e;
    out[GDN_OFF_META + GDN_C + lane] = e;
    beta[lane] = round_dt<BF16>(sigmoid_f32(ld_dt<BF16>(b_lin, (tok0 + lane) * nv + hv)));
  }
  __syncthreads();

  // k_s.k_t and k_s.q_t for the tiles of the lower triangle, as products of rows s with rows t: the
  // result lane holds column t = 16 b + l % 16, rows s = 16 a + 4 (l / 16) + i, i.e. row t's fragment.
#pragma unroll
  for (int u = 0; u < 5; ++u) {
    const int pi = wave + 4 * u, pair = pi < 10 ? pi : pi - 10;
    const int b = pair >= 6 ? 3 : pair >= 3 ? 2 : pair >= 1 ? 1 : 0, a = pair - tri(b, 0);
    const float* rt = (pi < 10 ? Ks : Qs) + (16 * b + lr) * LD + 4 * lq;
    const float* rs = Ks + (16 * a + lr) * LD + 4 * lq;
    f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4_t x = *reinterpret_cast<const f32x4_t*>(rs + 16 * j);
      const f32x4_t y = *reinterpret_cast<const f32x4_t*>(rt + 16 * j);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = mfma16x16x4(x[e], y[e], acc);
    }
    const int t = 16 * b + lr;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int s = 16 * a + 4 * lq + i;
      const float d = s <= t ? expf(cs[t] - cs[s]) : 0.0f;
      acc[i] = pi < 10 ? (s < t ? -(beta[t] * acc[i] * d) : 0.0f) : acc[i] * d;
    }
    if (pi < 10) *reinterpret_cast<f32x4_t*>(&Af[pair][4 * lane]) = acc;
    else *reinterpret_cast<f32x4_t*>(out + GDN_OFF_QK + pair * GDN_FRAG + 4 * lane) = acc;
  }
  __syncthreads();

  {
    // Column lr of (I + A_bb)^-1 for block b = wave: x_t = delta - sum_{s < t} A[t, s] x_s.
    const float* blk = Af[tri(wave, wave)];
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      float v = t == lr ? 1.0f : 0.0f;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (4 * g >= t) break;
        const f32x4_t r = *reinterpret_cast<const f32x4_t*>(blk + 4 * (t + 16 * g));
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (4 * g + e < t) v = fmaf(r[e], x[4 * g + e], v);
      }
      x[t] = v;
    }
    if (lq == 0) {
#pragma unroll
      for (int t = 0; t < 16; ++t) If[wave][4 * (t + 16 * (lr >> 2)) + (lr & 3)] = x[t];
    }
  }
  __syncthreads();

#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int ct = 2 * wave + u;  // column tile: 0-3 of Dv, 4-7 of Dk
    f32x4_t X[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      f32x4_t acc;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 16 * b + 4 * lq + i;
        acc[i] = ct < 4 ? Vs[r * LD + 16 * ct + lr] * beta[r] : (Ks[r * LD + 16 * (ct - 4) + lr] * beta[r]) * ec[r];
      }
#pragma unroll
      for (int a = 0; a < b; ++a) {
        const f32x4_t f = *reinterpret_cast<const f32x4_t*>(&Af[tri(b, a)][4 * lane]);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = mfma16x16x4(f[e], X[a][e], acc);
      }
      const f32x4_t f = *reinterpret_cast<const f32x4_t*>(&If[b][4 * lane]);
      X[b] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int e = 0; e < 4; ++e) X[b] = mfma16x16x4(f[e], acc[e], X[b]);
      if (ct < 4) {
        *reinterpret_cast<f32x4_t*>(out + (4 * b + ct) * GDN_FRAG + 4 * lane) = X[b];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) Qs[(16 * b + 4 * lq + i) * LD + 16 * (ct - 4) + lr] = X[b][i];
      }
    }
  }
  __syncthreads();
  const float last = cs[GDN_C - 1];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    *reinterpret_cast<f32x4_t*>(out + GDN_OFF_DK + (4 * wave + j) * GDN_FRAG + 4 * lane) =
        *reinterpret_cast<const f32x4_t*>(&Qs[(16 * wave + lr) * LD + 16 * j + 4 * lq]);
    f32x4_t kw;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = 16 * j + 4 * lq + e;
      kw[e] = Ks[t * LD + 16 * wave + lr] * expf(last - cs[t]);
    }
    *reinterpret_cast<f32x4_t*>(out + GDN_OFF_KW + (4 * wave + j) * GDN_FRAG + 4 * lane) = kw;
  }
}

// The recurrence over chunks of one (sequence, value head) and 16 of its 64 value columns (they are
// independent): four workgroups per head, placed on one XCD (block b runs on XCD b % 8) so that the
// fragments they share come from its L2. Wave w owns rows 16 w .. of D, O and S; the S and D fragments
// of the others come through LDS, two barriers per chunk. Each operand register is reloaded for the
// next chunk as soon as it is used. O goes to o_frag in dt, fragment order [chunk][w][column tile].
template <bool BF16>
__global__ __launch_bounds__(256, 3) void gdn_scan_kernel(const void* __restrict__ qkv, const float* __restrict__ ws,
                                                          void* __restrict__ o_frag, int heads, int S, int nk,
                                                          int nv) {
  __shared__ __attribute__((aligned(16))) float Dx[4][GDN_FRAG];
  __shared__ __attribute__((aligned(16))) float Sx[4][GDN_FRAG];
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = (int)blockIdx.x >> 3, ct = m & 3, head = (m >> 2) * 8 + ((int)blockIdx.x & 7);
  if (head >= heads) return;
  const int n = S / GDN_C;
  const int bb = head / nv, hk = (head % nv) / (nv / nk);
  const int C = (2 * nk + nv) * 64;
  const float* ck = ws + (int64_t)head * n * GDN_CHUNK_FLOATS;
  const int64_t q0 = ((int64_t)bb * S + 16 * wave + lr) * C + 64 * hk + 4 * lq;
  auto frag = [&](const float* base, int off, int i) {
    return *reinterpret_cast<const f32x4_t*>(base + off + i * GDN_FRAG + 4 * lane);
  };
  f32x4_t s[4], dk[4], kw[4], qk[4], q[4], dv;
  float rq, eq, carry;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    s[j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    dk[j] = frag(ck, GDN_OFF_DK, 4 * wave + j);
    q[j] = ld4_dt<BF16>(qkv, q0 + 16 * j);
    kw[j] = frag(ck, GDN_OFF_KW, 4 * wave + j);
    qk[j] = frag(ck, GDN_OFF_QK, tri(wave, min(j, wave)));
  }
  dv = frag(ck, 0, 4 * wave + ct);
  rq = ck[GDN_OFF_META + 16 * wave + lr];
  eq = ck[GDN_OFF_META + GDN_C + 16 * wave + lr];
  carry = load_uniform(ck + GDN_OFF_META + 2 * GDN_C - 1);
  for (int i = 0; i < n; ++i) {
    const float* nx = i + 1 < n ? ck + GDN_CHUNK_FLOATS : ck;
    const int64_t qn = q0 + (int64_t)(i + 1 < n ? i + 1 : i) * GDN_C * C;
    f32x4_t d = {0.0f, 0.0f, 0.0f, 0.0f}, o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4_t qr;
#pragma unroll
      for (int e = 0; e < 4; ++e) qr[e] = ((q[j][e] * rq) * 0.125f) * eq;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        d = mfma16x16x4(dk[j][e], s[j][e], d);
        o = mfma16x16x4(qr[e], s[j][e], o);
      }
      dk[j] = frag(nx, GDN_OFF_DK, 4 * wave + j);
      q[j] = ld4_dt<BF16>(qkv, qn + 16 * j);
    }
    d = dv - d;
    *reinterpret_cast<f32x4_t*>(&Dx[wave][4 * lane]) = d;
    dv = frag(nx, 0, 4 * wave + ct);
    rq = nx[GDN_OFF_META + 16 * wave + lr];
    eq = nx[GDN_OFF_META + GDN_C + 16 * wave + lr];
    __syncthreads();
    f32x4_t sn = s[0];  // this wave's own rows of S
#pragma unroll
    for (int j = 1; j < 4; ++j) sn = j == wave ? s[j] : sn;
    sn = sn * carry;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4_t dj = *reinterpret_cast<const f32x4_t*>(&Dx[j][4 * lane]);
#pragma unroll
      for (int e = 0; e < 4; ++e) sn = mfma16x16x4(kw[j][e], dj[e], sn);
      if (j <= wave) {
#pragma unroll
        for (int e = 0; e < 4; ++e) o = mfma16x16x4(qk[j][e], dj[e], o);
      }
    }
    *reinterpret_cast<f32x4_t*>(&Sx[wave][4 * lane]) = sn;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      kw[j] = frag(nx, GDN_OFF_KW, 4 * wave + j);
      qk[j] = frag(nx, GDN_OFF_QK, tri(wave, min(j, wave)));
    }
    carry = load_uniform(nx + GDN_OFF_META + 2 * GDN_C - 1);
    st4_dt<BF16>(o_frag, (((int64_t)head * n + i) * 16 + 4 * wave + ct) * GDN_FRAG + 4 * lane, o);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] = *reinterpret_cast<const f32x4_t*>(&Sx[j][4 * lane]);
    ck = nx;
  }
}

// Gated RMS norm of the heads' outputs (modeling:132-148): normalise in fp32, round to dt, times w
// rounded, times silu(z) rounded; out [B, S, nv * 64]. One block per (chunk, head): the fragments are
// transposed through LDS, four threads per row of 64.
template <bool BF16>
__global__ __launch_bounds__(256) void gdn_norm_kernel(const void* __restrict__ o_frag, const void* __restrict__ z,
                                                       const void* __restrict__ w, void* __restrict__ out, int S,
                                                       int nv, float eps) {
  constexpr int LD = 68;
  __shared__ __attribute__((aligned(16))) float os[GDN_C * LD];
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lq = lane >> 4, wave = tid >> 6;
  const int n = S / GDN_C;
  const int hv = (int)(blockIdx.x % nv), ci = (int)(blockIdx.x / nv) % n, bb = (int)(blockIdx.x / nv) / n;
  const int64_t chunk = (int64_t)(bb * nv + hv) * n + ci;
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
    const f32x4_t v = ld4_dt<BF16>(o_frag, (chunk * 16 + 4 * wave + ct) * GDN_FRAG + 4 * lane);
#pragma unroll
    for (int i = 0; i < 4; ++i) os[(16 * wave + 4 * lq + i) * LD + 16 * ct + lr] = v[i];
  }
  __syncthreads();
  const int row = tid >> 2, c0 = 16 * (tid & 3);
  const int64_t at = ((int64_t)bb * S + ci * GDN_C + row) * nv * 64 + 64 * hv + c0;
  f32x4_t x[4];
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[i] = *reinterpret_cast<const f32x4_t*>(&os[row * LD + c0 + 4 * i]);
#pragma unroll
    for (int e = 0; e < 4; ++e) s = fmaf(x[i][e], x[i][e], s);
  }
  s += __shfl_xor(s, 1);
  s += __shfl_xor(s, 2);
  const float r = rsqrtf(s / 64.0f + eps);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x4_t zv = ld4_dt<BF16>(z, at + 4 * i), wv = ld4_dt<BF16>(w, c0 + 4 * i);
    f32x4_t y;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      y[e] = round_dt<BF16>(wv[e] * round_dt<BF16>(x[i][e] * r)) * silu_f32(zv[e]);
    st4_dt<BF16>(out, at + 4 * i, y);
  }
}

// ---- QSA block-sparse attention -----------------------------------------------------------------

// Zero-centred RMS norm of the query and key heads (64 wide) and the partial rotary embedding of their
// first `rot` features (modeling:1117-1143, 580-623), roundings as the torch code's: the norm to dt, both
// products of the rotation and their sum to dt. Queries come from the q projection [T, H, 128] (query,
// gate), keys from [T, KV, 64]. Sixteen lanes per head, 4 features each; feature i's partner i +- rot / 2
// lies in another of the lanes (rot a multiple of 8). HBM-bound: 65-69 us for 250 MB at 16384 x 40 heads
// (a dozen torch passes before).
template <bool BF16>
__global__ __launch_bounds__(256) void qsa_prep_kernel(const void* __restrict__ qg, const void* __restrict__ k,
                                                       const void* __restrict__ q_norm,
                                                       const void* __restrict__ k_norm,
                                                       const void* __restrict__ cos_t,
                                                       const void* __restrict__ sin_t, void* __restrict__ q_out,
                                                       void* __restrict__ k_out, int64_t rows, int S, int H, int KV,
                                                       int rot, float eps) {
  const int64_t row = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);  // (token, head): H query, KV key heads
  const int l16 = threadIdx.x & 15, c = 4 * l16;
  if (row >= rows) return;
  const int64_t t = row / (H + KV);
  const int hd = (int)(row - t * (H + KV));
  const bool is_q = hd < H;
  const f32x4_t x = is_q ? ld4_dt<BF16>(qg, (t * H + hd) * 128 + c) : ld4_dt<BF16>(k, (t * KV + hd - H) * 64 + c);
  const f32x4_t w = ld4_dt<BF16>(is_q ? q_norm : k_norm, c);
  float s = 0.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) s = fmaf(x[e], x[e], s);
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) s += __shfl_xor(s, o);
  const float r = rsqrtf(s / 64.0f + eps);
  f32x4_t y;
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = round_dt<BF16>((x[e] * r) * (1.0f + w[e]));
  const int half = rot / 2;
  const int src = (threadIdx.x & 48) + (c < half ? l16 + half / 4 : c < rot ? l16 - half / 4 : l16);
  f32x4_t p;
#pragma unroll
  for (int e = 0; e < 4; ++e) p[e] = __shfl(y[e], src);
  if (c < rot) {
    const int64_t at = (t % S) * rot + c;
    const f32x4_t cs = ld4_dt<BF16>(cos_t, at), sn = ld4_dt<BF16>(sin_t, at);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float turned = c < half ? -p[e] : p[e];
      y[e] = __fadd_rn(round_dt<BF16>(__fmul_rn(y[e], cs[e])), round_dt<BF16>(__fmul_rn(turned, sn[e])));
    }
  }
  if (is_q) st4_dt<BF16>(q_out, (t * H + hd) * 64 + c, y);
  else st4_dt<BF16>(k_out, (t * KV + hd - H) * 64 + c, y);
}

// Zero in the place of every infinite bf16 value.
__device__ __forceinline__ void drop_infinities(u32x4_t& v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if ((v[i] & 0x7fffu) == 0x7f80u) v[i] &= 0xffff0000u;
    if ((v[i] & 0x7fff0000u) == 0x7f800000u) v[i] &= 0xffffu;
  }
}

// Attention of each 64-query block over its selected 64-key blocks, times sigmoid of the gate
// (modeling:1143-1165): scores, softmax and sums in fp32. A workgroup takes the query block of one
// sequence and key head for `hpw` of the query heads that share it; the key and value blocks lie in LDS
// (128 KiB for 8 blocks), and each wave runs 16 queries of one head over all of them with its scores (512
// per query) in registers, so the softmax is one pass over exact maxima and nothing is rescaled.
//
// Scores are computed transposed (K rows x queries): result lane l holds 4 keys of query l % 16, which
// is, register for register, the right-hand operand of O^T = V^T P^T.
// bf16: K Q^T by mfma_f32_16x16x32_bf16 (exact products, fp32 sums). The fp32 probabilities enter V^T P^T
// as three bf16 parts by truncation, whose sum is the probability exactly (8 + 8 + 8 bits), so the
// products with the bf16 values are exact too and only the fp32 sums round, as in an fp32 product; V
// fragments come through the transposing LDS read, in the scores' key order. An infinite value times a
// part that is zero would be NaN where the fp32 product is infinite: a wave that sees a NaN repeats its
// sums with infinities in the high part's product alone (the test costs 350.7 -> 352.3 us, launched alone
// at the sizes below; 10.6 -> 10.8 at 1 x 192).
// fp32: mfma_f32_16x16x4_f32 for both; the values take the keys' place in LDS after the scores, so a wave
// runs one set of 16 queries (hpw = 2).
// VALU-bound (exponentials and the three-way split, about 15 operations per score) next to 4 K MFMA
// cycles per 16 queries: 385-400 us in a prefill of 4 x 4096 tokens, 38 heads on 2, 8 blocks (the torch operations,
// fp32 products on gathered blocks with 2.5 GB of scores in memory, about 5 ms).
template <bool BF16>
__global__ __launch_bounds__(512, 2) void qsa_attention_kernel(const void* __restrict__ q, const void* __restrict__ k,
                                                               const void* __restrict__ v,
                                                               const void* __restrict__ qg,
                                                               const int64_t* __restrict__ sel,
                                                               void* __restrict__ out, int S, int H, int KV, int kk,
                                                               int hpw, float scale) {
  constexpr int ROWB = BF16 ? 128 : 256;  // bytes per row of 64
  constexpr int CPR = ROWB / 16;
  __shared__ __attribute__((aligned(16))) uint8_t buf[512 * 256];
  uint8_t* const kbuf = buf;
  uint8_t* const vbuf = BF16 ? buf + 512 * 128 : buf;
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nb = S / 64, G = H / KV;
  const int qb = (int)blockIdx.x % nb, b = (int)blockIdx.x / nb, g = (int)blockIdx.y;
  const int h0 = g * G + (int)blockIdx.z * hpw, hn = min(hpw, (g + 1) * G - h0);
  const int nblk = min(qb + 1, kk);
  const int64_t tok0 = (int64_t)b * S;
  int kb[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    kb[j] = j < nblk ? min(max((int)load_uniform(sel + ((int64_t)b * nb + qb) * kk + j), 0), nb - 1) : 0;

  auto copy_blocks = [&](const void* src, uint8_t* dst, bool values) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j >= nblk) break;
#pragma unroll
      for (int i = 0; i < CPR / 8; ++i) {
        const int id = i * 512 + tid, r = id / CPR, pos = id % CPR;
        const int c = pos ^ (!BF16 ? r & 15 : values ? 2 * ((r >> 1) & 3) : r & 7);
        const uint8_t* s = static_cast<const uint8_t*>(src) + ((tok0 + 64 * kb[j] + r) * KV + g) * ROWB + 16 * c;
        load_lds16(s, dst + j * 64 * ROWB + 16 * (i * 512 + 64 * wave));
      }
    }
  };
  copy_blocks(k, kbuf, false);
  if (BF16) copy_blocks(v, vbuf, true);
  wait_vmcnt0();
  __syncthreads();

  const uint32_t vbase = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)vbuf;
  typedef short i16x4_t __attribute__((ext_vector_type(4)));
  const int tasks = 4 * hn;  // (head, 16 queries)
  for (int task = wave; BF16 ? task < tasks : task == wave; task += 8) {
    const bool on = task < tasks;  // fp32: every wave passes the barriers
    const int head = h0 + (on ? task >> 2 : 0), rg = task & 3;
    const int64_t qtok = tok0 + 64 * qb + 16 * rg + lr;
    f32x4_t sc[8][4];
    const int64_t qat = (qtok * H + head) * 64;
    u32x4_t qf16[2];
    f32x4_t qf32[4];
    if (BF16) {
#pragma unroll
      for (int s = 0; s < 2; ++s) qf16[s] = ld16(static_cast<const uint16_t*>(q) + qat + 32 * s + 8 * lq);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) qf32[j] = ld4_dt<false>(q, qat + 16 * j + 4 * lq);
    }
    float m = -__builtin_inff();
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j >= nblk) break;
      // Keys past the query: key position 64 kb + 16 t + 4 lq + i > 64 qb + 16 rg + lr.
      const int ahead = 64 * (kb[j] - qb) - 16 * rg - lr;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = 64 * j + 16 * t + lr;
        f32x4_t a = {0.0f, 0.0f, 0.0f, 0.0f};
        if (BF16) {
#pragma unroll
          for (int s = 0; s < 2; ++s)
            a = mfma16x16x32(ld16(kbuf + r * ROWB + (((4 * s + lq) ^ (r & 7)) << 4)), qf16[s], a);
        } else {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const f32x4_t f = *reinterpret_cast<const f32x4_t*>(kbuf + r * ROWB + (((4 * u + lq) ^ (r & 15)) << 4));
#pragma unroll
            for (int e = 0; e < 4; ++e) a = mfma16x16x4(f[e], qf32[u][e], a);
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          a[i] = ahead + 16 * t + 4 * lq + i > 0 ? -__builtin_inff() : a[i] * scale;
          m = fmaxf(m, a[i]);
        }
        sc[j][t] = a;
      }
    }
    m = fmaxf(m, __shfl_xor(m, 16));
    m = fmaxf(m, __shfl_xor(m, 32));
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j >= nblk) break;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          sc[j][t][i] = expf(sc[j][t][i] - m);
          sum += sc[j][t][i];
        }
    }
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    if (!BF16) {
      __syncthreads();
      copy_blocks(v, vbuf, true);
      wait_vmcnt0();
      __syncthreads();
    }
    f32x4_t o[4];
    auto weigh_bf16 = [&](auto infinite) {
#pragma unroll
      for (int d = 0; d < 4; ++d) o[d] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (j >= nblk) break;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          // Probabilities of keys 32 u + {4 lq + e, 16 + 4 lq + e}: high, middle and low 8 bits.
          u32x4_t part[3];
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            float x0 = sc[j][2 * u + (w >> 1)][2 * (w & 1)], x1 = sc[j][2 * u + (w >> 1)][2 * (w & 1) + 1];
#pragma unroll
            for (int z = 0; z < 3; ++z) {
              const uint32_t b0 = __float_as_uint(x0), b1 = __float_as_uint(x1);
              part[z][w] = __builtin_amdgcn_perm(b1, b0, 0x07060302u);  // high halves, x0 low
              x0 -= __uint_as_float(b0 & 0xffff0000u);
              x1 -= __uint_as_float(b1 & 0xffff0000u);
            }
          }
          const int key = 64 * j + 32 * u + 4 * lq + (lr >> 2);  // row this lane addresses (second read: + 16)
          const uint32_t row = vbase + key * 128;
          const int sw = 2 * ((key >> 1) & 3);
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            const uint32_t at = row + ((((2 * d + ((lr & 3) >> 1)) ^ sw) << 4) | (8 * (lr & 1)));
            typedef __attribute__((address_space(3))) i16x4_t* lds_t;
            const uint2 x = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(uintptr_t)at));
            const uint2 y =
                __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(uintptr_t)(at + 16 * 128)));
            u32x4_t vf = {x.x, x.y, y.x, y.y};
#pragma unroll
            for (int z = 0; z < 3; ++z) {
              if (decltype(infinite)::value && z == 1) drop_infinities(vf);
              o[d] = mfma16x16x32(vf, part[z], o[d]);
            }
          }
        }
      }
    };
    if constexpr (BF16) {
      weigh_bf16(std::false_type{});
      float any = 0.0f;  // NaN if a sum is (or sums of both infinities meet)
#pragma unroll
      for (int d = 0; d < 4; ++d) any += (o[d][0] + o[d][1]) + (o[d][2] + o[d][3]);
      if (__builtin_expect(ballot64(any != any) != 0, 0)) weigh_bf16(std::true_type{});
    } else {
#pragma unroll
      for (int d = 0; d < 4; ++d) o[d] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (j >= nblk) break;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int key = 64 * j + 16 * t + 4 * lq + e;
#pragma unroll
            for (int d = 0; d < 4; ++d) {
              const float vf = *reinterpret_cast<const float*>(
                  vbuf + key * ROWB + (((4 * d + (lr >> 2)) ^ (key & 15)) << 4) + 4 * (lr & 3));
              o[d] = mfma16x16x4(vf, sc[j][t][e], o[d]);
            }
          }
      }
    }
    if (!on) continue;
    // Lane: features 16 d + 4 lq .. + 3 of query lr.
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int c = 16 * d + 4 * lq;
      const f32x4_t gate = ld4_dt<BF16>(qg, (qtok * H + head) * 128 + 64 + c);
      f32x4_t y;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        y[e] = round_dt<BF16>(o[d][e] / sum) * round_dt<BF16>(sigmoid_f32(gate[e]));
      st4_dt<BF16>(out, qat + c, y);
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

hipError_t launch_gdn_conv(const void* qkv, const void* w, void* out, int64_t B, int S, int C, bool bf16,
                           hipStream_t stream) {
  const int64_t runs = B * ((S + GDN_TS - 1) / GDN_TS);
  if (runs == 0) return hipSuccess;
  if (runs * (C / 4) + 255 >= (int64_t)1 << 32) return hipErrorInvalidValue;  // 32-bit thread ids
  const dim3 grid((unsigned)((runs * (C / 4) + 255) / 256));
  if (bf16) hipLaunchKernelGGL(gdn_conv_kernel<true>, grid, dim3(256), 0, stream, qkv, w, out, (uint32_t)runs, S, C);
  else hipLaunchKernelGGL(gdn_conv_kernel<false>, grid, dim3(256), 0, stream, qkv, w, out, (uint32_t)runs, S, C);
  return hipGetLastError();
}

size_t gdn_workspace_floats(int64_t B, int S, int nv) { return (size_t)B * nv * (S / GDN_C) * GDN_CHUNK_FLOATS; }

template <bool BF16>
static hipError_t launch_gdn_delta_t(const void* qkv, const void* b_lin, const void* a_lin, const void* A_log,
                                     const void* dt_bias, const void* z, const void* norm_w, float* ws, void* o_frag,
                                     void* out, int64_t B, int S, int nk, int nv, float eps, hipStream_t stream) {
  const unsigned chunks = (unsigned)(B * nv * (S / GDN_C));
  hipLaunchKernelGGL(gdn_chunk_kernel<BF16>, dim3(chunks), dim3(256), 0, stream, qkv, b_lin, a_lin, A_log, dt_bias, ws,
                     S, nk, nv);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int heads = (int)(B * nv);
  hipLaunchKernelGGL(gdn_scan_kernel<BF16>, dim3((unsigned)((heads + 7) / 8 * 32)), dim3(256), 0, stream, qkv, ws,
                     o_frag, heads, S, nk, nv);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(gdn_norm_kernel<BF16>, dim3(chunks), dim3(256), 0, stream, o_frag, z, norm_w, out, S, nv, eps);
  return hipGetLastError();
}

hipError_t launch_gdn_delta(const void* qkv, const void* b_lin, const void* a_lin, const void* A_log,
                            const void* dt_bias, const void* z, const void* norm_w, float* ws, void* o_frag, void* out,
                            int64_t B, int S, int nk, int nv, float eps, bool bf16, hipStream_t stream) {
  if (B == 0 || S == 0) return hipSuccess;
  if (S % GDN_C != 0 || nv % nk != 0) return hipErrorInvalidValue;
  return bf16 ? launch_gdn_delta_t<true>(qkv, b_lin, a_lin, A_log, dt_bias, z, norm_w, ws, o_frag, out, B, S, nk, nv,
                                         eps, stream)
              : launch_gdn_delta_t<false>(qkv, b_lin, a_lin, A_log, dt_bias, z, norm_w, ws, o_frag, out, B, S, nk, nv,
                                          eps, stream);
}

hipError_t launch_qsa_prep(const void* qg, const void* k, const void* q_norm, const void* k_norm, const void* cos_t,
                           const void* sin_t, void* q_out, void* k_out, int64_t T, int S, int H, int KV, int rot,
                           float eps, bool bf16, hipStream_t stream) {
  const int64_t rows = T * (H + KV);
  if (rows == 0) return hipSuccess;
  const dim3 grid((unsigned)((rows + 15) / 16));
  if (bf16)
    hipLaunchKernelGGL(qsa_prep_kernel<true>, grid, dim3(256), 0, stream, qg, k, q_norm, k_norm, cos_t, sin_t, q_out,
                       k_out, rows, S, H, KV, rot, eps);
  else
    hipLaunchKernelGGL(qsa_prep_kernel<false>, grid, dim3(256), 0, stream, qg, k, q_norm, k_norm, cos_t, sin_t, q_out,
                       k_out, rows, S, H, KV, rot, eps);
  return hipGetLastError();
}

hipError_t launch_qsa_attention(const void* q, const void* k, const void* v, const void* qg, const int64_t* sel,
                                void* out, int64_t B, int S, int H, int KV, int kk, float scale, bool bf16,
                                hipStream_t stream) {
  if (B == 0 || S == 0) return hipSuccess;
  if (S % 64 != 0 || H % KV != 0 || kk < 1 || kk > 8) return hipErrorInvalidValue;
  // Four heads per workgroup (two rounds of its eight waves on one copy of the blocks) where that still
  // gives every CU a few workgroups; two heads, and always in fp32, otherwise.
  const int G = H / KV;
  const int hpw = bf16 && B * (S / 64) * KV * ((G + 3) / 4) >= 2 * device_cus() ? 4 : 2;
  const dim3 grid((unsigned)(B * (S / 64)), (unsigned)KV, (unsigned)((G + hpw - 1) / hpw));
  if (bf16)
    hipLaunchKernelGGL(qsa_attention_kernel<true>, grid, dim3(512), 0, stream, q, k, v, qg, sel, out, S, H, KV, kk, hpw,
                       scale);
  else
    hipLaunchKernelGGL(qsa_attention_kernel<false>, grid, dim3(512), 0, stream, q, k, v, qg, sel, out, S, H, KV, kk,
                       hpw, scale);
  return hipGetLastError();
}

}  // namespace q38
