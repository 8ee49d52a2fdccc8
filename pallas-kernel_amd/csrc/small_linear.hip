// Bias-free projections of a few rows (decode steps): y_i = x W_i^T for up to kSmallMaxW
// weights of one input, x [M, K] with M <= 128, W_i [n_i, K] bf16, in one launch; and the
// low-rank gate's second matrix with the log-sigmoid gate. Reference: the dense layers and gate
// of tops/layers/gla.py:259-288, 343.
//
// What bounds it: the latency of one round of loads, and the L2 traffic of every block's x (128
// KB at M = 32, hidden 2048) beside its 64 KB of weights; the weights alone (25 MB for q, k, v,
// the gate's first matrix and the output gate) would take 5 us from HBM. A block takes 16 rows
// of one weight and all M rows of x; its eight waves split K, so that a wave's loads are issued
// before its first product, and their sums meet in LDS. Measured, M = 32, hidden 2048: 15 us for
// the five projections in one launch (five hipBLASLt calls: 43 us on the GPU and about 20 us
// each on the host, which is what a decode step waits for), 16 us for the output projection of
// float32 rows (a float32 GEMM and the weight's conversion: 19 us); the layer's decode step at
// batch 32 256 -> 123 us (85 us with a cheaper host path).
//
// bf16 x: bf16 MFMA 16x16x32, float32 sums, results rounded once. float32 x: each value enters
// as three bf16 (exactly; the weights are bf16), float32 results.
#include "common.hpp"
#include "kernels.hpp"

namespace tops {

namespace {

constexpr int SLW = 8;              // waves per block, each an eighth of K
constexpr int SLT = SLW * 64;
constexpr float kBf16Max = 3.38953139e38f;   // 0x7f7f0000
constexpr int SLP = 20;             // LDS row pitch: the 16 rows of a store spread over the banks

// Eight floats as three bf16 fragments that sum to them exactly. An infinity or NaN is the
// first part alone (the rest would be inf - inf), and a finite value that rounds to an infinity
// (from 0x7f7f8000) starts with the largest bf16 instead.
__device__ __forceinline__ void split8(const float (&x)[8], Frag<bf16> (&f)[3]) {
  float y[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t m = __float_as_uint(x[e]) & 0x7fffffffu;
    const bool finite = m < 0x7f800000u;
    y[e] = finite ? (m >= 0x7f7f8000u ? copysignf(kBf16Max, x[e]) : x[e]) : x[e];
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = pack2_bf16(y[2 * e], y[2 * e + 1]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float hi = e & 1 ? bf16_hi(w[e / 2]) : bf16_lo(w[e / 2]);
      const bool finite = (__float_as_uint(x[e]) & 0x7fffffffu) < 0x7f800000u;
      y[e] = finite ? (i == 0 ? x[e] : y[e]) - hi : 0.f;
    }
    f[i].d = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// w without its infinities and NaN (zeros in their place).
__device__ __forceinline__ Frag<bf16> finite_part(const Frag<bf16>& w) {
  const uint32_t x[4] = {w.d.x, w.d.y, w.d.z, w.d.w};
  uint32_t y[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t lo = (x[e] & 0x7f80u) != 0x7f80u ? 0xffffu : 0u;
    const uint32_t hi = (x[e] & 0x7f800000u) != 0x7f800000u ? 0xffff0000u : 0u;
    y[e] = x[e] & (lo | hi);
  }
  Frag<bf16> r;
  r.d = make_uint4(y[0], y[1], y[2], y[3]);
  return r;
}

}  // namespace

// MT: 16-row tiles of x. TX: x's type.
template <typename TX, int MT>
__global__ __launch_bounds__(SLT) void small_linear_kernel(SmallLinearArgs p) {
  extern __shared__ __attribute__((aligned(16))) float sl_sm[];
  // [SLW][MT * 16][SLP]: the waves' sums
  auto part = [&](int ww, int m) { return sl_sm + (ww * MT * 16 + m) * SLP; };
  int b = blockIdx.x, wi = 0;
#pragma unroll
  for (int i = 0; i < kSmallMaxW; ++i)   // the weight of this block's tile (uniform)
    if (wi == i && i < p.nw && b >= (p.n[i] + 15) / 16) {
      b -= (p.n[i] + 15) / 16;
      wi = i + 1;
    }
  const bf16* __restrict__ W = (const bf16*)p.w[0];
  void* y = p.y[0];
  int n = p.n[0];
#pragma unroll
  for (int i = 1; i < kSmallMaxW; ++i)
    if (wi == i) {
      W = (const bf16*)p.w[i];
      y = p.y[i];
      n = p.n[i];
    }
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int K = p.K, M = p.M, KW = K / SLW;   // this wave's columns: [w KW, + KW)
  const int n0 = b * 16;
  const bf16* wr = W + (long)min(n0 + li, n - 1) * K + w * KW + 8 * g;
  const TX* xr[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
    xr[t] = (const TX*)p.x + (long)min(t * 16 + li, M - 1) * K + w * KW + 8 * g;
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = zero4();
  // U steps of 32 columns at a time, their loads together (about 100 registers)
  constexpr int U = 32 / (int)sizeof(TX) / (MT < 2 ? 2 : MT);
  for (int k = 0; k < KW; k += 32 * U) {
    Frag<bf16> wf[U];
    uint4 xf[U][MT][sizeof(TX) / 2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = min(k + 32 * u, KW - 32);
      wf[u] = ld_frag(wr + c);
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int h = 0; h < (int)sizeof(TX) / 2; ++h)
          xf[u][t][h] = reinterpret_cast<const uint4*>(xr[t] + c)[h];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k + 32 * u >= KW) break;   // uniform
      // the lower parts of x are often 0: they leave out weights that are not finite, whose product
      // with x's first part has x's sign (or is NaN for x = 0) already
      Frag<bf16> wl;
      if constexpr (sizeof(TX) == 4) wl = finite_part(wf[u]);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        if constexpr (sizeof(TX) == 2) {
          Frag<bf16> f;
          f.d = xf[u][t][0];
          mma(acc[t], wf[u], f);
        } else {
          float x[8];
          Frag<bf16> f[3];
          __builtin_memcpy(x, &xf[u][t][0], 32);
          split8(x, f);
#pragma unroll
          for (int i = 2; i >= 1; --i) mma(acc[t], wl, f[i]);
          mma(acc[t], wf[u], f[0]);
        }
      }
    }
  }
  // accumulators: rows 4 g + r of the weight tile, column li = row of x
#pragma unroll
  for (int t = 0; t < MT; ++t)
    *reinterpret_cast<float4*>(part(w, t * 16 + li) + 4 * g) =
        make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
  __syncthreads();
  for (int i = threadIdx.x; i < MT * 16 * 4; i += SLT) {
    const int m = i >> 2, c = (i & 3) * 4;
    if (m >= M || n0 + c >= n) continue;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ww = 0; ww < SLW; ++ww) {
      const float4 a = *reinterpret_cast<const float4*>(part(ww, m) + c);
      s[0] += a.x;
      s[1] += a.y;
      s[2] += a.z;
      s[3] += a.w;
    }
    const long at = (long)m * n + n0 + c;
    if constexpr (sizeof(TX) == 4) {
      *reinterpret_cast<float4*>((float*)y + at) = make_float4(s[0], s[1], s[2], s[3]);
    } else {
      const uint2 o = make_uint2(pack2_bf16(s[0], s[1]), pack2_bf16(s[2], s[3]));
      if (p.f32_mask >> wi & 1)   // the rounded values, as floats
        *reinterpret_cast<float4*>((float*)y + at) =
            make_float4(bf16_lo(o.x), bf16_hi(o.x), bf16_lo(o.y), bf16_hi(o.y));
      else
        *reinterpret_cast<uint2*>((bf16*)y + at) = o;
    }
  }
}

// y[m][c] = max(log_sigmoid(bf16(x[m] . w[c] + bias[c])) inv_n, clamp): one thread per column,
// its weight row (R values, 16 in the layer) read once for LGM rows of x.
constexpr int LGM = 4;
__global__ __launch_bounds__(256) void low_rank_gate_kernel(
    const bf16* __restrict__ x, const bf16* __restrict__ w, const bf16* __restrict__ bias,
    bf16* __restrict__ y, int M, int N, int R, float inv_n, int has_clamp, float clamp) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= N) return;
  const int m0 = blockIdx.y * LGM;
  float s[LGM];
#pragma unroll
  for (int j = 0; j < LGM; ++j) s[j] = 0.f;
  for (int r = 0; r < R; r += 8) {
    const uint4 wv = *reinterpret_cast<const uint4*>(w + (long)c * R + r);
#pragma unroll
    for (int j = 0; j < LGM; ++j) {
      const uint4 xv = *reinterpret_cast<const uint4*>(x + (long)min(m0 + j, M - 1) * R + r);
      const uint32_t a[4] = {wv.x, wv.y, wv.z, wv.w}, b[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[j] = fmaf(bf16_lo(a[e]), bf16_lo(b[e]), s[j]);
        s[j] = fmaf(bf16_hi(a[e]), bf16_hi(b[e]), s[j]);
      }
    }
  }
  const float bv = bias ? to_f32(bias[c]) : 0.f;
#pragma unroll
  for (int j = 0; j < LGM; ++j) {
    if (m0 + j >= M) break;
    const float v = to_f32(from_f32<bf16>(s[j] + bv));
    // log_sigmoid(v) = min(v, 0) - log(1 + exp(-|v|)), as the gate's own kernel takes it
    float o = (fminf(v, 0.f) - __logf(1.f + __expf(-fabsf(v)))) * inv_n;
    if (has_clamp) o = fmaxf(o, clamp);
    y[(long)(m0 + j) * N + c] = from_f32<bf16>(o);
  }
}

template <typename TX, int MT>
static hipError_t launch_small_mt(const SmallLinearArgs& p, long blocks, hipStream_t st) {
  constexpr int lds = SLW * MT * 16 * SLP * 4;
  const hipError_t e = hipFuncSetAttribute((const void*)small_linear_kernel<TX, MT>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((small_linear_kernel<TX, MT>), dim3((unsigned)blocks), dim3(SLT), lds, st,
                     p);
  return hipGetLastError();
}

template <typename TX>
static hipError_t launch_small(const SmallLinearArgs& p, long blocks, hipStream_t st) {
  if (p.M <= 16) return launch_small_mt<TX, 1>(p, blocks, st);
  if (p.M <= 32) return launch_small_mt<TX, 2>(p, blocks, st);
  if (p.M <= 64) return launch_small_mt<TX, 4>(p, blocks, st);
  return launch_small_mt<TX, 8>(p, blocks, st);
}

hipError_t run_small_linear(const SmallLinearArgs& p, int x_dtype, hipStream_t st) {
  long blocks = 0;
  for (int i = 0; i < p.nw; ++i) blocks += (p.n[i] + 15) / 16;
  if (blocks == 0 || p.M == 0) return hipSuccess;
  return x_dtype == DT_F32 ? launch_small<float>(p, blocks, st)
                           : launch_small<bf16>(p, blocks, st);
}

hipError_t run_low_rank_gate(const void* x, const void* w, const void* bias, void* y, int M,
                             int N, int R, float inv_n, int has_clamp, float clamp,
                             hipStream_t st) {
  if (M == 0 || N == 0) return hipSuccess;
  hipLaunchKernelGGL(low_rank_gate_kernel, dim3((unsigned)((N + 255) / 256),
                                                (unsigned)((M + LGM - 1) / LGM)),
                     dim3(256), 0, st, (const bf16*)x, (const bf16*)w, (const bf16*)bias,
                     (bf16*)y, M, N, R, inv_n, has_clamp, clamp);
  return hipGetLastError();
}

}  // namespace tops
