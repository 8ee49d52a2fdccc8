// Fused recurrent GLA forward for bf16 inputs on the matrix cores, at float32 accuracy: the
// recurrence
//   S_t = e^{g_t} (.) S_{t-1} + k_t v_t^T,  o_t = scale q_t S_t   (reference:
// tops/ops/gla/fused_recurrent.py:139-227) taken 16 tokens at a time. With E_i the gates'
// sum from the middle of the 16 tokens to token i (negative before it: E_7 = 0, E_8 = g_8),
// qa_i = q_i e^{E_i}, ka_j = k_j e^{-E_j} and S' the state decayed to the middle,
//   o_i = scale (qa_i S' + sum_{j <= i} (qa_i . ka_j) v_j),   S <- e^{E_15} (S' + ka^T v).
//
// Precision. qa, ka, S' and A = qa ka^T are float32 and enter the bf16 MFMAs as exact sums of
// three bf16 (v is bf16 already): six products for qa S' and A, three for A v and ka^T v, all
// accumulated in float32. Both gate sums are taken from the middle outwards, so no exponent is
// a difference of sums, and an exponential's argument is carried as a rounded product and its
// remainder. Error against float64 (2-norm, B8 T2048 H4 K256 V512): o 9.6e-8, ht 7.1e-8; the
// VALU scan of recurrent.hip, which rounds the state at every token, has 1.4e-7 and 1.1e-7.
//
// What bounds it: VALU issue of the splits and of the producers' exponentials (bf16 MFMAs run
// beside other waves' VALU work; float32 MFMAs do not -- 923 us of them and 575 us of FMAs in
// another wave of the SIMD took 1444 us together, bf16 ones 971 -> 986 -- and are a sixteenth
// as fast: this kernel with them ran at 520 us instead of 458). The state never leaves the
// registers: a wave holds all K rows of 16 (or 32) columns as accumulators (rows 4g + r,
// column l & 15 in lane l = 16 g + column), which is also the B operand of an MFMA over those
// rows, so qa S' and ka^T v need no transposition and no exchange between waves. Measured: B8
// T2048 H4 K256 V512 951 -> 458 us, B64 T64 H16 K=V=128 131 -> 101 us (92 with inputs left in
// the caches), B3 T1000 H16 K=V=64 317 -> 149 us (the VALU scan and this kernel). VALU busy 65 %,
// the MFMA pipe 29 % in the first.
//
// Block = (sequence, head, 64 or 128 columns): four consumer waves, each 16 or 32 columns,
// and KP / 64 producer waves. While the consumers work on tokens 16 n .., the producers make
// qa, ka, the 16 x 16 products A (each over its own 64 key columns, summed by the reader) and
// the decays of the next 16 in the other LDS buffer: one barrier per 16 tokens.
//
// Range. A factored operand above 2^50 (gates below about -4 a token over half a chunk) or not
// finite, a half's decay above 8 or NaN (the first row's gate is in the decays alone, not in an
// operand), a v above 2^20 or not finite, an infinite state or one above 2^56: the block takes the
// sequence from that chunk on as the recurrence is written, on the VALU (below), so that
// non-finite values stay where the recurrence puts them; after 8 chunks, then 32 and so on, it
// comes back to the matrix cores. Measured, the VALU scan of recurrent.hip and this kernel, gates
// near -8 / one gate of -60 in a sequence: B8 T2048 H4 K256 V512 950 and 943 / 491 us, B8 T2048
// H16 K=V=128 666 and 586 / 377, B3 T1000 H16 K=V=64 313 and 205 / 160; only the start weighs on
// short sequences (B64 T64 H16 K=V=128 124 and 159 / 145). Without a way back the dense gates took
// 921, 561, 198 and 159 us, a single one up to as much; token by token from the registers of the
// matrix path a chunk cost 15 to 37 us in place of 3.6.
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace tops {

namespace {

constexpr int QC = 16;             // tokens per chunk
constexpr int QCW = 4;             // consumer waves
constexpr int QTP = 20;            // LDS pitch (floats) of rows of 16
constexpr float kOperandMax = 1125899906842624.f;   // 2^50
constexpr float kStateMax = 72057594037927936.f;    // 2^56
constexpr float kDecayWeight = 1.5845633e29f;       // 2^97
constexpr uint32_t kValueMaxBits = 0x4980u;         // 2^20 as bf16

constexpr int RTB = 8;             // tokens per stage of the element-wise phase
constexpr int kSpan = 8;           // chunks of its first stretch; each is four times the one before

template <int KP, int NVT>
struct QLayout {   // byte offsets of one buffer
  static constexpr int QP = KP + 8, KQ = KP + 16;    // row pitches (bf16) of qa and ka
  static constexpr int PW = KP / 64;                 // producer waves
  static constexpr int qa = 0;                       // [3][16][QP] bf16
  static constexpr int ka = qa + 3 * QC * QP * 2;    // [3][16][KQ] bf16
  static constexpr int A = ka + 3 * QC * KQ * 2;     // [PW][16][QTP] f32
  // decays f32 [KP] each, in the order of the producers' row groups: the previous chunk's
  // post x pre; pre = e^{sum of rows 0..7}; post = e^{sum of rows 8..15}; the previous post
  static constexpr int dec = A + PW * QC * QTP * 4;
  static constexpr int pre = dec + KP * 4, post = pre + KP * 4, ppost = post + KP * 4;
  static constexpr int flag = ppost + KP * 4;        // [4] of the producers, [4] of the consumers
  static constexpr int buf = flag + 32;
  // element-wise phase, in the same place: k, so q, e^g [RTB][KP] and v [RTB][CB] f32, twice; the
  // consumers' sums [QCW][RTB][CB] f32, twice; before it the state [KP][CB + 4] f32
  static constexpr int CB = QCW * NVT * 16;
  static constexpr int stage = RTB * (3 * KP + CB) * 4, sums = QCW * RTB * CB * 4;
  static constexpr int cmax(int a, int b) { return a > b ? a : b; }
  static constexpr int bytes =
      cmax(2 * buf, cmax(2 * (stage + sums), KP * (CB + 4) * 4));
};

constexpr float kLog2e = 1.44269502162933349609375f;   // log2(e) rounded to float
constexpr float kLog2eRest = 1.92596299e-8f;           // log2(e) - kLog2e
// e^x and e^-x to about an ulp at any size of x: x log2(e) as a rounded product plus its
// remainder.
__device__ __forceinline__ void exp_pair(float x, float& p, float& n) {
  const float hi = x * kLog2e;
  const float lo = fmaf(x, kLog2eRest, fmaf(x, kLog2e, -hi)) * 0.693147181f;
  p = __builtin_amdgcn_exp2f(hi);
  n = __builtin_amdgcn_exp2f(-hi);
  p = fmaf(p, lo, p);
  n = fmaf(n, -lo, n);
}
// e^x alone, for the decays. Where x log2(e) passes the float range (x = -inf among them) the
// remainder is inf - inf; the maximum drops that NaN, so that e^x is 0 there (a NaN x stays).
__device__ __forceinline__ float exp_one(float x) {
  const float hi = x * kLog2e;
  const float lo = fmaf(x, kLog2eRest, fmaf(x, kLog2e, -hi)) * 0.693147181f;
  const float p = __builtin_amdgcn_exp2f(hi);
  return fmaf(p, fmaxf(lo, -1.f), p);
}

__device__ __forceinline__ float comp(const float4& x, int i) {   // i known once unrolled
  return i == 0 ? x.x : i == 1 ? x.y : i == 2 ? x.z : x.w;
}

__device__ __forceinline__ float4 add4(const float4& a, const float4& b) {
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}

// Four floats as the sum of three bf16 each, exactly: x rounded to bf16, the rest rounded, and
// the rest of that (8 significand bits each and a sign). Rounded rather than cut off, the
// lower parts have either sign, so that the products of two lower parts, which are left out
// below, do not add up (cut off, o came out 7e-8 to 1e-7 too small).
struct Split {
  s4_t p[3];
};
__device__ __forceinline__ Split split3(const float (&x)[4]) {
  Split r;
  float y[4] = {x[0], x[1], x[2], x[3]};
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const uint2 w = make_uint2(pack2_bf16(y[0], y[1]), pack2_bf16(y[2], y[3]));
    r.p[i] = __builtin_bit_cast(s4_t, w);
    if (i < 2) {
      y[0] -= bf16_lo(w.x);
      y[1] -= bf16_hi(w.x);
      y[2] -= bf16_lo(w.y);
      y[3] -= bf16_hi(w.y);
    }
  }
  return r;
}

__device__ __forceinline__ f32x4 mma16(const s4_t& a, const s4_t& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
// a . b of split operands: of the nine products of their parts the six that reach a float's
// last bit, in sums of their own (no product waits on the one before it).
__device__ __forceinline__ void mma_split(const s4_t (&a)[3], const s4_t (&b)[3], f32x4& main,
                                          f32x4 (&rest)[3]) {
  main = mma16(a[0], b[0], main);
  rest[0] = mma16(a[2], b[0], rest[0]);
  rest[1] = mma16(a[0], b[2], rest[1]);
  rest[2] = mma16(a[1], b[1], rest[2]);
  rest[0] = mma16(a[1], b[0], rest[0]);
  rest[1] = mma16(a[0], b[1], rest[1]);
}

}  // namespace

// The element-wise phase: tokens t0 .. t1 - 1 as the recurrence is written, from and (`again`) to a
// state in LDS.
// The producers stage RTB tokens' k, so q, e^g and v as floats and write the outputs of the stage
// before; a consumer wave has KP / 4 state rows of all CB columns, a lane KP / 16 rows of four
// (eight) columns, so that an operand read from LDS meets four products, and its sums over the
// rows meet the other waves' in LDS. VALU issue bounds it (three operations a state value); one
// barrier a stage, a token's LDS reads under the products of the one before (944 -> 921 us at B8
// T2048 H4 K256 V512).
template <int KP, int NVT, bool VEC>
__device__ __forceinline__ void rec_elements_producer(const RecScanArgs& p, unsigned char* qsm,
                                                      int t0, int t1, bool again, int bos,
                                                      int eos, int hh, int ct, int pw, int lane) {
  using Lay = QLayout<KP, NVT>;
  constexpr int PW = Lay::PW, CB = Lay::CB, NV = RTB * CB / (PW * 64);
  asm volatile("" : "+v"(lane));   // nothing that depends on it is kept over the matrix path
  const int H = p.H, K = p.R, V = p.C;
  const long rsK = (long)H * K, rsV = (long)H * V;
  const bf16* q = (const bf16*)p.o + (long)hh * K;
  const bf16* k = (const bf16*)p.a + (long)hh * K;
  const bf16* gk = (const bf16*)(p.ga ? p.ga : p.a) + (long)hh * K;
  const bf16* v = (const bf16*)p.b + (long)hh * V;
  const uint32_t gmask = p.ga ? ~0u : 0u;
  const int NS = (t1 - t0 + RTB - 1) / RTB, c0 = pw * 64 + 4 * (lane & 15);
  auto tok = [&](int t) { return (long)(p.dir ? eos - 1 - t : bos + t); };
  uint2 raw[2][3];      // two tokens of four key columns
  uint32_t rv[NV];      // values: token and column of index (i PW + pw) 64 + lane
  auto load = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const long at = tok(min(t0 + s * RTB + 2 * (lane >> 4) + u, t1 - 1)) * rsK;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const bf16* base = (a == 0 ? q : a == 1 ? k : gk) + at;
        if constexpr (VEC) {
          raw[u][a] = *reinterpret_cast<const uint2*>(base + max(min(c0, K - 4), 0));
        } else {
          uint32_t x[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] = base[min(c0 + e, K - 1)].u;
          raw[u][a] = make_uint2(x[0] | (x[1] << 16), x[2] | (x[3] << 16));
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int x = (i * PW + pw) * 64 + lane;
      rv[i] = v[tok(min(t0 + s * RTB + x / CB, t1 - 1)) * rsV + min(ct * CB + x % CB, V - 1)].u;
    }
  };
  auto store = [&](int s) __attribute__((always_inline)) {   // tokens past the end are not read
    float* B = reinterpret_cast<float*>(qsm + (s & 1) * Lay::stage);
    uint32_t cm[2];
#pragma unroll
    for (int e = 0; e < 2; ++e)
      cm[e] = (c0 + 2 * e < K ? 0xffffu : 0u) | (c0 + 2 * e + 1 < K ? 0xffff0000u : 0u);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int at = (2 * (lane >> 4) + u) * KP + c0;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const uint32_t m = a == 2 ? gmask : ~0u;
        const uint32_t x = raw[u][a].x & cm[0] & m, y = raw[u][a].y & cm[1] & m;
        float f[4] = {bf16_lo(x), bf16_hi(x), bf16_lo(y), bf16_hi(y)};
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = a == 0 ? p.so * f[e] : a == 2 ? gexp<bf16>(f[e]) : f[e];
        // k, so q, e^g
        *reinterpret_cast<float4*>(B + (a == 0 ? 1 : a == 1 ? 0 : 2) * RTB * KP + at) =
            make_float4(f[0], f[1], f[2], f[3]);
      }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int x = (i * PW + pw) * 64 + lane;
      B[3 * RTB * KP + x] = ct * CB + x % CB < V ? bf16_lo(rv[i]) : 0.f;
    }
  };
  auto output = [&](int s) __attribute__((always_inline)) {
    const float* O = reinterpret_cast<const float*>(qsm + 2 * Lay::stage + (s & 1) * Lay::sums);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int x = (i * PW + pw) * 64 + lane, t = t0 + s * RTB + x / CB, c = ct * CB + x % CB;
      if (t < t1 && c < V)
        ((float*)p.out)[tok(t) * rsV + (long)hh * V + c] =
            (O[x] + O[RTB * CB + x]) + (O[2 * RTB * CB + x] + O[3 * RTB * CB + x]);
    }
  };
  load(0);
  __syncthreads();
  __syncthreads();   // the state is in LDS
  __syncthreads();   // and out of it
  store(0);
  if (NS > 1) load(1);
  for (int s = 0; s < NS; ++s) {
    __syncthreads();
    if (s + 1 < NS) store(s + 1);
    if (s + 2 < NS) load(s + 2);
    if (s > 0) output(s - 1);
  }
  __syncthreads();
  output(NS - 1);
  if (again) {
    __syncthreads();   // the sums are read
    __syncthreads();   // the state is in LDS
    __syncthreads();   // and out of it
  }
}

template <int KP, int NVT>
__device__ __forceinline__ void rec_elements_consumer(const RecScanArgs& p, unsigned char* qsm,
                                                      int t0, int t1, bool again, float* sN,
                                                      int ct, int w, int lane) {
  using Lay = QLayout<KP, NVT>;
  constexpr int CB = Lay::CB, R = KP / 16;
  const int K = p.R, V = p.C;
  asm volatile("" : "+v"(lane));   // as above
  const int cg = 4 * (lane & 15), r0 = (w * 4 + (lane >> 4)) * R;
  const int NS = (t1 - t0 + RTB - 1) / RTB;
  float S[R][NVT][4];
  __syncthreads();   // the state is in LDS
  {
    const float* X = reinterpret_cast<const float*>(qsm);
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
      for (int u = 0; u < NVT; ++u) {
        const float4 x = *reinterpret_cast<const float4*>(X + (r0 + j) * (CB + 4) + 64 * u + cg);
        S[j][u][0] = x.x;
        S[j][u][1] = x.y;
        S[j][u][2] = x.z;
        S[j][u][3] = x.w;
      }
  }
  __syncthreads();
  for (int s = 0; s < NS; ++s) {
    __syncthreads();
    const float* B = reinterpret_cast<const float*>(qsm + (s & 1) * Lay::stage);
    float* O = reinterpret_cast<float*>(qsm + 2 * Lay::stage + (s & 1) * Lay::sums) + w * RTB * CB;
    const int nt = min(RTB, t1 - t0 - s * RTB);
    // a token's operands, read while the one before it is computed
    struct Step {
      float4 b[NVT], a[R / 4], o[R / 4], e[R / 4];
    };
    auto load = [&](int t, Step& x) __attribute__((always_inline)) {
      t = min(t, RTB - 1);   // past the stage: not used
#pragma unroll
      for (int u = 0; u < NVT; ++u)
        x.b[u] = *reinterpret_cast<const float4*>(B + 3 * RTB * KP + t * CB + 64 * u + cg);
#pragma unroll
      for (int j = 0; j < R / 4; ++j) {
        const float4* row = reinterpret_cast<const float4*>(B + t * KP + r0) + j;
        x.a[j] = row[0];
        x.o[j] = row[RTB * KP / 4];
        x.e[j] = row[2 * RTB * KP / 4];
      }
    };
    auto step = [&](int t, const Step& x) __attribute__((always_inline)) {
      float sum[NVT][4];
#pragma unroll
      for (int u = 0; u < NVT; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[u][i] = 0.f;
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const float a = comp(x.a[j / 4], j % 4), o = comp(x.o[j / 4], j % 4);
        const float e = comp(x.e[j / 4], j % 4);
#pragma unroll
        for (int u = 0; u < NVT; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float& st = S[j][u][i];
            st *= e;
            st = fmaf(a, comp(x.b[u], i), st);
            sum[u][i] = fmaf(o, st, sum[u][i]);
          }
      }
      // over the wave's four row groups: lane l ends with column 4 (l & 15) + (l >> 4)
#pragma unroll
      for (int u = 0; u < NVT; ++u) {
        const auto p0 = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum[u][0]),
                                                         __float_as_uint(sum[u][2]), false, false);
        const auto p1 = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum[u][1]),
                                                         __float_as_uint(sum[u][3]), false, false);
        const float u0 = __uint_as_float(p0[0]) + __uint_as_float(p0[1]);
        const float u1 = __uint_as_float(p1[0]) + __uint_as_float(p1[1]);
        const auto p2 = __builtin_amdgcn_permlane16_swap(__float_as_uint(u0), __float_as_uint(u1),
                                                         false, false);
        O[t * CB + 64 * u + cg + (lane >> 4)] = __uint_as_float(p2[0]) + __uint_as_float(p2[1]);
      }
    };
    Step x0, x1;
    load(0, x0);
#pragma unroll 1
    for (int t = 0; t < nt; t += 2) {
      load(t + 1, x1);
      __builtin_amdgcn_sched_barrier(0);   // the reads issue before the token's products
      step(t, x0);
      if (t + 1 >= nt) break;
      load(t + 2, x0);
      __builtin_amdgcn_sched_barrier(0);
      step(t + 1, x1);
    }
  }
  __syncthreads();
  if (again) {
    __syncthreads();   // the sums are read
    float* X = reinterpret_cast<float*>(qsm);
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
      for (int u = 0; u < NVT; ++u)
        *reinterpret_cast<float4*>(X + (r0 + j) * (CB + 4) + 64 * u + cg) =
            make_float4(S[j][u][0], S[j][u][1], S[j][u][2], S[j][u][3]);
    __syncthreads();   // the state is in LDS
    return;
  }
  if (sN) {
    const bool whole = V % 4 == 0 && ((uintptr_t)sN & 15) == 0;
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
      for (int u = 0; u < NVT; ++u) {
        const int c = ct * CB + 64 * u + cg;
        if (whole && r0 + j < K && c < V)
          *reinterpret_cast<float4*>(sN + (uint32_t)(r0 + j) * (uint32_t)V + (uint32_t)c) =
              make_float4(S[j][u][0], S[j][u][1], S[j][u][2], S[j][u][3]);
      }
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
      for (int u = 0; u < NVT; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int c = ct * CB + 64 * u + cg + i;
          if (!whole && r0 + j < K && c < V)
            sN[(uint32_t)(r0 + j) * (uint32_t)V + (uint32_t)c] = S[j][u][i];
        }
  }
}

// KP: K rounded up to 64, 128 or 256; NVT: 16-column tiles per consumer wave; VEC: K % 4 == 0
// and q, k, g rows aligned to 8 bytes.
template <int KP, int NVT, bool VEC>
__global__ __launch_bounds__((QCW + KP / 64) * 64, KP < 256 && NVT == 1 ? 3 : 2)
    void rec_chunk_kernel(RecScanArgs p) {
  using Lay = QLayout<KP, NVT>;
  constexpr int PW = Lay::PW, KT = KP / 16, CB = Lay::CB;
  constexpr int NOM = KT == 16 ? 4 : 2;   // sums of o's main products, by tile
  extern __shared__ __attribute__((aligned(16))) unsigned char qsm[];
  const int H = p.H, K = p.R, V = p.C;
  const int NCT = (V + CB - 1) / CB;
  const int L = xcd_remap(blockIdx.x, gridDim.x);
  const int ct = L % NCT, sh = L / NCT;
  const int seq = sh / H, hh = sh % H;
  int bos, eos;
  seq_bounds(p.si, seq, bos, eos);
  const int T = eos - bos, NC = (T + QC - 1) / QC;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long rsK = (long)H * K, rsV = (long)H * V;
  const bf16* __restrict__ q = (const bf16*)p.o + (long)hh * K;
  const bf16* __restrict__ k = (const bf16*)p.a + (long)hh * K;
  // without gates k's rows are loaded in their place and masked out
  const uint32_t gmask = p.ga ? ~0u : 0u;
  const bf16* __restrict__ gk = (const bf16*)(p.ga ? p.ga : p.a) + (long)hh * K;
  const bf16* __restrict__ v = (const bf16*)p.b + (long)hh * V;

  // Row i of a chunk of len rows, as an element offset from the chunk's first token in memory
  // order (rows past the sequence: its last row), from the row's offset i * stride.
  auto row_off = [&](uint32_t o, uint32_t lastrow) __attribute__((always_inline)) {
    const uint32_t x = min(o, lastrow);
    return p.dir ? lastrow - x : x;
  };
  auto chunk_t0 = [&](int n, int len) {   // uniform: the chunk's first token in memory order
    return (long)(p.dir ? eos - n * QC - len : bos + n * QC);
  };

  // Whether the block leaves for the element-wise phase at chunk n: a producer could not factor its
  // columns of it, or a consumer asked for it before the chunk. The same for every wave: chunk n's
  // flags stand between its barrier and the next.
  auto leaves = [&](int n) __attribute__((always_inline)) {
    const int* f = reinterpret_cast<const int*>(qsm + (n & 1) * Lay::buf + Lay::flag);
    int x = f[4] | f[5] | f[6] | f[7];
#pragma unroll
    for (int j = 0; j < PW; ++j) x |= f[j];
    return __builtin_amdgcn_readfirstlane(x) != 0;
  };
  // The matrix path from chunk `start` to the end or to chunk `left`, from there the element-wise
  // phase for `span` chunks, and again.
  int start = 0, span = kSpan, left = NC;

  if (w >= QCW) {
    // ---- producers: lane = 4 key columns (lane & 15) x 4 rows (lane >> 4) ----
    // a single producer wave is what the block waits for (B3 T1000 H16 K=V=64 156 -> 149 us; four
    // of them take the consumers' slots: B8 T2048 H4 K256 V512 462 -> 522)
    if constexpr (PW == 1 && NVT == 1) __builtin_amdgcn_s_setprio(1);
    const int pw = w - QCW, rg = lane >> 4, c0 = pw * 64 + 4 * (lane & 15);
    const uint32_t cv = (uint32_t)max(min(c0, K - 4), 0);
    uint32_t cm[2];   // masks of the columns past the head
#pragma unroll
    for (int e = 0; e < 2; ++e)
      cm[e] = (c0 + 2 * e < K ? 0xffffu : 0u) | (c0 + 2 * e + 1 < K ? 0xffff0000u : 0u);
    // this lane's rows, outwards from the middle: groups 0, 1 go down from rows 3 and 7
    auto row_of = [&](int u) { return rg < 2 ? 4 * rg + 3 - u : 4 * rg + u; };
    uint32_t ro[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) ro[u] = (uint32_t)row_of(u) * (uint32_t)rsK;
    uint2 Rq[4], Rk[4], Rg[4];
    auto ld4 = [&](const bf16* base, uint32_t off) __attribute__((always_inline)) {
      if constexpr (VEC) {
        return *reinterpret_cast<const uint2*>(base + (off + cv));
      } else {
        uint32_t x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = base[off + (uint32_t)min(c0 + e, K - 1)].u;
        return make_uint2(x[0] | (x[1] << 16), x[2] | (x[3] << 16));
      }
    };
    auto issue = [&](int n) __attribute__((always_inline)) {
      n = min(n, NC - 1);
      const int len = min(QC, T - n * QC);
      const long at = chunk_t0(n, len) * rsK;
      const uint32_t lr = (uint32_t)(len - 1) * (uint32_t)rsK;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t off = row_off(ro[u], lr);
        Rq[u] = ld4(q + at, off);
        Rk[u] = ld4(k + at, off);
        Rg[u] = ld4(gk + at, off);
      }
    };
    for (;;) {
      // per column: the previous chunk's rows 8..15 in sum and as a factor (groups 2, 3)
      float lsum[4], lpost[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lsum[e] = 0.f;
        lpost[e] = 1.f;
      }
      if (NC > 0) issue(start);
      for (int n = start; n < NC; ++n) {
        {
          unsigned char* B = qsm + (n & 1) * Lay::buf;
          const int len = T - n * QC;
          float xq[4][4], xk[4][4], xg[4][4];   // [row][column]
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const uint32_t m = row_of(u) < len ? ~0u : 0u, m0 = m & cm[0], m1 = m & cm[1];
            const uint32_t wq[2] = {Rq[u].x & m0, Rq[u].y & m1};
            const uint32_t wk[2] = {Rk[u].x & m0, Rk[u].y & m1};
            const uint32_t wg[2] = {Rg[u].x & m0 & gmask, Rg[u].y & m1 & gmask};
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              xq[u][2 * e] = bf16_lo(wq[e]);
              xq[u][2 * e + 1] = bf16_hi(wq[e]);
              xk[u][2 * e] = bf16_lo(wk[e]);
              xk[u][2 * e + 1] = bf16_hi(wk[e]);
              xg[u][2 * e] = bf16_lo(wg[e]);
              xg[u][2 * e + 1] = bf16_hi(wg[e]);
            }
          }
          issue(n + 1);
          float dout[4];
          // sum of the operands' squares and four decays x 2^97: above kOperandMax^2 where an
          // operand is too large or the decays sum to more than 8
          float sq = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float tot = (xg[0][e] + xg[1][e]) + (xg[2][e] + xg[3][e]);
            // permlane16_swap of x with itself: [0] holds the even group of the lane's pair of
            // groups, [1] the odd one
            const auto pr = __builtin_amdgcn_permlane16_swap(__float_as_uint(tot),
                                                             __float_as_uint(tot), false, false);
            const float even = __uint_as_float(pr[0]), odd = __uint_as_float(pr[1]);
            const float half = even + odd;   // groups 0, 1: rows 0..7; groups 2, 3: rows 8..15
            // the sum from the middle to this group's inner edge: groups 1 and 2 start there
            float run = rg == 0 ? odd : rg == 3 ? even : 0.f;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              const float nx = run + xg[u][e];
              const float sum = rg < 2 ? -run : nx;   // E: rows before the middle exclude their own
              run = nx;
              float f, fi;
              exp_pair(sum, f, fi);
              xq[u][e] *= f;
              xk[u][e] *= fi;
              sq = fmaf(xq[u][e], xq[u][e], sq);
              sq = fmaf(xk[u][e], xk[u][e], sq);
            }
            // decays: groups 0, 1 make pre and (with the previous chunk's rows 8..15, held by
            // groups 2, 3) dec; groups 2, 3 post
            const auto ps = __builtin_amdgcn_permlane32_swap(__float_as_uint(lsum[e]),
                                                             __float_as_uint(lsum[e]), false,
                                                             false);
            const float prev = __uint_as_float(ps[1]);   // the upper half's value
            const float d = exp_one(rg == 0 ? half + prev : half);
            sq = fmaf(d, kDecayWeight, sq);
            dout[e] = rg == 3 ? lpost[e] : d;
            lpost[e] = d;
            lsum[e] = half;
          }
          const bool good = __ballot(sq <= kOperandMax * kOperandMax) == ~0ull;
          if (lane == 0) reinterpret_cast<int*>(B + Lay::flag)[pw] = good ? 0 : 1;
          *reinterpret_cast<float4*>(B + Lay::dec + (rg * KP + c0) * 4) =
              make_float4(dout[0], dout[1], dout[2], dout[3]);
          bf16* sQ = reinterpret_cast<bf16*>(B + Lay::qa);
          bf16* sK = reinterpret_cast<bf16*>(B + Lay::ka);
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const Split x = split3(xq[u]), y = split3(xk[u]);
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              *reinterpret_cast<s4_t*>(sQ + (i * QC + row_of(u)) * Lay::QP + c0) = x.p[i];
              *reinterpret_cast<s4_t*>(sK + (i * QC + row_of(u)) * Lay::KQ + c0) = y.p[i];
            }
          }
          // A over this wave's 64 columns: its own LDS rows, in order behind the writes
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
          f32x4 am[2], ar[3];
          am[0] = am[1] = ar[0] = ar[1] = ar[2] = zero4();
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int kb = pw * 64 + t * 16 + 4 * (lane >> 4), li = lane & 15;
            s4_t x[3], y[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              x[i] = *reinterpret_cast<const s4_t*>(sQ + (i * QC + li) * Lay::QP + kb);
              y[i] = *reinterpret_cast<const s4_t*>(sK + (i * QC + li) * Lay::KQ + kb);
            }
            mma_split(x, y, am[t & 1], ar);
          }
          am[0] = (am[0] + am[1]) + (ar[0] + ar[1] + ar[2]);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            reinterpret_cast<float*>(B + Lay::A)[(pw * QC + 4 * (lane >> 4) + r) * QTP +
                                                 (lane & 15)] = am[0][r];
        }
        __syncthreads();
        if (__builtin_expect(leaves(n), 0)) {
          left = n;
          break;
        }
      }
      if (left == NC) break;
      const int end = min(left + span, NC);
      rec_elements_producer<KP, NVT, VEC>(p, qsm, left * QC, min(T, end * QC), end < NC, bos, eos,
                                          hh, ct, pw, lane);
      if (end == NC) return;
      start = end;
      span *= 4;
      left = NC;
    }
    __syncthreads();
    return;
  }

  // ---- consumers: all K rows of NVT 16-column tiles ----
  int g4 = lane >> 4, li = lane & 15;
  int cb = ct * CB + w * NVT * 16 + li;   // this lane's column of tile 0
  // a lane's state element (kt, r): uniform base plus a 32-bit offset
  const long sbase = ((long)seq * H + hh) * K * V;
  const float* __restrict__ s0 = p.s0 ? p.s0 + sbase : nullptr;
  float* __restrict__ sN = p.sN ? p.sN + sbase : nullptr;
  f32x4 S[NVT][KT];
#pragma unroll
  for (int i = 0; i < NVT; ++i)
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        S[i][kt][r] = 0.f;
  if (s0) {   // one run of loads, masked when all are under way
#pragma unroll
    for (int i = 0; i < NVT; ++i)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          S[i][kt][r] = s0[(uint32_t)min(kt * 16 + 4 * g4 + r, K - 1) * (uint32_t)V +
                           (uint32_t)min(cb + i * 16, V - 1)];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NVT; ++i)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          S[i][kt][r] = kt * 16 + 4 * g4 + r < K && cb + i * 16 < V ? S[i][kt][r] : 0.f;
  }
  // An infinite state (or one large enough to leave the range within a few chunks) is left to the
  // recurrence as written: split into bf16 it would turn to NaN. A NaN stays one, and in its row
  // and column, so it stays here (NaN in v, B8 T2048 H4 K256 V512: 946 -> 510 us). Looked at
  // before the first chunk and after every eighth. Between, decays of at most 8 a half and 16
  // products of 2^50 2^20 a chunk keep a value below 2^48 (2^56 + 8 * 2^74).
  auto state_ok = [&]() __attribute__((always_inline)) {
    bool s_ok = true;
#pragma unroll
    for (int i = 0; i < NVT; ++i)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) s_ok = s_ok && !(fabsf(S[i][kt][r]) > kStateMax);
    return s_ok;
  };
  __builtin_amdgcn_sched_barrier(0);
  // the next chunk's v, as loaded: extended at the load, every load is waited for (two tiles a
  // wave, B64 T64 H16 K=V=128: 90 against 123 us). With two producers and one tile that wait, in
  // the middle of the chunk, leaves issue slots to the producers, which the block waits for (B8
  // T2048 H16 K=V=128 372 -> 357 us).
  std::conditional_t<PW == 2 && NVT == 1, uint32_t, uint16_t> Rv[NVT][4];
  uint32_t vo[4];
  auto issue_v = [&](int n) __attribute__((always_inline)) {
    n = min(n, NC - 1);
    const int len = min(QC, T - n * QC);
    const bf16* vb = v + chunk_t0(n, len) * rsV;
    const uint32_t lr = (uint32_t)(len - 1) * (uint32_t)rsV;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const uint32_t off = row_off(vo[m], lr);
#pragma unroll
      for (int i = 0; i < NVT; ++i) Rv[i][m] = vb[off + (uint32_t)min(cb + i * 16, V - 1)].u;
    }
  };
  auto mul_rows = [&](const unsigned char* f) __attribute__((always_inline)) {   // S rows x f[k]
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      const float4 x = *reinterpret_cast<const float4*>(f + (kt * 16 + 4 * g4) * 4);
#pragma unroll
      for (int i = 0; i < NVT; ++i) {
        S[i][kt][0] *= x.x;
        S[i][kt][1] *= x.y;
        S[i][kt][2] *= x.z;
        S[i][kt][3] *= x.w;
      }
    }
  };
  // whether S still has the last chunk's post factor to come (it meets the next chunk's pre
  // in one factor)
  bool owed = false;
  s4_t vv[NVT];   // rows 4 g4 .. 4 g4 + 3 of the lane's column
  // chunk n's v as operands, once loaded; ok: whether every value is small enough
  auto take_v = [&](int n) __attribute__((always_inline)) {
    const int len = T - n * QC;
    bool ok = true;
#pragma unroll
    for (int i = 0; i < NVT; ++i) {
      uint32_t x[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        x[m] = 4 * g4 + m < len && cb + i * 16 < V ? (uint32_t)Rv[i][m] : 0u;
        ok = ok && (x[m] & 0x7fffu) <= kValueMaxBits;
      }
      const uint2 w = make_uint2(x[0] | (x[1] << 16), x[2] | (x[3] << 16));
      vv[i] = __builtin_bit_cast(s4_t, w);
    }
    return ok;
  };
  // this wave's request for chunk n: its v or the state are not fit for the matrix cores
  auto request = [&](int n, bool ok) __attribute__((always_inline)) {
    const int x = __ballot(ok) == ~0ull ? 0 : 1;
    if (lane == 0) reinterpret_cast<int*>(qsm + (n & 1) * Lay::buf + Lay::flag)[4 + w] = x;
  };
  for (;;) {
    // what follows from these is formed anew after the element-wise phase, not kept over it
    asm volatile("" : "+v"(g4), "+v"(li), "+v"(cb));
#pragma unroll
    for (int m = 0; m < 4; ++m) vo[m] = (uint32_t)(4 * g4 + m) * (uint32_t)rsV;
    if (NC > 0) {
      issue_v(start);
      const bool s_ok = state_ok();
      request(start, take_v(start) && s_ok);
    }
    __syncthreads();
#pragma unroll 1
    for (int n = start; n < NC; ++n) {
      const unsigned char* B = qsm + (n & 1) * Lay::buf;
      const int len = min(QC, T - n * QC);
      issue_v(n + 1);
      if (__builtin_expect(leaves(n), 0)) {
        left = n;
        break;
      }
      f32x4 o[NVT];
      const float* dec = reinterpret_cast<const float*>(B + (owed ? Lay::dec : Lay::pre)) + 4 * g4;
      const bf16* pq = reinterpret_cast<const bf16*>(B + Lay::qa) + li * Lay::QP + 4 * g4;
      // transposed reads of 4 rows x 16 columns: this lane's address is row li >> 2 of its
      // group's four, columns 4 (li & 3); it receives column li
      const bf16* pk = reinterpret_cast<const bf16*>(B + Lay::ka) +
                       (4 * g4 + (li >> 2)) * Lay::KQ + 4 * (li & 3);
      float4 d[2];
      s4_t x[2][3], y[2][3];
      auto operands = [&](int kt) __attribute__((always_inline)) {
        d[kt & 1] = *reinterpret_cast<const float4*>(dec + kt * 16);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          x[kt & 1][i] = *reinterpret_cast<const s4_t*>(pq + i * QC * Lay::QP + kt * 16);
          y[kt & 1][i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) s4_t*)(pk + i * QC * Lay::KQ + kt * 16));
        }
      };
      operands(0);
      // Step kt: tile kt's qa S' (the main products in NOM sums, the others in three)
      // and ka^T v onto the state, with the next tile decayed to the chunk's middle and split
      // meanwhile and the one after it read from LDS. The order of the products keeps those of
      // one sum apart, and the VALU work sits between them (an MFMA occupies its own pipe for
      // 16 cycles, a VALU operation 4).
      f32x4 om[NVT][NOM], orest[NVT][3];
      float4 ap[PW];
      Split sp[NVT][2];
      auto decay = [&](int kt) __attribute__((always_inline)) {   // S' of tile kt, split
        const float4 dd = d[kt & 1];
#pragma unroll
        for (int i = 0; i < NVT; ++i) {
          S[i][kt][0] *= dd.x;
          S[i][kt][1] *= dd.y;
          S[i][kt][2] *= dd.z;
          S[i][kt][3] *= dd.w;
          const float t[4] = {S[i][kt][0], S[i][kt][1], S[i][kt][2], S[i][kt][3]};
          sp[i][kt & 1] = split3(t);
        }
      };
      decay(0);
      operands(1);
#pragma unroll
      for (int i = 0; i < NVT; ++i) {
#pragma unroll
        for (int j = 0; j < NOM; ++j) om[i][j] = zero4();
#pragma unroll
        for (int j = 0; j < 3; ++j) orest[i][j] = zero4();
      }
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        const int c = kt & 1;
        s4_t xx[3], yy[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          xx[j] = x[c][j];
          yy[j] = y[c][j];
        }
#pragma unroll
        for (int i = 0; i < NVT; ++i) {
          const s4_t(&b)[3] = sp[i][c].p;
          f32x4(&r)[3] = orest[i];
          f32x4& t = S[i][kt];
          om[i][kt % NOM] = mma16(xx[0], b[0], om[i][kt % NOM]);
          t = mma16(yy[2], vv[i], t);
          r[0] = mma16(xx[2], b[0], r[0]);
          r[1] = mma16(xx[0], b[2], r[1]);
          t = mma16(yy[1], vv[i], t);
          r[2] = mma16(xx[1], b[1], r[2]);
          r[0] = mma16(xx[1], b[0], r[0]);
          t = mma16(yy[0], vv[i], t);
          r[1] = mma16(xx[0], b[1], r[1]);
        }
        if (kt + 1 < KT) decay(kt + 1);
        if (kt + 2 < KT) {
          operands(kt + 2);
        } else if (kt + 2 == KT) {
#pragma unroll
          for (int j = 0; j < PW; ++j)
            ap[j] = *reinterpret_cast<const float4*>(
                B + Lay::A + ((j * QC + li) * QTP + 4 * g4) * 4);
        }
#pragma unroll
        for (int j = 0; j < 9 * NVT; ++j) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);   // one MFMA, four VALU
          __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // A v: row li, tokens 4 g4 ..; those after the row left out
      const float4 am = PW == 1   ? ap[0]
                        : PW == 2 ? add4(ap[0], ap[PW / 2])
                                  : add4(add4(ap[0], ap[1 % PW]), add4(ap[PW / 2], ap[PW - 1]));
      const int after = li - 4 * g4;
      const float aa[4] = {after >= 0 ? am.x : 0.f, after >= 1 ? am.y : 0.f,
                           after >= 2 ? am.z : 0.f, after >= 3 ? am.w : 0.f};
      const Split as = split3(aa);
#pragma unroll
      for (int i = 0; i < NVT; ++i) {
        f32x4 u = zero4();
#pragma unroll
        for (int j = 2; j >= 0; --j) u = mma16(as.p[j], vv[i], u);
        u += orest[i][0] + orest[i][1] + orest[i][2];
#pragma unroll
        for (int st = NOM / 2; st > 0; st /= 2)
#pragma unroll
          for (int j = 0; j < st; ++j) om[i][j] += om[i][j + st];
        o[i] = om[i][0] + u;
      }
      owed = true;
      {   // before the output's stores, which a wait for v behind them would wait for too
        bool ok = take_v(n + 1);
        if ((n & 7) == 7) ok = ok && state_ok();
        request(n + 1, ok);
      }
      {
        float* ob = (float*)p.out + chunk_t0(n, len) * rsV + (long)hh * V;
#pragma unroll
        for (int i = 0; i < NVT; ++i) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int row = 4 * g4 + r;
            if (row < len && cb + i * 16 < V)
              ob[(uint32_t)(p.dir ? len - 1 - row : row) * (uint32_t)rsV +
                 (uint32_t)(cb + i * 16)] = p.so * o[i][r];
          }
        }
      }
      __syncthreads();
    }
    if (__builtin_expect(left == NC, 1)) break;
    if (owed) mul_rows(qsm + (left & 1) * Lay::buf + Lay::ppost);
    owed = false;
    __syncthreads();   // the factors are read
    float* X = reinterpret_cast<float*>(qsm);
    int gl = g4, cl = w * NVT * 16 + li;
    asm volatile("" : "+v"(gl), "+v"(cl));
#pragma unroll
    for (int i = 0; i < NVT; ++i)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          X[(kt * 16 + 4 * gl + r) * (CB + 4) + cl + i * 16] = S[i][kt][r];
    const int end = min(left + span, NC);
    rec_elements_consumer<KP, NVT>(p, qsm, left * QC, min(T, end * QC), end < NC, sN, ct, w, lane);
    if (end == NC) return;
    asm volatile("" : "+v"(gl), "+v"(cl));
#pragma unroll
    for (int i = 0; i < NVT; ++i)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          S[i][kt][r] = X[(kt * 16 + 4 * gl + r) * (CB + 4) + cl + i * 16];
    __syncthreads();   // the state is out of LDS
    start = end;
    span *= 4;
    left = NC;
  }
  if (owed) mul_rows(qsm + ((NC - 1) & 1) * Lay::buf + Lay::post);
  if (sN) {
    int gl = g4, cl = cb;
    asm volatile("" : "+v"(gl), "+v"(cl));
#pragma unroll
    for (int i = 0; i < NVT; ++i)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int kk = kt * 16 + 4 * gl + r, c = cl + i * 16;
          if (kk < K && c < V) sN[(uint32_t)kk * (uint32_t)V + (uint32_t)c] = S[i][kt][r];
        }
  }
}

namespace {

template <int KP, int NVT, bool VEC>
hipError_t launch_rec_chunk(const RecScanArgs& p, hipStream_t st) {
  using Lay = QLayout<KP, NVT>;
  static_assert(Lay::bytes <= 163840, "LDS budget exceeded");
  constexpr int CB = QCW * NVT * 16;
  const long blocks = (long)p.si.N * p.H * ((p.C + CB - 1) / CB);
  if (blocks == 0) return hipSuccess;
  const hipError_t e = hipFuncSetAttribute((const void*)rec_chunk_kernel<KP, NVT, VEC>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           Lay::bytes);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((rec_chunk_kernel<KP, NVT, VEC>), dim3((unsigned)blocks),
                     dim3((QCW + Lay::PW) * 64), Lay::bytes, st, p);
  return hipGetLastError();
}

template <int KP>
hipError_t launch_rec_chunk_k(const RecScanArgs& p, hipStream_t st) {
  const bool vec = p.R % 4 == 0 &&
                   (((uintptr_t)p.o | (uintptr_t)p.a | (uintptr_t)p.ga) & 7) == 0;
  if (!vec) return launch_rec_chunk<KP, 1, false>(p, st);
  // 32 columns a wave (the producers' work shared by 128 columns) when that fills the chip
  if constexpr (KP <= 128)
    if ((long)p.si.N * p.H * (p.C / 128) >= 256) return launch_rec_chunk<KP, 2, true>(p, st);
  return launch_rec_chunk<KP, 1, true>(p, st);
}

}  // namespace

bool rec_chunk_supported(const RecScanArgs& p, int dtype, int o_dtype) {
  return dtype == DT_BF16 && o_dtype == DT_F32 && p.gb == nullptr && p.dg == nullptr &&
         !p.s_trans && !p.shift && !p.final_gate && p.flags.p == nullptr && p.sa == 1.f &&
         p.R <= 256 &&
         // 32-bit offsets within a chunk and a state
         16L * p.H * (p.R > p.C ? p.R : p.C) < (1L << 30) && (long)p.R * p.C < (1L << 30);
}

hipError_t run_rec_chunk(const RecScanArgs& p, hipStream_t st) {
  if (p.R <= 64) return launch_rec_chunk_k<64>(p, st);
  if (p.R <= 128) return launch_rec_chunk_k<128>(p, st);
  return launch_rec_chunk_k<256>(p, st);
}

}  // namespace tops
