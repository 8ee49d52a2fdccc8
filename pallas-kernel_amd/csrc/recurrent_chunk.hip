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
// as fast: this kernel with them ran at 520 us instead of 461). The state never leaves the
// registers: a wave holds all K rows of 16 (or 32) columns as accumulators (rows 4g + r,
// column l & 15 in lane l = 16 g + column), which is also the B operand of an MFMA over those
// rows, so qa S' and ka^T v need no transposition and no exchange between waves. Measured: B8
// T2048 H4 K256 V512 951 -> 461 us, B64 T64 H16 K=V=128 131 -> 92 us, B3 T1000 H16 K=V=64
// 317 -> 155 us (the VALU scan and this kernel).
//
// Block = (sequence, head, 64 or 128 columns): four consumer waves, each 16 or 32 columns,
// and KP / 64 producer waves. While the consumers work on tokens 16 n .., the producers make
// qa, ka, the 16 x 16 products A (each over its own 64 key columns, summed by the reader) and
// the decays of the next 16 in the other LDS buffer: one barrier per 16 tokens.
//
// Range: where a factored operand is above 2^50 (gates below about -4 a token over half a
// chunk) or not finite, or a half's decay is above 8 or NaN (the first row's gate is in the decays
// alone, not in an operand), the 64 key columns of that producer are taken token by token from
// the inputs, as the recurrence is written (37 us instead of 3.6 us a chunk when all of them
// are), and all columns where v or the state is not finite or the state is large: non-finite
// values, also of a state that overflows on the way, then stay where the recurrence puts them.
#include <type_traits>
#include <utility>

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

template <int KP>
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
  static constexpr int bad = ppost + KP * 4;         // [4] ints
  static constexpr int buf = bad + 16;
  static constexpr int bytes = 2 * buf;
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

// f(0), f(1), .. with the indices as types: a loop that is unrolled before anything else is
// done to it, also around an inner run-time loop.
template <class F, int... I>
__device__ __forceinline__ void each_tile(F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
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

// KP: K rounded up to 64, 128 or 256; NVT: 16-column tiles per consumer wave; VEC: K % 4 == 0
// and q, k, g rows aligned to 8 bytes.
template <int KP, int NVT, bool VEC>
__global__ __launch_bounds__((QCW + KP / 64) * 64, KP < 256 && NVT == 1 ? 3 : 2)
    void rec_chunk_kernel(RecScanArgs p) {
  using Lay = QLayout<KP>;
  constexpr int PW = Lay::PW, KT = KP / 16, CB = QCW * NVT * 16;
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

  if (w >= QCW) {
    // ---- producers: lane = 4 key columns (lane & 15) x 4 rows (lane >> 4) ----
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
    // per column: the previous chunk's rows 8..15 in sum and as a factor (groups 2, 3)
    float lsum[4], lpost[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      lsum[e] = 0.f;
      lpost[e] = 1.f;
    }
    if (NC > 0) issue(0);
    for (int n = 0; n < NC; ++n) {
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
        float dout[4], prevpost[4];
        // sum of the operands' squares and four decays x 2^97: above kOperandMax^2 where an operand
        // is too large or the decays sum to more than 8
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
          const auto pp = __builtin_amdgcn_permlane32_swap(__float_as_uint(lpost[e]),
                                                           __float_as_uint(lpost[e]), false,
                                                           false);
          prevpost[e] = __uint_as_float(pp[1]);
          sq = fmaf(d, kDecayWeight, sq);
          dout[e] = rg == 3 ? lpost[e] : d;
          lpost[e] = d;
          lsum[e] = half;
        }
        const bool good = __ballot(sq <= kOperandMax * kOperandMax) == ~0ull;
        if (lane == 0) reinterpret_cast<int*>(B + Lay::bad)[pw] = !good;
        if (!good) {
          // these 64 columns are left to the recurrence as written: operands that add nothing
          // and leave the state as it enters the chunk
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            dout[e] = rg == 0 ? prevpost[e] : rg == 3 ? dout[e] : 1.f;
            lpost[e] = 1.f;
            lsum[e] = 0.f;
#pragma unroll
            for (int u = 0; u < 4; ++u) xq[u][e] = xk[u][e] = 0.f;
          }
        }
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
    }
    __syncthreads();
    return;
  }

  // ---- consumers: all K rows of NVT 16-column tiles ----
  const int g4 = lane >> 4, li = lane & 15;
  const int cb = ct * CB + w * NVT * 16 + li;   // this lane's column of tile 0
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
      for (int r = 0; r < 4; ++r) {
        const int kk = kt * 16 + 4 * g4 + r, c = cb + i * 16;
        const float x = s0 ? s0[(uint32_t)min(kk, K - 1) * (uint32_t)V + (uint32_t)min(c, V - 1)]
                           : 0.f;
        S[i][kt][r] = kk < K && c < V ? x : 0.f;
      }
  // A state that is not finite (or large enough to leave the range within a few chunks) stays with
  // the recurrence as written: split into bf16 it would turn to NaN. Looked at before the first
  // chunk and after every eighth and after columns taken as written. Between, decays of at most 8
  // a half and 16 products of 2^50 2^20 a chunk keep a value below 2^48 (2^56 + 8 * 2^74).
  auto state_ok = [&]() __attribute__((always_inline)) {
    bool s_ok = true;
#pragma unroll
    for (int i = 0; i < NVT; ++i)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) s_ok = s_ok && fabsf(S[i][kt][r]) <= kStateMax;
    return __ballot(s_ok) == ~0ull;
  };
  bool check = true;
  __builtin_amdgcn_sched_barrier(0);
  uint32_t Rv[NVT][4], vo[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) vo[m] = (uint32_t)(4 * g4 + m) * (uint32_t)rsV;
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
  if (NC > 0) issue_v(0);
  __syncthreads();
#pragma unroll 1
  for (int n = 0; n < NC; ++n) {
    const unsigned char* B = qsm + (n & 1) * Lay::buf;
    const int len = min(QC, T - n * QC);
    s4_t vv[NVT];   // rows 4 g4 .. 4 g4 + 3 of the lane's column
    bool ok = true;
#pragma unroll
    for (int i = 0; i < NVT; ++i) {
      uint32_t x[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        x[m] = 4 * g4 + m < len && cb + i * 16 < V ? Rv[i][m] : 0u;
        ok = ok && (x[m] & 0x7fffu) <= kValueMaxBits;
      }
      const uint2 w = make_uint2(x[0] | (x[1] << 16), x[2] | (x[3] << 16));
      vv[i] = __builtin_bit_cast(s4_t, w);
    }
    issue_v(n + 1);
    // key column groups (a producer's 64) to be taken token by token: those flagged, or all
    // where this wave's columns of v or its state are not finite
    int seq_groups = 0;
#pragma unroll
    for (int j = 0; j < PW; ++j)
      seq_groups |= (reinterpret_cast<const int*>(B + Lay::bad)[j] != 0) << j;
    seq_groups = __builtin_amdgcn_readfirstlane(seq_groups);
    bool all_seq = __ballot(ok) != ~0ull;
    if (__builtin_expect(check, 0)) all_seq = all_seq || !state_ok();
    f32x4 o[NVT];
    if (__builtin_expect(!all_seq, 1)) {
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
    } else {
      if (owed) mul_rows(B + Lay::ppost);
      owed = false;
      seq_groups = (1 << PW) - 1;
#pragma unroll
      for (int i = 0; i < NVT; ++i) o[i] = zero4();
    }
    check = seq_groups != 0 || (n & 7) == 7;
    if (__builtin_expect(seq_groups != 0, 0)) {
      // the recurrence as written for the tiles of these groups, four tokens at a time (their
      // inputs from global memory, the next tile's under the work on this one); a row's part of
      // o is summed over the tiles and lanes and joins the lanes that hold the tokens' rows
#pragma unroll 1
      for (int b4 = 0; b4 < 4 && 4 * b4 < len; ++b4) {
        // the lane's indices through an empty asm: formed anew here, not held in registers
        // (for every tile) around the loops of the other path
        int gl = g4, cl = cb;
        asm volatile("" : "+v"(gl), "+v"(cl));
        // rows past the sequence: its last row's address, gate 0, k and q 0
        const long at = chunk_t0(n, len);
        uint32_t to[4];
        float xv[NVT][4], os[NVT][4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int row = min(4 * b4 + j, len - 1);
          to[j] = (uint32_t)(p.dir ? len - 1 - row : row);
#pragma unroll
          for (int i = 0; i < NVT; ++i) {
            xv[i][j] = to_f32(v[(at + to[j]) * rsV + min(cl + i * 16, V - 1)]);
            os[i][j] = 0.f;
          }
          to[j] *= (uint32_t)rsK;
        }
        uint2 w[2][3][4];
        auto load = [&](int kt) __attribute__((always_inline)) {
          const int k0 = kt * 16 + 4 * gl;   // this lane's four rows
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            const bf16* base = (a == 0 ? q : a == 1 ? k : gk) + at * rsK;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              if constexpr (VEC) {
                w[kt & 1][a][j] = *reinterpret_cast<const uint2*>(
                    base + (to[j] + (uint32_t)max(min(k0, K - 4), 0)));
              } else {
                uint32_t x[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = base[to[j] + (uint32_t)min(k0 + e, K - 1)].u;
                w[kt & 1][a][j] = make_uint2(x[0] | (x[1] << 16), x[2] | (x[3] << 16));
              }
            }
          }
        };
        load(0);
        auto tile = [&](auto tile_index) __attribute__((always_inline)) {
          constexpr int kt = decltype(tile_index)::value;
          if constexpr (kt + 1 < KT) load(kt + 1);
          const int k0 = kt * 16 + 4 * gl;
          if (seq_groups >> (kt / 4) & 1) {   // uniform
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const uint32_t m = 4 * b4 + j < len ? ~0u : 0u;
              const uint2 wq = w[kt & 1][0][j], wk = w[kt & 1][1][j], wg = w[kt & 1][2][j];
              const uint32_t qw[2] = {wq.x & m, wq.y & m}, kw[2] = {wk.x & m, wk.y & m};
              const uint32_t gw[2] = {wg.x & m & gmask, wg.y & m & gmask};
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const bool in = k0 + r < K;
                const float qx = r & 1 ? bf16_hi(qw[r >> 1]) : bf16_lo(qw[r >> 1]);
                const float kx = r & 1 ? bf16_hi(kw[r >> 1]) : bf16_lo(kw[r >> 1]);
                const float eg = gexp<bf16>(r & 1 ? bf16_hi(gw[r >> 1]) : bf16_lo(gw[r >> 1]));
#pragma unroll
                for (int i = 0; i < NVT; ++i) {
                  const float x = m ? xv[i][j] : 0.f;
                  S[i][kt][r] = fmaf(in ? kx : 0.f, x, S[i][kt][r] * (in ? eg : 1.f));
                  os[i][j] = fmaf(in ? qx : 0.f, S[i][kt][r], os[i][j]);
                }
              }
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        };
        each_tile(tile, std::make_integer_sequence<int, KT>{});
#pragma unroll
        for (int i = 0; i < NVT; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            os[i][j] += __shfl_xor(os[i][j], 16);
            os[i][j] += __shfl_xor(os[i][j], 32);
            if (g4 == b4) o[i][j] += os[i][j];
          }
      }
    }
    {
      float* ob = (float*)p.out + chunk_t0(n, len) * rsV + (long)hh * V;
#pragma unroll
      for (int i = 0; i < NVT; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 4 * g4 + r;
          if (row < len && cb + i * 16 < V)
            ob[(uint32_t)(p.dir ? len - 1 - row : row) * (uint32_t)rsV + (uint32_t)(cb + i * 16)] =
                p.so * o[i][r];
        }
      }
    }
    __syncthreads();
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
  using Lay = QLayout<KP>;
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
