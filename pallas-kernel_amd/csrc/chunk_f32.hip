// Per-chunk products of float32 inputs at chunk 64 over whole rows of the value dimension: the
// forward's output and the backward's dv (reference: tops/ops/gla/chunk.py:441-496, 504-560).
// With g~ the chunk-local cumsum, gamma its last row and r = (g~_first + gamma) / 2:
//   qg = q e^{g~-r},  kg = k e^{r-g~},  A = scale qg kg^T
//   o  = tril(A) v    + qg (scale e^{r} h)
//   dv = tril(A)^T do + kg (e^{gamma-r} dh)
// which are one computation: out = M x + L (f (.) S), L [64][K] in LDS.
//
// What bounds it: the float32 MFMAs (16x16x4, 256 FLOP a cycle and CU). One 256-thread block
// takes a (chunk, head) and up to 256 value columns, so that A and the gating are formed once
// for them; a wave takes 64 of the columns and 16 to 64 of the rows. x (v, do) and the state
// rows (h, dh) go from global memory to the MFMA operand registers and never through LDS: a
// lane's 16 bytes are four columns of one row, i.e. the operand of four 16-column tiles (tile j
// holds the columns 4 n + j), so no operand is transposed and a row of outputs is stored in 16
// bytes a lane. Each LDS fragment (four contraction steps of 16 rows) feeds 16 products, each
// global load four to sixteen. Tiles of A above the diagonal are neither formed nor read. LDS 53
// KB at K = 128 (the tile of the other operand is reused for A): three blocks a CU.
// B4 T2048 H4 K128 V256: o 199 -> 47 us, dv 124 -> 47 us. Replaced
// here: one block of 104 KB LDS a CU with transposing stores of v and h (o), one block
// per 64 columns with A formed in each (dv); both stay for the other chunk sizes, bf16, rows
// that are not 16-byte aligned, and given A or cumulative gates.
#include <initializer_list>

#include "common.hpp"
#include "kernels.hpp"

namespace tops {

namespace {

constexpr int FC = 64;          // rows of a chunk
constexpr int FP = FC + 4;      // LDS pitch of 64-wide rows

int f32_lds_bytes(int K) {
  const int KP = (K + 63) / 64 * 64;
  return (FC * (KP + 4) + FC * FP + KP + 2 * 5 * 64) * 4;
}

// Lower tiles of A in the order they are dealt to the waves.
__device__ __forceinline__ void lower_tile(int t, int& mi, int& ni) {
  mi = t < 1 ? 0 : t < 3 ? 1 : t < 6 ? 2 : 3;
  ni = t - mi * (mi + 1) / 2;
}

// Chunk-local cumsum of one column (lane) whose 16 rows of this wave are in g: in place without
// the earlier waves' rows, which are `off`. st: [5][64]. One barrier.
__device__ __forceinline__ void segment_cumsum(float (&g)[16], float* st, int w, int lane,
                                               float& first, float& off, float& gamma) {
  if (w == 0) st[4 * 64 + lane] = g[0];
#pragma unroll
  for (int i = 1; i < 16; ++i) g[i] += g[i - 1];
  st[w * 64 + lane] = g[15];
  __syncthreads();
  off = gamma = 0.f;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const float x = st[s * 64 + lane];
    off += s < w ? x : 0.f;
    gamma += x;
  }
  first = st[4 * 64 + lane];
}

}  // namespace

struct F32RowArgs {
  const float *q, *k, *g;
  const float* x;      // v or do [tokens, H, V]
  const float* s;      // h or dh [NC, H, K, V] (nullable)
  float* out;          // o or dv [tokens, H, V]
  int* flags;          // gate-range flags [NC, H] (gate_range.hip; nullable)
  float scale;
  int H, K, V;
  SeqInfo si;
};

// DV: dv instead of o. NV: 64-column groups of a block (waves: NV column x 4 / NV row groups).
template <bool DV, int NV>
__global__ __launch_bounds__(256, 3) void chunk_f32_kernel(F32RowArgs p) {
  constexpr int RT = NV;   // 16-row tiles of a wave
  extern __shared__ __attribute__((aligned(16))) float fsm[];
  const int H = p.H, K = p.K, V = p.V;
  const int KT = (K + 63) >> 6, KP = KT * 64, PL = KP + 4;
  float* sL = fsm;                  // [64][PL]: qg (o) or kg (dv)
  float* sT = sL + FC * PL;         // [64][FP]: the other operand's K tile, then M
  float* sR = sT + FC * FP;         // [KP]: the state rows' factors
  float* sTot = sR + KP;            // [2][5][64]: segment sums of g, first row

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, gr = lane >> 4;
  const int NB = (V + 64 * NV - 1) / (64 * NV);
  const int L = xcd_remap(blockIdx.x, gridDim.x);
  const int c = L / NB / H, hh = L / NB % H;
  int seq, t0, len;
  chunk_range(p.si, c, seq, t0, len);
  (void)seq;
  const long rsK = (long)H * K, rsV = (long)H * V;
  const long baseK = ((long)t0 * H + hh) * K, baseV = ((long)t0 * H + hh) * V;

  const float *qb = p.q + baseK, *kb = p.k + baseK, *gb = p.g + baseK;
  const float* xbase = p.x + baseV;

  // ---- L, M = tril(A) or its transpose ----
  f32x4 accA[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) accA[j] = zero4();
  int wide = 0;   // a column's |g~ - r| beyond the factors' range, as gate_range_kernel has it
  for (int kt = 0; kt < KT; ++kt) {
    const int col = kt * 64 + lane;   // thread: one column, rows 16 w .. 16 w + 15
    const uint32_t cc = (uint32_t)min(col, K - 1);
    float gv[16], qv[16], kv[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {   // no branches: all loads are in flight together
      const uint32_t at = (uint32_t)min(16 * w + i, len - 1) * (uint32_t)rsK + cc;
      gv[i] = gb[at];
      qv[i] = qb[at];
      kv[i] = kb[at];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (16 * w + i >= len || col >= K) gv[i] = qv[i] = kv[i] = 0.f;
    float first, off, gamma;   // two buffers of sums: one barrier between write and read
    segment_cumsum(gv, sTot + (kt & 1) * 5 * 64, w, lane, first, off, gamma);
    const float r = 0.5f * (first + gamma);
    float mx = -3.0e38f, mn = 3.0e38f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {   // rows past the chunk repeat its last one
      mx = fmaxf(mx, gv[i] + off);
      mn = fminf(mn, gv[i] + off);
    }
    wide |= fmaxf(mx - r, r - mn) * 1.4426950408889634f > kGateLimit2 ? 1 : 0;
    if (w == 0) sR[col] = DV ? gexp<float>(gamma - r) : p.scale * gexp<float>(r);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 16 * w + i;
      const float d = gv[i] + off - r;
      const float qg = qv[i] * gexp<float>(d), kg = kv[i] * gexp<float>(-d);
      sL[row * PL + col] = DV ? kg : qg;
      sT[row * FP + lane] = DV ? qg : kg;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int t = w + 4 * j;
      if (t >= 10) break;   // uniform
      int mi, ni;
      lower_tile(t, mi, ni);
      const float* a = DV ? sT + mi * 16 * FP : sL + mi * 16 * PL + kt * 64;
      const float* b = DV ? sL + ni * 16 * PL + kt * 64 : sT + ni * 16 * FP;
      mma_tile<float>(accA[j], a, DV ? FP : PL, b, DV ? PL : FP, 64, lane);
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int t = w + 4 * j;
    if (t >= 10) break;
    int mi, ni;
    lower_tile(t, mi, ni);
    const int jj = ni * 16 + li, ii = mi * 16 + 4 * gr;   // rows ii + r
    float a[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = jj <= ii + r ? accA[j][r] * p.scale : 0.f;
    if (DV) {
      *reinterpret_cast<float4*>(sT + jj * FP + ii) = make_float4(a[0], a[1], a[2], a[3]);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) sT[(ii + r) * FP + jj] = a[r];
    }
  }
  wide = __syncthreads_or(wide);
  if (tid == 0 && p.flags && L % NB == 0) p.flags[L / NB] = wide ? 1 : 0;

  // ---- out = M x + L (f (.) S): this wave's 64 columns and 16 RT rows ----
  const int vb = (L % NB * NV + w % NV) * 64, rt0 = w / NV * RT;
  if (vb >= V) return;   // uniform; no barrier follows
  const int vcol = min(vb + 4 * li, V - 4);
  const bool vok = vb + 4 * li < V;
  f32x4 acc[RT][4];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[t][j] = zero4();

  // 16 contraction steps: step e of the lane's group is row 4 gr + e of the 16
  auto products = [&](const float* M, int pitch, const float4 (&b)[4], int lo, int hi) {
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      if (rt0 + t < lo || rt0 + t > hi) continue;   // uniform
      const float4 m = *reinterpret_cast<const float4*>(M + ((rt0 + t) * 16 + li) * pitch + 4 * gr);
      const float me[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(me[e], b[e].x, acc[t][0], 0, 0, 0);
        acc[t][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(me[e], b[e].y, acc[t][1], 0, 0, 0);
        acc[t][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(me[e], b[e].z, acc[t][2], 0, 0, 0);
        acc[t][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(me[e], b[e].w, acc[t][3], 0, 0, 0);
      }
    }
  };
  auto load_x = [&](int s, float4 (&b)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 16 * s + 4 * gr + e;
      const float4 x =
          *reinterpret_cast<const float4*>(xbase + (uint32_t)min(row, len - 1) * (uint32_t)rsV + vcol);
      b[e] = row < len ? x : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  const float* srow = p.s + ((long)c * H + hh) * K * V;
  auto load_s = [&](int s, float4 (&b)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      b[e] = *reinterpret_cast<const float4*>(
          srow + (uint32_t)min(16 * s + 4 * gr + e, K - 1) * (uint32_t)V + vcol);
  };
  float4 xa[4], xb[4];
  load_x(0, xa);
#pragma unroll
  for (int s = 0; s < 4; ++s) {   // the next 16 rows are loaded under these products
    float4(&cur)[4] = s & 1 ? xb : xa;
    float4(&nxt)[4] = s & 1 ? xa : xb;
    if (s < 3) load_x(s + 1, nxt);
    products(sT + 16 * s, FP, cur, DV ? 0 : s, DV ? s : 3);
  }
  if (p.s) {
    const int NS = (K + 15) / 16;
    auto scaled = [&](int s, const float4 (&b)[4]) {
      const float4 f = *reinterpret_cast<const float4*>(sR + 16 * s + 4 * gr);
      const float fe[4] = {f.x, f.y, f.z, f.w};
      float4 y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool in = 16 * s + 4 * gr + e < K;
        y[e] = in ? make_float4(b[e].x * fe[e], b[e].y * fe[e], b[e].z * fe[e], b[e].w * fe[e])
                  : make_float4(0.f, 0.f, 0.f, 0.f);
      }
      products(sL + 16 * s, PL, y, 0, 3);
    };
    load_s(0, xa);
    for (int s = 0; s < NS; s += 2) {
      if (s + 1 < NS) load_s(s + 1, xb);
      scaled(s, xa);
      if (s + 1 >= NS) break;
      if (s + 2 < NS) load_s(s + 2, xa);
      scaled(s + 1, xb);
    }
  }
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = (rt0 + t) * 16 + 4 * gr + r;
      if (row < len && vok)
        *reinterpret_cast<float4*>(p.out + baseV + (uint32_t)row * (uint32_t)rsV + vcol) =
            make_float4(acc[t][0][r], acc[t][1][r], acc[t][2][r], acc[t][3][r]);
    }
}

template <bool DV, int NV>
static hipError_t launch_f32(const F32RowArgs& p, hipStream_t st) {
  const long blocks = (long)p.si.NC * p.H * ((p.V + 64 * NV - 1) / (64 * NV));
  if (blocks == 0) return hipSuccess;
  const int lds = f32_lds_bytes(p.K);
  const hipError_t e = hipFuncSetAttribute((const void*)chunk_f32_kernel<DV, NV>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((chunk_f32_kernel<DV, NV>), dim3((unsigned)blocks), dim3(256), lds, st, p);
  return hipGetLastError();
}

// Columns of a block: as many as V has, up to 256, unless that leaves fewer blocks than CUs.
template <bool DV>
static hipError_t pick_f32(const F32RowArgs& p, hipStream_t st) {
  const long nch = (long)p.si.NC * p.H;
  if (p.V > 128 && nch * ((p.V + 255) / 256) >= 256) return launch_f32<DV, 4>(p, st);
  if (p.V > 64 && nch * ((p.V + 127) / 128) >= 256) return launch_f32<DV, 2>(p, st);
  return launch_f32<DV, 1>(p, st);
}

// K up to 384: the LDS of a block (118 KB there) stays below that of the kernels replaced.
// 32-bit offsets within a chunk's rows and a state.
static bool f32_sizes(int C, int H, int K, int V, std::initializer_list<const void*> ptrs) {
  if (C != FC || K <= 0 || K > 384 || V % 4 != 0) return false;
  if (64L * H * (K > V ? K : V) >= (1L << 30) || (long)K * V >= (1L << 30)) return false;
  for (const void* x : ptrs)
    if ((uintptr_t)x & 15u) return false;
  return true;
}

// ---------------------------------------------------------------------------
// Per-chunk states: forward h (a = k, b = v) and reverse dh (a = q, b = do), reference
// tops/ops/common/chunk_h.py:18-119, 399-591, in two passes. The first forms every chunk's
// update U_n = a~^T b (a~ = k e^{gamma - g~}, or scale q e^{g~}) at the state's place and its
// decay e^{gamma_n}, all chunks at once; the second walks the chunks, S <- e^{gamma_n} S + U_n,
// one thread per four values, and leaves in U_n's place the state entering (reverse: leaving)
// the chunk.
//
// What bounds it: memory, the states written, read and written again. The scan that this replaces
// (state_scan_kernel, which writes them once) walks the chunks with the gating and the products in
// the chain: 3.1 us a chunk whatever the number of sequences. B4 T2048 H4 K128 V256, a direction:
// 100 us -> 36 (updates) + 22 (states); forward + backward 438 -> 354 us. It was faster at every
// size tried, from B1 T200 (one block of 64 x 32 a state tile) to 512 (sequence, head) pairs of four
// chunks and 64 pairs of 32 (B4 T2048 H16 K=V=128), so it runs wherever the workspace holds the
// decays.
// ---------------------------------------------------------------------------

// a~ in LDS (row-major, 17 KB), b from global memory to the operand registers as above; a block
// takes 64 key columns and up to 256 value columns of one chunk and head.
template <bool REV, int NV>
__global__ __launch_bounds__(256, 3) void f32_update_kernel(ScanArgs p) {
  constexpr int RT = NV;   // 16-row tiles (of keys) of a wave
  __shared__ __attribute__((aligned(16))) float sA[FC * FP];
  __shared__ float sTot[5 * 64];
  const int H = p.H, K = p.K, V = p.V;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, gr = lane >> 4;
  const int KT = (K + 63) >> 6, NB = (V + 64 * NV - 1) / (64 * NV);
  const int L = xcd_remap(blockIdx.x, gridDim.x);
  const int kt = L / NB % KT, ch = L / NB / KT;
  const int c = ch / H, hh = ch % H;
  int seq, t0, len;
  chunk_range(p.si, c, seq, t0, len);
  (void)seq;
  const uint32_t rsK = (uint32_t)H * K, rsV = (uint32_t)H * V;
  const long baseK = ((long)t0 * H + hh) * K, baseV = ((long)t0 * H + hh) * V;
  const float *ab = (const float*)p.a + baseK, *gb = (const float*)p.g + baseK;
  const float* bb = (const float*)p.b + baseV;

  const int vb = (L % NB * NV + w % NV) * 64, rt0 = w / NV * RT;
  const int vcol = min(vb + 4 * li, V - 4);
  auto load_b = [&](int s, float4 (&b)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 16 * s + 4 * gr + e;
      const float4 x = *reinterpret_cast<const float4*>(bb + (uint32_t)min(row, len - 1) * rsV + vcol);
      b[e] = row < len ? x : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  const int col = kt * 64 + lane;
  const uint32_t cc = (uint32_t)min(col, K - 1);
  float gv[16], av[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const uint32_t at = (uint32_t)min(16 * w + i, len - 1) * rsK + cc;
    gv[i] = gb[at];
    av[i] = ab[at];
  }
  float4 xa[4], xb[4];
  load_b(0, xa);
#pragma unroll
  for (int i = 0; i < 16; ++i)
    if (16 * w + i >= len || col >= K) gv[i] = av[i] = 0.f;
  float first, off, gamma;
  segment_cumsum(gv, sTot, w, lane, first, off, gamma);
  if (w == 0 && L % NB == 0 && col < K) p.dec[(long)ch * K + col] = gexp<float>(gamma);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float x = gv[i] + off;
    sA[(16 * w + i) * FP + lane] =
        av[i] * (REV ? p.scale * gexp<float>(x) : gexp<float>(gamma - x));
  }
  __syncthreads();
  if (vb >= V) return;   // uniform; no barrier follows

  f32x4 acc[RT][4];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[t][j] = zero4();
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    float4(&cur)[4] = s & 1 ? xb : xa;
    float4(&nxt)[4] = s & 1 ? xa : xb;
    if (s < 3) load_b(s + 1, nxt);
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = sA[(16 * s + 4 * gr + e) * FP + (rt0 + t) * 16 + li];
        acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, cur[e].x, acc[t][0], 0, 0, 0);
        acc[t][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, cur[e].y, acc[t][1], 0, 0, 0);
        acc[t][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, cur[e].z, acc[t][2], 0, 0, 0);
        acc[t][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, cur[e].w, acc[t][3], 0, 0, 0);
      }
  }
  float* u = (float*)p.s_all + (long)ch * K * V;
  const bool vok = vb + 4 * li < V;
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = kt * 64 + (rt0 + t) * 16 + 4 * gr + r;
      if (k < K && vok)
        *reinterpret_cast<float4*>(u + (uint32_t)k * (uint32_t)V + vcol) =
            make_float4(acc[t][0][r], acc[t][1][r], acc[t][2][r], acc[t][3][r]);
    }
}

// One thread per four values of a (sequence, head)'s state; two batches of SD chunks' updates
// in registers, so that loads are in flight while a batch is added up.
constexpr int SD = 8;
template <bool REV>
__global__ __launch_bounds__(256) void f32_state_kernel(ScanArgs p) {
  const int H = p.H, K = p.K, V4 = p.V / 4;
  const int NB = (K * V4 + 255) / 256;
  const int bh = blockIdx.x / NB, e = blockIdx.x % NB * 256 + (int)threadIdx.x;
  const int seq = bh / H, hh = bh % H;
  if (e >= K * V4) return;
  int bos, eos, c0, nc;
  seq_range(p.si, seq, bos, eos, c0, nc);
  (void)bos;
  (void)eos;
  const long step = (long)H * K * V4;   // float4s from a chunk to the next
  float4* s = (float4*)p.s_all + ((long)c0 * H + hh) * K * V4 + e;
  const float* dec = p.dec + ((long)c0 * H + hh) * K + e / V4;
  const long at = ((long)seq * H + hh) * K * V4 + e;
  float4 S = p.s_init ? ((const float4*)p.s_init)[at] : make_float4(0.f, 0.f, 0.f, 0.f);
  auto chunk = [&](int n) { return REV ? nc - 1 - n : n; };
  struct Batch {
    float4 u[SD];
    float d[SD];
  };
  auto load = [&](int n0, Batch& b) {
#pragma unroll
    for (int i = 0; i < SD; ++i) {
      const int n = chunk(min(n0 + i, nc - 1));   // past the end: the last chunk again, unused
      b.u[i] = s[n * step];
      b.d[i] = dec[(long)n * H * K];
    }
  };
  auto walk = [&](int n0, const Batch& b) {
#pragma unroll
    for (int i = 0; i < SD; ++i) {
      if (n0 + i >= nc) break;   // uniform
      s[chunk(n0 + i) * step] = S;
      S.x = fmaf(b.d[i], S.x, b.u[i].x);
      S.y = fmaf(b.d[i], S.y, b.u[i].y);
      S.z = fmaf(b.d[i], S.z, b.u[i].z);
      S.w = fmaf(b.d[i], S.w, b.u[i].w);
    }
  };
  if (nc > 0) {
    Batch A, B;
    load(0, A);
    for (int n = 0; n < nc; n += 2 * SD) {
      load(n + SD, B);
      walk(n, A);
      if (n + SD >= nc) break;
      load(n + 2 * SD, A);
      walk(n + SD, B);
    }
  }
  if (p.s_final) ((float4*)p.s_final)[at] = S;
}

template <bool REV, int NV>
static hipError_t launch_update(const ScanArgs& p, hipStream_t st) {
  const long blocks =
      (long)p.si.NC * p.H * ((p.K + 63) / 64) * ((p.V + 64 * NV - 1) / (64 * NV));
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL((f32_update_kernel<REV, NV>), dim3((unsigned)blocks), dim3(256), 0, st, p);
  return hipGetLastError();
}

template <bool REV>
static hipError_t run_f32_scan_dir(const ScanArgs& p, hipStream_t st) {
  const hipError_t e = p.V > 128 ? launch_update<REV, 4>(p, st)
                       : p.V > 64 ? launch_update<REV, 2>(p, st)
                                  : launch_update<REV, 1>(p, st);
  if (e != hipSuccess) return e;
  const long blocks = (long)p.si.N * p.H * ((p.K * (p.V / 4) + 255) / 256);
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL((f32_state_kernel<REV>), dim3((unsigned)blocks), dim3(256), 0, st, p);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// dq, dk and dg (reference: tops/ops/gla/chunk.py:504-743), with dA = scale tril(do v^T):
//   Xq = dA kg + (scale e^{r}) do h^T,   Xm = e^{gamma-r} v dh^T,   Xk = dA^T qg + Xm
//   dq = e^{g~-r} Xq,  dk = e^{r-g~} Xk,
//   dg = revcumsum(qg Xq - kg Xk) + e^{gamma} sum_v h dh + sum_j kg Xm
//
// What bounds it: the float32 MFMAs, 10 us of them a block of 64 key columns at V = 256. The
// operands' value columns go through LDS 32 at a time (37 KB for do, v, h and dh), which with
// qg and kg makes 72 KB and two blocks a CU, so that one block's loads and barriers lie under the
// other's products; chunk_bwd_dqkg_kernel, which stages 64 columns and q, k and g raw, has 139 KB
// and one (B4 T2048 H4 K128 V256: 127 -> 93 us; its 300 MB take about 55 at the rate of a large
// copy). A wave's 16 key columns of every row stay in its accumulators to the end: dg's sums
// over the rows are sums within a lane and across its four lane groups, without an exchange.
// ---------------------------------------------------------------------------

constexpr int DVW = 32, DVP = DVW + 4;   // value columns staged, their pitch
struct DqkgF32 {
  static constexpr int tile = FC * FP, vt = FC * DVP;   // floats
  static constexpr int qg = 0, kg = tile, stage = 2 * tile;   // stage: do, v, h, dh
  static constexpr int dA = stage, d = stage + tile;          // after the value columns
  static constexpr int fac = stage + 4 * vt;                  // sR, sEg, sGm, sHd [64], sums
  static constexpr int bytes = (fac + 4 * 64 + 5 * 64) * 4;
  static_assert(d + tile <= fac, "dA and d lie in the staged tiles' place");
};

__global__ __launch_bounds__(256, 2) void f32_dqkg_kernel(BwdArgs p) {
  extern __shared__ __attribute__((aligned(16))) float fsm[];
  float *sQg = fsm + DqkgF32::qg, *sKg = fsm + DqkgF32::kg, *sS = fsm + DqkgF32::stage;
  float *sdA = fsm + DqkgF32::dA, *sD = fsm + DqkgF32::d;
  float *sR = fsm + DqkgF32::fac, *sEg = sR + 64, *sGm = sR + 128, *sHd = sR + 192,
        *sTot = sR + 256;
  const int H = p.H, K = p.K, V = p.V;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, gr = lane >> 4;
  const int KT = (K + 63) >> 6, VT = (V + DVW - 1) / DVW;
  const int L = xcd_remap(blockIdx.x, gridDim.x);
  const int kb = L % KT * 64, ch = L / KT;
  const int c = ch / H, hh = ch % H;
  int seq, t0, len;
  chunk_range(p.si, c, seq, t0, len);
  (void)seq;
  const uint32_t rsK = (uint32_t)H * K, rsV = (uint32_t)H * V;
  const long baseK = ((long)t0 * H + hh) * K + kb, baseV = ((long)t0 * H + hh) * V;
  const long baseS = ((long)ch * K + kb) * V;
  const int klen = min(64, K - kb);
  const float* src[4] = {(const float*)p.dout + baseV, (const float*)p.v + baseV,
                         (const float*)p.h + baseS, (const float*)p.dh + baseS};

  // 16-byte pieces of the staged tiles: rows tid / 8 and + 32, columns 4 (tid % 8)
  const int pr = tid >> 3, pc = 4 * (tid & 7);
  float4 st[4][2];
  auto load = [&](int vt) {
    const int col = min(vt * DVW + pc, V - 4);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = min(pr + 32 * i, (t < 2 ? len : klen) - 1);
        st[t][i] = *reinterpret_cast<const float4*>(src[t] + (uint32_t)row * (t < 2 ? rsV : (uint32_t)V) + col);
      }
  };
  auto stage = [&](int vt) {
    const bool in = vt * DVW + pc < V;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = pr + 32 * i;
        const bool ok = in && row < (t < 2 ? len : klen);
        *reinterpret_cast<float4*>(sS + t * DqkgF32::vt + row * DVP + pc) =
            ok ? st[t][i] : make_float4(0.f, 0.f, 0.f, 0.f);
      }
  };

  // ---- qg, kg; d = g~ - r of this thread's column and 16 rows ----
  float d[16];
  {
    const bool cok = lane < klen;
    const uint32_t cc = (uint32_t)min(lane, klen - 1);
    const float *qb = (const float*)p.q + baseK, *kbp = (const float*)p.k + baseK,
                *gb = (const float*)p.g + baseK;
    float qv[16], kv[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t at = (uint32_t)min(16 * w + i, len - 1) * rsK + cc;
      d[i] = gb[at];
      qv[i] = qb[at];
      kv[i] = kbp[at];
    }
    load(0);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (16 * w + i >= len || !cok) d[i] = qv[i] = kv[i] = 0.f;
    float first, off, gamma;
    segment_cumsum(d, sTot, w, lane, first, off, gamma);
    const float r = 0.5f * (first + gamma);
    if (w == 0) {
      sR[lane] = p.scale * gexp<float>(r);
      sEg[lane] = gexp<float>(gamma - r);
      sGm[lane] = gexp<float>(gamma);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      d[i] += off - r;
      sQg[(16 * w + i) * FP + lane] = qv[i] * gexp<float>(d[i]);
      sKg[(16 * w + i) * FP + lane] = kv[i] * gexp<float>(-d[i]);
    }
  }

  // ---- dA = do v^T (lower tiles), do h^T and v dh^T (this wave's 16 key columns) ----
  f32x4 dA[3], Xq[4], Xm[4];
#pragma unroll
  for (int j = 0; j < 3; ++j) dA[j] = zero4();
#pragma unroll
  for (int j = 0; j < 4; ++j) Xq[j] = Xm[j] = zero4();
  float hd = 0.f;   // sum_v h dh of key column tid / 4 over this thread's eight columns a tile
  const float *sDo = sS, *sV = sS + DqkgF32::vt, *sH = sS + 2 * DqkgF32::vt,
              *sDh = sS + 3 * DqkgF32::vt;
  for (int vt = 0; vt < VT; ++vt) {
    if (vt > 0) __syncthreads();   // the previous columns' readers are done
    stage(vt);
    __syncthreads();
    if (vt + 1 < VT) load(vt + 1);
    const Frag<float> fh = ld_frag(sH + (16 * w + li) * DVP + 8 * gr);
    const Frag<float> fd = ld_frag(sDh + (16 * w + li) * DVP + 8 * gr);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      mma(Xq[j], ld_frag(sDo + (16 * j + li) * DVP + 8 * gr), fh);
      mma(Xm[j], ld_frag(sV + (16 * j + li) * DVP + 8 * gr), fd);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int t = w + 4 * j;
      if (t >= 10) break;   // uniform
      int mi, ni;
      lower_tile(t, mi, ni);
      mma_tile<float>(dA[j], sDo + mi * 16 * DVP, DVP, sV + ni * 16 * DVP, DVP, DVW, lane);
    }
    const float* a = sH + (tid >> 2) * DVP + 8 * (tid & 3);
    const float* b = sDh + (tid >> 2) * DVP + 8 * (tid & 3);
#pragma unroll
    for (int i = 0; i < 8; i += 4) {
      const float4 x = *reinterpret_cast<const float4*>(a + i);
      const float4 y = *reinterpret_cast<const float4*>(b + i);
      hd += x.x * y.x + x.y * y.y + (x.z * y.z + x.w * y.w);
    }
  }
  hd += __shfl_xor(hd, 1);
  hd += __shfl_xor(hd, 2);
  if ((tid & 3) == 0) sHd[tid >> 2] = hd;
  __syncthreads();   // the staged tiles are dead
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int t = w + 4 * j;
    if (t >= 10) break;
    int mi, ni;
    lower_tile(t, mi, ni);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int ii = mi * 16 + 4 * gr + r, jj = ni * 16 + li;
      sdA[ii * FP + jj] = jj <= ii ? dA[j][r] * p.scale : 0.f;
    }
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) sD[(16 * w + i) * FP + lane] = d[i];
  __syncthreads();

  // ---- dA kg and dA^T qg: lane l's step e of 16 rows is row 4 (l >> 4) + e ----
  const int kc = 16 * w + li;
  const float fr = sR[kc], fe = sEg[kc];
  f32x4 Xk[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    Xq[j] *= fr;
    Xm[j] *= fe;
    Xk[j] = Xm[j];
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    float bk[4], bq[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      bk[e] = sKg[(16 * s + 4 * gr + e) * FP + kc];
      bq[e] = sQg[(16 * s + 4 * gr + e) * FP + kc];
    }
#pragma unroll
    for (int j = s; j < 4; ++j) {   // rows 16 j.. of dq: columns of dA up to them
      const float4 m = *reinterpret_cast<const float4*>(sdA + (16 * j + li) * FP + 16 * s + 4 * gr);
      const float me[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
      for (int e = 0; e < 4; ++e)
        Xq[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(me[e], bk[e], Xq[j], 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j <= s; ++j)   // rows 16 j.. of dk: rows of dA from them on
#pragma unroll
      for (int e = 0; e < 4; ++e)
        Xk[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
            sdA[(16 * s + 4 * gr + e) * FP + 16 * j + li], bq[e], Xk[j], 0, 0, 0);
  }

  // ---- dq, dk, dg: this lane's column, rows 16 j + 4 gr + r ----
  float *dq = (float*)p.dq + baseK, *dk = (float*)p.dk + baseK, *dg = (float*)p.dg + baseK;
  const bool cok = kc < klen;
  float suf[4][4], dki = 0.f;
#pragma unroll
  for (int j = 3; j >= 0; --j)
#pragma unroll
    for (int r = 3; r >= 0; --r) {
      const int row = 16 * j + 4 * gr + r;
      const float dd = sD[row * FP + kc], qg = sQg[row * FP + kc], kg = sKg[row * FP + kc];
      suf[j][r] = qg * Xq[j][r] - kg * Xk[j][r] + (r < 3 ? suf[j][r < 3 ? r + 1 : 3] : 0.f);
      dki += kg * Xm[j][r];
      if (row < len && cok) {
        dq[(uint32_t)row * rsK + kc] = gexp<float>(dd) * Xq[j][r];
        dk[(uint32_t)row * rsK + kc] = gexp<float>(-dd) * Xk[j][r];
      }
    }
  dki += __shfl_xor(dki, 16);
  dki += __shfl_xor(dki, 32);
  float tail = sGm[kc] * sHd[kc] + dki, after = 0.f;   // after: the later 16-row tiles
#pragma unroll
  for (int j = 3; j >= 0; --j) {
    const float x1 = __shfl_xor(suf[j][0], 16), both = suf[j][0] + x1;
    const float x2 = __shfl_xor(both, 32);
    const float off = ((gr & 1) == 0 ? x1 : 0.f) + ((gr & 2) == 0 ? x2 : 0.f) + after;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * j + 4 * gr + r;
      if (row < len && cok) dg[(uint32_t)row * rsK + kc] = suf[j][r] + off + tail;
    }
    after += both + x2;
  }
}

bool f32_dqkg_supported(const BwdArgs& p) {
  return p.dg != nullptr && f32_sizes(p.si.C, p.H, p.K, p.V, {p.v, p.dout, p.h, p.dh});
}
hipError_t run_f32_dqkg(const BwdArgs& p, hipStream_t st) {
  const long blocks = (long)p.si.NC * p.H * ((p.K + 63) / 64);
  if (blocks == 0) return hipSuccess;
  const hipError_t e =
      hipFuncSetAttribute((const void*)f32_dqkg_kernel,
                          hipFuncAttributeMaxDynamicSharedMemorySize, DqkgF32::bytes);
  if (e != hipSuccess) return e;
  ktimer_mark(KT_BWD_DQKG, false, st);
  hipLaunchKernelGGL(f32_dqkg_kernel, dim3((unsigned)blocks), dim3(256), DqkgF32::bytes, st, p);
  ktimer_mark(KT_BWD_DQKG, true, st);
  return hipGetLastError();
}

bool f32_scan_supported(const ScanArgs& p) {
  return p.dec != nullptr && p.s_all != nullptr && !p.g_is_cumsum &&
         f32_sizes(p.si.C, p.H, p.K, p.V, {p.b, p.s_all, p.s_init, p.s_final});
}
hipError_t run_f32_scan(const ScanArgs& p, bool reverse, hipStream_t st) {
  return reverse ? run_f32_scan_dir<true>(p, st) : run_f32_scan_dir<false>(p, st);
}

bool f32_fwd_o_supported(const FwdOArgs& p) {
  return p.o != nullptr && p.A_in == nullptr && p.A_out == nullptr && !p.g_is_cumsum &&
         f32_sizes(p.si.C, p.H, p.K, p.V, {p.v, p.h, p.o});
}
hipError_t run_f32_fwd_o(const FwdOArgs& p, hipStream_t st) {
  F32RowArgs a = {(const float*)p.q, (const float*)p.k, (const float*)p.g, (const float*)p.v,
                  (const float*)p.h, (float*)p.o,       p.flags,           p.scale,
                  p.H,               p.K,               p.V,               p.si};
  return pick_f32<false>(a, st);
}

bool f32_dv_supported(const BwdArgs& p) {
  return f32_sizes(p.si.C, p.H, p.K, p.V, {p.dout, p.dh, p.dv});
}
hipError_t run_f32_dv(const BwdArgs& p, hipStream_t st) {
  F32RowArgs a = {(const float*)p.q,  (const float*)p.k, (const float*)p.g, (const float*)p.dout,
                  (const float*)p.dh, (float*)p.dv,      p.flags,           p.scale,
                  p.H,                p.K,               p.V,               p.si};
  return pick_f32<true>(a, st);
}

}  // namespace tops
