// The reference's Winograd / Toom-Cook 1-D conv op family (wino_tf[_snake|_leaky]_lc_f32_gpu,
// wino_mm[_res][_stats]_lc_f32_gpu, wino_adain_affine_lc_f32_gpu: python/lokinfer/ops/winograd.py:120-218,
// kernels/gpu/winograd.cpp:73-160 in lariaus/lokinfer), with the reference's operand layouts so that a graph built
// on those ops runs unchanged:
//   V  [d, A, rmax, C]: V[rho, xi, r, c] = sum_j BT[xi, j] h[rho + d (r M + j - pad / d), c], h = act(x), zero
//                       outside the residue class's rows
//   U  [A, N Ci, Co]   = G w per tap group (host wino_weights), tr = [BT (A x A) | AT (M x A)]
//   out[o, co] = (b + sum_xi AT[j, xi] sum_{g, ci} V[rho, xi, t + g, ci] U[xi, g Ci + ci, co] [+ res]) * scale,
//                o = rho + d (t M + j)
//   stats [d chunks, Co, 2]: (mean, M2) of each 128 output rows of a residue class
// The same kernels run this backend's Kokoro graph wherever their grid fills the chip (the generator's resblock
// and noise convs, the decoder's wide convs, conv_post).
//
// wino_mm: one workgroup per (64 output channels, 64 tiles, residue); 4 waves in 2 x 2, each 32 tiles x 32 channels.
// Steps = points x 16-channel chunks; the point's GEMM accumulates over the groups with the A rows shifted by g, and
// after a point's last chunk AT[j, xi] folds it into the M output accumulators. Small grids split the steps over
// workgroups (split-K) and sum the partial rows in winoSplitReduceKernel (statistics then from the channel-stats
// kernel).
#include "common.h"
#include "lokinfer_hip.h"
#include "split3.h"

#include <algorithm>
#include <cstdint>

namespace lkh {
int residueStats(const float* x, float* st, int64_t l, int64_t c, int d, int64_t chunks, hipStream_t s);  // kokoro.hip
}  // namespace lkh

namespace lkd {

typedef float v4w __attribute__((ext_vector_type(4)));

constexpr int kWinoRows = 128;  // output rows per statistics chunk

// V[rho, xi, r, c4 .. c4 + 3] for R consecutive tile rows r per thread, i.e. per (rho, r / R, c4), channel quad fastest:
// the R tiles share their overlapping input rows, so a thread loads and activates M R + A - M rows once (R = 2: 1.4x
// the input instead of A / M = 1.75x at M = 4, A = 7) and writes R A rows of V. act: 0 none, 1 snake(affine), 2
// leaky(affine); rows outside the residue class are zero (the conv pads after the activation).
template <int M, int A, int R>
__global__ __launch_bounds__(256) void winoTfKernel(const float* __restrict__ x, const float* __restrict__ tr,
                                                   const float* __restrict__ af, const float* __restrict__ alpha,
                                                   float* __restrict__ v, int64_t l, int64_t c, int d, int padq,
                                                   int64_t rmax, int act, float slope) {
  constexpr int XR = M * R + A - M;  // input rows behind R tiles
  const int64_t c4n = c / 4;
  const int64_t groups = (rmax + R - 1) / R;
  const int64_t total = static_cast<int64_t>(d) * groups * c4n;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t c4 = i % c4n, rg = (i / c4n) % groups;
    const int rho = static_cast<int>(i / (c4n * groups));
    const int64_t lr = rho < l ? (l - rho + d - 1) / d : 0;
    const int64_t r0 = rg * R;
    const int64_t q0 = r0 * M - padq;
    v4w mean = {0.f, 0.f, 0.f, 0.f}, scale = {1.f, 1.f, 1.f, 1.f}, beta = {0.f, 0.f, 0.f, 0.f};
    v4w al = {1.f, 1.f, 1.f, 1.f}, inv = {1.f, 1.f, 1.f, 1.f};
    if (act != 0) {
      mean = *reinterpret_cast<const v4w*>(af + 4 * c4);
      scale = *reinterpret_cast<const v4w*>(af + c + 4 * c4);
      beta = *reinterpret_cast<const v4w*>(af + 2 * c + 4 * c4);
    }
    if (act == 1) {
      al = *reinterpret_cast<const v4w*>(alpha + 4 * c4);
#pragma unroll
      for (int e = 0; e < 4; ++e) inv[e] = 1.0f / al[e];
    }
    v4w raw[XR];
#pragma unroll
    for (int j = 0; j < XR; ++j) {
      const int64_t q = q0 + j;
      const int64_t qc = min<int64_t>(max<int64_t>(q, 0), max<int64_t>(lr - 1, 0));
      raw[j] = *reinterpret_cast<const v4w*>(x + min<int64_t>(rho + qc * d, l - 1) * c + 4 * c4);
    }
#pragma unroll
    for (int j = 0; j < XR; ++j) {
      const int64_t q = q0 + j;
      v4w h = raw[j];
      if (act == 1) {
        h = (h - mean) * scale + beta;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = h[e] + inv[e] * snakeSinSq(al[e] * h[e]);
      } else if (act == 2) {
        h = (h - mean) * scale + beta;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = h[e] >= 0.0f ? h[e] : h[e] * slope;
      }
      const bool in = q >= 0 && q < lr;
#pragma unroll
      for (int e = 0; e < 4; ++e) raw[j][e] = in ? h[e] : 0.0f;
    }
#pragma unroll
    for (int t = 0; t < R; ++t) {
      const int64_t rr = r0 + t;
      if (rr >= rmax) break;
#pragma unroll
      for (int xi = 0; xi < A; ++xi) {
        v4w o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < A; ++j) o += tr[xi * A + j] * raw[M * t + j];
        *reinterpret_cast<v4w*>(v + ((static_cast<int64_t>(rho) * A + xi) * rmax + rr) * c + 4 * c4) = o;
      }
    }
  }
}

// A raw buffer resource over `bytes` bytes from p, both the same in every lane (read from the first, so that they are
// held in scalar registers).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t uniformRsrc(const void* p, unsigned bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  const uint64_t lo = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(a)));
  const uint64_t hi = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(a >> 32)));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(hi << 32 | lo), 0,
                                           __builtin_amdgcn_readfirstlane(static_cast<int>(bytes)), 0x00020000);
}

struct WinoMmArgs {
  const float* v;
  const float* u;
  const float* bias;
  const float* res;
  float* out;
  const float* tr;
  float* stats;
  float* part;  // split > 1: per-split raw output rows [split][Lo][Co], summed by winoSplitReduceKernel
  int64_t lo, ci, co, rmax, chunks;
  int d, split;
  float scale;
};

// MFMA-bound: the products run on the bf16 matrix cores as three-part splits (split3.h), 6 N S MFMAs of 32 cycles per
// wave and step of S 16-channel chunks, at three workgroups per CU (at most 168 registers): the y accumulators leave
// room for one 32 x 32 block per wave, and it takes three waves per SIMD to cover a step's loads, LDS stores and
// barrier (two blocks per wave at two waves per SIMD ran 5 - 35% slower).
//
// A: the step's V rows (64 tiles + N - 1 for the group shift) are split once while staging and held in LDS as three bf16
// planes, [row][2 halves of 8 channels], half swizzled by (row >> 3) & 1 so that 16 lanes of a 16-byte read cover all 64
// banks. B bypasses LDS: a wave's fragment (16 k x 32 columns) comes straight from U, one step ahead, in coalesced
// 16-byte loads.
//
// Measured (graph replay, one box; with statistics), the f32 MFMA form of this kernel over U tiled, which could not overlap
// its vector instructions with its MFMAs, against this one over U split: L = 293281, 128 -> 128 channels, K = 11 d = 5 427,
// 321 us (under the profiler 362), K = 7 d = 3 311, 251, K = 3 with residual 252, 163; L = 48880, 256 -> 256, K = 11 d = 3
// 281, 207; L = 5740, 256 -> 256, K = 7 d = 3 65, 47; L = 287, 1104 -> 1024, K = 3 40, 34. Of the first, with parts taken
// out: 269 without the V staging, 301 without the U loads, 148 its bf16 MFMAs alone (of 333 before V was scaled).
//
// UL, the layout of U:
//   0  U [A, N Ci, Co]: eight 4-byte loads per fragment, split before its MFMAs;
//   1  tiled (ops u_layout = 1), Ut [A, Co / 64, (Ci / 16) N 4 64 4]: per point and 64-column block, for each 16-channel
//      chunk and tap group the 16 x 64 slab stored k-quad-major, [k4][col][4] (U row g Ci + 16 c + 4 k4 + q, column
//      64 cb + col): two 16-byte loads;
//   2  split (ops u_layout = 2), Us [A, Co / 64, 2, Ci / 16, N, 3, 64, 8] bf16: per 32-column half, chunk and group the
//      three parts (h, m, l) in fragment order, lane 32 lk + lr holding k = 8 lk .. 8 lk + 7 of column lr: three 16-byte
//      loads and nothing to split.
template <int M, int A, int N, int S, int UL>
__global__ __launch_bounds__(256, 3) void winoMmKernel(WinoMmArgs p) {
  constexpr int TT = 64;            // tiles per workgroup
  constexpr int ROWS = TT + N - 1;  // staged V rows (group shift)
  constexpr int E = N * S;          // B fragments of a step: e = N (chunk) + (tap group)
  using Stage = u32x4[S][3][ROWS * 2];
  using RawB = f32x4[UL == 2 ? 3 : 2];
  __shared__ Stage As0, As1;  // two objects, so that the compiler sees that a step's stores and reads never meet
  __shared__ float red[2][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1, lr = lane & 31, lk = lane >> 5;
  // XCD-aware order: the channel blocks of a tile block read its V rows through one L2
  const GridItem wk = xcdOrder();
  const int d = p.d, rho = wk.z % d, sp = wk.z / d;
  const int64_t lor = rho < p.lo ? (p.lo - rho + d - 1) / d : 0;  // output rows of this residue class
  const int64_t t0 = static_cast<int64_t>(wk.y) * TT;
  if (t0 * M >= lor) return;
  const int64_t c0 = static_cast<int64_t>(wk.x) * 64;
  const int ci = static_cast<int>(p.ci), co = static_cast<int>(p.co);
  const int chunks = ci / (16 * S);
  const int steps = A * chunks;
  // split-K: this workgroup runs steps [sb, se) of the point-major step sequence; a point cut by the range is
  // folded with AT at the range's end, and AT is linear, so the splits' outputs sum to the full one
  const int sb = static_cast<int>(static_cast<int64_t>(steps) * sp / p.split);
  const int se = static_cast<int>(static_cast<int64_t>(steps) * (sp + 1) / p.split);
  const int64_t nci = static_cast<int64_t>(N) * ci;
  const int arow = 32 * wm + lr, bcol = 32 * wn + lr;

  // Operand addresses are a uniform pointer, advanced per step by scalar arithmetic, plus a 32-bit per-lane offset.
  // V: rows past rmax (they only feed tiles never stored) read the last one.
  auto vAt = [&](int xi, int ch) {
    return p.v + ((static_cast<int64_t>(rho) * A + xi) * p.rmax + t0) * ci + static_cast<int64_t>(ch) * 16 * S;
  };
  constexpr int kSet = UL == 0 ? 0 : UL == 1 ? 1024 : 768;  // floats of a fragment's slab (UL 2: of its 32-column half)
  auto uAt = [&](int xi, int ch) {
    if constexpr (UL == 0) return p.u + (static_cast<int64_t>(xi) * nci + ch * 16 * S) * co + c0;
    return p.u + (static_cast<int64_t>(xi) * (co / 64) + c0 / 64) * nci * (UL == 1 ? 64 : 96) +
           static_cast<int64_t>(ch) * E * kSet;
  };
  // from one step's operands to the next one's, and what a new point adds
  const int64_t vWrap = (p.rmax - 1) * ci;
  const int64_t uStep = UL == 0 ? static_cast<int64_t>(16 * S) * co : E * kSet;
  const int64_t uWrap = UL == 0   ? (nci - ci) * co
                        : UL == 1 ? (co / 64 - 1) * nci * 64
                                  : (co / 64) * nci * 96 - nci * 48;
  auto vRow = [&](int row) { return static_cast<unsigned>(min<int64_t>(row, p.rmax - 1 - t0)) * ci; };
  // Raw V of a step: a float4 of row tid / 4 (quad tid % 4) per chunk, and one float of the N - 1 extra rows, held by
  // every 16 (N - 1) S threads alike.
  struct RawA {
    f32x4 v[S];
    float x;
  } ra0, ra1;
  const int srow = tid >> 2, squad = tid & 3;
  constexpr int XN = N > 1 ? N - 1 : 1;
  const int xch = tid & 15, xrow = TT + (tid >> 4) % XN, xsub = (tid >> 4) / XN % S;
  const unsigned aoff = vRow(srow) + 4 * squad, xoff = vRow(xrow) + 16 * xsub + xch;
  const unsigned boff = UL == 0   ? 8 * lk * co + bcol
                        : UL == 1 ? (2 * lk * 64 + bcol) * 4
                                  : static_cast<unsigned>(wn * nci * 48) + lane * 4;
  auto loadA = [&](const float* vx, RawA& ra) {
#pragma unroll
    for (int i = 0; i < S; ++i) ra.v[i] = *reinterpret_cast<const f32x4*>(vx + 16 * i + aoff);
    if constexpr (N > 1) ra.x = vx[xoff];
  };
  auto storeA = [&](Stage& As, const RawA& ra) {
#pragma unroll
    for (int i = 0; i < S; ++i) {
      u32x2 h, m, l;
      split3(ra.v[i], kSplitScale, h, m, l);
      const int s2 = 4 * srow + 2 * ((squad >> 1) ^ ((srow >> 3) & 1)) + (squad & 1);
      reinterpret_cast<u32x2*>(As[i][0])[s2] = h;
      reinterpret_cast<u32x2*>(As[i][1])[s2] = m;
      reinterpret_cast<u32x2*>(As[i][2])[s2] = l;
    }
    if constexpr (N > 1) {
      unsigned h, m, l;
      split3(ra.x, 0.0f, kSplitScale, h, m, l);
      const int s8 = 8 * (xrow * 2 + ((xch >> 3) ^ ((xrow >> 3) & 1))) + (xch & 7);
      reinterpret_cast<unsigned short*>(As[xsub][0])[s8] = static_cast<unsigned short>(h);
      reinterpret_cast<unsigned short*>(As[xsub][1])[s8] = static_cast<unsigned short>(m);
      reinterpret_cast<unsigned short*>(As[xsub][2])[s8] = static_cast<unsigned short>(l);
    }
  };
  // channels 8 lk .. 8 lk + 7 of fragment e's 16, column c0 + bcol
  auto loadB = [&](const float* ux, int e, RawB& r) {
    if constexpr (UL == 0) {
      const float* ue = ux + (static_cast<int64_t>(e % N) * ci + (e / N) * 16) * co;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int q = 0; q < 4; ++q) r[h][q] = ue[static_cast<int64_t>(4 * h + q) * co + boff];
    } else {
#pragma unroll
      for (int h = 0; h < (UL == 1 ? 2 : 3); ++h)
        r[h] = *reinterpret_cast<const f32x4*>(ux + e * kSet + h * 256 + boff);
    }
  };
  auto partsB = [&](const RawB& r) {
    if constexpr (UL == 2)
      return Frag3{__builtin_bit_cast(bf16x8, r[0]), __builtin_bit_cast(bf16x8, r[1]),
                   __builtin_bit_cast(bf16x8, r[2])};
    else
      return split3(r[0], r[1], kSplitScale);
  };

  f32x16 acc;
  float y[M][16];
  auto clear = [&](auto& x) {
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = 0.0f;
  };
  // a finished point (or this split's part of it), its sums in units of 1 / unit, folds into the output rows
  auto fold = [&](int xi, float unit) {
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const float at = p.tr[A * A + j * A + xi] * unit;
#pragma unroll
      for (int r = 0; r < 16; ++r) y[j][r] += at * acc[r];
    }
    clear(acc);
  };
  clear(acc);
#pragma unroll
  for (int j = 0; j < M; ++j) clear(y[j]);

  // A step computes from one LDS buffer. Its first work is to split and store the next step's V rows, loaded two steps
  // earlier, into the other one, and to load those of the step after the next but one into the same registers (V comes
  // from HBM). Past the last step the operands of the last are loaded again. cv, cu: chunk of the step whose V / U
  // pointer is vp / up; xs, cs: point and chunk of the step being computed.
  int xs = sb / chunks, cs = sb - xs * chunks, cv = cs, cu = cs;
  const float *vp = vAt(xs, cs), *up = uAt(xs, cs);
  auto nextV = [&](bool more) {
    const bool wrap = cv + 1 == chunks;
    vp += more ? 16 * S + (wrap ? vWrap : 0) : 0;
    cv = more ? (wrap ? 0 : cv + 1) : cv;
  };
  auto nextU = [&](bool more) {
    const bool wrap = cu + 1 == chunks;
    up += more ? uStep + (wrap ? uWrap : 0) : 0;
    cu = more ? (wrap ? 0 : cu + 1) : cu;
  };
  RawB rb[E];
  loadA(vp, ra0);
  nextV(sb + 1 < se);
  loadA(vp, ra1);
#pragma unroll
  for (int e = 0; e < E; ++e) loadB(up, e, rb[e]);
  storeA(As0, ra0);
  nextV(sb + 2 < se);
  loadA(vp, ra0);
  __syncthreads();
  auto step = [&](int s, Stage& As, Stage& other, RawA& ra) {
    storeA(other, ra);
    nextV(s + 3 < se);
    nextU(s + 1 < se);
    loadA(vp, ra);
    auto fragA = [&](int e) {
      const int row = arow + e % N, slot = row * 2 + (lk ^ ((row >> 3) & 1));
      return Frag3{__builtin_bit_cast(bf16x8, As[e / N][0][slot]), __builtin_bit_cast(bf16x8, As[e / N][1][slot]),
                   __builtin_bit_cast(bf16x8, As[e / N][2][slot])};
    };
    Frag3 af = fragA(0);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const Frag3 bf = partsB(rb[e]), cur = af;
      if (e + 1 < E) af = fragA(e + 1);  // the next fragment's reads cover this one's MFMAs
      acc = mfma3(cur, bf, acc);
      loadB(up, e, rb[e]);  // the next step's
    }
    const bool wrap = cs + 1 == chunks;
    if (wrap || s == se - 1) fold(xs, UL == 2 ? kSplitUnscale : kSplitUnscale * kSplitUnscale);
    cs = wrap ? 0 : cs + 1;
    xs += wrap;
    __syncthreads();
  };
  int s = sb;
  for (; s + 1 < se; s += 2) {
    step(s, As0, As1, ra1);
    step(s + 1, As1, As0, ra0);
  }
  if (s < se) step(s, As0, As1, ra1);

  // an infinity or NaN may come from the split (split3.h): such a wave runs its steps again on f32 MFMAs, operands
  // straight from memory
  float bad = 0.0f;
#pragma unroll
  for (int j = 0; j < M; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) bad = fmaf(y[j][r], 0.0f, bad);  // NaN after either
  if (__any(bad != bad)) {
#pragma unroll
    for (int j = 0; j < M; ++j) clear(y[j]);
#pragma unroll 1
    for (int f = sb; f < se; ++f) {
      const int xf = f / chunks, cf = f - xf * chunks;
      const float *vf = vAt(xf, cf), *uf = uAt(xf, cf);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        RawB bq;
        loadB(uf, e, bq);
        if constexpr (UL == 2) joinParts(bq, 1.0f);
        const float* vr = vf + vRow(arow + e % N) + 16 * (e / N) + 8 * lk;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 aq = *reinterpret_cast<const f32x4*>(vr + 4 * h);
#pragma unroll
          for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(aq[q], bq[h][q], acc, 0, 0, 0);
        }
      }
      if (cf == chunks - 1 || f == se - 1) fold(xf, 1.0f);
    }
  }

  // Register r = tile tb0 + 8 (r / 4) + 4 lk + r % 4, channel c0 + bcol. Output rows go through buffer resources that
  // end with the tensor (a row past the residue class is past the tensor): loads there give 0 and stores are dropped,
  // with no branch per element. One resource per 8-tile row group keeps the lane offsets in 32 bits; rows too long for
  // that (32 of them past 4 GB) are addressed one by one.
  const int64_t tb0 = t0 + 32 * __builtin_amdgcn_readfirstlane(wm);
  const int left = static_cast<int>(min<int64_t>(lor - tb0 * M, 32 * M)) - 4 * lk * M;  // output rows from this lane's
  auto orow = [&](int j, int r) { return (8 * (r >> 2) + (r & 3)) * M + j; };
  const int64_t stride = static_cast<int64_t>(d) * co;
  const bool wide = stride >= int64_t{1} << 25;
  const unsigned rowBytes = static_cast<unsigned>(stride) * 4;
  const unsigned ooff = 4 * lk * M * rowBytes + static_cast<unsigned>(c0 + bcol) * 4;
  auto rows = [&](const float* base, int rg) {  // the 8-tile group rg
    const int64_t first = rho + (tb0 + 8 * rg) * M * d;
    const int64_t bytes = base ? min<int64_t>(max<int64_t>(p.lo - first, 0) * co * 4, 0xfffffff0) : 0;
    return uniformRsrc(base + (bytes ? first * co : 0), static_cast<unsigned>(bytes));
  };
  const int64_t wideOff = rho * static_cast<int64_t>(co) + (tb0 + 4 * lk) * M * stride + c0 + bcol;
  auto store = [&](float* base) {
    if (wide) {
#pragma unroll
      for (int j = 0; j < M; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (orow(j, r) < left) base[wideOff + orow(j, r) * stride] = y[j][r];
      return;
    }
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) {
      const auto rs = rows(base, rg);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < M; ++j)
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y[j][4 * rg + r]), rs, ooff + (r * M + j) * rowBytes, 0,
                                                0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (p.split > 1) {  // raw partial rows; bias, residual, scale and statistics come in the reduction
    store(p.part + static_cast<int64_t>(sp) * p.lo * co);
    return;
  }

  const float bias = p.bias[c0 + bcol];
  // every residual load before the first store; no residual: an empty resource, whose loads give 0
  const __amdgpu_buffer_rsrc_t rs[4] = {rows(p.res, 0), rows(p.res, 1), rows(p.res, 2), rows(p.res, 3)};
#pragma unroll
  for (int j = 0; j < M; ++j) {
    float rv[16];
    if (wide) {
#pragma unroll
      for (int r = 0; r < 16; ++r) rv[r] = p.res && orow(j, r) < left ? p.res[wideOff + orow(j, r) * stride] : 0.0f;
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        rv[r] = __uint_as_float(
            __builtin_amdgcn_raw_buffer_load_b32(rs[r >> 2], ooff + ((r & 3) * M + j) * rowBytes, 0, 0));
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) y[j][r] = ((y[j][r] + bias) + rv[r]) * p.scale;
    __builtin_amdgcn_sched_barrier(0);
  }
  store(p.out);
  if (p.stats) {
    // chunks of 128 rows of this residue class. M = 4: 32 tiles, one wave row, reduced in the wave; M = 2: the
    // workgroup's 64 tiles, the two wave rows combined through LDS.
    constexpr int TPC = kWinoRows / M;  // tiles per chunk
    const int64_t chunk = tb0 / TPC;
    const float nrows = static_cast<float>(min<int64_t>(kWinoRows, lor - chunk * kWinoRows));
    const bool whole = lor - tb0 * M >= 32 * M;
    auto rowSum = [&](auto term) {
      float t = 0.0f;
      if (whole) {
#pragma unroll
        for (int j = 0; j < M; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) t += term(y[j][r]);
      } else {
#pragma unroll
        for (int j = 0; j < M; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) t += orow(j, r) < left ? term(y[j][r]) : 0.0f;
      }
      t += __shfl_xor(t, 32, 64);
      if constexpr (TPC == 64) {
        __syncthreads();
        if (lk == 0) red[wm][bcol] = t;
        __syncthreads();
        t = red[0][bcol] + red[1][bcol];
      }
      return t;
    };
    const float mean = rowSum([](float v) { return v; }) / nrows;
    const float m2 = rowSum([&](float v) { return (v - mean) * (v - mean); });
    if (lk == 0 && (TPC == 32 || wm == 0) && nrows > 0.0f) {
      float* st = p.stats + ((static_cast<int64_t>(rho) * p.chunks + chunk) * co + c0 + bcol) * 2;
      st[0] = mean;
      st[1] = m2;
    }
  }
}

// Ut (u_layout 1) -> Us (u_layout 2), a fragment's 8 values per thread.
__global__ __launch_bounds__(256) void winoSplitUKernel(const float* __restrict__ ut, u32x4* __restrict__ us,
                                                       int64_t slabs, int64_t sets) {
  const int64_t total = slabs * sets * 128;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int lane = static_cast<int>(i & 63), half = static_cast<int>(i >> 6) & 1;
    const int64_t set = (i >> 7) % sets, slab = (i >> 7) / sets;
    const float* src = ut + (slab * sets + set) * 1024 + ((lane >> 5) * 128 + half * 32 + (lane & 31)) * 4;
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = src[(k >> 2) * 256 + (k & 3)];
    u32x4 parts[3];
    splitExact(v, 1.0f, parts);
#pragma unroll
    for (int q = 0; q < 3; ++q) us[((slab * 2 + half) * sets + set) * 192 + q * 64 + lane] = parts[q];
  }
}

// Split-K reduction: out = (sum_s part[s] + bias [+ res]) * scale, the s sum in split order; one
// float4 of one row per thread, grid-stride (Co % 64 == 0, so a float4 never straddles two rows).
__global__ __launch_bounds__(256) void winoSplitReduceKernel(const float* __restrict__ part, int split,
                                                            const float* __restrict__ bias,
                                                            const float* __restrict__ res, float* __restrict__ out,
                                                            int64_t lo, int64_t co, float scale) {
  const int64_t n4 = lo * co / 4, plane = lo * co;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n4;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t e = 4 * i, col = e % co;
    v4w sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int sp = 0; sp < 8; ++sp)  // split <= 8
      if (sp < split) sum += *reinterpret_cast<const v4w*>(part + sp * plane + e);
    v4w o = sum + *reinterpret_cast<const v4w*>(bias + col);
    if (res) o += *reinterpret_cast<const v4w*>(res + e);
    *reinterpret_cast<v4w*>(out + e) = o * scale;
  }
}

// AdaIN affine from wino_mm statistics (chunks per residue class of the dilation), 4 channels x 64 chunk slices
// per workgroup.
__global__ __launch_bounds__(kAffineThreads) void winoAffineKernel(const float* __restrict__ st,
                                                                  const float* __restrict__ gb,
                                                                  float* __restrict__ af, int64_t l, int64_t c, int d,
                                                                  int64_t chunks, int64_t creal, float eps) {
  adainAffineSlices(st, gb, af, l, c, d, chunks, creal, eps);
}

}  // namespace lkd

extern "C" {

int lk_hip_wino_tf_lc_f32(const float* x, const float* tr, const float* affine, const float* alpha, float* v,
                          int64_t l, int64_t c, int dilation, int padding, int kernel, int tile, int64_t v_rows,
                          int act, float slope, void* stream) {
  if (c % 4 != 0 || dilation < 1 || padding % dilation != 0 || (tile != 2 && tile != 4)) return 1;
  const int a = tile == 2 ? 4 : kernel == 3 ? 6 : 7;
  if (v_rows % (static_cast<int64_t>(dilation) * a) != 0) return 1;
  const int64_t rmax = v_rows / (static_cast<int64_t>(dilation) * a);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int padq = padding / dilation;
  const auto threads = [&](int r) { return static_cast<int64_t>(dilation) * ((rmax + r - 1) / r) * (c / 4); };
  if (threads(1) == 0) return 0;
  const auto go = [&](auto kernel, int r) {
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(std::min<int64_t>((threads(r) + 255) / 256, 65536))),
                       dim3(256), 0, s, x, tr, affine, alpha, v, l, c, dilation, padq, rmax, act, slope);
  };
  // One tile row per thread while that is what fills the chip (latency-bound: a thread's loads and stores are one round
  // trip each), two beyond: in us with one / two / four rows per thread, (L, C, K, d) = (287, 1104, 3, 1) 4.9 / 6.2 /
  // 8.4, (5740, 256, 7, 3) 7.5 / 8.0 / 10.2, (34441, 128, 7, 3) 13.1 / 14.3 / 15.1, (100000, 128, 11, 1) 28.7 / 28.0 /
  // 30.2, (293281, 128, 11, 5) 86.9 / 85.1 / 89.2.
  const auto pick = [&](auto one, auto two) { threads(1) < 524288 ? go(one, 1) : go(two, 2); };
  if (a == 4)
    pick(lkd::winoTfKernel<2, 4, 1>, lkd::winoTfKernel<2, 4, 2>);
  else if (a == 6)
    pick(lkd::winoTfKernel<4, 6, 1>, lkd::winoTfKernel<4, 6, 2>);
  else
    pick(lkd::winoTfKernel<4, 7, 1>, lkd::winoTfKernel<4, 7, 2>);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

}  // extern "C"

namespace {

template <int UL>
int winoMm(const float* v, const float* u, const float* bias, const float* res, float* out, const float* tr,
           float* stats, int64_t v_rows, int64_t ci, int64_t co, int64_t lo, int dilation, int groups, int kernel,
           int tile, float scale, void* workspace, int64_t workspace_bytes, void* stream) {
  const int a = tile == 2 ? 4 : kernel == 3 ? 6 : 7;
  if (ci % 16 != 0 || co % 64 != 0 || dilation < 1 || groups < 1 || groups > 3 || lo < 1) return 1;
  if (v_rows % (static_cast<int64_t>(dilation) * a) != 0) return 1;  // V holds whole (residue, point) row blocks
  if ((tile == 2 && groups != 1) || (a == 6 && groups != 1) || (a == 7 && groups < 2)) return 1;
  const int64_t rmax = v_rows / (static_cast<int64_t>(dilation) * a);
  const int m = tile;
  const int64_t tiles = ((lo + dilation - 1) / dilation + m - 1) / m;  // residue class 0 is the longest
  if (rmax < tiles + groups - 1) return 1;  // V must hold every tile and its group shifts
  // split-K when the grid is too small to fill the chip (two workgroups per CU): at least 32 steps per split (fewer
  // measured slower than no split on MI355X: the partial rows' round trip and the second launch outweigh the extra
  // workgroups; so did splits up to three workgroups per CU at 16 steps), partials in the workspace past its 64 KiB
  // counter area
  // lane offsets of 32 bits: 66 rows of V, 8 rows of U (operands of more than 150 GB)
  if ((63 + groups) * ci >= int64_t{1} << 32 || 8 * co >= int64_t{1} << 32) return 1;
  const int64_t base = (co / 64) * ((tiles + 63) / 64) * dilation;
  const int steps = a * static_cast<int>(ci / 16);  // in 16-channel units
  // one tap group: 48 or 32 channels per pipeline step where they divide Ci (with more groups the second chunk's
  // fragments spill: K = 11 333 -> 543 us)
  const int sub = groups == 1 && tile == 4 ? ((ci / 16) % 3 == 0 ? 3 : (ci / 16) % 2 == 0 ? 2 : 1) : 1;
  int split = 1;
  if (workspace && base < 512) {
    split = static_cast<int>(std::min<int64_t>({8, 512 / base, steps / 32}));
    while (split > 1 && 65536 + static_cast<int64_t>(split) * lo * co * 4 > workspace_bytes) --split;
    split = std::max(split, 1);
  }
  float* part = split > 1 ? reinterpret_cast<float*>(static_cast<char*>(workspace) + 65536) : nullptr;
  lkd::WinoMmArgs p{v, u, bias, res, out, tr, stats, part, lo, ci, co, rmax,
                    ((lo + dilation - 1) / dilation + lkd::kWinoRows - 1) / lkd::kWinoRows, dilation, split, scale};
  const dim3 grid(static_cast<unsigned>(co / 64), static_cast<unsigned>((tiles + 63) / 64),
                  static_cast<unsigned>(dilation * split));
  hipStream_t s = static_cast<hipStream_t>(stream);
  const auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, p); };
  if (a == 4)
    go(lkd::winoMmKernel<2, 4, 1, 1, UL>);
  else if (a == 6)
    sub == 3 ? go(lkd::winoMmKernel<4, 6, 1, 3, UL>) : sub == 2 ? go(lkd::winoMmKernel<4, 6, 1, 2, UL>)
                                                                : go(lkd::winoMmKernel<4, 6, 1, 1, UL>);
  else
    groups == 2 ? go(lkd::winoMmKernel<4, 7, 2, 1, UL>) : go(lkd::winoMmKernel<4, 7, 3, 1, UL>);
  if (split > 1) {
    hipLaunchKernelGGL(lkd::winoSplitReduceKernel,
                       dim3(static_cast<unsigned>(std::min<int64_t>((lo * co / 4 + 255) / 256, 8192))), dim3(256), 0,
                       s, part, split, bias, res, out, lo, co, scale);
    // the statistics of the summed output, per residue class as the fused epilogue writes them
    if (stats && lkh::residueStats(out, stats, lo, co, dilation, p.chunks, s)) return 2;
  }
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

}  // namespace

extern "C" {

int lk_hip_wino_mm_lc_f32(const float* v, const float* u, const float* bias, const float* res, float* out,
                          const float* tr, float* stats, int64_t v_rows, int64_t ci, int64_t co, int64_t lo,
                          int dilation, int groups, int kernel, int tile, float scale, void* workspace,
                          int64_t workspace_bytes, void* stream) {
  return winoMm<0>(v, u, bias, res, out, tr, stats, v_rows, ci, co, lo, dilation, groups, kernel, tile, scale,
                   workspace, workspace_bytes, stream);
}

int lk_hip_wino_mm_ut_lc_f32(const float* v, const float* ut, const float* bias, const float* res, float* out,
                             const float* tr, float* stats, int64_t v_rows, int64_t ci, int64_t co, int64_t lo,
                             int dilation, int groups, int kernel, int tile, float scale, void* workspace,
                             int64_t workspace_bytes, void* stream) {
  return winoMm<1>(v, ut, bias, res, out, tr, stats, v_rows, ci, co, lo, dilation, groups, kernel, tile, scale,
                   workspace, workspace_bytes, stream);
}

int lk_hip_wino_mm_us_lc_f32(const float* v, const void* us, const float* bias, const float* res, float* out,
                             const float* tr, float* stats, int64_t v_rows, int64_t ci, int64_t co, int64_t lo,
                             int dilation, int groups, int kernel, int tile, float scale, void* workspace,
                             int64_t workspace_bytes, void* stream) {
  return winoMm<2>(v, static_cast<const float*>(us), bias, res, out, tr, stats, v_rows, ci, co, lo, dilation, groups,
                   kernel, tile, scale, workspace, workspace_bytes, stream);
}

// Ut [A, Co / 64, N Ci 64] -> Us [A, Co / 64, N Ci 96] (bf16 parts), n = N Ci a multiple of 16, slabs = A Co / 64.
int lk_hip_wino_split_u_f32(const float* ut, void* us, int64_t slabs, int64_t n, void* stream) {
  if (slabs < 0 || n < 0 || n % 16 != 0) return 1;
  if (slabs == 0 || n == 0) return 0;
  hipLaunchKernelGGL(lkd::winoSplitUKernel, dim3(static_cast<unsigned>(std::min<int64_t>(lkh::ceilDiv(slabs * n * 8, 256), 8192))),
                     dim3(256), 0, static_cast<hipStream_t>(stream), ut, static_cast<lkd::u32x4*>(us), slabs, n / 16);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int lk_hip_wino_adain_affine_lc_f32(const float* stats, const float* gb, float* af, int64_t s, int64_t c,
                                    int64_t creal, int dilation, int64_t length, float eps, void* stream) {
  if (dilation < 1 || s % dilation != 0 || length < 1 || creal > c) return 1;
  hipLaunchKernelGGL(lkd::winoAffineKernel, dim3(lkh::ceilDiv(c, lkd::kAffineCh)), dim3(lkd::kAffineThreads), 0,
                     static_cast<hipStream_t>(stream),
                     stats, gb, af, length, c, dilation, s / dilation, creal, eps);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

}  // extern "C"

namespace lkh {

namespace {

// wino_tf[_snake|_leaky]_lc_f32_gpu. ptrs: x, tr, [affine], [alpha], v. ints: x(L, C), tr(T), [affine(3, C)],
// [alpha(C)], v(R, C), dilation, groups, kernel, padding, tile; floats (leaky): slope.
template <int ACT>
void runWinoTf(ExecCtx& ctx, const KernelArgs& a) {
  const int64_t l = a.ints[0], c = a.ints[1];
  const int o = ACT == 1 ? 6 : ACT == 2 ? 5 : 3;  // v dims
  const int64_t vr = a.ints[o];
  const int d = static_cast<int>(a.ints[o + 2]), k = static_cast<int>(a.ints[o + 4]);
  const int pad = static_cast<int>(a.ints[o + 5]), tile = static_cast<int>(a.ints[o + 6]);
  LK_REQUIRE(ctx, a.ints[o + 1] == c, "wino_tf: v must be f32[R, C]");
  const int vp = ACT == 1 ? 4 : ACT == 2 ? 3 : 2;
  const float slope = ACT == 2 && a.numFloats > 0 ? static_cast<float>(a.floats[0]) : 0.0f;
  if (lk_hip_wino_tf_lc_f32(P<float>(a, 0), P<float>(a, 1), ACT ? P<float>(a, 2) : nullptr,
                            ACT == 1 ? P<float>(a, 3) : nullptr, P<float>(a, vp), l, c, d, pad, k, tile, vr, ACT, slope,
                            ctx.stream))
    ctx.error = "wino_tf: invalid configuration";
}

// wino_mm[_res][_stats]_lc_f32_gpu. ptrs: v, u, b, tr, x, [res], out, [stats]. ints: v(R, Ci), u(A, N Ci, Co),
// b(Co), tr(T), x(L, Ci), [res(Lo, Co)], out(Lo, Co), [stats(d chunks, Co, 2)], dilation, groups, kernel,
// padding, tile, [u_layout]; floats: [oscale]. u_layout (this backend's addition; absent = 0, the reference's
// layout): 1, u is U tiled, Ut(A, Co / 64, N Ci 64); 2, U split, Us(A, Co / 64, N Ci 96) (winoMmKernel's UL layouts).
template <bool RES, bool STATS>
void runWinoMm(ExecCtx& ctx, const KernelArgs& a) {
  const int64_t vr = a.ints[0], ci = a.ints[1];
  const int o = RES ? 11 : 9;
  const int at = o + 2 + (STATS ? 3 : 0);
  const int64_t co = a.ints[o + 1], lo = a.ints[o];
  const int d = static_cast<int>(a.ints[at]), groups = static_cast<int>(a.ints[at + 1]);
  const int k = static_cast<int>(a.ints[at + 2]), tile = static_cast<int>(a.ints[at + 4]);
  const int64_t ul = a.numInts > static_cast<uint32_t>(at + 5) ? a.ints[at + 5] : 0;
  LK_REQUIRE(ctx,
             ul == 1 || ul == 2 ? (a.ints[3] * 64 == co && a.ints[4] == groups * ci * (ul == 1 ? 64 : 96))
                                : (a.ints[4] == co && a.ints[3] == groups * ci),
             "wino_mm: u must be f32[A, N Ci, Co] (u_layout 1: f32[A, Co / 64, N Ci 64], 2: f32[A, Co / 64, N Ci 96])");
  const int64_t alpha = tile == 2 ? 4 : k == 3 ? 6 : 7;  // transform points of this kernel size and tile
  LK_REQUIRE(ctx, a.ints[2] == alpha, "wino_mm: u's leading dim must be the transform's point count");
  LK_REQUIRE(ctx, d >= 1 && vr % (static_cast<int64_t>(d) * alpha) == 0,
             "wino_mm: v rows must be a multiple of dilation * points");
  const int outp = RES ? 6 : 5;
  const float scale = RES && a.numFloats > 0 ? static_cast<float>(a.floats[0]) : 1.0f;
  const auto mm = ul == 1 ? winoMm<1> : ul == 2 ? winoMm<2> : winoMm<0>;
  if (mm(P<float>(a, 0), P<float>(a, 1), P<float>(a, 2), RES ? P<float>(a, 5) : nullptr, P<float>(a, outp),
         P<float>(a, 3), STATS ? P<float>(a, outp + 1) : nullptr, vr, ci, co, lo, d, groups, k, tile, scale,
         ctx.workspace, static_cast<int64_t>(ctx.workspaceBytes), ctx.stream))
    ctx.error = "wino_mm: invalid configuration";
}

// wino_split_u_f32_gpu. ptrs: ut, us. ints: ut(A, Co / 64, N Ci 64), us(A, Co / 64, N Ci 96).
void runWinoSplitU(ExecCtx& ctx, const KernelArgs& a) {
  LK_REQUIRE(ctx, a.ints[2] % 1024 == 0 && a.ints[3] == a.ints[0] && a.ints[4] == a.ints[1] &&
             a.ints[5] * 2 == a.ints[2] * 3, "wino_split_u: ut f32[A, Co / 64, N Ci 64], us f32[A, Co / 64, N Ci 96]");
  if (lk_hip_wino_split_u_f32(P<float>(a, 0), P<float>(a, 1), a.ints[0] * a.ints[1], a.ints[2] / 64, ctx.stream))
    ctx.error = "wino_split_u: invalid configuration";
}

// wino_adain_affine_lc_f32_gpu. ptrs: stats, gb, af. ints: stats(S, C, 2), gb(2 Creal), af(3, C), dilation,
// length; floats: eps.
void runWinoAffine(ExecCtx& ctx, const KernelArgs& a) {
  const int64_t s = a.ints[0], c = a.ints[1], g2 = a.ints[3];
  const int d = static_cast<int>(a.ints[6]);
  const int64_t length = a.ints[7];
  const float eps = a.numFloats > 0 ? static_cast<float>(a.floats[0]) : 1e-5f;
  LK_REQUIRE(ctx, a.ints[2] == 2 && g2 % 2 == 0 && g2 / 2 <= c, "wino_adain_affine: bad stats / gb");
  if (lk_hip_wino_adain_affine_lc_f32(P<float>(a, 0), P<float>(a, 1), P<float>(a, 2), s, c, g2 / 2, d, length, eps,
                                      ctx.stream))
    ctx.error = "wino_adain_affine: invalid configuration";
}

}  // namespace

void registerWinogradKernels() {
  const Device G = Device::Gpu;
  registerKernel({"wino_tf_lc_f32_gpu", G, runWinoTf<0>, 2, 1});
  registerKernel({"wino_tf_snake_lc_f32_gpu", G, runWinoTf<1>, 4, 1});
  registerKernel({"wino_tf_leaky_lc_f32_gpu", G, runWinoTf<2>, 3, 1});
  registerKernel({"wino_mm_lc_f32_gpu", G, runWinoMm<false, false>, 5, 1});
  registerKernel({"wino_mm_res_lc_f32_gpu", G, runWinoMm<true, false>, 6, 1});
  registerKernel({"wino_mm_stats_lc_f32_gpu", G, runWinoMm<false, true>, 5, 2});
  registerKernel({"wino_mm_res_stats_lc_f32_gpu", G, runWinoMm<true, true>, 6, 2});
  registerKernel({"wino_split_u_f32_gpu", G, runWinoSplitU, 1, 1});
  registerKernel({"wino_adain_affine_lc_f32_gpu", G, runWinoAffine, 2, 1});
}

}  // namespace lkh
