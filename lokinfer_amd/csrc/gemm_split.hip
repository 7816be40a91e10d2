// f32 GEMM over split weights (MI355X backend): out[M, N] = (act(A W + bias) + res) * scale on the bf16 matrix cores,
// both operands as three exact bf16 parts and six MFMAs per product (split3.h). A weight is laid out once by
// splitWeightKernel, in matrix-fragment order: Ws [ceil(N / 32), ceil(K / 16), 3, 64, 8] bf16, per 32-column block and
// 16 k the parts h, m, l, lane 32 lk + lr holding k = 8 lk .. 8 lk + 7 of column lr (zero past N and K). A wave's B
// fragment is then three coalesced 16-byte loads that bypass LDS and need no arithmetic; A is split once per workgroup
// on its way to LDS.
//
// The models' projections (ALBERT, the GPT-2 prompt chunk, the generator's transposed convs) run here; GEMMs over a
// plain f32 B stay on gemm.hip's f32 MFMA kernels, which read B as it is.
#include "common.h"
#include "lokinfer_hip.h"
#include "split3.h"

#include <algorithm>

namespace lkd {

enum : int { WS_ACT_NONE = 0, WS_ACT_RELU = 1, WS_ACT_GELU = 2 };

struct GemmWsParams {
  const float* a;
  const u32x4* ws;
  const float* bias;  // [N] or null
  const float* res;   // [M, N] or null
  float* c;
  int64_t m, n, k;
  int act;
  float scale;
  int planes;  // > 1: grid z = K range of an equal part of the steps, raw sums to c [planes, M, N]
  float wUnscale;  // inverse of the factor that the parts of W carry
};

// One fragment's 8 values per thread; w [K, N] (nt 0) or [N, K] (nt 1).
__global__ __launch_bounds__(256) void splitWeightKernel(const float* __restrict__ w, u32x4* __restrict__ ws, int64_t n,
                                                        int64_t k, int nt, float scale) {
  const int64_t kb = (k + 15) / 16, total = (n + 31) / 32 * kb * 64;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int lane = static_cast<int>(i & 63);
    const int64_t kc = (i >> 6) % kb, nb = (i >> 6) / kb;
    const int64_t col = nb * 32 + (lane & 31), k0 = kc * 16 + 8 * (lane >> 5);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = col < n && k0 + e < k ? w[nt ? col * k + k0 + e : (k0 + e) * n + col] : 0.0f;
    u32x4 parts[3];
    splitExact(v, scale, parts);
#pragma unroll
    for (int q = 0; q < 3; ++q) ws[(nb * kb + kc) * 192 + q * 64 + lane] = parts[q];
  }
}

// Bound by what feeds the MFMAs: 1.1 to 2.3 times the f32 MFMA kernels' rate (the launcher's table, and 53 shapes of the
// models' ranges). On the large tiles the matrix pipes are busy 46 - 49% of the time while waves wait to issue for half of
// their cycles (A's conversion and LDS stores, 1.7 conflict cycles per LDS instruction, 3 KB of B for 98 ns of a 32 x 32
// block's MFMAs); at (487, 768, 2304) they are busy 16%, at (59, 768, 2304) 3%, which is latency.
//
// Workgroup tile 32 TM rows x 32 NW columns; NW KG waves, wave (kg, wn) computing 32 TM x 32 over the K range of group kg
// (the groups' partial tiles meet in LDS at the end, summed in order). A step is KS deep in every group: its A tile is
// split while staged, double-buffered as [chunk of 16 k][part][row][2 halves of 8 k], half swizzled by (row >> 3) & 1; A and B
// are loaded D steps ahead.
template <int TM, int NW, int KG, int KS, int D>
__global__ __launch_bounds__(64 * NW * KG) void gemmWsKernel(GemmWsParams p) {
  constexpr int BM = 32 * TM, TG = 64 * NW;  // rows of the tile, threads of a K group
  constexpr int KC = KS / 16;                // 16-k chunks per step
  constexpr int UF = BM * KS / 8 < TG ? 1 : 2;  // float4s per unit of the A tile: 8 floats, or 4 where those are too few
  constexpr int UNITS = BM * KS / (4 * UF);
  constexpr int UA = UNITS / TG;
  static_assert(UA >= 1 && UNITS % TG == 0, "whole A units per thread");
  using Stage = u32x4[KC][3][BM * 2];
  constexpr int RED = KG > 1 ? (KG - 1) * BM * 32 * NW * 4 : 16;
  constexpr int BYTES = sizeof(Stage) * KG > RED / 2 ? static_cast<int>(sizeof(Stage)) * KG : RED / 2;
  // two objects, so that the compiler sees that a step's stores and reads never meet; the reduction reuses both
  __shared__ __attribute__((aligned(16))) char smem[2][BYTES];
  Stage* st0 = reinterpret_cast<Stage*>(smem[0]);
  Stage* st1 = reinterpret_cast<Stage*>(smem[1]);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lk = lane >> 5, wn = wave % NW, kg = wave / NW, gt = tid % TG;
  // a K group of one wave stages for itself: its LDS accesses are in order, and only the compiler has to keep them so
  auto meet = [] {
    if constexpr (NW == 1) __builtin_amdgcn_wave_barrier();
    else __syncthreads();
  };
  const GridItem gi = xcdOrderYFast();  // row blocks of one column block share an XCD's L2: W is read once per XCD
  const int64_t m0 = static_cast<int64_t>(gi.y) * BM;
  const int64_t nb = static_cast<int64_t>(gi.x) * NW + wn, nBlocks = (p.n + 31) / 32;
  const int64_t nbc = min<int64_t>(nb, nBlocks - 1);  // a wave past the last block repeats it and stores nothing
  const int kChunks = static_cast<int>((p.k + 15) / 16), allSteps = (kChunks + KC - 1) / KC;
  const int zb = allSteps * gi.z / p.planes, zn = allSteps * (gi.z + 1) / p.planes - zb;  // this workgroup's steps
  const int sb = zb + zn * kg / KG, se = zb + zn * (kg + 1) / KG;
  const int maxSteps = (zn + KG - 1) / KG;
  const int last = max(se - 1, 0);  // what a group loads past its range (one with no steps at all too)
  const int ik = static_cast<int>(p.k);
  const int64_t lastRow = p.m - 1;

  // A units of this thread: 4 UF consecutive k of one row; k past K loads the row's start and is zeroed when split
  const float* arow[UA];
  int aslot[UA], ak[UA];
#pragma unroll
  for (int u = 0; u < UA; ++u) {
    constexpr int PR = KS / (4 * UF);  // units per row
    const int idx = gt + u * TG, row = idx / PR;
    arow[u] = p.a + min<int64_t>(m0 + row, lastRow) * p.k;
    ak[u] = 4 * UF * (idx % PR);
    const int half = ak[u] >> 3;  // 8-k half of the step
    aslot[u] = ((half >> 1) * 3 * BM * 2 + row * 2 + ((half & 1) ^ ((row >> 3) & 1))) * (2 / UF) + (UF == 1 ? (ak[u] >> 2) & 1 : 0);
  }
  f32x4 ra[D][UA][UF];
  u32x4 rb[D][KC][3];
  auto loadA = [&](int s, f32x4(&r)[UA][UF]) {
    const int k0 = min(s, last) * KS;
#pragma unroll
    for (int u = 0; u < UA; ++u)
#pragma unroll
      for (int h = 0; h < UF; ++h) {
        const int kk = k0 + ak[u] + 4 * h;
        r[u][h] = *reinterpret_cast<const f32x4*>(arow[u] + (kk < ik ? kk : 0));
      }
  };
  auto storeA = [&](Stage* st, int s, const f32x4(&r)[UA][UF]) {
    // zero past K, and past the range of a group with fewer steps than the others: its products add nothing, and no
    // load or MFMA sits behind a branch (which would make the compiler wait for the loads just issued). The zero is the
    // split's scale, so it takes no instruction of its own (an infinity there becomes NaN, but its row holds one as well).
    const int k0 = s < se ? s * KS : ik;
#pragma unroll
    for (int u = 0; u < UA; ++u) {
      const float scale = k0 + ak[u] < ik ? kSplitScale : 0.0f;  // K % 8 == 0: a unit ends within K or starts past it
      if constexpr (UF == 2) {
        const Frag3 f = split3(r[u][0], r[u][1], scale);
        u32x4* dst = &st[kg][0][0][0] + aslot[u];
        dst[0] = __builtin_bit_cast(u32x4, f.h);
        dst[BM * 2] = __builtin_bit_cast(u32x4, f.m);
        dst[2 * BM * 2] = __builtin_bit_cast(u32x4, f.l);
      } else {
        u32x2* dst = reinterpret_cast<u32x2*>(&st[kg][0][0][0]) + aslot[u];
        split3(r[u][0], scale, dst[0], dst[BM * 4], dst[2 * BM * 4]);
      }
    }
  };
  const u32x4* wb = p.ws + nbc * kChunks * 192 + lane;
  auto loadB = [&](int s, int c, u32x4(&r)[3]) {
    const int64_t chunk = min(min(s, last) * KC + c, kChunks - 1);  // past K: A is zero there
#pragma unroll
    for (int q = 0; q < 3; ++q) r[q] = wb[chunk * 192 + q * 64];
  };

  f32x16 acc[TM], low[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = low[i][r] = 0.0f;
  // A of step t sits in register set t % D from D steps before it is stored, its B fragments in set t % D from D steps
  // before they are used
#pragma unroll
  for (int t = 0; t < D; ++t) {
    loadA(sb + t, ra[t]);
#pragma unroll
    for (int c = 0; c < KC; ++c) loadB(sb + t, c, rb[t][c]);
  }
  storeA(st0, sb, ra[0]);
  loadA(sb + D, ra[0]);
  meet();
  auto step = [&](int s, Stage* st, Stage* other, f32x4(&a)[UA][UF], u32x4(&b)[KC][3]) {
    storeA(other, s + 1, a);
    loadA(s + 1 + D, a);
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const Frag3 bf{__builtin_bit_cast(bf16x8, b[c][0]), __builtin_bit_cast(bf16x8, b[c][1]),
                     __builtin_bit_cast(bf16x8, b[c][2])};
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int row = 32 * i + lr, slot = row * 2 + (lk ^ ((row >> 3) & 1));
        const Frag3 af{__builtin_bit_cast(bf16x8, st[kg][c][0][slot]), __builtin_bit_cast(bf16x8, st[kg][c][1][slot]),
                       __builtin_bit_cast(bf16x8, st[kg][c][2][slot])};
        mfma3(af, bf, acc[i], low[i]);
      }
      loadB(s + D, c, b[c]);
    }
    meet();
  };
  int s = 0;
  for (; s + D <= maxSteps; s += D) {
#pragma unroll
    for (int t = 0; t < D; ++t)
      step(sb + s + t, t & 1 ? st1 : st0, t & 1 ? st0 : st1, ra[(t + 1) % D], rb[t]);
  }
#pragma unroll
  for (int t = 0; t < D - 1; ++t)
    if (s + t < maxSteps) step(sb + s + t, t & 1 ? st1 : st0, t & 1 ? st0 : st1, ra[(t + 1) % D], rb[t]);

  // an infinity or NaN may come from the split (split3.h): such a wave sums its K range again on f32 MFMAs
  float bad = 0.0f;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc[i][r] = (acc[i][r] + low[i][r]) * (kSplitUnscale * p.wUnscale);
      bad = fmaf(acc[i][r], 0.0f, bad);  // NaN after either
    }
  if (__any(bad != bad)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
#pragma unroll 1
    for (int c = sb * KC; c < min(se * KC, kChunks); ++c) {
      f32x4 b[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) b[q] = __builtin_bit_cast(f32x4, wb[static_cast<int64_t>(c) * 192 + q * 64]);
      joinParts(b, p.wUnscale);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const float* ar = p.a + min<int64_t>(m0 + 32 * i + lr, lastRow) * p.k;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int kk = c * 16 + 8 * lk + e;
          const float av = kk < ik ? ar[kk] : 0.0f;
          acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(av, b[e >> 2][e & 3], acc[i], 0, 0, 0);
        }
      }
    }
  }

  if constexpr (KG > 1) {  // partial tiles of groups 1 .. KG - 1 -> LDS (the stages are free after the last barrier)
    float* red = reinterpret_cast<float*>(&smem[0][0]);
    if constexpr (NW == 1) __syncthreads();  // another wave may still read the stages that the partial tiles overwrite
    auto at = [&](int g, int i, int r) {
      return ((g * NW + wn) * TM + i) * 1024 + (8 * (r >> 2) + 4 * lk + (r & 3)) * 32 + lr;
    };
    if (kg > 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) red[at(kg - 1, i, r)] = acc[i][r];
    }
    __syncthreads();
    if (kg > 0) return;
    for (int g = 0; g < KG - 1; ++g)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] += red[at(g, i, r)];
  }
  // accumulator r = row 8 (r / 4) + 4 lk + r % 4, column lr; residual loads before the first store
  const int64_t col = nb * 32 + lr;
  if (col >= p.n) return;
  float* c = p.c + static_cast<int64_t>(gi.z) * p.m * p.n;
  const float bias = p.bias ? p.bias[col] : 0.0f;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int64_t row0 = m0 + 32 * i + 4 * lk;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float v = acc[i][r] + bias;
      if (p.act == WS_ACT_RELU) v = fmaxf(v, 0.0f);
      else if (p.act == WS_ACT_GELU) v = geluTanh(v);
      acc[i][r] = v;
    }
    if (p.res) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][r] += p.res[min<int64_t>(row0 + 8 * (r >> 2) + (r & 3), lastRow) * p.n + col];
    }
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int64_t row = m0 + 32 * i + 4 * lk + 8 * (r >> 2) + (r & 3);
      if (row <= lastRow) c[row * p.n + col] = acc[i][r] * p.scale;
    }
}

}  // namespace lkd

namespace {

int splitWeight(const float* w, void* ws, int64_t n, int64_t k, int nt, float scale, void* stream) {
  if (n < 0 || k < 0) return 1;
  if (n == 0 || k == 0) return 0;
  const int64_t total = (n + 31) / 32 * ((k + 15) / 16) * 64;
  hipLaunchKernelGGL(lkd::splitWeightKernel, dim3(static_cast<unsigned>(std::min<int64_t>((total + 255) / 256, 16384))),
                     dim3(256), 0, static_cast<hipStream_t>(stream), w, static_cast<lkd::u32x4*>(ws), n, k, nt, scale);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int gemmWs(const float* a, const void* ws, const float* bias, const float* res, float* out, int64_t m, int64_t n,
           int64_t k, int act, float scale, int planes, float wUnscale, void* stream) {
  if (m < 0 || n < 0 || k <= 0 || k % 8 != 0 || k > (int64_t{1} << 30)) return 1;
  if (((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(ws)) & 15) != 0) return 1;
  if (m == 0 || n == 0) return 0;
  const lkd::GemmWsParams p{a, static_cast<const lkd::u32x4*>(ws), bias, res, out, m, n, k, act, scale, planes, wUnscale};
  hipStream_t s = static_cast<hipStream_t>(stream);
  const auto go = [&](auto kernel, int tm, int nw, int kg) {
    hipLaunchKernelGGL(kernel, dim3(lkh::ceilDiv(n, 32 * nw), lkh::ceilDiv(m, 32 * tm), static_cast<unsigned>(planes)),
                       dim3(64 * nw * kg), 0, s, p);
  };
  // Workgroups with tiles of 32 x 32, 32 x 64, 32 x 128 and 64 x 128. Smaller tiles read A and B more often, larger ones
  // leave CUs idle, so the rule is the smallest tile that fits the chip in one round of workgroups: one to each of the 256
  // CUs where K is spread over the waves (eight waves), then as many as the registers admit, three or two of four waves;
  // beyond that the largest tile. In us (graph replay) at (M, K, N), gemm.hip's f32 MFMA kernels (with their split-K
  // reduction), then the forms around the line:
  //   32 x 32 | 32 x 64, K over eight / four waves: (96, 768, 2304) 13.4, 8.3 | 9.8; (128, 768, 2304) 13.5, 17.0 | 10.0;
  //     (320, 768, 768) 18.0, 14.0 | 15.0; (360, 768, 768) 18.5, 19.9 | 15.2
  //   32 x 64 | 32 x 128 over two: (200, 768, 2304) 13.7, 10.2 | 12.5; (256, 768, 2304) 20.5, 14.4 | 13.6; (600, 2048, 768)
  //     39.8, 26.0 | 34.4; (700, 2048, 768) 49.7, 35.3 | 34.8
  //   32 x 128 over two | 32 x 64 over two with four waves: (430, 768, 2304) 23.0, 14.5 | 16.5; (460, 768, 2304) 28.4, 21.8
  //     | 20.5; (600, 768, 2048) 31.3, 23.6 | 22.6
  //   32 x 64 over two | 32 x 128: (512, 768, 3072) 32.1, 26.1 | 27.7; (600, 768, 3072) 40.9, 32.0 | 27.9; (900, 768, 2048)
  //     40.5, 31.2 | 26.0
  //   32 x 128 | 64 x 128: (1200, 256, 1536) 19.7, 11.9 | 12.4; (2400, 256, 1536) 41.2, 22.0 | 18.7; (800, 512, 5120) 64.1,
  //     33.7 | 40.7 (520 of the larger tiles: a second round for 8 of them); (1200, 512, 5120) 86.8, 51.1 | 44.3; (48880, 256,
  //     1536) 328, - | 268
  // One block of rows leaves most CUs without a workgroup and waits for W: four waves that load four steps ahead instead of
  // eight that load two, W from memory: (32, 768, 2304) 11.4 against 12.0, f32 10.9; (32, 3072, 768) in four ranges 18.1
  // against 18.8, f32 19.6; W in the caches 8.5 against 7.7, f32 10.1. Narrow W keeps the eight: (32, 768, 768) 11.9, 12.7.
  // The 32 x 64 tiles take steps of 32 k for a long K in one range, for the same reason. Steps of 16 | 32, W from memory:
  // (512, 3072, 768) 31.9 | 29.6, (512, 2048, 768) 22.5 | 21.7, (512, 768, 768) 11.6 | 11.7, (160, 3072, 768) in four ranges 12.8
  // | 12.8; in the caches 25.0 | 26.5, 18.3 | 19.4, 10.1 | 10.8, 9.7 | 10.5. A GPT-2 chunk of 512 tokens 1561 | 1532.
  const int64_t rows = static_cast<int64_t>(lkh::ceilDiv(m, 32)) * planes;
  const int64_t g1 = rows * lkh::ceilDiv(n, 32), g2 = rows * lkh::ceilDiv(n, 64), g4 = rows * lkh::ceilDiv(n, 128);
  const int64_t g8 = static_cast<int64_t>(lkh::ceilDiv(m, 64)) * lkh::ceilDiv(n, 128) * planes;
  if (m <= 32 && g1 > 64 && g1 <= 256)
    go(lkd::gemmWsKernel<1, 1, 4, 16, 4>, 1, 1, 4);
  else if (g1 <= 256)
    go(lkd::gemmWsKernel<1, 1, 8, 16, 2>, 1, 1, 8);
  else if (g2 <= 256 && planes == 1 && k >= 2560)
    go(lkd::gemmWsKernel<1, 2, 4, 32, 2>, 1, 2, 4);
  else if (g2 <= 256)
    go(lkd::gemmWsKernel<1, 2, 4, 16, 2>, 1, 2, 4);
  else if (g4 <= 256)
    go(lkd::gemmWsKernel<1, 4, 2, 32, 2>, 1, 4, 2);
  else if (g2 <= 768)
    go(lkd::gemmWsKernel<1, 2, 2, 32, 2>, 1, 2, 2);
  else if (g4 <= 512 || (g4 <= 1024 && g8 > 512))
    go(lkd::gemmWsKernel<1, 4, 1, 32, 4>, 1, 4, 1);
  else
    go(lkd::gemmWsKernel<2, 4, 1, 32, 2>, 2, 4, 1);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

}  // namespace

extern "C" {

int lk_hip_split_weight_f32(const float* w, void* ws, int64_t n, int64_t k, int nt, void* stream) {
  return splitWeight(w, ws, n, k, nt, lkd::kSplitScale, stream);
}

int lk_hip_gemm_ws_f32(const float* a, const void* ws, const float* bias, const float* res, float* out, int64_t m,
                       int64_t n, int64_t k, int act, float scale, void* stream) {
  return gemmWs(a, ws, bias, res, out, m, n, k, act, scale, 1, lkd::kSplitUnscale, stream);
}

int lk_hip_gemm_ws_splitk_f32(const float* a, const void* ws, float* part, int64_t m, int64_t n, int64_t k, int planes,
                              void* stream) {
  if (planes < 1 || planes > 64) return 1;
  return gemmWs(a, ws, nullptr, nullptr, part, m, n, k, 0, 1.0f, planes, lkd::kSplitUnscale, stream);
}

}  // extern "C"

namespace lkh {

namespace {

// The kernels' attr `scaled`: 1, the parts of W are those of kSplitScale W. Graphs saved before it existed name none; their
// weights are laid out, and read, unscaled.
bool scaledAttr(const KernelArgs& a, uint32_t at) { return a.numInts > at && a.ints[at] == 1; }

// split_weight_f32_gpu. ptrs: w, ws. ints: w(K, N) (nt: (N, K)), ws(ceil(N / 32), ceil(K / 16) 768), nt, [scaled].
void runSplitWeight(ExecCtx& ctx, const KernelArgs& a) {
  const bool nt = a.ints[4] != 0;
  const int64_t k = a.ints[nt ? 1 : 0], n = a.ints[nt ? 0 : 1];
  LK_REQUIRE(ctx, a.ints[2] == (n + 31) / 32 && a.ints[3] == (k + 15) / 16 * 768,
             "split_weight: ws must be f32[ceil(N / 32), ceil(K / 16) 768]");
  status(ctx,
         splitWeight(P<float>(a, 0), P<void>(a, 1), n, k, nt, scaledAttr(a, 5) ? lkd::kSplitScale : 1.0f, ctx.stream),
         "split_weight: launch failed");
}

// gemm_ws[_bias[_relu|_gelu|_res]]_f32_gpu. ptrs: a, ws, [bias], [res], out. ints: a(M, K), ws(..), [bias(N)],
// [res(M, N)], out(M, N), [scaled].
template <bool BIAS, int ACT, bool RES>
void runGemmWs(ExecCtx& ctx, const KernelArgs& a) {
  const int o = 4 + (BIAS ? 1 : 0) + (RES ? 2 : 0);
  const int64_t m = a.ints[0], k = a.ints[1], n = a.ints[o + 1];
  LK_REQUIRE(ctx, a.ints[o] == m && a.ints[2] == (n + 31) / 32 && a.ints[3] == (k + 15) / 16 * 768,
             "gemm_ws: a f32[M, K], ws of an f32[K, N] weight, out f32[M, N]");
  const int outp = 2 + (BIAS ? 1 : 0) + (RES ? 1 : 0);
  status(ctx,
         gemmWs(P<float>(a, 0), P<void>(a, 1), BIAS ? P<float>(a, 2) : nullptr, RES ? P<float>(a, 3) : nullptr,
                P<float>(a, outp), m, n, k, ACT, 1.0f, 1, scaledAttr(a, o + 2) ? lkd::kSplitUnscale : 1.0f, ctx.stream),
         "gemm_ws: K must be a multiple of 8 and the operands 16-byte aligned");
}

// gemm_ws_splitk_f32_gpu. ptrs: a, ws, parts. ints: a(M, K), ws(..), parts(S, M, N), [scaled], splits: the first
// splitKPlanes planes hold the K ranges' sums, as gemm_splitk's.
void runGemmWsSplitK(ExecCtx& ctx, const KernelArgs& a) {
  const int64_t m = a.ints[0], k = a.ints[1], splits = a.ints[4], n = a.ints[6];
  LK_REQUIRE(ctx, a.ints[5] == m && a.ints[2] == (n + 31) / 32 && a.ints[3] == (k + 15) / 16 * 768 && splits >= 1,
             "gemm_ws_splitk: a f32[M, K], ws of an f32[K, N] weight, parts f32[S, M, N]");
  const int64_t planes = splitKPlanes(m, n, splits);
  LK_REQUIRE(ctx, planes <= 64, "gemm_ws_splitk: S must be at most 64");
  const bool scaled = a.numInts > 8 && scaledAttr(a, 7);
  status(ctx, gemmWs(P<float>(a, 0), P<void>(a, 1), nullptr, nullptr, P<float>(a, 2), m, n, k, 0, 1.0f,
                     static_cast<int>(planes), scaled ? lkd::kSplitUnscale : 1.0f, ctx.stream),
         "gemm_ws_splitk: K must be a multiple of 8 and the operands 16-byte aligned");
}

}  // namespace

void registerGemmSplitKernels() {
  const Device G = Device::Gpu;
  registerKernel({"split_weight_f32_gpu", G, runSplitWeight, 1, 1});
  registerKernel({"gemm_ws_f32_gpu", G, runGemmWs<false, 0, false>, 2, 1});
  registerKernel({"gemm_ws_splitk_f32_gpu", G, runGemmWsSplitK, 2, 1});
  registerKernel({"gemm_ws_bias_f32_gpu", G, runGemmWs<true, 0, false>, 3, 1});
  registerKernel({"gemm_ws_bias_relu_f32_gpu", G, runGemmWs<true, 1, false>, 3, 1});
  registerKernel({"gemm_ws_bias_gelu_f32_gpu", G, runGemmWs<true, 2, false>, 3, 1});
  registerKernel({"gemm_ws_bias_res_f32_gpu", G, runGemmWs<true, 0, true>, 4, 1});
}

}  // namespace lkh
