// Row passes of the fused depth steps (the column passes and the order of the
// three passes of a step: step_kernels.hip), and the presence masks.
//
// LaneFft::NB rows per wave (one at 512 and 1024 points), loaded and
// stored straight from / to memory at the positions the first / last stage
// needs.  These passes move one or two wavefields and do one or two
// transforms per row: with the transforms free of index arithmetic they are
// bound by memory at the long rows (1024^2 x 128 planes, forward rows: 5.1 TB/s,
// 92 % of the stream copy) and by latency at small grids.
#include "fwix_kernels.h"
#include "fwix_launch.h"

namespace fwix {

// ------------------------------------------------------------------ row passes
// A row workgroup covers rows R0 .. R0 + RW NB - 1 (RW = kRowWaves, R0 a
// multiple of RW NB), its waves' LDS regions hold those rows in order, STRIDE
// apart.  In the quad-block layout the same rows are one contiguous run of
// elements from R0 N, so the workgroup moves them between LDS and memory with
// consecutive lanes on consecutive elements (whole 128-byte lines).
template <int N>
struct RowStage {
  using F = LaneFft<N>;
  static constexpr int ROWS = kRowWaves * F::NB, TOT = ROWS * N, PER = TOT / kRowThreads;
  static_assert(ROWS % 4 == 0 && PER * kRowThreads == TOT, "run must divide evenly");
  static __device__ __forceinline__ int row(int j) { return 4 * (j / (4 * N)) + (((j % (4 * N)) & 15) >> 2); }
  static __device__ __forceinline__ int col(int j) { return (((j % (4 * N)) >> 4) << 2) + (j & 3); }
  static __device__ __forceinline__ int addr(int j) { return row(j) * F::STRIDE + col(j); }
  // run (quad-block memory) -> LDS rows; rows at or beyond nrows read as zero
  static __device__ __forceinline__ void load(float2* lds, const float2* __restrict__ src, int R0, int nrows) {
    float2 t[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int j = threadIdx.x + k * kRowThreads;
      t[k] = R0 + row(j) < nrows ? src[(size_t)R0 * N + j] : czero();
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) lds[addr(threadIdx.x + k * kRowThreads)] = t[k];
  }
  // LDS rows -> run (quad-block memory), rows below nrows
  static __device__ __forceinline__ void store(const float2* lds, float2* __restrict__ dst, int R0, int nrows) {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int j = threadIdx.x + k * kRowThreads;
      if (R0 + row(j) < nrows) dst[(size_t)R0 * N + j] = lds[addr(j)];
    }
  }
};

// out = (add ? out : 0) + post(scale * F_x(pre * in))   along x
// (in / out are K when qin / qout: in the quad-block layout, staged through LDS)
template <int N, bool INV, bool PRE_TAPER, bool POST_TAPER>
__global__ __launch_bounds__(kRowThreads) void k_rows(KArgs a) {
  using F = LaneFft<N>;
  __shared__ float2 lds[kRowWaves * F::NB * F::STRIDE];
  const RowLane<N, float2> w(a);
  const int R0 = blockIdx.x * kRowWaves * F::NB;
  // K in the quad-block layout goes through LDS as whole lines; row-major K
  // is read and written like any wavefield
  const bool qin = a.qin && a.quad, qout = a.qout && a.quad;
  if (w.empty() && !qin && !qout) return;  // (the stagings are the whole workgroup's)
  float2* line = lds + ((threadIdx.x >> 6) * F::NB + w.b) * F::STRIDE;
  const float s = a.scale;  // row normalisation 1/sqrt(NX)
  // positions a transform reads and leaves its values at
  auto ci = [](int e) { return INV ? F::last_c(e) : F::first_c(e); };
  auto co = [](int e) { return INV ? F::first_c(e) : F::last_c(e); };
  float2 v[F::V];
  if (!qin) {
    const RowBuf<N, float2> in(a.in, w, false);
#pragma unroll
    for (int e = 0; e < F::V; ++e) v[e] = in.load(ci(e));
  } else {
    RowStage<N>::load(lds, a.in, R0, w.nrows);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < F::V; ++e) v[e] = line[w.l + ci(e)];
    wave_sync();  // the transform reuses the region it was read from
  }
  if constexpr (PRE_TAPER) {
    const float ty = a.tapy[w.iy];
    const float* tx = a.tapx + w.l;
#pragma unroll
    for (int e = 0; e < F::V; ++e) v[e] = cscale(v[e], tx[ci(e)] * ty);
  }
  // one transform, no loop: the twiddles come straight from memory (L1), which
  // leaves LDS for a fourth workgroup per CU at 1024 points
  F::template run<INV>(v, line, a.twx, w.l);
  if constexpr (POST_TAPER) {
    const float ty = a.tapy[w.iy];
    const float* tx = a.tapx + w.l;
#pragma unroll
    for (int e = 0; e < F::V; ++e) v[e] = cscale(cscale(v[e], s), tx[co(e)] * ty);
  } else {
#pragma unroll
    for (int e = 0; e < F::V; ++e) v[e] = cscale(v[e], s);
  }
  if (qout) {  // K is never added to
    wave_sync();
#pragma unroll
    for (int e = 0; e < F::V; ++e) line[w.l + co(e)] = v[e];
    __syncthreads();
    RowStage<N>::store(lds, a.out, R0, w.nrows);
    return;
  }
  if (w.empty()) return;
  const RowBuf<N, float2> out(a.out, w, false);
  if (a.add) {
#pragma unroll
    for (int e = 0; e < F::V; ++e) v[e] = cadd(v[e], out.load(co(e)));
  }
#pragma unroll
  for (int e = 0; e < F::V; ++e) out.store(v[e], co(e));
}

// rows_fanout: W_r = scale * F_x([labels == r] * in) for every reference r
// (T: arithmetic type of the transforms, float2 or double2)
template <int N, bool MAP, class T = float2>
__global__ __launch_bounds__(kRowThreads) void k_rows_fanout(KArgs a) {
  using F = LaneFft<N, T>;
  __shared__ T lds[kRowWaves * F::NB * F::STRIDE];
  __shared__ T twl[F::TW];
  const RowLane<N, T> w(a);
  T* line = lds + ((threadIdx.x >> 6) * F::NB + w.b) * F::STRIDE;
  T u[F::V];
  Labels<F::V> lab;
  {
    const RowBuf<N, T> in(a.in, w, false);
#pragma unroll
    for (int e = 0; e < F::V; ++e) u[e] = from_f2<T>(in.load(F::first_c(e)));
    lab.load(a.labels + ((size_t)(model_iw<MAP>(a, w.iw) * a.NY + w.iy) * N + w.l),
             [](int e) { return F::first_c(e); });
  }
  row_twiddles<N>(twl, twx_of(a, (T*)nullptr));
  __syncthreads();
  if (w.empty()) return;
  const real_of<T> s = a.scale;
  const uint32_t wm = wave_row_mask<N, T, MAP>(a, w);
  int turn = (int)blockIdx.y;  // part blockIdx.y takes every gridDim.y-th of the wave's references
  for (int r = 0; r < a.nref; ++r) {
    if (r < 32 && !((wm >> r) & 1u)) continue;  // rows without reference r: the column pass reads zeros
    if (turn-- != 0) continue;
    turn = (int)gridDim.y - 1;
    T x[F::V];
#pragma unroll
    for (int e = 0; e < F::V; ++e) x[e] = (lab.at(e) == r) ? u[e] : cz<T>();
    F::template run<false>(x, line, twl, w.l);
    const RowBuf<N, T> W(a.W + (size_t)r * a.wstride, w, a.quad != 0);
#pragma unroll
    for (int e = 0; e < F::V; ++e) W.store(to_f2(cscale(x[e], s)), F::last_c(e));
  }
}

// rows_select: out = (add ? out : 0) + sum_r [labels == r] * scale * F_x^-1(W_r)
// KNEXT: also K = scale * F_x(taper * out) (quad-block), the first row pass of
// a next step that propagates out further: one transform more here instead of
// a pass that reads out back.
// G: waves that share the rows of one, each taking every G-th of their
// references (launches that leave the chip idle, term_split).
template <int N, bool MAP, bool KNEXT = false, int G = 1>
__global__ __launch_bounds__(kRowThreads) void k_rows_select(KArgs a) {
  using F = LaneFft<N>;
  __shared__ float2 lds[kRowWaves * F::NB * F::STRIDE];
  __shared__ float2 twl[F::TW];
  static_assert(kRowWaves % G == 0, "a workgroup holds whole groups");
  const RowLane<N, float2> w(a, G);
  const int g = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6) % G);
  float2* line = lds + ((threadIdx.x >> 6) * F::NB + w.b) * F::STRIDE;
  Labels<F::V> lab;
  float2 acc[F::V];
  lab.load(a.labels + ((size_t)(model_iw<MAP>(a, w.iw) * a.NY + w.iy) * N + w.l),
           [](int e) { return F::first_c(e); });
#pragma unroll
  for (int e = 0; e < F::V; ++e) acc[e] = czero();
  // references present in this wave's rows (wave-uniform)
  const uint32_t wm = wave_row_mask<N, float2, MAP>(a, w);
  const uint32_t live = a.nref >= 32 ? wm : (wm & ((1u << a.nref) - 1u));
  float2 nxt[F::V];
  auto fetch = [&](int r) {
    const RowBuf<N, float2> W(a.W + (size_t)r * a.wstride, w, a.quad != 0);
#pragma unroll
    for (int e = 0; e < F::V; ++e) nxt[e] = W.load(F::last_c(e));
  };
  // absent references contribute nothing to these rows: skip their loads and
  // transforms.  The next reference's row is fetched into registers during
  // this one's transform, except at 16 values per lane or more, where holding
  // it would cost a wave of occupancy
  constexpr bool PREFETCH = F::V < 16;
  const int rend = w.empty() ? 0 : a.rowmask ? 32 : a.nref;
  auto after = [&](int r, int k) {  // the k-th reference after r, rend or more when there is none
    for (int i = 0; i < k && r < rend; ++i) r = a.rowmask ? next_bit(live, r) : r + 1;
    return r;
  };
  int r = after(a.rowmask ? next_bit(live, -1) : 0, g);
  if (r < rend) fetch(r);
  row_twiddles<N>(twl, a.twx);
  __syncthreads();
  if (G == 1 && w.empty()) return;
  while (r < rend) {
    float2 x[F::V];
#pragma unroll
    for (int e = 0; e < F::V; ++e) x[e] = nxt[e];
    const int rn = after(r, G);
    if (PREFETCH && rn < rend) fetch(rn);
    F::template run<true>(x, line, twl, w.l);
    if (!PREFETCH && rn < rend) fetch(rn);
    // every node has one label, so its sum over the references is one term
#pragma unroll
    for (int e = 0; e < F::V; ++e)
      if (lab.at(e) == r) acc[e] = x[e];
    r = rn;
  }
  if constexpr (G > 1) {  // the first wave of a group gathers the nodes of the others (each node has one owner)
    wave_sync();
#pragma unroll
    for (int e = 0; e < F::V; ++e)
      if (g > 0) line[w.l + F::first_c(e)] = acc[e];
    __syncthreads();
    if (g > 0 || w.empty()) return;
#pragma unroll
    for (int h = 1; h < G; ++h)
#pragma unroll
      for (int e = 0; e < F::V; ++e) acc[e] = cadd(acc[e], line[h * F::NB * F::STRIDE + w.l + F::first_c(e)]);
    wave_sync();
  }
  const float s = a.scale;
  const RowBuf<N, float2> out(a.out, w, false);
#pragma unroll
  for (int e = 0; e < F::V; ++e) acc[e] = cscale(acc[e], s);
  if (a.add) {
#pragma unroll
    for (int e = 0; e < F::V; ++e) acc[e] = cadd(acc[e], out.load(F::first_c(e)));
  }
  if (!KNEXT || a.knext != 2) {
#pragma unroll
    for (int e = 0; e < F::V; ++e) out.store(acc[e], F::first_c(e));
  }
  if constexpr (KNEXT) {
    const float ty = a.tapy[w.iy];
    const float* tx = a.tapx + w.l;
#pragma unroll
    for (int e = 0; e < F::V; ++e) acc[e] = cscale(acc[e], tx[F::first_c(e)] * ty);
    F::template run<false>(acc, line, twl, w.l);
    const RowBuf<N, float2> K(a.K, w, a.quad != 0);
#pragma unroll
    for (int e = 0; e < F::V; ++e) K.store(cscale(acc[e], s), F::last_c(e));
  }
}

// ------------------------------------------------------------------ presence masks
// Presence masks of reference labels: bit r of rowmask[row] is set when
// label r occurs in that (w, y) row; planemask is the OR over a plane's rows.
__global__ __launch_bounds__(kThreads) void k_presence(const uint8_t* __restrict__ labels, uint32_t* rowmask,
                                                       int NX, long long nrows) {
  const long long row = (long long)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= nrows) return;
  uint32_t m = 0;
  for (int x = lane; x < NX; x += 64) {
    const int l = labels[row * NX + x];
    if (l < 32) m |= 1u << l;
  }
  for (int off = 32; off > 0; off >>= 1) m |= (uint32_t)__shfl_xor((int)m, off);
  if (lane == 0) rowmask[row] = m;
}
__global__ __launch_bounds__(kThreads) void k_planemask(const uint32_t* __restrict__ rowmask, uint32_t* planemask,
                                                        int NY, long long nplanes) {
  const long long p = (long long)blockIdx.x * kThreads + threadIdx.x;
  if (p >= nplanes) return;
  uint32_t m = 0;
  for (int y = 0; y < NY; ++y) m |= rowmask[p * NY + y];
  planemask[p] = m;
}
// number of present (row, reference) pairs of every plane
__global__ __launch_bounds__(kThreads) void k_present_count(const uint32_t* __restrict__ rowmask, int* cnt, int NY,
                                                            long long nplanes, uint32_t refs) {
  const long long p = (long long)blockIdx.x * kThreads + threadIdx.x;
  if (p >= nplanes) return;
  int c = 0;
  for (int y = 0; y < NY; ++y) c += __builtin_popcount(rowmask[p * NY + y] & refs);
  cnt[p] = c;
}
hipError_t launch_present_count(const uint32_t* rowmask, int* cnt, int NY, long long nplanes, int nref,
                                hipStream_t st) {
  const uint32_t refs = nref >= 32 ? 0xffffffffu : ((1u << nref) - 1u);
  hipLaunchKernelGGL(k_present_count, dim3((unsigned)((nplanes + kThreads - 1) / kThreads)), dim3(kThreads), 0, st,
                     rowmask, cnt, NY, nplanes, refs);
  return hipGetLastError();
}

hipError_t launch_presence(const uint8_t* labels, uint32_t* rowmask, uint32_t* planemask, int NX, int NY,
                           long long nplanes, hipStream_t st) {
  const long long nrows = nplanes * NY;
  hipLaunchKernelGGL(k_presence, dim3((unsigned)((nrows + kThreads / 64 - 1) / (kThreads / 64))), dim3(kThreads), 0, st, labels,
                     rowmask, NX, nrows);
  hipLaunchKernelGGL(k_planemask, dim3((unsigned)((nplanes + kThreads - 1) / kThreads)), dim3(kThreads), 0, st,
                     rowmask, planemask, NY, nplanes);
  return hipGetLastError();
}

// ------------------------------------------------------------------ launchers
// kind: 0 plain forward, 1 plain inverse, 2 forward with pre-taper,
//       3 inverse with post-taper
hipError_t launch_rows(int kind, const KArgs& a, hipStream_t st) {
  return dispatch_n(a.NX, [&](auto nc) -> hipError_t {
    constexpr int N = decltype(nc)::value;
    const dim3 g = row_grid<N, float2>(a.np * a.NY);
    switch (kind) {
      case 0: hipLaunchKernelGGL((k_rows<N, false, false, false>), g, dim3(kRowThreads), 0, st, a); break;
      case 1: hipLaunchKernelGGL((k_rows<N, true, false, false>), g, dim3(kRowThreads), 0, st, a); break;
      case 2: hipLaunchKernelGGL((k_rows<N, false, true, false>), g, dim3(kRowThreads), 0, st, a); break;
      case 3: hipLaunchKernelGGL((k_rows<N, true, false, true>), g, dim3(kRowThreads), 0, st, a); break;
      default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
  });
}

hipError_t launch_rows_fanout(const KArgs& a, hipStream_t st) {
  return dispatch_n(a.NX, [&](auto nc) -> hipError_t {
    constexpr int N = decltype(nc)::value;
    auto go = [&](auto map, auto t) {
      using T = decltype(t);
      dim3 g = row_grid<N, T>(a.np * a.NY);
      g.y = term_split(row_waves<N, T>(a.np * a.NY), live_refs(a), 4, 2048);
      hipLaunchKernelGGL((k_rows_fanout<N, decltype(map)::value, T>), g, dim3(kRowThreads), 0, st, a);
      return hipGetLastError();
    };
    if (a.f64) return a.mplane ? go(std::true_type{}, double2{}) : go(std::false_type{}, double2{});
    return a.mplane ? go(std::true_type{}, float2{}) : go(std::false_type{}, float2{});
  });
}

hipError_t launch_rows_select(const KArgs& a, hipStream_t st) {
  return dispatch_n(a.NX, [&](auto nc) -> hipError_t {
    constexpr int N = decltype(nc)::value;
    auto go = [&](auto map, auto knext) {
      constexpr bool M = decltype(map)::value, K = decltype(knext)::value;
      const int nrows = a.np * a.NY;
      const bool split = term_split(row_waves<N, float2>(nrows), live_refs(a), kRowWaves, 1024) > 1;
      const dim3 g = row_grid<N, float2>(nrows, split ? kRowWaves : 1);
      if (split) hipLaunchKernelGGL((k_rows_select<N, M, K, kRowWaves>), g, dim3(kRowThreads), 0, st, a);
      else hipLaunchKernelGGL((k_rows_select<N, M, K>), g, dim3(kRowThreads), 0, st, a);
      return hipGetLastError();
    };
    if (a.knext) return a.mplane ? go(std::true_type{}, std::true_type{}) : go(std::false_type{}, std::true_type{});
    return a.mplane ? go(std::true_type{}, std::false_type{}) : go(std::false_type{}, std::false_type{});
  });
}

}  // namespace fwix
