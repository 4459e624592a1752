// cols_fanin: K = F_y^-1[sum_r M_r * F_y(W_r)] / NY.
//
// Every term present in the plane is loaded (the rows where it is present),
// transformed and added to the spectrum of the tile in registers, times its
// multiplier M_r (TermMult<MODE>); one inverse transform ends the pass.
#include "col_kernels.h"

namespace fwix {

// Waves per SIMD the kernel is compiled for under a budget.  LDS admits 3 at
// 1024 points: 3 (166 registers) beats 2 for the phase-shift terms (1024^2 x 16
// planes, 202 against 214 us), not for the Taylor terms (75 against 73).  At 384
// points it admits 4, which the scheduler then has to aim at (219 against 227 us, Taylor terms 70
// against 78; col_wpe_built).
constexpr int fanin_waves(int n, int mode, int wpe, bool f64) {
  if (f64) return 2;
  if (n == 1024) return mode == 2 ? 2 : 3;
  return wpe;
}

// (T: arithmetic type of the transforms, float2 or double2; G: groups of
// threads that share a tile's terms, group g taking every G-th, their sums
// added in group order)
template <int N, int MODE, int WPE, class T, int CWX, int G>
__global__ __launch_bounds__((TileFft<N, T, CWX>::THREADS * G)) __attribute__((amdgpu_waves_per_eu(fanin_waves(N, MODE, WPE, sizeof(T) == 16)))) void k_cols_fanin(KArgs a) {
  using F = TileFft<N, T, CWX>;
  using S = real_of<T>;
  constexpr int SM = G > 1 && F::SMEM < N * F::CW ? N * F::CW : F::SMEM;
  __shared__ __align__(16) T regions[G * SM];
  __shared__ __align__(16) T twl[F::TW];
  __shared__ uint32_t rmk[N];
  const int g = G > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.y) : 0;
  T* region = regions + g * SM;
  const F f(region, twl);
  int p, c0;
  col_tile<F>(p, c0);
  const size_t pb = (size_t)p * a.NX * N;
  const ColOffs<F, true> o(f, c0, a.NX, a.quad != 0);
  const int iw = plane_iw(a, p);
  const int im = model_iw_any(a, iw);
  const uint32_t* rm = (MODE != 2 && a.rowmask) ? a.rowmask + im * a.NY : nullptr;
  const uint32_t pm = (MODE != 2 && a.planemask) ? a.planemask[im] : 0xffffffffu;
  const uint32_t live = a.nterm >= 32 ? pm : (pm & ((1u << a.nterm) - 1u));
  const bool masked = rm != nullptr;
  const int rend = masked ? 32 : a.nterm;
  col_twiddles<F>(twl, twy_of(a, (T*)nullptr));
  col_row_masks<F, N>(rmk, rm);
  constexpr bool HELD = sizeof(S) == 4 && F::V != 12;
  __shared__ float kyl[HELD ? 1 : N];
  const ColumnK2<F, N, S, HELD> k2(f, a, c0, kyl);
  const S w2 = a.w2[iw];
  if constexpr (G > 1) __syncthreads();
  else F::sync();
  // the next term's tile is fetched into registers during this term's
  // transform, as it is stored (float32)
  float2 nxt[F::V];
  auto fetch = [&](int r) {
    const PlaneBuf W(a.W + (size_t)r * a.wstride + pb, plane_bytes(a));
    if (masked) {
#pragma unroll
      for (int e = 0; e < F::V; ++e)
        nxt[e] = W.load(off_if(rmk[f.l0 + F::first_c(e)], r, o.voff(e)), o.soff(e));
    } else {
#pragma unroll
      for (int e = 0; e < F::V; ++e) nxt[e] = W.load(o.voff(e), o.soff(e));
    }
  };
  T acc[F::V];
#pragma unroll
  for (int e = 0; e < F::V; ++e) acc[e] = cz<T>();
  // the k-th term after r, rend or more when there is none
  auto after = [&](int r, int k) {
    for (int i = 0; i < k && r < rend; ++i) r = masked ? next_bit(live, r) : r + 1;
    return r;
  };
  int lead = masked ? next_bit(live, -1) : 0;  // group 0's term: the groups wait for each other, so all go as far
  int r = after(lead, g);
  if (r < rend) fetch(r);
  while (lead < rend) {
    lead = after(lead, G);
    if (G > 1 && F::ONE && r >= rend) break;  // no waits in a tile of one wave
    T x[F::V];
#pragma unroll
    for (int e = 0; e < F::V; ++e) x[e] = G > 1 && r >= rend ? cz<T>() : from_f2<T>(nxt[e]);
    const int rn = after(r, G);
    if (rn < rend) fetch(rn);
    f.forward(x);
    if (G == 1 || r < rend) {
      const TermMult<MODE, T> tm(a, r, iw, w2);
      auto mult = [&](auto real) {
#pragma unroll
        for (int e = 0; e < F::V; ++e) acc[e] = tm.template apply<decltype(real)::value, true>(x[e], k2.at(e), acc[e]);
      };
      if (tm.real) mult(std::true_type{});
      else mult(std::false_type{});
    }
    r = rn;
  }
  if constexpr (G > 1) {
    __syncthreads();
#pragma unroll
    for (int e = 0; e < F::V; ++e)
      if (g > 0) region[e * F::THREADS + threadIdx.x] = acc[e];
    __syncthreads();
    if (F::ONE && g > 0) return;
    // the other groups run along to the end for its waits
#pragma unroll
    for (int h = 1; h < G; ++h)
#pragma unroll
      for (int e = 0; e < F::V; ++e)
        if (g == 0) acc[e] = cadd(acc[e], regions[h * SM + e * F::THREADS + threadIdx.x]);
  }
  const S s2 = a.scale;
#pragma unroll
  for (int e = 0; e < F::V; ++e) acc[e] = cscale(acc[e], s2);
  f.inverse(acc);
  if (g > 0) return;
  const PlaneBuf K(a.K + pb, plane_bytes(a));
#pragma unroll
  for (int e = 0; e < F::V; ++e) K.store(to_f2(acc[e]), o.voff(e), o.soff(e));
}

template <int N, int MODE, int WPE, class T, int CWX, int G>
struct FanIn {
  static constexpr auto kernel = &k_cols_fanin<N, MODE, WPE, T, CWX, G>;
};
hipError_t launch_cols_fanin(int mode, const KArgs& a, hipStream_t st) {
  return launch_col_terms<FanIn, true>(1, mode, a, st);
}

}  // namespace fwix
