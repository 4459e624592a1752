// cols_fanin: K = F_y^-1[sum_r M_r * F_y(W_r)] / NY.
//
// Every term present in the plane is loaded (the rows where it is present),
// transformed and added to the spectrum of the tile in registers, times its
// multiplier M_r (TermMult<MODE>); one inverse transform ends the pass.
#include "col_kernels.h"

namespace fwix {

// (T: arithmetic type of the transforms, float2 or double2)
template <int N, int MODE, int WPE, class T, int CWX>
__global__ __launch_bounds__((TileFft<N, T, CWX>::THREADS)) __attribute__((amdgpu_waves_per_eu(WPE))) void k_cols_fanin(KArgs a) {
  using F = TileFft<N, T, CWX>;
  using S = real_of<T>;
  __shared__ __align__(16) T region[F::SMEM];
  __shared__ __align__(16) T twl[F::TW];
  __shared__ uint32_t rmk[N];
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
  S k2v[F::V];
  column_k2(k2v, f, a, c0);
  const S w2 = a.w2[iw];
  F::sync();
  // the next term's tile is fetched into registers during this term's
  // transform, as it is stored (float32)
  float2 nxt[F::V];
  auto fetch = [&](int r) {
    const PlaneBuf W(a.W + (size_t)r * a.wstride + pb, plane_bytes(a));
    if (masked) {
#pragma unroll
      for (int e = 0; e < F::V; ++e)
        nxt[e] = W.load((rmk[f.l0 + F::first_c(e)] >> r) & 1u ? o.voff(e) : kOff, o.soff(e));
    } else {
#pragma unroll
      for (int e = 0; e < F::V; ++e) nxt[e] = W.load(o.voff(e), o.soff(e));
    }
  };
  T acc[F::V];
#pragma unroll
  for (int e = 0; e < F::V; ++e) acc[e] = cz<T>();
  int r = masked ? next_bit(live, -1) : 0;
  if (r < rend) fetch(r);
  while (r < rend) {
    T x[F::V];
#pragma unroll
    for (int e = 0; e < F::V; ++e) x[e] = from_f2<T>(nxt[e]);
    const int rn = masked ? next_bit(live, r) : r + 1;
    if (rn < rend) fetch(rn);
    f.forward(x);
    const TermMult<MODE, T> tm(a, r, iw, w2);
    auto mult = [&](auto real) {
#pragma unroll
      for (int e = 0; e < F::V; ++e) acc[e] = cadd(acc[e], tm.template apply<decltype(real)::value>(x[e], k2v[e]));
    };
    if (tm.real) mult(std::true_type{});
    else mult(std::false_type{});
    r = rn;
  }
  const S s2 = a.scale;
#pragma unroll
  for (int e = 0; e < F::V; ++e) acc[e] = cscale(acc[e], s2);
  f.inverse(acc);
  const PlaneBuf K(a.K + pb, plane_bytes(a));
#pragma unroll
  for (int e = 0; e < F::V; ++e) K.store(to_f2(acc[e]), o.voff(e), o.soff(e));
}

template <int N, int MODE, int WPE, class T, int CWX>
struct FanIn {
  static constexpr auto kernel = &k_cols_fanin<N, MODE, WPE, T, CWX>;
};
hipError_t launch_cols_fanin(int mode, const KArgs& a, hipStream_t st) {
  return launch_col_terms<FanIn>(1, mode, a, st);
}

}  // namespace fwix
