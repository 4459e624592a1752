// cols_fanout: W_r = F_y^-1[M_r * F_y(K)] / NY for every term r.
//
// The spectrum of a column tile stays in registers and every term present in
// the plane is one multiplication and one inverse transform from it, its
// multiplier M_r (TermMult<MODE>) evaluated on the fly.
#include "col_kernels.h"

namespace fwix {

// (T: arithmetic type of the transforms, float2 or double2)
template <int N, int MODE, int WPE, class T, int CWX>
__global__ __launch_bounds__((TileFft<N, T, CWX>::THREADS)) __attribute__((amdgpu_waves_per_eu(WPE))) void k_cols_fanout(KArgs a) {
  using F = TileFft<N, T, CWX>;
  using S = real_of<T>;
  __shared__ __align__(16) T region[F::SMEM];
  __shared__ __align__(16) T twl[F::TW];
  __shared__ uint32_t rmk[N];
  const F f(region, twl);
  int p, c0;
  col_tile<F>(p, c0);
  const size_t pb = (size_t)p * a.NX * N;
  const int iw = plane_iw(a, p);
  const int im = model_iw_any(a, iw);
  const uint32_t* rm = (MODE != 2 && a.rowmask) ? a.rowmask + im * a.NY : nullptr;
  const uint32_t pm = (MODE != 2 && a.planemask) ? a.planemask[im] : 0xffffffffu;
  const ColOffs<F, true> o(f, c0, a.NX, a.quad != 0);
  T spec[F::V];
  {
    const PlaneBuf K(a.K + pb, plane_bytes(a));
#pragma unroll
    for (int e = 0; e < F::V; ++e) spec[e] = from_f2<T>(K.load(o.voff(e), o.soff(e)));
  }
  col_twiddles<F>(twl, twy_of(a, (T*)nullptr));
  col_row_masks<F, N>(rmk, rm);
  constexpr bool HELD = sizeof(S) == 4;
  __shared__ float kyl[HELD ? 1 : N];
  const ColumnK2<F, N, S, HELD> k2(f, a, c0, kyl);
  F::sync();
  f.forward(spec);
  const S w2 = a.w2[iw];
  const S s2 = a.scale;  // 1/NY: forward and inverse column normalisation together
#pragma unroll
  for (int e = 0; e < F::V; ++e) spec[e] = cscale(spec[e], s2);
  // part blockIdx.z takes every gridDim.z-th of the plane's terms
  int turn = (int)blockIdx.z;
  for (int r = 0; r < a.nterm; ++r) {
    if (r < 32 && !((pm >> r) & 1u)) continue;  // reference absent from the plane: W_r is never read
    if (turn-- != 0) continue;
    turn = (int)gridDim.z - 1;
    const TermMult<MODE, T> tm(a, r, iw, w2);
    T x[F::V];
    auto mult = [&](auto real) {
#pragma unroll
      for (int e = 0; e < F::V; ++e) x[e] = tm.template apply<decltype(real)::value, false>(spec[e], k2.at(e), spec[e]);
    };
    if (tm.real) mult(std::true_type{});
    else mult(std::false_type{});
    f.inverse(x);
    const PlaneBuf W(a.W + (size_t)r * a.wstride + pb, plane_bytes(a));
    if (rm && r < 32) {
      // only the rows where the reference is present are read later
#pragma unroll
      for (int e = 0; e < F::V; ++e)
        W.store(to_f2(x[e]), off_if(rmk[f.l0 + F::first_c(e)], r, o.voff(e)), o.soff(e));
    } else {
#pragma unroll
      for (int e = 0; e < F::V; ++e) W.store(to_f2(x[e]), o.voff(e), o.soff(e));
    }
  }
}

template <int N, int MODE, int WPE, class T, int CWX, int G>
struct FanOut {
  static constexpr auto kernel = &k_cols_fanout<N, MODE, WPE, T, CWX>;
};
hipError_t launch_cols_fanout(int mode, const KArgs& a, hipStream_t st) {
  return launch_col_terms<FanOut, false>(0, mode, a, st);
}

}  // namespace fwix
