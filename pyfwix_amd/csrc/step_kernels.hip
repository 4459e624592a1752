// Fused one-way depth-step kernels: three passes per PSPI / NSPS step.
//
//   PSPI forward   (propagator/src/PSPI.cpp:6-24, :66-83)
//     rows_fwd(pre-taper)  ->  cols_fanout(Phi_r)  ->  rows_select
//   PSPI adjoint   (PSPI.cpp:85-103)
//     rows_fanout(mask)    ->  cols_fanin(Phi_r^adj) -> rows_inv(post-taper)
//   NSPS forward   (propagator/src/NSPS.cpp:27-45)
//     rows_fanout(mask)    ->  cols_fanin(Phi_r)    -> rows_inv
//   NSPS adjoint   (corrected; NSPS.cpp:6-25 passes swapped arguments)
//     rows_fwd             ->  cols_fanout(Phi_r^adj) -> rows_select
//
// Row passes: row_kernels.hip.  Column passes: cols_fanout.hip and
// cols_fanin.hip (the fan-out keeps the spectrum of a column tile in registers and
// runs all nref inverse transforms from it; the fan-in accumulates all nref
// spectra in registers before a single inverse transform); here the plain
// column transform and the tables that choose among the column kernels.
#include "col_kernels.h"

namespace fwix {

// out = (add ? out : 0) + scale * F_y(in) on each plane (plain 2-D FFT column pass)
template <int N, bool INV>
__global__ __launch_bounds__((TileFft<N, float2, 8>::THREADS)) __attribute__((amdgpu_waves_per_eu(N == 1024 ? 2 : 4))) void k_cols(KArgs a) {
  using F = TileFft<N, float2, 8>;
  __shared__ __align__(16) float2 region[F::SMEM];
  // one transform, no loop: the twiddles come straight from memory (L1)
  const F f(region, a.twy);
  int p, c0;
  col_tile<F>(p, c0);
  const size_t pb = (size_t)p * a.NX * N;
  const ColOffs<F, !INV> oi(f, c0, a.NX, false);
  const ColOffs<F, INV> oo(f, c0, a.NX, false);
  float2 v[F::V];
  {
    const PlaneBuf in(a.in + pb, plane_bytes(a));
#pragma unroll
    for (int e = 0; e < F::V; ++e) v[e] = in.load(oi.voff(e), oi.soff(e));
  }
  if constexpr (INV) f.inverse(v);
  else f.forward(v);
  const float s = a.scale;  // column normalisation 1/sqrt(NY)
#pragma unroll
  for (int e = 0; e < F::V; ++e) v[e] = cscale(v[e], s);
  const PlaneBuf out(a.out + pb, plane_bytes(a));
  if (a.add) {
#pragma unroll
    for (int e = 0; e < F::V; ++e) v[e] = cadd(v[e], out.load(oo.voff(e), oo.soff(e)));
  }
#pragma unroll
  for (int e = 0; e < F::V; ++e) out.store(v[e], oo.voff(e), oo.soff(e));
}

// ------------------------------------------------------------------ launchers
bool fft_size_supported(int n) {
  switch (n) {
#define CASE(S) case S:
    FWIX_SIZES(CASE)
#undef CASE
    return true;
    default: return false;
  }
}

hipError_t launch_cols(bool inv, const KArgs& a, hipStream_t st) {
  return dispatch_n(a.NY, [&](auto nc) -> hipError_t {
    constexpr int N = decltype(nc)::value;
    using F = TileFft<N, float2, 8>;
    if (inv) hipLaunchKernelGGL((k_cols<N, true>), col_grid<F>(a), dim3(F::THREADS), 0, st, a);
    else hipLaunchKernelGGL((k_cols<N, false>), col_grid<F>(a), dim3(F::THREADS), 0, st, a);
    return hipGetLastError();
  });
}

// ------------------------------------------------------------------ occupancy variants
// Every fan-out / fan-in column kernel is built for three register budgets:
// 2, 4 or 6 waves per SIMD (256, 128 or 80 VGPRs).  More waves hide more
// latency but may spill; which wins depends on the size and the transform,
// so the choice is a runtime table (kernel, mode, size) that an autotuner
// sets from timed launches; the defaults (col_wpe_default) are the winners
// of such timings.
static constexpr int kSizeList[] = {8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512, 768, 1024};
static constexpr int kNumSizes = sizeof(kSizeList) / sizeof(int);
static int size_slot(int n) {
  for (int i = 0; i < kNumSizes; ++i)
    if (kSizeList[i] == n) return i;
  return -1;
}
static int g_wpe[2][3][kNumSizes];
static bool g_wpe_ready = false;
static void wpe_init() {
  if (g_wpe_ready) return;
  for (int k = 0; k < 2; ++k)
    for (int m = 0; m < 3; ++m)
      for (int i = 0; i < kNumSizes; ++i) g_wpe[k][m][i] = col_wpe_default(k, m, kSizeList[i]);
  g_wpe_ready = true;
}
int col_wpe_get(int kind, int mode, int n) {
  const int i = size_slot(n);
  if (kind < 0 || kind > 1 || mode < 0 || mode > 2 || i < 0) return -1;
  wpe_init();
  return g_wpe[kind][mode][i];
}
// Layout of the 1024-point column transforms, per kind (0 fan-out, 1 fan-in)
// and mode: 0 tiles of 8 columns (512 threads), 1 tiles of 4 (256 threads).
static int g_layout[2][3] = {{1, 1, 1}, {1, 1, 1}};
// Layout of the K / W scratch per lateral size (the column length NY): 1
// quad-block, 0 row-major.  The quad-block layout pays where the column tiles
// are 4 columns wide (1024-point columns, whole lines instead of quarter
// lines); at 8 columns the row passes' partial-line accesses cost more than
// the column passes gain.
static int g_quad[16] = {};
static bool g_quad_init = false;
static void quad_init() {
  if (g_quad_init) return;
  g_quad[size_slot(1024)] = 1;
  g_quad_init = true;
}
int scratch_quad_get(int n) {
  const int i = size_slot(n);
  if (i < 0) return -1;
  quad_init();
  return g_quad[i];
}
int scratch_quad_set(int n, int quad) {
  const int i = size_slot(n);
  if (i < 0 || (quad != 0 && quad != 1)) return -1;
  quad_init();
  g_quad[i] = quad;
  return 0;
}
int col_layout_get(int kind, int mode, int n) {
  if (kind < 0 || kind > 1 || mode < 0 || mode > 2 || size_slot(n) < 0) return -1;
  return n == 1024 ? g_layout[kind][mode] : 0;
}
int col_layout_set(int kind, int mode, int n, int layout) {
  if (kind < 0 || kind > 1 || mode < 0 || mode > 2 || size_slot(n) < 0) return -1;
  if (layout != 0 && !(layout == 1 && n == 1024)) return -1;
  if (n == 1024) g_layout[kind][mode] = layout;
  return 0;
}
int col_wpe_set(int kind, int mode, int n, int wpe) {
  const int i = size_slot(n);
  if (kind < 0 || kind > 1 || mode < 0 || mode > 2 || i < 0) return -1;
  if (wpe != 2 && wpe != 4 && wpe != 6) return -1;
  wpe_init();
  g_wpe[kind][mode][i] = wpe;
  return 0;
}

}  // namespace fwix
