// Shared kernel argument block, tile geometry and per-point physics for the
// PSPI / NSPS / Born depth-step kernels.
#pragma once
#include "fwix_fft.h"

namespace fwix {

// Supported lateral FFT sizes: 2^a and 3*2^a between 8 and 1024.
constexpr bool size_has3(int N) { return N % 3 == 0; }

// Row passes: workgroups of 4 waves, each with LaneFft::NB rows (64 / NB lanes a
// row).  (8 waves to share one twiddle table at 1024 points, 16 waves per CU
// instead of 12, cap the registers at 128: the chained select pass spills and
// takes 1298 instead of 824 us per 128-plane launch.)
constexpr int kRowWaves = 4;
constexpr int kRowThreads = 64 * kRowWaves;
// Default register budget (waves per SIMD) of the column kernels, from timed
// launches of every budget on MI355X: kind 0 the fan-out transforms, kind 1
// the fan-in transforms; mode 2 the scattering terms.  (Every mode of a kind
// has the same winners so far; mode stays in the key.)  The fan-out needs at most
// 93 registers (118 at 1024 points) and is the same code at every budget but
// for its schedule (within 3 %).  The fan-in fits 4 waves at V = 8 (16 M points,
// 512: 235 us at 2, 215 at 4, 210 to 275 at 6, which spills) and, with k^2 formed
// from LDS, at V = 12, where the budgets are within 4 % (192: 130 / 130 / 129 us,
// 384: 219 at 2 and 4, 222 at 6, 768: 256 / 252 / 249; Taylor terms at 768: 112 / 83 / 112).
constexpr int col_wpe_default(int kind, int mode, int N) {
  const bool pow2 = !size_has3(N);
  (void)mode;
  if (kind == 0) return N == 1024 ? 2 : pow2 ? 6 : 4;
  return (pow2 && N <= 512) || N == 768 ? 4 : 2;
}
// The budget that a kernel is built for when `wpe` is asked for: where
// budgets give the same instructions there is one kernel.  At 1024 points that is every budget
// (LDS decides the waves), in the fan-in at 384 points 2 is 4.
constexpr int col_wpe_built(int kind, int N, int wpe) {
  return N == 1024 ? 2 : kind == 1 && N == 384 && wpe == 2 ? 4 : wpe;
}
constexpr int kThreads = 256;

// One argument block for every step kernel (passed by value).
struct KArgs {
  const float2* in;        // input wavefield, already offset to the chunk's first plane
  float2* out;             // output wavefield, same offset
  float2* K;               // chunk spectrum scratch (np planes)
  float2* W;               // per-reference / per-Taylor-term scratch (nterm * np planes)
  const uint8_t* labels;   // (NW, NY, NX) reference labels of the current depth
  const uint32_t* rowmask; // (NW, NY) bit r set: reference r labels a node of that row (null: all)
  const uint32_t* planemask; // (NW) OR of rowmask over the plane's rows (null: all)
  const float2* sref;      // (nref, NW) reference slownesses of the current depth
  const int* mplane;       // (NW) model plane of every plane (null: the plane itself)
  const float* kx;         // (NX) wavenumbers
  const float* ky;         // (NY)
  const float* w2;         // (NW) (2 pi f)^2
  const float* w;          // (NW) 2 pi f
  const float* tapx;       // (NX) taper weights
  const float* tapy;       // (NY)
  const float2* twx;       // (NX) stage twiddles of the row transforms (twiddle_exp)
  const float2* twy;       // (NY) stage twiddles of the column transforms
  const double2* twx64;    // the same tables and taper weights in float64, for the
  const double2* twy64;    //   passes that run in float64 arithmetic (f64)
  const double* tapx64;
  const double* tapy64;
  const float2* slow;      // (NW, ny, nx) unpadded slowness slice (Born scatter)
  const float2* dslow;     // (NW, ny, nx) model perturbation slice (Born IC)
  const float2* bg;        // background wavefield slice, chunk offset (Born IC)
  const float2* addin;     // extra wavefield added before the taper (Born: dU_z)
  float2* aux;             // extra output (checkpoint copy / image)
  int NX, NY, NW, NS, nx, ny;
  int nref, nterm;
  int live;                // most references present in a plane of the launch (0: unknown)
  int p0, np;              // chunk: first global plane, number of planes
  long long wstride;       // elements between consecutive W terms (np*NX*NY)
  float dz, eps, eps_s;
  float scale;             // normalisation applied by the kernel (set per launch)
  int add;
  int f64;                 // the launch runs its transforms in float64 arithmetic
  int qin, qout;           // k_rows: in / out are K (in the scratch layout below)
  int quad;                // K and W in the quad-block layout (else row-major)
  int knext;               // k_rows_select: also K = scale * F_x(taper * out), the next step's spectrum
                           //   (2: K only, out itself is not needed)
};

// Quad-block layout of the column-pass scratch (K and the W terms, where the
// launch's a.quad says so; row-major otherwise): a 128-byte
// line holds a 4 x 4 block (rows 4q..4q+3 x columns 4p..4p+3, row-major inside),
// blocks row-major.  A column tile of 4 or 8 columns then loads and stores
// whole lines, and the 4 rows of a row-pass workgroup share every line they
// touch.  y counts rows over all planes of the chunk (NY is a multiple of 4).
__device__ __forceinline__ unsigned qidx(int y, int x, int NX) {
  return (unsigned)(((((y >> 2) * (NX >> 2)) + (x >> 2)) << 4) + ((y & 3) << 2) + (x & 3));
}

// twiddle tables of the arithmetic type T (float2 or double2)
__device__ __forceinline__ const float2* twx_of(const KArgs& a, float2*) { return a.twx; }
__device__ __forceinline__ const double2* twx_of(const KArgs& a, double2*) { return a.twx64; }
__device__ __forceinline__ const float2* twy_of(const KArgs& a, float2*) { return a.twy; }
__device__ __forceinline__ const double2* twy_of(const KArgs& a, double2*) { return a.twy64; }

__device__ __forceinline__ int plane_iw(const KArgs& a, int p_local) { return (a.p0 + p_local) % a.NW; }
// Index into the model-sized arrays (labels, presence masks, slowness, model
// perturbation): plane iw itself, or the shot it belongs to when planes of
// several shots share one launch.
// MAP is a template flag so that the per-element index of the unbatched
// kernels carries no branch (a per-element test of a.mplane split the
// unrolled loads into separate blocks and cost the row passes 7-17 %).
template <bool MAP>
__device__ __forceinline__ int model_iw(const KArgs& a, int iw) {
  if constexpr (MAP) return a.mplane[iw];
  else return iw;
}
// once-per-workgroup form (column kernels)
__device__ __forceinline__ int model_iw_any(const KArgs& a, int iw) { return a.mplane ? a.mplane[iw] : iw; }

// The rows of one wave of a row pass, as one lane sees them: row rb + b of the
// chunk, at lane l of its LaneFft::L lanes.  Rows at or beyond nrows (the last
// wave's) are computed on zeros and never stored.
template <int N, class T>
struct RowLane {
  using F = LaneFft<N, T>;
  int l, b, rb, nrows;
  bool live;
  int iw, iy;  // frequency plane and row of the plane (of the last row for dead lanes)
  // groups: this many consecutive waves share the rows of one
  __device__ __forceinline__ explicit RowLane(const KArgs& a, int groups = 1) {
    const int lane = (int)threadIdx.x & 63;
    l = (int)((unsigned)lane % F::L);
    b = (int)((unsigned)lane / F::L);
    nrows = a.np * a.NY;
    rb = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * kRowWaves + (threadIdx.x >> 6)) / groups * F::NB));
    const int lr = rb + b;
    live = lr < nrows;
    const int row = live ? lr : nrows - 1;
    const int p = row / a.NY;
    iy = row - p * a.NY;
    iw = plane_iw(a, p);
  }
  // no row at all (wave-uniform): such a wave must not store
  __device__ __forceinline__ bool empty() const { return rb >= nrows; }
};
// The wave's rows of a wavefield (row-major) or of the K / W scratch (in the
// launch's layout) as a buffer resource: a lane's elements sit at one 32-bit
// lane offset plus a uniform offset per element, so they cost no address
// arithmetic, and the hardware range check reads zero / drops stores of
// rows beyond the last.  The check counts on a wave with at least one row: the
// lane offset of a row beyond the last is then past the resource whether or not
// the uniform offset (less than a row, or a quad of rows) is part of it.  A wave
// without rows gets the resource of the first rows, to load from and not to
// store to: one of no bytes based past the array would let accesses through if
// the check is lane offset >= size - uniform offset, which wraps.  (No branch
// around the loads instead: rows_fanout 73.5 against 78.2 us, 768^2 x 24 planes.)
template <int N, class T>
struct RowBuf {
  using F = LaneFft<N, T>;
  __amdgpu_buffer_rsrc_t r;
  unsigned v, row;
  int cs, l;
  __device__ __forceinline__ RowBuf(const float2* base, const RowLane<N, T>& w, bool quad) : l(w.l) {
    const int rb = w.empty() ? 0 : w.rb, r0 = quad ? rb & ~3 : rb;
    const int left = w.nrows - r0, most = F::NB + 4;
    const int rows = left < most ? left : most;
    r = __builtin_amdgcn_make_buffer_rsrc((void*)(base + (size_t)r0 * N), (short)0,
                                          __builtin_amdgcn_readfirstlane(rows * N * 8), 0x00020000);
    const unsigned y = (unsigned)(rb - r0 + w.b);
    row = quad ? ((y >> 2) * N + (y & 3)) * 32u : y * N * 8u;
    v = row + (quad ? (((unsigned)l >> 2) << 4) + ((unsigned)l & 3u) : (unsigned)l) * 8u;
    cs = quad ? 32 : 8;
  }
  // column l + C (C a compile-time constant after unrolling)
  __device__ __forceinline__ unsigned voff(int C) const {
    if constexpr (F::L % 4 == 0) return v;
    const unsigned x = (unsigned)(l + C);
    return cs == 32 ? row + (((x >> 2) << 4) + (x & 3u)) * 8u : row + x * 8u;
  }
  __device__ __forceinline__ int soff(int C) const { return F::L % 4 == 0 ? C * cs : 0; }
  __device__ __forceinline__ float2 load(int C) const {
    return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff(C), soff(C), 0));
  }
  // where the lane's condition holds, else zero without touching memory: every
  // element's load is in flight at once, which a branch around each would forbid
  __device__ __forceinline__ float2 load_if(bool on, int C) const {
    return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, on ? (int)voff(C) : (int)0x80000000u, soff(C), 0));
  }
  __device__ __forceinline__ void store(float2 x, int C) const {
    using U2 = __attribute__((ext_vector_type(2))) unsigned;
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, x), r, (int)voff(C), soff(C), 0);
  }
};
// x[e] = f(e) for the elements of a lane, in groups: a group's loads are in
// flight together, and its results are formed before the next group's loads
// are issued, which bounds the registers that loads of several arrays take at
// once (left alone the compiler issues every element's loads first).
// A group holds the elements at positions from r0 N / R(0) on (first_c order),
// and groups that start at or beyond column `cols` are skipped: nothing of
// theirs is needed (the padding of an imaging or scattering source).
__device__ __forceinline__ void pin(float2& x) { asm volatile("" : "+v"(x.x), "+v"(x.y) : : "memory"); }
__device__ __forceinline__ void pin(double2& x) { asm volatile("" : "+v"(x.x), "+v"(x.y) : : "memory"); }
template <class F, class T, class Fn>
__device__ __forceinline__ void in_groups(T* x, int cols, Fn&& f) {
  constexpr int R = F::R(0), Q = F::V / R, most = sizeof(T) == 16 || F::V == 16 ? 4 : 8;
  constexpr int G = Q >= most ? 1 : most / Q < R ? most / Q : R;  // butterfly inputs per group
#pragma unroll
  for (int r0 = 0; r0 < R; r0 += G) {
    if (r0 * (F::L * Q) < cols) {
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int r = r0; r < (r0 + G < R ? r0 + G : R); ++r) x[q * R + r] = f(q * R + r);
    }
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int r = r0; r < (r0 + G < R ? r0 + G : R); ++r) pin(x[q * R + r]);
  }
}
// labels of a lane's elements, four to a register
template <int V>
struct Labels {
  uint32_t w[(V + 3) / 4];
  template <class Pos>
  __device__ __forceinline__ void load(const uint8_t* __restrict__ p, Pos&& pos) {
#pragma unroll
    for (int k = 0; k < (V + 3) / 4; ++k) w[k] = 0;
#pragma unroll
    for (int e = 0; e < V; ++e) w[e / 4] |= (uint32_t)p[pos(e)] << (8 * (e % 4));
  }
  __device__ __forceinline__ int at(int e) const { return (int)((w[e / 4] >> (8 * (e % 4))) & 255u); }
};
// this workgroup's copy of the row transforms' twiddle table; the caller
// synchronises.  In LDS because a global load inside the term loops would
// wait (one counter for all vector memory operations) for the term's
// stores or the next term's loads still in flight.
template <int N, class T>
__device__ __forceinline__ void row_twiddles(T* twl, const T* __restrict__ tw) {
  for (int i = threadIdx.x; i < LaneFft<N, T>::TW; i += kRowThreads) twl[i] = tw[i];
}
// references present in any row of this wave (all bits when there are no masks)
template <int N, class T, bool MAP>
__device__ __forceinline__ uint32_t wave_row_mask(const KArgs& a, const RowLane<N, T>& w) {
  if (!a.rowmask) return 0xffffffffu;
  uint32_t m = a.rowmask[model_iw<MAP>(a, w.iw) * a.NY + w.iy];
#pragma unroll
  for (int o = LaneFft<N, T>::L; o < 64; o <<= 1) m |= (uint32_t)__shfl_xor((int)m, o);
  return __builtin_amdgcn_readfirstlane(m);
}

// lowest set bit of m above position r (32 when none); r = -1 gives the lowest
__device__ __forceinline__ int next_bit(uint32_t m, int r) {
  const uint32_t rest = r >= 31 ? 0u : (m & ~((2u << r) - 1u));
  return rest ? __builtin_ctz(rest) : 32;
}

// sin and cos of x (radians) from the transcendental unit: v_sin_f32 /
// v_cos_f32 take revolutions, so x is scaled by 1/(2 pi) and reduced to
// [0, 1) with v_fract_f32.  Measured on gfx950 over [-2, 2) revolutions:
// |error| <= 1.3e-7 against double-precision sin / cos, float rounding level
// for the phases of a depth step (|kz dz| well below one revolution).
__device__ __forceinline__ void fast_sincos(float x, float* s, float* c) {
  const float r = __builtin_amdgcn_fractf(x * 0.159154943091895336f);
  *s = __builtin_amdgcn_sinf(r);
  *c = __builtin_amdgcn_cosf(r);
}

// Phase-shift multiplier exp(-i kz dz) for one reference slowness.
// Reference formula (propagator/src/phase_shift.cu:36-59): a = w2 Re s - k^2,
// b = w2 (Im s - eps Re s), kr = sqrt((c+a)/2), ki = sqrt((c-a)/2),
// c = sqrt(a^2+b^2).  Evaluated as the numerically stable complex square
// root (the smaller of kr, ki from kr*ki = |b|/2): identical in exact
// arithmetic, free of the float32 cancellation in c-a / c+a.
// MODE 0: forward  exp(-ki dz) exp(-i kr dz)
// MODE 1: adjoint  kr -> -kr if b > 0; exp(-ki dz) exp(+i kr dz)
// MODE 2: inverse  kr -> -kr if b > 0; exp(+ki dz) exp(+i kr dz)
// b depends only on (frequency, reference): callers test b == 0 once and
// use ps_real (kz real or purely imaginary) for the whole plane.
template <int MODE>
__device__ __forceinline__ float2 ps_real(float a, float dz) {
  const float t = __builtin_amdgcn_sqrtf(fabsf(a)) * dz;
  float sn, cs;
  fast_sincos(t, &sn, &cs);
  const float e = __expf(MODE == 2 ? t : -t);
  if (a >= 0.f) return MODE == 0 ? make_float2(cs, -sn) : make_float2(cs, sn);
  return make_float2(e, 0.f);
}
template <int MODE>
__device__ __forceinline__ float2 ps_general(float a, float b, float dz) {
  const float c = __builtin_amdgcn_sqrtf(fmaf(a, a, b * b));
  const float big = __builtin_amdgcn_sqrtf(0.5f * (c + fabsf(a)));
  const float small = 0.5f * fabsf(b) * __builtin_amdgcn_rcpf(big);
  float kr = a >= 0.f ? big : small;
  const float ki = a >= 0.f ? small : big;
  if (MODE != 0 && b > 0.f) kr = -kr;
  const float att = __expf((MODE == 2 ? ki : -ki) * dz);
  float sn, cs;
  fast_sincos(kr * dz, &sn, &cs);
  return MODE == 0 ? make_float2(att * cs, -att * sn) : make_float2(att * cs, att * sn);
}
// The same multipliers in float64 arithmetic (the float64 scattering passes:
// near the evanescent boundary a = w2 Re s - k^2 cancels, and a float32
// phase there is the largest error left once the transforms run in float64).
// sincospi of the phase in half turns: sincos reduces an argument of any size,
// which costs the column kernels registers they spill (768^2 x 6 planes fan-in:
// 117 registers spilled, 0.6 GB of scratch traffic, against 16).
constexpr double kInvPi = 0.31830988618379067154;
template <int MODE>
__device__ __forceinline__ double2 ps_general64(double a, double b, double dz) {
  const double c = sqrt(fma(a, a, b * b));
  const double big = sqrt(0.5 * (c + fabs(a)));
  const double small = 0.5 * fabs(b) / big;
  double kr = a >= 0.0 ? big : small;
  const double ki = a >= 0.0 ? small : big;
  if (MODE != 0 && b > 0.0) kr = -kr;
  const double att = exp((MODE == 2 ? ki : -ki) * dz);
  double sn, cs;
  sincospi(kr * (dz * kInvPi), &sn, &cs);
  return MODE == 0 ? make_double2(att * cs, -att * sn) : make_double2(att * cs, att * sn);
}

template <int MODE>
__device__ __forceinline__ float2 ps_mult(float w2, float sre, float sim, float k2, float dz, float eps) {
  const float a = fmaf(w2, sre, -k2);
  const float b = w2 * (sim - eps * sre);
  return b == 0.f ? ps_real<MODE>(a, dz) : ps_general<MODE>(a, b, dz);
}

}  // namespace fwix
