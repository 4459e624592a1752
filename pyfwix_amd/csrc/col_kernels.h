// Column passes of the fused depth steps: the tile of a workgroup and its
// memory accesses, the spectral multipliers, and the launch geometry (kernels:
// cols_fanout.hip, cols_fanin.hip; the plain transform: step_kernels.hip).
//
// A workgroup transforms CW columns of N points (TileFft), loaded from and
// stored to memory without a staging tile: a wave's access covers 64 / CW
// rows of CW consecutive columns.
//
// What bounds them: vector instructions and memory about equally.  A fan-out
// of a 512^2 x 64 plane launch with all four references present runs one forward and
// four inverse transforms, 203 VALU instructions per point (40 per term: 31 of the
// transform, the rest the multiplier), VALU 60 % busy, while it moves
// 0.52 GB (3.6 TB/s); LDS is active 36 % of the time without bank conflicts.
// The form before staged every tile through LDS on the way in and out (one
// exchange and a barrier more per term) and computed every position and LDS address
// per element.  Before -> now, us per launch: fan-out 512^2 x 64 planes 175 ->
// 143, 384^2 x 200 375 -> 255, 1024^2 x 128 1012 -> 877, 192 x 384 x 26 (complex
// slowness) 92 -> 50, 96 x 128 x 24 25 -> 11; fan-in 212 -> 180, 572 -> 281, 1237 -> 960,
// 121 -> 54, 25 -> 10; float64 768^2 x 6 fan-out 222 -> 95, fan-in 443 -> 102 (134 and
// 272 with sincos and k^2 held, 117 registers spilled; 16 now).
#pragma once
#include "fwix_kernels.h"
#include "fwix_launch.h"

#include <type_traits>

namespace fwix {

// Workgroups are handed to the 8 XCDs round-robin by linear id, and each
// XCD has its own L2.  A column tile reads CW * 8 bytes of every row; with
// CW = 8 (4) that is a half (quarter) of a 128-byte line, so G = 2 (4)
// neighbouring tiles share every line they read.  Linear ids L, L + 8, ...
// run on the same XCD back to back, so they take the G parts: within each
// group of 8G ids, 8G g + 8h + q gets the logical tile 8G g + G q + h (a
// trailing partial group keeps the identity).  Logical tile J is column
// tile J % gridDim.x of plane J / gridDim.x.
template <class F>
__device__ __forceinline__ void col_tile(int& plane, int& c0) {
  const int nb = gridDim.x;
  const int L = blockIdx.y * nb + blockIdx.x;
  int J = L;
  constexpr int G = 128 / (F::CW * 8);
  if constexpr (G > 1) {
    const int total = nb * gridDim.y;
    const int r = L % (8 * G);
    if (L - r + 8 * G <= total) J = L - r + G * (r % 8) + r / 8;
  }
  plane = J / nb;
  c0 = (J - plane * nb) * F::CW;
}

// Columns per workgroup: 8 (half a line of memory per row; 16 would take the
// LDS of a second workgroup), 4 for float64 columns from 512 points on (twice
// the LDS per value) and for 1024 points in the 4-column layout, the default
// there: its waves access whole quad blocks and three workgroups fit a CU
// (1024^2 x 16 planes: fan-out 160 us against 227 with 8 columns, fan-in 210 against
// 253).
constexpr int col_cw(int N, bool f64, int layout) { return (f64 && N >= 512) || (N == 1024 && layout == 1) ? 4 : 8; }

// One plane of a wavefield (or of a term buffer) as a buffer resource: the
// base address sits in scalar registers, an element costs one 32-bit lane
// offset and a uniform offset.  Offsets at or beyond the plane's size read as
// zero and drop stores (hardware range check), which replaces the per-element
// bounds and presence branches: such elements get the offset kOff.
constexpr unsigned kOff = 0x80000000u;
__device__ __forceinline__ unsigned plane_bytes(const KArgs& a) { return (unsigned)(a.NX * a.NY) * 8u; }
struct PlaneBuf {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ PlaneBuf(const float2* base, unsigned bytes)
      : r(__builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)bytes, 0x00020000)) {}
  __device__ __forceinline__ float2 load(unsigned off, int soff) const {
    return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, soff, 0));
  }
  __device__ __forceinline__ void store(float2 v, unsigned off, int soff) const {
    using U2 = __attribute__((ext_vector_type(2))) unsigned;
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), r, (int)off, soff, 0);
  }
};
// Byte offsets of this thread's elements: its column at rows row + C, C the
// first (FIRST: row l0) or last positions of the transform, in a row-major
// plane or (quad) one in the quad-block layout.  When every C is a multiple of
// 4, C rows move the offset by C NX elements in both layouts; the short columns where
// one is not (8, 12 and 24 points) form the offset per element.
template <class F, bool FIRST>
struct ColOffs {
  static constexpr int C(int e) { return FIRST ? F::first_c(e) : F::last_c(e); }
  static constexpr bool by4() {
    for (int e = 0; e < F::V; ++e)
      if (C(e) % 4) return false;
    return true;
  }
  unsigned o;
  int row, col, NX, step;
  bool quad;
  __device__ __forceinline__ ColOffs(const F& f, int c0, int NX_, bool quad_)
      : row(FIRST ? f.l0 : f.lane), col(c0 + f.col), NX(NX_), step(NX_ * 8), quad(quad_) {
    o = col >= NX ? kOff : (quad ? qidx(row, col, NX) : (unsigned)(row * NX + col)) * 8u;
  }
  __device__ __forceinline__ unsigned voff(int e) const {
    if constexpr (by4()) return o;
    if (col >= NX) return kOff;
    return (quad ? qidx(row + C(e), col, NX) : (unsigned)((row + C(e)) * NX + col)) * 8u;
  }
  __device__ __forceinline__ int soff(int e) const { return by4() ? C(e) * step : 0; }
};

// this workgroup's copy of the column transforms' twiddle table and of the
// plane's row masks, inverted (absent references set; none when masks are off);
// the caller synchronises.
// In LDS because one wait counter covers vector loads and stores: a global
// load in the loop over the terms would wait for the term's stores or for the
// next term's tile in flight.
// (every thread group of a workgroup writes the same values)
template <class F, class T>
__device__ __forceinline__ void col_twiddles(T* twl, const T* __restrict__ tw) {
  for (int i = threadIdx.x; i < F::TW; i += F::THREADS) twl[i] = tw[i];
}
template <class F, int N>
__device__ __forceinline__ void col_row_masks(uint32_t* rml, const uint32_t* __restrict__ rm) {
  for (int i = threadIdx.x; i < N; i += F::THREADS) rml[i] = rm ? ~rm[i] : 0u;
}
// offset off of an element whose row has reference r (< 32), else kOff
__device__ __forceinline__ unsigned off_if(uint32_t absent, int r, unsigned off) {
  return off | ((absent << (31 - r)) & kOff);
}
// Reference slowness r of the plane, by a scalar load (through a
// constant-address-space pointer): that load waits on the scalar counter
// only, and every workgroup of the plane reads the same few values.
__device__ __forceinline__ float2 term_sref(const KArgs& a, int r, int iw) {
  using CP = const __attribute__((address_space(4))) float*;
  const CP p = (CP)(const void*)a.sref + 2 * (r * a.NW + iw);
  return make_float2(p[0], p[1]);
}

// ------------------------------------------------------------------ multipliers
// Pointwise spectral multiplier of term r at (kx, ky) of frequency iw.
// MULT 0 / 1: forward / adjoint phase shift of reference slowness r
// (propagator/src/phase_shift.cu); MULT 2: Born scattering wavenumber factor
// (|k|/w)^(2it) = (k^2/w^2)^it of Taylor order it = r + 1 (scatter.cu:23-59);
// order 0 is the identity and is applied in space by the row kernels.
// The term's uniform part (reference slowness, real/complex branch) is set up
// once per (plane, term) so the unrolled per-sample loops carry no divergent
// or if-converted paths.
// The phase sqrt(a) dz goes to revolutions in one fused product with dz / 2 pi in two
// parts: rounded to one float32 that factor is up to 6e-8 off, by dz, the same for every
// wavenumber, frequency and depth, and a recursion adds it up (per radian, mean of 256
// frequencies over 100 steps: 7.9e-8 at dz = 6.284, 4.3e-8 at 7.3; in two parts 3.1e-8 and 2.5e-8).
// The product it costs is skipped with the sine where no lane propagates (downward 512^2, 11
// references: 22.43 -> 22.47 ms).
template <int MULT, class T>
struct TermMult {
  using S = real_of<T>;
  S w2, sre, b, iw2, dz;
  S turns, turns_lo, decay;  // phase in revolutions and log2 of the amplitude per sqrt|a| (the phase in two parts)
  int r;
  bool real;
  __device__ __forceinline__ TermMult(const KArgs& a, int r_, int iw, S w2_) : w2(w2_), r(r_), dz(a.dz) {
    if constexpr (MULT == 2) {
      iw2 = (S)1 / w2;
      real = true; sre = 0; b = 0;
    } else {
      const float2 sr = term_sref(a, r_, iw);
      sre = sr.x;
      b = w2 * ((S)sr.y - (S)a.eps * (S)sr.x);
      real = b == 0;
      iw2 = 0;
      turns = (S)((double)a.dz * 0.15915494309189533577);
      turns_lo = (S)((double)a.dz * 0.15915494309189533577 - (double)turns);
      decay = (S)((double)a.dz * -1.44269504088896340736);
    }
  }
  // x times the multiplier at k2, plus acc where ADD
  template <bool ADD>
  __device__ __forceinline__ static T times(T x, S m, T acc) {
    if constexpr (!ADD) return cscale(x, m);
    else return CX<T>::mk(fma_(x.x, m, acc.x), fma_(x.y, m, acc.y));
  }
  template <bool ADD>
  __device__ __forceinline__ static T times(T x, T m, T acc) {
    if constexpr (!ADD) return cmul(x, m);
    else return CX<T>::mk(fma_(x.x, m.x, fma_(-x.y, m.y, acc.x)), fma_(x.x, m.y, fma_(x.y, m.x, acc.y)));
  }
  __device__ __forceinline__ static float fma_(float a, float b, float c) { return fmaf(a, b, c); }
  __device__ __forceinline__ static double fma_(double a, double b, double c) { return fma(a, b, c); }
  template <bool REAL, bool ADD>
  __device__ __forceinline__ T apply(T x, S k2, T acc) const {
    if constexpr (MULT == 2) {
      const S q = sizeof(S) == 8 ? k2 / w2 : k2 * iw2;
      S m = q;
      for (int i = 0; i < r; ++i) m *= q;
      return times<ADD>(x, m, acc);
    } else if constexpr (sizeof(S) == 8) {
      if constexpr (!REAL) {
        return times<ADD>(x, ps_general64<MULT>(w2 * sre - k2, b, dz), acc);
      } else {
        const S a = w2 * sre - k2, q = sqrt(fabs(a));
        if (a < 0) return times<ADD>(x, exp(-q * dz), acc);
        S sn, cs;
        sincospi(q * (dz * kInvPi), &sn, &cs);
        return times<ADD>(x, CX<T>::mk(cs, MULT == 0 ? -sn : sn), acc);
      }
    } else if constexpr (!REAL) {
      return times<ADD>(x, ps_general<MULT>(fmaf(w2, sre, -k2), b, dz), acc);
    } else {
      // Past the evanescent boundary the multiplier is real and needs no sine
      // or cosine.  A wave's samples are neighbours in (kx, ky), so most
      // waves lie on one side (the propagating disc of a 10-20 m grid covers
      // 3-15 % of the plane): one test of the wave skips both.
      const float a = fmaf(w2, sre, -k2), q = __builtin_amdgcn_sqrtf(fabsf(a));
      const float e = __builtin_amdgcn_exp2f(q * decay);
      if (__builtin_amdgcn_ballot_w64(a >= 0.f) == 0) return times<ADD>(x, e, acc);
      const float rev = __builtin_amdgcn_fractf(fmaf(q, turns, q * turns_lo));
      const float sn = __builtin_amdgcn_sinf(rev), cs = __builtin_amdgcn_cosf(rev);
      const float2 m = a >= 0.f ? make_float2(cs, MULT == 0 ? -sn : sn) : make_float2(e, 0.f);
      return times<ADD>(x, m, acc);
    }
  }
};
// k^2 = kx^2 + ky^2 at this thread's samples after a forward transform (the
// positions of the last stage): HELD in registers over the terms, or formed
// from the wavenumbers staged in LDS (the caller synchronises) where those registers
// cost waves.  Float64 kernels are at their budget (the phase-shift fan-in with V = 12 still spills 6 to 17
// of 256); the float32 fan-in with V = 12 goes from 145 to 128 registers at 384 points (3
// spilled), a fourth wave per SIMD, and from 15 spilled to 2 at 768 (8 references, 34 planes: 543 ->
// 466 us); with V = 8 the wave more is not reached (512: 215 us held, 222 not).
template <class F, int N, class S, bool HELD>
struct ColumnK2 {
  S v[HELD ? F::V : 1];
  const float* ky;
  __device__ __forceinline__ ColumnK2(const F& f, const KArgs& a, int c0, float* lds) {
    const int col = c0 + f.col;
    const S kxv = a.kx[col < a.NX ? col : 0];
    if constexpr (HELD) {
      ky = a.ky + f.lane;
#pragma unroll
      for (int e = 0; e < F::V; ++e) {
        const S kyv = ky[F::last_c(e)];
        if constexpr (sizeof(S) == 8) v[e] = fma(kxv, kxv, kyv * kyv);
        else v[e] = fmaf(kxv, kxv, kyv * kyv);
      }
    } else {
      for (int i = threadIdx.x; i < N; i += F::THREADS) lds[i] = a.ky[i];
      ky = lds + f.lane;
      v[0] = kxv;
    }
  }
  __device__ __forceinline__ S at(int e) const {
    if constexpr (HELD) return v[e];
    const S kyv = ky[F::last_c(e)];
    if constexpr (sizeof(S) == 8) return fma(v[0], v[0], kyv * kyv);
    else return fmaf(v[0], v[0], kyv * kyv);
  }
};

// ------------------------------------------------------------------ launch geometry
template <class F>
inline dim3 col_grid(const KArgs& a) {
  return dim3((a.NX + F::CW - 1) / F::CW, a.np);
}
template <class Fn>
hipError_t dispatch_wpe(int wpe, Fn&& fn) {
  switch (wpe) {
    case 2: return fn(std::integral_constant<int, 2>{});
    case 4: return fn(std::integral_constant<int, 4>{});
    case 6: return fn(std::integral_constant<int, 6>{});
    default: return hipErrorInvalidValue;
  }
}
// mode 0..2 as a constant
template <class Fn>
hipError_t dispatch_mode(int mode, Fn&& fn) {
  switch (mode) {
    case 0: return fn(std::integral_constant<int, 0>{});
    case 1: return fn(std::integral_constant<int, 1>{});
    case 2: return fn(std::integral_constant<int, 2>{});
    default: return hipErrorInvalidValue;
  }
}
// One column kernel per (size, mode) and, in float32, register budget (2, 4
// or 6 waves per SIMD, col_wpe_get, col_wpe_built) and at 1024 points tile width
// (col_layout_get); float64 arithmetic (a.f64) has one budget.  Launches that
// leave the chip idle split their terms (term_split): a fan-out over more
// workgroups (each with its own forward transform), a fan-in (GROUPS) over thread groups
// of its workgroups.  K<N, MODE, WPE, T, CW, G>::kernel
// Tiles of 8 waves (512 and 768 points, 1024 in 8 columns) keep one group: with
// two of them waiting for each other 4 references take longer on one plane (96 x 512:
// 16.4 us in two groups, 15.3 in one; 96 x 768: 24.3, 23.9), one present takes 10.9 against
// 8.9 and 15.3 against 11.9, and 8 gain little (23.5 against 24.2, 36.7 against 39.6).
// Groups start at 3 terms (one plane or few, 2 terms, whole -> split: 128 x 128 x 4
// 8.6 -> 9.3 us, 192 x 192 x 4 10.8 -> 11.7, 384 x 384 13.3 -> 12.9; 3 terms 10.1 -> 9.6, 13.1 ->
// 12.0, 16.7 -> 16.7), at 256 points at 4 (3: 11.0 -> 11.8; 4: 13.2 -> 12.8, with complex
// slowness 13.4 -> 13.8; 8: 20.0 -> 18.0).
constexpr int col_groups(int threads, int N) { return threads <= 128 || N == 256 ? 4 : 2; }
template <template <int, int, int, class, int, int> class K, bool GROUPS>
hipError_t launch_col_terms(int kind, int mode, const KArgs& a, hipStream_t st) {
  return dispatch_n(a.NY, [&](auto nc) {
    constexpr int N = decltype(nc)::value;
    return dispatch_mode(mode, [&](auto mc) {
      constexpr int M = decltype(mc)::value;
      auto go = [&](auto wc, auto cc, auto t) -> hipError_t {
        using T = decltype(t);
        constexpr int CW = decltype(cc)::value;
        constexpr int W = sizeof(T) == 16 ? 2 : col_wpe_built(GROUPS ? 1 : 0, N, decltype(wc)::value);
        using F = TileFft<N, T, CW>;
        dim3 g = col_grid<F>(a), b(F::THREADS);
        const long long waves = (long long)g.x * g.y * F::WAVES;
        const int terms = M == 2 ? a.nterm : live_refs(a);
        if constexpr (!GROUPS) {
          g.z = term_split(waves, terms, 4, 2048);
        } else if constexpr (M != 2 && sizeof(T) == 8 && F::WAVES < 8) {
          constexpr int G = col_groups(F::THREADS, N);
          if (term_split(waves, terms, G, 512, N == 256 ? 4 : 3) > 1) {
            b.y = G;
            hipLaunchKernelGGL((K<N, M, 2, T, CW, G>::kernel), g, b, 0, st, a);
            return hipGetLastError();
          }
        }
        hipLaunchKernelGGL((K<N, M, W, T, CW, 1>::kernel), g, b, 0, st, a);
        return hipGetLastError();
      };
      constexpr std::integral_constant<int, col_cw(N, true, 0)> cw64{};
      if (a.f64) return go(std::integral_constant<int, 2>{}, cw64, double2{});
      return dispatch_wpe(col_wpe_get(kind, mode, N), [&](auto wc) {
        if constexpr (N == 1024) {
          if (col_layout_get(kind, mode, N) == 1) return go(wc, std::integral_constant<int, col_cw(N, false, 1)>{}, float2{});
        }
        return go(wc, std::integral_constant<int, col_cw(N, false, 0)>{}, float2{});
      });
    });
  });
}

}  // namespace fwix
