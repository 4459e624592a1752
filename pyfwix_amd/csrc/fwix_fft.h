// Wave-level Stockham FFT for gfx950 (CDNA4, 64-lane wavefronts).
//
// One wavefront transforms NB batches of N points held as V = NB*N/64 complex
// values per lane.  The radix plan (8, 4, 3, 2) is fixed at compile time from
// N and V so every loop unrolls and every index is a constant-folded shift or
// multiply.  Stages exchange data through the wave's own LDS region and only
// need wave-level ordering, never a workgroup barrier.
//
// Position conventions (Stockham autosort, decimation in time):
//   stage radix R, sub-transform size Ns (product of earlier radices):
//     butterfly (b, j), j < N/R, reads  x[b][j + r*N/R]
//     writes y[b][(j/Ns)*Ns*R + j%Ns + r*Ns]
//   The first stage therefore reads positions j + r*N/R0 and the last stage
//   writes positions j + r*N/RL, both contiguous across lanes: kernels load
//   the first stage straight from global memory and store the last stage
//   straight back.  The inverse plan is the forward plan reversed, so the
//   inverse's first stage reads exactly the positions the forward's last
//   stage wrote: a forward -> pointwise multiply -> inverse chain never leaves
//   registers between the two transforms.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fwix {

// ----------------------------------------------------------------- complex helpers
// float2 (complex64) is the storage and default arithmetic type; the same
// helpers exist for double2, so a transform can run in float64 arithmetic on
// values loaded from and stored to complex64 arrays.
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(fmaf(a.x, b.x, -a.y * b.y), fmaf(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ float2 cmulc(float2 a, float2 b) {  // a * conj(b)
  return make_float2(fmaf(a.x, b.x, a.y * b.y), fmaf(a.y, b.x, -a.x * b.y));
}
__device__ __forceinline__ float2 cconj(float2 a) { return make_float2(a.x, -a.y); }
__device__ __forceinline__ float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
__device__ __forceinline__ float2 czero() { return make_float2(0.f, 0.f); }

__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ double2 cmulc(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, a.y * b.y), fma(a.y, b.x, -a.x * b.y));
}
__device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
__device__ __forceinline__ double2 cscale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }

// the arithmetic type T's scalar and constructor; conversions from / to the
// complex64 storage type
template <class T> struct CX;
template <> struct CX<float2> {
  using S = float;
  __device__ __forceinline__ static float2 mk(float x, float y) { return make_float2(x, y); }
};
template <> struct CX<double2> {
  using S = double;
  __device__ __forceinline__ static double2 mk(double x, double y) { return make_double2(x, y); }
};
template <class T> using real_of = typename CX<T>::S;
template <class T> __device__ __forceinline__ T cz() { return CX<T>::mk(0, 0); }
template <class T> __device__ __forceinline__ T from_f2(float2 a) { return CX<T>::mk(a.x, a.y); }
__device__ __forceinline__ float2 to_f2(float2 a) { return a; }
__device__ __forceinline__ float2 to_f2(double2 a) { return make_float2((float)a.x, (float)a.y); }

// multiply by sgn*i, sgn = -1 for the forward (e^{-i}) transform, +1 for the inverse
template <bool INV, class T>
__device__ __forceinline__ T mul_si(T a) {
  return INV ? CX<T>::mk(-a.y, a.x) : CX<T>::mk(a.y, -a.x);
}

// ----------------------------------------------------------------- compile-time plan
constexpr int kRadices[4] = {8, 4, 3, 2};

constexpr int plan_len(int N, int V) {
  int n = N, c = 0;
  for (int k = 0; k < 4; ++k) {
    const int R = kRadices[k];
    while (n % R == 0 && V % R == 0) { n /= R; ++c; }
  }
  return n == 1 ? c : -1;
}

constexpr int plan_radix(int N, int V, int s) {
  int n = N, c = 0;
  for (int k = 0; k < 4; ++k) {
    const int R = kRadices[k];
    while (n % R == 0 && V % R == 0) {
      if (c == s) return R;
      n /= R; ++c;
    }
  }
  return 0;
}

// radix of stage s of the forward (INV=false) or inverse (reversed) plan
template <int N, int V, bool INV>
struct Plan {
  static constexpr int S = plan_len(N, V);
  static_assert(S > 0, "FFT size has no radix plan for this register budget");
  static constexpr int radix(int s) { return plan_radix(N, V, INV ? (S - 1 - s) : s); }
  static constexpr int ns(int s) {  // product of the radices of stages < s
    int p = 1;
    for (int k = 0; k < s; ++k) p *= radix(k);
    return p;
  }
  static constexpr int first() { return radix(0); }
  static constexpr int last() { return radix(S - 1); }
};

// ----------------------------------------------------------------- in-register DFTs
template <int R, bool INV> struct Dft;

template <bool INV> struct Dft<2, INV> {
  template <class T>
  __device__ __forceinline__ static void run(T* x) {
    T a = x[0], b = x[1];
    x[0] = cadd(a, b); x[1] = csub(a, b);
  }
};

template <bool INV> struct Dft<4, INV> {
  template <class T>
  __device__ __forceinline__ static void run(T* x) {
    T a = cadd(x[0], x[2]), b = csub(x[0], x[2]);
    T c = cadd(x[1], x[3]), e = mul_si<INV>(csub(x[1], x[3]));
    x[0] = cadd(a, c); x[2] = csub(a, c);
    x[1] = cadd(b, e); x[3] = csub(b, e);
  }
};

template <bool INV> struct Dft<3, INV> {
  template <class T>
  __device__ __forceinline__ static void run(T* x) {
    using S = real_of<T>;
    const S h = (S)0.86602540378443864676;  // sin(2*pi/3)
    T t1 = cadd(x[1], x[2]);
    T t2 = mul_si<INV>(cscale(csub(x[1], x[2]), h));
    T m = CX<T>::mk(x[0].x - (S)0.5 * t1.x, x[0].y - (S)0.5 * t1.y);
    x[0] = cadd(x[0], t1);
    x[1] = cadd(m, t2);
    x[2] = csub(m, t2);
  }
};

template <bool INV> struct Dft<8, INV> {
  template <class T>
  __device__ __forceinline__ static void run(T* x) {
    using S = real_of<T>;
    T e[4] = {x[0], x[2], x[4], x[6]};
    T o[4] = {x[1], x[3], x[5], x[7]};
    Dft<4, INV>::run(e);
    Dft<4, INV>::run(o);
    const S r = (S)0.70710678118654752440;
    // W8^k = exp(sgn*2*pi*i*k/8), sgn = -1 forward
    T o1 = cscale(cadd(o[1], mul_si<INV>(o[1])), r);           // (1 + sgn i)/sqrt2
    T o2 = mul_si<INV>(o[2]);                                   // sgn i
    T o3 = cscale(csub(mul_si<INV>(o[3]), o[3]), r);           // (-1 + sgn i)/sqrt2
    x[0] = cadd(e[0], o[0]); x[4] = csub(e[0], o[0]);
    x[1] = cadd(e[1], o1);   x[5] = csub(e[1], o1);
    x[2] = cadd(e[2], o2);   x[6] = csub(e[2], o2);
    x[3] = cadd(e[3], o3);   x[7] = csub(e[3], o3);
  }
};

// 16 = 4 x 4; the twiddles between the two layers are multiples of pi/8
template <bool INV> struct Dft<16, INV> {
  template <class T>
  __device__ __forceinline__ static void run(T* x) {
    using S = real_of<T>;
    const S r = (S)0.70710678118654752440, c = (S)0.92387953251128675613, s = (S)0.38268343236508977173;
    T y[4][4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
#pragma unroll
      for (int a = 0; a < 4; ++a) y[b][a] = x[4 * a + b];
      Dft<4, INV>::run(y[b]);
    }
    auto rot = [&](T v, S cr, S si) {  // v * (cr + sgn i si), sgn = -1 forward
      return INV ? cmul(v, CX<T>::mk(cr, si)) : cmulc(v, CX<T>::mk(cr, si));
    };
    auto w2 = [&](T v) { return cscale(cadd(v, mul_si<INV>(v)), r); };       // pi/4
    auto w6 = [&](T v) { return cscale(csub(mul_si<INV>(v), v), r); };       // 3 pi/4
    y[1][1] = rot(y[1][1], c, s);   y[1][2] = w2(y[1][2]);           y[1][3] = rot(y[1][3], s, c);
    y[2][1] = w2(y[2][1]);          y[2][2] = mul_si<INV>(y[2][2]);  y[2][3] = w6(y[2][3]);
    y[3][1] = rot(y[3][1], s, c);   y[3][2] = w6(y[3][2]);           y[3][3] = rot(y[3][3], -c, -s);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      T z[4] = {y[0][k], y[1][k], y[2][k], y[3][k]};
      Dft<4, INV>::run(z);
#pragma unroll
      for (int d = 0; d < 4; ++d) x[k + 4 * d] = z[d];
    }
  }
};

// R = A * B with coprime A, B by the prime-factor map, free of twiddles:
// input n = (B n1 + A n2) mod R, output k with k mod A = k1, k mod B = k2
template <int A, int B, bool INV> struct DftPfa {
  static constexpr int R = A * B;
  static constexpr int crt(int k1, int k2) {
    for (int k = 0; k < R; ++k)
      if (k % A == k1 && k % B == k2) return k;
    return 0;
  }
  template <class T>
  __device__ __forceinline__ static void run(T* x) {
    T y[A][B];  // [n1][k2]
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) {
#pragma unroll
      for (int n2 = 0; n2 < B; ++n2) y[n1][n2] = x[(B * n1 + A * n2) % R];
      Dft<B, INV>::run(y[n1]);
    }
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) {
      T z[A];
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) z[n1] = y[n1][k2];
      Dft<A, INV>::run(z);
#pragma unroll
      for (int k1 = 0; k1 < A; ++k1) x[crt(k1, k2)] = z[k1];
    }
  }
};
template <bool INV> struct Dft<6, INV> : DftPfa<3, 2, INV> {};
template <bool INV> struct Dft<12, INV> : DftPfa<3, 4, INV> {};

// ----------------------------------------------------------------- wave ordering
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ----------------------------------------------------------------- positions
// Butterfly t = lane + 64*q of a radix-R stage owns batch b and index j.
// BFAST: batch index varies fastest across lanes (column tiles), else the
// position within the batch does (rows).
// (Unsigned arithmetic: t is never negative, and the lane index is opaque to
// the compiler inside a transform, so signed division would cost sign fix-ups.)
template <int N, int NB, int R, bool BFAST>
__device__ __forceinline__ void bj(int t, int& b, int& j) {
  const unsigned u = (unsigned)t;
  if (BFAST) { b = (int)(u % NB); j = (int)(u / NB); }
  else { b = (int)(u / (N / R)); j = (int)(u % (N / R)); }
}

// (batch, position) of value v = q*R + r at the input of a stage of radix R
// when it is the first stage, or at the output when it is the last stage.
template <int N, int NB, int R, bool BFAST>
__device__ __forceinline__ void edge_pos(int lane, int v, int& b, int& i) {
  const int q = v / R, r = v % R;
  int j;
  bj<N, NB, R, BFAST>(lane + 64 * q, b, j);
  i = j + r * (N / R);
}

// ----------------------------------------------------------------- the transform
// LDS layout policy: L::addr(b, i) gives the element offset of batch b, point i
// inside the wave's region.  T is the arithmetic type of the values, the LDS
// region and the twiddle table (float2, or double2 for float64 arithmetic).
template <int N, int NB, bool BFAST, bool INV, class L, class T = float2>
struct WaveFft {
  static constexpr int V = NB * N / 64;
  using P = Plan<N, V, INV>;
  static constexpr int S = P::S;

  template <int R, int Ns>
  __device__ __forceinline__ static void butterflies(T* v, const T* __restrict__ tw, int lane) {
#pragma unroll
    for (int q = 0; q < V / R; ++q) {
      T* x = v + q * R;
      if constexpr (Ns > 1) {
        int b, j;
        bj<N, NB, R, BFAST>(lane + 64 * q, b, j);
        const int k = (int)((unsigned)j % Ns);
        constexpr int step = N / (Ns * R);
#pragma unroll
        for (int r = 1; r < R; ++r) {
          T w = tw[r * k * step];
          if (INV) w.y = -w.y;
          x[r] = cmul(x[r], w);
        }
      }
      Dft<R, INV>::run(x);
    }
  }

  template <int R, int Ns, int R2>
  __device__ __forceinline__ static void exchange(T* v, T* lds, int lane) {
#pragma unroll
    for (int q = 0; q < V / R; ++q) {
      int b, j;
      bj<N, NB, R, BFAST>(lane + 64 * q, b, j);
      const unsigned uj = (unsigned)j;
      const int base = (int)((uj / Ns) * Ns * R + (uj % Ns));
#pragma unroll
      for (int r = 0; r < R; ++r) lds[L::addr(b, base + r * Ns)] = v[q * R + r];
    }
    wave_sync();
#pragma unroll
    for (int q = 0; q < V / R2; ++q) {
      int b, j;
      bj<N, NB, R2, BFAST>(lane + 64 * q, b, j);
#pragma unroll
      for (int r = 0; r < R2; ++r) v[q * R2 + r] = lds[L::addr(b, j + r * (N / R2))];
    }
    wave_sync();
  }

  template <int s>
  __device__ __forceinline__ static void stages(T* v, T* lds, const T* __restrict__ tw, int lane) {
    if constexpr (s < S) {
      constexpr int R = P::radix(s);
      constexpr int Ns = P::ns(s);
      butterflies<R, Ns>(v, tw, lane);
      if constexpr (s + 1 < S) {
        exchange<R, Ns, P::radix(s + 1)>(v, lds, lane);
        stages<s + 1>(v, lds, tw, lane);
      }
    }
  }

  // v holds the values at first-stage input positions (edge_pos<..., P::first()>);
  // on return it holds the spectrum at last-stage output positions
  // (edge_pos<..., P::last()>).  Unnormalized.
  __device__ __forceinline__ static void run(T* v, T* lds, const T* __restrict__ tw, int lane) {
    // Keep the twiddles and the per-element twiddle / LDS addresses next to
    // their use: without these fences the compiler hoists every stage's
    // (loop-invariant) loads and addresses out of the per-reference loops
    // of the fused kernels and runs out of registers.  The lane index is
    // made opaque here, so the index arithmetic derived from it is redone
    // per transform (a few integer ops) instead of held in registers.
    asm volatile("" ::: "memory");
    asm volatile("" : "+v"(lane));
    stages<0>(v, lds, tw, lane);
  }
};

// ================================================================= lane transform
// The transforms of the row passes.  L = N / V lanes hold one line of N
// points, V values each, and a wave holds 64 / L lines; lane l of a line owns
// the butterflies j = l + L q of every stage.  The plans below take few,
// wide stages (their count is what sets the LDS exchanges), with V a multiple
// of every radix and L a divisor (or a multiple) of every sub-transform
// length, so that every position, LDS address and twiddle index of a value is
// a per-lane base plus a compile-time constant: the loops carry no index
// arithmetic (the transforms it replaced spent half of their VALU
// instructions on it).
//
//   forward stage s (radix R, sub-transform length Ns): butterfly j reads
//     positions j + r N/R, multiplies by W_{Ns R}^(r (j mod Ns)), and leaves
//     output r at position (j / Ns) Ns R + j mod Ns + r Ns
//   inverse: the forward stages undone in reverse order (butterfly, then the
//     conjugate twiddles, exchanges written where the forward reads and read
//     where it writes), so it starts at the positions the forward ends at and
//     ends where the forward starts.
struct PlanDef {
  int V, S, R[4];
};
// Short lines take narrow plans (V <= 12): their launches are small and more
// waves in flight are worth more than a stage less (256 points: Born adjoint
// rows 21.3 us at V = 16, two stages, 17.5 us at V = 8, three).  The long
// lines with a factor 3 take V = 24 (768 points: 4 stages of V = 12 against 3);
// float64 lines hold at most 16 values per lane (twice the registers each).
__host__ __device__ constexpr PlanDef plan_def(int N, bool f64) {
  switch (N) {
    case 8: return {4, 2, {4, 2}};
    case 12: return {12, 1, {12}};
    case 16: return {4, 2, {4, 4}};
    case 24: return {12, 2, {4, 6}};
    case 32: return {8, 2, {8, 4}};
    case 48: return {12, 2, {4, 12}};
    case 64: return {8, 2, {8, 8}};
    case 96: return {12, 3, {4, 2, 12}};
    case 128: return {8, 3, {8, 4, 4}};
    case 192: return {12, 3, {4, 4, 12}};
    case 256: return {8, 3, {8, 8, 4}};
    case 384: return f64 ? PlanDef{12, 4, {4, 4, 4, 6}} : PlanDef{24, 3, {8, 8, 6}};
    case 512: return {8, 3, {8, 8, 8}};
    case 768: return f64 ? PlanDef{12, 4, {4, 4, 4, 12}} : PlanDef{24, 3, {8, 8, 12}};
    case 1024: return {16, 3, {16, 8, 8}};
    default: return {0, 0, {}};
  }
}
__host__ __device__ constexpr int plan_ns(const PlanDef& d, int s) {
  int p = 1;
  for (int k = 0; k < s; ++k) p *= d.R[k];
  return p;
}
// Entry i of a length's twiddle table: the exponent e of exp(-2 pi i e / N).
// Stage s holds its R - 1 rows of Ns factors one after another ([r][k], k
// fastest), so a lane reads W^(rk) at a base of its own plus r Ns, neighbouring
// lanes on neighbouring entries.  Entries past the last stage's are zero.
__host__ __device__ constexpr int twiddle_exp(int N, bool f64, int i) {
  const PlanDef d = plan_def(N, f64);
  int o = 0;
  for (int s = 1; s < d.S; ++s) {
    const int Ns = plan_ns(d, s), n = (d.R[s] - 1) * Ns;
    if (i < o + n) {
      const int r = (i - o) / Ns + 1, k = (i - o) % Ns;
      return r * k * (N / (Ns * d.R[s]));
    }
    o += n;
  }
  return 0;
}

template <int N, class T = float2>
struct LaneFft {
  // (a constexpr array member would be a device constant, loaded at run time:
  // the plan is only ever read through these functions)
  static constexpr bool F64 = sizeof(T) == 16;
  static constexpr int V = plan_def(N, F64).V, S = plan_def(N, F64).S, L = N / V, NB = 64 / L;
  static_assert(V > 0 && L * V == N && NB * L == 64, "lanes must divide the line and the wave");
  static constexpr int R(int s) { return plan_def(N, F64).R[s]; }
  static constexpr int Ns(int s) { return plan_ns(plan_def(N, F64), s); }
  static constexpr int tw_off(int s) {
    int o = 0;
    for (int k = 1; k < s; ++k) o += (R(k) - 1) * Ns(k);
    return o;
  }
  static constexpr int TW = tw_off(S) > 0 ? tw_off(S) : 1;  // table entries (N - R(0))

  // Padding of the exchange between stages s and s + 1, in positions: Ns more
  // after each block of G, but none where the sum reaches a row of banks (32).
  // 32 lanes then write runs of Ns positions NsR apart to distinct banks,
  // and still read 32 consecutive positions without a gap.
  static constexpr int G(int s) {
    int g = R(s) * Ns(s);
    while (g < 32) g *= 2;
    return g;
  }
  static constexpr int WR(int s) { return Ns(s) >= 32 ? 1 : 32 / Ns(s); }
  __host__ __device__ static constexpr int pad(int s, int blk) {
    const unsigned b = (unsigned)blk, w = (unsigned)WR(s);
    return (int)(b % w + b / w * (w - 1)) * Ns(s);
  }
  static constexpr int stride_min() {
    int m = N;
    for (int s = 0; s + 1 < S; ++s) {
      const int p = pad(s, (N - 1) / G(s));
      if (N + p > m) m = N + p;
    }
    return m;
  }
  // lines of a wave: short lines side by side in the banks (stride = L mod
  // 32); the others 8 past a multiple of 32, so that four rows staged as
  // quads fall into distinct banks
  static constexpr int STRIDE = stride_min() + ((L < 32 ? L : 8) + 32 * 64 - stride_min() % 32) % 32;

  // position of value v of lane l before the first forward stage (= after the
  // inverse) and after the last (= before the inverse): lane base + constant
  static constexpr int in_c(int s, int v) { return L * (v / R(s)) + (v % R(s)) * (N / R(s)); }
  static constexpr int first_c(int v) { return in_c(0, v); }
  static constexpr int last_c(int v) { return in_c(S - 1, v); }

  // exchange after stage s: LDS offset of value v where stage s + 1 reads
  // (IN) and where stage s wrote (OUT), as a lane base and a constant
  template <int s>
  __device__ __forceinline__ static int in_base(int l) {
    return l + pad(s, (int)((unsigned)l / (unsigned)G(s)));
  }
  template <int s>
  static constexpr int in_const(int v) {
    const int C = in_c(s + 1, v);
    return C + pad(s, C / G(s));
  }
  template <int s>
  static constexpr bool in_ok() {
    for (int v = 0; v < V; ++v) {
      const int C = in_c(s + 1, v);
      // the lane part stays in its block, or the constant is whole blocks
      // and the sum of the block numbers adds no bank row of its own
      const int blk = C / G(s), span = (L - 1) / G(s);
      if (!(C % G(s) + L <= G(s) || (C % G(s) == 0 && (blk % WR(s) == 0 || blk % WR(s) + span < WR(s)))))
        return false;
    }
    return true;
  }
  template <int s>
  __device__ __forceinline__ static int out_base(int l) {
    constexpr int n = Ns(s), g = G(s) / (n * R(s));
    const unsigned a = (unsigned)l / (unsigned)n;
    return (int)(a * n * R(s) + (unsigned)l % (unsigned)n) + pad(s, (int)(a / g));
  }
  template <int s>
  static constexpr int out_const(int v) {
    constexpr int n = Ns(s), g = G(s) / (n * R(s));
    const int q = v / R(s), r = v % R(s);
    return q * L * R(s) + r * n + pad(s, q * (L / n) / g);
  }
  template <int s>
  static constexpr bool out_ok() {
    constexpr int n = Ns(s), g = G(s) / (n * R(s));
    if (L % n) return false;
    for (int q = 0; q < V / R(s); ++q) {
      const int a = q * (L / n), span = (L / n - 1) / g;  // blocks the lane part reaches past the constant's
      const bool whole = a % g == 0 || a % g + L / n <= g;
      if (!whole) return false;
      if ((a / g) % WR(s) != 0 && (a / g) % WR(s) + span >= WR(s)) return false;
    }
    return true;
  }

  template <int s, bool INV>
  __device__ __forceinline__ static void twiddle(T* v, const T* __restrict__ tw, int l) {
    if constexpr (s > 0) {
      constexpr int n = Ns(s);
      static_assert(L % n == 0 || n % L == 0, "a lane's twiddles must sit at constant offsets");
      const T* t = tw + tw_off(s) + (L % n == 0 ? (int)((unsigned)l % (unsigned)n) : l);
#pragma unroll
      for (int q = 0; q < V / R(s); ++q) {
        const int kc = L % n == 0 ? 0 : (L * q) % n;
#pragma unroll
        for (int r = 1; r < R(s); ++r) {
          const T w = t[(r - 1) * n + kc];
          T& x = v[q * R(s) + r];
          x = INV ? cmulc(x, w) : cmul(x, w);
        }
      }
    }
  }
  template <int s, bool INV>
  __device__ __forceinline__ static void butterflies(T* v) {
#pragma unroll
    for (int q = 0; q < V / R(s); ++q) Dft<R(s), INV>::run(v + q * R(s));
  }
  template <int s>
  __device__ __forceinline__ static void put_out(const T* v, T* line, int l) {
    static_assert(out_ok<s>(), "exchange positions must split into lane base and constant");
    T* p = line + out_base<s>(l);
#pragma unroll
    for (int e = 0; e < V; ++e) p[out_const<s>(e)] = v[e];
  }
  template <int s>
  __device__ __forceinline__ static void get_out(T* v, const T* line, int l) {
    const T* p = line + out_base<s>(l);
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = p[out_const<s>(e)];
  }
  template <int s>
  __device__ __forceinline__ static void put_in(const T* v, T* line, int l) {
    static_assert(in_ok<s>(), "exchange positions must split into lane base and constant");
    T* p = line + in_base<s>(l);
#pragma unroll
    for (int e = 0; e < V; ++e) p[in_const<s>(e)] = v[e];
  }
  template <int s>
  __device__ __forceinline__ static void get_in(T* v, const T* line, int l) {
    const T* p = line + in_base<s>(l);
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = p[in_const<s>(e)];
  }

  // stages FROM .. TO - 1 of the forward transform, with the exchanges between
  // them (through this line's own LDS: wave ordering is enough)
  template <int FROM, int TO>
  __device__ __forceinline__ static void forward(T* v, T* line, const T* __restrict__ tw, int l) {
    if constexpr (FROM < TO) {
      twiddle<FROM, false>(v, tw, l);
      butterflies<FROM, false>(v);
      if constexpr (FROM + 1 < TO) {
        put_out<FROM>(v, line, l);
        wave_sync();
        get_in<FROM>(v, line, l);
        wave_sync();
        forward<FROM + 1, TO>(v, line, tw, l);
      }
    }
  }
  // stages FROM - 1 .. TO of the inverse
  template <int FROM, int TO>
  __device__ __forceinline__ static void inverse(T* v, T* line, const T* __restrict__ tw, int l) {
    if constexpr (FROM > TO) {
      butterflies<FROM - 1, true>(v);
      twiddle<FROM - 1, true>(v, tw, l);
      if constexpr (FROM - 1 > TO) {
        put_in<FROM - 2>(v, line, l);
        wave_sync();
        get_out<FROM - 2>(v, line, l);
        wave_sync();
        inverse<FROM - 1, TO>(v, line, tw, l);
      }
    }
  }
  // Whole transforms of a line held by one wave, unnormalized: v at
  // first_c / last_c positions in, at last_c / first_c out.  The memory
  // clobber keeps the twiddle loads next to their use (hoisted out of a
  // per-reference loop they would cost two registers each).
  template <bool INV>
  __device__ __forceinline__ static void run(T* v, T* line, const T* __restrict__ tw, int l) {
    asm volatile("" ::: "memory");
    if constexpr (INV) inverse<S, 0>(v, line, tw, l);
    else forward<0, S>(v, line, tw, l);
  }
};

}  // namespace fwix
