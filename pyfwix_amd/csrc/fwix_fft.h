// FFTs of lines held in registers for gfx950 (CDNA4, 64-lane wavefronts).
//
// L = N / V lanes hold one line of N points, V complex values each, with the
// radix plan fixed at compile time.  Stages exchange data through LDS.  Two
// owners of a line: LaneFft, a line inside one wave (the row passes), and
// TileFft, the columns of a tile across the waves of a workgroup (the column
// passes).
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

// 16 = 4 x 4; the twiddles between the two layers are multiples of pi/8.  In
// float32 sqrt(1/2) and sin(pi/8) both round down, cos(pi/8) lies in the middle
// of two values (3.1e-8 and 3.4e-8 off): the upper one makes up for the others, and the
// gain |F|^2 - 1 of a 1024-point transform {4, 16, 16} is -1e-8 in the mean
// instead of -6.5e-8, the same at every step of a recursion (its own rounding 1.07e-7
// instead of 1.10e-7; FWI gradient at 1024^2 0.50e-6 instead of 1.05e-6 from float64).
template <bool INV> struct Dft<16, INV> {
  template <class T>
  __device__ __forceinline__ static void run(T* x) {
    using S = real_of<T>;
    const S r = (S)0.70710678118654752440, s = (S)0.38268343236508977173;
    const S c = sizeof(S) == 8 ? (S)0.92387953251128675613 : (S)0.92387956381f;
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

// ================================================================= stages
// L = N / V lanes hold one line of N points; lane l of a line owns the
// butterflies j = l + L q of every stage.  The plans below take few, wide
// stages (their count is what sets the LDS exchanges), with V a multiple
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
//     ends where the forward starts: a forward -> pointwise multiply -> inverse
//     chain never leaves registers between the two transforms.
struct PlanDef {
  int V, S, R[4];
};
// Row plans and column plans, float32 and float64 arithmetic.
enum PlanKind { kRow32 = 0, kRow64 = 1, kCol32 = 2, kCol64 = 3 };
// Narrow plans (V <= 12 below 1024 points): the kernels hold two or three
// arrays of V values per lane, short lines' launches are small, and waves in flight
// are worth more than a stage less (256-point rows: Born adjoint 21.3 us at V = 16,
// two stages, 17.5 us at V = 8, three; 384 points, V = 24, three stages, against 12, four,
// 200 planes: scattering adjoint rows 203 -> 151 us, its imaging 129 -> 94, fan-out
// rows 160 -> 146, fan-out columns 193 -> 180 at 16 M points, fan-in 233 -> 211;
// 768 points, 5 planes: fan-out rows 52 -> 46 us, the select 39 -> 44).
// Rows of 12 and 24 points hold 6 values per lane, two and four lanes to a row: with 12, one and
// two lanes, an access touches 64 or 32 rows (12 x 1024 x 341 planes: plain rows 26 -> 17 us,
// scattering rows 48 -> 28, imaging rows 47 -> 27; 24 x 768 x 227: 18 -> 14, 31 -> 22, 32 -> 21).
// Columns lie across a tile and keep 12.
// The order of the stages decides which twiddles' rounding a recursion
// adds up step after step: columns of 384 points as
// {4, 2, 12, 4} take the time of {4, 4, 4, 6} (FWI gradient 384^2 x 200 15.8 ms, steps within
// 1 %) and leave that gradient 0.93e-6 from float64 instead of 1.27e-6; rows so ordered
// would halve it again, but read five twiddles more (plain rows 57 -> 62 us, 128 planes).
// Columns: a first radix R(0) that divides the lanes a wave holds of a column (TileFft).
__host__ __device__ constexpr PlanDef plan_def(int N, PlanKind kind) {
  switch (N) {
    case 8: return {4, 2, {4, 2}};
    case 12: return kind >= kCol32 ? PlanDef{12, 1, {12}} : PlanDef{6, 2, {6, 2}};
    case 16: return {4, 2, {4, 4}};
    case 24: return kind >= kCol32 ? PlanDef{12, 2, {4, 6}} : PlanDef{6, 3, {2, 6, 2}};
    case 32: return {8, 2, {8, 4}};
    case 48: return {12, 2, {4, 12}};
    case 64: return {8, 2, {8, 8}};
    case 96: return {12, 3, {4, 2, 12}};
    case 128: return {8, 3, {8, 4, 4}};
    case 192: return {12, 3, {4, 4, 12}};
    case 256: return {8, 3, {8, 8, 4}};
    case 384: return kind >= kCol32 ? PlanDef{12, 4, {4, 2, 12, 4}} : PlanDef{12, 4, {4, 4, 4, 6}};
    case 512: return {8, 3, {8, 8, 8}};
    case 768: return {12, 4, {4, 4, 4, 12}};
    case 1024:
      if (kind == kCol64) return {8, 4, {4, 4, 8, 8}};
      return kind == kCol32 ? PlanDef{16, 3, {4, 16, 16}} : PlanDef{16, 3, {16, 8, 8}};
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
__host__ __device__ constexpr int twiddle_exp(int N, PlanKind kind, int i) {
  const PlanDef d = plan_def(N, kind);
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

// the plan of a line, its positions, twiddles and butterflies
template <int N, class T, bool COL>
struct Stages {
  // (a constexpr array member would be a device constant, loaded at run time:
  // the plan is only ever read through these functions)
  static constexpr PlanKind KIND = COL ? (sizeof(T) == 16 ? kCol64 : kCol32) : (sizeof(T) == 16 ? kRow64 : kRow32);
  static constexpr int V = plan_def(N, KIND).V, S = plan_def(N, KIND).S, L = N / V;
  static_assert(V > 0 && L * V == N, "lanes must divide the line");
  static constexpr int R(int s) { return plan_def(N, KIND).R[s]; }
  static constexpr int Ns(int s) { return plan_ns(plan_def(N, KIND), s); }
  static constexpr int tw_off(int s) {
    int o = 0;
    for (int k = 1; k < s; ++k) o += (R(k) - 1) * Ns(k);
    return o;
  }
  static constexpr int TW = tw_off(S) > 0 ? tw_off(S) : 1;  // table entries (N - R(0))

  // position of value v of lane l before the first forward stage (= after the
  // inverse) and after the last (= before the inverse): lane base + constant
  static constexpr int in_c(int s, int v) { return L * (v / R(s)) + (v % R(s)) * (N / R(s)); }
  static constexpr int first_c(int v) { return in_c(0, v); }
  static constexpr int last_c(int v) { return in_c(S - 1, v); }

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
};

// ================================================================= lines of one wave
// A wave holds NB = 64 / L lines, each on its own L lanes.
template <int N, class T = float2>
struct LaneFft : Stages<N, T, false> {
  using B = Stages<N, T, false>;
  using B::L; using B::S; using B::V; using B::R; using B::Ns; using B::in_c;
  static constexpr int NB = 64 / L;
  static_assert(NB * L == 64, "lanes must divide the wave");

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
      B::template twiddle<FROM, false>(v, tw, l);
      B::template butterflies<FROM, false>(v);
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
      B::template butterflies<FROM - 1, true>(v);
      B::template twiddle<FROM - 1, true>(v, tw, l);
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

// ================================================================= columns of a workgroup
// A tile of CW columns of N points on CW L threads: thread t holds column
// t % CW at lane t / CW, V values.  Values are loaded from and stored to
// memory straight at the positions the first stage reads (a wave's access
// touches 64 / CW rows of 8 CW bytes) or the last stage writes; no staging
// tile.  LDS is only the exchange region, in slots of CW values, and a wave
// holds LW = 64 / CW lanes of every column.
//
// Exchange 0 stays inside the waves: position p of it belongs to the wave
// (p % L) / LW that reads it for stage 1 (lane p % L), and the first stage's
// lanes are dealt out so that the same wave has written it: lane
//   l0 = (i / D) (L / R(0)) + D w + i % D,   D = LW / R(0)
// for place i of wave w.  Each wave's positions form a section of SEC slots;
// exchange 1 keeps a wave's output positions of stage 1 in its own section
// too.  So a forward transform waits for the workgroup before its first
// write (the exchange before may still be read) and once in exchange 1, an
// inverse before and in exchange 1, and nothing else (a fourth stage adds one
// exchange over the whole region, two waits).
// Tiles of one wave (short columns) need no wait at all.
template <int N, class T, int CWX>
struct TileFft : Stages<N, T, true> {
  using B = Stages<N, T, true>;
  using B::L; using B::S; using B::V; using B::R; using B::Ns; using B::in_c;
  static constexpr int CW = CWX * L >= 64 ? CWX : 64 / L;
  static constexpr int THREADS = CW * L, WAVES = THREADS / 64, LW = 64 / CW;
  static constexpr bool ONE = WAVES == 1;
  static constexpr bool SECT = S > 1 && LW % R(0) == 0;
  static constexpr int D = SECT ? LW / R(0) : 1;
  static constexpr int ROWL = LW + D, SEC = V * ROWL;  // a section: V rows of LW positions, padded
  static_assert(THREADS % 64 == 0 && LW * CW == 64, "a wave must hold whole lanes of the tile");
  static_assert(ONE || S < 3 || SECT, "the first radix must divide a wave's lanes");
  // slots of the region: the sections, or (one wave, first radix above its
  // lanes) the positions with one more slot per first-stage butterfly
  static constexpr int SLOTS = S == 1 ? 1 : SECT ? WAVES * SEC : N + N / R(0);
  static constexpr int SMEM = SLOTS * CW;
  // Slot of position p of the exchange after stage s.  Padding: 32 (16 for
  // float64) lanes of an access sit on 32 / CW places, which must fall into
  // distinct rows of banks; written places of exchange 0 are a row of the
  // section or R(0) positions apart, of exchange 1 Ns R(1) positions apart
  // at each Ns-th.
  template <int s>
  __host__ __device__ static constexpr int slot(int pos) {
    const unsigned p = (unsigned)pos;
    constexpr unsigned r0 = R(0);
    if constexpr (s == 0) {
      if constexpr (!SECT) return (int)(p + p / r0);
      const unsigned w = p % L / LW, m = p / L, x = p % LW;
      return (int)(w * SEC + m * ROWL + x + (D > 1 ? x / r0 : 0u));
    } else if constexpr (s == 1 && !ONE) {
      constexpr unsigned blk = LW * R(1), grp = Ns(1) * R(1), pad = Ns(1) < 32 / CW ? Ns(1) : 0;
      static_assert((int)(blk + pad * (blk / grp)) * (V / R(1)) <= SEC, "a wave's stage-1 outputs must fit its section");
      const unsigned b = p / blk, x = p % blk;
      return (int)(b % WAVES * SEC + b / WAVES * (blk + pad * (blk / grp)) + x + x / grp * pad);
    } else {
      return pos;
    }
  }
  // the positions of value v of lane l after stage s (written by the
  // forward), and before stage s + 1 (read): lane part and constant part
  template <int s> __host__ __device__ static constexpr int out_l(int l) {
    constexpr unsigned n = Ns(s), r = R(s);
    return (int)((unsigned)l / n * n * r + (unsigned)l % n);
  }
  template <int s> static constexpr int out_v(int v) {
    constexpr int n = Ns(s), r = R(s);
    return v / r * L * r + v % r * n;
  }
  template <int s> static constexpr int in_v(int v) {
    constexpr int r = R(s + 1);
    return v / r * L + v % r * (N / r);
  }
  __host__ __device__ static constexpr int lane0(int lane) {
    if constexpr (S == 1 || !SECT) return lane;
    constexpr unsigned r0 = R(0);
    const unsigned w = (unsigned)lane / LW, i = (unsigned)lane % LW;
    return (int)(i / D * (L / r0) + D * w + i % D);
  }
  // slots split into lane part and constant, and exchanges 0 and 1 stay in
  // the sections they must
  template <int s>
  static constexpr bool slots_ok() {
    if (s > 1 || (s == 1 && ONE)) return true;  // a slot is its position
    int so[V] = {}, si[V] = {};
    for (int v = 0; v < V; ++v) so[v] = slot<s>(out_v<s>(v)), si[v] = slot<s>(in_v<s>(v));
    for (int l = 0; l < L; ++l) {
      const int ol = out_l<s>(s == 0 ? lane0(l) : l), lo = slot<s>(ol), li = slot<s>(l);
      for (int v = 0; v < V; ++v) {
        const int o = slot<s>(ol + out_v<s>(v)), i = slot<s>(l + in_v<s>(v));
        if (o >= SLOTS || i >= SLOTS || o != lo + so[v] || i != li + si[v]) return false;
        if (!ONE && (o / SEC != l / LW || (s == 0 && i / SEC != l / LW))) return false;
      }
    }
    return true;
  }

  const int col, lane, l0;  // this thread's column of the tile, lane, and lane of the first stage
  T* const lds;             // the exchange region, at this thread's column
  const T* const tw;
  __device__ __forceinline__ TileFft(T* region, const T* tw_)
      : col((int)(threadIdx.x % (unsigned)CW)), lane((int)(threadIdx.x / (unsigned)CW)),
        l0(lane0((int)(threadIdx.x / (unsigned)CW))), lds(region + threadIdx.x % (unsigned)CW), tw(tw_) {}

  __device__ __forceinline__ static void sync() {
    if constexpr (ONE) wave_sync();
    else __syncthreads();
  }
  template <int s, bool IN, bool PUT>
  __device__ __forceinline__ void move(T* v) const {
    static_assert(slots_ok<s>(), "exchange slots must split into lane base and constant, inside their sections");
    T* p = lds + slot<s>(IN ? lane : out_l<s>(s == 0 ? l0 : lane)) * CW;
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const int k = slot<s>(IN ? in_v<s>(e) : out_v<s>(e)) * CW;
      if constexpr (PUT) p[k] = v[e];
      else v[e] = p[k];
    }
  }
  template <int s>
  __device__ __forceinline__ void forward_from(T* v) const {
    B::template twiddle<s, false>(v, tw, lane);
    B::template butterflies<s, false>(v);
    if constexpr (s + 1 < S) {
      if constexpr (s != 1) sync();
      move<s, false, true>(v);
      if constexpr (s == 0) wave_sync();
      else sync();
      move<s, true, false>(v);
      wave_sync();
      forward_from<s + 1>(v);
    }
  }
  // v: values at l0 + first_c -> spectrum at lane + last_c, unnormalized
  __device__ __forceinline__ void forward(T* v) const {
    asm volatile("" ::: "memory");
    forward_from<0>(v);
  }
  template <int s>
  __device__ __forceinline__ void inverse_from(T* v) const {
    B::template butterflies<s, true>(v);
    B::template twiddle<s, true>(v, tw, lane);
    if constexpr (s > 0) {
      if constexpr (s > 1) sync();
      move<s - 1, true, true>(v);
      if constexpr (s > 1) sync();
      else wave_sync();
      move<s - 1, false, false>(v);
      wave_sync();
      inverse_from<s - 1>(v);
    }
  }
  // v: spectrum at lane + last_c -> values at l0 + first_c, unnormalized
  __device__ __forceinline__ void inverse(T* v) const {
    asm volatile("" ::: "memory");
    inverse_from<S - 1>(v);
  }
};

}  // namespace fwix
