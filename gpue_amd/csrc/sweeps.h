// sweeps.h -- fused split-operator sweeps for gfx950.
//
// One "sweep" reads psi once from HBM, applies a chain of 1-D transforms
// along one axis with GPUE's pointwise operators fused between them, and
// writes psi once.  GPUE's step (src/evolution.cu:727-870) maps onto
//   2D: [V/2, FFTx] [FFTy, K, IFFTy] [IFFTx, V/2 (,x-gauge)] (+gauge sweeps)
//   3D: [V/2, FFTx] [FFTy] [FFTz, K, IFFTz] [IFFTy] [IFFTx, V/2 (,x-gauge)] (+gauge)
//   1D: [V/2, FFT, K, IFFT, V/2 (,gauge)]
// The imaginary-time renormalisation (parSum, src/split_op.cu:83-129) is
// fused: the last sweep of a step leaves per-workgroup partial sums of |psi|^2, a
// finalize kernel or every wave of the next step's first sweep reduces them in one
// fixed order to norm = sqrt(sum * dV), and that first sweep divides by it.
// Operator fields are regenerated in-kernel from 1-D coordinate arrays
// (harmonic V, rotation A, standard K) or read from tables (equation-string
// or file fields), so the only per-step HBM traffic is psi itself.
#pragma once
#include <type_traits>

#include "fft_core.h"

namespace gpue {

// V: separable 1-D value tables (harmonic trap + 1/2 m |A|^2 of the rotation gauge)
// or a full table (file / equation fields).  Time-dependent equation fields
// (V_EQN, K_EQN, A_EQN; V_TRAP_A is the harmonic trap plus 1/2 m |A|^2 of a
// time-dependent A, as GPUE builds V after A, src/operators.cu:726-829) are host
// states only: a fill kernel writes their tables before each step (k_fields_at)
// and the sweeps read them as V_TABLE, K_TABLE and A_TABLE.
enum { V_SEP = 0, V_TABLE = 1, V_EQN = 2, V_TRAP_A = 3 };
enum { A_ROTATION = 0, A_ZERO = 1, A_TABLE = 2, A_EQN = 3 };
enum { K_SEP = 0, K_TABLE = 1, K_EQN = 2 };

// Sweep modes: row (x) and strided (y/z) kernels.
// RM_INV_FWD / RM_GAUGE_FWD / CM_GAUGE_FWD: the last sweep of a real-time step
// fused with the first of the next one on the same axis:
// ..., [V/2 of step i+1 (F_HALFV_PRE)], FFT.
// RM_K: FFT, K, IFFT along x (a step that leads with the y axis).
// CM_FWD_V: [scale] [V/2] FFT along y/z (a step that leads with that axis);
// CM_INV_VG: IFFT [V/2] [FFT, A, IFFT] along y/z (its closing sweep).
enum { RM_FWD = 0, RM_INV = 1, RM_GAUGE = 2, RM_FULL = 3, RM_KSUM = 4, RM_INV_FWD = 5, RM_GAUGE_FWD = 6, RM_K = 7 };
enum { CM_FWD = 0, CM_INV = 1, CM_K = 2, CM_GAUGE = 3, CM_KSUM = 4, CM_FWD_V = 5, CM_INV_VG = 6, CM_GAUGE_FWD = 7 };

// Strided-sweep modes that apply an operator (real time runs their bit-16 kernels).
__host__ __device__ inline bool col_phase_mode(int mode) {
  return mode == CM_K || mode == CM_GAUGE || mode == CM_FWD_V || mode == CM_INV_VG || mode == CM_GAUGE_FWD;
}

// Flags of a sweep (runtime-uniform).
enum : unsigned {
  F_SCALE_IN = 1u,     // divide loaded psi by *norm_in (pending renormalisation)
  F_HALFV_PRE = 2u,    // V/2 (+ nonlinearity) before the first transform
  F_HALFV_POST = 4u,   // V/2 (+ nonlinearity) after the inverse transform
  F_GAUGE_POST = 8u,   // extra [FFT, A_axis, IFFT] after the post op
  F_NORM = 16u,        // accumulate |psi_out|^2 and produce norm_out
  F_SCALE_PART = 32u,  // with F_SCALE_IN: the norm is reduced here from the previous
                       // sweep's partials (norm_nb of them), and block 0 stores it
                       // to norm_out, instead of a separate finalize
  F_DEFER = 64u,       // host only: the finalize of this F_NORM sweep is left to
                       // the next sweep (F_SCALE_PART)
  F_ASUM = 128u,       // KSUM modes: weight A_axis * k_axis (the gauge term of the
                       // evolved Hamiltonian) instead of K
  F_KAX = 256u,        // KSUM modes: weight ks[axis][k_axis], this axis's part of a
                       // separable K (Parseval along the other axes needs no transform)
};

// Time-dependent equation program (postfix): CONST pushes val, X/Y/Z/T push a
// coordinate, OP+k pops (a, b) and pushes GPUE operator k (src/dynamic.cu:568-600);
// EQ_UNI marks an op whose result is the same at every point (no x, y, z below it).
enum : int { EQ_CONST = 0, EQ_X = 1, EQ_Y = 2, EQ_Z = 3, EQ_T = 4, EQ_OP = 16, EQ_UNI = 64 };
constexpr int EQ_MAX = 48;
constexpr int EQ_REG_DEPTH = 8;   // largest stack of a time-dependent program (k_fields_at)
struct EqnProg {
  int n;
  int depth;   // largest stack depth the program reaches
  int op[EQ_MAX];
  double val[EQ_MAX];
};

struct Phys {
  int xDim, yDim, zDim, dimnum;
  int gstate, gpe;
  int v_kind, a_kind, k_kind;
  double cV;      // Dt / (2 hbar)          (GV/EV exponent, src/operators.cu:1081,1100)
  double cH;      // (0.5*Dt) / hbar        (cMultDensity, src/kernels.cu:372)
  double g;       // interaction * gDenConst
  double cK;      // Dt / hbar              (GK/EK, src/operators.cu:1082,1102)
  double Dt;      // gauge exponent scale   (GpA/EpA, src/operators.cu:1093-1110)
  double omega, omegaX, omegaY;
  const double *xg, *yg, *zg, *pxg, *pyg, *pzg;
  const double *vs[3];   // V_SEP: V = vs[0][x] + vs[1][y] + vs[2][z]
  const double *ks[3];   // K_SEP: K = ks[0][kx] + ks[1][ky] + ks[2][kz]
  const double *kf[3];   // K_SEP: per-axis factors of the K operator for this gstate,
                         // interleaved (re, im): exp(-K_a Dt/hbar) or exp(-i K_a Dt/hbar)
  const float *vsf[3];   // FP32 contexts: vs and kf rounded to FP32 once (the FP32
  const float *kff[3];   // sweeps read these; null for FP64 contexts)
  const double *Vt, *Kt, *At[3];
  const double* Vt_next;  // V table of the next step's first V/2 (bridge sweeps; Vt unless V depends on time)
};

struct SweepArgs {
  int active;         // batched launches: 0 skips this instance
  const void* in;
  void* out;
  const void* tw;
  Phys ph;
  int lines;          // row sweeps: yDim*zDim
  int axis;           // 0 x (row), 1 y, 2 z
  int gauge_axis;     // axis of the A operator applied by F_GAUGE_POST / gauge modes
  unsigned flags;
  double invN;        // normalisation folded into K (1/N) or A (1/n_axis)
  const double* norm_in;   // pending renormalisation divisor (F_SCALE_IN)
  double* partials;        // per-workgroup partial sums (F_NORM, KSUM modes)
  int norm_nb;             // F_SCALE_PART: partials of the previous sweep
  double norm_scale;       // F_SCALE_PART: dV
  double* norm_out;        // F_SCALE_PART: where block 0 stores the norm
};

// Of three scalar arguments the one of axis a, by value (an index or a select of
// addresses would keep the arguments in memory).
template <typename U>
__device__ __forceinline__ U pick(int a, U x, U y, U z) { return a == 0 ? x : a == 1 ? y : z; }

// ---------------------------------------------------------------------------
// Field evaluation (GPUE operators.cu kernels restated per point)
// ---------------------------------------------------------------------------
__device__ __forceinline__ double A_val(const Phys& p, int axis, int xi, int yi, int zi, long gid) {
  if (p.a_kind == A_ROTATION) {           // krotation_Ax/Ay, kconstant_A (:630-647, :621-627)
    if (axis == 0) return -p.yg[yi] * p.omega * p.omegaX;
    if (axis == 1) return p.xg[xi] * p.omega * p.omegaY;
    return 0.0;
  }
  if (p.a_kind == A_ZERO) return 0.0;
  return pick(axis, p.At[0], p.At[1], p.At[2])[gid];
}

// kharmonic_V (src/operators.cu:994-1008) is a sum of per-axis terms once the
// rotation gauge is written out (Ax = Ax(y), Ay = Ay(x), Az = 0), so it is
// carried as three 1-D tables; other fields are full tables.
__device__ __forceinline__ double V_val(const Phys& p, int xi, int yi, int zi, long gid) {
  if (p.v_kind == V_SEP) return p.vs[0][xi] + p.vs[1][yi] + p.vs[2][zi];
  return p.Vt[gid];
}

// simple_K (src/operators.cu:460-469): hbar^2/(2m) (kx^2 + ky^2 + kz^2)
__device__ __forceinline__ double K_val(const Phys& p, int xi, int yi, int zi, long gid) {
  if (p.k_kind == K_SEP) return p.ks[0][xi] + p.ks[1][yi] + p.ks[2][zi];
  return p.Kt[gid];
}

__device__ __forceinline__ long gid_of(const Phys& p, int xi, int yi, int zi) {
  return (long)xi + (long)p.xDim * ((long)yi + (long)p.yDim * (long)zi);
}

// FP64 exp and sincos for the fused operators.  The library versions carry
// general special-case handling that dominates the cost of the V/2 sweeps; here
// the arguments are finite and moderate, so a short form suffices:
// Cody-Waite argument reduction (W. J. Cody and W. Waite, "Software Manual for
// the Elementary Functions", 1980) followed by the Taylor polynomial of the
// reduced argument in Horner form.  The split constants are ln 2 and pi/2
// rounded to 42 and 3x33 significant bits, so k*C_hi is exact for every k that
// occurs.  exp: |r| <= ln2/2, degree 13 (truncation < 5e-18 relative).
// sin/cos: |r| <= pi/4, degrees 17 and 18 (truncation < 1e-19).  Arguments
// outside |x| < 2^20 (sincos) go to the library; NaN propagates.
namespace fm {
constexpr double LN2_HI = 0.6931471805598903;
constexpr double LN2_LO = 5.497923018708371e-14;
constexpr double INV_LN2 = 1.4426950408889634;
constexpr double PIO2_1 = 1.5707963267341256;
constexpr double PIO2_2 = 6.077100506303966e-11;
constexpr double PIO2_3 = 2.0222662487959506e-21;
constexpr double TWO_OVER_PI = 0.6366197723675814;
// 1/k!
constexpr double F2 = 0.5, F3 = 0.16666666666666666, F4 = 0.041666666666666664, F5 = 0.008333333333333333,
                 F6 = 0.001388888888888889, F7 = 0.0001984126984126984, F8 = 2.48015873015873e-05,
                 F9 = 2.7557319223985893e-06, F10 = 2.755731922398589e-07, F11 = 2.505210838544172e-08,
                 F12 = 2.08767569878681e-09, F13 = 1.6059043836821613e-10, F14 = 1.1470745597729725e-11,
                 F15 = 7.647163731819816e-13, F16 = 4.779477332387385e-14, F17 = 2.8114572543455206e-15,
                 F18 = 1.5619206968586225e-16;
}  // namespace fm

__device__ __forceinline__ double exp_cw(double x) {
  using namespace fm;
  x = x < -750.0 ? -750.0 : x;   // below -745.14 the result rounds to 0; comparisons keep NaN
  x = x > 710.0 ? 710.0 : x;
  const double k = rint(x * INV_LN2);
  double r = fma(-k, LN2_HI, x);
  r = fma(-k, LN2_LO, r);
  double p = F13;
  p = fma(p, r, F12); p = fma(p, r, F11); p = fma(p, r, F10); p = fma(p, r, F9); p = fma(p, r, F8);
  p = fma(p, r, F7); p = fma(p, r, F6); p = fma(p, r, F5); p = fma(p, r, F4); p = fma(p, r, F3);
  p = fma(p, r, F2); p = fma(p, r, 1.0); p = fma(p, r, 1.0);
  return ldexp(p, (int)k);
}

// |x| <= 1/32: Taylor polynomials without a reduction (the V/2 phases of
// real time and most imaginary-time exponents are this small); the first
// omitted terms, x^9/9! and r^9/9!, r^10/10!, are below 1e-18 relative.
constexpr double SMALL_ARG = 0.03125;
__device__ __forceinline__ double exp_small(double x) {
  using namespace fm;
  double p = F8;
  p = fma(p, x, F7); p = fma(p, x, F6); p = fma(p, x, F5); p = fma(p, x, F4); p = fma(p, x, F3);
  p = fma(p, x, F2); p = fma(p, x, 1.0);
  return fma(p, x, 1.0);
}
__device__ __forceinline__ void sincos_small(double r, double* sn_out, double* cs_out) {
  using namespace fm;
  const double z = r * r;
  double ps = -F7;
  ps = fma(ps, z, F5); ps = fma(ps, z, -F3);
  *sn_out = fma(r * z, ps, r);            // r - r^3/3! + r^5/5! - r^7/7!
  double pc = F8;
  pc = fma(pc, z, -F6); pc = fma(pc, z, F4); pc = fma(pc, z, -F2);
  *cs_out = fma(z, pc, 1.0);              // 1 - r^2/2! + ... + r^8/8!
}

// sin and cos of |r| <= pi/4 (no reduction)
__device__ __forceinline__ void sincos_poly(double r, double* sn_out, double* cs_out) {
  using namespace fm;
  const double z = r * r;
  double ps = -F17;
  ps = fma(ps, z, F15); ps = fma(ps, z, -F13); ps = fma(ps, z, F11); ps = fma(ps, z, -F9);
  ps = fma(ps, z, F7); ps = fma(ps, z, -F5); ps = fma(ps, z, F3);
  const double sn = fma(-r * z, ps, r);   // r - r^3/3! + ...
  double pc = F18;
  pc = fma(pc, z, -F16); pc = fma(pc, z, F14); pc = fma(pc, z, -F12); pc = fma(pc, z, F10);
  pc = fma(pc, z, -F8); pc = fma(pc, z, F6); pc = fma(pc, z, -F4); pc = fma(pc, z, F2);
  const double cs = fma(-z, pc, 1.0);     // 1 - r^2/2! + ...
  *sn_out = sn;
  *cs_out = cs;
}

// core for |x| < 2^20 (no branch, so the polynomial chains of several points
// can be interleaved); sincos_cw adds the library path for other arguments
__device__ __forceinline__ void sincos_core(double x, double* s, double* c) {
  using namespace fm;
  const double q = rint(x * TWO_OVER_PI);
  double r = fma(-q, PIO2_1, x);
  r = fma(-q, PIO2_2, r);
  r = fma(-q, PIO2_3, r);
  double sn, cs;
  sincos_poly(r, &sn, &cs);
  const int n = ((int)q) & 3;
  const double s0 = (n & 1) ? cs : sn, c0 = (n & 1) ? sn : cs;
  *s = (n & 2) ? -s0 : s0;
  *c = ((n + 1) & 2) ? -c0 : c0;
}

__device__ __forceinline__ bool sincos_small_ok(double x) { return fabs(x) <= 0.78539816339744828; }

__device__ __forceinline__ bool sincos_fast_ok(double x) { return fabs(x) < 1048576.0; }

__device__ __forceinline__ void sincos_cw(double x, double* s, double* c) {
  if (!sincos_fast_ok(x)) {   // large, infinite or NaN: library
    sincos(x, s, c);
    return;
  }
  sincos_core(x, s, c);
}

// FP32 sincos in the same form: pi/2 split into 12+12 significant bits and a
// rounded tail (q*P1, q*P2 exact for |q| < 2^12), Taylor degrees 9 and 10 on
// |r| <= pi/4 (truncation < 2e-9, below FP32 rounding); |x| >= 6000, infinities
// and NaN go to the library.
__device__ __forceinline__ void sincos_poly(float r, float* sn_out, float* cs_out) {
  const float z = r * r;
  float ps = 2.7557318844628753e-06f;
  ps = fmaf(ps, z, -0.00019841270113829523f);
  ps = fmaf(ps, z, 0.008333333767950535f);
  ps = fmaf(ps, z, -0.1666666716337204f);
  const float sn = fmaf(r * z, ps, r);
  float pc = -2.755731998149713e-07f;
  pc = fmaf(pc, z, 2.4801587642286904e-05f);
  pc = fmaf(pc, z, -0.0013888889225199819f);
  pc = fmaf(pc, z, 0.0416666679084301f);
  pc = fmaf(pc, z, -0.5f);
  const float cs = fmaf(z, pc, 1.0f);
  *sn_out = sn;
  *cs_out = cs;
}

__device__ __forceinline__ void sincos_core(float x, float* s, float* c) {
  const float q = rintf(x * 0.6366197466850281f);
  float r = fmaf(-q, 1.57080078125f, x);
  r = fmaf(-q, -4.453584551811218e-06f, r);
  r = fmaf(-q, -8.705515752716053e-10f, r);
  float sn, cs;
  sincos_poly(r, &sn, &cs);
  const int n = ((int)q) & 3;
  const float s0 = (n & 1) ? cs : sn, c0 = (n & 1) ? sn : cs;
  *s = (n & 2) ? -s0 : s0;
  *c = ((n + 1) & 2) ? -c0 : c0;
}

__device__ __forceinline__ bool sincos_small_ok(float x) { return fabsf(x) <= 0.78539816f; }

__device__ __forceinline__ bool sincos_fast_ok(float x) { return fabsf(x) < 6000.0f; }

__device__ __forceinline__ void sincos_cw(float x, float* s, float* c) {
  if (!sincos_fast_ok(x)) {
    sincosf(x, s, c);
    return;
  }
  sincos_core(x, s, c);
}

// exp and sincos of the verification entry (gpue_math_eval) and of the library
// fallback.
template <typename T>
struct WMath;
template <>
struct WMath<double> {
  static __device__ __forceinline__ double ex(double a) { return exp_cw(a); }
  static __device__ __forceinline__ void sc(double a, double* s, double* c) { sincos_cw(a, s, c); }
};
template <>
struct WMath<float> {
  // hardware exp2 of a*log2(e) (__expf): the FP32 step rounds its operands to
  // FP32 anyway, and |a| stays small (V dt/2, K dt), so the product's rounding
  // adds |a|*2^-24 relative
  static __device__ __forceinline__ float ex(float a) { return __expf(a); }
  static __device__ __forceinline__ void sc(float a, float* s, float* c) { sincos_cw(a, s, c); }
};

// ---------------------------------------------------------------------------
// Pointwise operators on the E points a lane holds of a line.
//
// Each operator comes in two parts: load() gathers what it needs from tables,
// and the rest computes.  Sweeps of small grids are a serial chain (a 512^2 FP64
// sweep is half a wave per SIMD; its waves waited 60 % of their life), so the
// variants for them issue every load() of the sweep at its start, next to psi's
// own, and derive factors that do not depend on psi while psi is on its way;
// a load left to its place of use costs a further memory round trip of 0.5-1 us
// in a sweep of 4-10 us.  At 512^2 FP64 with rotation (4 MiB psi, 32-step graphs)
// loading up front took the step from 29.6 to 26.9 us in imaginary and from 26.2 to
// 23.5 us in real time (sweeps 6.3-9.5 -> 6.1-8.9 and 6.4-10.9 -> 6.1-9.6 us), the
// 256^2 step without rotation from 14.2 to 12.7 and from 9.8 to 8.8 us.  Sweeps of
// large grids load at the place of use (other waves cover the wait, registers are
// what they lack).
//
// The arithmetic runs in the working precision T: FP64 sweeps in double; FP32
// sweeps in float, with table values held in double rounded once.  Reductions,
// gauge factors and real-time phase factors stay in FP64 in the FP32 form.
// ---------------------------------------------------------------------------
// Marks loaded values as needed from here on.  Without it the compiler moves their
// first arithmetic up to the loads (a sum of two table values next to them), and its
// wait stands in front of every later load.
template <typename U>
__device__ __forceinline__ void arrive(U& x) { asm volatile("" : "+v"(x)); }
template <typename U>
__device__ __forceinline__ void arrive(cx<U>& x) {
  arrive(x.x);
  arrive(x.y);
}

// A scaled point, rounded here: contracted into the butterfly that follows it, results
// would depend on what the compiler sees next to each other.
template <typename T>
__device__ __forceinline__ cx<T> scaled(cx<T> v, T s) {
  cx<T> r = cscale(v, s);
  arrive(r);
  return r;
}

// A line of N points along axis ax: element e at flat index base + e*es; i0, i1:
// the indices on the other two axes, in ascending order.  The lane holds points
// tid + bpos(0, r).
struct LineAt {
  int ax, tid;
  long base, es;
  int i0, i1;
  __device__ __forceinline__ int o0() const { return ax == 0 ? 1 : 0; }
  __device__ __forceinline__ int o1() const { return ax == 2 ? 1 : 2; }
};

template <typename T>
struct VTab;
template <>
struct VTab<double> {
  static __device__ __forceinline__ const double* get(const Phys& p, int a) { return pick(a, p.vs[0], p.vs[1], p.vs[2]); }
};
template <>
struct VTab<float> {
  static __device__ __forceinline__ const float* get(const Phys& p, int a) { return pick(a, p.vsf[0], p.vsf[1], p.vsf[2]); }
};

// v times the phase (cs, sn) and s: see apply_phase_all.
template <typename T>
__device__ __forceinline__ cx<T> times_phase(cx<T> v, T cs, T sn, double s_) {
  if constexpr (sizeof(T) == 8) {
    return cmul(mk(cs * s_, sn * s_), v);
  } else {
    const double c0 = cs, d0 = sn;
    const double f = fma(-0.5, fma(c0, c0, d0 * d0), 1.5) * s_;
    const cx<double> w = cmul(mk(c0 * f, d0 * f), mk((double)v.x, (double)v.y));
    return mk((float)w.x, (float)w.y);
  }
}

// E points whose arguments may need the library (huge, infinite, NaN): one at a time,
// the arrays rotating through their first slot, so that the kernel holds one copy of the
// library code instead of E (they made up most of a sweep's 36-107 KB) and no array is
// indexed by a variable.  The factors ...
template <typename T, int E>
__device__ __forceinline__ void sincos_any(T (&x)[E], T (&sn)[E], T (&cs)[E]) {
#pragma unroll
  for (int r = 0; r < E; ++r) sn[r] = cs[r] = (T)0;
#pragma unroll 1
  for (int k = 0; k < E; ++k) {
    T s, c;
    WMath<T>::sc(x[0], &s, &c);
#pragma unroll
    for (int r = 0; r + 1 < E; ++r) {
      x[r] = x[r + 1];
      sn[r] = sn[r + 1];
      cs[r] = cs[r + 1];
    }
    sn[E - 1] = s;
    cs[E - 1] = c;
  }
}
// ... or the points times their phases.
template <typename T, int E>
__device__ __forceinline__ void phase_any(cx<T>* v, T (&x)[E], double s) {
#pragma unroll 1
  for (int k = 0; k < E; ++k) {
    T sn, cs;
    WMath<T>::sc(x[0], &sn, &cs);
    const cx<T> u = times_phase(v[0], cs, sn, s);
#pragma unroll
    for (int r = 0; r + 1 < E; ++r) {
      x[r] = x[r + 1];
      v[r] = v[r + 1];
    }
    v[E - 1] = u;
  }
}

// psi * exp(-arg) (imaginary time) or psi * exp(-i arg) (REAL), times s.
// FP64: a lane whose arguments are all small takes the short polynomials.
// FP32 real time: the phase factor is formed in FP32, then its modulus is
// corrected in FP64 by one Newton step towards 1/sqrt(c^2 + s^2), and the
// product is formed in FP64 and rounded to FP32 once.  A factor rounded to FP32
// carries a modulus error of ~1e-7 that is the same at every step for static V,
// A and K, so the norm and energy would drift linearly with the steps; after the
// Newton step the modulus is 1 within ~1e-14, and what is left (the FP32 phase,
// ~1e-7 relative) acts like a rounded V and does not grow.
// AHEAD (real time): all factors before the first product, for serial chains with
// registers to spare (line_body, and sweeps of small grids with up to 8 points a lane).
// Elsewhere each branch finishes its points: factors kept across the join, and through the
// loop of the library branch, are 4 registers a point, which left FP64 lanes of 16 points
// one wave per SIMD and made 1024-lane workgroups spill (real time, us a step, with / without:
// 384 x 4096 FP32 69 / 46, 1024 x 4096 FP64 107 / 81, 64 x 64 x 512 FP64 61.6 / 54.9; the other
// way a line of 4096 points takes 8.4 / 10.1, one of 1024 3.19 / 3.27, 384^2 loses 1 %).
template <typename T, int E, bool REAL, bool AHEAD>
__device__ __forceinline__ void apply_phase_all(cx<T>* v, const T (&arg)[E], double s_) {
  const T s = (T)s_;
  if constexpr (!REAL) {
    if constexpr (sizeof(T) == 8) {
      bool tiny = true;
#pragma unroll
      for (int r = 0; r < E; ++r) tiny = tiny && fabs(arg[r]) <= SMALL_ARG;
      if (tiny) {
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = scaled(v[r], exp_small(-arg[r]) * s);
        return;
      }
    }
#pragma unroll
    for (int r = 0; r < E; ++r) v[r] = scaled(v[r], WMath<T>::ex(-arg[r]) * s);
  } else {
    // one range check for the lane's E arguments, then branch-free forms
    T x[E];
    bool small = true, fast = true;
#pragma unroll
    for (int r = 0; r < E; ++r) {
      x[r] = -arg[r];
      small = small && (sizeof(T) == 8 ? fabs((double)x[r]) <= SMALL_ARG : sincos_small_ok(x[r]));
      fast = fast && sincos_fast_ok(x[r]);
    }
    if constexpr (AHEAD) {
      T sn[E], cs[E];
      if (small) {
#pragma unroll
        for (int r = 0; r < E; ++r) {
          if constexpr (sizeof(T) == 8) sincos_small(x[r], &sn[r], &cs[r]);
          else sincos_poly(x[r], &sn[r], &cs[r]);
        }
      } else if (fast) {
#pragma unroll
        for (int r = 0; r < E; ++r) sincos_core(x[r], &sn[r], &cs[r]);
      } else {
        sincos_any<T, E>(x, sn, cs);
      }
#pragma unroll
      for (int r = 0; r < E; ++r) v[r] = times_phase(v[r], cs[r], sn[r], s_);
    } else if (small) {
#pragma unroll
      for (int r = 0; r < E; ++r) {
        T sn, cs;
        if constexpr (sizeof(T) == 8) sincos_small(x[r], &sn, &cs);
        else sincos_poly(x[r], &sn, &cs);
        v[r] = times_phase(v[r], cs, sn, s_);
      }
    } else if (fast) {
#pragma unroll
      for (int r = 0; r < E; ++r) {
        T sn, cs;
        sincos_core(x[r], &sn, &cs);
        v[r] = times_phase(v[r], cs, sn, s_);
      }
    } else {
      phase_any<T, E>(v, x, s_);
    }
  }
}

// V/2 with the nonlinear density term: cMultDensity (src/kernels.cu:365-388)
// with GV/EV (src/operators.cu:1081,1100) merged into one exponential.
template <typename T, int N, int TPL, int R, int E>
struct VOp {
  T e[E], f0, f1;   // V = e + (f0 + f1): the line's own axis and the other two; a table: e
  // no branch joins around the FP64 loads and f0, f1: a join copies registers, which
  // waits for the values there
  __device__ __forceinline__ void load(const Phys& p, const double* __restrict__ Vt, const LineAt& l) {
    const bool sep = p.v_kind == V_SEP;
    f0 = VTab<T>::get(p, l.o0())[l.i0];
    f1 = VTab<T>::get(p, l.o1())[l.i1];
    const double* vt = Vt + l.base + (long)l.tid * l.es;
    if constexpr (sizeof(T) == 8) {
      const double* ve = sep ? VTab<T>::get(p, l.ax) + l.tid : vt;
      const long es = sep ? 1 : l.es;
#pragma unroll
      for (int r = 0; r < E; ++r) e[r] = ve[bpos<N, TPL, R>(0, r) * es];
    } else if (sep) {
      const T* ve = VTab<T>::get(p, l.ax) + l.tid;
#pragma unroll
      for (int r = 0; r < E; ++r) e[r] = ve[bpos<N, TPL, R>(0, r)];
    } else {
#pragma unroll
      for (int r = 0; r < E; ++r) e[r] = (T)vt[bpos<N, TPL, R>(0, r) * l.es];
    }
  }
  __device__ __forceinline__ void ready() {
    arrive(f0);
    arrive(f1);
#pragma unroll
    for (int r = 0; r < E; ++r) arrive(e[r]);
  }
  // exponents of the half step on v.  FP32 adds the axes in the order x, y, z, and the
  // density takes the square of x after that of y in a step's first half, before it in
  // its second (CLOSES).  The order is fixed so that every kernel rounds alike; V cV is
  // rounded before the density term for the same reason.
  template <bool CLOSES>
  __device__ __forceinline__ void args(const Phys& p, const LineAt& l, const cx<T>* v, T (&arg)[E]) const {
    const T cV = (T)p.cV;
    if constexpr (sizeof(T) == 8) {
      const T f = p.v_kind == V_SEP ? f0 + f1 : (T)0;
#pragma unroll
      for (int r = 0; r < E; ++r) arg[r] = (e[r] + f) * cV;
    } else if (p.v_kind == V_SEP) {
#pragma unroll
      for (int r = 0; r < E; ++r) arg[r] = (l.ax == 2 ? (f0 + f1) + e[r] : (e[r] + f0) + f1) * cV;
    } else {
#pragma unroll
      for (int r = 0; r < E; ++r) arg[r] = e[r] * cV;
    }
    if (p.gpe) {
      const T g = (T)p.g, cH = (T)p.cH;
#pragma unroll
      for (int r = 0; r < E; ++r) {
        arrive(arg[r]);   // rounded before the sum
        const T d = CLOSES ? fma(v[r].x, v[r].x, v[r].y * v[r].y) : fma(v[r].y, v[r].y, v[r].x * v[r].x);
        arg[r] = fma(g * d, cH, arg[r]);
      }
    }
  }
  template <bool REAL, bool CLOSES, bool AHEAD>
  __device__ __forceinline__ void half(const Phys& p, const LineAt& l, cx<T>* v) const {
    T arg[E];
    args<CLOSES>(p, l, v, arg);
    apply_phase_all<T, E, REAL, AHEAD>(v, arg, 1.0);
  }
};

// The gauge operator along the line's axis: GpA*/EpA* (src/operators.cu:1089-1110)
// with both 1/sqrt(n) of the axis transforms folded into invn.
//
// The rotation gauge on a line along x (A_x = -y omega omegaX) or y (A_y = x omega
// omegaY) is constant along the line, so the point of signed wave-number index m
// is multiplied by exp(-a m) (imaginary time) or exp(-i a m) (real time), a = A dk
// Dt, dk = k[1].  In the boundary layout of radix R a lane holds the points
// tid + TPL q + (N/R) s (r = q R + s), less N from the Nyquist index on, so the E
// factors are products of four per-lane factors and their powers: exp(-a tid),
// exp(-a N/R), exp(-a TPL) and exp(a N), i.e. three or four exponentials per lane
// instead of E (each product adds a rounding: a few ulp).  Other gauges, FP32, or an
// |a| N large enough for exp(a N) to leave the double range take E exponentials.
template <typename T, int N, int TPL, int R, int E, bool REAL>
struct GOp {
  static constexpr int Q = E / R, NR = N / R;
  static constexpr bool LIN = sizeof(T) == 8;
  double A, dk;
  bool lin;
  cx<double> b, W, U, Z;   // imaginary time: real factors, in .x
  T at[E], kk[E];          // not lin: A and k of the points
  __device__ __forceinline__ void load_points(const Phys& p, const LineAt& l) {
    const double* kt = pick(l.ax, p.pxg, p.pyg, p.pzg) + l.tid;
    const double* ap = pick(l.ax, p.At[0], p.At[1], p.At[2]) + l.base + (long)l.tid * l.es;
#pragma unroll
    for (int r = 0; r < E; ++r) kk[r] = (T)kt[bpos<N, TPL, R>(0, r)];
    if (p.a_kind == A_TABLE) {
#pragma unroll
      for (int r = 0; r < E; ++r) at[r] = (T)ap[bpos<N, TPL, R>(0, r) * l.es];
    }
  }
  __device__ __forceinline__ void load(const Phys& p, const LineAt& l) {
    A = pick(l.ax, p.yg, p.xg, p.xg)[l.i0];   // the rotation's coordinate (A_z = 0)
    dk = pick(l.ax, p.pxg, p.pyg, p.pzg)[1];
  }
  __device__ __forceinline__ void prep(const Phys& p, const LineAt& l, double invn) {
    A = A * pick(l.ax, -p.omega, p.omega, p.omega) * pick(l.ax, p.omegaX, p.omegaY, p.omegaY);
    A = p.a_kind == A_ROTATION && l.ax < 2 ? A : 0.0;
    const double a = A * dk * p.Dt;
    lin = LIN && p.a_kind != A_TABLE && fabs(a) * N <= 600.0;
    if constexpr (!LIN) return;
    if constexpr (!REAL) {
      b.x = exp_cw(-a * l.tid) * invn;
      W.x = exp_cw(-a * NR);
      Z.x = exp_cw(a * N);
      if constexpr (Q > 1) U.x = exp_cw(-a * TPL);
    } else {
      auto ph = [](double x) {   // exp(-i x)
        double sn, cs;
        sincos_core(x, &sn, &cs);
        return mk(cs, -sn);
      };
      const cx<double> b0 = ph(a * l.tid);
      b = mk(b0.x * invn, b0.y * invn);
      W = ph(a * NR);
      Z = ph(-a * N);
      if constexpr (Q > 1) U = ph(a * TPL);
    }
  }
  __device__ __forceinline__ void apply_lin(cx<T>* v, const LineAt& l) const {
    cx<double> w[R];
    w[0] = b;
#pragma unroll
    for (int k = 1; k < R; ++k) {
      if constexpr (REAL) w[k] = cmul(w[k - 1], W);
      else w[k].x = w[k - 1].x * W.x;
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const int r = q * R + k;
        const bool wrap = l.tid + TPL * q + NR * k >= N / 2;
        if constexpr (REAL) v[r] = cmul(wrap ? cmul(w[k], Z) : w[k], v[r]);
        else v[r] = scaled(v[r], wrap ? w[k].x * Z.x : w[k].x);
      }
      if (q + 1 < Q) {
#pragma unroll
        for (int k = 0; k < R; ++k) {
          if constexpr (REAL) w[k] = cmul(w[k], U);
          else w[k].x *= U.x;
        }
      }
    }
  }
  // `early`: load_points() was called up front where A is a table
  template <bool AHEAD>
  __device__ __forceinline__ void apply(const Phys& p, cx<T>* v, const LineAt& l, double invn, bool early) {
    if constexpr (LIN) {
      if (lin) {
        apply_lin(v, l);
        return;
      }
    }
    if (!(early && p.a_kind == A_TABLE)) load_points(p, l);
    T arg[E];
    const T Dt = (T)p.Dt;
#pragma unroll
    for (int r = 0; r < E; ++r) arg[r] = (p.a_kind == A_TABLE ? at[r] : (T)A) * kk[r] * Dt;
    apply_phase_all<T, E, REAL, AHEAD>(v, arg, invn);
  }
};

// K step: GK/EK (src/operators.cu:1082,1102) with both 1/sqrt(N) of
// src/evolution.cu:761,777 folded into invN.  For the separable K the operator
// is the product of per-axis factors (no transcendental per point): the other
// two axes' product times the line's own.  FP32 real time reads the FP64 tables
// and forms the product in FP64 (see apply_phase_all).
template <typename T, int N, int TPL, int R, int E, bool REAL>
struct KOp {
  using F = typename std::conditional<REAL, double, T>::type;
  cx<F> e[E], f0, f1;   // imaginary time: real factors, in .x; K tables: K itself in e.x
  static __device__ __forceinline__ const F* tab(const Phys& p, int a) {
    if constexpr (sizeof(F) == 4) return pick(a, p.kff[0], p.kff[1], p.kff[2]);
    else return pick(a, p.kf[0], p.kf[1], p.kf[2]);
  }
  static __device__ __forceinline__ cx<F> one(const F* t, int i) {
    return mk(t[2 * i], REAL ? t[2 * i + 1] : (F)0);
  }
  __device__ __forceinline__ void load(const Phys& p, const LineAt& l) {
    f0 = one(tab(p, l.o0()), l.i0);
    f1 = one(tab(p, l.o1()), l.i1);
    if (p.k_kind == K_SEP) {
      const F* t = tab(p, l.ax) + 2 * l.tid;
#pragma unroll
      for (int r = 0; r < E; ++r) e[r] = one(t, bpos<N, TPL, R>(0, r));
    } else {
      const double* kt = p.Kt + l.base + (long)l.tid * l.es;
#pragma unroll
      for (int r = 0; r < E; ++r) e[r] = mk((F)kt[bpos<N, TPL, R>(0, r) * l.es], (F)0);
    }
  }
  __device__ __forceinline__ void ready() {
    arrive(f0);
    arrive(f1);
#pragma unroll
    for (int r = 0; r < E; ++r) arrive(e[r]);
  }
  // A separable K: f0 f1 and 1/N once, then a factor a point.  FP32 imaginary time
  // multiplies the axes' factors in the order x, y, z.
  struct Sep {
    cx<F> f0, f1, f;
    double invN;
    bool z;
    __device__ __forceinline__ Sep(const LineAt& l, cx<F> f0_, cx<F> f1_, double invN_)
        : f0(f0_), f1(f1_), invN(invN_), z(l.ax == 2) {
      if constexpr (REAL) f = cscale(cmul(f0, f1), invN);
      else f = mk(f0.x * f1.x * (F)invN, (F)0);
    }
    __device__ __forceinline__ cx<T> operator()(cx<F> e, cx<T> v) const {
      if constexpr (REAL) {
        const cx<double> u = cmul(cmul(e, f), mk((double)v.x, (double)v.y));
        return mk((T)u.x, (T)u.y);
      } else if constexpr (sizeof(T) == 8) {
        return scaled(v, e.x * f.x);
      } else {
        return scaled(v, (z ? f0.x * f1.x * e.x : e.x * f0.x * f1.x) * (T)invN);
      }
    }
  };
  // on factors loaded up front
  template <bool AHEAD>
  __device__ __forceinline__ void apply(const Phys& p, const LineAt& l, cx<T>* v, double invN) const {
    if (p.k_kind == K_SEP) {
      const Sep k(l, f0, f1, invN);
#pragma unroll
      for (int r = 0; r < E; ++r) v[r] = k(e[r], v[r]);
    } else {
      T arg[E];
      const T cK = (T)p.cK;
#pragma unroll
      for (int r = 0; r < E; ++r) arg[r] = (T)e[r].x * cK;
      apply_phase_all<T, E, REAL, AHEAD>(v, arg, invN);
    }
  }
  // Real time, loads included, each next to its use: held together, the factors take 4
  // registers a point, and the widest workgroups spilled.  (Imaginary time has 2 a point,
  // and gains 1-9 % from loading them together.)
  static __device__ __forceinline__ void load_apply(const Phys& p, const LineAt& l, cx<T>* v, double invN) {
    if (p.k_kind == K_SEP) {
      const Sep k(l, one(tab(p, l.o0()), l.i0), one(tab(p, l.o1()), l.i1), invN);
      const F* t = tab(p, l.ax) + 2 * l.tid;
#pragma unroll
      for (int r = 0; r < E; ++r) v[r] = k(one(t, bpos<N, TPL, R>(0, r)), v[r]);
    } else {
      const double* kt = p.Kt + l.base + (long)l.tid * l.es;
      T arg[E];
      const T cK = (T)p.cK;
#pragma unroll
      for (int r = 0; r < E; ++r) arg[r] = (T)kt[bpos<N, TPL, R>(0, r) * l.es] * cK;
      apply_phase_all<T, E, REAL, false>(v, arg, invN);
    }
  }
};

// ---------------------------------------------------------------------------
// Deterministic two-stage reduction of NA doubles: every workgroup writes its
// partial sums (plain stores, no fences), a one-workgroup finalize kernel
// launched after it sums them in a fixed order.  The result is the same for
// every run and independent of scheduling.
// ---------------------------------------------------------------------------
// Sum over the lanes of a wave (xor 1, 2, 4, 8 by DPP within rows of 16: once two
// groups hold their own totals, mirroring pairs them as the xor would; 16 and 32 by
// the row swaps), every lane gets it.  LDS-routed shuffles took ~130 cycles a level.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double x) {
  union { double d; int i[2]; } u, w;
  u.d = x;
  w.i[0] = __builtin_amdgcn_update_dpp(0, u.i[0], CTRL, 0xf, 0xf, false);
  w.i[1] = __builtin_amdgcn_update_dpp(0, u.i[1], CTRL, 0xf, 0xf, false);
  return w.d;
}
template <int ROW>
__device__ __forceinline__ double row_swap_add(double x) {
  union { double d; unsigned i[2]; } u, w0, w1;
  u.d = x;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    auto r = ROW == 16 ? __builtin_amdgcn_permlane16_swap(u.i[h], u.i[h], false, false)
                       : __builtin_amdgcn_permlane32_swap(u.i[h], u.i[h], false, false);
    w0.i[h] = r[0];
    w1.i[h] = r[1];
  }
  return w0.d + w1.d;
}
__device__ __forceinline__ double wave_sum(double x, int width) {
  x += dpp_move<0xB1>(x);    // quad_perm [1,0,3,2]
  x += dpp_move<0x4E>(x);    // quad_perm [2,3,0,1]
  x += dpp_move<0x141>(x);   // row_half_mirror
  x += dpp_move<0x140>(x);   // row_mirror
  if (width > 16) x = row_swap_add<16>(x);
  if (width > 32) x = row_swap_add<32>(x);
  return x;
}

// Lanes tx of a block of `width` (the workgroup, or a part of one whose other parts sum
// in step); lane 0 gets the totals.
template <int NA>
__device__ __forceinline__ void block_sum(double (&v)[NA], double* sh /* >= NA * 16 */, int tx, int width) {
  // a workgroup smaller than a wave (strided sweeps of 16- and 32-point lines
  // with narrow tiles) has lanes past its end: the sum stays within the
  // workgroup's lanes
#pragma unroll
  for (int a = 0; a < NA; ++a) v[a] = wave_sum(v[a], width);
  const int w = tx >> 6, nw = (width + 63) >> 6;
  if (nw == 1) return;   // every lane holds the total
  __syncthreads();
  if ((tx & 63) == 0) {
#pragma unroll
    for (int a = 0; a < NA; ++a) sh[a * 16 + w] = v[a];
  }
  __syncthreads();
  if (tx == 0) {
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      double s = 0.0;
      for (int i = 0; i < nw; ++i) s += sh[a * 16 + i];
      v[a] = s;
    }
  }
}

// Sum of nb partials in a fixed order, as lane t of a B-lane finalize block
// adds them: elements t, t+B, t+2B, ... in four interleaved accumulators (so
// four loads are in flight per lane).  The order depends only on nb and B.
__device__ __forceinline__ double fin_sum_at(const double* __restrict__ p, int nb, int t, int B) {
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  int i = t;
  for (; i + 3 * B < nb; i += 4 * B) {
    const double a = p[i], b = p[i + B], c = p[i + 2 * B], d = p[i + 3 * B];
    s0 += a;
    s1 += b;
    s2 += c;
    s3 += d;
  }
  for (; i < nb; i += B) s0 += p[i];
  return (s0 + s1) + (s2 + s3);
}

// The 1024-lane form (nb >= 4096): eight accumulators, so eight loads are in
// flight per lane (a 32768-partial sum takes four rounds instead of eight).
__device__ __forceinline__ double fin_sum8_at(const double* __restrict__ p, int nb, int t, int B) {
  double s[8] = {};
  int i = t;
  for (; i + 7 * B < nb; i += 8 * B) {
    double x[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = p[i + k * B];
#pragma unroll
    for (int k = 0; k < 8; ++k) s[k] += x[k];
  }
  for (; i < nb; i += B) s[0] += p[i];
  return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
}

// The finalize block size for nb partials (launch_finalize).
__host__ __device__ constexpr int fin_block(int nb) { return nb >= 4096 ? 1024 : 256; }

// The parSum norm sqrt(sum * scale) of nb < 4096 partials, computed by one full
// wave (every lane gets it; the host defers a norm only to sweeps whose
// workgroups are whole waves) with the additions of k_finalize in its 256-lane
// form, bit for bit.  Lane l stands for the finalize lanes t = l + 64j (j < 4): in
// chunks of four consecutive elements per t (element t + (4c+q)*256, zero past
// nb), a chunk is one iteration of fin_sum_at's first loop while t + (4c+3)*256 <
// nb, else its elements go one by one into its s0, as the second loop takes them
// (adding an exact zero changes nothing).  Each j is one finalize wave, reduced by
// the same wave_sum, and the four wave totals are added in order.
// load() issues the first chunk (1024 partials: all of them for most sweeps), so
// that they are on their way before psi; indices are clamped, not branched on.
struct PartNorm {
  double v[4][4];
  static __device__ __forceinline__ void chunk(const double* __restrict__ p, int nb, int c, double (&v)[4][4]) {
    const int l = threadIdx.x & 63;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int e = (4 * c + q) * 256;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = e + l + 64 * j;
        v[j][q] = p[i < nb ? i : nb - 1];
      }
    }
  }
  __device__ __forceinline__ void load(const double* __restrict__ p, int nb) { chunk(p, nb, 0, v); }
  __device__ __forceinline__ double norm(const double* __restrict__ p, int nb, double scale) {
    const int l = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) arrive(v[j][q]);
    double s[4][4] = {};
    const int nch = (nb + 1023) / 1024;
    for (int c = 0; c < nch; ++c) {
      if (c > 0) chunk(p, nb, c, v);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = 4 * c * 256 + l + 64 * j;
        if (i + 3 * 256 < nb) {
#pragma unroll
          for (int q = 0; q < 4; ++q) s[j][q] += v[j][q];
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) s[j][0] += i + q * 256 < nb ? v[j][q] : 0.0;
        }
      }
    }
    double tot = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) tot += wave_sum((s[j][0] + s[j][1]) + (s[j][2] + s[j][3]), 64);
    return sqrt(tot * scale);
  }
};

// Block b of nb (of one problem) stores its NA partial sums.
template <int NA>
__device__ __forceinline__ void block_partial(double (&v)[NA], double* partials, double* sh, unsigned b,
                                              unsigned nb, int tx, int width) {
  block_sum<NA>(v, sh, tx, width);
  if (tx == 0 && b < nb) {
#pragma unroll
    for (int a = 0; a < NA; ++a) partials[(size_t)a * nb + b] = v[a];
  }
}

}  // namespace gpue
