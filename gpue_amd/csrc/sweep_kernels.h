// sweep_kernels.h -- row (x, contiguous) and strided (y/z) sweep kernels.
#pragma once
#include "sweeps.h"

namespace gpue {

// Workgroup shapes.  Row sweeps: LPW lines of TPL lanes.  Strided sweeps: TC
// adjacent x-lines (lanes vary fastest in x for coalescing) of TPL lanes.
// RV is the row-sweep variant: bit 0 the plan, bit 1 twiddles loaded before
// the first pass of each transform (fft_regs PRE).
template <int N, int RV>
struct RowCfg {
  static constexpr int V = RV & 1;
  static constexpr int TPL = Plan<N, V>::TPL;
  static constexpr int WGr = V == 0 ? 128 : 64;
  static constexpr int WG = TPL >= WGr ? TPL : WGr;
  static constexpr int LPW = WG / TPL;
  // elements of a line (the larger of both precisions) and of the workgroup
  static constexpr int FOOT64 = lds_span<N, V, lds_lanes<double, 1>()>(), FOOT32 = lds_span<N, V, lds_lanes<float, 1>()>();
  static constexpr int FOOT = FOOT64 > FOOT32 ? FOOT64 : FOOT32;
  static constexpr int LDS = Plan<N, V>::NP > 1 ? LPW * FOOT : 1;
};

// Strided sweeps read TC adjacent x-lines per row of the tile: at least one
// 128-byte cache line (8 complex doubles, 16 complex floats) and up to 256
// lanes' worth for short transforms, within 1024 lanes per workgroup.
// Measured at 256^3: FP64 8-column tiles run the strided FFT at copy speed
// (2-4 columns lose 40-70 %); FP32 8-column tiles fetch every line twice.
//
// CV is the strided-sweep variant: bit 0 the plan, bits 1-2 narrow the tile
// to a half or a quarter of that width. Small grids have few tiles (64 of
// them for 512 FP64 columns), so narrower tiles put more CUs to work; the
// tiles that share a 128-byte line then run on one XCD (col_sweep), so the
// line is fetched into one L2 only.  Narrowed FP64 tiles also load each
// transform's twiddles before its first pass (these launches are latency
// bound and have registers to spare); FP32 tiles keep per-pass loads, since
// the up-front tables (hi + lo parts) cost 60-100 more VGPRs and FP32 tiles
// serve batches whose sweeps are limited by occupancy (82 VGPRs: 5 waves per
// SIMD; 141-180 with the tables: 2-3).
template <typename T, int N, int CV>
struct ColCfg {
  static constexpr int PV = CV & 1, NARROW = CV >> 1;
  static constexpr int TPL = Plan<N, PV>::TPL;
  static constexpr int TCmin = 128 / (2 * (int)sizeof(T));
  static constexpr int TCa = 256 / TPL > TCmin ? 256 / TPL : TCmin;
  static constexpr int TCb = TCa > 64 ? 64 : TCa;
  static constexpr int TCw = TPL * TCb > 1024 ? 1024 / TPL : TCb;
  // the tile's LDS (TC lines of N points) within 128 KiB of the 160 KiB per workgroup
  static constexpr int TCm = 131072 / (N * 2 * (int)sizeof(T));
  static constexpr int TC0 = TCw < TCm ? TCw : TCm;
  static constexpr int TC = (TC0 >> NARROW) > 0 ? (TC0 >> NARROW) : 1;
  // tiles that share 128-byte lines, or make up a default-width one: on one XCD (xcd_tile).
  // (FP64 tiles of 2048 points are 4 columns, half lines; a line in two L2s made the K
  // sweep of 2048^2 take 51 us next to 31 of a row sweep.  With it, and the exchange gaps
  // of fft_core.h, an imaginary step there takes 101 instead of 112 us.)
  static constexpr int G = TC0 < TCmin ? TCmin / TC : TC0 / TC;
  static constexpr int WG = TPL * TC;
  static constexpr int LDS = Plan<N, PV>::NP > 1 ? TC * lds_span<N, PV, lds_lanes<T, TC>()>() : 1;   // elements
  static_assert(TC0 >= 1 && G >= 1 && WG <= 1024, "strided tile does not fit a workgroup");
};

// scalarDiv_wfcNorm (src/kernels.cu:479-486) divides by sqrt(sum * dV); the
// fused form multiplies by its reciprocal (within 1 ulp of the quotient).
template <typename T>
__device__ __forceinline__ cx<T> scale_norm(cx<T> v, T inv) {
  return scaled(v, inv);
}

template <typename T>
__device__ __forceinline__ double abs2d(cx<T> v) {
  return fma((double)v.x, (double)v.x, (double)v.y * (double)v.y);
}

// Mode bits above the sweep kind (RM_*, CM_*): 16, the real-time kernel (phases;
// the plain one is imaginary time); 64, RM_INV compiled without the gauge operator
// (its three-transform path sets the register count of the whole kernel, and so
// the waves per SIMD), for sweeps whose flags carry no F_GAUGE_POST.

using OpeningHalf = std::integral_constant<bool, false>;
using ClosingHalf = std::integral_constant<bool, true>;

// The pending norm's reciprocal for the sweep that opens an imaginary-time step.
struct NormIn {
  PartNorm part;
  __device__ __forceinline__ void load(const SweepArgs& a) {
    if (a.flags & F_SCALE_PART) part.load(a.partials, a.norm_nb);
  }
  // a deferred renormalisation: the norm reduced here from the previous sweep's
  // partials by every wave (all lanes active), stored once by block 0
  __device__ __forceinline__ double inverse(const SweepArgs& a, int bid, int tx) {
    double nrm;
    if (a.flags & F_SCALE_PART) {
      nrm = part.norm(a.partials, a.norm_nb, a.norm_scale);
      if (bid == 0 && tx == 0) *a.norm_out = nrm;
    } else {
      nrm = *a.norm_in;
    }
    return 1.0 / nrm;
  }
};

// Brings the scalar arguments of a sweep into registers in one go at its start: left
// to their places of use they are separate scalar loads (selects between them become
// loads through selected addresses), each with its own wait in the serial chain ahead
// of psi's loads and of the operators.
// (Pointers go through the asm as global ones, or their loads would become flat.)
template <typename U>
__device__ __forceinline__ void pin_ptr(U*& p) {
  auto g = (__attribute__((address_space(1))) U*)p;
  asm volatile("" : "+s"(g));
  p = (U*)g;
}
template <typename... P>
__device__ __forceinline__ void pin_ptrs(P&... p) { (pin_ptr(p), ...); }
#define GPUE_PIN(...) asm volatile("" : __VA_ARGS__)
template <bool VHALF, bool KSTEP, bool GAUGE, bool OPENS>
__device__ __forceinline__ void pin_args(SweepArgs& a) {
  Phys& p = a.ph;
  pin_ptrs(a.in, a.out, a.tw);
  GPUE_PIN("+s"(a.flags), "+s"(p.yDim), "+s"(p.zDim), "+s"(p.xDim));
  if constexpr (VHALF) {
    pin_ptrs(p.vs[0], p.vs[1], p.vs[2], p.vsf[0], p.vsf[1], p.vsf[2], p.Vt, p.Vt_next);
    GPUE_PIN("+s"(p.v_kind), "+s"(p.cV), "+s"(p.g), "+s"(p.cH), "+s"(p.gpe));
  }
  if constexpr (KSTEP) {
    pin_ptrs(p.kf[0], p.kf[1], p.kf[2], p.kff[0], p.kff[1], p.kff[2], p.Kt);
    GPUE_PIN("+s"(p.k_kind), "+s"(a.invN));
  }
  if constexpr (GAUGE) {
    pin_ptrs(p.xg, p.yg, p.pxg, p.pyg, p.pzg, p.At[0], p.At[1], p.At[2]);
    GPUE_PIN("+s"(p.a_kind), "+s"(p.omega), "+s"(p.omegaX), "+s"(p.omegaY), "+s"(p.Dt), "+s"(a.invN));
  }
  if constexpr (OPENS) {
    pin_ptrs(a.partials, a.norm_in, a.norm_out);
    GPUE_PIN("+s"(a.norm_nb), "+s"(a.norm_scale));
  }
}
#undef GPUE_PIN

// ---------------------------------------------------------------------------
// Row sweep: lines are contiguous x-rows, line = y + yDim*z.
// ---------------------------------------------------------------------------
// Block `bid` of nblk of a sweep, by the lanes tx = 0 .. RowCfg::WG - 1 on the LDS at
// lds (RowCfg::LDS elements) and sh (16 doubles).  ONEWAVE: see lds_sync.
template <typename T, int N, int RV, int MODE_, bool ONEWAVE = false, bool TWPRE = true>
__device__ __forceinline__ void row_body(SweepArgs a, int bid, int nblk, int tx, cx<T>* lds, double* sh) {
  constexpr int MODE = MODE_ & 15;
  constexpr bool REAL = (MODE_ & 16) != 0, NG = (MODE_ & 64) != 0;
  constexpr int V = RV & 1;
  constexpr bool EARLY = (RV >> 1) != 0;     // operands loaded up front
  constexpr bool PRE = EARLY && TWPRE;       // and every twiddle
  constexpr bool GAUGE = (MODE == RM_INV && !NG) || MODE == RM_GAUGE || MODE == RM_GAUGE_FWD || MODE == RM_FULL;
  constexpr bool KSTEP = MODE == RM_K || MODE == RM_FULL;
  constexpr bool OPENS = !REAL && (MODE == RM_FWD || MODE == RM_FULL);
  constexpr bool GEARLY = EARLY && sizeof(T) == 8;
  constexpr bool VHALF = MODE != RM_GAUGE && MODE != RM_K && MODE != RM_KSUM;
  using P = Plan<N, V>;
  constexpr int TPL = P::TPL, E = P::E, LPW = RowCfg<N, RV>::LPW;
  constexpr bool AHEAD = EARLY && E <= 8;   // see apply_phase_all
  if constexpr (EARLY) pin_args<VHALF, KSTEP, GAUGE, OPENS>(a);
  const Phys& p = a.ph;
  const unsigned flags = a.flags;
  const int tid = tx % TPL, lw = tx / TPL;
  const int line = bid * LPW + lw;
  const bool active = line < a.lines;
  const int ln = active ? line : 0;
  int yi = ln, zi = 0;
  if (p.zDim > 1) {
    zi = ln / p.yDim;
    yi = ln - zi * p.yDim;
  }
  const LineAt l{0, tid, (long)ln * N, 1, yi, zi};
  const cx<T>* __restrict__ in = (const cx<T>*)a.in + l.base;
  cx<T>* __restrict__ out = (cx<T>*)a.out + l.base;
  const auto* __restrict__ tw = (const typename TwE<T>::type*)a.tw;
  const LdsLine<T, 1, ONEWAVE> la{lw * RowCfg<N, RV>::FOOT};
  constexpr int RF0 = Seq<N, V, ORD_FWD>::first(), RFL = Seq<N, V, ORD_FWD>::last();
  constexpr int RIN = MODE == RM_INV || MODE == RM_INV_FWD ? RFL : RF0;
  cx<T> v[E];
  double acc = 0.0;
  TwRegs<T, N, V> twr;
  NormIn nin;
  VOp<T, N, TPL, RF0, E> vo;          // V/2 sits between transforms: first-radix layout
  KOp<T, N, TPL, RFL, E, REAL> ko;    // K and A in the last radix's
  GOp<T, N, TPL, RFL, E, REAL> go;
  const double* __restrict__ Vt = MODE == RM_GAUGE_FWD ? p.Vt_next : p.Vt;
  auto fwd = [&]() { fft_regs_tw<T, N, V, ORD_FWD, -1, PRE>(v, tid, tw, twr, lds, la); };
  auto inv = [&]() { fft_regs_tw<T, N, V, ORD_REV, +1, PRE>(v, tid, tw, twr, lds, la); };
  auto half = [&](auto closes) {
    if constexpr (EARLY) vo.ready();
    else vo.load(p, Vt, l);
    vo.template half<REAL, decltype(closes)::value, AHEAD>(p, l, v);
  };
  auto kstep = [&]() {
    if constexpr (!EARLY && REAL) {
      ko.load_apply(p, l, v, a.invN);
    } else {
      if constexpr (EARLY) ko.ready();
      else ko.load(p, l);
      ko.template apply<AHEAD>(p, l, v, a.invN);
    }
  };
  auto gauge = [&]() {
    if constexpr (!EARLY) {
      go.load(p, l);
      go.prep(p, l, a.invN);
    }
    go.template apply<AHEAD>(p, v, l, a.invN, GEARLY);
  };

  if constexpr (EARLY && GAUGE) go.load(p, l);
  if constexpr (OPENS) nin.load(a);
#pragma unroll
  for (int r = 0; r < E; ++r) v[r] = in[bpos<N, TPL, RIN>(tid, r)];
  if constexpr (EARLY) {
    if constexpr (VHALF) vo.load(p, Vt, l);
    if constexpr (KSTEP) ko.load(p, l);
    if constexpr (GAUGE && GEARLY) {
      if (p.a_kind == A_TABLE) go.load_points(p, l);
    }
    if constexpr (PRE) twr.load(tid, tw);
    if constexpr (GAUGE) go.prep(p, l, a.invN);
  }

  if constexpr (MODE == RM_INV || MODE == RM_INV_FWD) {
    inv();
    if constexpr (MODE == RM_INV_FWD && sizeof(T) == 8) {
      // the closing V/2 of this step and the opening one of the next: phases, which
      // leave |psi|^2, so one phase of the summed exponents
      if constexpr (EARLY) vo.ready();
      else vo.load(p, Vt, l);
      T arg[E];
      vo.template args<true>(p, l, v, arg);
      if (p.Vt_next != p.Vt) {   // V(t): the next step's table
        VOp<T, N, TPL, RF0, E> vn;
        vn.load(p, p.Vt_next, l);
        T arg2[E];
        vn.template args<false>(p, l, v, arg2);
#pragma unroll
        for (int r = 0; r < E; ++r) arg[r] += arg2[r];
      } else {
#pragma unroll
        for (int r = 0; r < E; ++r) arg[r] += arg[r];
      }
      apply_phase_all<T, E, REAL, AHEAD>(v, arg, 1.0);
      fwd();
    } else if constexpr (MODE == RM_INV_FWD) {
      half(ClosingHalf());   // FP32 (static V): each half's phase rounds psi, as in single steps
      half(OpeningHalf());
      fwd();
    } else {
      if (flags & F_HALFV_POST) half(ClosingHalf());
      if constexpr (GAUGE) {
        fwd();
        gauge();
        inv();
      }
    }
  } else {
    if constexpr (OPENS) {
      if (flags & F_SCALE_IN) {
        const T s = (T)nin.inverse(a, bid, tx);
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = scale_norm(v[r], s);
      }
    }
    if constexpr (MODE == RM_FWD || MODE == RM_FULL) {
      if (flags & F_HALFV_PRE) half(OpeningHalf());
    }
    fwd();
    if constexpr (MODE == RM_GAUGE || MODE == RM_GAUGE_FWD) {
      gauge();
      inv();
    } else if constexpr (KSTEP) {
      kstep();
      inv();
      if constexpr (MODE == RM_FULL) {
        if (flags & F_HALFV_POST) half(ClosingHalf());
        if (flags & F_GAUGE_POST) {
          fwd();
          gauge();
          inv();
        }
      }
    } else if constexpr (MODE == RM_KSUM) {
      if (active) {
#pragma unroll
        for (int r = 0; r < E; ++r) {
          const int xi = bpos<N, TPL, RFL>(tid, r);
          const long gid = gid_of(p, xi, yi, zi);
          const double w = (flags & F_ASUM)  ? A_val(p, 0, xi, yi, zi, gid) * p.pxg[xi]
                           : (flags & F_KAX) ? p.ks[0][xi]
                                             : K_val(p, xi, yi, zi, gid);
          acc += w * abs2d(v[r]);
        }
      }
    }
    if constexpr (MODE == RM_GAUGE_FWD) {   // continue with the next step's first row sweep
      half(OpeningHalf());
      fwd();
    }
  }

  // store: forward sweeps leave the forward layout (last radix), the others the first radix
  constexpr bool FWD_OUT = MODE == RM_FWD || MODE == RM_INV_FWD || MODE == RM_GAUGE_FWD;
  constexpr int ROUT = FWD_OUT ? RFL : RF0;
  constexpr bool NORM = !REAL && !FWD_OUT && MODE != RM_KSUM;
  if constexpr (MODE != RM_KSUM) {
    if (active) {
#pragma unroll
      for (int r = 0; r < E; ++r) {
        out[bpos<N, TPL, ROUT>(tid, r)] = v[r];
        if (NORM && (flags & F_NORM)) acc += abs2d(v[r]);
      }
    }
  }
  if (MODE == RM_KSUM || (NORM && (flags & F_NORM))) {
    double pv[1] = {acc};
    block_partial<1>(pv, a.partials, sh, bid, nblk, tx, RowCfg<N, RV>::WG);
  }
}

// ---------------------------------------------------------------------------
// Strided sweep: lines along y (axis 1, stride xDim) or z (axis 2, stride
// xDim*yDim); a workgroup owns TC adjacent x-lines, lanes vary fastest in x.
// ---------------------------------------------------------------------------
template <typename T, int N, int CV, int MODE_, bool ONEWAVE = false, bool TWPRE = true>
__device__ __forceinline__ void col_body(SweepArgs a, int bid, int nblk, int tx, cx<T>* lds, double* sh) {
  constexpr int MODE = MODE_ & 15;
  constexpr bool REAL = (MODE_ & 16) != 0;
  constexpr int V = CV & 1;
  constexpr bool EARLY = (CV >> 1) != 0;               // operands loaded up front
  constexpr bool PRE = EARLY && TWPRE && sizeof(T) == 8;   // and every twiddle
  constexpr bool GAUGE = MODE == CM_INV_VG || MODE == CM_GAUGE || MODE == CM_GAUGE_FWD;
  constexpr bool GEARLY = EARLY && sizeof(T) == 8;
  constexpr bool VHALF = MODE == CM_FWD_V || MODE == CM_INV_VG || MODE == CM_GAUGE_FWD;
  constexpr bool OPENS = !REAL && MODE == CM_FWD_V;
  using P = Plan<N, V>;
  constexpr int TC = ColCfg<T, N, CV>::TC, E = P::E, TPL = P::TPL;
  constexpr bool AHEAD = EARLY && E <= 8;   // see apply_phase_all
  if constexpr (EARLY) pin_args<VHALF, MODE == CM_K, GAUGE, OPENS>(a);
  const Phys& p = a.ph;
  const unsigned flags = a.flags;
  const int c = tx % TC, tid = tx / TC;
  const int tiles = (p.xDim + TC - 1) / TC;
  const int bq = bid < nblk ? bid : 0;   // blocks past the last (parts of a merged workgroup) read block 0
  const int o = bq / tiles, xt = bq - o * tiles;
  const int xi = xt * TC + c;
  const bool active = xi < p.xDim && bid < nblk;
  const int xq = xi < p.xDim ? xi : 0;   // lanes past xDim (a last partial tile) read column 0
  const bool ay = a.axis == 1;
  const LineAt l{a.axis, tid, ay ? (long)xq + (long)o * p.xDim * p.yDim : (long)xq + (long)o * p.xDim,
                 ay ? (long)p.xDim : (long)p.xDim * p.yDim, xq, o};
  const long es = l.es;
  // a lane's points lie at (tid + bpos(0, r)) * es from the tile's base:
  // one per-lane pointer, then per register a uniform offset bpos(0, r) * es
  // (scalar arithmetic) instead of a 64-bit multiply per access
  const cx<T>* __restrict__ in = (const cx<T>*)a.in + l.base + (long)tid * es;
  cx<T>* __restrict__ out = (cx<T>*)a.out + l.base + (long)tid * es;
  const auto* __restrict__ tw = (const typename TwE<T>::type*)a.tw;
  const LdsLine<T, TC, ONEWAVE> la{c};
  constexpr int RF0 = Seq<N, V, ORD_FWD>::first(), RFL = Seq<N, V, ORD_FWD>::last();
  constexpr int RIN = MODE == CM_INV || MODE == CM_INV_VG ? RFL : RF0;
  cx<T> v[E];
  double acc = 0.0;
  TwRegs<T, N, V> twr;
  NormIn nin;
  VOp<T, N, TPL, RF0, E> vo;
  KOp<T, N, TPL, RFL, E, REAL> ko;
  GOp<T, N, TPL, RFL, E, REAL> go;
  const double* __restrict__ Vt = MODE == CM_GAUGE_FWD ? p.Vt_next : p.Vt;
  auto fwd = [&]() { fft_regs_tw<T, N, V, ORD_FWD, -1, PRE>(v, tid, tw, twr, lds, la); };
  auto inv = [&]() { fft_regs_tw<T, N, V, ORD_REV, +1, PRE>(v, tid, tw, twr, lds, la); };
  auto half = [&](auto closes) {
    if constexpr (EARLY) vo.ready();
    else vo.load(p, Vt, l);
    vo.template half<REAL, decltype(closes)::value, AHEAD>(p, l, v);
  };
  auto gauge = [&]() {
    if constexpr (!EARLY) {
      go.load(p, l);
      go.prep(p, l, a.invN);
    }
    go.template apply<AHEAD>(p, v, l, a.invN, GEARLY);
  };

  if constexpr (EARLY && GAUGE) go.load(p, l);
  if constexpr (OPENS) nin.load(a);
#pragma unroll
  for (int r = 0; r < E; ++r) v[r] = in[bpos<N, TPL, RIN>(0, r) * es];
  if constexpr (EARLY) {
    if constexpr (VHALF) vo.load(p, Vt, l);
    if constexpr (MODE == CM_K) ko.load(p, l);
    if constexpr (GAUGE && GEARLY) {
      if (p.a_kind == A_TABLE) go.load_points(p, l);
    }
  }
  if constexpr (PRE) twr.load(tid, tw);
  if constexpr (EARLY && GAUGE) go.prep(p, l, a.invN);

  if constexpr (MODE == CM_INV || MODE == CM_INV_VG) {
    inv();
    if constexpr (MODE == CM_INV_VG) {
      // the closing sweep of a step that leads with this axis: V/2, then this
      // axis' gauge operator
      half(ClosingHalf());
      fwd();
      gauge();
      inv();
    }
  } else {
    if constexpr (OPENS) {   // the opening sweep of a step that leads with this axis
      if (flags & F_SCALE_IN) {
        const T s = (T)nin.inverse(a, bid, tx);
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = scale_norm(v[r], s);
      }
    }
    if constexpr (MODE == CM_FWD_V) half(OpeningHalf());
    fwd();
    if constexpr (MODE == CM_KSUM) {
      if (active) {
#pragma unroll
        for (int r = 0; r < E; ++r) {
          const int e = bpos<N, TPL, RFL>(tid, r);
          const int yi = ay ? e : o, zi = ay ? o : e;
          const long gid = gid_of(p, xi, yi, zi);
          const double w = (flags & F_ASUM)  ? A_val(p, a.axis, xi, yi, zi, gid) * (ay ? p.pyg[yi] : p.pzg[zi])
                           : (flags & F_KAX) ? (ay ? p.ks[1][yi] : p.ks[2][zi])
                                             : K_val(p, xi, yi, zi, gid);
          acc += w * abs2d(v[r]);
        }
      }
    } else if constexpr (MODE == CM_K) {
      if constexpr (!EARLY && REAL) {
        ko.load_apply(p, l, v, a.invN);
      } else {
        if constexpr (EARLY) ko.ready();
        else ko.load(p, l);
        ko.template apply<AHEAD>(p, l, v, a.invN);
      }
      inv();
    } else if constexpr (GAUGE) {
      gauge();
      inv();
      if constexpr (MODE == CM_GAUGE_FWD) {   // bridge: the next step's V/2 and its first transform along this axis
        half(OpeningHalf());
        fwd();
      }
    }
  }

  constexpr bool FWD_OUT = MODE == CM_FWD || MODE == CM_FWD_V || MODE == CM_GAUGE_FWD;
  constexpr int ROUT = FWD_OUT ? RFL : RF0;
  constexpr bool NORM = !REAL && (MODE == CM_INV_VG || MODE == CM_GAUGE);
  if constexpr (MODE != CM_KSUM) {
    if (active) {
#pragma unroll
      for (int r = 0; r < E; ++r) {
        out[bpos<N, TPL, ROUT>(0, r) * es] = v[r];
        if (NORM && (flags & F_NORM)) acc += abs2d(v[r]);
      }
    }
  }
  if (MODE == CM_KSUM || (NORM && (flags & F_NORM))) {
    double pv[1] = {acc};
    block_partial<1>(pv, a.partials, sh, bid, nblk, tx, ColCfg<T, N, CV>::WG);
  }
}

// ---------------------------------------------------------------------------
// 1D problems: a run of whole steps in one launch.  The line fits one workgroup, so
// psi stays in registers from step to step ([V/2, FFT, K, IFFT, V/2 (, gauge)], the
// operators and their arithmetic as in RM_FULL) and the renormalisation is a block
// sum, with the additions of a sweep's partial and its finalize: results are those
// of steps launched one by one.  What bounds it is the dependent chain of a step
// (N = 1024: eight passes and their exchanges, two V/2 and the block sum): about 4 us
// at N = 1024 FP64, 1e2 steps in one launch, where a sweep and a finalize a step,
// most of them launch and first loads, took 11.7 us.
// The norm of the last step is left pending in *norm_out.
// ---------------------------------------------------------------------------
template <typename T, int N, int RV, bool REAL>
__device__ __forceinline__ void line_body(const SweepArgs& a, int nsteps) {
  constexpr int V = RV & 1;
  constexpr bool PRE = (RV >> 1) != 0;   // twiddles in registers for the whole run
  using P = Plan<N, V>;
  constexpr int TPL = P::TPL, E = P::E, WG = RowCfg<N, RV>::WG, NW = (WG + 63) / 64;
  __shared__ cx<T> lds[RowCfg<N, RV>::LDS];
  __shared__ double sh[16];
  const Phys& p = a.ph;
  const unsigned flags = a.flags;
  const int tid = threadIdx.x % TPL, lw = threadIdx.x / TPL;
  const bool active = lw == 0;   // further lines of the workgroup repeat line 0
  const LineAt l{0, tid, 0, 1, 0, 0};
  const auto* __restrict__ tw = (const typename TwE<T>::type*)a.tw;
  const LdsLine<T, 1> la{lw * RowCfg<N, RV>::FOOT};
  constexpr int RF0 = Seq<N, V, ORD_FWD>::first(), RFL = Seq<N, V, ORD_FWD>::last();
  cx<T> v[E];
  TwRegs<T, N, V> twr;
  VOp<T, N, TPL, RF0, E> vo;
  KOp<T, N, TPL, RFL, E, REAL> ko;
  GOp<T, N, TPL, RFL, E, REAL> go;
  const bool gauge = (flags & F_GAUGE_POST) != 0;
#pragma unroll
  for (int r = 0; r < E; ++r) v[r] = ((const cx<T>*)a.in)[bpos<N, TPL, RF0>(tid, r)];
  vo.load(p, p.Vt, l);
  ko.load(p, l);
  if constexpr (PRE) twr.load(tid, tw);
  if (gauge) {
    go.load(p, l);
    go.prep(p, l, a.invN);
  }
  double nrm = !REAL && (flags & F_SCALE_IN) ? *a.norm_in : 1.0;
  auto fwd = [&]() { fft_regs_tw<T, N, V, ORD_FWD, -1, PRE>(v, tid, tw, twr, lds, la); };
  auto inv = [&]() { fft_regs_tw<T, N, V, ORD_REV, +1, PRE>(v, tid, tw, twr, lds, la); };
#pragma unroll 1
  for (int s = 0; s < nsteps; ++s) {
    if constexpr (!REAL) {
      const T f = (T)(1.0 / nrm);
#pragma unroll
      for (int r = 0; r < E; ++r) v[r] = scale_norm(v[r], f);
    }
    vo.template half<REAL, false, true>(p, l, v);
    fwd();
    ko.template apply<true>(p, l, v, a.invN);
    inv();
    vo.template half<REAL, true, true>(p, l, v);
    if (gauge) {
      fwd();
      go.template apply<true>(p, v, l, a.invN, false);
      inv();
    }
    if constexpr (!REAL) {
      double acc = 0.0;
#pragma unroll
      for (int r = 0; r < E; ++r)
        if (active) acc += abs2d(v[r]);
      double tot = wave_sum(acc, 64);
      if constexpr (NW > 1) {
        if constexpr (P::NP == 1) __syncthreads();   // else the exchanges' barriers follow the last read of sh
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = tot;
        __syncthreads();
        tot = 0.0;
#pragma unroll
        for (int w = 0; w < NW; ++w) tot += sh[w];
      }
      nrm = sqrt(tot * a.norm_scale);
    }
  }
  if (active) {
#pragma unroll
    for (int r = 0; r < E; ++r) ((cx<T>*)a.out)[bpos<N, TPL, RF0>(tid, r)] = v[r];
    if (!REAL && tid == 0) *a.norm_out = nrm;
  }
}

template <typename T, int N, int V, bool REAL>
__global__ void __launch_bounds__((RowCfg<N, V>::WG)) line_steps(SweepArgs a, int nsteps) {
  line_body<T, N, V, REAL>(a, nsteps);
}

// One problem per launch (arguments by value) ...
template <typename T, int N, int V, int MODE>
__global__ void __launch_bounds__((RowCfg<N, V>::WG)) row_sweep(SweepArgs a) {
  __shared__ cx<T> lds[RowCfg<N, V>::LDS];
  __shared__ double sh[16];
  row_body<T, N, V, MODE>(a, blockIdx.x, gridDim.x, threadIdx.x, lds, sh);
}
// Workgroups are dealt to the 8 XCDs round robin (block b runs on XCD b % 8).
// With narrowed tiles, the G tiles of one default-width tile (one 128-byte
// line per row) are given blocks on the same XCD: block b = x + 8q takes
// tile G*(x + 8*(q/G)) + q%G. Blocks past the last whole group of 8G keep
// their own index, so the map is a permutation of [0, nblk).
template <int G>
__device__ __forceinline__ int xcd_tile(int b, int nblk) {
  if constexpr (G == 1) {
    return b;
  } else {
    const int full = nblk - nblk % (8 * G);
    if (b >= full) return b;
    const int x = b & 7, q = b >> 3;
    return G * (x + 8 * (q / G)) + q % G;
  }
}

template <typename T, int N, int CV, int MODE>
__global__ void __launch_bounds__((ColCfg<T, N, CV>::WG)) col_sweep(SweepArgs a) {
  __shared__ cx<T> lds[ColCfg<T, N, CV>::LDS];
  __shared__ double sh[16];
  col_body<T, N, CV, MODE>(a, xcd_tile<ColCfg<T, N, CV>::G>(blockIdx.x, gridDim.x), gridDim.x, threadIdx.x, lds, sh);
}

// ... or many problems of one shape per launch: blocks [i*bpi, (i+1)*bpi) work
// on instance i, whose arguments are read from device memory.
template <typename T, int N, int V, int MODE>
__global__ void __launch_bounds__((RowCfg<N, V>::WG)) row_sweep_b(const SweepArgs* __restrict__ args, int bpi) {
  const SweepArgs& a = args[blockIdx.x / bpi];
  if (!a.active) return;
  __shared__ cx<T> lds[RowCfg<N, V>::LDS];
  __shared__ double sh[16];
  row_body<T, N, V, MODE>(a, blockIdx.x % bpi, bpi, threadIdx.x, lds, sh);
}
template <typename T, int N, int CV, int MODE>
__global__ void __launch_bounds__((ColCfg<T, N, CV>::WG)) col_sweep_b(const SweepArgs* __restrict__ args, int bpi) {
  const SweepArgs& a = args[blockIdx.x / bpi];
  if (!a.active) return;
  __shared__ cx<T> lds[ColCfg<T, N, CV>::LDS];
  __shared__ double sh[16];
  col_body<T, N, CV, MODE>(a, blockIdx.x % bpi, bpi, threadIdx.x, lds, sh);
}

}  // namespace gpue
