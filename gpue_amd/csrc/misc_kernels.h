// misc_kernels.h -- launchers for the pointwise kernels around the sweeps.
#pragma once
#include "sweeps.h"

namespace gpue {

constexpr int REDUCE_BLOCKS = 1024;   // grid of the standalone reductions

struct EqnProg;
hipError_t launch_eqn_field(const EqnProg& prog, double* out, int xDim, int yDim, int zDim, double dx, double dy,
                            double dz, double xMax, double yMax, double zMax, double t, hipStream_t s);
// Time-dependent fields into their tables (k_fields_at).
struct FieldArgs {
  const EqnProg* eq[5];    // programs of V, K, Ax, Ay, Az; null where the field is static
  double* out[5];          // their tables; null: not written
  const double* At[3];     // trap: the static components of A
  const double* vst[3];    // trap: per-axis terms of the harmonic trap without 1/2 m |A|^2
  double mass;
  int trap;                // out[0] is the harmonic trap plus 1/2 m |A|^2 (V_TRAP_A)
  int xDim, yDim, zDim;
  long N;
  double org[3], dxyz[3];  // coordinates x = dx * xi - xMax (src/dynamic.cu:613-615)
  const double* tbase;     // device: step index of the captured block's first step (null: 0)
  double Dt, tstep;        // t = Dt * (*tbase + tstep) (src/evolution.cu:408)
};
hipError_t launch_fields_at(const FieldArgs& f, int depth, hipStream_t s);
template <typename T>
hipError_t launch_apply_norm(void* psi, long N, const double* norm, hipStream_t s);
template <typename T>
hipError_t launch_norm_sum(const void* psi, long N, double* partials, int* nb, hipStream_t s);
hipError_t launch_finalize(const double* partials, int nb, int na, int mode, double scale, double* out, hipStream_t s);
template <typename T>
hipError_t launch_energy_pos(const void* psi, const Phys& p, int gauge, double hbar, double dx, double dy, double dz,
                             double* partials, int* nb, hipStream_t s);
template <typename T>
hipError_t launch_vortex(const void* psi, const unsigned char* mask, int xDim, int* cand, int* marker, int* found,
                         hipStream_t s);

// sweep dispatch (sweep_inst_*.hip)
hipError_t launch_sweep(int prec, bool row, int N, int var, int mode, const SweepArgs& a, hipStream_t s,
                        bool* handled);
hipError_t launch_line(int prec, int N, int plan, const SweepArgs& a, int nsteps, hipStream_t s, bool* handled);
int sweep_blocks(int prec, bool row, int N, int var, int lines_or_xdim, int others);
bool sweep_full_waves(int prec, bool row, int N, int var);
hipError_t launch_sweep_batched(int prec, bool row, int N, int var, int mode, unsigned flags, int gstate,
                                const SweepArgs* d, int ninst, int lx, int others, hipStream_t s, bool* handled);

// One launch over problems of different sizes (sweep_merged.h): lanes of a block and LDS
// bytes of a workgroup for an axis length (0 lanes: no such kernel), and the launch.
struct MergeMap;
int merged_shape(int prec, bool row, int n, int* lds);
hipError_t launch_sweep_merged(int prec, bool row, int mode, unsigned flags, int gstate, const SweepArgs* d,
                               const MergeMap* map, int grid, int lds, hipStream_t s);

// Second stage of a batched reduction: one workgroup per instance.
struct FinArgs {
  int active;
  int nb, na, mode;
  double scale;
  const double* partials;
  double* out;
};
hipError_t launch_finalize_batched(const FinArgs* d, int ninst, hipStream_t s);
hipError_t launch_set_double(double* p, double v, hipStream_t s);
hipError_t launch_energy_fold(double* results, int naxes, hipStream_t s);
hipError_t launch_copy16(const void* in, void* out, size_t bytes, hipStream_t s);
hipError_t launch_math_eval(int fn, const double* x, double* y, long n, hipStream_t s);
// variant = plan (bit 0: 0 wide lines, 1 narrow lines) + 2 * narrow, where the
// strided sweeps' tiles are 2^narrow times narrower (narrow 0..2) and, for
// narrow > 0, every sweep loads its transforms' twiddles up front (row sweeps
// have variants 0..3 only)
constexpr int N_VARIANTS = 6;
bool sweep_supported(int N);

}  // namespace gpue
