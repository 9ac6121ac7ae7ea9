// The library's host code on the runtime of fake_hip.cpp: what it launches and with
// which arguments, and what it leaves behind where memory runs out.  Built and run by
// tests/test_host_logic.py, one argument: the check to run.
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <thread>
#include <vector>

#include "../../gpue_amd/csrc/ctx_internal.h"
#include "../../gpue_amd/csrc/sweep_merged.h"
#include "fake_hip.h"

using namespace gpue;

static int failures = 0;
#define CHECK(cond, ...)                                          \
  do {                                                            \
    if (!(cond) && ++failures <= 20) {                            \
      std::printf("%s:%d: %s: ", __FILE__, __LINE__, #cond);      \
      std::printf(__VA_ARGS__);                                   \
      std::printf("\n");                                          \
    }                                                             \
  } while (0)

// Looks at every launch: a sweep's kernel is built for the length of the axis that its
// arguments name, its psi is as large as its grid, and the norm an imaginary step divides
// by is there: reduced by a finalize into the slot, or by the opening sweep itself from
// all the partials of the sweep before, in workgroups of whole waves.
struct Audit {
  struct Norm {
    int nb = 0;
    bool settled = true;
  };
  std::map<const void*, Norm> norms;   // by partials
  long sweeps = 0, from_partials = 0;
  std::map<std::string, long> kernels;

  void sweep(const fake::Launch& l, const SweepArgs& a, int n, int nblk, int wg, int mode, bool row) {
    if (!a.active) return;
    ++sweeps;
    const int dims[3] = {a.ph.xDim, a.ph.yDim, a.ph.zDim};
    CHECK(a.axis >= 0 && a.axis < 3 && (a.axis == 0) == row && dims[a.axis] == n, "%s on axis %d of %d x %d x %d",
          l.kernel.c_str(), a.axis, dims[0], dims[1], dims[2]);
    const size_t es = l.kernel.find("<double") != std::string::npos ? 16 : 8;
    CHECK(fake::bytes_at(a.in) >= es * dims[0] * dims[1] * dims[2], "%s: psi", l.kernel.c_str());
    CHECK(fake::bytes_at(a.tw) > 0, "%s: twiddles", l.kernel.c_str());
    const double all = 1.0 / ((double)dims[0] * dims[1] * dims[2]), one = 1.0 / dims[a.axis];
    const int op = mode & 15;
    const bool k_op = row ? op == RM_K || op == RM_FULL : op == CM_K;
    const bool a_op = row ? op == RM_GAUGE || op == RM_GAUGE_FWD || (op == RM_INV && (a.flags & F_GAUGE_POST))
                          : op == CM_GAUGE || op == CM_GAUGE_FWD || (op == CM_INV_VG && (a.flags & F_GAUGE_POST));
    CHECK(!k_op || a.invN == all, "%s: K normalised by %g", l.kernel.c_str(), a.invN);
    CHECK(!a_op || a.invN == one, "%s: A normalised by %g", l.kernel.c_str(), a.invN);
    Norm& m = norms[a.partials];
    const bool ksum = (mode & 15) == (row ? (int)RM_KSUM : (int)CM_KSUM);
    if (a.flags & F_SCALE_IN) {
      if (a.flags & F_SCALE_PART) {
        ++from_partials;
        CHECK(wg % 64 == 0, "%s: %d lanes reduce a norm", l.kernel.c_str(), wg);
        CHECK(a.norm_nb < 4096 && a.norm_nb == m.nb, "%s: norm of %d partials, there are %d", l.kernel.c_str(), a.norm_nb,
              m.nb);
      } else {
        CHECK(m.settled, "%s: the norm is still in its partials", l.kernel.c_str());
      }
      m.settled = true;
    }
    if (ksum) m.nb = -1;
    if (a.flags & F_NORM) m = Norm{nblk, false};
  }
  void finalize(const void* partials, int nb, int mode) {
    Norm& m = norms[partials];
    if (mode != 1) return;
    CHECK(m.nb == nb || m.settled, "finalize of %d partials, there are %d", nb, m.nb);
    m.settled = true;
  }
  void operator()(const fake::Launch& l) {
    const std::string& k = l.kernel;
    ++kernels[k.substr(0, k.find('<'))];
    if (k.rfind("gpue::k_finalize_b", 0) == 0) {
      const FinArgs* f = *(const FinArgs**)l.args[0];
      for (unsigned i = 0; i < l.grid; ++i)
        if (f[i].active) finalize(f[i].partials, f[i].nb, f[i].mode);
      return;
    }
    if (k.rfind("gpue::k_finalize", 0) == 0) {
      finalize(*(const void**)l.args[0], *(int*)l.args[1], *(int*)l.args[3]);
      return;
    }
    const bool row = k.rfind("gpue::row_", 0) == 0, col = k.rfind("gpue::col_", 0) == 0;
    if (!row && !col) return;
    const char* t = k.c_str() + k.find(", ") + 2;   // after the type
    if (k.find("_merged<") != std::string::npos) {
      const SweepArgs* d = *(const SweepArgs**)l.args[0];
      const MergeMap* map = *(const MergeMap**)l.args[1];
      std::map<int, bool> seen;
      for (unsigned i = 0; i < l.grid; ++i)
        if (map[i].inst >= 0 && !seen[map[i].inst]) {
          seen[map[i].inst] = true;
          sweep(l, d[map[i].inst], map[i].n, map[i].nblk, 64, std::atoi(t), row);
        }
      return;
    }
    int n = 0, var = 0, mode = 0;
    std::sscanf(t, "%d, %d, %d", &n, &var, &mode);
    if (k.find("_sweep_b<") != std::string::npos) {
      const SweepArgs* d = *(const SweepArgs**)l.args[0];
      const int bpi = *(int*)l.args[1];
      for (unsigned i = 0; i < l.grid / bpi; ++i) sweep(l, d[i], n, bpi, l.block, mode, row);
    } else {
      sweep(l, *(const SweepArgs*)l.args[0], n, (int)l.grid, l.block, mode, row);
    }
  }
};

static gpue_ctx* make(std::vector<int> n, int prec, int gauge) {
  gpue_params p;
  gpue_params_default(&p);
  p.dimnum = (int)n.size();
  n.resize(3, 1);
  p.xDim = n[0];
  p.yDim = n[1];
  p.zDim = n[2];
  p.hbar = p.mass = p.omegaX = p.omegaY = p.omegaZ = 1.0;
  p.xMax = p.yMax = p.zMax = 6.0;
  p.g = 10.0;
  p.gpe = 1;
  p.omega = 0.3;
  p.corotating = gauge;
  p.precision = prec;
  gpue_ctx* c = nullptr;
  if (gpue_create(&p, &c) != GPUE_OK) {
    std::printf("gpue_create failed\n");
    std::exit(1);
  }
  return c;
}

// A batch whose instances (a shape without merged kernels) defer their norms runs the
// variants its tuner tries, in both precisions and step parities: axes of 16 and 32
// points have tiles of less than a wave in some variants.  A member whose variants are
// set by hand stays in step with its group.
static void batch_norms() {
  const std::vector<std::vector<int>> shapes = {{64, 16}, {64, 32}, {48, 16}, {16, 48, 32}, {32, 16, 16}};
  for (int prec : {64, 32})
    for (const auto& shape : shapes)
      for (int gauge : {0, 1}) {
        Audit audit;
        fake::on_launch = [&](const fake::Launch& l) { audit(l); };
        gpue_ctx* c[2] = {make(shape, prec, gauge), make(shape, prec, gauge)};
        gpue_batch* b = nullptr;
        CHECK(gpue_batch_create(c, 2, &b) == GPUE_OK, "batch");
        CHECK(gpue_batch_evolve(b, 5, 0) == GPUE_OK, "evolve");
        CHECK(audit.from_partials > 0, "no norm was deferred");
        CHECK(gpue_batch_autotune(b, 0, 4, nullptr, nullptr) == GPUE_OK, "autotune");
        CHECK(gpue_batch_evolve(b, 37, 0) == GPUE_OK, "evolve");
        CHECK(gpue_batch_set_graph_mode(b, 2) == GPUE_OK, "graph mode");
        for (int v = 0; v < N_VARIANTS; ++v) {
          const int vars[3] = {v, v, v};
          gpue_set_variants(c[0], vars);
          CHECK(gpue_batch_evolve(b, 3, 0) == GPUE_OK, "evolve");
          gpue_set_variants(c[1], vars);
          CHECK(gpue_batch_evolve(b, 2, 0) == GPUE_OK, "evolve");
          gpue_batch_set_active(b, 0, v % 2);
          CHECK(gpue_batch_evolve(b, 3, 0) == GPUE_OK, "evolve");
        }
        double e[2], m[2];
        CHECK(gpue_batch_evolve(b, 2, 1) == GPUE_OK && gpue_batch_evolve(b, 2, 0) == GPUE_OK, "evolve");
        (void)gpue_batch_energy(b, e, m);
        CHECK(gpue_batch_evolve(b, 3, 0) == GPUE_OK, "evolve");
        gpue_batch_destroy(b);
        gpue_destroy(c[0]);
        gpue_destroy(c[1]);
      }
}

// A batch goes on with the schedule it was created for when a member's A_z becomes a
// field, which would lead the member's own even steps along z: kernels, axes and
// normalisations stay in step.  (Merged boxes of different sizes, and a group of one
// shape without merged kernels.)
static void batch_members_change() {
  const std::vector<std::vector<int>> shapes = {{64, 128, 64}, {64, 64, 96}, {128, 64, 64}, {64, 96, 64}, {64, 64, 64},
                                                 {48, 64, 16},  {48, 64, 16}};
  for (int prec : {64, 32}) {
    Audit audit;
    fake::on_launch = [&](const fake::Launch& l) { audit(l); };
    std::vector<gpue_ctx*> c;
    for (const auto& s : shapes) c.push_back(make(s, prec, 1));
    gpue_batch* b = nullptr;
    CHECK(gpue_batch_create(c.data(), (int)c.size(), &b) == GPUE_OK, "batch");
    CHECK(gpue_batch_set_graph_mode(b, 2) == GPUE_OK, "graph mode");
    for (size_t k = 0; k < c.size(); ++k) {
      const std::vector<double> az(c[k]->N, 0.1 + (double)k);
      CHECK(gpue_set_field(c[k], GPUE_FIELD_AZ, az.data()) == GPUE_OK, "A_z");
      CHECK(gpue_batch_set_active(b, (int)k, 0) == GPUE_OK && gpue_batch_set_active(b, (int)k, 1) == GPUE_OK, "active");
      for (int gstate : {0, 1}) CHECK(gpue_batch_evolve(b, 3, gstate) == GPUE_OK, "evolve");
    }
    CHECK(audit.kernels["gpue::col_merged"] > 0 && audit.kernels["gpue::col_sweep_b"] > 0, "kernels");
    gpue_batch_destroy(b);
    for (gpue_ctx* x : c) gpue_destroy(x);
  }
}

// What the steps read: the fields' kinds and, by step parity, the V table.
struct Fields {
  int v_kind, a_kind, k_kind;
  bool az_zero, t_dep, two_v;
  bool prog[5];
  explicit Fields(const gpue_ctx* c)
      : v_kind(c->v_kind), a_kind(c->a_kind), k_kind(c->k_kind), az_zero(c->az_zero), t_dep(c->t_dep),
        two_v(v_table(c, 0) != v_table(c, 1)) {
    for (int k = 0; k < 5; ++k) prog[k] = c->deq[k] != nullptr;
  }
  bool operator==(const Fields& o) const {
    return v_kind == o.v_kind && a_kind == o.a_kind && k_kind == o.k_kind && az_zero == o.az_zero && t_dep == o.t_dep &&
           two_v == o.two_v && std::memcmp(prog, o.prog, sizeof(prog)) == 0;
  }
};

// Time-dependent fields where the n-th device allocation fails: the call reports it and
// the fields stay as they were; with memory again it succeeds, and nothing leaks.
static void field_out_of_memory() {
  const char* td = "0.5*(x*x+y*y)*(1+0.1*sin(2*t))";
  for (int before = 0; before < 4; ++before)   // trap; V(t); a table of V; a table of A_x
    for (int which = GPUE_FIELD_V; which <= GPUE_FIELD_AZ; ++which) {
      const size_t live = fake::live();
      long fails = 0;
      for (long n = 0;; ++n) {
        gpue_ctx* c = make({32, 16, 16}, 64, 1);
        const std::vector<double> table(c->N, 0.5);
        if (before == 1) CHECK(gpue_set_field_eqn(c, GPUE_FIELD_V, td, nullptr, nullptr, 0) == GPUE_OK, "V(t)");
        if (before == 2) CHECK(gpue_set_field(c, GPUE_FIELD_V, table.data()) == GPUE_OK, "V");
        if (before == 3) CHECK(gpue_set_field(c, GPUE_FIELD_AX, table.data()) == GPUE_OK, "A_x");
        const Fields was(c);
        fake::mallocs_left = n;
        const gpue_status st = gpue_set_field_eqn(c, which, td, nullptr, nullptr, 0);
        fake::mallocs_left = -1;
        if (st != GPUE_OK) {
          ++fails;
          CHECK(st == GPUE_ENOMEM && Fields(c) == was, "field %d, allocation %ld: half set", which, n);
          CHECK(gpue_evolve(c, 0, 4, 1, 0, -1.0, nullptr, 0, nullptr) == GPUE_OK, "evolve after the failure");
          CHECK(gpue_set_field_eqn(c, which, td, nullptr, nullptr, 0) == GPUE_OK, "with memory");
        }
        CHECK(c->t_dep && c->deq[which] && c->tbase && (which != GPUE_FIELD_V || c->Vt2), "field %d", which);
        for (int a = 0; a < 3; ++a) CHECK(c->v_kind != V_TRAP_A || (c->Vt && c->vst[a]), "field %d: trap", which);
        CHECK(gpue_evolve(c, 0, 4, 1, 0, -1.0, nullptr, 0, nullptr) == GPUE_OK, "evolve");
        gpue_destroy(c);
        CHECK(fake::live() == live, "%zu allocations left", fake::live() - live);
        if (st == GPUE_OK) break;
      }
      CHECK(fails > 0, "no allocation failed");
    }
}

// psi to the device and back where no pinned memory can be had, one or two buffers, or all:
// parts of a chunk, several chunks, transfers that use threads.
static void pinned_memory() {
  const std::vector<std::vector<int>> shapes = {{16},          {32, 32},     {32, 48},   {128, 128},   {192, 192},    {384, 256},
                                                 {192, 192, 16}, {1024, 512}, {512, 384}, {192, 96, 96}, {2048, 1024}};
  for (long pinned : {0L, 1L, 2L, 3L, -1L})
    for (int prec : {64, 32})
      for (const auto& shape : shapes) {
        const size_t live = fake::live();
        fake::pinned_left = pinned;
        gpue_ctx* c = make(shape, prec, 0);
        std::vector<double> in(2 * c->N), out(2 * c->N, -1.0);
        for (size_t k = 0; k < in.size(); ++k) in[k] = 0.1 * (double)(k % 9973) + (double)k;
        for (int again = 0; again < 2; ++again) {
          CHECK(gpue_upload_wfc(c, in.data()) == GPUE_OK, "upload: %s", gpue_last_error(c));
          CHECK(gpue_download_wfc(c, out.data()) == GPUE_OK, "download: %s", gpue_last_error(c));
          bool same = true;
          for (size_t k = 0; k < in.size(); ++k) same = same && out[k] == (prec == 64 ? in[k] : (double)(float)in[k]);
          CHECK(same, "%ld pinned allocations, %d bits, %ld points", pinned, prec, c->N);
        }
        double e = 0.0, m = 0.0;
        CHECK(gpue_energy(c, &e, &m) == GPUE_OK, "energy: %s", gpue_last_error(c));
        gpue_destroy(c);
        fake::pinned_left = -1;
        CHECK(fake::live() == live, "%zu allocations left", fake::live() - live);
      }
}

// Step blocks of every length are captured once and kept, in both gstates.
static void step_blocks() {
  fake::on_launch = [&](const fake::Launch& l) {   // norms must be numbers
    if (l.kernel.rfind("gpue::k_set_double", 0) == 0) **(double**)l.args[0] = *(double*)l.args[1];
  };
  gpue_ctx* c = make({64, 32}, 64, 1);
  auto captures = [&](int n, int gstate) {
    const long before = fake::captures;
    CHECK(gpue_evolve(c, 0, n, gstate, 0, -1.0, nullptr, 0, nullptr) == GPUE_OK, "evolve: %s", gpue_last_error(c));
    return fake::captures - before;
  };
  for (int round = 0; round < 3; ++round)
    for (int gstate : {0, 1})
      for (int n = 2; n <= 32; n += 2) {
        const long got = captures(n, gstate);
        CHECK(got == (round == 0), "%ld captures for %d steps in round %d", got, n, round);
      }
  CHECK(captures(100, 0) == 0 && captures(100, 1) == 0, "three blocks of 32 and a tail");
  CHECK(gpue_set_g(c, 20.0) == GPUE_OK && captures(100, 0) == 2 && captures(100, 0) == 0, "dropped with the parameters");
  gpue_destroy(c);
}

// 1D runs: launches of at most 2^20 point steps and 1024 steps, up to each energy
// evaluation, that make up the call.
static void line_runs() {
  for (int n : {16, 1024, 2048, 4096})
    for (int every : {0, 700}) {
      std::vector<int> runs;
      fake::on_launch = [&](const fake::Launch& l) {
        if (l.kernel.rfind("gpue::k_set_double", 0) == 0) **(double**)l.args[0] = *(double*)l.args[1];
        if (l.kernel.rfind("gpue::line_steps", 0) == 0) runs.push_back(*(int*)l.args[1]);
      };
      gpue_ctx* c = make({n}, 64, 0);
      double e[8];
      CHECK(gpue_evolve(c, 0, 2500, 0, every, -1.0, e, 8, nullptr) == GPUE_OK, "evolve: %s", gpue_last_error(c));
      int done = 0;
      for (int r : runs) {
        CHECK(r > 0 && r <= 1024 && (long)r * n <= 1 << 20, "%d steps of %d points in one launch", r, n);
        if (every)
          for (int i = done; i < done + r - 1; ++i) CHECK(i % every != 0, "energy step %d inside a launch", i);
        done += r;
      }
      CHECK(done == 2500, "%d steps", done);
      gpue_destroy(c);
    }
}

// 1D: the profile and the traffic are those of the launches that the step loop makes.
static void line_reports() {
  for (int n : {64, 4096})
    for (int gstate : {0, 1}) {
      long lines = 0, sweeps = 0, steps = 0;
      void *in = nullptr, *psi = nullptr;
      fake::on_launch = [&](const fake::Launch& l) {
        if (l.kernel.rfind("gpue::k_set_double", 0) == 0) **(double**)l.args[0] = *(double*)l.args[1];
        if (l.kernel.rfind("gpue::line_steps", 0) == 0) {
          ++lines;
          steps = *(int*)l.args[1];
          in = (void*)((const SweepArgs*)l.args[0])->in;
        }
        if (l.kernel.find("_sweep<") != std::string::npos) ++sweeps;
      };
      gpue_ctx* c = make({n}, 64, 1);
      psi = c->psi;
      int kinds = 0;
      const char* names[4];
      double us[4], per[4], bytes = 0.0, count = 0.0;
      CHECK(gpue_sweep_profile(c, gstate, 5, 4, &kinds, names, us, per) == GPUE_OK, "profile: %s", gpue_last_error(c));
      CHECK(kinds == 1 && std::string(names[0]) == "line_steps" && lines > 0 && sweeps == 0, "%d kinds, %s", kinds, names[0]);
      CHECK(in != psi && c->psi == psi && c->results[0] == 1.0, "the state is untouched");
      CHECK(per[0] == 1.0 / steps, "%g launches a step", per[0]);
      CHECK(gpue_step_bytes(c, gstate, &bytes, &count) == GPUE_OK && count == 1.0 / steps && bytes == 32.0 * n / steps,
            "%g bytes a step", bytes);
      CHECK(gpue_set_graph_steps(c, 0) == GPUE_OK && gpue_step_bytes(c, gstate, &bytes, &count) == GPUE_OK && count == 1.0 &&
                gpue_sweep_profile(c, gstate, 5, 4, &kinds, names, us, per) == GPUE_OK && kinds == 1 && per[0] == 1.0 && sweeps > 0,
            "steps launched one by one");
      gpue_destroy(c);
    }
}

// A request of the service captures one block a phase where its chunks allow it.
static void service_captures() {
  fake::on_launch = [&](const fake::Launch& l) {
    if (l.kernel.rfind("gpue::k_set_double", 0) == 0) **(double**)l.args[0] = *(double*)l.args[1];
  };
  struct Case { int imag, real, every, captures; };
  for (const Case& k : {Case{40, 0, 100, 1}, Case{60, 0, 100, 1}, Case{100, 0, 100, 1}, Case{200, 0, 100, 1}, Case{20, 40, 100, 2},
                        Case{0, 90, 30, 1}, Case{41, 0, 100, 2}, Case{62, 0, 100, 2}, Case{4, 0, 100, 1}, Case{1, 0, 100, 0}}) {
    gpue_server* sv = nullptr;
    CHECK(gpue_server_create(0, 1e9, 2, &sv) == GPUE_OK, "server");
    gpue_ctx* like = make({64, 64}, 64, 0);
    for (int again = 0; again < 2; ++again) {   // a new context, then a reused one
      gpue_request r;
      std::memset(&r, 0, sizeof(r));
      r.params = like->p;
      r.max_imag_steps = k.imag;
      r.real_steps = k.real;
      r.check_every = k.every;
      r.quench_factor = 1.1;
      const long before = fake::captures;
      CHECK(gpue_server_submit(sv, &r, 1) == GPUE_OK && gpue_server_drain(sv, 20.0) == GPUE_OK, "request");
      gpue_result got;
      CHECK(gpue_server_poll(sv, &got, 1) == 1 && got.status == GPUE_OK && got.imag_steps == k.imag && got.real_steps == k.real,
            "status %d, %d + %d steps", got.status, (int)got.imag_steps, (int)got.real_steps);
      CHECK(fake::captures - before == k.captures, "%d + %d steps: %ld captures", k.imag, k.real, fake::captures - before);
    }
    gpue_server_destroy(sv);
    gpue_destroy(like);
  }
}

// A tuner that fails before it has chosen anything leaves a context with its default
// variants: the kernels of a real-time step are those from before.
static void tuner_fails() {
  gpue_ctx* c = make({128, 64, 192}, 64, 0);
  std::string kernels;
  fake::on_launch = [&](const fake::Launch& l) { kernels += l.kernel + "\n"; };
  auto step = [&]() {
    kernels.clear();
    CHECK(gpue_set_graph_steps(c, 0) == GPUE_OK && gpue_evolve(c, 0, 1, 1, 0, -1.0, nullptr, 0, nullptr) == GPUE_OK, "step");
    return kernels;
  };
  const std::string before = step();
  int was[3], now[3];
  gpue_get_variants(c, was);
  for (long n : {0L, 1L, 5L}) {
    fake::instantiates_left = n;
    CHECK(gpue_autotune(c, 2, now) != GPUE_OK, "the tuner");
    fake::instantiates_left = -1;
    CHECK(std::memcmp(was, now, sizeof(was)) == 0 && step() == before, "other kernels after a failed tuner");
  }
  gpue_destroy(c);
}

// The batch's tuner compares steps, not the captures before them: blocks of steps cost
// less than pairs here, but their captures more.
static void tuner_times_steps() {
  for (int steps : {20, 19, 4, 3}) {
    gpue_ctx* c[3] = {make({48, 64}, 64, 0), make({48, 64}, 64, 0), make({32, 64}, 64, 0)};
    gpue_batch* b = nullptr;
    CHECK(gpue_batch_create(c, 3, &b) == GPUE_OK, "batch");
    fake::capture_us = 5000;
    fake::replay_us = steps > 16 ? 200 : 0;
    double us = 0.0;
    int mode = -1;
    CHECK(gpue_batch_autotune(b, 0, steps, &us, &mode) == GPUE_OK, "autotune");
    fake::capture_us = fake::replay_us = 0;
    CHECK(us < 1000.0, "%g us a step", us);
    CHECK(steps < 16 || mode == 0, "mode %d", mode);
    gpue_batch_destroy(b);
    for (gpue_ctx* x : c) gpue_destroy(x);
  }
}

// The batch's tuner takes merged launches apart where launches by shape are faster, keeps
// them (and the contexts' variants) where they are not or where there is no memory to try.
static void tuner_regroups() {
  for (int slow : {0, 1, 2}) {   // merged launches; launches by shape; those, and no memory
    const size_t live = fake::live();
    Audit audit;
    std::vector<gpue_ctx*> c;
    for (int n : {64, 128, 64, 96}) c.push_back(make({n, 64}, 64, 1));
    c.push_back(make({48, 64}, 64, 1));   // has no merged kernels
    gpue_batch* b = nullptr;
    CHECK(gpue_batch_create(c.data(), (int)c.size(), &b) == GPUE_OK && gpue_batch_set_graph_mode(b, 2) == GPUE_OK, "batch");
    fake::on_launch = [&](const fake::Launch& l) {
      audit(l);
      if ((l.kernel.find("_merged") != std::string::npos) == (slow == 0))
        std::this_thread::sleep_for(std::chrono::microseconds(300));
    };
    fake::mallocs_left = slow == 2 ? 3 : -1;
    CHECK(gpue_batch_autotune(b, 0, 4, nullptr, nullptr) == GPUE_OK, "%s", gpue_batch_last_error(b));
    fake::mallocs_left = -1;
    fake::on_launch = [&](const fake::Launch& l) { audit(l); };
    audit.kernels.clear();
    CHECK(gpue_batch_set_graph_mode(b, 2) == GPUE_OK && gpue_batch_set_active(b, 1, 0) == GPUE_OK, "active");
    for (int gstate : {0, 1, 0}) CHECK(gpue_batch_evolve(b, 37, gstate) == GPUE_OK, "evolve");
    CHECK((audit.kernels["gpue::row_merged"] == 0) == (slow == 0) && audit.kernels["gpue::row_sweep_b"] > 0,
          "%ld merged row sweeps, slow %d", audit.kernels["gpue::row_merged"], slow);
    if (slow)
      for (int k = 0; k < 4; ++k)
        CHECK(c[k]->var[0] == MERGE_ROW && c[k]->var[1] == MERGE_COL, "variants of member %d", k);
    gpue_batch_destroy(b);
    for (gpue_ctx* x : c) gpue_destroy(x);
    CHECK(fake::live() == live, "%zu allocations left", fake::live() - live);
  }
}

// FP64 boxes share merged launches beyond four shapes, FP32 ones and planes always.
static void batch_boxes() {
  const std::vector<std::vector<int>> shapes = {{64, 64, 64}, {64, 64, 96}, {64, 96, 64}, {96, 64, 64}, {64, 64, 128}};
  for (int prec : {64, 32})
    for (int kinds = 1; kinds <= 5; ++kinds) {
      Audit audit;
      std::vector<gpue_ctx*> c;
      for (int k = 0; k < kinds + 2; ++k) c.push_back(make(shapes[k % kinds], prec, 1));
      c.push_back(make({64, 96}, prec, 1));
      gpue_batch* b = nullptr;
      CHECK(gpue_batch_create(c.data(), (int)c.size(), &b) == GPUE_OK, "batch");
      fake::on_launch = [&](const fake::Launch& l) { audit(l); };
      CHECK(gpue_batch_evolve(b, 3, 0) == GPUE_OK && gpue_batch_evolve(b, 3, 1) == GPUE_OK, "evolve");
      const bool by_shape = audit.kernels["gpue::col_sweep_b"] > 0;
      CHECK(audit.kernels["gpue::col_merged"] > 0, "the plane");
      CHECK(by_shape == (prec == 64 && kinds <= 4), "%d kinds of boxes, %d bits", kinds, prec);
      gpue_batch_destroy(b);
      for (gpue_ctx* x : c) gpue_destroy(x);
    }
}

int main(int argc, char** argv) {
  const std::map<std::string, std::function<void()>> checks = {
      {"batch_norms", batch_norms},
      {"batch_members_change", batch_members_change},
      {"field_out_of_memory", field_out_of_memory},
      {"pinned_memory", pinned_memory},
      {"step_blocks", step_blocks},
      {"line_runs", line_runs},
      {"service_captures", service_captures},
      {"line_reports", line_reports},
      {"tuner_fails", tuner_fails},
      {"batch_boxes", batch_boxes},
      {"tuner_times_steps", tuner_times_steps},
      {"tuner_regroups", tuner_regroups},
  };
  const auto it = checks.find(argc > 1 ? argv[1] : "");
  if (it == checks.end()) {
    std::printf("no such check\n");
    return 2;
  }
  it->second();
  std::printf(failures ? "%d failures\n" : "ok\n", failures);
  return failures != 0;
}
