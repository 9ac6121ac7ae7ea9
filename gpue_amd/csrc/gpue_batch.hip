// gpue_batch.hip -- many independent problems advanced together.
//
// Instances of one precision, dimension and gauge whose axes have merged kernels
// (sweep_merged.h; FP64 boxes only where they have more shapes than there are streams) form
// a merged group: every sweep of the step is one launch over all of them, whatever their
// sizes.  Others group by shape (grid sizes and kernel variants
// too): for every sweep one batched kernel covers the group, blocks [i*bpi, (i+1)*bpi)
// working on instance i.  The instances' SweepArgs live in a device array.  GPUE's gauge
// order alternates with the step parity (src/evolution.cu:837,842).  When the
// odd-step sweep list is a prefix of the even-step one in kernel kind, both
// parities share one launch per position, with per-instance flags; otherwise each parity
// has its own sequence.  Imaginary-time norms are reduced in the next step's opening
// sweep (groups whose partials allow it), with one batched finalize at the end of a
// call, or else by a batched finalize after every step.  The groups run on at most
// four streams (the process's hardware queues; the groups with the most work
// get one each, the others share the last), with blocks of 16 and 2 consecutive steps
// of a group captured once per gstate as HIP graphs and replayed, so the groups of
// different shapes (the small ones latency bound) overlap on the device.
// Device memory is allocated only in gpue_batch_create and by the tuner, which compares
// merged launches with launches by shape.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <chrono>
#include <cmath>
#include <cstring>
#include <numeric>
#include <vector>

#include "ctx_internal.h"
#include "sweep_merged.h"

using namespace gpue;

namespace {

struct Merged {                     // a merged launch (sweep_merged.h): which blocks a workgroup takes
  MergeMap* map = nullptr;          // device array [grid]
  int grid = 0, lds = 0;
};

struct BSeq {                       // one launch sequence of a group for (gstate, phase)
  std::vector<Sweep> keys;          // kernel kind per position (flags come per instance)
  int mask = 3;                     // step parities it serves (bit p: parity p)
  std::vector<SweepArgs*> dargs;    // per position: device array [members]
  std::vector<std::vector<SweepArgs>> hargs;
  // imaginary time: the opening sweep of a call's first step, which scales by the norm
  // slot also where the group defers its norms to the next step's opening sweep
  SweepArgs* dopen = nullptr;
  std::vector<SweepArgs> hopen;
  std::vector<Merged> merged;       // per position, merged groups only
  FinArgs* dfin = nullptr;          // imaginary time: device array [members]
  std::vector<FinArgs> hfin;
  bool any = true;                  // some member takes this sequence (else it is not launched)
};

// Steps of a group's captured graphs: a replay costs some 10-20 us beside its steps,
// the pair covers what is left.
constexpr int kGraphLens[] = {16, 2};
constexpr int kGraphKinds = 2;

struct Group {
  std::vector<int> members;
  gpue_ctx* proto;                  // first member: shape and variants
  bool merged = false;              // members of different shapes, launched together
  int vars[3] = {};                 // kernel variants (unmerged): its contexts' when the batch
                                    // was created, then what its tuner chose
  bool defer = false;               // norms reduced in the next step's opening sweep (can_defer, of vars)
  std::vector<Sweep> sched[2][2];   // [gstate][parity]
  std::vector<BSeq> seqs[2][2];     // [gstate][phase]
  hipStream_t stream = nullptr;     // one of the batch's streams (not owned)
  hipGraph_t graph[2][kGraphKinds] = {};   // [gstate][kGraphLens]
  hipGraphExec_t gexec[2][kGraphKinds] = {};
  int var(int axis) const { return !merged ? vars[axis] : axis == 0 ? MERGE_ROW : MERGE_COL; }
};

// Problems that may share launches with others of their kind: every axis has a merged
// kernel, and the variants are those it runs (the defaults of small grids).
bool can_merge(const gpue_ctx* c) {
  if (c->p.dimnum < 2) return false;
  for (int a = 0; a < c->p.dimnum; ++a) {
    int lds = 0;
    if (!merged_shape(c->prec, a == 0, c->dims[a], &lds)) return false;
    if (a == 0 ? c->var[a] != MERGE_ROW : c->var[a] != MERGE_COL) return false;
  }
  return true;
}
bool same_kind_of_problem(const gpue_ctx* a, const gpue_ctx* b) {
  return a->prec == b->prec && a->p.dimnum == b->p.dimnum && a->p.corotating == b->p.corotating &&
         a->az_zero == b->az_zero && a->p.device == b->p.device;
}

// Workgroups (= partials) of a member's sweep.
int blocks_of(const Group& g, const gpue_ctx* c, const Sweep& s) {
  const int n = c->dims[s.axis], var = g.var(s.axis);
  return s.row ? sweep_blocks(c->prec, true, n, var, c->dims[1] * c->dims[2], 1)
               : sweep_blocks(c->prec, false, n, var, c->dims[0], s.axis == 1 ? c->dims[2] : c->dims[1]);
}

// The normalisation of a member's sweep (schedule's, for its own sizes): of the whole
// transform where K is applied, of the axis with a gauge operator.
double inv_n(const gpue_ctx* c, const Sweep& s) {
  if (s.invN == 0.0) return 0.0;
  const bool k = s.row ? s.mode == RM_K || s.mode == RM_FULL : s.mode == CM_K;
  return k ? 1.0 / (double)c->N : 1.0 / c->dims[s.axis];
}

// Whether every member's norm can be left to the next step's opening sweep (as
// defer_norm decides for one context).  Asked again whenever the variants change: some
// have tiles of less than a wave for axes of 16 and 32 points.
bool can_defer(const Group& g, const std::vector<gpue_ctx*>& ctx) {
  for (int idx : g.members) {
    const gpue_ctx* c = ctx[idx];
    if (c->p.dimnum < 2) return false;
    for (int par = 0; par < 2; ++par) {
      const Sweep& open = g.sched[0][par].front();
      if (blocks_of(g, c, g.sched[0][par].back()) >= 4096 ||
          !sweep_full_waves(c->prec, open.row, c->dims[open.axis], g.var(open.axis)))
        return false;
    }
  }
  return true;
}

bool same_shape(const gpue_ctx* a, const gpue_ctx* b) {
  return a->prec == b->prec && a->p.dimnum == b->p.dimnum && a->dims[0] == b->dims[0] && a->dims[1] == b->dims[1] &&
         a->dims[2] == b->dims[2] && a->var[0] == b->var[0] && a->var[1] == b->var[1] && a->var[2] == b->var[2] &&
         a->p.corotating == b->p.corotating && a->az_zero == b->az_zero && a->p.device == b->p.device;
}

bool same_kind(const Sweep& x, const Sweep& y) { return x.row == y.row && x.axis == y.axis && x.mode == y.mode; }

constexpr size_t kBatchStreams = 4;   // the process's hardware queues

// the shorter list's kinds are a prefix of the longer list's
bool mergeable(const std::vector<Sweep>& a, const std::vector<Sweep>& b) {
  const size_t n = std::min(a.size(), b.size());
  for (size_t k = 0; k < n; ++k)
    if (!same_kind(a[k], b[k])) return false;
  return true;
}

// The instances as groups, and what belongs to them.
struct Grouping {
  std::vector<Group> groups;
  // at most four streams (default priority), owned here: the groups with the
  // most work get one each, the others share the last
  std::vector<hipStream_t> streams;
  std::vector<size_t> by_work;     // group indices, most work first (launch order of the replays)
  std::vector<hipEvent_t> join_ev;   // per group (graph mode 1)
};

}  // namespace

struct gpue_batch : Grouping {
  int device = 0;
  std::vector<gpue_ctx*> ctx;
  std::vector<int> active;
  std::vector<int> cls;            // parity class: the instance's step parity at phase 0
  int phase = 0;
  // graph mode 1: one graph per pair of steps for the whole batch, captured on
  // `origin` with a branch per shape group (forked to the group streams and
  // joined back), so a pair of steps of every group is one launch
  int graph_mode = 0;
  hipStream_t origin = nullptr;
  hipEvent_t fork_ev = nullptr;
  hipGraph_t wgraph[2] = {nullptr, nullptr};
  hipGraphExec_t wexec[2] = {nullptr, nullptr};
  double* terms = nullptr;         // pinned: 6 energy terms per instance (gpue_batch_energy)
  std::string err;
};

static gpue_status bfail(gpue_batch* b, gpue_status s, const std::string& m) {
  if (b) b->err = m;
  return s;
}

#define BHIP(b, expr)                                                                           \
  do {                                                                                          \
    hipError_t e_ = (expr);                                                                     \
    if (e_ != hipSuccess) return bfail((b), GPUE_EHIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

// Fill the host argument arrays of every sequence from the members' current
// state; returns true when the set of sequences that are launched changed
// (captured graphs hold the launches, so they are captured again).
static bool fill_args(gpue_batch* b) {
  bool pattern = false;
  for (Group& g : b->groups)
    for (int gs = 0; gs < 2; ++gs)
      for (int ph = 0; ph < 2; ++ph)
        for (BSeq& s : g.seqs[gs][ph]) {
          bool any = false;
          for (size_t m = 0; m < g.members.size(); ++m) {
            const int idx = g.members[m];
            gpue_ctx* c = b->ctx[idx];
            const int par = (b->cls[idx] + ph) % 2;   // the instance's step parity at this phase
            const bool in = b->active[idx] && ((s.mask >> par) & 1);
            any = any || in;
            // The group's schedule, which the launches and their maps were laid out for: a
            // member's own may change after (A_z set to a field leads even steps along z).
            const std::vector<Sweep>& sc = g.sched[gs][par];
            const Phys phys = make_phys(c, gs, 0);
            for (size_t k = 0; k < s.keys.size(); ++k) {
              const bool on = in && k < sc.size();
              const Sweep& sw = on ? sc[k] : s.keys[k];
              SweepArgs& a = s.hargs[k][m];
              std::memset(&a, 0, sizeof(a));
              // every context holds the tables of both plans for each of its
              // axes; a missing one would leave the sweep off rather than fault
              const auto twi = c->tw.find(2 * c->dims[sw.axis] + (g.var(sw.axis) & 1));
              a.active = on && twi != c->tw.end();
              a.in = c->psi;
              a.out = c->psi;
              a.tw = twi == c->tw.end() ? nullptr : twi->second;
              a.ph = phys;
              a.lines = c->dims[1] * c->dims[2];
              a.axis = sw.axis;
              a.gauge_axis = sw.axis;
              a.flags = sw.flags;
              a.invN = inv_n(c, sw);
              a.norm_in = c->results;
              a.partials = c->partials;
              if (k == 0 && s.dopen) {
                s.hopen[m] = a;
                if (g.defer) {   // the previous step's norm from its partials (its last sweep's)
                  a.flags |= F_SCALE_PART;
                  a.norm_nb = blocks_of(g, c, g.sched[gs][1 - par].back());
                  a.norm_scale = c->d[0] * c->d[1] * c->d[2];
                  a.norm_out = c->results;
                }
              }
            }
            if (s.dfin) {
              // the partials come from the instance's F_NORM sweep (its last)
              FinArgs& f = s.hfin[m];
              std::memset(&f, 0, sizeof(f));
              f.active = in;
              f.nb = blocks_of(g, c, sc.back());
              f.na = 1;
              f.mode = 1;
              f.scale = c->d[0] * c->d[1] * c->d[2];
              f.partials = c->partials;
              f.out = c->results;
            }
          }
          if (any != s.any) pattern = true;
          s.any = any;
        }
  return pattern;
}

static gpue_status upload_args(gpue_batch* b) {
  for (Group& g : b->groups)
    for (int gs = 0; gs < 2; ++gs)
      for (int ph = 0; ph < 2; ++ph)
        for (BSeq& s : g.seqs[gs][ph]) {
          for (size_t k = 0; k < s.keys.size(); ++k)
            BHIP(b, hipMemcpy(s.dargs[k], s.hargs[k].data(), s.hargs[k].size() * sizeof(SweepArgs),
                              hipMemcpyHostToDevice));
          if (s.dopen)
            BHIP(b, hipMemcpy(s.dopen, s.hopen.data(), s.hopen.size() * sizeof(SweepArgs), hipMemcpyHostToDevice));
          if (s.dfin)
            BHIP(b, hipMemcpy(s.dfin, s.hfin.data(), s.hfin.size() * sizeof(FinArgs), hipMemcpyHostToDevice));
        }
  return GPUE_OK;
}

// One step (one phase) of group g for gstate, on the group's stream.  `first`: the first
// step of a call (deferring groups scale by the norm slot).  Groups that do not defer
// close every imaginary-time step with their finalize.
static gpue_status launch_group_phase(gpue_batch* b, Group& g, int gs, int ph, bool first) {
  gpue_ctx* c = g.proto;
  for (BSeq& s : g.seqs[gs][ph]) {
    if (!s.any) continue;   // the step parity no member has
    for (size_t k = 0; k < s.keys.size(); ++k) {
      const Sweep& sw = s.keys[k];
      const SweepArgs* args = k == 0 && first && s.dopen ? s.dopen : s.dargs[k];
      bool handled = true;
      hipError_t e;
      if (g.merged) {
        const Merged& m = s.merged[k];
        e = launch_sweep_merged(c->prec, sw.row, sw.mode, sw.flags, gs, args, m.map, m.grid, m.lds, g.stream);
      } else {
        const int n = c->dims[sw.axis];
        const int lx = sw.row ? c->dims[1] * c->dims[2] : c->dims[0];
        const int others = sw.row ? 1 : (sw.axis == 1 ? c->dims[2] : c->dims[1]);
        e = launch_sweep_batched(c->prec, sw.row, n, g.var(sw.axis), sw.mode, sw.flags, gs, args,
                                 (int)g.members.size(), lx, others, g.stream, &handled);
      }
      if (!handled || e != hipSuccess) return bfail(b, GPUE_EHIP, "batched sweep launch");
    }
    if (s.dfin && !g.defer) {
      hipError_t e = launch_finalize_batched(s.dfin, (int)g.members.size(), g.stream);
      if (e != hipSuccess) return bfail(b, GPUE_EHIP, "batched finalize launch");
    }
  }
  return GPUE_OK;
}

static gpue_status launch_phase(gpue_batch* b, int gs, int ph, bool first) {
  for (size_t k : b->by_work) {
    gpue_status st = launch_group_phase(b, b->groups[k], gs, ph, first);
    if (st != GPUE_OK) return st;
  }
  return GPUE_OK;
}

// The norms that deferring groups' last step (phase ph) left in its partials, into the
// norm slots: every call ends with them there.
static gpue_status settle_norms(gpue_batch* b, int ph) {
  for (Group& g : b->groups) {
    if (!g.defer) continue;
    for (BSeq& s : g.seqs[0][ph])
      if (s.any && launch_finalize_batched(s.dfin, (int)g.members.size(), g.stream) != hipSuccess)
        return bfail(b, GPUE_EHIP, "batched finalize launch");
  }
  return GPUE_OK;
}

static void drop_group_graphs(Group& grp) {
  for (int g = 0; g < 2; ++g)
    for (int j = 0; j < kGraphKinds; ++j) {
      if (grp.gexec[g][j]) (void)hipGraphExecDestroy(grp.gexec[g][j]);
      if (grp.graph[g][j]) (void)hipGraphDestroy(grp.graph[g][j]);
      grp.gexec[g][j] = nullptr;
      grp.graph[g][j] = nullptr;
    }
}

static void drop_whole_graphs(gpue_batch* b) {
  for (int g = 0; g < 2; ++g) {
    if (b->wexec[g]) (void)hipGraphExecDestroy(b->wexec[g]);
    if (b->wgraph[g]) (void)hipGraphDestroy(b->wgraph[g]);
    b->wexec[g] = nullptr;
    b->wgraph[g] = nullptr;
  }
}

static void drop_batch_graphs(gpue_batch* b) {
  for (Group& grp : b->groups) drop_group_graphs(grp);
  drop_whole_graphs(b);
}

static gpue_status sync_groups(gpue_batch* b) {
  for (hipStream_t st : b->streams)
    if (st) BHIP(b, hipStreamSynchronize(st));
  if (b->origin) BHIP(b, hipStreamSynchronize(b->origin));
  return GPUE_OK;
}

// Graph mode 1: capture a pair of steps of every group as one graph on
// `origin`: fork to each group's stream, launch its two phases there, join back.
static gpue_status build_whole_graph(gpue_batch* b, int gstate) {
  BHIP(b, hipStreamBeginCapture(b->origin, hipStreamCaptureModeThreadLocal));
  gpue_status st = GPUE_OK;
  hipError_t e = hipEventRecord(b->fork_ev, b->origin);
  for (size_t k = 0; k < b->groups.size() && st == GPUE_OK && e == hipSuccess; ++k) {
    Group& grp = b->groups[k];
    e = hipStreamWaitEvent(grp.stream, b->fork_ev, 0);
    if (e == hipSuccess) st = launch_group_phase(b, grp, gstate, 0, false);
    if (st == GPUE_OK && e == hipSuccess) st = launch_group_phase(b, grp, gstate, 1, false);
    if (st == GPUE_OK && e == hipSuccess) e = hipEventRecord(b->join_ev[k], grp.stream);
    if (st == GPUE_OK && e == hipSuccess) e = hipStreamWaitEvent(b->origin, b->join_ev[k], 0);
  }
  hipGraph_t g = nullptr;
  const hipError_t ec = hipStreamEndCapture(b->origin, &g);
  if (st != GPUE_OK || e != hipSuccess || ec != hipSuccess) {
    if (g) (void)hipGraphDestroy(g);
    return st != GPUE_OK ? st : bfail(b, GPUE_EHIP, "whole-batch graph capture");
  }
  if (hipGraphInstantiate(&b->wexec[gstate], g, nullptr, nullptr, 0) != hipSuccess) {
    (void)hipGraphDestroy(g);
    return bfail(b, GPUE_EHIP, "whole-batch graph instantiate");
  }
  b->wgraph[gstate] = g;
  return GPUE_OK;
}

// Capture kGraphLens[j] steps (from phase 0, norms deferred where the group does) of a group.
static gpue_status build_group_graph(gpue_batch* b, Group& grp, int gstate, int j) {
  BHIP(b, hipStreamBeginCapture(grp.stream, hipStreamCaptureModeThreadLocal));
  gpue_status st = GPUE_OK;
  for (int s = 0; s < kGraphLens[j] && st == GPUE_OK; ++s) st = launch_group_phase(b, grp, gstate, s & 1, false);
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(grp.stream, &g);
  if (st != GPUE_OK || e != hipSuccess) {
    if (g) (void)hipGraphDestroy(g);
    return st != GPUE_OK ? st : bfail(b, GPUE_EHIP, "batch graph capture");
  }
  if (hipGraphInstantiate(&grp.gexec[gstate][j], g, nullptr, nullptr, 0) != hipSuccess) {
    (void)hipGraphDestroy(g);
    grp.gexec[gstate][j] = nullptr;
    return bfail(b, GPUE_EHIP, "batch graph instantiate");
  }
  grp.graph[gstate][j] = g;
  return GPUE_OK;
}

// Lay out a merged launch: each member's blocks in runs of a workgroup's worth, the
// members with the longest axes first (their blocks take longest).  Workgroups are dealt
// to the 8 XCDs round robin; those whose tiles share 128-byte lines of psi (the quarter
// tiles of one default tile) are given positions on one XCD, so that the lines are
// fetched into one L2 (xcd_tile does this within a lone launch).
static gpue_status build_map(gpue_batch* b, const Group& g, const Sweep& sw, Merged& out) {
  constexpr int XCDS = 8;
  std::vector<size_t> order(g.members.size());
  std::iota(order.begin(), order.end(), size_t(0));
  std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) {
    return b->ctx[g.members[x]]->dims[sw.axis] > b->ctx[g.members[y]]->dims[sw.axis];
  });
  std::vector<MergeMap> queue[XCDS];
  for (size_t m : order) {
    const gpue_ctx* c = b->ctx[g.members[m]];
    const int n = c->dims[sw.axis], nblk = blocks_of(g, c, sw);
    int lds = 0;
    const int wg = merged_shape(c->prec, sw.row, n, &lds);
    if (wg <= 0) return GPUE_EUNSUPPORTED;
    out.lds = std::max(out.lds, lds);
    const int per = MERGE_WG / wg;                              // blocks of a workgroup
    const int share = sw.row ? per : std::max(per, MERGE_TILES);   // blocks that stay on one XCD
    for (int k0 = 0; k0 < nblk; k0 += share) {
      std::vector<MergeMap>* q = &queue[0];
      for (int x = 1; x < XCDS; ++x)
        if (queue[x].size() < q->size()) q = &queue[x];
      for (int k = k0; k < std::min(k0 + share, nblk); k += per) q->push_back(MergeMap{(int)m, k, n, nblk});
    }
  }
  size_t longest = 0;
  for (const auto& q : queue) longest = std::max(longest, q.size());
  std::vector<MergeMap> map(longest * XCDS, MergeMap{-1, 0, 0, 0});   // -1: nothing to do
  for (int x = 0; x < XCDS; ++x)
    for (size_t i = 0; i < queue[x].size(); ++i) map[i * XCDS + x] = queue[x][i];
  out.grid = (int)map.size();
  if (hipMalloc((void**)&out.map, map.size() * sizeof(MergeMap)) != hipSuccess) return GPUE_ENOMEM;
  return hipMemcpy(out.map, map.data(), map.size() * sizeof(MergeMap), hipMemcpyHostToDevice) == hipSuccess ? GPUE_OK
                                                                                                            : GPUE_EHIP;
}

static void free_grouping(Grouping& gr) {
  for (hipStream_t st : gr.streams)
    if (st) (void)hipStreamSynchronize(st);
  for (Group& g : gr.groups) drop_group_graphs(g);
  for (hipEvent_t ev : gr.join_ev)
    if (ev) (void)hipEventDestroy(ev);
  for (Group& g : gr.groups)
    for (int gs = 0; gs < 2; ++gs)
      for (int ph = 0; ph < 2; ++ph)
        for (BSeq& s : g.seqs[gs][ph]) {
          for (auto* p : s.dargs)
            if (p) (void)hipFree(p);
          if (s.dfin) (void)hipFree(s.dfin);
          if (s.dopen) (void)hipFree(s.dopen);
          for (Merged& m : s.merged)
            if (m.map) (void)hipFree(m.map);
        }
  for (hipStream_t st : gr.streams)
    if (st) (void)hipStreamDestroy(st);
  gr = Grouping();
}

// Whether instances of c's kind run merged by default.  FP64 boxes do beyond four shapes
// only: up to there each shape has a stream, and its own kernels, with twiddles up front
// and the registers of one length, win (us a step, merged / by shape: eight 64^3 62.6 / 56.3
// and rotating in real time 105.5 / 82.7, four 96^3 121 / 107, three shapes 52.4 / 39.0, four
// rotating 201 / 170; six rotating 123 / 143, twelve 189 / 334).  FP32 boxes and planes gain
// from merging with equal shapes too (sweep_merged.h).
static bool merge_pays(const gpue_batch* b, const gpue_ctx* c) {
  if (c->p.dimnum != 3 || c->prec != 64) return true;
  std::vector<const gpue_ctx*> shapes;
  for (const gpue_ctx* x : b->ctx) {
    if (!can_merge(x) || !same_kind_of_problem(x, c)) continue;
    if (std::none_of(shapes.begin(), shapes.end(), [&](const gpue_ctx* y) { return same_shape(x, y); })) shapes.push_back(x);
    if (shapes.size() > kBatchStreams) return true;
  }
  return false;
}

// Group the instances (those with merged kernels together if `merge`) and lay out their
// launches; a part of it may be there after a failure (free_grouping).
static gpue_status make_grouping(gpue_batch* b, bool merge, Grouping& gr) {
  for (int i = 0; i < (int)b->ctx.size(); ++i) {
    bool placed = false;
    const bool mg = merge && can_merge(b->ctx[i]) && merge_pays(b, b->ctx[i]);
    for (Group& g : gr.groups)
      if (mg ? g.merged && same_kind_of_problem(g.proto, b->ctx[i]) : !g.merged && same_shape(g.proto, b->ctx[i])) {
        g.members.push_back(i);
        placed = true;
        break;
      }
    if (!placed) {
      Group g;
      g.proto = b->ctx[i];
      g.merged = mg;
      std::copy(g.proto->var, g.proto->var + 3, g.vars);
      g.members.push_back(i);
      gr.groups.push_back(g);
    }
  }
  {
    // A process gets four hardware queues (GPU_MAX_HW_QUEUES); more streams
    // than that share queues in FIFO order wherever the runtime places them.
    // So the groups are ranked by work (instances x points), the first three
    // get a stream each and the rest share the last one, where their graphs
    // run one after another.
    std::vector<size_t> order(gr.groups.size());
    std::iota(order.begin(), order.end(), size_t(0));
    auto work = [&](size_t k) {
      double n = 0.0;
      for (int idx : gr.groups[k].members) n += (double)b->ctx[idx]->N;
      return n;
    };
    std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) { return work(x) > work(y); });
    const size_t ns = std::min<size_t>(gr.groups.size(), kBatchStreams);
    for (size_t i = 0; i < ns; ++i) {
      hipStream_t st = nullptr;
      if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess) return GPUE_EHIP;
      gr.streams.push_back(st);
    }
    for (size_t r = 0; r < order.size(); ++r) gr.groups[order[r]].stream = gr.streams[std::min(r, ns - 1)];
    gr.by_work = order;
  }
  gr.join_ev.assign(gr.groups.size(), nullptr);
  for (hipEvent_t& ev : gr.join_ev)
    if (hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) return GPUE_EHIP;
  for (Group& g : gr.groups)
    for (int gs = 0; gs < 2; ++gs) {
      // imaginary time: the norm slot holds 1.0 whenever nothing is pending, so
      // the renormalising first sweep is always safe
      for (int par = 0; par < 2; ++par) schedule(g.proto, gs, par, gs == 0, g.sched[gs][par]);
      if (gs == 0) g.defer = can_defer(g, b->ctx);
      const std::vector<Sweep>& s0 = g.sched[gs][0];
      const std::vector<Sweep>& s1 = g.sched[gs][1];
      for (int ph = 0; ph < 2; ++ph) {
        std::vector<BSeq>& seqs = g.seqs[gs][ph];
        if (mergeable(s0, s1)) {
          seqs.resize(1);
          seqs[0].keys = s0.size() >= s1.size() ? s0 : s1;
          seqs[0].mask = 3;
        } else {
          seqs.resize(2);
          for (int par = 0; par < 2; ++par) {
            seqs[par].keys = g.sched[gs][par];
            seqs[par].mask = 1 << par;
          }
        }
        const size_t M = g.members.size();
        for (BSeq& s : seqs) {
          s.hargs.assign(s.keys.size(), std::vector<SweepArgs>(M));
          s.dargs.assign(s.keys.size(), nullptr);
          for (size_t k = 0; k < s.keys.size(); ++k)
            if (hipMalloc((void**)&s.dargs[k], M * sizeof(SweepArgs)) != hipSuccess) return GPUE_ENOMEM;
          if (g.merged) {
            s.merged.resize(s.keys.size());
            for (size_t k = 0; k < s.keys.size(); ++k) {
              const gpue_status st = build_map(b, g, s.keys[k], s.merged[k]);
              if (st != GPUE_OK) return st;
            }
          }
          if (gs == 0) {
            s.hopen.assign(M, SweepArgs{});
            if (hipMalloc((void**)&s.dopen, M * sizeof(SweepArgs)) != hipSuccess) return GPUE_ENOMEM;
          }
          if (gs == 0) {
            s.hfin.assign(M, FinArgs{});
            if (hipMalloc((void**)&s.dfin, M * sizeof(FinArgs)) != hipSuccess) return GPUE_ENOMEM;
          }
        }
      }
    }
  return GPUE_OK;
}

extern "C" {

void gpue_batch_destroy(gpue_batch* b) {
  if (!b) return;
  if (b->origin) (void)hipStreamSynchronize(b->origin);
  for (hipStream_t st : b->streams)
    if (st) (void)hipStreamSynchronize(st);
  drop_batch_graphs(b);
  free_grouping(*b);
  if (b->fork_ev) (void)hipEventDestroy(b->fork_ev);
  if (b->origin) (void)hipStreamDestroy(b->origin);
  if (b->terms) (void)hipHostFree(b->terms);
  delete b;
}

const char* gpue_batch_last_error(const gpue_batch* b) { return b ? b->err.c_str() : "null batch"; }

gpue_status gpue_batch_set_graph_mode(gpue_batch* b, int mode) {
  if (!b || mode < 0 || mode > 2) return GPUE_EINVAL;
  if (mode != b->graph_mode) {
    gpue_status st = sync_groups(b);
    if (st != GPUE_OK) return st;
    drop_batch_graphs(b);
    b->graph_mode = mode;
  }
  return GPUE_OK;
}

gpue_status gpue_batch_create(gpue_ctx* const* ctxs, int n, gpue_batch** out) {
  if (!ctxs || n <= 0 || !out) return GPUE_EINVAL;
  *out = nullptr;
  gpue_batch* b = new gpue_batch();
  for (int i = 0; i < n; ++i) {
    gpue_ctx* c = ctxs[i];
    if (!c || c->t_dep || c->ramp_type || c->p.device != ctxs[0]->p.device) {
      gpue_batch_destroy(b);
      return GPUE_EINVAL;   // time-dependent V or ramp and mixed devices are run per context
    }
    b->ctx.push_back(c);
    b->active.push_back(1);
    b->cls.push_back(c->next_step % 2);
  }
  b->device = ctxs[0]->p.device;
  if (hipSetDevice(b->device) != hipSuccess ||
      hipHostMalloc((void**)&b->terms, (size_t)n * 6 * sizeof(double), hipHostMallocDefault) != hipSuccess) {
    gpue_batch_destroy(b);
    return GPUE_EHIP;
  }
  if (hipStreamCreateWithFlags(&b->origin, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreateWithFlags(&b->fork_ev, hipEventDisableTiming) != hipSuccess) {
    gpue_batch_destroy(b);
    return GPUE_EHIP;
  }
  {
    const gpue_status st = make_grouping(b, true, *b);
    if (st != GPUE_OK) {
      gpue_batch_destroy(b);
      return st;
    }
  }
  fill_args(b);
  if (upload_args(b) != GPUE_OK) {
    gpue_batch_destroy(b);
    return GPUE_EHIP;
  }
  *out = b;
  return GPUE_OK;
}

gpue_status gpue_batch_set_active(gpue_batch* b, int index, int active) {
  if (!b || index < 0 || index >= (int)b->ctx.size()) return GPUE_EINVAL;
  b->active[index] = active ? 1 : 0;
  // graphs keep their argument pointers, only the contents change, unless a
  // sequence starts or stops being launched (every evolve call ends synchronised,
  // so no replay is in flight here)
  if (fill_args(b)) drop_batch_graphs(b);
  return upload_args(b);
}

// Advance every active instance by nsteps steps of gstate.
gpue_status gpue_batch_evolve(gpue_batch* b, int nsteps, int gstate) {
  if (!b || nsteps < 0 || (gstate != 0 && gstate != 1)) return GPUE_EINVAL;
  // settle per-instance state on the instances' own streams first
  bool changed = false;
  for (size_t i = 0; i < b->ctx.size(); ++i) {
    gpue_ctx* c = b->ctx[i];
    if (!b->active[i]) continue;
    if (gstate == 1 && c->pending_norm) {
      if (apply_pending(c) != GPUE_OK) return bfail(b, GPUE_EHIP, c->err);
    }
    BHIP(b, hipStreamSynchronize(c->stream));
    const int cls = (c->next_step + b->phase) % 2;   // parity at phase 0 of the current pair
    if (cls != b->cls[i]) {
      b->cls[i] = cls;
      changed = true;
    }
  }
  if (changed) {
    if (fill_args(b)) drop_batch_graphs(b);
    gpue_status st = upload_args(b);
    if (st != GPUE_OK) return st;
  }
  int s = 0, last_phase = 0;
  auto single = [&](bool first) {   // the next step, launched on its own
    const gpue_status st = launch_phase(b, gstate, b->phase, first);
    last_phase = b->phase;
    b->phase ^= 1;
    ++s;
    return st;
  };
  // imaginary time: the first step scales by the norm slots, not by partials of a call
  // before (which other work may have replaced)
  const bool slots = gstate == 0 && std::any_of(b->groups.begin(), b->groups.end(), [](const Group& g) { return g.defer; });
  if (slots && s < nsteps) {
    gpue_status st = single(true);
    if (st != GPUE_OK) return st;
  }
  if (b->phase == 1 && s < nsteps) {   // up to the start of a pair
    gpue_status st = single(false);
    if (st != GPUE_OK) return st;
  }
  if (nsteps - s >= 2 && b->graph_mode == 1) {
    if (!b->wexec[gstate]) {
      gpue_status st = build_whole_graph(b, gstate);
      if (st != GPUE_OK) return st;
    }
    // the whole graph runs on `origin` after the groups' earlier work, and their
    // later work waits for it
    for (size_t k = 0; k < b->groups.size(); ++k) {
      BHIP(b, hipEventRecord(b->join_ev[k], b->groups[k].stream));
      BHIP(b, hipStreamWaitEvent(b->origin, b->join_ev[k], 0));
    }
    for (; nsteps - s >= 2; s += 2) BHIP(b, hipGraphLaunch(b->wexec[gstate], b->origin));
    last_phase = 1;
    BHIP(b, hipEventRecord(b->fork_ev, b->origin));
    for (Group& grp : b->groups) BHIP(b, hipStreamWaitEvent(grp.stream, b->fork_ev, 0));
  }
  if (b->graph_mode == 2) {   // no graphs: every phase launched on its own (kernel traces)
    while (nsteps - s >= 2) {
      gpue_status st = single(false);
      if (st == GPUE_OK) st = single(false);
      if (st != GPUE_OK) return st;
    }
  }
  // blocks of steps, the groups' graphs interleaved across their streams, the group
  // with the most work (the critical path) first
  for (int j = 0; j < kGraphKinds; ++j) {
    const int len = kGraphLens[j];
    if (nsteps - s < len) continue;
    for (Group& grp : b->groups)
      if (!grp.gexec[gstate][j]) {
        gpue_status st = build_group_graph(b, grp, gstate, j);
        if (st != GPUE_OK) return st;
      }
    for (; nsteps - s >= len; s += len)
      for (size_t k : b->by_work) BHIP(b, hipGraphLaunch(b->groups[k].gexec[gstate][j], b->groups[k].stream));
    last_phase = 1;
  }
  if (s < nsteps) {
    gpue_status st = single(false);
    if (st != GPUE_OK) return st;
  }
  if (gstate == 0 && nsteps > 0) {
    gpue_status st = settle_norms(b, last_phase);
    if (st != GPUE_OK) return st;
  }
  {
    gpue_status st = sync_groups(b);
    if (st != GPUE_OK) return st;
  }
  for (size_t i = 0; i < b->ctx.size(); ++i) {
    if (!b->active[i]) continue;
    b->ctx[i]->next_step += nsteps;
    if (gstate == 0) b->ctx[i]->pending_norm = true;
  }
  return GPUE_OK;
}

// Host time per step of `steps` steps of the whole batch, after as many (twice, for an
// odd number: from the same phase) that capture every graph the current choice needs.
// A capture in the timed steps outweighs what candidates differ by: blocks of 16 steps
// of sixteen 128^2 instances added 15 us to a step of 27.
static gpue_status time_batch(gpue_batch* b, int gstate, int steps, double* us) {
  gpue_status st = gpue_batch_evolve(b, steps, gstate);
  if (st == GPUE_OK && (steps & 1)) st = gpue_batch_evolve(b, steps, gstate);
  if (st != GPUE_OK) return st;
  const auto t0 = std::chrono::steady_clock::now();
  st = gpue_batch_evolve(b, steps, gstate);   // returns after the groups' streams finished
  if (st != GPUE_OK) return st;
  *us = std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count() / steps;
  return GPUE_OK;
}

// Every member of group g takes variant v on axis a; the launch arguments and
// graphs of the batch follow.
static gpue_status set_group_variant(gpue_batch* b, Group& g, int a, int v) {
  g.vars[a] = v;
  g.defer = can_defer(g, b->ctx);
  for (int idx : g.members) {
    gpue_ctx* c = b->ctx[idx];
    int vars[3] = {c->var[0], c->var[1], c->var[2]};
    vars[a] = v;
    gpue_status st = gpue_set_variants(c, vars);
    if (st != GPUE_OK) return bfail(b, st, c->err);
  }
  if (fill_args(b)) drop_batch_graphs(b);
  drop_group_graphs(g);   // the other groups' launches stay as they are
  drop_whole_graphs(b);
  return upload_args(b);
}

// The arguments of a grouping that has just come into use.
static gpue_status load_grouping(gpue_batch* b) {
  fill_args(b);
  return upload_args(b);
}

// The time per step of the batch, and the variants of its unmerged groups that lower it:
// coordinate descent over the groups, those with the most points first, then each axis.
static gpue_status tune_groups(gpue_batch* b, int gstate, int steps, double* best) {
  gpue_status st = time_batch(b, gstate, steps, best);
  std::vector<size_t> order(b->groups.size());
  for (size_t k = 0; k < order.size(); ++k) order[k] = k;
  std::sort(order.begin(), order.end(), [&](size_t x, size_t y) {
    return b->groups[x].proto->N * (long)b->groups[x].members.size() >
           b->groups[y].proto->N * (long)b->groups[y].members.size();
  });
  for (size_t k = 0; k < order.size() && st == GPUE_OK; ++k) {
    Group& g = b->groups[order[k]];
    if (g.merged) continue;   // merged launches run one set of variants
    for (int a = 0; a < g.proto->p.dimnum && st == GPUE_OK; ++a) {
      const int keep = g.vars[a];
      int pick = keep;
      // row sweeps: plan and twiddle loading (variants 0-3); strided: plan and tile width (0-5)
      const int nv = a == 0 ? 4 : N_VARIANTS;
      for (int v = 0; v < nv && st == GPUE_OK; ++v) {
        if (v == keep) continue;
        st = set_group_variant(b, g, a, v);
        double us = 0.0;
        if (st == GPUE_OK) st = time_batch(b, gstate, steps, &us);
        if (st == GPUE_OK && us < *best) {
          *best = us;
          pick = v;
        }
      }
      if (st == GPUE_OK && g.vars[a] != pick) st = set_group_variant(b, g, a, pick);
    }
  }
  return st;
}

gpue_status gpue_batch_autotune(gpue_batch* b, int gstate, int steps, double* us_per_step, int* graph_mode) {
  if (!b || steps < 2 || (gstate != 0 && gstate != 1)) return GPUE_EINVAL;
  gpue_status st = sync_groups(b);
  if (st != GPUE_OK) return st;
  // save every instance's state: psi into its scratch buffer, the step counter,
  // the pending norm and its value
  const size_t n = b->ctx.size();
  std::vector<int> next(n), pend(n), cls = b->cls;
  std::vector<double> nrm(n);
  const int phase = b->phase;
  for (size_t i = 0; i < n; ++i) {
    gpue_ctx* c = b->ctx[i];
    next[i] = c->next_step;
    pend[i] = c->pending_norm;
    BHIP(b, hipMemcpyAsync(c->tmp, c->psi, c->N * c->esz, hipMemcpyDeviceToDevice, c->stream));
    BHIP(b, hipMemcpyAsync(&nrm[i], c->results, sizeof(double), hipMemcpyDeviceToHost, c->stream));
    BHIP(b, hipStreamSynchronize(c->stream));
  }
  double best = 0.0;
  st = tune_groups(b, gstate, steps, &best);
  // Launches by shape, which have variants to choose, in place of merged ones: they win
  // where a few groups fill the chip (us a step in imaginary time with rotation, merged /
  // by shape and tuned: eight 512^2 FP64 84 / 73, sixty-four 256^2 FP64 138 / 120), and
  // lose where there are more shapes than streams (fifteen 128^2-512^2 FP32 59 / 68).
  // Merged launches stay unless more than the timings' noise is gained.
  bool merged = false;
  for (const Group& g : b->groups) merged = merged || g.merged;
  if (st == GPUE_OK && merged) {
    std::vector<std::array<int, 3>> vars(n);
    for (size_t i = 0; i < n; ++i) std::copy(b->ctx[i]->var, b->ctx[i]->var + 3, vars[i].begin());
    Grouping by_shape;
    if (make_grouping(b, false, by_shape) != GPUE_OK) {
      (void)hipGetLastError();   // no memory to try it: the batch stays merged
    } else {
      drop_batch_graphs(b);
      std::swap((Grouping&)*b, by_shape);
      double us = 0.0;
      st = load_grouping(b);
      if (st == GPUE_OK) st = tune_groups(b, gstate, steps, &us);
      if (st == GPUE_OK && us < 0.99 * best) {
        best = us;
      } else {
        (void)sync_groups(b);
        drop_batch_graphs(b);
        std::swap((Grouping&)*b, by_shape);
        for (size_t i = 0; i < n; ++i) (void)gpue_set_variants(b->ctx[i], vars[i].data());
        const gpue_status back = load_grouping(b);
        if (st == GPUE_OK) st = back;
      }
    }
    free_grouping(by_shape);
  }
  // then the graph mode: per-group graphs or one graph for the whole batch
  if (st == GPUE_OK) {
    const int m0 = b->graph_mode == 2 ? 0 : b->graph_mode, m1 = 1 - m0;
    st = gpue_batch_set_graph_mode(b, m0);
    double us0 = best, us1 = 0.0;
    if (st == GPUE_OK) st = time_batch(b, gstate, steps, &us0);
    if (st == GPUE_OK) st = gpue_batch_set_graph_mode(b, m1);
    if (st == GPUE_OK) st = time_batch(b, gstate, steps, &us1);
    if (st == GPUE_OK && us0 <= us1) st = gpue_batch_set_graph_mode(b, m0);
    best = std::min(us0, us1);
  }
  // restore the states (also after a failure, as far as the device allows)
  gpue_status rs = sync_groups(b);
  for (size_t i = 0; i < n; ++i) {
    gpue_ctx* c = b->ctx[i];
    if (hipMemcpyAsync(c->psi, c->tmp, c->N * c->esz, hipMemcpyDeviceToDevice, c->stream) != hipSuccess ||
        hipMemcpyAsync(c->results, &nrm[i], sizeof(double), hipMemcpyHostToDevice, c->stream) != hipSuccess ||
        hipStreamSynchronize(c->stream) != hipSuccess)
      rs = bfail(b, GPUE_EHIP, "restoring an instance after tuning");
    c->next_step = next[i];
    c->pending_norm = pend[i];
  }
  b->cls = cls;
  b->phase = phase;
  fill_args(b);
  drop_batch_graphs(b);
  if (rs == GPUE_OK) rs = upload_args(b);
  if (st == GPUE_OK) st = rs;
  if (st == GPUE_OK && us_per_step) *us_per_step = best;
  if (st == GPUE_OK && graph_mode) *graph_mode = b->graph_mode;
  return st;
}

gpue_status gpue_batch_energy(gpue_batch* b, double* energy, double* mu) {
  if (!b || !energy || !mu) return GPUE_EINVAL;
  const size_t n = b->ctx.size();
  for (size_t i = 0; i < n; ++i) {   // queue every instance's evaluation first
    gpue_status st = energy_launch_graph(b->ctx[i], b->terms + 6 * i);
    if (st != GPUE_OK) return bfail(b, st, b->ctx[i]->err);
  }
  gpue_status out = GPUE_OK;
  for (size_t i = 0; i < n; ++i) {
    gpue_ctx* c = b->ctx[i];
    BHIP(b, hipStreamSynchronize(c->stream));
    energy_combine(c, b->terms + 6 * i, &energy[i], &mu[i]);
    if (!std::isfinite(energy[i]) && out == GPUE_OK) out = bfail(b, GPUE_ENONFINITE, "energy is not finite");
  }
  return out;
}

}  // extern "C"
