// sht_batch.hip -- ensemble batches: members of uneven truncation and level
// count, grouped by grid, transformed by one launch per stage of all the
// smaller grids, beside the larger grids' own as branches of a hipGraph.
//
// Layout: for each group (members with the same nmax, im, jm) the batch owns
// one resident field batch -- canonical spectra in and out [K][2 * nf_group]
// and grid [nf_group][jm][im] -- and member j is the field range
// [f0_j, f0_j + nfield_j) of its group.  Each stage kernel of a group therefore
// covers all of the group's members in a single launch (its tiles are spread
// over the whole chip).  Groups on grids of up to 64 latitude pairs also share
// their launches (batch_units); groups on larger grids run beside them as
// branches of a captured graph, which forks from the launch stream and joins
// back.
#include <algorithm>
#include <map>
#include <new>
#include <tuple>

#include "sht_internal.h"

namespace sht {

struct BatchGroup {
  int nmax = 0, im = 0, jm = 0, nf = 0;
  bool can_share = false;  // its built-in shapes' results are those of the shared launches
  sht_plan *plan = nullptr;
  double *spec_in = nullptr, *grid = nullptr, *spec_out = nullptr;
  hipStream_t stream = nullptr;
  hipEvent_t done = nullptr;
};

struct BatchMember {
  int group = 0, f0 = 0, nf = 0;
};

int run_dir_on(sht_plan *plan, const double *spec_in, double *grid, double *spec_out, int nf,
               int dir, hipStream_t s);

}  // namespace sht

struct sht_batch {
  std::vector<sht::BatchGroup> groups;
  std::vector<sht::BatchMember> members;
  std::vector<std::vector<int>> units;  // group indexes, see batch_units
  bool share = true;                    // see pick_sharing
  hipEvent_t fork = nullptr;
  hipGraphExec_t exec[3] = {nullptr, nullptr, nullptr};
  hipGraph_t graph[3] = {nullptr, nullptr, nullptr};
};

namespace sht {

static void drop_graphs(sht_batch *b) {
  for (int d = 0; d < 3; ++d) {
    if (b->exec[d]) (void)hipGraphExecDestroy(b->exec[d]);
    if (b->graph[d]) (void)hipGraphDestroy(b->graph[d]);
    b->exec[d] = nullptr;
    b->graph[d] = nullptr;
  }
}

static void batch_release(sht_batch *b) {
  drop_graphs(b);
  for (auto &g : b->groups) {
    if (g.plan) sht_plan_destroy(g.plan);
    if (g.spec_in) (void)hipFree(g.spec_in);
    if (g.grid) (void)hipFree(g.grid);
    if (g.spec_out) (void)hipFree(g.spec_out);
    if (g.stream) (void)hipStreamDestroy(g.stream);
    if (g.done) (void)hipEventDestroy(g.done);
  }
  if (b->fork) (void)hipEventDestroy(b->fork);
  delete b;
}

// The independent pieces of a batch's work: all groups that can share their
// stages' launches (multi_available) as one piece of up to kMaxMulti groups,
// kMaxMultiBlocks workgroups and kMaxMultiGrid bytes of grids, largest first, and
// every other group on its own.  Shared launches because
// small groups' kernels neither fill the chip nor overlap: one after the
// other each pays its launch and its latency chain, and as branches of a graph
// they pay the hand-offs between queues.  12 members, T21/T42/T85, fp16, round
// trip: 84.5 us group by group, 89-110 us as graph branches, 55 us shared.  Large
// groups lose by it: a group's stages then no longer follow each other while its
// data are in the Infinity Cache.  T42 and T85 of 800 / 1200 / 1500 fields each (262 /
// 393 / 491 MB of grids), FP64, shared 228 / 399 / 568 us, graph branches 226 / 388 /
// 523; x6 205 / 293 / 402 and 205 / 284 / 397; T21 and T42 of 5000 (410 MB), x6 333 and 292.
constexpr size_t kMaxMultiGrid = 400000000;
static std::vector<std::vector<int>> batch_units(const sht_batch *b) {
  std::vector<int> shared;
  std::vector<std::vector<int>> units;
  for (int i = 0; i < (int)b->groups.size(); ++i) {
    if (b->share && b->groups[i].can_share)
      shared.push_back(i);
    else
      units.push_back({i});
  }
  auto grid_bytes = [&](int i) {
    return sizeof(double) * b->groups[i].nf * b->groups[i].jm * b->groups[i].im;
  };
  std::stable_sort(shared.begin(), shared.end(), [&](int x, int y) { return grid_bytes(x) > grid_bytes(y); });
  long blocks = 0;
  size_t bytes = 0;
  for (int i : shared) {
    const long more = multi_blocks(b->groups[i].plan->p, b->groups[i].nf);
    if (blocks == 0 || blocks + more > kMaxMultiBlocks || bytes + grid_bytes(i) > kMaxMultiGrid ||
        units.back().size() == kMaxMulti) {
      units.emplace_back();
      blocks = 0;
      bytes = 0;
    }
    units.back().push_back(i);
    blocks += more;
    bytes += grid_bytes(i);
  }
  return units;
}

static int enqueue_unit(sht_batch *b, const std::vector<int> &unit, int dir, hipStream_t s) {
  if (unit.size() == 1) {
    BatchGroup &g = b->groups[unit[0]];
    return run_dir_on(g.plan, g.spec_in, g.grid, g.spec_out, g.nf, dir, s);
  }
  MultiGroup m[kMaxMulti];
  const int n = (int)unit.size();
  for (int i = 0; i < n; ++i) {
    const BatchGroup &g = b->groups[unit[i]];
    m[i] = {&g.plan->p, g.spec_in, g.grid, g.spec_out, g.nf};
  }
  const bool f64 = m[0].p->prec == SHT_PREC_FP64;
  int rc = SHT_OK;
  if (dir != SHT_DIR_FORWARD) {
    rc = f64 ? launch_leg_inv_f64_multi(m, n, s) : launch_leg_inv_mixed_multi(m, n, s);
    if (!rc) rc = launch_fft_inv_multi(m, n, s);
  }
  if (!rc && dir != SHT_DIR_INVERSE) {
    rc = launch_fft_fwd_multi(m, n, s);
    if (!rc) rc = f64 ? launch_leg_fwd_f64_multi(m, n, s) : launch_leg_fwd_mixed_multi(m, n, s);
  }
  return rc;
}

// Enqueue every unit's work; with fork_join the units go to streams of their
// own (for capture into parallel graph branches), else all on s.
static int enqueue_all(sht_batch *b, int dir, hipStream_t s, bool fork_join) {
  if (fork_join) SHT_HIP(hipEventRecord(b->fork, s));
  for (const auto &u : b->units) {
    BatchGroup &g = b->groups[u[0]];
    const hipStream_t us = fork_join ? g.stream : s;
    if (fork_join) SHT_HIP(hipStreamWaitEvent(us, b->fork, 0));
    int rc = enqueue_unit(b, u, dir, us);
    if (rc) return rc;
    if (fork_join) {
      SHT_HIP(hipEventRecord(g.done, us));
      SHT_HIP(hipStreamWaitEvent(s, g.done, 0));
    }
  }
  return SHT_OK;
}

// All units of one direction on s: directly if there is one, else as a graph,
// captured on the first call.
static int run_units(sht_batch *b, int dir, hipStream_t s) {
  // a single piece has no branches to run side by side, and its launches take
  // less than a graph's
  if (b->units.size() == 1) return enqueue_all(b, dir, s, false);
  if (!b->exec[dir]) {
    // capture on a private stream so the caller's stream may be the legacy one
    hipStream_t cap = nullptr;
    SHT_HIP(hipStreamCreateWithFlags(&cap, hipStreamNonBlocking));
    hipError_t e = hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal);
    int rc = (e == hipSuccess) ? enqueue_all(b, dir, cap, true)
                               : fail(SHT_ERR_DEVICE, "sht_batch_run: hipStreamBeginCapture failed");
    hipGraph_t graph = nullptr;
    hipError_t e2 = hipStreamEndCapture(cap, &graph);
    (void)hipStreamDestroy(cap);
    if (rc) {
      if (graph) (void)hipGraphDestroy(graph);
      return rc;
    }
    if (e2 != hipSuccess) return fail(SHT_ERR_DEVICE, "sht_batch_run: hipStreamEndCapture failed");
    hipGraphExec_t exec = nullptr;
    if (hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) != hipSuccess) {
      (void)hipGraphDestroy(graph);
      return fail(SHT_ERR_DEVICE, "sht_batch_run: hipGraphInstantiate failed");
    }
    b->graph[dir] = graph;
    b->exec[dir] = exec;
  }
  SHT_HIP(hipGraphLaunch(b->exec[dir], s));
  return SHT_OK;
}

// Whether the groups that can share launches are to: times the round trip of
// those groups' shared launches against that of each group's own kernels (the
// tuned shapes), on scratch data and the plans' own Fourier scratch, and keeps
// sharing unless the latter is at least 3 % faster.  Without memory for the
// scratch data the choice stays.  Called while the batch is idle.
static int pick_sharing(sht_batch *b, int reps) {
  sht_batch t;  // the groups in question over scratch data
  b->share = true;
  for (const auto &u : batch_units(b))
    if (u.size() > 1)
      for (int i : u) t.groups.push_back(b->groups[i]);
  if (t.groups.empty()) return SHT_OK;
  t.fork = b->fork;
  int cur = 0, rc = SHT_OK;
  bool memory = true;
  hipStream_t s = nullptr;
  hipEvent_t e[2] = {nullptr, nullptr};
  SHT_HIP(hipGetDevice(&cur));
  SHT_HIP(hipSetDevice(t.groups[0].plan->p.device));
  for (auto &g : t.groups) g.spec_in = g.spec_out = g.grid = nullptr;
  for (auto &g : t.groups) {
    const size_t nspec = sizeof(double) * g.plan->p.K * 2 * g.nf, ngrid = sizeof(double) * g.nf * g.jm * g.im;
    memory = hipMalloc(&g.spec_in, nspec) == hipSuccess && hipMalloc(&g.grid, ngrid) == hipSuccess &&
             hipMemset(g.spec_in, 0, nspec) == hipSuccess && hipMemset(g.grid, 0, ngrid) == hipSuccess;
    g.spec_out = g.spec_in;
    if (!memory) break;
  }
  double best[2] = {0.0, 0.0};
  if (memory) {
    if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess || hipEventCreate(&e[0]) != hipSuccess ||
        hipEventCreate(&e[1]) != hipSuccess || hipDeviceSynchronize() != hipSuccess)
      rc = fail(SHT_ERR_DEVICE, "sht_batch_autotune: stream or event creation failed");
    // three interleaved rounds, as for the shapes: a drift hits both alike
    for (int round = 0; round < 6 && !rc; ++round) {
      t.share = round % 2 == 0;
      t.units = batch_units(&t);
      drop_graphs(&t);
      rc = run_units(&t, SHT_DIR_ROUNDTRIP, s);  // captures, loads code
      if (!rc) rc = run_units(&t, SHT_DIR_ROUNDTRIP, s);
      if (!rc && hipEventRecord(e[0], s) != hipSuccess) rc = fail(SHT_ERR_DEVICE, "sht_batch_autotune: hipEventRecord");
      for (int r = 0; r < reps && !rc; ++r) rc = run_units(&t, SHT_DIR_ROUNDTRIP, s);
      float ms = 0.f;
      if (!rc && (hipEventRecord(e[1], s) != hipSuccess || hipEventSynchronize(e[1]) != hipSuccess ||
                  hipEventElapsedTime(&ms, e[0], e[1]) != hipSuccess))
        rc = fail(SHT_ERR_DEVICE, "sht_batch_autotune: timing failed");
      double &x = best[t.share ? 0 : 1];
      if (!rc && (round < 2 || ms < x)) x = ms;
    }
    (void)hipDeviceSynchronize();
    b->share = rc || best[1] > 0.97 * best[0];
  } else {
    (void)hipGetLastError();
  }
  drop_graphs(&t);
  for (auto &g : t.groups) {
    if (g.spec_in) (void)hipFree(g.spec_in);
    if (g.grid) (void)hipFree(g.grid);
  }
  for (hipEvent_t x : e)
    if (x) (void)hipEventDestroy(x);
  if (s) (void)hipStreamDestroy(s);
  (void)hipSetDevice(cur);
  return rc;
}

}  // namespace sht

using namespace sht;

extern "C" {

int sht_batch_create(const sht_member_desc *members, int nmember, int precision, sht_batch **out) {
  if (!out) return fail(SHT_ERR_INVALID, "sht_batch_create: out is NULL");
  *out = nullptr;
  if (!members || nmember < 1) return fail(SHT_ERR_INVALID, "sht_batch_create: no members");
  sht_batch *b = new (std::nothrow) sht_batch;
  if (!b) return fail(SHT_ERR_NOMEM, "sht_batch_create: host allocation failed");
  std::map<std::tuple<int, int, int>, int> gid;
  for (int j = 0; j < nmember; ++j) {
    const sht_member_desc &d = members[j];
    if (d.nfield < 1) {
      batch_release(b);
      return fail(SHT_ERR_INVALID, "sht_batch_create: member with nfield < 1");
    }
    auto key = std::make_tuple(d.nmax, d.im, d.jm);
    auto it = gid.find(key);
    int g;
    if (it == gid.end()) {
      g = (int)b->groups.size();
      gid[key] = g;
      BatchGroup grp;
      grp.nmax = d.nmax;
      grp.im = d.im;
      grp.jm = d.jm;
      b->groups.push_back(grp);
    } else {
      g = it->second;
    }
    BatchMember m;
    m.group = g;
    m.f0 = b->groups[g].nf;
    m.nf = d.nfield;
    b->groups[g].nf += d.nfield;
    b->members.push_back(m);
  }
  hipError_t e = hipEventCreateWithFlags(&b->fork, hipEventDisableTiming);
  if (e != hipSuccess) {
    batch_release(b);
    return fail(SHT_ERR_DEVICE, "sht_batch_create: hipEventCreate failed");
  }
  for (auto &g : b->groups) {
    sht_desc d{g.nmax, g.im, g.jm, g.nf, precision, 0};
    int rc = sht_plan_create(&d, &g.plan);
    if (rc) {
      std::string keep = sht_last_error();
      batch_release(b);
      return fail(rc, "sht_batch_create: " + keep);
    }
    const size_t K = (size_t)(g.nmax + 1) * (g.nmax + 2) / 2;
    const size_t nspec = K * 2 * g.nf, ngrid = (size_t)g.nf * g.jm * g.im;
    if (hipMalloc(&g.spec_in, sizeof(double) * nspec) != hipSuccess ||
        hipMalloc(&g.spec_out, sizeof(double) * nspec) != hipSuccess ||
        hipMalloc(&g.grid, sizeof(double) * ngrid) != hipSuccess) {
      batch_release(b);
      return fail(SHT_ERR_NOMEM, "sht_batch_create: member state allocation failed");
    }
    if (hipStreamCreateWithFlags(&g.stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&g.done, hipEventDisableTiming) != hipSuccess) {
      batch_release(b);
      return fail(SHT_ERR_DEVICE, "sht_batch_create: stream/event creation failed");
    }
    // defined contents before the first run
    if (hipMemset(g.spec_in, 0, sizeof(double) * nspec) != hipSuccess ||
        hipMemset(g.spec_out, 0, sizeof(double) * nspec) != hipSuccess ||
        hipMemset(g.grid, 0, sizeof(double) * ngrid) != hipSuccess) {
      batch_release(b);
      return fail(SHT_ERR_DEVICE, "sht_batch_create: hipMemset failed");
    }
  }
  if (hipDeviceSynchronize() != hipSuccess) {
    batch_release(b);
    return fail(SHT_ERR_DEVICE, "sht_batch_create: device synchronisation failed");
  }
  for (auto &g : b->groups) g.can_share = multi_available(g.plan->p, g.nf);
  b->units = batch_units(b);
  *out = b;
  return SHT_OK;
}

void sht_batch_destroy(sht_batch *b) {
  if (b) batch_release(b);
}

int sht_batch_member(const sht_batch *b, int j, double **spec_in, double **grid, double **spec_out,
                     int *ld) {
  if (!b || j < 0 || j >= (int)b->members.size())
    return fail(SHT_ERR_INVALID, "sht_batch_member: bad batch or member index");
  const BatchMember &m = b->members[j];
  const BatchGroup &g = b->groups[m.group];
  if (spec_in) *spec_in = g.spec_in + 2 * (size_t)m.f0;
  if (spec_out) *spec_out = g.spec_out + 2 * (size_t)m.f0;
  if (grid) *grid = g.grid + (size_t)m.f0 * g.jm * g.im;
  if (ld) *ld = 2 * g.nf;
  return SHT_OK;
}

int sht_batch_run(sht_batch *b, int dir, void *stream) {
  if (!b) return fail(SHT_ERR_INVALID, "sht_batch_run: batch is NULL");
  if (dir < SHT_DIR_INVERSE || dir > SHT_DIR_ROUNDTRIP)
    return fail(SHT_ERR_INVALID, "sht_batch_run: bad direction");
  return run_units(b, dir, (hipStream_t)stream);
}

int sht_batch_autotune(sht_batch *b, int reps, const char *cache_path) {
  return sht_batch_autotune_flags(b, reps, cache_path, 0);
}

int sht_batch_autotune_flags(sht_batch *b, int reps, const char *cache_path, int flags) {
  if (!b) return fail(SHT_ERR_INVALID, "sht_batch_autotune: batch is NULL");
  // the tuner runs on a stream of its own through each group plan's Fourier
  // scratch: a graph or eager run still in flight on any stream would share it
  SHT_HIP(hipDeviceSynchronize());
  // graphs captured before hold the old kernels (dropped before the first shape
  // changes, so that an error leaves none): capture again on the next run
  drop_graphs(b);
  int rc = SHT_OK;
  for (auto &g : b->groups) {
    rc = sht_plan_autotune_flags(g.plan, g.nf, reps, cache_path, flags, nullptr);
    if (rc) break;
  }
  if (!rc) rc = pick_sharing(b, reps);
  b->units = batch_units(b);
  if (rc) return rc;
  SHT_HIP(hipDeviceSynchronize());
  return SHT_OK;
}

int sht_batch_run_eager(sht_batch *b, int dir, void *stream) {
  if (!b) return fail(SHT_ERR_INVALID, "sht_batch_run_eager: batch is NULL");
  if (dir < SHT_DIR_INVERSE || dir > SHT_DIR_ROUNDTRIP)
    return fail(SHT_ERR_INVALID, "sht_batch_run_eager: bad direction");
  return enqueue_all(b, dir, (hipStream_t)stream, false);
}

}  // extern "C"
