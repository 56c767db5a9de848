// runtime_check.cpp -- the host side of the runtime (fivonagi_amd/csrc/
// fv_runtime.cpp) on a stand-in for the HIP runtime (hip/hip_runtime.h here),
// one check per run (argv[1]).  The kernels are stand-ins too: a step attempt is
// always accepted.  Prints "ok", or what was wrong.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>

#include "../../fivonagi_amd/csrc/fv_adjoint.h"
#include "../../fivonagi_amd/csrc/fv_types.h"
#include "../../include/fivonagi.h"

namespace {
std::string trace;                       // launches: s = step (and its collect), c = collection
void note(char what, int phase, int collect) {
  trace += what + std::to_string(phase) + (what == 's' && collect > 0 ? "+c " : " ");
}
}  // namespace

extern "C" {
hipError_t fv_launch_step(const fv::InstDesc* d, const fv::WorkItem*, const uint64_t*, int,
                          int phase, int n, fv::Ctl*, fv::SyncSlots*, int, int, int, int,
                          int collect, hipStream_t) {
  fake::launch([=] {
    note('s', phase, collect);
    for (int k = 0; k < n; ++k) {
      fv::Ctl& o = d[k].ctl[(phase + 1) & 1];
      o = d[k].ctl[phase & 1];
      if (o.n_acc >= o.target_acc || !(o.T < o.T_stop)) continue;
      o.T += o.dt;
      o.cur ^= 1;
      ++o.n_acc;
      ++o.n_att;
    }
  });
  return hipSuccess;
}
hipError_t fv_launch_settle(const fv::InstDesc* d, int n, int phase, fv::Ctl* mirror, hipStream_t) {
  fake::launch([=] {
    for (int k = 0; k < n; ++k) {
      d[k].ctl[(phase + 1) & 1] = d[k].ctl[phase & 1];
      if (mirror) mirror[k] = d[k].ctl[phase & 1];
    }
  });
  return hipSuccess;
}
hipError_t fv_launch_targets(const fv::InstDesc* d, int n, int phase, const int64_t* targets,
                             int64_t target, double T_stop, hipStream_t) {
  fake::launch([=] {
    for (int k = 0; k < n; ++k) {
      d[k].ctl[phase & 1].target_acc = targets ? targets[k] : target;
      d[k].ctl[phase & 1].T_stop = T_stop;
    }
  });
  return hipSuccess;
}
hipError_t fv_launch_collect(const fv::InstDesc*, int, int, int phase, hipStream_t) {
  fake::launch([=] { note('c', phase, 0); });
  return hipSuccess;
}
hipError_t fv_launch_taylor_ghosts(const fv::InstDesc*, int, int, int, int, hipStream_t) {
  return hipSuccess;
}
hipError_t fv_step_waves_per_cu(int* w, int fp64) { *w = fp64 ? 8 : 16; return hipSuccess; }
hipError_t fv_adj_occupancy(int* w) { *w = 8; return hipSuccess; }
hipError_t fv_scratch_get(void**, size_t*) { return hipErrorInvalidValue; }
// (no check runs the adjoint)
hipError_t fv_adj_reverse(const fv::AdjDesc*, const fv::AdjItem*, const int32_t*, int, int,
                          fv::StateSlot, fv::StateSlot, int, int, hipStream_t) { return 1; }
hipError_t fv_adj_begin(const fv::AdjDesc*, int, size_t, int, int, fv::SyncSlots*, int,
                        hipStream_t) { return 1; }
hipError_t fv_adj_segment(const fv::AdjDesc*, int, int, int, int, fv::StateSlot, fv::InstDesc*,
                          fv::Ctl*, hipStream_t) { return 1; }
hipError_t fv_adj_back(const fv::InstDesc*, int, size_t, int, hipStream_t) { return 1; }
hipError_t fv_adj_log(const fv::AdjDesc*, int, int, hipStream_t) { return 1; }
hipError_t fv_adj_end(const fv::AdjDesc*, int, size_t, int, hipStream_t) { return 1; }
}

namespace {

#define EXPECT(cond, ...)                                    \
  do {                                                       \
    if (!(cond)) {                                           \
      std::printf("line %d: %s: ", __LINE__, #cond);         \
      std::printf(__VA_ARGS__);                              \
      std::printf("\n");                                     \
      return 1;                                              \
    }                                                        \
  } while (0)

fivonagi_params grid(int nx, int ny, int bc = FIVONAGI_BC_ZEROGRAD) {
  fivonagi_params p;
  std::memset(&p, 0, sizeof(p));
  p.nx = nx; p.ny = ny;
  p.dx = p.dy = 0.05;
  p.beta = 3.5; p.delta = 1e-4;
  p.cfl_max = 1.0; p.cfl_wish = 0.9;
  p.dt0 = 0.005;
  p.bc = bc;
  p.cfl_mode = FIVONAGI_CFL_ALL;
  return p;
}

fivonagi_ctx* context(const std::vector<fivonagi_params>& ps) {
  static std::vector<float> q;                 // (of a large grid nothing is read)
  size_t n = 0;
  for (const auto& p : ps) n = std::max(n, (size_t)p.nx * p.ny);
  if (4 * n < fake::kLarge) q.assign(n, 0.25f);
  std::vector<const float*> host(3 * ps.size(), q.data());
  static const float some = 0.f;
  if (4 * n >= fake::kLarge) host.assign(3 * ps.size(), &some);
  fivonagi_ctx* c = nullptr;
  if (fivonagi_init(&c, ps.data(), (int)ps.size(), host.data()) != 0) {
    std::printf("init: %s\n", fivonagi_last_error());
    std::exit(1);
  }
  return c;
}

}  // namespace

// A Taylor field that leaves no room for its ghost ring (4 GiB): the cells are
// written into the grid before each attempt, so the attempt before it must have
// been collected by then.
static int check_collect_without_ring() {
  for (int nx : {64, 32768}) {
    fivonagi_ctx* c = context({grid(nx, nx, FIVONAGI_BC_TAYLOR)});
    fivonagi_collect_opts o;
    std::memset(&o, 0, sizeof(o));
    o.eta = 1.0;
    EXPECT(fivonagi_set_collect(c, 0, &o) == 0, "%s", fivonagi_last_error());
    trace.clear();
    EXPECT(fivonagi_enqueue(c, 6) == 0, "%s", fivonagi_last_error());
    const char* want = nx == 64 ? "s0 s1+c s2+c s3+c s4+c s5+c c5 "
                                : "s0 c0 s1 c1 s2 c2 s3 c3 s4 c4 s5 c5 ";
    EXPECT(trace == want, "%d: %s", nx, trace.c_str());
    fivonagi_destroy(c);
  }
  return 0;
}

// A download whose second copy is refused: when the call returns, nothing of it
// may still write the staging buffer, which another context may have by then.
static int check_download_error() {
  for (int nx : {100, 1500}) {                 // one wait; a ring of slots
    fivonagi_ctx* c = context({grid(nx, nx)});
    EXPECT(fivonagi_step(c, 1) == 0, "%s", fivonagi_last_error());
    std::vector<float> q(3 * (size_t)nx * nx);
    float* f[3] = {q.data(), q.data() + (size_t)nx * nx, q.data() + 2 * (size_t)nx * nx};
    fake::st().fail_copy = 1;
    EXPECT(fivonagi_collect(c, 0, f[0], f[1], f[2], nullptr, nullptr, nullptr, nullptr) != 0, "%d",
           nx);
    for (const auto* s : fake::st().streams)
      EXPECT(s->queued.empty(), "%d: %zu copies in flight", nx, s->queued.size());
    fake::st().fail_copy = -1;
    EXPECT(fivonagi_collect(c, 0, f[0], f[1], f[2], nullptr, nullptr, nullptr, nullptr) == 0, "%s",
           fivonagi_last_error());
    fivonagi_destroy(c);
  }
  return 0;
}

// A download by a caller whose current device is another than the context's
// (every launch before it done: only copies are left to do).
static int check_download_device() {
  for (int nx : {100, 1500}) {
    fivonagi_ctx* c = context({grid(nx, nx)});
    EXPECT(fivonagi_step(c, 1) == 0, "%s", fivonagi_last_error());
    std::vector<float> q((size_t)nx * nx);
    fake::device() = 1;
    EXPECT(fivonagi_collect(c, 0, q.data(), q.data(), q.data(), nullptr, nullptr, nullptr,
                            nullptr) == 0, "%d: %s", nx, fivonagi_last_error());
    EXPECT(fake::device() == 1, "device %d", fake::device());
    EXPECT(q[5] == 0.25f, "%g", (double)q[5]);
    fake::device() = 0;
    fivonagi_destroy(c);
  }
  return 0;
}

// Attempts enqueued while the caller captures the stream: accepted where they
// are launches alone; refused where the stop conditions have to be set first,
// which the replays would set again, from host memory used for other targets by
// then.
static int check_enqueue_under_capture() {
  for (int n : {1, 3}) {
    fivonagi_ctx* c = context(std::vector<fivonagi_params>(n, grid(64, 64)));
    hipStream_t s;
    (void)hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
    EXPECT(fivonagi_set_stream(c, s) == 0, "%s", fivonagi_last_error());
    for (bool first : {true, false}) {
      hipGraph_t g;
      (void)hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
      const int rc = fivonagi_enqueue(c, 3);
      (void)hipStreamEndCapture(s, &g);
      EXPECT((rc != 0) == first, "%d instances, first %d: %d", n, first, rc);
      EXPECT(g->nodes.size() == (first ? 0u : 3u), "%zu nodes", g->nodes.size());
      (void)hipGraphDestroy(g);
      if (first) EXPECT(fivonagi_enqueue(c, 3) == 0, "%s", fivonagi_last_error());
    }
    EXPECT(fivonagi_set_stream(c, nullptr) == 0, "%s", fivonagi_last_error());
    (void)hipStreamDestroy(s);
    fivonagi_destroy(c);
  }
  return 0;
}

// The autotuner keeps the fastest of its trials: the split the context started
// with where that is it -- also when another was chosen meanwhile -- and one of
// the others where those are.
static int check_autotune() {
  std::vector<std::vector<fivonagi_params>> all = {
      {grid(400, 400)}, {grid(1024, 1024)}, {grid(4096, 1024)}, {grid(8192, 2048)},
      std::vector<fivonagi_params>(16, grid(512, 512)), {grid(200, 300), grid(700, 100)}};
  all.back()[0].rows_per_wave = 21;
  for (const auto& ps : all) {
    fivonagi_ctx* c = context(ps);
    fivonagi_info_t a, b;
    int32_t rows = 0;
    EXPECT(fivonagi_info(c, 0, &a) == 0, "%s", fivonagi_last_error());
    for (int fastest : {0, 3, 0, 15, 0}) {
      auto& g = fake::st();
      g.elapsed.assign(100, 2.0f);
      g.elapsed[fastest] = 1.0f;
      g.asked = 0;
      EXPECT(fivonagi_autotune(c, 20, &rows) == 0, "%s", fivonagi_last_error());
      EXPECT(fivonagi_info(c, 0, &b) == 0, "%s", fivonagi_last_error());
      const bool same = a.n_items == b.n_items && a.skew == b.skew && a.rotate == b.rotate;
      EXPECT(fastest != 0 || same, "%dx%d: %d items skew %g, had %d skew %g", ps[0].nx, ps[0].ny,
             b.n_items, b.skew, a.n_items, a.skew);
      EXPECT(fastest != 3 || !same, "%dx%d: %d items", ps[0].nx, ps[0].ny, b.n_items);
      EXPECT(rows > 0 && (fastest != 0 || rows == a.rows_per_wave), "%d rows", rows);
    }
    fivonagi_destroy(c);
  }
  return 0;
}

// A process with no pinned memory left: contexts are made, step (also when their
// instances have different targets) and are read as with it.
static int check_no_pinned_memory() {
  fake::st().no_pinned = true;
  for (int n : {1, 3, 50}) {
    fivonagi_ctx* c = context(std::vector<fivonagi_params>(n, grid(64, 40)));
    EXPECT(fivonagi_step(c, 5) == 0, "%s", fivonagi_last_error());
    EXPECT(fivonagi_enqueue(c, 2) == 0, "%s", fivonagi_last_error());
    EXPECT(fivonagi_step(c, 4) == 0, "%s", fivonagi_last_error());
    std::vector<float> q(64 * 40);
    for (int k = 0; k < n; ++k) {
      int64_t acc = 0;
      double T = 0.0;
      EXPECT(fivonagi_collect(c, k, q.data(), nullptr, nullptr, &T, nullptr, &acc, nullptr) == 0,
             "%s", fivonagi_last_error());
      EXPECT(acc == 11 && std::abs(T - 11 * 0.005) < 1e-12, "%lld steps, T %g", (long long)acc, T);
    }
    fivonagi_destroy(c);
  }
  return 0;
}

int main(int argc, char** argv) {
  const std::string name = argc > 1 ? argv[1] : "";
  int rc = 1;
  if (name == "collect_without_ring") rc = check_collect_without_ring();
  if (name == "download_error") rc = check_download_error();
  if (name == "download_device") rc = check_download_device();
  if (name == "enqueue_under_capture") rc = check_enqueue_under_capture();
  if (name == "autotune") rc = check_autotune();
  if (name == "no_pinned_memory") rc = check_no_pinned_memory();
  if (rc == 0 && !fake::st().blocks.empty()) {
    std::printf("%zu blocks not freed\n", fake::st().blocks.size());
    rc = 1;
  }
  if (rc == 0) std::printf("ok\n");
  return rc;
}
