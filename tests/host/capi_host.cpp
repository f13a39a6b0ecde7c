// The C ABI's host code (bmx_capi.hip) over a simulated device: HIP calls and
// kernel launches are the stand-ins below, which run on the host and keep
// what the bookkeeping has to agree with -- the buffers the last executed
// reorder, row build and step left -- and fail where a case asks for it.
// Launches inside a stream capture run when the graph is launched.
// Usage: capi_host CASE; exit code 0 when every check holds.
#include "bmx_capi.hip"

#include <cstdlib>
#include <functional>
#include <tuple>

namespace sim {
bool capturing = false;
std::vector<std::function<void()>> graph;
std::string fail_at;  // the operation that returns an error
int fail_after = 0;   // ... after this many successful ones

// left by the launches executed so far
const void *chem = nullptr, *oid = nullptr, *rows = nullptr, *counts = nullptr;
long builds = 0;
double radius = 7e-5;  // the largest one the records hold
bool counts_zero = false;
int bad = 0;

hipError_t op(const char *name, std::function<void()> f) {
  if (fail_at == name && fail_after-- == 0) return hipErrorUnknown;
  if (capturing)
    graph.push_back(std::move(f));
  else
    f();
  return hipSuccess;
}
}  // namespace sim

#define CHECK(x)                                             \
  do {                                                       \
    if (!(x)) {                                              \
      std::printf("line %d: %s\n", __LINE__, #x);            \
      sim::bad++;                                            \
    }                                                        \
  } while (0)

// ---- the HIP runtime
extern "C" {
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "simulated"; }
hipError_t hipMalloc(void **p, size_t n) { *p = std::calloc(n, 1); return hipSuccess; }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = std::calloc(n, 1); return hipSuccess; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  return sim::op("copy", [=] { std::memmove(d, s, n); });
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)8; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)8; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)8; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  sim::capturing = true;
  sim::graph.clear();
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  sim::capturing = false;
  *g = (hipGraph_t)8;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  return sim::op("instantiate", [=] { *x = (hipGraphExec_t)8; });
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
  return sim::op("graph", [] { for (auto &f : sim::graph) f(); });
}
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
}

// ---- the launches (those that no case reaches are left out)
namespace bmx {
int32_t tile_count(int64_t n, int tile) { return (int32_t)std::max<int64_t>(1, (n + tile - 1) / tile); }
int64_t flat_entries(int64_t ncap, int, int32_t maxn) { return ncap * maxn + 128; }
int flat_tile(int, int64_t, double row) { return row > 4.0 ? 4 : 64; }
int64_t scan_scratch_elems(int64_t nb) { return nb / 2048 + 2; }
int32_t adj_blocks(int64_t n, int tile) { return tile_count(n, 4 * tile); }
int32_t adj_loss_blocks(int64_t n) { return tile_count(n, 256); }

hipError_t launch_fill_i32(int32_t *p, int64_t n, int32_t v, hipStream_t) {
  return sim::op("fill", [=] {
    std::fill(p, p + n, v);
    if (p == sim::counts) sim::counts_zero = v == 0;
  });
}
hipError_t launch_fill_u64(unsigned long long *p, int64_t n, unsigned long long v, hipStream_t) {
  return sim::op("fill", [=] { std::fill(p, p + n, v); });
}
hipError_t launch_aos_unpack(const uint8_t *, AosLayout, int64_t, const int32_t *, const BoxGeom *,
                             BoxGeom, StaticArrays st, DynArrays, unsigned long long *stats,
                             hipStream_t) {
  return sim::op("unpack", [=] {
    std::memcpy(stats, &sim::radius, 8);
    stats[1] = 0;  // no segments
    stats[2] = 1;
    sim::oid = st.oid;
  });
}
hipError_t launch_aos_refresh(const uint8_t *, AosLayout, int64_t, BoxGeom, StaticArrays, DynArrays,
                              uint32_t, unsigned long long *stats, hipStream_t) {
  return sim::op("refresh", [=] { std::memcpy(stats, &sim::radius, 8); });
}
hipError_t launch_mesh_bin(const double4 *, const int32_t *, int64_t, const MeshGeom &, int, int32_t *,
                           int32_t *, int32_t *, int32_t *, int32_t *, unsigned long long *, int,
                           int32_t *, unsigned long long *, hipStream_t) {
  return sim::op("mesh_bin", [] {});
}
hipError_t launch_mesh_to_particle(double *, int64_t, const MeshGeom &, const int32_t *,
                                   const int32_t *, const Topo *, double4 *, double4 *, const double *,
                                   const double *, int, int, const double[10], double, int,
                                   unsigned long long *maxima, int32_t *, hipStream_t) {
  return sim::op("mesh", [=] {
    std::memcpy(maxima, &sim::radius, 8);
    maxima[1] = 0;
  });
}
hipError_t launch_mesh_out(int32_t *err, const unsigned long long *maxima, int32_t *out_err,
                           unsigned long long *out_max, hipStream_t) {
  return sim::op("mesh_out", [=] {
    *out_err = *err;
    *err = 0;
    if (maxima) std::memcpy(out_max, maxima, 16);
  });
}
hipError_t launch_bin_count(const double4 *, const int32_t *, const BoxGeom *, BoxGeom, int, int64_t,
                            int32_t *, int32_t *, int32_t *count, hipStream_t, SkinCheck) {
  return sim::op("count", [=] {
    if (sim::counts == count) CHECK(sim::counts_zero);
    sim::counts = count;
    sim::counts_zero = false;
  });
}
hipError_t launch_scan(int32_t *, int32_t *, int64_t, int32_t *, hipStream_t, SkinCheck) {
  return sim::op("scan", [] { sim::counts_zero = true; });
}
hipError_t launch_bin_scatter(const int32_t *, const int32_t *, const int32_t *, const int32_t *,
                              int64_t, unsigned long long *, hipStream_t) {
  return sim::op("scatter", [] {});
}
hipError_t launch_sort_gather(const unsigned long long *, const int32_t *, int64_t, StaticArrays ss,
                              StaticArrays ds, DynArrays, DynArrays, const int32_t *, int, int,
                              int32_t *, hipStream_t, const double *from, double *to) {
  return sim::op("gather", [=] {
    CHECK(ss.oid == sim::oid);
    sim::oid = ds.oid;
    if (from) {
      CHECK(from == sim::chem);
      sim::chem = to;
    }
  });
}
hipError_t launch_build_nbr(const double4 *, const int32_t *, const int32_t *, const double4 *,
                            const BoxGeom *, BoxGeom, int, int, const int32_t *, const int32_t *,
                            int64_t, int, double, double, double, int32_t *, int32_t *, int64_t,
                            int32_t, int32_t *, int32_t *, FlatRows flat, int, hipStream_t) {
  return sim::op("build", [=] {
    sim::rows = flat.cidx;
    sim::builds++;
  });
}
hipError_t launch_force_sphere_flat(const double4 *, double4 *, const int32_t *, const uint8_t *,
                                    const int32_t *, const int32_t *, int64_t, int, int32_t,
                                    const int32_t *, const BoxGeom *, BoxGeom, int, ForceParams,
                                    double *, double *, int32_t *, LaunchShape, hipStream_t) {
  return sim::op("force", [] {});
}
hipError_t launch_skin_check(double *, int32_t, int32_t, double, int, unsigned long long *, int32_t *,
                             hipStream_t) {
  return sim::op("skin", [] {});
}
hipError_t launch_flags_out(const int32_t *, int32_t, int32_t *, unsigned long long *, int32_t *err,
                            int32_t *out, int add, hipStream_t) {
  return sim::op("flags", [=] {
    out[0] = add ? out[0] | *err : *err;
    *err = 0;
  });
}
hipError_t launch_fc_to_orig(const double *, const int32_t *, int64_t, double *, hipStream_t) {
  return sim::op("fc", [] {});
}
hipError_t launch_chem_unpack(const uint8_t *, AosLayout, int64_t, int, const int32_t *, double *state,
                              hipStream_t) {
  return sim::op("chem", [=] { sim::chem = state; });
}
hipError_t launch_to_orig4(const double4 *, const int32_t *, int64_t, double4 *, hipStream_t) {
  return sim::op("reorder", [] {});
}
hipError_t launch_from_orig4(const double4 *, const int32_t *, int64_t, double4 *, hipStream_t) {
  return sim::op("reorder", [] {});
}
hipError_t launch_adj_loss(const double4 *, const int32_t *, const double *, int64_t, BoxGeom,
                           double4 *, double *, hipStream_t) {
  return sim::op("loss", [] {});
}
hipError_t launch_adj_step(const double4 *, const int32_t *, const uint8_t *, const int32_t *,
                           const int32_t *, int, int32_t, const int32_t *, int64_t, BoxGeom,
                           ForceParams, const double4 *, double4 *, double *, double *, hipStream_t) {
  return sim::op("adj_step", [] {});
}
hipError_t launch_export_counts(const int32_t *, const int32_t *, int64_t n, int64_t *out, hipStream_t) {
  return sim::op("export", [=] { std::fill(out, out + n, 0); });
}
hipError_t launch_sum_partials(const double *, int64_t, int, double *, hipStream_t) {
  return sim::op("sum", [] {});
}
}  // namespace bmx

namespace {

constexpr int64_t kN = 300;
constexpr int32_t kEvery = 10;
const double kForce[9] = {6e-6, 1.0, 0, 0, 1.0, 0, 0, 0, 1.0};

bmx_ctx *bound(std::vector<uint8_t> &recs) {
  bmx_layout L{};
  L.n_real = 40;
  L.n_int = 40;
  L.pos_offset = 0;
  L.rdata_offset = 24;
  L.idata_offset = 24 + 8 * L.n_real;
  L.id_offset = L.cpu_offset = L.idata_offset;
  L.stride_bytes = L.idata_offset + 4 * L.n_int;
  recs.assign((size_t)(kN * L.stride_bytes), 0);
  bmx_ctx *c = nullptr;
  CHECK(bmx_ctx_create(&c, 0) == BMX_OK);
  CHECK(bmx_set_force_params(c, kForce) == BMX_OK);
  bmx_geometry g{};
  for (int d = 0; d < 3; d++) {
    g.prob_hi[d] = 1.0e-3;
    g.periodic[d] = 1;
    g.n_cell[d] = 4;
  }
  CHECK(bmx_set_geometry(c, &g) == BMX_OK);
  bmx_neighbor_params p{};
  p.mode = BMX_NBR_VERLET;
  p.rebuild_every = kEvery;
  p.skin = 2e-5;
  CHECK(bmx_set_neighbor_params(c, &p) == BMX_OK);
  CHECK(bmx_bind_particles_aos(c, recs.data(), kN, &L, BMX_AOS_HOST) == BMX_OK);
  return c;
}

// The host's idea of the current buffers against what was executed.
void check_buffers(bmx_ctx *c) {
  CHECK(c->oid[c->cs].p == sim::oid);
  if (c->have_chem) CHECK(c->d_chemst[c->cc].p == sim::chem);
  CHECK(c->rebuilds_total == sim::builds);
  if (c->have_list) CHECK(c->d_cidx.p == sim::rows);
}

// What a step changes on the host.
auto bookkeeping(const bmx_ctx *c) {
  return std::make_tuple(c->step, c->last_build, c->rebuilds_total, c->row_nblk, c->cs,
                         c->cd, c->cc, c->have_list, c->count_clear, c->wrote_step,
                         c->fc_orig, c->fc_cs);
}

const double kXpar[3] = {0, 0, 0};

void graph_with_chem() {
  std::vector<uint8_t> recs;
  bmx_ctx *c = bound(recs);
  CHECK(bmx_exchange(c, kXpar, 1.0) == BMX_OK);
  check_buffers(c);
  // one rebuild in the graph, captured and then replayed; then two
  for (int32_t steps : {kEvery, kEvery, 2 * kEvery, 3}) {
    CHECK(bmx_evolve_graph(c, 1e-3, steps) == BMX_OK);
    check_buffers(c);
  }
  CHECK(bmx_exchange(c, kXpar, 1.0) == BMX_OK);
  check_buffers(c);
  CHECK(bmx_evolve(c, 1e-3, 25) == BMX_OK);
  check_buffers(c);
  bmx_ctx_destroy(c);
}

// A capture that fails (in a launch, or when it is instantiated) and a graph
// that does not launch leave the context where it was.
void failed_capture() {
  for (const char *where : {"force", "build", "instantiate", "graph"}) {
    std::vector<uint8_t> recs;
    sim::builds = 0;
    bmx_ctx *c = bound(recs);
    for (int32_t steps : {0, 4, kEvery}) {  // before the first row build, in
      if (steps) CHECK(bmx_evolve(c, 1e-3, steps) == BMX_OK);  // a period, at its end
      if (steps == 4) CHECK(bmx_exchange(c, kXpar, 1.0) == BMX_OK);
      const auto m = bookkeeping(c);
      sim::fail_at = where;
      sim::fail_after = sim::fail_at == "force" ? 12 : 0;
      CHECK(bmx_evolve_graph(c, 1e-3, 2 * kEvery) == BMX_ERR_HIP);
      sim::fail_at.clear();
      CHECK(bookkeeping(c) == m);
      check_buffers(c);
      CHECK(bmx_evolve_graph(c, 1e-3, 3) == BMX_OK);
      check_buffers(c);
    }
    bmx_ctx_destroy(c);
  }
}

// A row build that fails inside a list period leaves no list: the particles
// are in another order than the rows.
void failed_build() {
  std::vector<uint8_t> recs;
  bmx_ctx *c = bound(recs);
  CHECK(bmx_evolve(c, 1e-3, 5) == BMX_OK);
  sim::fail_at = "build";
  sim::fail_after = 0;
  CHECK(bmx_exchange(c, kXpar, 1.0) == BMX_ERR_HIP);
  sim::fail_at.clear();
  CHECK(!c->have_list);
  CHECK(bmx_evolve(c, 1e-3, 1) == BMX_OK);
  check_buffers(c);
  CHECK(c->have_list && sim::builds == 2);
  bmx_ctx_destroy(c);
}

// An adjoint call whose reverse pass fails: its recomputed rows went to the
// history, so the context must not take its own rows as current.
void adjoint_error() {
  for (const char *where : {"adj_step", "force", "copy", "sum"}) {
    std::vector<uint8_t> recs;
    sim::builds = 0;
    bmx_ctx *c = bound(recs);
    CHECK(bmx_evolve(c, 1e-3, 5) == BMX_OK);
    const std::vector<double> target(3 * kN, 0.0);
    std::vector<double> grad_r(kN);
    double loss = 0.0, grad[3];
    sim::fail_at = where;
    // past the forward pass: 40 steps of forces; 2 copies in, the error word
    sim::fail_after = sim::fail_at == "force" ? 45 : sim::fail_at == "copy" ? 4 : 0;
    CHECK(bmx_adjoint(c, 1e-3, 40, 2 * kEvery, target.data(), &loss, grad, grad_r.data(),
                      nullptr) == BMX_ERR_HIP);
    sim::fail_at.clear();
    CHECK(sim::rows != c->d_cidx.p);  // the reverse pass had built rows
    check_buffers(c);
    int64_t total, offsets[kN + 1];
    CHECK(bmx_get_neighbors(c, offsets, nullptr, 0, &total) == BMX_ERR_STATE);
    bmx_ctx_destroy(c);
  }
}

// The tile follows the reach, as a new bind with that reach would choose it,
// and the arrays laid out by tiles with it.
void check_tile(bmx_ctx *c, int tile) {
  CHECK(c->flat_tile == tile && c->flat_tile == flat_tile(0, c->n, row_estimate(c)));
  const size_t tiles = (size_t)tile_count(c->ncap, tile);
  CHECK(c->vstride == (int32_t)tiles && c->d_vpart.n >= tiles * c->vmax_slots);
  CHECK(c->d_wtot.n >= tiles && c->d_redo.n >= tiles && c->d_bstats.n >= 2 * tiles);
  CHECK(bmx_evolve(c, 1e-3, 3) == BMX_OK);
  check_buffers(c);
  CHECK(bmx_evolve_graph(c, 1e-3, 3) == BMX_OK);
  check_buffers(c);
}
void tile_follows_reach() {
  std::vector<uint8_t> recs;
  bmx_ctx *c = bound(recs);
  check_tile(c, 64);
  double fpar[9];
  std::memcpy(fpar, kForce, sizeof fpar);
  for (double band : {1.5e-4, 6e-6}) {  // the adhesion band W_A
    fpar[0] = band;
    CHECK(bmx_set_force_params(c, fpar) == BMX_OK);
    check_tile(c, band > 1e-4 ? 4 : 64);
  }
  for (double radius : {1.3e-4, 7e-5}) {
    sim::radius = radius;
    CHECK(bmx_refresh_from_aos(c, nullptr, kFieldSizes) == BMX_OK);
    check_tile(c, radius > 1e-4 ? 4 : 64);
  }
  const double chempar[10] = {};
  const std::vector<double> x(3 * 6 * 6 * 6, 1.0);
  for (double radius : {1.3e-4, 7e-5}) {
    sim::radius = radius;
    CHECK(bmx_calc_txfr_particle(c, chempar, x.data(), x.data(), 1.0, 1, 0, 0, 0) == BMX_OK);
    check_tile(c, radius > 1e-4 ? 4 : 64);
  }
  bmx_ctx_destroy(c);
}

}  // namespace

int main(int argc, char **argv) {
  std::setvbuf(stdout, nullptr, _IONBF, 0);
  const std::string name = argc > 1 ? argv[1] : "";
  if (name == "graph_with_chem") graph_with_chem();
  else if (name == "failed_capture") failed_capture();
  else if (name == "failed_build") failed_build();
  else if (name == "tile_follows_reach") tile_follows_reach();
  else if (name == "adjoint_error") adjoint_error();
  else return 2;
  return sim::bad ? 1 : 0;
}
