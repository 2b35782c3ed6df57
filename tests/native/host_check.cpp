// Checks of the library's host code on the host, over the HIP runtime of
// fake_hip.hpp: what is asked of the runtime, in which order, and what the
// library does when a call fails.  One check per run, named by the argument.
#include "fake_hip.hpp"

#include <cstdlib>
#include <functional>

#include "../../include/csaw.h"

#define NEED(x)                                                                                 \
  do {                                                                                          \
    if (!(x)) {                                                                                 \
      std::printf("line %d: %s (last error: %s)\n", __LINE__, #x, csaw_last_error());           \
      std::exit(1);                                                                             \
    }                                                                                           \
  } while (0)

// V vertices of degree d each; ids are read by no host code and reserved only
static csaw_graph* regular_graph(int64_t V, int64_t d) {
  std::vector<int64_t> off(V + 1);
  for (int64_t v = 0; v <= V; ++v) off[v] = v * d;
  const size_t bytes = sizeof(int32_t) * (size_t)off[V] + 1;
  void* ids = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  NEED(ids != MAP_FAILED);
  csaw_graph* g = nullptr;
  NEED(csaw_graph_create(off.data(), 1, (const int32_t*)ids, nullptr, V, off[V], &g) == CSAW_OK);
  munmap(ids, bytes);
  return g;
}

static csaw_request request(int32_t samples, std::vector<int32_t> fanouts, int32_t bias, const int32_t* seeds) {
  csaw_request r;
  memset(&r, 0, sizeof(r));
  r.samples = samples;
  r.depth = (int32_t)fanouts.size();
  for (size_t h = 0; h < fanouts.size(); ++h) r.fanouts[h] = fanouts[h];
  r.bias = bias;
  r.dedup = 1;
  r.seeds = seeds;
  return r;
}

// Degree bias over hubs whose lists hold 2^32 entries and more together: a CDF's
// place among them does not fit the 32 bits that the batch build keeps of it, so
// such a graph is searched by the kernels that keep 64.
static void hub_positions() {
  const int64_t d = 4097;  // hubs: beyond 1,024 neighbours
  const int32_t n = 40000;
  std::vector<int32_t> seeds(n, 0);
  const csaw_request r = request(n, {25, 10}, CSAW_BIAS_DEGREE, seeds.data());
  auto batch_built = [&](int64_t V) {
    csaw_graph* g = regular_graph(V, d);
    csaw_plan* p = nullptr;
    NEED(csaw_plan_create(g, &r, 1, nullptr, &p) == CSAW_OK);
    fake().log.clear();
    NEED(csaw_plan_run(p, nullptr, 1) == CSAW_OK);
    NEED(fake().logged("k_expand_plain"));
    const bool built = fake().logged("k_expand_plainILi1ELb0ELi1ELb0ELb1E");
    csaw_plan_destroy(p);
    csaw_graph_destroy(g);
    return built;
  };
  const int64_t fit = ((int64_t(1) << 32) - 1) / d;
  NEED(batch_built(1000));
  NEED(batch_built(fit));
  NEED(!batch_built(fit + 1));
}

// A plan run but not waited for, destroyed while another device is current: the
// wait is for the plan's device, and the caller's device stays current.  What the
// plan held goes to the next plan of its device and to none of another's.
static void wait_on_own_device() {
  csaw_graph* g = regular_graph(100, 8);
  const std::vector<int32_t> seeds(50, 1);
  const csaw_request r = request(50, {4, 4}, CSAW_BIAS_UNIFORM, seeds.data());
  csaw_plan_opts o;
  memset(&o, 0, sizeof(o));
  o.mode = CSAW_MODE_BATCHED;
  csaw_plan *p = nullptr, *q = nullptr;
  NEED(csaw_plan_create(g, &r, 1, &o, &p) == CSAW_OK);
  NEED(csaw_plan_run(p, nullptr, 0) == CSAW_OK);
  fake().device = 1;
  fake().log.clear();
  csaw_plan_destroy(p);
  NEED(fake().logged("wait for device 0"));
  NEED(!fake().logged("wait for device 1"));
  NEED(fake().device == 1);
  const size_t before = fake().allocs.size();
  const uintptr_t handles = fake().handles;
  NEED(csaw_plan_create(g, &r, 1, &o, &p) == CSAW_OK);  // of device 1
  NEED(fake().allocs.size() == before + 1 && fake().handles > handles);
  fake().device = 0;
  const uintptr_t made = fake().handles;
  NEED(csaw_plan_create(g, &r, 1, &o, &q) == CSAW_OK);  // of device 0: what p left
  NEED(fake().allocs.size() == before + 1 && fake().handles == made);
  csaw_plan_destroy(p);
  csaw_plan_destroy(q);
  csaw_graph_destroy(g);
}

// A wait that fails leaves the plan's work where it may be: its memory and
// streams go to no other plan.
static void failed_wait() {
  csaw_graph* g = regular_graph(100, 8);
  const std::vector<int32_t> seeds(50, 1);
  const csaw_request r = request(50, {4, 4}, CSAW_BIAS_UNIFORM, seeds.data());
  csaw_plan_opts o;
  memset(&o, 0, sizeof(o));
  o.mode = CSAW_MODE_BATCHED;
  csaw_plan* p = nullptr;
  NEED(csaw_plan_create(g, &r, 1, &o, &p) == CSAW_OK);
  NEED(csaw_plan_run(p, nullptr, 0) == CSAW_OK);
  fake().fail_in["hipDeviceSynchronize"] = 1;
  fake().log.clear();
  csaw_plan_destroy(p);
  NEED(fake().logged("free on 0"));
  const size_t before = fake().allocs.size();
  const uintptr_t handles = fake().handles;
  NEED(csaw_plan_create(g, &r, 1, &o, &p) == CSAW_OK);
  NEED(fake().allocs.size() == before + 1 && fake().handles > handles);
  csaw_plan_destroy(p);
  csaw_graph_destroy(g);
}

// Calls that wait for what they launch and fail before they have: the plan is
// waited for when it goes, before its memory is anyone else's.
static void failed_copy_out() {
  csaw_graph* g = regular_graph(100, 8);
  const std::vector<int32_t> seeds(50, 1);
  auto waits = [&](const std::function<void()>& destroy) {
    fake().log.clear();
    destroy();
    return fake().logged("wait for device 0");
  };
  // csaw_sample: the run waits and brings the bounds home (the first copy), then
  // the edges are packed and copied (the second)
  csaw_params prm;
  memset(&prm, 0, sizeof(prm));
  prm.samples = 50;
  prm.frontier_size = 1;
  prm.neighbor_size = 4;
  prm.depth = 2;
  prm.dedup = 1;
  csaw_edges* e = nullptr;
  NEED(!waits([&] { NEED(csaw_sample(g, &prm, seeds.data(), &e, nullptr) == CSAW_OK); }));
  csaw_edges_free(e);
  NEED(waits([&] {
    fake().fail_in["hipMemcpyAsync"] = 2;
    NEED(csaw_sample(g, &prm, seeds.data(), &e, nullptr) != CSAW_OK && !e);
  }));
  NEED(waits([&] {
    fake().fail_in["hipStreamSynchronize"] = 2;
    NEED(csaw_sample(g, &prm, seeds.data(), &e, nullptr) != CSAW_OK && !e);
  }));
  // a plan's copy to device buffers and its digest
  const csaw_request r = request(50, {4, 4}, CSAW_BIAS_UNIFORM, seeds.data());
  std::vector<int32_t> out(3000);
  uint64_t digest = 0;
  for (int what = 0; what < 3; ++what) {
    csaw_plan* p = nullptr;
    NEED(csaw_plan_create(g, &r, 1, nullptr, &p) == CSAW_OK);
    NEED(csaw_plan_run(p, nullptr, 1) == CSAW_OK);
    NEED(csaw_plan_copy_device(p, 0, out.data(), nullptr, nullptr, nullptr, nullptr, 1) == CSAW_OK);
    NEED(csaw_plan_digest(p, 0, &digest) == CSAW_OK);
    if (what) fake().fail_in["hipStreamSynchronize"] = 1;
    if (what == 1) NEED(csaw_plan_copy_device(p, 0, out.data(), nullptr, nullptr, nullptr, nullptr, 1) != CSAW_OK);
    if (what == 2) NEED(csaw_plan_digest(p, 0, &digest) != CSAW_OK);
    NEED(waits([&] { csaw_plan_destroy(p); }) == (what != 0));
  }
  csaw_graph_destroy(g);
}

// A set of streams and events that could be made in part only: the next plan
// makes what it lacks.
static void partial_streams() {
  const std::vector<int32_t> seeds(50, 1);
  const csaw_request r = request(50, {4, 4}, CSAW_BIAS_UNIFORM, seeds.data());
  csaw_plan_opts o;
  memset(&o, 0, sizeof(o));
  o.mode = CSAW_MODE_BATCHED;
  const std::pair<const char*, int> made[] = {
      {"hipStreamCreateWithFlags", 4}, {"hipEventCreate", 2}, {"hipEventCreateWithFlags", 4}};
  for (const auto& m : made)
    for (int k = 1; k <= m.second; ++k) {
      csaw_graph* g = regular_graph(100, 8);
      csaw_plan* p = nullptr;
      fake().fail_in[m.first] = k;
      NEED(csaw_plan_create(g, &r, 1, &o, &p) != CSAW_OK);
      NEED(csaw_plan_create(g, &r, 1, &o, &p) == CSAW_OK);
      NEED(csaw_plan_run(p, nullptr, 1) == CSAW_OK);
      csaw_plan_destroy(p);
      csaw_graph_destroy(g);
    }
}

// No allocation of the library fails while a pool holds memory that would do.
static void pool_makes_room() {
  csaw_graph* g = regular_graph(2000, 8);
  csaw_graph* hubs = regular_graph(100, 2000);
  csaw_host_graph* hg = nullptr;
  {
    std::vector<int64_t> off(1001);
    for (int64_t v = 0; v <= 1000; ++v) off[v] = 8 * v;
    const std::vector<int32_t> ids(8000, 0);
    NEED(csaw_host_graph_from_csr(off.data(), ids.data(), 1000, 8000, &hg) == CSAW_OK);
  }
  const std::vector<int32_t> seeds(4000, 1);
  // a block of about 11 MB in the pool of g, and no other memory left than that
  auto fill = [&] {
    const csaw_request r = request(4000, {25, 8}, CSAW_BIAS_UNIFORM, seeds.data());
    csaw_plan* p = nullptr;
    fake().limit = SIZE_MAX;
    NEED(csaw_plan_create(g, &r, 1, nullptr, &p) == CSAW_OK);
    NEED(csaw_plan_run(p, nullptr, 1) == CSAW_OK);
    csaw_plan_destroy(p);
    fake().limit = fake().used;
  };
  std::vector<int32_t> out(4000 * 8), walks(4000 * 9);
  std::vector<int64_t> offs(4001);
  fill();
  csaw_mlp* m = nullptr;
  NEED(csaw_mlp_create(1, &m) == CSAW_OK);
  fill();
  std::vector<float> X(16, 0.f), Y(16);
  NEED(csaw_mlp_forward(m, X.data(), 1, Y.data()) == CSAW_OK);
  fill();
  NEED(csaw_random_walk(g, CSAW_BIAS_DEGREE, 1, 0, seeds.data(), 4000, 8, walks.data(), nullptr) == CSAW_OK);
  fill();
  NEED(csaw_mdrw(g, 1, 0, 2000, 2, 8, seeds.data(), out.data(), out.data(), offs.data(), nullptr) == CSAW_OK);
  fill();
  NEED(csaw_seeds(g, 1, 0, 100, out.data()) == CSAW_OK);
  fill();
  csaw_graph* other = regular_graph(10, 2);
  csaw_graph_destroy(other);
  for (int cache = 0; cache < 2; ++cache) {
    fill();
    const csaw_request r = request(10, {5}, CSAW_BIAS_DEGREE, seeds.data());
    csaw_plan_opts o;
    memset(&o, 0, sizeof(o));
    o.cdf_cache = cache;
    csaw_plan* p = nullptr;
    NEED(csaw_plan_create(hubs, &r, 1, &o, &p) == CSAW_OK);
    uint64_t digest = 0;
    NEED(csaw_plan_run(p, nullptr, 1) == CSAW_OK);
    fill();
    NEED(csaw_plan_digest(p, 0, &digest) == CSAW_OK);
    csaw_plan_destroy(p);
  }
  fill();
  const csaw_request r = request(10, {5}, CSAW_BIAS_UNIFORM, seeds.data());
  csaw_edges* e = nullptr;
  csaw_stream_stats st;
  NEED(csaw_stream_sample(hg, &r, 8 << 20, 2, &e, &st) == CSAW_OK);
  csaw_edges_free(e);
  // and one that is too large for the device all the same says so
  fill();
  const csaw_request big = request(4000, {64, 64}, CSAW_BIAS_UNIFORM, seeds.data());
  csaw_plan* p = nullptr;
  NEED(csaw_plan_create(g, &big, 1, nullptr, &p) == CSAW_ERR_OOM);
  // an allocation refused for another reason (a stream is being captured) leaves the
  // pools as they are
  fill();
  fake().limit = SIZE_MAX;
  fake().log.clear();
  fake().fail_in["hipMalloc as unsupported"] = 1;
  NEED(csaw_seeds(g, 1, 0, 100, out.data()) == CSAW_ERR_HIP);
  NEED(!fake().logged("free on"));
  csaw_mlp_destroy(m);
  csaw_host_graph_destroy(hg);
  csaw_graph_destroy(hubs);
  csaw_graph_destroy(g);
}

// The 32-bit copy of the hub CDFs is made for plans that read it (degree bias
// without the CDF cache), and by a later plan where the first one found no room.
static void narrow_hubs_when_read() {
  const int32_t n = 4000;  // 13 MB a plan
  const std::vector<int32_t> seeds(n, 0);
  const csaw_request r = request(n, {25, 10}, CSAW_BIAS_DEGREE, seeds.data());
  const int64_t entries = 5000 * 2000;  // 40 MB narrow
  csaw_graph* g = regular_graph(5000, 2000);
  auto asked = [&] {  // allocations of the copy's size
    int k = 0;
    for (size_t a : fake().allocs) k += a == sizeof(uint32_t) * entries;
    return k;
  };
  auto batch_built = [&](int cache) {
    csaw_plan_opts o;
    memset(&o, 0, sizeof(o));
    o.cdf_cache = cache;
    csaw_plan* p = nullptr;
    fake().allocs.clear();
    NEED(csaw_plan_create(g, &r, 1, &o, &p) == CSAW_OK);
    fake().log.clear();
    NEED(csaw_plan_run(p, nullptr, 1) == CSAW_OK);
    csaw_plan_destroy(p);
    return fake().logged("k_expand_plainILi1ELb0ELi1ELb0ELb1E");
  };
  NEED(!batch_built(1) && asked() == 1);  // the CDF cache itself
  NEED(!batch_built(1) && asked() == 0);
  fake().limit = fake().used + (20 << 20);  // the plan fits, the copy does not
  NEED(!batch_built(0));
  NEED(!batch_built(0));
  fake().limit = SIZE_MAX;
  NEED(batch_built(0) && asked() == 1);
  NEED(batch_built(0) && asked() == 0);
  csaw_graph_destroy(g);
  NEED(fake().used == 0);
}

// The autotuner tries what the plan's hops read and leaves the rest at its
// default.  Every run takes less time than the one before it here, so that the
// last of the values tried is kept.
static void autotune_reads() {
  csaw_graph* g = regular_graph(100, 8);
  const std::vector<int32_t> seeds(50, 1);
  const csaw_request r = request(50, {4, 4}, CSAW_BIAS_UNIFORM, seeds.data());
  auto tune = [&](int mode, int sched) {
    csaw_plan_opts o;
    memset(&o, 0, sizeof(o));
    o.mode = mode;
    o.sched = sched;
    o.variant = CSAW_VAR_THREAD;
    csaw_tuning t;
    double ms = 0;
    fake().ms = 1000.0f;
    fake().ms_step = 1.0f;
    NEED(csaw_autotune(g, &r, 1, &o, &t, &ms) == CSAW_OK);
    NEED(t.count_per_cu == 16 && t.group_min == 16);
    return t;
  };
  csaw_tuning t = tune(CSAW_MODE_BATCHED, CSAW_SCHED_HEURISTIC);  // hops expanded whole
  NEED(t.expand_per_cu == 8 && t.thread_per_cu == 4 && t.block_per_cu == 2 && t.chunk_min == 8);
  NEED(t.grid_override == 64 * 256);
  t = tune(CSAW_MODE_PLAIN, CSAW_SCHED_HEURISTIC);
  NEED(t.expand_per_cu == 16 && t.thread_per_cu == 4 && t.block_per_cu == 2 && t.chunk_min == 8);
  NEED(t.grid_override == 0);
  t = tune(CSAW_MODE_BATCHED, CSAW_SCHED_FORCED);  // binned
  NEED(t.expand_per_cu == 16 && t.thread_per_cu == 16 && t.block_per_cu == 16 && t.chunk_min == 256);
  NEED(t.grid_override == 0);
  csaw_graph_destroy(g);
}

int main(int argc, char** argv) {
  const std::map<std::string, std::function<void()>> checks = {
      {"hub_positions", hub_positions},
      {"wait_on_own_device", wait_on_own_device},
      {"failed_wait", failed_wait},
      {"failed_copy_out", failed_copy_out},
      {"partial_streams", partial_streams},
      {"pool_makes_room", pool_makes_room},
      {"narrow_hubs_when_read", narrow_hubs_when_read},
      {"autotune_reads", autotune_reads},
  };
  const auto it = checks.find(argc > 1 ? argv[1] : "");
  if (it == checks.end()) return 2;
  it->second();
  std::printf("ok\n");
  return 0;
}
