// Sampling plans: the host side of Sampler() (non-stream/main.cu:196-308),
// re-designed around reusable device buffers.
//
// A plan holds every buffer a run needs in one block (sized at creation by the
// per-request upper bound S * F_0 * ... * F_h per hop, taken from the graph's
// pool), so csaw_plan_run allocates nothing and its launch sequence can be
// captured in a hipGraph.
// PLAIN mode executes one request after another (one unit per request, a
// wave per frontier entry, synchronising after each request like a call of
// the reference's Sampler()); BATCHED mode puts all requests into one unit:
// one launch sequence per hop over the concatenated frontiers: a kernel per bias
// kind in frontier order, or degree binning and a kernel variant per chunk
// (plan_bins_hop).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <numeric>
#include <vector>

#include "graph.hpp"
#include "plan.hpp"

namespace csaw {

void EventTimer::begin(int which, hipStream_t s) {
  if (!enabled) return;
  if (used >= pool.size()) {
    Rec r;
    r.kind = which;
    if (hipEventCreate(&r.a) != hipSuccess || hipEventCreate(&r.b) != hipSuccess) return;
    pool.push_back(r);
  }
  pool[used].kind = which;
  (void)hipEventRecord(pool[used].a, s);
}

void EventTimer::end(int which, hipStream_t s) {
  if (!enabled || used >= pool.size()) return;
  (void)which;
  (void)hipEventRecord(pool[used].b, s);
  ++used;
}

void EventTimer::collect() {
  for (size_t i = 0; i < used; ++i) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, pool[i].a, pool[i].b) == hipSuccess) {
      total_ms[pool[i].kind] += ms;
      launches[pool[i].kind] += 1;
    }
  }
  used = 0;
}

EventTimer::~EventTimer() {
  for (auto& r : pool) {
    (void)hipEventDestroy(r.a);
    (void)hipEventDestroy(r.b);
  }
}

// csaw_sample packs results of at most this many words (64 MB) for one copy; the
// time of larger ones is the copy's own
constexpr int64_t kStageWords = 16 << 20;

static int64_t ub_mul(int64_t a, int64_t b) {
  if (a == 0 || b == 0) return 0;
  if (a > (int64_t)1 << 40 || b > (int64_t)1 << 40 || a > ((int64_t)1 << 62) / b) return (int64_t)1 << 62;
  return a * b;
}

}  // namespace csaw

using namespace csaw;

static int validate_request(const csaw_graph* g, const csaw_request& r) {
  if (r.samples < 0 || r.depth < 0 || r.depth > CSAW_MAX_HOPS) return CSAW_ERR_INVALID_ARG;
  if (r.bias < CSAW_BIAS_UNIFORM || r.bias > CSAW_BIAS_USER) return CSAW_ERR_INVALID_ARG;
  if (r.dedup < 0 || r.dedup > 2) return CSAW_ERR_INVALID_ARG;
  if (r.bias == CSAW_BIAS_WEIGHT && !g->w) return CSAW_ERR_INVALID_ARG;
  if (r.request_id >= (1u << 20)) return CSAW_ERR_INVALID_ARG;
  for (int h = 0; h < r.depth; ++h)
    if (r.fanouts[h] < 0 || r.fanouts[h] > CSAW_MAX_FANOUT) return CSAW_ERR_INVALID_ARG;
  if (r.samples > 0 && !r.seeds) return CSAW_ERR_INVALID_ARG;
  for (int32_t s = 0; s < r.samples; ++s)
    if (r.seeds[s] < 0 || r.seeds[s] >= g->V) return CSAW_ERR_INVALID_ARG;
  return CSAW_OK;
}

namespace csaw {

int PlanStreams::create(bool with_side) {
  // (each by itself: an earlier call may have failed half-way)
  if (!main) CSAW_HIP(hipStreamCreateWithFlags(&main, hipStreamNonBlocking));
  if (!begin) CSAW_HIP(hipEventCreate(&begin));
  if (!end) CSAW_HIP(hipEventCreate(&end));
  if (with_side) {
    if (!fork) CSAW_HIP(hipEventCreateWithFlags(&fork, hipEventDisableTiming));
    for (int i = 0; i < kSide; ++i) {
      if (!side[i]) CSAW_HIP(hipStreamCreateWithFlags(&side[i], hipStreamNonBlocking));
      if (!join[i]) CSAW_HIP(hipEventCreateWithFlags(&join[i], hipEventDisableTiming));
    }
  }
  return CSAW_OK;
}

void PlanStreams::destroy() {
  for (hipEvent_t e : {begin, end, fork, join[0], join[1], join[2]})
    if (e) (void)hipEventDestroy(e);
  for (hipStream_t x : {main, side[0], side[1], side[2]})
    if (x) (void)hipStreamDestroy(x);
  *this = PlanStreams();
}

int Workspace::take(size_t bytes, Block* b) {
  int device = 0;
  CSAW_HIP(hipGetDevice(&device));
  {
    std::lock_guard<std::mutex> lock(mu);
    size_t best = blocks.size();
    for (size_t i = 0; i < blocks.size(); ++i)
      if (blocks[i].device == device && blocks[i].bytes >= bytes && blocks[i].bytes <= 4 * bytes + (1u << 20) &&
          (best == blocks.size() || blocks[i].bytes < blocks[best].bytes))
        best = i;
    if (best < blocks.size()) {
      *b = blocks[best];
      held -= b->bytes;
      blocks.erase(blocks.begin() + best);
      return CSAW_OK;
    }
  }
  b->bytes = (bytes + 65535) & ~(size_t)65535;
  b->device = device;
  CSAW_HIP(device_malloc(&b->p, b->bytes));
  return CSAW_OK;
}

void Workspace::give(Block b) {
  if (!b.p) return;
  {
    std::lock_guard<std::mutex> lock(mu);
    if (!closed && b.bytes <= kBlockBytes && held + b.bytes <= kHeldBytes) {
      blocks.push_back(b);
      held += b.bytes;
      return;
    }
  }
  (void)hipFree(b.p);
}

int Workspace::take_streams(bool with_side, PlanStreams* s) {
  int device = 0;
  CSAW_HIP(hipGetDevice(&device));
  {
    std::lock_guard<std::mutex> lock(mu);
    for (size_t i = streams.size(); i-- > 0;)
      if (streams[i].device == device) {
        *s = streams[i];
        streams.erase(streams.begin() + i);
        break;
      }
  }
  s->device = device;
  return s->create(with_side);
}

void Workspace::give_streams(PlanStreams s) {
  {
    std::lock_guard<std::mutex> lock(mu);
    if (!closed && streams.size() < kHeldStreams && s.main) {
      streams.push_back(s);
      return;
    }
  }
  s.destroy();
}

void Workspace::drain(std::vector<Block>* out) {
  std::lock_guard<std::mutex> lock(mu);
  out->insert(out->end(), blocks.begin(), blocks.end());
  blocks.clear();
  held = 0;
}

void Workspace::close() {
  std::vector<Block> out;
  std::vector<PlanStreams> sets;
  drain(&out);
  {
    std::lock_guard<std::mutex> lock(mu);
    closed = true;
    sets.swap(streams);
  }
  for (Block& b : out) (void)hipFree(b.p);
  for (PlanStreams& s : sets) s.destroy();
}

// The pools that exist, for device_malloc.  (Never destroyed: a graph may go
// after this file's statics.)
namespace {
struct Pools {
  std::mutex mu;
  std::vector<Workspace*> all;
};
Pools& pools() {
  static Pools* p = new Pools;
  return *p;
}
}  // namespace

Workspace::Workspace() {
  Pools& P = pools();
  std::lock_guard<std::mutex> lock(P.mu);
  P.all.push_back(this);
}

Workspace::~Workspace() {
  {
    Pools& P = pools();
    std::lock_guard<std::mutex> lock(P.mu);
    P.all.erase(std::find(P.all.begin(), P.all.end(), this));
  }
  close();
}

hipError_t device_malloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipSuccess) return e;
  (void)hipGetLastError();
  if (e != hipErrorOutOfMemory) return e;  // (a stream being captured, for one: frees are refused then too)
  std::vector<Workspace::Block> out;
  {
    Pools& P = pools();
    std::lock_guard<std::mutex> lock(P.mu);
    for (Workspace* w : P.all) w->drain(&out);
  }
  if (out.empty()) return e;
  for (Workspace::Block& b : out) (void)hipFree(b.p);
  e = hipMalloc(p, bytes);
  if (e != hipSuccess) (void)hipGetLastError();
  return e;
}

}  // namespace csaw

// Waits for everything on `device`, which need not be the current one.
static hipError_t wait_for_device(int device) {
  int cur = device;
  hipError_t e = hipGetDevice(&cur);
  if (e == hipSuccess && cur != device) e = hipSetDevice(device);
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (cur != device) (void)hipSetDevice(cur);
  return e;
}

static void plan_free(csaw_plan* p) {
  if (!p) return;
  // work that a call has not waited for may still use the workspace, on a stream
  // of the caller's; where that wait fails nothing goes back to the pool
  const bool idle = p->unwaited == 0 || wait_for_device(p->slab.device) == hipSuccess;
  if (!idle) (void)hipGetLastError();
  if (p->gexec) (void)hipGraphExecDestroy(p->gexec);
  if (p->work && idle) {
    p->work->give(p->slab);
    p->work->give_streams(p->st);
  } else {
    (void)hipFree(p->slab.p);
    p->st.destroy();
  }
  delete p;
}

static int build_unit(csaw_plan* p, Unit& u) {
  // requests sorted by depth descending: the active set at hop h is a prefix
  std::stable_sort(u.reqs.begin(), u.reqs.end(),
                   [&](int a, int b) { return p->reqs[a].depth > p->reqs[b].depth; });
  u.G = 0;
  u.depth_max = 0;
  u.kinds[0] = u.kinds[1] = u.kinds[2] = false;
  u.remap = false;
  std::vector<ReqDev> rd;
  for (int ri : u.reqs) {
    const csaw_request& r = p->reqs[ri];
    ReqDev d;
    memset(&d, 0, sizeof(d));
    for (int h = 0; h < CSAW_MAX_HOPS; ++h) d.fanout[h] = h < r.depth ? r.fanouts[h] : 0;
    d.depth = r.depth;
    d.bias = r.bias;
    d.dedup = r.dedup == 2 ? 2 : (r.dedup ? 1 : 0);
    d.samples = r.samples;
    d.key_lo = (uint32_t)r.seed;
    d.key_hi = (uint32_t)(r.seed >> 32);
    d.request_id = r.request_id;
    d.slot = (uint32_t)ri;
    d.gbase = u.G;
    u.gbase.push_back(u.G);
    rd.push_back(d);
    u.G += r.samples;
    u.depth_max = std::max(u.depth_max, r.depth);
    if (r.depth > 0 && r.samples > 0) u.kinds[bias_kind(r.bias)] = true;
    if (r.dedup == 2) u.remap = true;
  }
  if (u.G > 0x7fffffffLL) return CSAW_ERR_CAPACITY;
  // per hop: first inactive global sample, edge capacity, max frontier entries
  u.gb.assign(u.depth_max, 0);
  u.cap.assign(u.depth_max, 0);
  u.nmax.assign(u.depth_max, 0);
  std::vector<int64_t> ub(u.reqs.size());
  for (size_t i = 0; i < u.reqs.size(); ++i) ub[i] = p->reqs[u.reqs[i]].samples;
  for (int h = 0; h < u.depth_max; ++h) {
    int64_t gb = 0, cap = 0, nm = 0;
    for (size_t i = 0; i < u.reqs.size(); ++i) {
      const csaw_request& r = p->reqs[u.reqs[i]];
      if (r.depth > h) {
        gb = u.gbase[i] + r.samples;
        nm += ub[i];
        ub[i] = ub_mul(ub[i], r.fanouts[h]);
        cap += ub[i];
      }
    }
    u.gb[h] = (int32_t)gb;
    u.cap[h] = cap;
    u.nmax[h] = nm;
    if (cap > ((int64_t)1 << 34) || nm > ((int64_t)1 << 32) - 1) {
      set_last_error("plan exceeds the per-hop capacity (2^32 frontier entries)");
      return CSAW_ERR_CAPACITY;
    }
  }
  u.d_eo.assign(u.depth_max, nullptr);
  u.d_src.assign(u.depth_max, nullptr);
  u.d_dst.assign(u.depth_max, nullptr);
  u.d_smp.assign(u.depth_max, nullptr);
  u.rd = std::move(rd);
  return CSAW_OK;
}

// Carves a plan's arrays from one block: a first pass with base null sizes it.
struct Carver {
  char* base = nullptr;
  size_t at = 0;
  template <typename T>
  void part(T** p, int64_t count) {
    if (base) *p = reinterpret_cast<T*>(base + at);
    at += (std::max<int64_t>(count, 1) * sizeof(T) + 255) & ~(size_t)255;
  }
};

struct PlanSizes {
  int64_t nmax = 1, depth = 1, bin_max = 0, staging = 0;
  bool several = false, mlp = false;
};

// What the host fills in comes first (`filled` bytes).
static void plan_layout(csaw_plan* p, const PlanSizes& z, Carver& c, size_t* filled) {
  const size_t state = kCtrBytes + kBoundsBytes * p->reqs.size();
  c.part(&p->counters, state / sizeof(uint32_t));
  if (c.base) p->bounds = reinterpret_cast<int64_t*>(reinterpret_cast<char*>(p->counters) + kCtrBytes);
  c.part(&p->bytes_acc, kNumKernKinds);
  for (auto& u : p->units) {
    c.part(&u.d_req, (int64_t)u.rd.size());
    c.part(&u.d_fv0, u.G);
  }
  *filled = c.at;
  for (auto& u : p->units) {
    c.part(&u.d_gs2req, u.G);
    c.part(&u.d_fs0, u.G);
    c.part(&u.d_fo0, u.G + 1);
  }
  for (auto& u : p->units)
    for (int h = 0; h < u.depth_max; ++h) {
      c.part(&u.d_eo[h], u.G + 1);
      c.part(&u.d_src[h], u.cap[h]);
      c.part(&u.d_dst[h], u.cap[h]);
      c.part(&u.d_smp[h], u.cap[h]);
    }
  const int64_t nblk = (z.nmax + kBlockEntries - 1) / kBlockEntries;
  c.part(&p->local_excl, z.nmax);
  c.part(&p->blk_excl, nblk);
  c.part(&p->blk_scan, std::min<int64_t>(nblk, 1024));
  c.part(&p->grp_excl, (nblk + 1023) / 1024);
  c.part(&p->totals, z.depth);
  if (z.several) c.part(&p->kind_mask, (z.nmax + kWave - 1) / kWave);
  if (z.bin_max > 0) {
    const int64_t bblk = (z.bin_max + kBlockEntries - 1) / kBlockEntries;
    const int64_t waves = (int64_t)p->L.num_cu * p->L.expand_per_cu * 4;
    p->chunk_cap = (uint32_t)std::min<int64_t>(bblk * kChunksPerBlock + waves, 0xFFFFFFF0LL);
    p->queue_cap = p->chunk_cap;
    c.part(&p->order, bblk * kBlockEntries);
    c.part(&p->chunks, p->chunk_cap);
    c.part(&p->queues, (int64_t)kNumQueues * p->queue_cap);
    c.part(&p->chosen, p->chunk_cap);
    if (p->opts.log_chunks) c.part(&p->log, p->chunk_cap);
  }
  if (z.mlp) c.part(&p->d_mlp, kMlpParams);
  if (z.staging > 0) c.part(&p->staging, z.staging);
}

namespace csaw {
// The first frontier besides its vertices: sample g at position g, of the last
// request whose first sample is not above g (and has samples).
__global__ void k_first_frontier(const ReqDev* __restrict__ R, int n_req, int64_t G, int32_t* __restrict__ gs2req,
                                 int32_t* __restrict__ fs, int64_t* __restrict__ fo) {
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g <= G; g += (int64_t)gridDim.x * blockDim.x) {
    fo[g] = g;
    if (g == G) continue;
    int lo = 0, hi = n_req;  // last request with gbase <= g
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (R[mid].gbase <= g) lo = mid; else hi = mid;
    }
    gs2req[g] = lo;
    fs[g] = (int32_t)g;
  }
}
}  // namespace csaw

// Requests and seeds, one copy in the block's own layout; the rest of the first
// frontier is written on the device.
static int upload_inputs(csaw_plan* p, const csaw_request* reqs, size_t filled) {
  std::vector<char> host(filled, 0);  // (zeroes: the counters, the bounds, the byte counts)
  auto at = [&](const void* dev) {
    return host.data() + (reinterpret_cast<const char*>(dev) - static_cast<char*>(p->slab.p));
  };
  for (auto& u : p->units) {
    if (!u.rd.empty()) memcpy(at(u.d_req), u.rd.data(), sizeof(ReqDev) * u.rd.size());
    for (size_t i = 0; i < u.reqs.size(); ++i) {
      const csaw_request& r = reqs[u.reqs[i]];
      if (r.samples > 0) memcpy(at(u.d_fv0) + sizeof(int32_t) * u.gbase[i], r.seeds, sizeof(int32_t) * r.samples);
    }
  }
  CSAW_HIP(hipMemcpy(p->slab.p, host.data(), filled, hipMemcpyHostToDevice));
  for (auto& u : p->units) {
    const int grid = (int)std::min<int64_t>(u.G / 256 + 1, (int64_t)p->L.num_cu * 8);
    k_first_frontier<<<grid, 256, 0, p->stream>>>(u.d_req, (int)u.rd.size(), u.G, u.d_gs2req, u.d_fs0, u.d_fo0);
    CSAW_LAUNCH_CHECK();
  }
  return CSAW_OK;
}

static HopDev make_hop(csaw_plan* p, Unit& u, int h) {
  HopDev H;
  H.fv = h == 0 ? u.d_fv0 : u.d_dst[h - 1];
  H.fs = h == 0 ? u.d_fs0 : u.d_smp[h - 1];
  H.fo = h == 0 ? u.d_fo0 : u.d_eo[h - 1];
  H.n_ptr = H.fo + u.gb[h];
  H.hop = h;
  H.gb = u.gb[h];
  H.local_excl = p->local_excl;
  H.blk_excl = p->blk_excl;
  H.blk_scan = p->blk_scan;
  H.grp_excl = p->grp_excl;
  H.order = p->order;
  H.chunks = p->chunks;
  H.n_chunks = p->counters + kCtrChunks;
  H.chunk_cap = p->chunk_cap;
  H.src = u.d_src[h];
  H.dst = u.d_dst[h];
  H.smp = u.d_smp[h];
  H.eo = u.d_eo[h];
  H.flags = p->counters + kCtrFlags;
  H.bytes = p->opts.timing ? p->bytes_acc : nullptr;
  H.expand_waves = p->L.num_cu * p->L.expand_per_cu * 4;  // 4 waves per 256-lane workgroup
  H.chunk_min = p->L.chunk_min;
  H.group_min = p->L.group_min;
  H.only_kind = 0;
  H.kind_mask = p->kind_mask;
  H.bounds = p->bounds;
  H.n_req = (int32_t)u.reqs.size();
  return H;
}

// Whether a batched hop of at most nmax entries is binned into chunks with a
// kernel variant each, or expanded in frontier order by one whole-hop kernel per
// bias kind.  Frontier order writes each wave's edges next to one another; a
// block's chunks are spread over the chip and fill the same output lines from
// several XCDs, which cost more than the variants gained wherever no entry has a
// CDF to build: 256 mixed requests over RMAT-22 take 22.7 ms binned, 17.3 ms in
// frontier order, 8 of 64 to 1,024 seeds 0.89 and 0.41.  Binning stays for integer
// biases whose CDFs neither a 32-bit cache holds nor a group's wave builds (the
// workgroup variants share those builds), and for what asks for chunks: forced and random variants, chunk logs.
static bool plan_bins_hop(const csaw_plan* p, const Unit& u, int64_t nmax) {
  if (p->opts.mode != CSAW_MODE_BATCHED) return false;
  if (p->opts.log_chunks || (p->opts.sched != CSAW_SCHED_HEURISTIC && p->opts.sched != CSAW_SCHED_MLP)) return true;
  if (nmax <= kSmallHopEntries) return false;
  if (!u.kinds[kInt]) return false;
  if (p->opts.cdf_cache) return p->g->int_cdf[0] || p->g->int_cdf[1];
  if (!p->g->build32 || u.remap) return true;
  for (int ri : u.reqs)
    if (p->reqs[ri].bias == CSAW_BIAS_USER) return true;
  return false;
}

static int run_unit(csaw_plan* p, Unit& u, hipStream_t st, TimingHook* th) {
  const GraphDev G = p->g->view(p->opts.cdf_cache != 0);
  const csaw_graph_view hv = p->g->hook_view();
  LaunchCfg L = p->L;
  L.stream = st;
  for (int h = 0; h < u.depth_max; ++h) {
    HopDev H = make_hop(p, u, h);
    const bool bin = u.bin[h];
    if (bin) {
      if (th) th->begin(kKernFill, st);
      CSAW_TRY(launch_fill(L, p->counters, 0u, kCtrCount - 1));  // keeps the flags word
      if (th) th->end(kKernFill, st);
    }
    if (th) th->begin(kKernCount, st);
    CSAW_TRY(launch_count(L, G, u.d_req, u.d_gs2req, H, bin, u.nmax[h]));
    if (th) th->end(kKernCount, st);
    if (th) th->begin(kKernScan, st);
    CSAW_TRY(launch_scans(L, H, u.d_req, p->totals + h, u.nmax[h]));
    if (th) th->end(kKernScan, st);
    if (bin) {
      ChooseArgs A;
      A.sched = p->opts.sched;
      A.variant = p->opts.variant;
      A.explore_key = p->opts.explore_key;
      A.qlen = p->counters + kCtrQlen;
      A.queues = p->queues;
      A.queue_cap = p->queue_cap;
      A.chosen = p->chosen;
      A.int_cache = p->opts.cdf_cache != 0;
      A.in_place = 0;
      A.mlp.w = p->d_mlp;
      A.mlp_w = p->d_mlp;
      if (th) th->begin(kKernChoose, st);
      CSAW_TRY(launch_choose(L, A, H, (int64_t)p->chunk_cap));
      if (th) th->end(kKernChoose, st);
      ExpandArgs E;
      E.queues = p->queues;
      E.queue_cap = p->queue_cap;
      E.qlen = p->counters + kCtrQlen;
      E.qhead = p->counters + kCtrQhead;
      E.log = p->opts.log_chunks ? p->log : nullptr;
      E.int_cache = p->opts.cdf_cache != 0;
      E.remap = u.remap ? 1 : 0;
      if (p->fan) {
        // the hop's expansion kernels (one per variant queue) run side by
        // side on four streams, so one kernel's last chunks overlap the
        // others' work; all join before the next hop (with timing on, each
        // kernel's events are recorded on the stream it runs on, so the
        // times are those of this concurrent schedule)
        hipStream_t ss[1 + PlanStreams::kSide] = {st};
        CSAW_HIP(hipEventRecord(p->st.fork, st));
        for (int i = 0; i < PlanStreams::kSide; ++i) {
          CSAW_HIP(hipStreamWaitEvent(p->st.side[i], p->st.fork, 0));
          ss[1 + i] = p->st.side[i];
        }
        CSAW_TRY(launch_expand_chunks(L, G, hv, u.d_req, u.d_gs2req, H, E, u.kinds, th, ss, 1 + PlanStreams::kSide));
        for (int i = 0; i < PlanStreams::kSide; ++i) {
          CSAW_HIP(hipEventRecord(p->st.join[i], p->st.side[i]));
          CSAW_HIP(hipStreamWaitEvent(st, p->st.join[i], 0));
        }
      } else {
        CSAW_TRY(launch_expand_chunks(L, G, hv, u.d_req, u.d_gs2req, H, E, u.kinds, th));
      }
      if (p->opts.log_chunks) {
        // keep this hop's chunks and log for the host
        p->hop_logs.emplace_back();
        p->pending_log_hops.push_back(h);
      }
    } else {
      // one launch per bias kind present (one for a plain unit, whose single
      // request has one kind); with several kinds each launch expands only
      // its own kind's entries, side by side on the plan's streams so that
      // one kind's last waves overlap the others' work
      int nk = 0;
      for (int k = 0; k < 3; ++k) nk += u.kinds[k] ? 1 : 0;
      const bool fan = nk > 1 && p->fan;
      if (fan) {
        CSAW_HIP(hipEventRecord(p->st.fork, st));
        for (int i = 0; i + 1 < nk; ++i) CSAW_HIP(hipStreamWaitEvent(p->st.side[i], p->st.fork, 0));
      }
      int next = 0;
      // integer and FP32 kinds first: their chains are the long ones
      for (int kind : {(int)kInt, (int)kF32, (int)kUniform}) {
        if (!u.kinds[kind]) continue;
        // sub-wave group size from the largest fanout of the kind's requests
        int fmax = 0;
        bool remap = false, user = false;
        for (int ri : u.reqs) {
          const csaw_request& r = p->reqs[ri];
          if (r.depth > h && bias_kind(r.bias) == kind) {
            user |= r.bias == CSAW_BIAS_USER;
            fmax = std::max(fmax, r.fanouts[h]);
            remap |= r.dedup == 2;
          }
        }
        const int gs = group_size_for(fmax, L.group_min);
        H.only_kind = nk > 1 ? 1 + kind : 0;
        LaunchCfg K = L;
        if (fan && next > 0) K.stream = p->st.side[next - 1];
        if (th) th->begin(kKernPlain, K.stream);
        CSAW_TRY(launch_expand_plain(K, kind, G, hv, u.d_req, u.d_gs2req, H, u.nmax[h], gs, remap, user));
        if (th) th->end(kKernPlain, K.stream);
        if (fan && next > 0) {
          CSAW_HIP(hipEventRecord(p->st.join[next - 1], K.stream));
          CSAW_HIP(hipStreamWaitEvent(st, p->st.join[next - 1], 0));
        }
        ++next;
      }
    }
    if (bin && p->opts.log_chunks) {
      // chunk log must be read before the next hop overwrites chunk storage
      CSAW_HIP(hipStreamSynchronize(st));
      uint32_t nch = 0;
      CSAW_HIP(hipMemcpy(&nch, p->counters + kCtrChunks, sizeof(uint32_t), hipMemcpyDeviceToHost));
      nch = std::min(nch, p->chunk_cap);
      HopLog& hl = p->hop_logs.back();
      hl.hop = h;
      hl.chunks.resize(nch);
      hl.log.resize(nch);
      if (nch) {
        CSAW_HIP(hipMemcpy(hl.chunks.data(), p->chunks, sizeof(Chunk) * nch, hipMemcpyDeviceToHost));
        CSAW_HIP(hipMemcpy(hl.log.data(), p->log, sizeof(ChunkLog) * nch, hipMemcpyDeviceToHost));
      }
    }
  }
  return CSAW_OK;
}

// stage: leave room for csaw_sample's packed result
static int plan_create(csaw_graph* g, const csaw_request* reqs, int32_t n_req, const csaw_plan_opts* opts, bool stage,
                       csaw_plan** out) {
  if (!g || !out || n_req < 0 || (n_req > 0 && !reqs)) return CSAW_ERR_INVALID_ARG;
  *out = nullptr;
  csaw_plan_opts o;
  memset(&o, 0, sizeof(o));
  if (opts) o = *opts;
  if (o.mode != CSAW_MODE_PLAIN && o.mode != CSAW_MODE_BATCHED) return CSAW_ERR_INVALID_ARG;
  if (o.sched < CSAW_SCHED_HEURISTIC || o.sched > CSAW_SCHED_RANDOM) return CSAW_ERR_INVALID_ARG;
  if (o.sched == CSAW_SCHED_FORCED && (o.variant < 0 || o.variant >= CSAW_NUM_VARIANTS)) return CSAW_ERR_INVALID_ARG;
  CSAW_TRY(validate_tuning(o.tuning));
  for (int i = 0; i < n_req; ++i) {
    int st = validate_request(g, reqs[i]);
    if (st != CSAW_OK) {
      set_last_error("invalid request " + std::to_string(i));
      return st;
    }
  }
  csaw_plan* p = new csaw_plan();
  p->g = g;
  p->work = g->work;
  p->opts = o;
  p->L.num_cu = g->num_cu;
  if (o.tuning) apply_tuning(p->L, o.tuning);
  // Whole-hop kernels: a plain plan's takes the tuned shape (8 by default: 4 to
  // 16 within 2% from 3,000 to 1,048,576 seeds, 32 up to 8% slower for degree bias).
  // A batched plan's tuned expand_per_cu is that of its side-by-side variant
  // kernels; its kinds' kernels skip one another's batches, and 32 evens out what
  // is left (32 requests of 64 to 4,096 seeds: 906 us at 32, 1,022 at 8).
  if (o.mode == CSAW_MODE_BATCHED) p->L.frontier_per_cu = 32;
  else if (o.tuning && o.tuning->expand_per_cu > 0) p->L.frontier_per_cu = o.tuning->expand_per_cu;
  auto body = [&]() -> int {
    for (int i = 0; i < n_req; ++i) {
      std::lock_guard<std::mutex> lock(g->prepare);
      CSAW_TRY(graph_prepare_bias(g, reqs[i].bias));
      if (o.cdf_cache) {
        CSAW_TRY(graph_prepare_index(g, reqs[i].bias));
        CSAW_TRY(graph_prepare_vertex_records(g, reqs[i].bias));
      } else if (reqs[i].bias == CSAW_BIAS_DEGREE) {
        CSAW_TRY(graph_prepare_build32(g));
      }
      p->reqs.push_back(reqs[i]);
      p->reqs.back().seeds = nullptr;
    }
    if (o.mode == CSAW_MODE_BATCHED) {
      p->units.emplace_back();
      for (int i = 0; i < n_req; ++i) p->units.back().reqs.push_back(i);
    } else {
      for (int i = 0; i < n_req; ++i) {
        p->units.emplace_back();
        p->units.back().reqs.push_back(i);
      }
    }
    PlanSizes z;
    for (auto& u : p->units) {
      CSAW_TRY(build_unit(p, u));
      for (int64_t v : u.nmax) {
        z.nmax = std::max(z.nmax, v);
        u.bin.push_back(plan_bins_hop(p, u, v));
        if (u.bin.back()) z.bin_max = std::max(z.bin_max, v);
      }
      z.several |= u.kinds[0] + u.kinds[1] + u.kinds[2] > 1;
      z.depth = std::max<int64_t>(z.depth, u.depth_max);
    }
    p->req_unit.assign(n_req, {-1, -1});
    for (size_t ui = 0; ui < p->units.size(); ++ui)
      for (size_t k = 0; k < p->units[ui].reqs.size(); ++k) p->req_unit[p->units[ui].reqs[k]] = {(int)ui, (int)k};
    z.mlp = o.mode == CSAW_MODE_BATCHED && o.sched == CSAW_SCHED_MLP;
    if (z.mlp && !o.mlp) {
      set_last_error("CSAW_SCHED_MLP needs a trained csaw_mlp");
      return CSAW_ERR_INVALID_ARG;
    }
    if (stage) {
      // the one request's offsets and edges, if they are worth packing
      int64_t words = 2 * (int64_t)reqs[0].depth * ((int64_t)reqs[0].samples + 1);
      for (int64_t c : p->units[0].cap) words += 3 * c;
      if (words <= kStageWords) z.staging = words;
    }
    size_t filled = 0;
    Carver size;
    plan_layout(p, z, size, &filled);
    CSAW_TRY(p->work->take(size.at, &p->slab));
    Carver c;
    c.base = static_cast<char*>(p->slab.p);
    plan_layout(p, z, c, &filled);
    p->h_state.assign((kCtrBytes + kBoundsBytes * (size_t)n_req) / sizeof(uint32_t), 0u);
    InFlight upload(p->unwaited);
    if (z.mlp) CSAW_TRY(mlp_upload_bf16(o.mlp, p->d_mlp));
    CSAW_TRY(p->work->take_streams(o.mode == CSAW_MODE_BATCHED && !o.serial_expand, &p->st));
    p->stream = p->st.main;
    p->fan = o.mode == CSAW_MODE_BATCHED && !o.serial_expand;
    CSAW_TRY(upload_inputs(p, reqs, filled));
    // (csaw_sample runs on the same stream and waits there)
    if (!stage) CSAW_HIP(hipStreamSynchronize(p->stream));
    upload.waited();
    p->timer.enabled = o.timing != 0;
    return CSAW_OK;
  };
  int st = body();
  if (st != CSAW_OK) {
    plan_free(p);
    return st;
  }
  *out = p;
  return CSAW_OK;
}

extern "C" int csaw_plan_create(csaw_graph* g, const csaw_request* reqs, int32_t n_req, const csaw_plan_opts* opts,
                                csaw_plan** out) {
  return plan_create(g, reqs, n_req, opts, false, out);
}

extern "C" int csaw_plan_run(csaw_plan* p, void* stream, int sync) {
  if (!p) return CSAW_ERR_INVALID_ARG;
  hipStream_t st = stream ? (hipStream_t)stream : p->stream;
  p->hop_logs.clear();
  p->pending_log_hops.clear();
  p->bounds_known = false;
  InFlight run(p->unwaited);
  TimingHook* th = p->timer.enabled ? &p->timer : nullptr;
  const bool wait = sync || th;
  if (wait) CSAW_HIP(hipEventRecord(p->st.begin, st));
  if (th) {
    LaunchCfg L = p->L;
    L.stream = st;
    CSAW_TRY(launch_fill(L, (uint32_t*)p->bytes_acc, 0u, 2 * kNumKernKinds));
  }
  const bool use_graph = p->opts.use_graph && p->opts.mode == CSAW_MODE_BATCHED && !th && !p->opts.log_chunks;
  if (use_graph) {
    if (!p->gexec || p->graph_stream != st) {
      if (p->gexec) {
        CSAW_HIP(hipGraphExecDestroy(p->gexec));
        p->gexec = nullptr;
      }
      hipGraph_t graph;
      CSAW_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
      int rs = CSAW_OK;
      for (auto& u : p->units) {
        rs = run_unit(p, u, st, nullptr);
        if (rs != CSAW_OK) break;
      }
      hipError_t ce = hipStreamEndCapture(st, &graph);
      if (rs != CSAW_OK) return rs;
      CSAW_HIP(ce);
      CSAW_HIP(hipGraphInstantiate(&p->gexec, graph, nullptr, nullptr, 0));
      CSAW_HIP(hipGraphDestroy(graph));
      p->graph_stream = st;
    }
    CSAW_HIP(hipGraphLaunch(p->gexec, st));
  } else {
    for (size_t i = 0; i < p->units.size(); ++i) {
      CSAW_TRY(run_unit(p, p->units[i], st, th));
      // (the last one's wait is the run's own, below)
      if (p->opts.mode == CSAW_MODE_PLAIN && !(wait && i + 1 == p->units.size())) CSAW_HIP(hipStreamSynchronize(st));
    }
  }
  if (wait) {
    CSAW_HIP(hipEventRecord(p->st.end, st));
    CSAW_HIP(hipMemcpyAsync(p->h_state.data(), p->counters, sizeof(uint32_t) * p->h_state.size(), hipMemcpyDeviceToHost,
                            st));
    CSAW_HIP(hipStreamSynchronize(st));
    run.waited();
    float ms = 0.f;
    CSAW_HIP(hipEventElapsedTime(&ms, p->st.begin, p->st.end));
    p->last_ms = ms;
    if (th) {
      p->timer.collect();
      unsigned long long b[kNumKernKinds];
      CSAW_HIP(hipMemcpy(b, p->bytes_acc, sizeof(b), hipMemcpyDeviceToHost));
      for (int k = 0; k < kNumKernKinds; ++k) p->timer.total_bytes[k] += (double)b[k];
    }
    if (p->h_state[kCtrFlags] & 1u) {
      set_last_error("chunk descriptor capacity exceeded");
      return CSAW_ERR_CAPACITY;
    }
    p->bounds_known = true;
  }
  p->runs += 1;
  return CSAW_OK;
}

// Per-request hop boundaries: hop h edges of request r are
// [eo_h[gbase], eo_h[gbase + S]) of its unit's hop-h arrays.  A synchronised
// run has brought them to the host; after any other they are read here.
static int request_bounds(const csaw_plan* p, int32_t req, std::vector<int64_t>& lo, std::vector<int64_t>& hi) {
  if (req < 0 || req >= (int32_t)p->reqs.size()) return CSAW_ERR_INVALID_ARG;
  const int32_t depth = p->reqs[req].depth;
  int64_t read[2 * CSAW_MAX_HOPS];
  const char* known = reinterpret_cast<const char*>(p->h_state.data()) + kCtrBytes + kBoundsBytes * (size_t)req;
  if (p->bounds_known) memcpy(read, known, kBoundsBytes);
  else CSAW_HIP(hipMemcpy(read, p->bounds + (size_t)req * 2 * CSAW_MAX_HOPS, kBoundsBytes, hipMemcpyDeviceToHost));
  lo.resize(depth);
  hi.resize(depth);
  for (int h = 0; h < depth; ++h) {
    lo[h] = read[2 * h];
    hi[h] = read[2 * h + 1];
  }
  return CSAW_OK;
}

extern "C" int csaw_plan_request_info(const csaw_plan* p, int32_t req, int64_t* n_edges) {
  if (!p || !n_edges) return CSAW_ERR_INVALID_ARG;
  std::vector<int64_t> lo, hi;
  CSAW_TRY(request_bounds(p, req, lo, hi));
  int64_t n = 0;
  for (size_t h = 0; h < lo.size(); ++h) n += hi[h] - lo[h];
  *n_edges = n;
  return CSAW_OK;
}

extern "C" int csaw_plan_copy(const csaw_plan* p, int32_t req, int32_t* src, int32_t* dst, int32_t* sample,
                              int64_t* hop_offsets) {
  if (!p) return CSAW_ERR_INVALID_ARG;
  std::vector<int64_t> lo, hi;
  CSAW_TRY(request_bounds(p, req, lo, hi));
  const auto [ui, k] = p->req_unit[req];
  const Unit& u = p->units[ui];
  const csaw_request& r = p->reqs[req];
  int64_t at = 0;
  for (int h = 0; h < r.depth; ++h) {
    const int64_t n = hi[h] - lo[h];
    if (n > 0) {
      if (src) CSAW_HIP(hipMemcpy(src + at, u.d_src[h] + lo[h], sizeof(int32_t) * n, hipMemcpyDeviceToHost));
      if (dst) CSAW_HIP(hipMemcpy(dst + at, u.d_dst[h] + lo[h], sizeof(int32_t) * n, hipMemcpyDeviceToHost));
      if (sample) {
        CSAW_HIP(hipMemcpy(sample + at, u.d_smp[h] + lo[h], sizeof(int32_t) * n, hipMemcpyDeviceToHost));
        for (int64_t i = 0; i < n; ++i) sample[at + i] -= (int32_t)u.gbase[k];
      }
    }
    if (hop_offsets) {
      std::vector<int64_t> eo(r.samples + 1);
      CSAW_HIP(hipMemcpy(eo.data(), u.d_eo[h] + u.gbase[k], sizeof(int64_t) * (r.samples + 1), hipMemcpyDeviceToHost));
      for (int32_t s = 0; s <= r.samples; ++s) hop_offsets[(int64_t)h * (r.samples + 1) + s] = at + eo[s] - lo[h];
    }
    at += n;
  }
  return CSAW_OK;
}

// csaw_plan_copy into device buffers, on the device (for callers that keep
// the edge lists on the GPU, e.g. as framework tensors).
static int copy_edges_device(const csaw_plan* p, int32_t req, const std::vector<int64_t>& lo,
                             const std::vector<int64_t>& hi, int32_t* src, int32_t* dst, int32_t* sample,
                             int64_t* hop_offsets, hipStream_t st) {
  const auto [ui, k] = p->req_unit[req];
  const Unit& u = p->units[ui];
  const csaw_request& r = p->reqs[req];
  CopyArgs A;
  memset(&A, 0, sizeof(A));
  int64_t at = 0;
  for (int h = 0; h < r.depth; ++h) {
    A.col[0][h] = u.d_src[h];
    A.col[1][h] = u.d_dst[h];
    A.col[2][h] = u.d_smp[h];
    A.eo[h] = u.d_eo[h] + u.gbase[k];
    A.lo[h] = lo[h];
    A.n[h] = hi[h] - lo[h];
    A.at[h] = at;
    at += A.n[h];
  }
  A.out[0] = src;
  A.out[1] = dst;
  A.out[2] = sample;
  A.hop_offsets = hop_offsets;
  A.rows = (int64_t)r.samples + 1;
  A.depth = r.depth;
  A.sub = (int32_t)u.gbase[k];
  return launch_copy_edges(st, A);
}

extern "C" int csaw_plan_copy_device(const csaw_plan* p, int32_t req, int32_t* src, int32_t* dst, int32_t* sample,
                                     int64_t* hop_offsets, void* stream, int sync) {
  if (!p) return CSAW_ERR_INVALID_ARG;
  std::vector<int64_t> lo, hi;
  CSAW_TRY(request_bounds(p, req, lo, hi));
  hipStream_t st = stream ? (hipStream_t)stream : p->stream;
  InFlight copy(p->unwaited);
  CSAW_TRY(copy_edges_device(p, req, lo, hi, src, dst, sample, hop_offsets, st));
  if (sync) {
    CSAW_HIP(hipStreamSynchronize(st));
    copy.waited();
  }
  return CSAW_OK;
}

extern "C" int csaw_plan_digest(const csaw_plan* p, int32_t req, uint64_t* digest) {
  if (!p || !digest) return CSAW_ERR_INVALID_ARG;
  std::vector<int64_t> lo, hi;
  CSAW_TRY(request_bounds(p, req, lo, hi));
  const auto [ui, k] = p->req_unit[req];
  const Unit& u = p->units[ui];
  unsigned long long* d;
  InFlight sum(p->unwaited);
  CSAW_HIP(device_malloc(&d, sizeof(unsigned long long)));
  CSAW_HIP(hipMemsetAsync(d, 0, sizeof(unsigned long long), p->stream));
  int64_t at = 0;
  int st = CSAW_OK;
  for (size_t h = 0; h < lo.size() && st == CSAW_OK; ++h) {
    st = launch_digest(p->stream, p->g->num_cu, u.d_src[h], u.d_dst[h], u.d_smp[h], lo[h], hi[h], at, u.gbase[k], d);
    at += hi[h] - lo[h];
  }
  unsigned long long v = 0;
  if (st == CSAW_OK) {
    CSAW_HIP(hipMemcpyAsync(&v, d, sizeof(v), hipMemcpyDeviceToHost, p->stream));
    CSAW_HIP(hipStreamSynchronize(p->stream));
    sum.waited();
  }
  (void)hipFree(d);
  *digest = (uint64_t)v ^ ((uint64_t)at * 0x100000001b3ull);
  return st;
}

extern "C" int csaw_plan_stats(const csaw_plan* p, csaw_stats* s) {
  if (!p || !s) return CSAW_ERR_INVALID_ARG;
  memset(s, 0, sizeof(*s));
  int64_t edges = 0;
  for (int32_t r = 0; r < (int32_t)p->reqs.size(); ++r) {
    int64_t n = 0;
    CSAW_TRY(csaw_plan_request_info(p, r, &n));
    edges += n;
  }
  s->edges = edges;
  s->kernel_ms = p->last_ms;
  if (p->opts.mode == CSAW_MODE_BATCHED && p->chosen) {
    // variant mix of the last hop (chunk storage is per hop)
    uint32_t nch = 0;
    CSAW_HIP(hipMemcpy(&nch, p->counters + kCtrChunks, sizeof(uint32_t), hipMemcpyDeviceToHost));
    (void)nch;
  }
  return CSAW_OK;
}

extern "C" int csaw_plan_kernel_times(const csaw_plan* p, char* names, size_t names_len, double* avg_ms,
                                      int64_t* launches, double* avg_bytes, int32_t max_kinds, int32_t* n_kinds) {
  if (!p) return CSAW_ERR_INVALID_ARG;
  int32_t n = 0;
  size_t pos = 0;
  for (int k = 0; k < kNumKernKinds; ++k) {
    if (p->timer.launches[k] == 0) continue;
    if (n < max_kinds) {
      if (avg_ms) avg_ms[n] = p->timer.total_ms[k] / (double)p->timer.launches[k];
      if (launches) launches[n] = p->timer.launches[k];
      if (avg_bytes) avg_bytes[n] = p->timer.total_bytes[k] / (double)p->timer.launches[k];
      if (names) {
        size_t l = strlen(kKernNames[k]) + 1;
        if (pos + l <= names_len) {
          memcpy(names + pos, kKernNames[k], l);
          pos += l;
        }
      }
    }
    ++n;
  }
  if (n_kinds) *n_kinds = n;
  return CSAW_OK;
}

extern "C" int csaw_plan_reset_times(csaw_plan* p) {
  if (!p) return CSAW_ERR_INVALID_ARG;
  for (int k = 0; k < kNumKernKinds; ++k) {
    p->timer.total_ms[k] = 0;
    p->timer.launches[k] = 0;
    p->timer.total_bytes[k] = 0;
  }
  return CSAW_OK;
}

extern "C" int csaw_plan_destroy(csaw_plan* p) {
  plan_free(p);
  return CSAW_OK;
}

// ------------------------------------------------------------ csaw_sample
// One block of offsets (hop_off), then src, dst and sample columns of n edges.
struct csaw_edges {
  int32_t depth = 0, samples = 0;
  int64_t n = 0, n_off = 0;
  std::unique_ptr<int64_t[]> block;
  void alloc(int64_t edges, int64_t offsets) {
    n = edges;
    n_off = offsets;
    block.reset(new int64_t[n_off + (3 * n + 1) / 2 + 1]);
  }
  int64_t* hop_off() const { return block.get(); }
  int32_t* col(int c) const { return reinterpret_cast<int32_t*>(block.get() + n_off) + c * n; }
};

// The request's offsets and columns packed on the device as csaw_edges holds
// them, then one copy to the host (a copy per hop and column, each its own round
// trip, took 0.12 ms of a small call).
static int copy_staged(const csaw_plan* p, const std::vector<int64_t>& lo, const std::vector<int64_t>& hi, csaw_edges* e) {
  int64_t* off = reinterpret_cast<int64_t*>(p->staging);
  int32_t* col = reinterpret_cast<int32_t*>(off + e->n_off);
  InFlight copy(p->unwaited);
  CSAW_TRY(copy_edges_device(p, 0, lo, hi, col, col + e->n, col + 2 * e->n, off, p->stream));
  CSAW_HIP(hipMemcpyAsync(e->block.get(), p->staging, sizeof(int64_t) * e->n_off + 3 * sizeof(int32_t) * e->n,
                          hipMemcpyDeviceToHost, p->stream));
  CSAW_HIP(hipStreamSynchronize(p->stream));
  copy.waited();
  return CSAW_OK;
}

extern "C" int csaw_sample(csaw_graph* g, const csaw_params* prm, const int32_t* seeds, csaw_edges** out,
                           csaw_stats* stats) {
  if (!g || !prm || !out) return CSAW_ERR_INVALID_ARG;
  *out = nullptr;
  if (prm->frontier_size > 1) {
    // FrontierSize > 1 runs the multi-dimensional random walk, as Sampler()
    // dispatches check_layer (main.cu:285-287); the result is one layer.
    if (prm->samples < 0 || prm->depth < 0 || (prm->samples > 0 && !seeds)) return CSAW_ERR_INVALID_ARG;
    const size_t cap = std::max<size_t>((size_t)prm->samples * prm->depth, 1);
    std::vector<int32_t> src(cap), dst(cap);
    std::vector<int64_t> off((size_t)prm->samples + 1);
    csaw_stats st;
    CSAW_TRY(csaw_mdrw(g, prm->seed, prm->request_id, prm->samples, prm->frontier_size, prm->depth, seeds, src.data(),
                       dst.data(), off.data(), &st));
    csaw_edges* e = new csaw_edges();
    e->depth = 1;
    e->samples = prm->samples;
    e->alloc(off[prm->samples], prm->samples + 1);
    memcpy(e->hop_off(), off.data(), sizeof(int64_t) * off.size());
    if (e->n > 0) {
      memcpy(e->col(0), src.data(), sizeof(int32_t) * e->n);
      memcpy(e->col(1), dst.data(), sizeof(int32_t) * e->n);
    }
    for (int32_t s = 0; s < prm->samples; ++s) std::fill(e->col(2) + off[s], e->col(2) + off[s + 1], s);
    if (stats) *stats = st;
    *out = e;
    return CSAW_OK;
  }
  if (prm->frontier_size != 1) return CSAW_ERR_INVALID_ARG;
  if (prm->depth < 0 || prm->depth > CSAW_MAX_HOPS) return CSAW_ERR_INVALID_ARG;
  csaw_request r;
  memset(&r, 0, sizeof(r));
  r.samples = prm->samples;
  r.depth = prm->depth;
  for (int h = 0; h < prm->depth; ++h) r.fanouts[h] = prm->fanouts ? prm->fanouts[h] : prm->neighbor_size;
  r.bias = prm->bias;
  r.dedup = prm->dedup;
  r.seed = prm->seed;
  r.request_id = prm->request_id;
  r.seeds = seeds;
  csaw_plan_opts o;
  memset(&o, 0, sizeof(o));
  const bool binned = prm->sched != CSAW_SCHED_HEURISTIC || prm->variant != 0;
  o.mode = binned ? CSAW_MODE_BATCHED : CSAW_MODE_PLAIN;
  o.sched = prm->sched == CSAW_SCHED_MLP ? CSAW_SCHED_HEURISTIC : prm->sched;
  o.variant = prm->variant;
  csaw_tuning t;
  memset(&t, 0, sizeof(t));
  if (prm->n_blocks > 0) {
    t.grid_override = prm->n_blocks;
    o.tuning = &t;
  }
  csaw_plan* p = nullptr;
  CSAW_TRY(plan_create(g, &r, 1, &o, true, &p));
  int st = csaw_plan_run(p, nullptr, 1);
  csaw_edges* e = nullptr;
  if (st == CSAW_OK) {
    e = new csaw_edges();
    e->depth = r.depth;
    e->samples = r.samples;
    std::vector<int64_t> lo, hi;
    st = request_bounds(p, 0, lo, hi);
    if (st == CSAW_OK) {
      int64_t n = 0;
      for (int32_t h = 0; h < r.depth; ++h) n += hi[h] - lo[h];
      e->alloc(n, (int64_t)r.depth * ((int64_t)r.samples + 1));
      st = p->staging ? copy_staged(p, lo, hi, e)
                      : csaw_plan_copy(p, 0, e->col(0), e->col(1), e->col(2), e->hop_off());
      if (st == CSAW_OK && stats) {
        memset(stats, 0, sizeof(*stats));
        stats->edges = n;
        stats->kernel_ms = p->last_ms;
      }
    }
  }
  csaw_plan_destroy(p);
  if (st != CSAW_OK) {
    delete e;
    return st;
  }
  *out = e;
  return CSAW_OK;
}

extern "C" int csaw_edges_info(const csaw_edges* e, int64_t* n_edges, int32_t* depth, int32_t* samples) {
  if (!e) return CSAW_ERR_INVALID_ARG;
  if (n_edges) *n_edges = e->n;
  if (depth) *depth = e->depth;
  if (samples) *samples = e->samples;
  return CSAW_OK;
}

extern "C" int csaw_edges_copy(const csaw_edges* e, int32_t* src, int32_t* dst, int32_t* sample, int64_t* hop_offsets) {
  if (!e) return CSAW_ERR_INVALID_ARG;
  int32_t* out[3] = {src, dst, sample};
  for (int c = 0; c < 3; ++c)
    if (out[c] && e->n > 0) memcpy(out[c], e->col(c), sizeof(int32_t) * e->n);
  if (hop_offsets && e->n_off > 0) memcpy(hop_offsets, e->hop_off(), sizeof(int64_t) * e->n_off);
  return CSAW_OK;
}

extern "C" void csaw_edges_free(csaw_edges* e) { delete e; }

extern "C" int csaw_edges_from_host(int32_t depth, int32_t samples, int64_t n, const int32_t* src, const int32_t* dst,
                                    const int32_t* smp, const int64_t* hop_off, csaw_edges** out) {
  if (!out || n < 0 || depth < 0 || samples < 0 || (n > 0 && (!src || !dst || !smp))) return CSAW_ERR_INVALID_ARG;
  csaw_edges* e = new csaw_edges();
  e->depth = depth;
  e->samples = samples;
  e->alloc(n, hop_off ? (int64_t)depth * (samples + 1) : 0);
  if (n > 0) {
    memcpy(e->col(0), src, sizeof(int32_t) * n);
    memcpy(e->col(1), dst, sizeof(int32_t) * n);
    memcpy(e->col(2), smp, sizeof(int32_t) * n);
  }
  if (e->n_off > 0) memcpy(e->hop_off(), hop_off, sizeof(int64_t) * e->n_off);
  *out = e;
  return CSAW_OK;
}

// C4 request mix (all draws from Philox with the mix key, domain kDomMix).
extern "C" int64_t csaw_request_mix(uint64_t mix_key, int32_t n, int32_t lo, int32_t hi, csaw_request* out) {
  if (n < 0 || lo < 1 || hi < lo || (n > 0 && !out)) return -1;
  int64_t total = 0;
  const double l0 = std::log2((double)lo), l1 = std::log2((double)hi);
  for (int32_t i = 0; i < n; ++i) {
    const U4 o = philox4x32_10((uint32_t)i, 0u, 0u, kDomMix << 28, (uint32_t)mix_key, (uint32_t)(mix_key >> 32));
    const double u = (double)(o.x >> 8) * (1.0 / 16777216.0);
    int64_t s = (int64_t)std::floor(std::exp2(l0 + u * (l1 - l0)));
    s = std::min<int64_t>(std::max<int64_t>(s, lo), hi);
    csaw_request& r = out[i];
    memset(&r, 0, sizeof(r));
    r.samples = (int32_t)s;
    if (o.y & 1u) {
      r.depth = 3;
      r.fanouts[0] = 15;
      r.fanouts[1] = 10;
      r.fanouts[2] = 5;
    } else {
      r.depth = 2;
      r.fanouts[0] = 25;
      r.fanouts[1] = 10;
    }
    r.bias = (int32_t)(o.z % 3u);  // uniform, degree, weight
    r.dedup = 1;
    r.seed = 42;
    r.request_id = (uint32_t)i;
    r.seeds = nullptr;
    total += s;
  }
  return total;
}
