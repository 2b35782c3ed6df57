// Host-side plan state (see plan.cpp).
#pragma once
#include <atomic>
#include <utility>
#include <vector>

#include "graph.hpp"
#include "sample_kernels.hpp"

namespace csaw {

// layout of the small counter block reset at every hop
enum : int {
  kCtrChunks = 0,
  kCtrQlen = 1,
  kCtrQhead = kCtrQlen + kNumQueues,
  kCtrFlags = kCtrQhead + kNumQueues,
  kCtrCount = kCtrFlags + 1
};
static_assert(kCtrCount <= 64, "the bounds table starts 64 words after the counters");
constexpr size_t kCtrBytes = 64 * sizeof(uint32_t);  // counters, padded
constexpr size_t kBoundsBytes = 2 * CSAW_MAX_HOPS * sizeof(int64_t);  // one request's edge bounds

struct EventTimer : TimingHook {
  struct Rec {
    int kind;
    hipEvent_t a, b;
  };
  bool enabled = false;
  std::vector<Rec> pool;
  size_t used = 0;
  double total_ms[kNumKernKinds] = {};
  int64_t launches[kNumKernKinds] = {};
  double total_bytes[kNumKernKinds] = {};
  void begin(int which, hipStream_t s) override;
  void end(int which, hipStream_t s) override;
  void collect();
  ~EventTimer() override;
};

struct Unit {
  std::vector<int> reqs;        // plan request indices, sorted by depth (desc)
  std::vector<int64_t> gbase;   // global sample base per unit request
  int64_t G = 0;
  int depth_max = 0;
  bool kinds[3] = {false, false, false};
  bool remap = false;           // some request uses the region-remap mode
  std::vector<int32_t> gb;      // per hop: first inactive global sample
  std::vector<int64_t> cap;     // per hop: edge capacity
  std::vector<int64_t> nmax;    // per hop: frontier entries upper bound
  std::vector<char> bin;        // per hop: binned into chunks (plan_bins_hop)
  std::vector<ReqDev> rd;       // the requests as the device sees them
  ReqDev* d_req = nullptr;
  int32_t* d_gs2req = nullptr;
  int32_t* d_fv0 = nullptr;
  int32_t* d_fs0 = nullptr;
  int64_t* d_fo0 = nullptr;
  std::vector<int64_t*> d_eo;
  std::vector<int32_t*> d_src, d_dst, d_smp;
};

struct HopLog {
  int hop = 0;
  std::vector<Chunk> chunks;
  std::vector<ChunkLog> log;
};

void apply_tuning(LaunchCfg& L, const csaw_tuning* t);
// CSAW_ERR_INVALID_ARG for shapes out of range (workgroups per CU 0..64,
// chunk_min a power of two in 8..1024, group_min 4..32; 0 keeps a default).
int validate_tuning(const csaw_tuning* t);
int mlp_upload_bf16(const csaw_mlp* m, uint16_t* dst);

// A call's device work on a plan's arrays, counted from before its first launch
// until the call has waited for it.  A call that does not wait, or whose launch or
// wait fails, leaves its count.
struct InFlight {
  std::atomic<int64_t>& n;
  explicit InFlight(std::atomic<int64_t>& count) : n(count) { ++n; }
  void waited() { --n; }
};

}  // namespace csaw

struct csaw_plan {
  csaw_graph* g = nullptr;
  std::vector<csaw_request> reqs;
  std::vector<std::pair<int, int>> req_unit;  // (unit, index in unit)
  csaw_plan_opts opts;
  std::vector<csaw::Unit> units;
  uint32_t* local_excl = nullptr;
  int32_t* order = nullptr;
  uint8_t* kind_mask = nullptr;  // whole-hop kernels of several kinds (HopDev)
  uint32_t* blk_excl = nullptr;
  uint32_t* blk_scan = nullptr;
  uint64_t* grp_excl = nullptr;
  csaw::Chunk* chunks = nullptr;
  uint32_t chunk_cap = 0;
  // every device array below and the units' (one allocation)
  std::shared_ptr<csaw::Workspace> work;
  csaw::Workspace::Block slab;
  mutable std::atomic<int64_t> unwaited{0};  // calls whose work may still use it (InFlight)
  int32_t* staging = nullptr;         // csaw_sample: the result, packed for one copy
  // counter block, then the requests' edge bounds (kCtrBytes + n_req *
  // kBoundsBytes): one copy into h_state after a synchronised run brings the
  // overflow flag and every request's place to the host
  uint32_t* counters = nullptr;
  int64_t* bounds = nullptr;          // in the same allocation
  std::vector<uint32_t> h_state;
  bool bounds_known = false;          // h_state is of the last run
  uint32_t* queues = nullptr;
  int64_t queue_cap = 0;
  int64_t* totals = nullptr;
  uint8_t* chosen = nullptr;
  csaw::ChunkLog* log = nullptr;
  uint16_t* d_mlp = nullptr;
  unsigned long long* bytes_acc = nullptr;  // algorithmic bytes per kernel kind (timing runs)
  csaw::LaunchCfg L;
  csaw::PlanStreams st;   // main stream; batched: side streams the expansion
                          // kernels of a hop fan out to, joined before the next hop
  hipStream_t stream = nullptr;
  bool fan = false;       // this plan uses the side streams
  hipGraphExec_t gexec = nullptr;
  hipStream_t graph_stream = nullptr;
  csaw::EventTimer timer;
  double last_ms = 0.0;
  int64_t runs = 0;
  std::vector<csaw::HopLog> hop_logs;
  std::vector<int> pending_log_hops;
};
