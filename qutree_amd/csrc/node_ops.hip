// Node-level contractions: mode-k products (matvec/tmatvec/ctmatvec semantics
// of LA_lib.f, matrixTensorBLAS semantics of TensorBLAS.cpp) and hole
// contractions (rhomat / contractionBLAS), single and grouped, all on MFMA
// tile kernels: a mode product is a GEMM over the flattened (before, after)
// rows, a hole contraction a GEMM over the flattened (before, after) reduction
// index.  Where 32-bit offsets reach, hole contractions and the products of
// large plans take the register-blocked kernels of gemm_block.hip (long
// reductions shared by workgroups, whose partial tiles are added in order),
// the rest those of gemm_ops.hip.
#include <algorithm>
#include <climits>
#include <cmath>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "common.hpp"
#include "gemm_ops.hpp"

namespace qtg {

static_assert(sizeof(qtg_mode_product_desc) == 64, "descriptor layout");
static_assert(sizeof(qtg_hole_contraction_desc) == 64, "descriptor layout");

namespace {

constexpr int64_t kSplitK = 512;  // K per task of a split hole contraction

int to_gm(const qtg_mode_product_desc& d, GmDesc& g) {
  if (d.before < 1 || d.after < 1 || d.nB < 1 || d.nC < 1 || d.op < 0 || d.op > 2) {
    set_error("mode product: need nB, nC, before, after >= 1 and op in {0,1,2}");
    return QTG_ESHAPE;
  }
  // the tile kernels index rows of the flattened (before, after) in 64 bits
  // and matrices in 32 bits; every product is checked before it is formed
  if (d.before > INT_MAX || d.after > INT_MAX || d.nB > INT_MAX || d.nC > INT_MAX ||
      d.before * d.after > ((int64_t)1 << 40) || d.nB * d.nC >= ((int64_t)1 << 31) ||
      d.before * d.after > (((int64_t)1 << 62) / std::max(d.nB, d.nC))) {
    set_error("mode product: dimensions out of range");
    return QTG_ESHAPE;
  }
  g = GmDesc{};
  g.x = d.offB;
  g.m = d.offM;
  g.out = d.offC;
  g.bef = (int32_t)d.before;
  g.nin = (int32_t)d.nB;
  g.nout = (int32_t)d.nC;
  g.aft = (int32_t)d.after;
  g.op = d.op;
  g.acc = d.add ? 1 : 0;
  g.are = 1.0;
  g.aim = 0.0;
  g.node = -1;
  g.ksplit = 1;
  return QTG_OK;
}

int to_gc(const qtg_hole_contraction_desc& d, GcDesc& g) {
  if (d.before < 1 || d.after < 1 || d.nA < 1 || d.nB < 1) {
    set_error("hole contraction: dimensions must be >= 1");
    return QTG_ESHAPE;
  }
  // The reduction walks k = b + a before over K = before * after and steps a
  // by before * n (gc_product): both stay in 32 bits only below 2^31, with
  // 16 more for the last k-step's overrun.
  const int64_t lim = (int64_t)1 << 31;
  if (d.before >= lim || d.after >= lim || d.nA >= lim || d.nB >= lim || d.before * d.after + 16 >= lim ||
      d.before * std::max(d.nA, d.nB) >= lim || d.nA * d.nB >= lim) {
    set_error("hole contraction: before*after and before*max(nA, nB) must stay below 2^31");
    return QTG_ESHAPE;
  }
  g = GcDesc{};
  g.x = d.offA;
  g.y = d.offB;
  g.out = d.offS;
  g.bef = (int32_t)d.before;
  g.nx = (int32_t)d.nA;
  g.ny = (int32_t)d.nB;
  g.aft = (int32_t)d.after;
  g.acc = d.accumulate ? 1 : 0;
  g.node = -1;
  g.ksplit = 1;
  g.sel = 2;  // X from the first input base, Y from the second
  return QTG_OK;
}

template <typename R>
int mode_product_one(const qtg_mode_product_desc& d, cplx<R>* C, const cplx<R>* M, const cplx<R>* B, hipStream_t s) {
  if (!C || !M || !B) {
    set_error("mode product: null pointer");
    return QTG_EARG;
  }
  GmDesc g;
  int rc = to_gm(d, g);
  if (rc) return rc;
  return launch_gm_single<R>(g, B, M, C, s);
}

// A plan: descriptors [0, nblock) run in a register-blocked kernel
// (gemm_block.hip), the rest in a general grouped kernel.
struct Plan {
  int kind = 0;  // 0 mode product, 1 hole contraction
  bool c64 = false;
  int64_t nblock = 0, block_tasks = 0, nsums = 0;
  int64_t ngen = 0, gen_tasks = 0;
  bool gen_lean = false;  // every general descriptor takes the lean form
  void* d_descs = nullptr;
  void* d_block = nullptr;  // gm_block: descriptor of every task; gc_block: GcBlockWg of every workgroup, then the sums
  void* d_wg = nullptr;     // general kernel: descriptor of every task
  double flops = 0, bytes = 0;
  // Shared reductions (nsums > 0): their partial macro tiles, which an
  // execution uses from its first launch to its last, in up to kPlanSlots sets
  // of part_bytes within kPlanPartBytes.  A stream keeps to the set it used
  // last, another takes the oldest; every set's uses are ordered by its event,
  // recorded behind each.  Under capture the plan runs unshared (d_descs1,
  // d_block1: a workgroup per macro tile), since a replay could not be ordered.
  // One set alone put the executions of all streams in one line: 16 tensors of
  // legs 8-31 on four streams 34 us each, 10 without shared reductions.
  struct Slot {
    hipEvent_t done = nullptr;
    hipStream_t last = nullptr;
    uint64_t use = 0;  // 0: never
  };
  static constexpr int kPlanSlots = 4;
  static constexpr size_t kPlanPartBytes = (size_t)32 << 20;
  void* d_part = nullptr;
  size_t part_bytes = 0;
  int nslots = 0;
  Slot slots[kPlanSlots];
  uint64_t uses = 0;
  void* d_descs1 = nullptr;
  void* d_block1 = nullptr;
  int64_t block_tasks1 = 0;
  std::mutex mu;
  ~Plan() {
    for (void* p : {d_descs, d_block, d_wg, d_part, d_descs1, d_block1})
      if (p) (void)hipFree(p);
    for (Slot& x : slots)
      if (x.done) (void)hipEventDestroy(x.done);
  }
};

template <typename X>
int upload(void** dst, const std::vector<X>& v) {
  *dst = nullptr;
  if (v.empty()) return QTG_OK;
  QTG_HIP_TRY(hipMalloc(dst, sizeof(X) * v.size()));
  QTG_HIP_TRY(hipMemcpy(*dst, v.data(), sizeof(X) * v.size(), hipMemcpyHostToDevice));
  return QTG_OK;
}

// The descriptors of the blocked kernel come first; uploads all tables.
template <typename D>
int finish_plan(Plan& p, std::vector<D>& block, std::vector<D>& gen, int64_t (*tasks)(const D&),
                bool (*lean_ok)(const D&)) {
  std::vector<int32_t> wg;
  p.nblock = (int64_t)block.size();
  p.ngen = (int64_t)gen.size();
  p.gen_tasks = order_tasks(gen, tasks);
  p.gen_lean = std::all_of(gen.begin(), gen.end(), lean_ok);
  gemm_wg_table(gen.data(), p.ngen, p.gen_tasks, wg);
  block.insert(block.end(), gen.begin(), gen.end());
  int rc = upload(&p.d_descs, block);
  if (!rc) rc = upload(&p.d_wg, wg);
  return rc;
}

// Mode products of more than 16 columns take 32 x 32 outputs a wavefront
// when the plan then still has kMinBlockTasks wavefronts (eight a SIMD):
// 500 tensors of legs 17-48 221 -> 195 us, 49-64 1300 -> 1023 us (complex128),
// 852 -> 643 us (complex64).  Below, and for up to 16 columns, one 16 x 16
// tile a wavefront is the faster form: 16 tensors of legs 8-64 14.5 against
// 19.5 us, 2000 of legs 3-20 25.9 against 33 us.
constexpr int64_t kMinBlockTasks = 8192;
bool gm_blocked(const GmDesc& g) { return gm_lean_ok(g) && g.nout > 16; }

// A hole contraction of a plan: blocked where its offsets fit 32 bits.
void add_gc(GcDesc& g, std::vector<GcDesc>& block, std::vector<GcDesc>& gen) {
  if (gc_lean_ok(g)) {
    block.push_back(g);
    return;
  }
  const int64_t K = (int64_t)g.bef * g.aft;
  if (K > 2 * kSplitK) g.ksplit = split_chunks(K, kGemmWaves, 1);
  gen.push_back(g);
}

// The workgroups of the blocked hole contractions: every reduction in
// `ksplit` shares, toward about kTargetWgs workgroups of equal work in all
// (two per CU) and at least kMinShare elements each (a share costs a 16 KB
// partial tile where it reads 64 columns).  The macro tiles of a share read
// the same operands, so they go to one XCD (workgroup index mod 8), where
// they meet in its L2: 1204 -> 1086 us for 4096 tensors of legs 8-64, 1279
// -> 984 us for 1000 of legs 33-48.  The shares are dealt to the XCD with the
// least work so far, the heaviest first, so the launch also ends with its
// short workgroups; where a queue has run out the others close up, which
// moves only the lightest units.
struct GcBlockPlan {
  std::vector<GcBlockWg> wgs, sums;
  int64_t parts = 0;  // partial macro tiles
};
constexpr int64_t kTargetWgs = 512;
GcBlockPlan plan_gc_blocks(std::vector<GcDesc>& v, int64_t targetWgs = kTargetWgs) {
  constexpr int kXcds = 8;
  constexpr int64_t kMinShare = 256;
  GcBlockPlan p;
  auto work = [](const GcDesc& d) {
    return (double)d.bef * d.aft * ((d.nx + 15) / 16) * ((d.ny + 15) / 16);
  };
  double total = 0.0;
  for (auto& d : v) total += work(d);
  struct Unit {
    double w;
    int32_t desc, share, part;
  };
  std::vector<Unit> units;
  for (size_t i = 0; i < v.size(); ++i) {
    GcDesc& d = v[i];
    const int64_t K = (int64_t)d.bef * d.aft, m = gc_block_macros(d);
    // m shares of more than total / kTargetWgs each: the partial tiles of a
    // plan stay below 2 kTargetWgs
    const int64_t want = (int64_t)std::ceil(work(d) / (double)m * (double)targetWgs / total);
    d.ksplit = (int32_t)std::max<int64_t>(1, std::min(want, K / kMinShare));
    for (int32_t s = 0; s < d.ksplit; ++s) units.push_back({work(d) / d.ksplit, (int32_t)i, s, (int32_t)p.parts});
    if (d.ksplit > 1) {
      for (int64_t t = 0; t < m; ++t) p.sums.push_back({(int32_t)i, (int32_t)t, (int32_t)(p.parts + t * d.ksplit), 0});
      p.parts += m * d.ksplit;
    }
  }
  std::stable_sort(units.begin(), units.end(), [](const Unit& a, const Unit& b) { return a.w > b.w; });
  std::vector<GcBlockWg> q[kXcds];
  double load[kXcds] = {};
  for (const Unit& u : units) {
    const int x = (int)(std::min_element(load, load + kXcds) - load);
    load[x] += u.w;
    const GcDesc& d = v[u.desc];
    const int64_t m = gc_block_macros(d);
    for (int64_t t = 0; t < m; ++t)
      q[x].push_back({u.desc, (int32_t)(t * d.ksplit + u.share), (int32_t)(u.part + t * d.ksplit + u.share), 0});
  }
  size_t len = 0;
  for (auto& x : q) len = std::max(len, x.size());
  for (size_t k = 0; k < len; ++k)
    for (auto& x : q)
      if (k < x.size()) p.wgs.push_back(x[k]);
  return p;
}

int upload_gc_blocks(Plan& p, std::vector<GcDesc>& v) {
  if (v.empty()) return QTG_OK;
  GcBlockPlan g = plan_gc_blocks(v);
  p.block_tasks = (int64_t)g.wgs.size();
  p.nsums = (int64_t)g.sums.size();
  g.wgs.insert(g.wgs.end(), g.sums.begin(), g.sums.end());
  if (g.parts > 0) {
    const size_t es = p.c64 ? sizeof(cplx<float>) : sizeof(cplx<double>);
    p.part_bytes = (size_t)g.parts * 1024 * es;
    p.nslots = (int)std::max<size_t>(1, std::min<size_t>(Plan::kPlanSlots, Plan::kPlanPartBytes / p.part_bytes));
    if (hipMalloc(&p.d_part, p.nslots * p.part_bytes) != hipSuccess) {
      (void)hipGetLastError();
      p.d_part = nullptr;
      set_error("plan: device allocation of the partial tiles failed");
      return QTG_ENOMEM;
    }
    for (int i = 0; i < p.nslots; ++i)
      QTG_HIP_TRY(hipEventCreateWithFlags(&p.slots[i].done, hipEventDisableTiming));
    std::vector<GcDesc> one = v;
    const GcBlockPlan g1 = plan_gc_blocks(one, 0);
    p.block_tasks1 = (int64_t)g1.wgs.size();
    int rc = upload(&p.d_descs1, one);
    if (!rc) rc = upload(&p.d_block1, g1.wgs);
    if (rc) return rc;
  }
  return upload(&p.d_block, g.wgs);
}

// (a query that fails counts as a capture: the launches then need no ordering)
bool capturing(hipStream_t s) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &cap) == hipSuccess) return cap != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return true;
}

template <typename T>
int run_plan(Plan& p, void* out, const void* first, const void* second, hipStream_t s) {
  int rc = QTG_OK;
  if (p.kind == 0) {
    // first = M base, second = B base
    const GmDesc* g = (const GmDesc*)p.d_descs;
    rc = launch_gm_block<T>(g, (const int32_t*)p.d_block, p.block_tasks, second, first, out, s);
    if (rc) return rc;
    return launch_gm<T, T, T>(g + p.nblock, (const int32_t*)p.d_wg, p.ngen, p.gen_tasks, second, second, first, out,
                              nullptr, 1.0, 0.0, s, nullptr, kGemmWaves, p.gen_lean);
  }
  // X (bra) from the first base, Y (ket) from the second: sel = 2 on every descriptor
  const GcDesc* g = (const GcDesc*)p.d_descs;
  const GcBlockWg* wgs = (const GcBlockWg*)p.d_block;
  if (p.nsums == 0) {
    rc = launch_gc_block<T>(g, wgs, p.block_tasks, wgs, 0, first, second, out, nullptr, s);
  } else if (capturing(s)) {
    const GcBlockWg* w1 = (const GcBlockWg*)p.d_block1;
    rc = launch_gc_block<T>((const GcDesc*)p.d_descs1, w1, p.block_tasks1, w1, 0, first, second, out, nullptr, s);
  } else {
    std::lock_guard<std::mutex> lock(p.mu);
    int k = 0;
    for (int i = 1; i < p.nslots; ++i)
      if (p.slots[i].use < p.slots[k].use) k = i;
    for (int i = 0; i < p.nslots; ++i)
      if (p.slots[i].use && p.slots[i].last == s) k = i;
    Plan::Slot& x = p.slots[k];
    if (x.use) QTG_HIP_TRY(hipStreamWaitEvent(s, x.done, 0));
    x.use = ++p.uses;
    x.last = s;
    rc = launch_gc_block<T>(g, wgs, p.block_tasks, wgs + p.block_tasks, p.nsums, first, second, out,
                            static_cast<unsigned char*>(p.d_part) + k * p.part_bytes, s);
    QTG_HIP_TRY(hipEventRecord(x.done, s));
  }
  if (rc) return rc;
  return launch_gc<T, T>(g + p.nblock, (const int32_t*)p.d_wg, p.ngen, p.gen_tasks, first, second, out, nullptr, s,
                         nullptr, p.gen_lean);
}

// ------------------------------------------------ no-allocation variant
// Device-resident staging of qtg_hole_contraction_grouped_noalloc_z: the
// converted descriptors, then the tables of a plan: the workgroups of the
// blocked kernel (at most one per 16 x 16 tile and 2 kTargetWgs shares) and
// its sums, or, for descriptors beyond the blocked kernel's 32-bit offsets,
// the descriptor of every task.  Each GPU holds its own copy for the life of
// the process.
constexpr int64_t kNoAllocMaxDescs = 4096;
constexpr int64_t kNoAllocMaxTasks = 1 << 18;
constexpr size_t kNoAllocTableOff = (size_t)kNoAllocMaxDescs * sizeof(GcDesc);
constexpr size_t kNoAllocBytes = kNoAllocTableOff + (size_t)(kNoAllocMaxTasks + 4 * kTargetWgs) * sizeof(GcBlockWg);
static_assert(kNoAllocTableOff % 256 == 0, "table alignment");

}  // namespace
}  // namespace qtg

// In host code these names are only handles for hipGetSymbolAddress: kernels
// receive the per-device address it returns (symbol_address).
static __device__ __align__(256) unsigned char scratch[qtg::kNoAllocBytes];
// Partial tiles of single hole contractions split over workgroups, in slots
// (see PartPool): 8 MiB hold the 128 shares of a 64 x 64 complex128 output.
constexpr int kPartSlots = 4;
constexpr size_t kPartBytes = (size_t)8 << 20;
static __device__ __align__(256) unsigned char part_scratch[kPartSlots * kPartBytes];

namespace qtg {
namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The current device's copy of a device array, looked up once per device
// with that device current (cache under mu, which the caller holds).
int symbol_address(const void* symbol, int dev, void* (&cache)[kMaxDevices], const char* what, void** out) {
  if (dev < 0 || dev >= kMaxDevices) {
    set_error(std::string(what) + ": device index out of range");
    return QTG_EDEVICE;
  }
  if (!cache[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, symbol);
    if (e != hipSuccess || !p) {
      set_error(std::string(what) + ": hipGetSymbolAddress: " + hipGetErrorString(e));
      return QTG_EDEVICE;
    }
    cache[dev] = p;
  }
  *out = cache[dev];
  return QTG_OK;
}

int scratch_address(void** out) {
  int dev = 0;
  QTG_HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return symbol_address(HIP_SYMBOL(scratch), dev, g_scratch_ptr, "no-allocation contraction", out);
}

// The slots of part_scratch, per device.  A call holds the lock while it
// enqueues its two launches and records the slot's event behind them; the
// next user of a slot, on whatever stream and thread, makes its stream wait
// for that event.  A stream keeps to the slot it used last, another takes the
// one used longest ago.  (Asking whether an event has passed would end a
// capture that is open on any other stream of the thread.)  Nothing is
// allocated but the events.
struct PartPool {
  std::mutex mu;
  void* base[kMaxDevices] = {};
  hipEvent_t ev[kMaxDevices][kPartSlots] = {};
  hipStream_t last[kMaxDevices][kPartSlots] = {};
  uint64_t use[kMaxDevices][kPartSlots] = {};  // 0: never
  uint64_t uses = 0;
};
PartPool g_parts;

// the array's address and the slots' events, which the first call makes (with
// captures on other streams left alone by it)
int part_slots(int dev, void** base) {
  if (g_parts.base[dev] && g_parts.ev[dev][kPartSlots - 1]) {
    *base = g_parts.base[dev];
    return QTG_OK;
  }
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  QTG_HIP_TRY(hipThreadExchangeStreamCaptureMode(&mode));
  int rc = symbol_address(HIP_SYMBOL(part_scratch), dev, g_parts.base, "hole contraction", base);
  for (int i = 0; i < kPartSlots && !rc; ++i)
    if (!g_parts.ev[dev][i] &&
        hipEventCreateWithFlags(&g_parts.ev[dev][i], hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      g_parts.ev[dev][i] = nullptr;
      set_error("hole contraction: hipEventCreate failed");
      rc = QTG_EDEVICE;
    }
  QTG_HIP_TRY(hipThreadExchangeStreamCaptureMode(&mode));
  return rc;
}

template <typename R>
int hole_split(const GcDesc& g, const GcOnePlan& p, const cplx<R>* A, const cplx<R>* B, cplx<R>* Sm, hipStream_t s) {
  int dev = 0;
  QTG_HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) {
    set_error("hole contraction: device index out of range");
    return QTG_EDEVICE;
  }
  std::lock_guard<std::mutex> lock(g_parts.mu);
  void* base = nullptr;
  int rc = part_slots(dev, &base);
  if (rc) return rc;
  int slot = 0;
  for (int i = 1; i < kPartSlots; ++i)
    if (g_parts.use[dev][i] < g_parts.use[dev][slot]) slot = i;
  for (int i = 0; i < kPartSlots; ++i)
    if (g_parts.use[dev][i] && g_parts.last[dev][i] == s) slot = i;
  if (g_parts.use[dev][slot]) QTG_HIP_TRY(hipStreamWaitEvent(s, g_parts.ev[dev][slot], 0));
  g_parts.use[dev][slot] = ++g_parts.uses;
  g_parts.last[dev][slot] = s;
  rc = launch_gc_one<R>(g, p, A, B, Sm, static_cast<unsigned char*>(base) + (size_t)slot * kPartBytes, s);
  // also after a failed launch: the first of the two may run
  const hipError_t e = hipEventRecord(g_parts.ev[dev][slot], s);
  if (!rc && e != hipSuccess) {
    set_error(std::string("hole contraction: hipEventRecord: ") + hipGetErrorString(e));
    rc = QTG_EDEVICE;
  }
  return rc;
}

// launch(base) with the slots as one buffer, behind their last uses; launch
// returns when its work on the device is done.
template <typename F>
int with_all_parts(hipStream_t s, F&& launch) {
  int dev = 0;
  QTG_HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) {
    set_error("hole contraction: device index out of range");
    return QTG_EDEVICE;
  }
  std::lock_guard<std::mutex> lock(g_parts.mu);
  void* base = nullptr;
  int rc = part_slots(dev, &base);
  if (rc) return rc;
  for (int i = 0; i < kPartSlots; ++i)
    if (g_parts.use[dev][i]) QTG_HIP_TRY(hipStreamWaitEvent(s, g_parts.ev[dev][i], 0));
  return launch(base);
}

// Reductions long enough for it split over workgroups (plan_gc_one), except
// under stream capture: a replayed graph would use its slot unordered with
// other calls.
template <typename R>
int hole_one(const qtg_hole_contraction_desc& d, cplx<R>* Sm, const cplx<R>* A, const cplx<R>* B, hipStream_t s) {
  if (!Sm || !A || !B) {
    set_error("hole contraction: null pointer");
    return QTG_EARG;
  }
  GcDesc g;
  int rc = to_gc(d, g);
  if (rc) return rc;
  if (!gc_lean_ok(g)) return launch_gc_single<R>(g, A, B, Sm, s);
  GcOnePlan p = plan_gc_one(g, (int64_t)(kPartBytes / sizeof(cplx<R>)));
  if (p.S > 1 && capturing(s)) p = plan_gc_one(g, 0);
  if (p.S > 1) return hole_split<R>(g, p, A, B, Sm, s);
  return launch_gc_one<R>(g, p, A, B, Sm, nullptr, s);
}

}  // namespace
}  // namespace qtg

using namespace qtg;

extern "C" {

int qtg_mode_product_z(double* C, const double* M, const double* B, int64_t before, int64_t nB, int64_t nC,
                       int64_t after, int op, int add, qtg_stream stream) {
  qtg_mode_product_desc d{0, 0, 0, before, nB, nC, after, op, add};
  return mode_product_one<double>(d, (cplx<double>*)C, (const cplx<double>*)M, (const cplx<double>*)B,
                                        S(stream));
}
int qtg_mode_product_c(float* C, const float* M, const float* B, int64_t before, int64_t nB, int64_t nC,
                       int64_t after, int op, int add, qtg_stream stream) {
  qtg_mode_product_desc d{0, 0, 0, before, nB, nC, after, op, add};
  return mode_product_one<float>(d, (cplx<float>*)C, (const cplx<float>*)M, (const cplx<float>*)B,
                                       S(stream));
}
int qtg_matvec_z(double* C, const double* B, const double* M, int64_t a, int64_t b, int64_t c, int add,
                 qtg_stream stream) {
  return qtg_mode_product_z(C, M, B, b, a, a, c, 0, add, stream);
}
int qtg_tmatvec_z(double* C, const double* B, const double* M, int64_t a, int64_t b, int64_t c, int add,
                  qtg_stream stream) {
  return qtg_mode_product_z(C, M, B, b, a, a, c, 1, add, stream);
}
int qtg_ctmatvec_z(double* C, const double* B, const double* M, int64_t a, int64_t b, int64_t c, int add,
                   qtg_stream stream) {
  return qtg_mode_product_z(C, M, B, b, a, a, c, 2, add, stream);
}
int qtg_hole_contraction_z(double* Sm, const double* A, const double* B, int64_t before, int64_t nA, int64_t nB,
                           int64_t after, int accumulate, qtg_stream stream) {
  qtg_hole_contraction_desc d{0, 0, 0, before, nA, nB, after, accumulate, 0};
  return hole_one<double>(d, (cplx<double>*)Sm, (const cplx<double>*)A, (const cplx<double>*)B,
                                S(stream));
}
int qtg_hole_contraction_c(float* Sm, const float* A, const float* B, int64_t before, int64_t nA, int64_t nB,
                           int64_t after, int accumulate, qtg_stream stream) {
  qtg_hole_contraction_desc d{0, 0, 0, before, nA, nB, after, accumulate, 0};
  return hole_one<float>(d, (cplx<float>*)Sm, (const cplx<float>*)A, (const cplx<float>*)B, S(stream));
}
int qtg_rhomat_z(const double* bra, const double* ket, double* M, int64_t a, int64_t b, int64_t c,
                 qtg_stream stream) {
  return qtg_hole_contraction_z(M, bra, ket, b, a, a, c, 0, stream);
}

int qtg_rmatvec_d(double* C, const double* B, const double* M, int64_t a, int64_t b, int64_t c, int add,
                  qtg_stream stream) {
  if (!C || !B || !M) {
    set_error("rmatvec: null pointer");
    return QTG_EARG;
  }
  qtg_mode_product_desc d{0, 0, 0, b, a, a, c, 0, add};
  GmDesc g;
  int rc = to_gm(d, g);
  if (rc) return rc;
  return launch_gm_real(g, B, M, C, S(stream));
}
int qtg_trmatvec_d(double* C, const double* B, const double* M, int64_t a, int64_t b, int64_t c, int add,
                   qtg_stream stream) {
  if (!C || !B || !M) {
    set_error("trmatvec: null pointer");
    return QTG_EARG;
  }
  qtg_mode_product_desc d{0, 0, 0, b, a, a, c, 1, add};
  GmDesc g;
  int rc = to_gm(d, g);
  if (rc) return rc;
  return launch_gm_real(g, B, M, C, S(stream));
}

int qtg_mode_product_plan_create(qtg_plan* plan, const qtg_mode_product_desc* descs, int64_t count,
                                 int complex64) {
  if (!plan || (!descs && count > 0) || count < 0 || count > INT_MAX) {
    set_error("plan: bad arguments");
    return QTG_EARG;
  }
  std::unique_ptr<Plan> p(new Plan());
  p->kind = 0;
  p->c64 = complex64 != 0;
  const double es = p->c64 ? 8.0 : 16.0;
  std::vector<GmDesc> block, gen;
  for (int64_t i = 0; i < count; ++i) {
    GmDesc g;
    int rc = to_gm(descs[i], g);
    if (rc) return rc;
    (gm_blocked(g) ? block : gen).push_back(g);
    const auto& d = descs[i];
    p->flops += 8.0 * d.before * d.after * d.nB * d.nC;
    p->bytes += es * (d.before * d.after * (d.nB + d.nC * (d.add ? 2 : 1)) + d.nB * d.nC);
  }
  for (auto& g : block) {
    g.tile0 = p->block_tasks;
    p->block_tasks += gm_block_tasks(g);
  }
  if (p->block_tasks < kMinBlockTasks) {
    gen.insert(gen.begin(), block.begin(), block.end());
    block.clear();
    p->block_tasks = 0;
  }
  std::vector<int32_t> wg;
  gemm_wg_table(block.data(), (int64_t)block.size(), p->block_tasks, wg);
  int rc = upload(&p->d_block, wg);
  if (!rc) rc = finish_plan<GmDesc>(*p, block, gen, gm_tasks, gm_lean_ok);
  if (rc) return rc;
  *plan = p.release();
  return QTG_OK;
}

int qtg_hole_contraction_plan_create(qtg_plan* plan, const qtg_hole_contraction_desc* descs, int64_t count,
                                     int complex64) {
  if (!plan || (!descs && count > 0) || count < 0 || count > INT_MAX) {
    set_error("plan: bad arguments");
    return QTG_EARG;
  }
  std::unique_ptr<Plan> p(new Plan());
  p->kind = 1;
  p->c64 = complex64 != 0;
  const double es = p->c64 ? 8.0 : 16.0;
  std::vector<GcDesc> block, gen;
  for (int64_t i = 0; i < count; ++i) {
    GcDesc g;
    int rc = to_gc(descs[i], g);
    if (rc) return rc;
    add_gc(g, block, gen);
    const auto& d = descs[i];
    const int64_t K = d.before * d.after;
    p->flops += 8.0 * K * d.nA * d.nB;
    p->bytes += es * (K * (d.nA + d.nB) + d.nA * d.nB * (d.accumulate ? 2 : 1));
  }
  int rc = upload_gc_blocks(*p, block);
  if (!rc) rc = finish_plan<GcDesc>(*p, block, gen, gc_tasks, gc_lean_ok);
  if (rc) return rc;
  *plan = p.release();
  return QTG_OK;
}

int qtg_plan_execute(qtg_plan plan, void* out_base, const void* first_base, const void* second_base,
                     qtg_stream stream) {
  auto* p = static_cast<Plan*>(plan);
  if (!p || !out_base || !first_base || !second_base) {
    set_error("plan execute: null argument");
    return QTG_EARG;
  }
  return p->c64 ? run_plan<float>(*p, out_base, first_base, second_base, S(stream))
                : run_plan<double>(*p, out_base, first_base, second_base, S(stream));
}

int qtg_hole_contraction_grouped_noalloc_z(const qtg_hole_contraction_desc* descs, int64_t count, double* S_base,
                                           const double* A_base, const double* B_base, qtg_stream stream) {
  if ((!descs && count > 0) || count < 0 || !S_base || !A_base || !B_base) {
    set_error("no-allocation contraction: bad arguments");
    return QTG_EARG;
  }
  if (count > kNoAllocMaxDescs) {
    set_error("no-allocation contraction: more than " + std::to_string(kNoAllocMaxDescs) + " descriptors");
    return QTG_ESHAPE;
  }
  if (count == 0) return QTG_OK;
  // the same descriptors, K shares and kernels as a plan of these descs
  std::vector<GcDesc> block, gen;
  int64_t tiles = 0;
  for (int64_t i = 0; i < count; ++i) {
    GcDesc g;
    int rc = to_gc(descs[i], g);
    if (rc) return rc;
    add_gc(g, block, gen);
    tiles += (int64_t)((g.nx + 15) / 16) * ((g.ny + 15) / 16) *
             ((int64_t)g.bef * g.aft > 2 * kSplitK ? kGemmWaves : 1);
  }
  if (tiles > kNoAllocMaxTasks) {
    set_error("no-allocation contraction: more than " + std::to_string(kNoAllocMaxTasks) + " 16 x 16 tiles");
    return QTG_ESHAPE;
  }
  void* base = nullptr;
  int rc = scratch_address(&base);
  if (rc) return rc;
  hipStream_t s = S(stream);
  GcDesc* d_descs = reinterpret_cast<GcDesc*>(base);
  unsigned char* d_table = static_cast<unsigned char*>(base) + kNoAllocTableOff;
  // the staging tables are host temporaries and the device copy is shared by
  // every call on this GPU: each part returns with its result written
  if (!block.empty()) {
    GcBlockPlan p = plan_gc_blocks(block);
    const int64_t nwg = (int64_t)p.wgs.size(), nsums = (int64_t)p.sums.size();
    p.wgs.insert(p.wgs.end(), p.sums.begin(), p.sums.end());
    if (p.wgs.size() * sizeof(GcBlockWg) > kNoAllocBytes - kNoAllocTableOff ||
        (size_t)p.parts * 1024 * sizeof(cplx<double>) > kPartSlots * kPartBytes) {
      set_error("no-allocation contraction: tables exceed the fixed array");
      return QTG_ESHAPE;
    }
    QTG_HIP_TRY(hipMemcpyAsync(d_descs, block.data(), sizeof(GcDesc) * block.size(), hipMemcpyHostToDevice, s));
    QTG_HIP_TRY(hipMemcpyAsync(d_table, p.wgs.data(), sizeof(GcBlockWg) * p.wgs.size(), hipMemcpyHostToDevice, s));
    const GcBlockWg* wgs = reinterpret_cast<const GcBlockWg*>(d_table);
    auto launch = [&](void* part) -> int {
      int e = launch_gc_block<double>(d_descs, wgs, nwg, wgs + nwg, nsums, A_base, B_base, S_base, part, s);
      if (e) return e;
      QTG_HIP_TRY(hipStreamSynchronize(s));
      return QTG_OK;
    };
    rc = p.parts > 0 ? with_all_parts(s, launch) : launch(nullptr);
    if (rc) return rc;
  }
  if (!gen.empty()) {
    const int64_t tasks = order_tasks(gen, gc_tasks);
    std::vector<int32_t> wg;
    gemm_wg_table(gen.data(), (int64_t)gen.size(), tasks, wg);
    QTG_HIP_TRY(hipMemcpyAsync(d_descs, gen.data(), sizeof(GcDesc) * gen.size(), hipMemcpyHostToDevice, s));
    QTG_HIP_TRY(hipMemcpyAsync(d_table, wg.data(), sizeof(int32_t) * wg.size(), hipMemcpyHostToDevice, s));
    rc = launch_gc<double, double>(d_descs, reinterpret_cast<const int32_t*>(d_table), (int64_t)gen.size(), tasks,
                                   A_base, B_base, S_base, nullptr, s);
    if (rc) return rc;
    QTG_HIP_TRY(hipStreamSynchronize(s));
  }
  return QTG_OK;
}

int qtg_plan_destroy(qtg_plan plan) {
  delete static_cast<Plan*>(plan);
  return QTG_OK;
}

int qtg_plan_counts(qtg_plan plan, double* flops, double* bytes) {
  auto* p = static_cast<Plan*>(plan);
  if (!p) return QTG_EARG;
  if (flops) *flops = p->flops;
  if (bytes) *bytes = p->bytes;
  return QTG_OK;
}

}  // extern "C"
