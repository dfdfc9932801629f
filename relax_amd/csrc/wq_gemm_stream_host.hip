// Host side of the streamed GEMM (wq_gemm_stream.hip): the planned launch and the library's own workspaces.
#include <string.h>

#include <mutex>

#include "../../include/mi355x_wq.h"
#include "wq_internal.h"
#include "wq_slots.h"

namespace wq {

bool launch_gemm_stream(const Problem& p, int variant, int ksplit, const SplitSpace& space) {
  if (!gemm_stream_applicable(p)) return false;
  return p.bits == 4 ? launch_gemm_stream_bits<4>(p, variant, ksplit, space) : launch_gemm_stream_bits<8>(p, variant, ksplit, space);
}

bool launch_gemm_strip(const Problem& p, int tiles) {
  if (!gemm_strip_applicable(p)) return false;
  return p.bits == 4 ? launch_gemm_strip_bits<4>(p, tiles) : launch_gemm_strip_bits<8>(p, tiles);
}

bool gemm_stream_applicable(const Problem& p) {
  // groups of at least 32 (a lane's k of a stage share a scale); output rows of a tile within a 32-bit buffer
  return p.group >= 32 && p.n <= (4 << 20);
}

namespace {

// Workspaces of the library's own for calls that bring none; from 257 rows on where split_clearly_ahead says so.
// The memory is part of the code object (zero at load, as the counters have to be).  A call that finds
// no slot runs its windows one after the other, with the same result (kSerial in wq_gemm_stream.hip).  What that costs where the chip is idle otherwise (us: split,
// in turn, whole): int8 99 x 5120 x 13824 31.7, 73.5, 43.1, 300 x 5120 x 13824 59.7, 70.0, 73.1, 259 x 1096 x 11520 18.8, 57.2, 22.5; 75 problems
// of more than 256 rows 1.38 times the unsplit call (1.0 - 2.1).  With twelve streams at work, which is when a slot is missing, these take 0.97 of the
// unsplit calls' time (0.73 - 1.16).  Unsplit instead, the bits of a result would depend on what other streams do.
constexpr int64_t kSlotBytes = kSplitCounterBytes + (20ll << 20);  // (the largest plan: 288 windows of 128 x 128 float32)
__device__ unsigned char stream_slots[kSlots][kSlotBytes];
__device__ unsigned char decode_slots[kDecodeSlots][kDecodeSplitBytes];

// Under capture nothing of the library's is used: a graph may be replayed beside anything.
bool capturing(hipStream_t s) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &status) == hipSuccess) return status != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return true;
}

template <int SLOTS, int64_t BYTES>
struct Slots {
  std::mutex mutex;
  SlotOwners<SLOTS> owners;
  char* base = nullptr;
  uint32_t* done = nullptr;  // [SLOTS][kSlotTiles], host memory that the kernels write
};

// The memory of a device's slots: the workspaces and, at the first call that needs one, 2 KB of pinned host memory for each.
template <int SLOTS, int64_t BYTES>
bool find_memory(Slots<SLOTS, BYTES>* o, const void* symbol) {
  if (o->done != nullptr) return true;
  void* base = nullptr;
  void* done = nullptr;
  // (another thread may be capturing, which an allocation must not end)
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  const bool relaxed = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
  const bool ok = relaxed && hipGetSymbolAddress(&base, symbol) == hipSuccess &&
                  hipHostMalloc(&done, sizeof(uint32_t) * SLOTS * kSlotTiles, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) == hipSuccess;
  if (relaxed) (void)hipThreadExchangeStreamCaptureMode(&mode);
  if (!ok) {
    (void)hipGetLastError();
    return false;
  }
  memset(done, 0, sizeof(uint32_t) * SLOTS * kSlotTiles);
  o->base = static_cast<char*>(base);
  o->done = static_cast<uint32_t*>(done);
  return true;
}

// how many of a slot's `done` a launch writes
int launch_marks(const GemmPlan& plan) { return (int)plan.tiles * (plan.shares ? plan.split : 1); }

template <int SLOTS, int64_t BYTES>
SplitSpace take_slot(Slots<SLOTS, BYTES>* o, const void* symbol, hipStream_t s, const GemmPlan& plan, std::unique_lock<std::mutex>* lock) {
  if (plan.bytes > BYTES) return {};
  *lock = std::unique_lock<std::mutex>(o->mutex);
  if (!find_memory(o, symbol)) return {};
  Slot* const slot = o->owners.take(s);
  if (slot == nullptr) return {};
  const int64_t i = slot - o->owners.slot;
  slot->done = o->done + i * kSlotTiles;
  slot->tiles = launch_marks(plan);
  return SplitSpace{o->base + i * BYTES, o->done + i * kSlotTiles, ++slot->launch};
}

// A workspace for one launch of a plan on `s`; empty where there is none.  The caller passes `lock` in and keeps it until
// its launch is in the stream: another thread's launch on the same stream must not come between the two.
SplitSpace library_space(hipStream_t s, const GemmPlan& plan, bool decode, std::unique_lock<std::mutex>* lock) {
  if (s == hipStreamPerThread || launch_marks(plan) > kSlotTiles) return {};  // (one handle for a stream in every thread)
  static Slots<kSlots, kSlotBytes> slots[kMaxDevices];
  static Slots<kDecodeSlots, kDecodeSplitBytes> small[kMaxDevices];
  const int device = current_device_slot();
  return decode ? take_slot(&small[device], HIP_SYMBOL(decode_slots), s, plan, lock) : take_slot(&slots[device], HIP_SYMBOL(stream_slots), s, plan, lock);
}

}  // namespace

namespace {

// Up to 16 rows the decode kernel and the register-activation kernel read the weights faster, but for the long K that
// launch_gemm_stream_decode takes.  With K below 1024 a launch is mostly start-up and the kernels are level -- 600 x 15323 x 512: 38.2 us there, 36.3 - 40.9 here -- so those stay.
bool in_range(const Problem& p) { return p.m > 16 && p.k >= 1024 && gemm_stream_applicable(p); }

}  // namespace

int64_t gemm_workspace_bytes(const Problem& p, bool skinny_family) {
  if (!in_range(p) || !(skinny_family || launch_gemm_streams(p))) return 0;
  const GemmPlan plan = plan_stream(p, true);
  return plan.split > 1 && plan.us <= (skinny_family ? skinny_cost(p) : other_gemm_cost(p)) ? plan.bytes : 0;
}

namespace {

bool captured(const Problem& p) { return capturing(p.stream); }

int launched(bool ok, const char* which) {
  if (!ok) return -1;
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("gemm kernel (%s) launch failed: %s", which, hipGetErrorString(e));
    return -1;
  }
  return 1;
}

// `slot`: on a workspace of the library's
int launch_plan(const Problem& p, const GemmPlan& plan, void* workspace, bool slot) {
  std::unique_lock<std::mutex> slot_lock;
  SplitSpace space{plan.split > 1 ? workspace : nullptr, nullptr, 0};
  if (plan.split > 1 && slot) space = library_space(p.stream, plan, p.m <= 16, &slot_lock);
  return launched(launch_gemm_stream(p, plan.variant, plan.split, space), "streamed operands");
}

}  // namespace

namespace {

// The streamed plan of a call that brings so much workspace; `slot`: its split is to run on one of the library's.
GemmPlan plan_call(const Problem& p, int64_t workspace_bytes, bool* slot) {
  const GemmPlan plan = plan_stream(p, true);
  *slot = plan.split > 1 && plan.bytes > workspace_bytes;
  if (!*slot || !(p.m > 256 || captured(p))) return plan;
  // (hipStreamPerThread never has a slot: many rows are not split there)
  const GemmPlan whole = plan_stream(p, false);
  *slot = p.stream != hipStreamPerThread && split_clearly_ahead(plan, whole) && !captured(p);
  return *slot ? plan : whole;
}

}  // namespace

int launch_gemm_stream_planned(const Problem& p, void* workspace, int64_t workspace_bytes, float other_us) {
  if (!in_range(p)) return 0;
  bool slot;
  const GemmPlan plan = plan_call(p, workspace_bytes, &slot);
  const GemmPlan strip = plan_strip(p);
  switch (choose_streamed(p, strip, plan, other_us)) {
    case kOtherKernel: return 0;
    case kStrips: return launched(launch_gemm_strip(p, strip.variant), "strip");
    default: return launch_plan(p, plan, workspace, slot);
  }
}

bool launch_gemm_stream_unwatched(const Problem& p) {
  bool slot = false;
  const GemmPlan plan = in_range(p) ? plan_call(p, 0, &slot) : GemmPlan{};
  if (!slot || !plan.shares || strip_ahead(p, plan_strip(p), plan)) return false;
  std::unique_lock<std::mutex> slot_lock;
  SplitSpace space = library_space(p.stream, plan, false, &slot_lock);
  space.looks = 0;
  return space.base != nullptr && launch_gemm_stream(p, plan.variant, plan.split, space);
}

namespace {

// (gelu onto its own residual stays with the kernels it is on)
bool decode_applicable(const Problem& p) { return gemm_stream_applicable(p) && !(p.activation == MI355X_WQ_ACT_GELU && p.residual == p.y && p.y != nullptr); }

}  // namespace

int64_t decode_workspace_bytes(const Problem& p) {
  const int64_t decode = gemv_split_workspace_bytes(p);
  if (decode > 0 || !decode_applicable(p)) return decode;
  const GemmPlan plan = plan_decode_stream(p);
  return plan.split > 1 ? plan.bytes : 0;
}

int launch_gemm_stream_decode(const Problem& p, void* workspace, int64_t workspace_bytes) {
  if (!decode_streams(p) || !decode_applicable(p)) return 0;
  if (workspace == nullptr ? p.stream == hipStreamPerThread || captured(p) : gemv_split_workspace_bytes(p) > 0) return 0;
  const GemmPlan plan = plan_decode_stream(p);
  if (plan.split == 1 || (workspace != nullptr && plan.bytes > workspace_bytes)) return 0;
  return launch_plan(p, plan, workspace, workspace == nullptr);
}

}  // namespace wq
