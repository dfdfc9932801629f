// Which stream owns which of the library's workspaces, and whether the last launch on one has ended (wq_gemm_stream_host.hip).
// Host arithmetic only: an owner may be busy, in capture or destroyed, and HIP is never asked about another caller's stream.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wq {

constexpr int kSlotTiles = 512;  // what a launch that splits K over workgroups marks: its tiles or its workgroups, at most 9/8 times the CUs

// Workspaces of a device.  Calls of up to 16 rows, whose launches are short and which a program may have on many streams at once, have
// small ones of their own: without a slot such a call takes 2.2 times as long as on the decode kernel (1.6 - 2.9 times in eight of
// ten of 726 problems), with one 0.79 times.
constexpr int kSlots = 8, kDecodeSlots = 24;

// One workspace: the stream that launches on it, and for every tile (workgroup, where those share the finishing of one: `tiles` of them)
// the number of the launch that has read its partial sums last, written by the kernel into host memory.
struct Slot {
  hipStream_t stream = nullptr;
  const volatile uint32_t* done = nullptr;
  uint32_t launch = 0;  // the last one's number
  int tiles = 0;

  bool idle() const {
    for (int t = 0; t < tiles; ++t)
      if (done[t] != launch) return false;
    return true;
  }
};

// A slot belongs to a stream, whose calls run one after the other, and passes to a stream that has none once its owner's
// last launch has ended.  (A new stream at a destroyed one's address has that one's slot: hipStreamDestroy returns after
// the stream's work -- 82 ms of queued products, measured on streams of both kinds.)
template <int SLOTS>
struct SlotOwners {
  int used = 0;
  Slot slot[SLOTS];

  // nullptr if every slot is another stream's and busy
  Slot* take(hipStream_t s) {
    for (int i = 0; i < used; ++i)
      if (slot[i].stream == s) return &slot[i];
    if (used < SLOTS) {
      slot[used].stream = s;
      return &slot[used++];
    }
    for (Slot& o : slot)
      if (o.idle()) {
        o.stream = s;
        return &o;
      }
    return nullptr;
  }
};

}  // namespace wq
