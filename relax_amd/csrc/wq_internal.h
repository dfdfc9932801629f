// Host-side contract between the C ABI (wq_capi.cpp) and the kernel launchers.
#pragma once
#include <atomic>
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wq {

struct Problem {
  const void* x;
  const void* wq;
  const void* scales;
  void* y;
  int64_t m, n, k;
  int bits, group, zero_point;
  hipStream_t stream;
  // fused epilogue (all optional): y = f16add(act(f16add(f16(acc), bias[n])), residual[m,n])
  const void* bias = nullptr;
  const void* residual = nullptr;
  int activation = 0;  // 0 none, 1 relu
  // wq / scales are in the tile-major layout written by launch_tile_weights (see wq_tiled.hip)
  bool tiled = false;
  // the choice between kernels whose sums differ in order goes by the layout's own times; not for a forced kernel family,
  // whose results are the same on either layout
  bool choose_by_layout = true;
};

// Head of every workspace a K split uses: arrival counters, one per tile, shared by the kernels that split (row tiles of the
// decode kernel: N <= 65536).
constexpr int64_t kSplitMaxTiles = 4096;
constexpr int64_t kSplitCounterBytes = kSplitMaxTiles * 4;
constexpr int kStreamCounterWords = 16;  // of the streamed GEMM's split, a tile
// Counters and partial tiles of a call of up to 16 rows on memory of the library's.
constexpr int64_t kDecodeSplitBytes = kSplitCounterBytes + 4 * 1024 * 1024;

// Tuning variant: 0 = library default for the shape, >0 = explicit choice
// (only reachable through mi355x_wq_matmul_ex; used by sweeps).
int launch_gemv(const Problem& p, int variant);
// How the decode kernel requests its weights: a lane its own chunks, pairs of lanes whole lines, whole lines non-temporally; and which
// of them its default shape (eight wavefronts, two-chunk super steps) takes on tiles of so many rows, in rounds or not.
enum { kReadOwn, kReadPairs, kReadOnce };
int weight_reads(const Problem& p, int tile_rows, bool rounds);
bool gemv_applicable(const Problem& p);  // M <= 16 and a default variant's LDS plan (slots + activations) fits
// The decode kernel with its tiles in rounds, where the default takes that: 1 launched, 0 not its problem, -1 failure.
int launch_gemv_rounds(const Problem& p);
// Cross-workgroup K split of the decode kernel (M <= 16): bytes of caller workspace it needs for `p`
// (0 = no split for this problem), and the launch (1 launched, 0 not applicable / workspace too small,
// -1 failure).  The workspace holds float32 partial tiles and per-tile arrival counters; the counters
// must be zero before the first use and are zero again when the kernel has finished.
int64_t gemv_split_workspace_bytes(const Problem& p);
int launch_gemv_split(const Problem& p, void* workspace, int64_t workspace_bytes);
// The library's own file-scope device array for that split (no caller workspace, no allocation); nullptr with the error set
// where it cannot be resolved.
void* static_scratch_address();
int64_t gemv_static_scratch_bytes();
// (a workspace lets the streamed GEMM, where it is the default, split K)
int launch_skinny(const Problem& p, int variant, void* workspace, int64_t workspace_bytes);
int launch_gemm(const Problem& p, int variant, void* workspace, int64_t workspace_bytes);
bool launch_gemm_streams(const Problem& p);  // whether the GEMM family's default may be the streamed kernel for `p`
bool gemm_pipe_applicable(const Problem& p);  // K % 64 == 0, operands below 1 GiB
bool launch_gemm_pipe(const Problem& p, int group_shift, int variant);
// The streamed GEMM (wq_gemm_stream.hip): its tiles, an explicit launch, and the one its cost model picks (wq_gemm_plan.cpp)
// -- K split over workgroups where `workspace` has room for that and it pays -- unless another kernel's time on the problem,
// `other_us`, is less.  1 launched, 0 not its problem, -1 failure.
enum { kStream128x256 = 1, kStream128x128, kStream256x256, kStream64x128, kStream64x64, kStream32x64, kStream32x128, kStream64x96, kStream32x96 };
bool gemm_stream_applicable(const Problem& p);
// Whether the windows of such a tile split over workgroups share the finishing of it; else the last to arrive does that.
constexpr bool stream_split_shares(int rows, int columns) { return rows >= 64 && columns == 128; }
constexpr int kMaxWindows = 8;
constexpr int kSplitLooks = 8;  // looks of such a workgroup at its tile's counter before it gives its fellows up (a trip to memory of about 1 us each)
// Whether a tile of so many rows and columns, `macro_step` of K at a time, asks for `p`'s scales in pieces; and the tiles that have a build for it.
constexpr bool stream_pieces_built(int bits, int rows, int columns) { return bits == 8 || rows > 32 || columns > 64; }
bool stream_scale_pieces(const Problem& p, int rows, int columns, int macro_step);
// A workspace for K in windows over workgroups: the caller's, or one of the library's own, whose launches are numbered and
// write their number to `done`, in host memory, for every workgroup (where those share the finishing of a tile, else tile) whose share of the
// partial sums has been read.
struct SplitSpace {
  void* base = nullptr;
  uint32_t* done = nullptr;
  uint32_t launch = 0;
  int looks = kSplitLooks;  // (tests: 0, as if every workgroup's fellows came late)
};
// (K in `ksplit` windows: over workgroups on a workspace, without one one after the other, with the same result)
bool launch_gemm_stream(const Problem& p, int variant, int ksplit, const SplitSpace& space);
template <int BITS>
bool launch_gemm_stream_bits(const Problem& p, int variant, int ksplit, const SplitSpace& space);  // of that bit width
int launch_gemm_stream_planned(const Problem& p, void* workspace, int64_t workspace_bytes, float other_us);
// (tests) The planned split on the library's memory, no workgroup of which looks whether its fellows are in: all but a tile's last to arrive
// resign.  False where the call runs strips, the plan does not split, its windows do not share the finishing, or there is no memory for it.
bool launch_gemm_stream_unwatched(const Problem& p);
// launch_gemm_stream_planned for up to 16 rows, where decode_streams says so.  With a workspace: on that, where the decode kernel does not split K and it is
// large enough.  Without: on a slot, but not under capture nor on hipStreamPerThread, where the library has none
// for it and the decode kernel is ahead of the unsplit form.
int launch_gemm_stream_decode(const Problem& p, void* workspace, int64_t workspace_bytes);
// The workspace that a call of up to 16 rows splits K on, in the decode kernel or the streamed one; 0 where it would not.
int64_t decode_workspace_bytes(const Problem& p);
bool decode_streams(const Problem& p);
// The workspace that a call of `p` from 17 rows on splits K on, 0 where it would not.  (A call that the strips take leaves it alone: then
// the size is that of the streamed plan, as it is for a call on either kernel.)
int64_t gemm_workspace_bytes(const Problem& p, bool skinny_family);
// The strip kernel (wq_gemm_strip.hip): where it applies, the blocks of eight rows in a slice of rows, whether a wavefront's share of the
// LDS holds its rings (and its partial sums) for so many column tiles of 16, and an explicit launch with that many.
constexpr int64_t kStripMaxM = 256;
constexpr int kStripWaves = 8, kStripMaxTiles = 4;
constexpr int strip_ring_bytes(int row_blocks, int tiles) { return row_blocks * 2048 + tiles * 2048 + 1024; }
constexpr bool strip_fits(int row_blocks, int tiles) {
  return strip_ring_bytes(row_blocks, tiles) * kStripWaves <= 160 * 1024 && (row_blocks + 1) / 2 * tiles * 1024 * kStripWaves <= 160 * 1024;
}
bool gemm_strip_applicable(const Problem& p);
int strip_row_blocks(int64_t m);
bool launch_gemm_strip(const Problem& p, int tiles);
template <int BITS>
bool launch_gemm_strip_bits(const Problem& p, int tiles);  // of that bit width
struct GemmPlan {
  int variant = 0, split = 1;  // tile, windows of K
  float us = 0.f, both_us = 0.f;  // on the problem's layout, on both together
  int64_t tiles = 0, bytes = 0;  // bytes of workspace
  bool shares = false;  // stream_split_shares
  float other_us = 0.f;  // on the other layout
};
GemmPlan plan_stream(const Problem& p, bool may_split);
bool split_clearly_ahead(const GemmPlan& split, const GemmPlan& whole);
GemmPlan plan_decode_stream(const Problem& p);
GemmPlan plan_strip(const Problem& p);  // `variant`: its column tiles, 0 where it does not apply (`us` is out of reach then)
bool strip_ahead(const Problem& p, const GemmPlan& strip, const GemmPlan& stream);
// What a call of 17 rows on runs, where the kernel that its family would run instead takes `other_us`.
enum StreamedChoice { kOtherKernel, kStreamedTiles, kStrips };
StreamedChoice choose_streamed(const Problem& p, const GemmPlan& strip, const GemmPlan& stream, float other_us);
float skinny_cost(const Problem& p);  // us by the cost model; out of reach where a kernel does not apply
float other_gemm_cost(const Problem& p);  // of the kernels launch_gemm takes where not the streamed one
bool gemm_direct_applicable(const Problem& p);  // K % 256 == 0, the standard group, operands below 1 GiB
int choose_gemm_direct(const Problem& p);  // the direct-weight kernel's variant for a problem that it applies to
int64_t gemm_full_round_cols(const Problem& p);  // of its variant 6
int choose_gemm_pipe(const Problem& p);
bool launch_gemm_direct(const Problem& p, int group_shift, int variant);
int launch_dequant(const Problem& p, void* wd);
// canonical -> tile-major (forward) or back; p.wq / p.scales are the source, p.y is unused
int launch_tile_weights(const Problem& p, void* wq_out, void* scales_out, bool forward);
// K and (bits, group) for which the tile-major layout is defined: int4 / group 32 with K % 256 == 0,
// int8 / group 128 with K % 128 == 0
bool tiled_layout_defined(int bits, int group, int64_t k);

// Upper bound of rows the skinny family accepts.
constexpr int64_t kSkinnyMaxM = 256;  // (above 64 rows as grid slices)

void set_error(const char* fmt, ...) __attribute__((format(printf, 1, 2)));

// Index of the current HIP device, clamped to the size of the per-device caches below.
constexpr int kMaxDevices = 64;
int current_device_slot();

// Raises a kernel's dynamic-LDS limit on the current device, once per device and kernel
// (the attribute is per device; `done` is the kernel's own flag array of kMaxDevices
// entries).  Returns false with the error set if the runtime refuses.
bool ensure_dynamic_lds(const void* kernel, int bytes, std::atomic<bool>* done);

// Compute units of the current device (cached per device).
int cu_count();

}  // namespace wq

// The packed boundary's pieces that the subgraph module (wq_module.cpp) shares.
struct mi355x_wq_callspec;
struct mi355x_wq_desc;
union mi355x_tvm_value;
namespace wq {
// The workspace that a call of `m` rows with this tail splits K on (MI355X_WQ_ACT_*), 0 where it would not; of a valid descriptor.
int64_t call_workspace_bytes(const mi355x_wq_desc* desc, int64_t m, bool tiled, int activation, bool residual);
// mi355x_wq_packed_call; when `wq_tiled` is given, a matmul reads these tile-major copies instead of
// the canonical tensors in the wq / scales slots (which are still validated and give N, K and group).
// `library_scratch`: decode matmuls go through mi355x_wq_matmul_static_ws (K split on the library's scratch array).
// `workspace`: device memory of the caller for the K split (mi355x_wq_matmul_ws); it takes precedence over the
// library's scratch array.
int packed_call_with_weights(const mi355x_wq_callspec* spec, mi355x_tvm_value* args, int* type_codes, int num_args,
                             const void* wq_tiled, const void* scales_tiled, bool library_scratch = false,
                             void* workspace = nullptr, int64_t workspace_bytes = 0);
// Forwards the recorded error to TVM's error slot when the process has one; returns -1.
int packed_fail();
}  // namespace wq
