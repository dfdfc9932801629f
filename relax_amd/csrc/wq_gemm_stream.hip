// MFMA GEMM whose operands stream through LDS: y[M,N] = x[M,K] @ dequant(Wq,S)^T, from 17 rows on and, with K split, for fewer rows
// of long K (decode_streams in wq_gemm_plan.cpp).
//
// What bounds it: with 128 rows and more per tile the matrix pipes and, on random data, the board's power (the chip clocks
// down); below that the vector instructions of the conversion (a weight is converted once per tile of rows: 8 per MFMA
// at 64 rows, 4 at 128, 2 at 256; up to six per MFMA hide behind it, measured) and, for few tiles, start and end of a launch.
//
// A workgroup owns a TM*32 x CW*TN*32 output tile.  Activations, packed weights and scales go from memory straight into LDS
// (buffer loads with the lds modifier: no registers, no stores), many stages ahead -- 60 to 110 KB in flight per CU,
// which a register-staged pipeline had no room for.  Weights and scales are staged by macro steps of 128 - 256 k, so
// that a request reads a row's whole 128-byte lines in either layout; activations by stages of 32 - 128 k.  K is an
// index of both operands, so a lane's k of a slice are chosen to be one packed word (int4) or two (int8) of its column,
// which it converts in registers to the float16 values of the CPU path, one slice ahead of the MFMAs that use them;
// the A fragments come from LDS, read once per 32 * TN columns.  K groups (G): wavefronts that share columns take
// different slices of every stage and add up at the end through LDS, in the order of the groups.
//
// Requests are sent by four wavefronts of their own (PROD = 4), so that a full address queue never holds up an MFMA; the
// 256 x 256 tile, whose accumulators take half of the register file, sends them from its four wavefronts, spread over
// the MFMAs.  Requests are counted, not tracked: every stage sends the same number (out of range once K is done), so
// "stage t + 1 has landed" is a constant s_waitcnt and one workgroup barrier per stage.
//
// Rows past M, columns past N, k past K and groups past the row's end are out-of-range buffer offsets: LDS gets zeros.
//
// Measured against the kernels it takes over from (us, weights from memory): int4 4096 x 11008 at 37 / 128 / 512 rows 24.7 /
// 34.8 / 69 -> 15.7 / 23.2 / 57, 12288 x 4096 at 64 / 256 rows 24.2 / 39.5 -> 17.0 / 32.3, int8 5120 x 13824 at 64 / 256
// rows 38.7 / 78 -> 22 / 54, 15360 x 5120 at 256 rows 73 -> 48.5; a layer of 4096 / 11008 at 2048 rows 809 -> 756 (power).
//
// Rings: what a tile has in flight decides below 128 rows.  int8 64 x 128 with 128-byte weight rows has 32 KB a macro step, and
// two of them leave one ahead: with 64-byte rows, four macro steps and two K groups 15360 x 5120 at 128 rows 37.9 -> 35.2 us,
// 27648 x 5120 at 99 71.7 -> 65.3, 5120 x 5120 at 256 29.5 -> 25.7.  int4 64 x 128 has enough in flight and gains from two K
// groups instead of four (half of the exchange at the end): 12288 x 4096 at 37 rows 20.2 -> 18.7.  Two of the tiles of 256
// columns, int8 128 x 256 and int4 256 x 256, whose ring had three stages of 64 k of activations, waited for them; six stages of 32 k in the same memory are 160 k
// ahead of the MFMAs and not 128: int8 128 x 256 256 x 15360 x 5120 84 -> 69 us (256 x 27648 x 5120 takes it now, one round for two of 128 x 128: 88 -> 79),
// int4 256 x 256 512 x 6144 x 4096 108 -> 87 (2048 x 22016 x 4096 338 -> 328, on 128 x 256 tiles 336).  256 x 128 tiles, which convert a weight half as often, are behind (int8 256 x 7680 x 5120 82 us
// against 67): twice the activations of a row's weights go through the L1.  32-row tiles for up to 32
// rows (half of the MFMAs and of the activation traffic; a remainder of up to 32 rows as well): int4 12288 x 4096 at 20 rows
// 14.0 -> 11.8, 22016 x 4096 21.1 -> 17.8, int8 27648 x 5120 at 32 rows 41.5 -> 32.7 us.  96 columns for
// matrices of more than one round of 64-column tiles and far less than one of 128-column tiles: int4 22016 x 4096 at 20 / 37
// rows (230 tiles, not 172) 18.7 / 22.5 -> 17.8 / 21.4, 18243 x 4352 at 59 0.85 of the time.  Level or behind: deeper rings
// elsewhere, reading fragments two slices ahead from LDS, one column wave, not requesting rows past M.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "wq_device.h"
#include "wq_internal.h"
#include "wq_split_share.h"

namespace wq {

namespace {
constexpr uint32_t kStreamOob = 0x80000000u;

template <int B, int E, class F>
__device__ __forceinline__ void static_for_s(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for_s<B + 1, E>(f);
  }
}

// One request of 64 lanes from a buffer straight into LDS: lane l's 16 bytes land at lds + 16 l (its two bytes, zero
// extended, at lds + 4 l); a lane whose offset is out of range writes zeros.  Written as assembly because the
// compiler would order every LDS read behind every such request in flight; the kernel orders them itself.  The
// destination is an operand in m0, which is the compiler's to write (a wait state apart from the request).  It does not see the wait
// states that a request needs behind a vector instruction which writes its scalar operands, so `lds`, `r` and `soff` have to be computed by
// scalar instructions alone (a branch on the way, or a call in the argument, and it refuses or moves one over right in front).  The built
// objects are read for that (tests/test_lds_requests_cpu.py): five wait states in every request instead cost 1 - 3 %.
__device__ __forceinline__ void dma_b128(uint32_t lds, uint32_t voff, rsrc_t r, uint32_t soff) {
  asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"{m0}"(lds), "v"(voff), "s"(r), "s"(soff) : "memory");
}
__device__ __forceinline__ void dma_u16(uint32_t lds, uint32_t voff, rsrc_t r, uint32_t soff) {
  asm volatile("s_nop 0\n\tbuffer_load_ushort %1, %2, %3 offen lds" ::"{m0}"(lds), "v"(voff), "s"(r), "s"(soff) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_dma() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
}  // namespace

// SV: scales come 16 bytes of a row at a time, eight groups, and only where a macro step begins such a piece or a window; the other
// macro steps send the same number of requests, out of range, into a place nobody reads.
template <int BITS, int TM, int TN, int CW, int G, int PROD, int KA, int KM, int NM, bool SV>
struct StreamShape {
  static constexpr int kBM = TM * 32, kBN = CW * TN * 32, kWaves = CW * G, kThreads = (kWaves + PROD) * 64;
  static constexpr int kIssuers = PROD > 0 ? PROD : kWaves;  // wavefronts that send requests
  static constexpr int kKM = KM;                       // k per macro step: what weights and scales are staged by
  static constexpr int kSPM = kKM / KA;                // activation stages per macro step
  static constexpr int kKG = KA / G;                   // k of a stage that one wavefront multiplies
  static constexpr int kSlices = kKG / 16;             // MFMA k slices of it
  static constexpr int kARow = KA * 2;                 // bytes of an activation row per stage
  static constexpr int kWRow = kKM * BITS / 8;         // packed bytes of a weight row per macro step
  static constexpr int kSub = kKM / 32;                // scales of a row per macro step (one dword per 32 k)
  static constexpr int kSRow = SV ? 16 : kSub * 4;     // bytes of a row's scales in LDS
  static constexpr int kABytes = kBM * kARow, kWBytes = kBN * kWRow, kSBytes = SV ? (kBN * 16 + 1023) / 1024 * 1024 : kBN * kSRow;
  static constexpr int kQA = kABytes / 1024, kQW = kWBytes / 1024, kQS = kSBytes / (SV ? 1024 : 256);  // requests
  static constexpr int kNA = kQA / kIssuers;                                    // ... of one of them
  static constexpr int kNW = (kQW + kIssuers - 1) / kIssuers;
  static constexpr int kNS = (kQS + kIssuers - 1) / kIssuers;
  static constexpr int kNWS = kNW + kNS;
  static constexpr bool kDummy = SV || kQW % kIssuers != 0 || kQS % kIssuers != 0;
  static constexpr int kLdsMax = 160 * 1024 - (kDummy ? 1024 : 0);
  static constexpr int kMacros = NM;                      // macro steps in the ring
  static constexpr int kRoom = (kLdsMax - kMacros * (kWBytes + kSBytes)) / kABytes;
  static constexpr int kStages = kRoom < 8 ? kRoom : 8;  // activation stages in the ring
  static constexpr int kWBase = kStages * kABytes, kSBase = kWBase + kMacros * kWBytes, kDummyBase = kSBase + kMacros * kSBytes;
  // end of the K loop: the G groups exchange partial sums, each finishing PG of the TM*4 row quads
  static constexpr int kPG = TM * 4 / G;
  static constexpr int kXPerTarget = (G - 1) * CW * kPG * TN * 1024;              // LDS bytes a target group receives
  static constexpr int kTargets = G == 1 ? 1 : (160 * 1024 / kXPerTarget < G ? 160 * 1024 / kXPerTarget : G);  // per phase
  // ... and so do the requests' wavefronts where they are whole groups that the row quads divide by: kFG groups finish kFPG quads each
  static constexpr bool kHelp = PROD > 0 && PROD % CW == 0 && TM * 4 % (G + PROD / CW) == 0;
  static constexpr int kFG = kHelp ? G + PROD / CW : G, kFPG = TM * 4 / kFG;
  static constexpr int kHelpLds = kHelp ? (G * (G - 1) + (kFG - G) * G) * CW * kFPG * TN * 1024 : 0;
  static constexpr int kLds = std::max({kDummyBase + (kDummy ? 1024 : 0), kTargets * kXPerTarget, kHelpLds});
  static_assert(kQA % kIssuers == 0 && kSlices >= 1 && kStages >= 3 && TM * 4 % G == 0 && kSPM % 2 == 0 && CW * G % 4 == 0 && kLds <= 160 * 1024, "shape");

  // Requests that may still be in flight at the top of stage t (of a macro step), where the activations of stage t + 1 and
  // the weights of stage t + kAhead have to be there.  Stage u issues the activations of stage u + kStages - 1, and a macro
  // step's first stage, before those, the weights of the macro step kMacros - 1 later.
  static constexpr int kAhead = kSlices == 1 ? 2 : 1;
  static constexpr int in_flight(int t) {
    const int t0 = t + 4 * kSPM * kMacros;  // (any macro step of the steady state)
    const int last_a = t0 + 2 - kStages;    // stage that issued the activations needed
    const int need_macro = (t0 + kAhead) / kSPM, u_w = (need_macro - kMacros + 1) * kSPM;
    int n = 0;
    for (int u = t0 - 1; u > last_a; --u) {
      n += kNA;
      if (u == u_w) return n;
      if (u % kSPM == 0) n += kNWS;
    }
    return n;
  }
};

// LDS rows hold their 16-byte chunks XOR-swizzled with the row so that sixteen consecutive rows reading the same chunk cover all
// 64 banks once.
__device__ __forceinline__ int stream_swizzle(int row, int chunks) { return (row / (16 / chunks)) % chunks; }

// The requests of one wavefront: request q of an operand fills 1 KB of its LDS area (64 dwords for scales).
template <class C, int BITS, int TN, bool TILED, bool SV>
struct StreamRequests {
  static constexpr int R = C::kIssuers;
  uint32_t av[C::kNA], wv[C::kNW], sv[C::kNS];
  int a_k, w_k, s_sub, me, k_begin, k_end, group_log2;
  int s_place = 0, s_fill = 0;  // SV: place in the ring of the last piece of scales, and whether this macro step begins one
  uint32_t lds0;
  rsrc_t rx, rw, rs;

  // LDS row r of the weights and scales is column tile r / 32 % TN of column wave r / (32 TN), lane r % 32: a matrix row such
  // that a lane ends up with TN adjacent outputs
  __device__ __forceinline__ static int matrix_row(int r) { return r / (32 * TN) * (32 * TN) + TN * (r & 31) + (TN == 1 ? 0 : (r >> 5) % TN); }

  __device__ __forceinline__ void init(int me_, int lane, int m0, int n0, int M, int N, int K, bool gated) {
    me = me_;
    const uint32_t row_bytes = (uint32_t)K * BITS / 8, groups_per_row = (uint32_t)K >> group_log2;
    {
      constexpr int CPR = C::kARow / 16, RPQ = 64 / CPR;  // chunks per row, rows per request
      static_assert(R * RPQ % 16 == 0, "the swizzle term is the same for all requests of a lane");
      const int r0 = me * RPQ + lane / CPR;
      const int chunk = (lane % CPR) ^ stream_swizzle(r0, CPR);
      a_k = chunk * 8;
#pragma unroll
      for (int i = 0; i < C::kNA; ++i) {
        const int m = m0 + r0 + i * R * RPQ;
        av[i] = m < M ? (uint32_t)m * (uint32_t)K * 2u + (uint32_t)chunk * 16u : kStreamOob;
      }
    }
    {
      constexpr int CPR = C::kWRow / 16, RPQ = 64 / CPR;
      static_assert(R * RPQ % 16 == 0, "the swizzle term is the same for all requests of a lane");
#pragma unroll
      for (int i = 0; i < C::kNW; ++i) {
        const int r = (me + i * R) * RPQ + lane / CPR;
        const int c = (lane % CPR) ^ stream_swizzle(r, CPR);
        const int n = n0 + matrix_row(r);
        w_k = c * (128 / BITS);
        if (r >= C::kBN || n >= N) {
          wv[i] = kStreamOob;
        } else if constexpr (TILED) {
          // chunk c of row n: 128-byte super step s = c / 8, chunk cc = c % 8 of it at ((n/16 * nsuper + s) * 2 + cc%2) * 1024 +
          // (cc/2 * 16 + n%16) * 16
          const uint32_t nsuper = row_bytes / 128u, cc = (uint32_t)c & 7u;
          wv[i] = ((((uint32_t)n >> 4) * nsuper + ((uint32_t)c >> 3)) * 2u + (cc & 1u)) * 1024u + ((cc >> 1) * 16u + ((uint32_t)n & 15u)) * 16u;
        } else {
          wv[i] = (uint32_t)(gated ? gated_physical_row(n, N) : n) * row_bytes + (uint32_t)c * 16u;
        }
      }
    }
    s_sub = SV ? 0 : lane % C::kSub;
    constexpr int SPR = SV ? 1 : C::kSub;  // lanes of a request that ask for a row's scales
#pragma unroll
    for (int i = 0; i < C::kNS; ++i) {
      const int r = (me + i * R) * (64 / SPR) + lane / SPR;
      const int n = n0 + matrix_row(r);
      if (r >= C::kBN || n >= N) sv[i] = kStreamOob;
      else if constexpr (TILED && BITS == 4) sv[i] = ((uint32_t)n >> 4) * (row_bytes / 128u) * 256u + (((uint32_t)s_sub >> 1) * 16u + ((uint32_t)n & 15u)) * 4u + ((uint32_t)s_sub & 1u) * 2u;
      else if constexpr (TILED) sv[i] = ((((uint32_t)n >> 4) * (row_bytes / 128u) + ((uint32_t)s_sub >> 2)) * 16u + ((uint32_t)n & 15u)) * 2u;
      else sv[i] = (uint32_t)(gated ? gated_physical_row(n, N) : n) * groups_per_row * 2u;
    }
  }

  // request P of the activations from k0 on, into the stage at LDS offset `buf`; lanes past k_end read zeros (a stage that is
  // all past k_end without a scalar offset: the hardware compares the lane's offset with the buffer's size less that one)
  template <int P>
  __device__ __forceinline__ void issue_a(int k0, uint32_t buf) const {
    dma_b128(lds0 + buf + (uint32_t)(me + P * R) * 1024u, k0 + a_k < k_end ? av[P] : kStreamOob, rx, k0 < k_end ? (uint32_t)k0 * 2u : 0u);
  }
  // request P of the weights and scales of the macro step from k0 on, into place `ring` of their rings
  template <int P>
  __device__ __forceinline__ void issue_ws(int k0, uint32_t ring) {
    if constexpr (P < C::kNW) {
      const int q = me + P * R;
      const bool mine = C::kQW % R == 0 || q < C::kQW;
      const uint32_t byte = k0 < k_end ? (uint32_t)k0 * BITS / 8u : 0u, off = TILED ? (byte >> 7) * 2048u + ((byte >> 5) & 3u) * 256u : byte;
      dma_b128(lds0 + (mine ? C::kWBase + ring * C::kWBytes + (uint32_t)q * 1024u : (uint32_t)C::kDummyBase), k0 + w_k < k_end ? wv[P] : kStreamOob, rw, off);
    } else if constexpr (SV) {
      constexpr int i = P - C::kNW;
      const int q = me + i * R;
      if constexpr (i == 0) {
        s_fill = k0 < k_end && (k0 == k_begin || (k0 & ((8 << group_log2) - 1)) == 0);
        if (k0 == k_begin) s_place = 0;
        else if (s_fill) s_place = s_place + 1 == C::kMacros ? 0 : s_place + 1;
      }
      dma_b128(lds0 + (s_fill && q < C::kQS ? C::kSBase + (uint32_t)s_place * C::kSBytes + (uint32_t)q * 1024u : (uint32_t)C::kDummyBase),
               s_fill ? sv[i] : kStreamOob, rs, s_fill ? (uint32_t)(k0 >> (group_log2 + 3)) * 16u : 0u);
    } else {
      constexpr int i = P - C::kNW;
      const int q = me + i * R;
      const bool mine = C::kQS % R == 0 || q < C::kQS;
      uint32_t v = sv[i], off = 0;
      if constexpr (TILED) off = k0 >= k_end ? 0u : BITS == 4 ? (uint32_t)k0 : (uint32_t)k0 / 4u;  // (256 bytes per 256 k, 32 per 128 k)
      else v += (uint32_t)((k0 + s_sub * 32) >> group_log2) * 2u;
      dma_u16(lds0 + (mine ? C::kSBase + ring * C::kSBytes + (uint32_t)q * 256u : (uint32_t)C::kDummyBase), k0 + s_sub * 32 < k_end ? v : kStreamOob, rs, off);
    }
  }
  // What stages -(kStages - 1) .. -1 would have issued, in their order; weights due before that first.
  template <int SPM, int KA, int KM>
  __device__ __forceinline__ void prologue() {
    auto issue_macro = [&](auto mm) __attribute__((always_inline)) {
      static_for_s<0, C::kNWS>([&](auto piece) __attribute__((always_inline)) { issue_ws<decltype(piece)::value>(k_begin + decltype(mm)::value * KM, decltype(mm)::value); });
    };
    static_for_s<0, C::kMacros - 1>([&](auto mm) __attribute__((always_inline)) {
      if constexpr ((C::kMacros - 1 - decltype(mm)::value) * SPM > C::kStages - 1) issue_macro(mm);
    });
    static_for_s<0, C::kStages - 1>([&](auto p) __attribute__((always_inline)) {
      constexpr int back = C::kStages - 1 - decltype(p)::value;  // stage -back
      if constexpr (back % SPM == 0 && back / SPM <= C::kMacros - 1) issue_macro(std::integral_constant<int, C::kMacros - 1 - back / SPM>{});
      static_for_s<0, C::kNA>([&](auto piece) __attribute__((always_inline)) { issue_a<decltype(piece)::value>(k_begin + decltype(p)::value * KA, decltype(p)::value * C::kABytes); });
    });
    wait_dma<C::in_flight(SPM - 1)>();
  }
};

// K in one piece; in windows, a workgroup each, that meet through a workspace; or the same windows one after the other in one
// workgroup -- slower, but without a workspace and with the sums in the same order, bit for bit.
enum { kWhole, kSplit, kSerial };

template <int BITS, int TM, int TN, int CW, int G, int PROD, int KA, int KM, int NM, bool TILED, int MODE, bool SV>
__global__ __launch_bounds__((CW * G + PROD) * 64, 1) void wq_gemm_stream_kernel(
    const half_t* __restrict__ x, const uint32_t* __restrict__ wq, const half_t* __restrict__ scales, int M, int N, int K,
    int shift_and_zero, int tiles_m, int tiles_n, int ksplit, half_t* y, const Epilogue ep, float* partials,
    unsigned int* counters, uint32_t* done, uint32_t launch, int looks) {
  using C = StreamShape<BITS, TM, TN, CW, G, PROD, KA, KM, NM, SV>;
  static_assert(!(TILED && SV), "tile-major scales lie as they are read");
  constexpr int BM = C::kBM, BN = C::kBN, WAVES = C::kWaves, SPM = C::kSPM, NS = C::kSlices;
  // The wavefronts that finish the tile.  One wavefront a SIMD is what the K loop has for 128 rows, and alone it is slow at the tail's chain of
  // conversions, loads and stores, so the requests' wavefronts take their share of the row quads through LDS (us): int4 333 x 10001 x 4224
  // with bias and gelu 42.8 -> 40.5, plain 333 x 10000 37.9 -> 37.0, 512 x 12288 on 128 x 256 tiles 55.9 -> 55.1; on 64 x 128 tiles, unsplit, 2 % behind.
  // (The windows of kSerial keep them busy to the end.)
  constexpr bool HELP = C::kHelp && MODE != kSerial && (TM > 2 || MODE == kSplit);
  constexpr int PG = HELP ? C::kFPG : C::kPG, FINISHERS = HELP ? WAVES + PROD : WAVES;
  constexpr bool SCATTER = MODE == kSplit && stream_split_shares(BM, BN);  // a split's windows share the finishing
  static_assert(!SCATTER || HELP, "the builds it was measured on");
  const int group_log2 = shift_and_zero & 0xFF, zero_point = (shift_and_zero >> 8) & 0xFF;  // group = 1 << group_log2 >= 32
  const bool gated = (shift_and_zero >> 16) & 1;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;

  // ---- which tile: workgroup ids go round the XCDs; give each XCD a contiguous range of the list (K windows, then
  // panels of eight column tiles, rows of the panel) so that it shares activation blocks and weight tiles in its L2
  static_assert(MODE != kSerial || PROD > 0, "the windows' requests come from wavefronts of their own");
  const int S = MODE == kWhole ? 1 : ksplit;
  const int ntiles = tiles_m * tiles_n, nblocks = MODE == kSplit ? ntiles * S : ntiles;
  const int xcd = blockIdx.x & 7, per_xcd = nblocks >> 3, extra = nblocks & 7;
  int lin = xcd * per_xcd + min(xcd, extra) + ((int)blockIdx.x >> 3);
  int ks = MODE == kSplit && S > 1 ? lin / ntiles : 0;
  const int tile_lin = lin - ks * ntiles;
  constexpr int PANEL = 8;
  const int full = tiles_n / PANEL, panel = min(tile_lin / (tiles_m * PANEL), full);
  const int width = panel < full ? PANEL : tiles_n - full * PANEL;
  const int rest = tile_lin - panel * tiles_m * PANEL;
  const int m0 = rest / width * BM, n0 = (panel * PANEL + rest % width) * BN;

  const int lane = threadIdx.x & 63, fr = lane & 31, fh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = wave / CW, cw = wave % CW;

  // macro steps [k_begin, k_end) / KM of this workgroup; lanes past k_end read zeros
  const int macros_all = (K + KM - 1) / KM, per_window = (macros_all + S - 1) / S;
  int k_begin = ks * per_window * KM, k_end = min(k_begin + per_window * KM, K);
  // (barriers of the exchange between the K groups at a window's end)
  constexpr int kExchangeBarriers = G == 1 ? 0 : 2 * ((G + C::kTargets - 1) / C::kTargets);

  float16_t acc[TM][TN];
  float4_t fin[PG][TN], total[MODE == kSerial ? PG : 1][TN];
  // HELP: where quad p of target group t from group g is in LDS, `lane`s apart
  auto handed = [&](int t, int g) __attribute__((always_inline)) {
    const int place = t < G ? t * (G - 1) + (g < t ? g : g - 1) : G * (G - 1) + (t - G) * G + g;
    return reinterpret_cast<float4_t*>(smem) + (place * CW + cw) * PG * TN * 64 + lane;
  };

  using std::integral_constant;
  StreamRequests<C, BITS, TN, TILED, SV> req;
  req.k_begin = k_begin;
  req.k_end = k_end;
  req.group_log2 = group_log2;
  req.lds0 = lds0;
  req.rx = make_rsrc(x, (uint32_t)M * (uint32_t)K * 2u);
  {
    const uint32_t n_stored = TILED ? ((uint32_t)N + 15u) / 16u * 16u : (uint32_t)N;
    req.rw = make_rsrc(wq, n_stored * ((uint32_t)K * BITS / 8));
    req.rs = make_rsrc(scales, n_stored * ((uint32_t)K >> group_log2) * 2u);
  }
  if constexpr (PROD > 0) {
    if (wave >= WAVES) {
      // producer wavefronts: requests only
      __builtin_amdgcn_s_setprio(2);
      req.init(wave - WAVES, lane, m0, n0, M, N, K, gated);
      for (;;) {
        req.template prologue<SPM, KA, KM>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        uint32_t abuf = (C::kStages - 1) * C::kABytes, ring = C::kMacros - 1;
        for (int k0 = k_begin; k0 < k_end; k0 += KM) {
          static_for_s<0, SPM>([&](auto tc) __attribute__((always_inline)) {
            constexpr int t = decltype(tc)::value;
            wait_dma<C::in_flight(t)>();
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if constexpr (t == 0) {
              static_for_s<0, C::kNWS>([&](auto piece) __attribute__((always_inline)) { req.template issue_ws<decltype(piece)::value>(k0 + (C::kMacros - 1) * KM, ring); });
              ring = ring + 1 == C::kMacros ? 0 : ring + 1;
            }
            static_for_s<0, C::kNA>([&](auto piece) __attribute__((always_inline)) { req.template issue_a<decltype(piece)::value>(k0 + (t + C::kStages - 1) * KA, abuf); });
            abuf = abuf + C::kABytes == C::kStages * C::kABytes ? 0 : abuf + C::kABytes;
          });
        }
        wait_dma<0>();
        __builtin_amdgcn_s_barrier();
        if constexpr (MODE == kSerial) {
          if (++ks == S) return;
          for (int i = 0; i < kExchangeBarriers + 1; ++i) __builtin_amdgcn_s_barrier();
          req.k_begin = k_begin = ks * per_window * KM;
          req.k_end = k_end = min(k_begin + per_window * KM, K);
        } else if constexpr (!HELP) {
          return;
        } else {
          break;
        }
      }
      if constexpr (HELP) {
        // the share of the row quads of a group that has no sums of its own
        __builtin_amdgcn_s_setprio(0);
        __syncthreads();
#pragma unroll
        for (int p = 0; p < PG; ++p)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            fin[p][j] = handed(grp, 0)[(p * TN + j) * 64];
#pragma unroll
            for (int g = 1; g < G; ++g) fin[p][j] += handed(grp, g)[(p * TN + j) * 64];
          }
      }
    }
  } else {
    req.init(wave, lane, m0, n0, M, N, K, gated);
    req.template prologue<SPM, KA, KM>();
  }

  if (!HELP || wave < WAVES) {
    // ---- LDS reads of this lane: KL contiguous k of a stage, from (grp * kKG + fh * KL) on ------------------------
    constexpr int KL = C::kKG / 2, WB = KL * BITS / 8, WL = WB > 16 ? WB / 16 : 1, WORDS = WB / 4;
    const int kl0 = grp * C::kKG + fh * KL;
    uint32_t a_rd[NS], w_rd[SPM][WL], s_rd[SPM];
#pragma unroll
    for (int kk = 0; kk < NS; ++kk) a_rd[kk] = (uint32_t)fr * C::kARow + (uint32_t)(((kl0 / 8 + kk) ^ stream_swizzle(fr, C::kARow / 16)) << 4);
    const int wrow = cw * TN * 32 + fr;  // + 32 j
#pragma unroll
    for (int t = 0; t < SPM; ++t) {
#pragma unroll
      for (int v = 0; v < WL; ++v) {
        const int byte = (t * KA + kl0) * BITS / 8 + v * 16;
        w_rd[t][v] = C::kWBase + (uint32_t)wrow * C::kWRow + (uint32_t)(((byte / 16) ^ stream_swizzle(wrow, C::kWRow / 16)) << 4) + (byte & 15);
      }
      s_rd[t] = C::kSBase + (uint32_t)(wrow * C::kSRow) + (SV ? (uint32_t)((t * KA + kl0) >> group_log2) * 2u : (uint32_t)((t * KA + kl0) / 32) * 4u);
    }

    const Q4Consts qc = make_q4_consts(zero_point);
    if constexpr (MODE == kSerial) {
#pragma unroll
      for (int p = 0; p < PG; ++p)
#pragma unroll
        for (int j = 0; j < TN; ++j) total[p][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    }

    struct Words {
      uint32_t w[TN][WORDS];
      half_t s[TN];
    };
    Words words[2];
    // (`piece`: where the macro step's scales are if they come in pieces; else by its place in the ring, as its weights)
    auto read_words = [&](Words& d, uint32_t ring, uint32_t piece, auto tt) __attribute__((always_inline)) {
      constexpr int t = decltype(tt)::value;
      const unsigned char* const wb = smem + ring * C::kWBytes;
      const unsigned char* const sb = smem + (SV ? piece : ring * C::kSBytes);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (WB >= 16) {
#pragma unroll
          for (int v = 0; v < WL; ++v) {
            const u32x4 q = *reinterpret_cast<const u32x4*>(wb + w_rd[t][v] + j * 32 * C::kWRow);
#pragma unroll
            for (int e = 0; e < 4; ++e) d.w[j][v * 4 + e] = q[e];
          }
        } else if constexpr (WB == 8) {
          const u32x2 q = *reinterpret_cast<const u32x2*>(wb + w_rd[t][0] + j * 32 * C::kWRow);
          d.w[j][0] = q[0], d.w[j][1] = q[1];
        } else {
          d.w[j][0] = *reinterpret_cast<const uint32_t*>(wb + w_rd[t][0] + j * 32 * C::kWRow);
        }
        d.s[j] = *reinterpret_cast<const half_t*>(sb + s_rd[t] + j * 32 * C::kSRow);
      }
    };
    // Weight pair PR (of four) of a lane's eight k of slice KK, column tile J, in two halves: integers with the float16
    // exponent bits in place, then the exact subtraction and the one rounding of the product with the scale.
    auto convert_front = [&](const Words& d, auto kk, auto jj, auto pp) __attribute__((always_inline)) -> uint32_t {
      constexpr int KK = decltype(kk)::value, J = decltype(jj)::value, PR = decltype(pp)::value;
      if constexpr (BITS == 4) {
        const uint32_t t = __builtin_amdgcn_perm(0u, d.w[J][KK], 0x0c000c00u | PR | (PR << 16));
        return (t & 0x00F0000Fu) | qc.magic;
      } else {
        return cvt_i8_lo<PR % 2 * 2>(d.w[J][2 * KK + PR / 2]);
      }
    };
    auto convert_back = [&](const Words& d, uint32_t f, auto kk, auto jj, auto pp) __attribute__((always_inline)) -> uint32_t {
      constexpr int KK = decltype(kk)::value, J = decltype(jj)::value, PR = decltype(pp)::value;
      if constexpr (BITS == 4) return as_u32(__builtin_elementwise_fma(as_h2(f), qc.mix_mul, -qc.mix_sub) * bcast_h2(d.s[J]));
      else return as_u32(as_h2(cvt_i8_hi<PR % 2 * 2 + 1>(f, d.w[J][2 * KK + PR / 2])) * bcast_h2(d.s[J]));
    };
    half8_t a[2][TM];
    uint32_t b[2][TN][4];
    constexpr int SLOTS = TM * TN, PAIRS = TN * 4;  // MFMAs and weight pairs of a slice

    // ---- K loop (program order is issue order: sched_barrier after every MFMA).  Slice q is multiplied while the A fragments of slice q + 1 are read and its weights converted; packed
    // words and scales are read a slice before their conversion begins.
    for (;;) {  // (a single window but for kSerial)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      // (SV: the group of a k0, which its macro step begins or lies within, is the sum of k0's and of the lane's own)
      auto in_piece = [&](int k0) __attribute__((always_inline)) { return (uint32_t)((k0 >> group_log2) & 7) * 2u; };
      uint32_t s_base = 0, s_off = SV ? in_piece(k_begin) : 0;
      read_words(words[0], 0, s_off, integral_constant<int, 0>{});
      if constexpr (NS == 1) read_words(words[1], 0, s_off, integral_constant<int, 1>{});
#pragma unroll
      for (int i = 0; i < TM; ++i) a[0][i] = *reinterpret_cast<const half8_t*>(smem + a_rd[0] + i * 32 * C::kARow);
      static_for_s<0, PAIRS>([&](auto q) __attribute__((always_inline)) {
        constexpr int j = decltype(q)::value / 4, pr = decltype(q)::value % 4;
        integral_constant<int, 0> kk;
        integral_constant<int, j> jj;
        integral_constant<int, pr> pp;
        b[0][j][pr] = convert_back(words[0], convert_front(words[0], kk, jj, pp), kk, jj, pp);
      });
      uint32_t abuf = 0, abuf_issue = (C::kStages - 1) * C::kABytes, ring = 0;
      for (int k0 = k_begin; k0 < k_end; k0 += KM) {
        const uint32_t ring_next = ring + 1 == C::kMacros ? 0 : ring + 1, ring_issue = ring == 0 ? C::kMacros - 1 : ring - 1;
        uint32_t s_next = 0;
        if constexpr (SV) {
          if (((k0 + KM) & ((8 << group_log2) - 1)) == 0) s_base = s_base + C::kSBytes == C::kMacros * C::kSBytes ? 0 : s_base + C::kSBytes;
          s_next = s_base + in_piece(k0 + KM);
        }
        static_for_s<0, SPM>([&](auto tc) __attribute__((always_inline)) {
          constexpr int t = decltype(tc)::value;
          const uint32_t abuf_next = abuf + C::kABytes == C::kStages * C::kABytes ? 0 : abuf + C::kABytes;
          if constexpr (PROD == 0) wait_dma<C::in_flight(t)>();  // (otherwise the producers have waited)
          __builtin_amdgcn_sched_barrier(0);
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
          static_for_s<0, NS>([&](auto kkc) __attribute__((always_inline)) {
            constexpr int kk = decltype(kkc)::value, q = t * NS + kk;         // slice of the macro step
            constexpr int t1 = (q + 1) / NS, kk1 = (q + 1) % NS;              // the next slice, being converted
            constexpr int t2 = (q + 2) / NS, kk2 = (q + 2) % NS;              // the one after it
            uint32_t front[PAIRS];
            static_for_s<0, SLOTS>([&](auto sc) __attribute__((always_inline)) {
              constexpr int s = decltype(sc)::value, i = s / TN, j = s % TN;
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                  a[q & 1][i], __builtin_bit_cast(half8_t, *reinterpret_cast<const u32x4*>(b[q & 1][j])), acc[i][j], 0, 0, 0);
              if constexpr (s < TM)
                a[(q + 1) & 1][s] = *reinterpret_cast<const half8_t*>(smem + (kk1 == 0 ? abuf_next : abuf) + a_rd[kk1] + s * 32 * C::kARow);
              if constexpr (s == 0 && kk2 == 0) read_words(words[t2 & 1], t2 >= SPM ? ring_next : ring, t2 >= SPM ? s_next : s_off, integral_constant<int, t2 % SPM>{});
              if constexpr (PROD == 0) {
                // requests of later stages, evenly over the slots: weights and scales first
                constexpr int slot = kk * SLOTS + s, WS = t == 0 ? C::kNWS : 0, ALL = WS + C::kNA;
                constexpr int P0 = slot * ALL / (NS * SLOTS), P1 = (slot + 1) * ALL / (NS * SLOTS);
                static_for_s<P0, P1>([&](auto pc) __attribute__((always_inline)) {
                  constexpr int P = decltype(pc)::value;
                  if constexpr (P < WS) req.template issue_ws<P>(k0 + (C::kMacros - 1) * KM, ring_issue);
                  else req.template issue_a<P - WS>(k0 + (t + C::kStages - 1) * KA, abuf_issue);
                });
              }
              constexpr int F0 = s * PAIRS / SLOTS, F1 = (s + 1) * PAIRS / SLOTS, B0 = s == 0 ? 0 : (s - 1) * PAIRS / SLOTS, B1 = s + 1 == SLOTS ? PAIRS : F0;
              static_for_s<F0, F1>([&](auto qc_) __attribute__((always_inline)) {
                constexpr int p = decltype(qc_)::value;
                front[p] = convert_front(words[t1 & 1], integral_constant<int, kk1>{}, integral_constant<int, p / 4>{}, integral_constant<int, p % 4>{});
              });
              static_for_s<B0, B1>([&](auto qc_) __attribute__((always_inline)) {
                constexpr int p = decltype(qc_)::value;
                b[(q + 1) & 1][p / 4][p % 4] = convert_back(words[t1 & 1], front[p], integral_constant<int, kk1>{}, integral_constant<int, p / 4>{}, integral_constant<int, p % 4>{});
              });
              __builtin_amdgcn_sched_barrier(0);
            });
          });
          abuf_issue = abuf;
          abuf = abuf_next;
        });
        ring = ring_next;
        s_off = s_next;
      }
      if constexpr (PROD == 0) wait_dma<0>();
      __builtin_amdgcn_s_barrier();  // the last requests (all out of range) have landed
      asm volatile("" ::: "memory");

      // ---- K groups: every group hands its partial sums of the other groups' row quads over through LDS ----------------
      auto part = [&](int pair, int j) __attribute__((always_inline)) {
        const float16_t& c = acc[pair / 4][j];
        const int v = pair % 4 * 4;
        return float4_t{c[v], c[v + 1], c[v + 2], c[v + 3]};
      };
      if constexpr (HELP) {
        static_for_s<0, C::kFG>([&](auto tt) __attribute__((always_inline)) {
          constexpr int t = decltype(tt)::value;
          if (t >= G || grp != t) {
            float4_t* const dst = handed(t, grp);
#pragma unroll
            for (int p = 0; p < PG; ++p)
#pragma unroll
              for (int j = 0; j < TN; ++j) dst[(p * TN + j) * 64] = part(t * PG + p, j);
          }
        });
        __syncthreads();
        static_for_s<0, G>([&](auto tt) __attribute__((always_inline)) {
          constexpr int t = decltype(tt)::value;
          if (grp == t) {
#pragma unroll
            for (int p = 0; p < PG; ++p)
#pragma unroll
              for (int j = 0; j < TN; ++j) {
                fin[p][j] = t == 0 ? part(p, j) : handed(t, 0)[(p * TN + j) * 64];
#pragma unroll
                for (int g = 1; g < G; ++g) fin[p][j] += g == t ? part(t * PG + p, j) : handed(t, g)[(p * TN + j) * 64];
              }
          }
        });
      } else if constexpr (G == 1) {
#pragma unroll
        for (int p = 0; p < PG; ++p)
#pragma unroll
          for (int j = 0; j < TN; ++j) fin[p][j] = part(p, j);
      } else {
        static_for_s<0, (G + C::kTargets - 1) / C::kTargets>([&](auto phase) __attribute__((always_inline)) {
          constexpr int T0 = decltype(phase)::value * C::kTargets, T1 = T0 + C::kTargets < G ? T0 + C::kTargets : G;
          __syncthreads();
          static_for_s<T0, T1>([&](auto tt) __attribute__((always_inline)) {
            constexpr int t = decltype(tt)::value;
            if (grp != t) {
              const int src = grp < t ? grp : grp - 1;
              float4_t* const dst = reinterpret_cast<float4_t*>(smem) + (((t - T0) * (G - 1) + src) * CW + cw) * PG * TN * 64 + lane;
#pragma unroll
              for (int p = 0; p < PG; ++p)
#pragma unroll
                for (int j = 0; j < TN; ++j) dst[(p * TN + j) * 64] = part(t * PG + p, j);
            }
          });
          __syncthreads();
          static_for_s<T0, T1>([&](auto tt) __attribute__((always_inline)) {
            constexpr int t = decltype(tt)::value;
            if (grp == t) {
              const float4_t* const sp = reinterpret_cast<const float4_t*>(smem) + ((t - T0) * (G - 1) * CW + cw) * PG * TN * 64 + lane;
#pragma unroll
              for (int p = 0; p < PG; ++p)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                  // (in the order of the groups, whichever of them adds: an output does not depend on its place in the tile)
                  float4_t f = t == 0 ? part(p, j) : sp[(p * TN + j) * 64];
#pragma unroll
                  for (int g = 1; g < G; ++g) f += g == t ? part(t * PG + p, j) : sp[((g < t ? g : g - 1) * CW * PG * TN + p * TN + j) * 64];
                  fin[p][j] = f;
                }
            }
          });
        });
      }

      if constexpr (MODE == kSerial) {
#pragma unroll
        for (int p = 0; p < PG; ++p)
#pragma unroll
          for (int j = 0; j < TN; ++j) total[p][j] += fin[p][j];
        if (++ks == S) break;
        __syncthreads();  // (the exchange has been read: the requests of the next window may land)
        k_begin = ks * per_window * KM, k_end = min(k_begin + per_window * KM, K);
      } else {
        break;
      }
    }
    if constexpr (MODE == kSerial) {
#pragma unroll
      for (int p = 0; p < PG; ++p)
#pragma unroll
        for (int j = 0; j < TN; ++j) fin[p][j] = total[p][j];
    }
  }

  uint32_t owned = ~0u;  // the wavefront's row quads that are this workgroup's to store
  if constexpr (MODE == kSplit) {
    // K split over workgroups: float32 partial tiles through the workspace, every output's sum in window order by one workgroup.  Partials and
    // counters are only touched by accesses performed at the memory side of the L2s (sc1).  A tile's counter has 64 bytes to
    // itself, as atomics to one line are performed one after the other (int4 20 x 4096 x 11008 in four 12.35 -> 12.05 us).
    constexpr uint32_t kWaveBytes = PG * TN * 1024u;
    const rsrc_t rp = make_rsrc(reinterpret_cast<char*>(partials) + (size_t)tile_lin * S * FINISHERS * kWaveBytes, (uint32_t)S * FINISHERS * kWaveBytes);
    const int counter = tile_lin * kStreamCounterWords;
    uint32_t* const word = reinterpret_cast<uint32_t*>(smem);
    auto live = [&](int p) __attribute__((always_inline)) { return (grp * PG + p) * 8 < M - m0; };  // (quads that begin past M are nobody's)
    auto place = [&](int q, int p, int j) __attribute__((always_inline)) { return (uint32_t)(q * FINISHERS + wave) * kWaveBytes + (p * TN + j) * 1024u; };
    if constexpr (SCATTER) {
      // Window w's workgroup finishes part w, every S-th quad: it writes the other parts, counts itself in, waits for the others, and reads its
      // part of theirs.  Bound by trips to memory: written, counted, seen, read.  Against the last to arrive finishing the whole tile, with
      // every workgroup writing all of its own (us): int8 256 x 5120 x 5120 in three 27.9 -> 25.9, 256 x 5120 x 13824 in three 49.7 -> 47.2, 99 x 5120 x
      // 13824 in six 34.7 -> 31.3, int4 256 x 4096 x 11008 in two 35.4 -> 32.5, 149 x 5760 x 6656 in two level at 27.7; 64 x 128 tiles 0.99.
      //
      // Nobody waits for long: a workgroup whose fellows are not in after `looks` looks at the counter resigns (wq_split_share.h).  Every access to the
      // counter but its return to zero is an add, so that all of them are in one order.  The addend is one that the compiler does not see: it would
      // make an add of zero a load, with which fourteen shapes take 1 % longer (int8 99 x 5120 x 13824 31.3 -> 31.8 us).
      auto part_of = [&](int w) __attribute__((always_inline)) {
        uint32_t quads = 0;
        int owner = wave * PG % S;
#pragma unroll
        for (int p = 0; p < PG; ++p) {
          quads |= owner == w ? 1u << p : 0u;
          owner = owner + 1 == S ? 0 : owner + 1;
        }
        return quads;
      };
      const uint32_t own = part_of(ks);
      auto write_parts = [&](uint32_t parts) __attribute__((always_inline)) {
        const uint32_t quads = (parts >> ks & 1u) != 0 ? own : ~own;
#pragma unroll
        for (int p = 0; p < PG; ++p)
          if ((quads >> p & 1u) != 0 && live(p)) {
#pragma unroll
            for (int j = 0; j < TN; ++j) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, fin[p][j]), rp, place(ks, p, j) + lane * 16u, 0, 0x10);
          }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
      };
      auto add = [&](uint32_t by) __attribute__((always_inline)) {
        asm volatile("" : "+v"(by));
        return __hip_atomic_fetch_add(&counters[counter], by, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      };
      auto one = [&](auto&& f) __attribute__((always_inline)) {
        if (threadIdx.x == 0) *word = f();
        __syncthreads();
        return (uint32_t)__builtin_amdgcn_readfirstlane(*word);
      };
      auto zero = [&](auto&& if_last) __attribute__((always_inline)) {
        if (threadIdx.x == 0 && if_last()) __hip_atomic_store(&counters[counter], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      };
      const uint32_t parts = split_parts(S, ks, looks, write_parts, one, add, zero);
      owned = 0;
      for (uint32_t todo = parts; todo != 0; todo &= todo - 1) owned |= part_of(__builtin_ctz(todo));
#pragma unroll
      for (int p = 0; p < PG; ++p)
        if ((owned >> p & 1u) != 0 && live(p)) {
          u32x4 win[kMaxWindows][TN];
#pragma unroll
          for (int q = 0; q < kMaxWindows; ++q)
            if (q < S && q != ks) {
#pragma unroll
              for (int j = 0; j < TN; ++j) win[q][j] = __builtin_amdgcn_raw_buffer_load_b128(rp, place(q, p, j) + lane * 16u, 0, 0x10);
            }
          float4_t sum[TN];
#pragma unroll
          for (int j = 0; j < TN; ++j) sum[j] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int q = 0; q < kMaxWindows; ++q)
            if (q < S) {
#pragma unroll
              for (int j = 0; j < TN; ++j) sum[j] += q == ks ? fin[p][j] : __builtin_bit_cast(float4_t, win[q][j]);
            }
#pragma unroll
          for (int j = 0; j < TN; ++j) fin[p][j] = sum[j];
        }
    } else {
      // The last to arrive finishes the tile, its own window still in registers: no trip to see the others arrive, which is worth more than
      // sharing the reads where a tile has few of them (64 x 64 and 32 rows: shared 0.3 - 0.6 us slower).
#pragma unroll
      for (int p = 0; p < PG; ++p)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, fin[p][j]), rp, (live(p) ? place(ks, p, j) : kStreamOob) + lane * 16u, 0, 0x10);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (threadIdx.x == 0)
        *word = __hip_atomic_fetch_add(&counters[counter], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(S - 1);
      __syncthreads();
      if (*word == 0) return;
      if (threadIdx.x == 0) __hip_atomic_store(&counters[counter], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      constexpr int PS = PG < 4 ? PG : 4, WIN = PS * TN <= 4 ? 4 : 2;  // row quads summed at a time, windows in flight
      static_for_s<0, PG / PS>([&](auto portion) __attribute__((always_inline)) {
        constexpr int p0 = decltype(portion)::value * PS;
        float4_t sum[PS][TN];
#pragma unroll
        for (int p = 0; p < PS; ++p)
#pragma unroll
          for (int j = 0; j < TN; ++j) sum[p][j] = float4_t{0.f, 0.f, 0.f, 0.f};
        for (int q = 0; q < S; q += WIN) {
          u32x4 win[WIN][PS][TN];
#pragma unroll
          for (int w = 0; w < WIN; ++w)
#pragma unroll
            for (int p = 0; p < PS; ++p)
#pragma unroll
              for (int j = 0; j < TN; ++j)
                win[w][p][j] = __builtin_amdgcn_raw_buffer_load_b128(rp, (q + w < S && q + w != ks && live(p0 + p) ? place(q + w, p0 + p, j) : kStreamOob) + lane * 16u, 0, 0x10);
#pragma unroll
          for (int w = 0; w < WIN; ++w)
#pragma unroll
            for (int p = 0; p < PS; ++p)
#pragma unroll
              for (int j = 0; j < TN; ++j) sum[p][j] += q + w == ks ? fin[p0 + p][j] : __builtin_bit_cast(float4_t, win[w][p][j]);
        }
#pragma unroll
        for (int p = 0; p < PS; ++p)
#pragma unroll
          for (int j = 0; j < TN; ++j) fin[p0 + p][j] = sum[p][j];
      });
    }
    if (done != nullptr) {
      // (a workspace of the library's: once every wavefront has read, and the counter, if it was this workgroup's to return, is back at
      // zero, the host may know)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (threadIdx.x == 0) __hip_atomic_store(&done[SCATTER ? tile_lin * S + ks : tile_lin], launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (SCATTER && owned == 0) return;
  }

  // ---- epilogue: lane holds columns n .. n + TN - 1, rows 8 (pair % 4) + 4 fh + e of row block pair / 4.  The tail's shape
  // is decided once; rows are addressed with 32-bit offsets from the first, rows past M go out of the buffer's range.
  const int n = n0 + cw * TN * 32 + TN * fr;
  const int pair0 = grp * PG;
  // (the offset of a row quad that is this workgroup's to store; around the comparison of rows, which the compiler otherwise lays out
  // differently in the unsplit builds too: int4 71 x 11776 x 2048 11.9 -> 12.3 us)
  auto kept = [&](int p, uint32_t off) __attribute__((always_inline)) {
    if constexpr (SCATTER) return (owned >> p & 1u) != 0 ? off : kStreamOob;
    else return off;
  };
  auto row_in_tile = [&](int p, int e) __attribute__((always_inline)) { return ((pair0 + p) >> 2) * 32 + ((pair0 + p) & 3) * 8 + fh * 4 + e; };
  if (gated) {
    // columns 2 c (gate) and 2 c + 1 (up) of the interleaved order: in one lane, or (one column tile) in a lane and the next
    const int rows = min(BM, M - m0), half_n = N >> 1;
    const rsrc_t ry = make_rsrc(y + (size_t)m0 * half_n, (uint32_t)rows * (uint32_t)half_n * 2u);
    const uint32_t col = (n & 1) == 0 && n + 1 < N ? (uint32_t)(n >> 1) * 2u : kStreamOob;
#pragma unroll
    for (int p = 0; p < PG; ++p)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t r = (uint32_t)row_in_tile(p, e);
        float up = fin[p][TN - 1][e];
        if constexpr (TN == 1) up = __shfl_down(up, 1);
        const half_t h = silu_mul((half_t)fin[p][0][e], (half_t)up);
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, h), ry, kept(p, r < (uint32_t)rows && col != kStreamOob ? r * (uint32_t)half_n * 2u + col : kStreamOob), 0, 0);
      }
    return;
  }
  // (in portions of four row quads, which keeps the registers of the loop's accumulators apart from the tail's)
  const int rows = min(BM, M - m0);
  const uint32_t bytes = (uint32_t)rows * (uint32_t)N * 2u, pitch = (uint32_t)N * 2u;
  const rsrc_t ry = make_rsrc(y + (size_t)m0 * N, bytes), rr = make_rsrc(ep.residual + (size_t)m0 * N, bytes), rb = make_rsrc(ep.bias, (uint32_t)N * 2u);
  constexpr int PC = PG < 4 ? PG : 4;
  const bool paired = TN == 2 && pair_store_ok(ep, y, N);
  const uint32_t col = n < N ? (uint32_t)n * 2u : kStreamOob, col1 = TN == 2 && n + 1 < N ? col + 2u : kStreamOob;
  const uint32_t base = (uint32_t)row_in_tile(0, 0) * pitch;
  // of row quad p, row e, column offset c; p = 0, e = 0 is `base`
  auto offset = [&](int p, int e, uint32_t c) __attribute__((always_inline)) {
    const int r = row_in_tile(p, e);
    return kept(p, r < rows && c != kStreamOob ? base + (uint32_t)(r - row_in_tile(0, 0)) * pitch + c : kStreamOob);
  };
  // of row quad p, row e of the pairs.  (A column beyond N: kStreamOob and less than 2^31 on top stays out of range, so that
  // only the row is compared.)
  auto pair_offset = [&](int p, int e) __attribute__((always_inline)) {
    const int r = row_in_tile(p, e);
    return kept(p, r < rows ? base + col + (uint32_t)(r - row_in_tile(0, 0)) * pitch : kStreamOob);
  };
  auto tail = [&](half2_t (&h)[PC][4], half2_t b2) __attribute__((always_inline)) {
    if (ep.bias != nullptr) {
#pragma unroll
      for (int p = 0; p < PC; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) h[p][e] = h[p][e] + b2;
    }
    if (ep.activation == 1) {
#pragma unroll
      for (int p = 0; p < PC; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int c = 0; c < 2; ++c) h[p][e][c] = h[p][e][c] > (half_t)0 ? h[p][e][c] : (half_t)0;
    }
    if (__builtin_expect(ep.activation == kActGelu, 0)) {
#pragma unroll
      for (int p = 0; p < PC; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) h[p][e] = half2_t{gelu_f16(h[p][e][0]), TN == 2 ? gelu_f16(h[p][e][1]) : (half_t)0};
    }
  };
  if (paired) {
    static_for_s<0, PG / PC>([&](auto portion) __attribute__((always_inline)) {
      constexpr int p0 = decltype(portion)::value * PC;
      half2_t h[PC][4];
#pragma unroll
      for (int p = 0; p < PC; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) h[p][e] = half2_t{(half_t)fin[p0 + p][0][e], (half_t)fin[p0 + p][TN - 1][e]};
      tail(h, ep.bias != nullptr ? as_h2(load_b32(rb, col)) : half2_t{});
      if (ep.residual != nullptr) {
        uint32_t res[PC][4];
#pragma unroll
        for (int p = 0; p < PC; ++p)
#pragma unroll
          for (int e = 0; e < 4; ++e) res[p][e] = load_b32(rr, pair_offset(p0 + p, e));
#pragma unroll
        for (int p = 0; p < PC; ++p)
#pragma unroll
          for (int e = 0; e < 4; ++e) h[p][e] = h[p][e] + as_h2(res[p][e]);
      }
#pragma unroll
      for (int p = 0; p < PC; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) __builtin_amdgcn_raw_buffer_store_b32(as_u32(h[p][e]), ry, pair_offset(p0 + p, e), 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    });
    return;
  }
  // One column per lane, an odd N or operands that are only 2-byte aligned.  Bound by the latency of what an element asks for: bias
  // and residual are requested for a portion at a time, and the tail's shape is not asked per element (int4 333 x 10001 x
  // 4224: plain 41.2 -> 38.5 us, bias and gelu 51.7 -> 40.9, residual 51.4 -> 40.8; 64 x 64 tiles, 37 x 4096 x 11008 with a residual
  // 18.0 -> 16.3).  Two columns: rows that begin on a 4-byte boundary (odd
  // N: every second one) are stored in pairs all the same, the others in pairs of the second column and the next lane's first
  // (what a half-wavefront's first and last lane have left over goes out as 2 bytes).
  const bool odd_n = N & 1, shifted0 = (reinterpret_cast<uintptr_t>(y) >> 1 & 1) ^ (odd_n & m0 & 1);
  static_for_s<0, PG / PC>([&](auto portion) __attribute__((always_inline)) {
    constexpr int p0 = decltype(portion)::value * PC;
    half2_t h[PC][4];
#pragma unroll
    for (int p = 0; p < PC; ++p)
#pragma unroll
      for (int e = 0; e < 4; ++e) h[p][e] = half2_t{(half_t)fin[p0 + p][0][e], (half_t)fin[p0 + p][TN - 1][e]};
    auto two = [](uint32_t first, uint32_t second) __attribute__((always_inline)) { return as_h2(first | second << 16); };
    tail(h, ep.bias != nullptr ? two(load_b16(rb, col), TN == 2 ? load_b16(rb, col1) : 0u) : half2_t{});
    if (ep.residual != nullptr) {
      uint32_t res[PC][4][TN];
#pragma unroll
      for (int p = 0; p < PC; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int j = 0; j < TN; ++j) res[p][e][j] = load_b16(rr, offset(p0 + p, e, j == 0 ? col : col1));
#pragma unroll
      for (int p = 0; p < PC; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) h[p][e] = h[p][e] + two(res[p][e][0], TN == 2 ? res[p][e][TN - 1] : 0u);
    }
    auto store_b16 = [&](uint32_t v, uint32_t off) __attribute__((always_inline)) { __builtin_amdgcn_raw_buffer_store_b16((uint16_t)v, ry, off, 0, 0); };
    if constexpr (TN == 1) {
#pragma unroll
      for (int p = 0; p < PC; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) store_b16(as_u32(h[p][e]), offset(p0 + p, e, col));
    } else {
#pragma unroll
      for (int p = 0; p < PC; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t v = as_u32(h[p][e]);
          if (shifted0 != (odd_n && (e & 1))) {
            const uint32_t next = (uint32_t)__shfl_down((int)v, 1);
            const bool whole = fr < 31 && n + 2 < N;
            __builtin_amdgcn_raw_buffer_store_b32(v >> 16 | next << 16, ry, offset(p0 + p, e, whole ? col1 : kStreamOob), 0, 0);
            store_b16(fr == 0 ? v : v >> 16, offset(p0 + p, e, fr == 0 ? col : whole ? kStreamOob : col1));
            // (the first lane's second column where it has no whole pair)
            if (n0 + cw * TN * 32 + 2 >= N) store_b16(v >> 16, offset(p0 + p, e, fr == 0 ? col1 : kStreamOob));
          } else {
            __builtin_amdgcn_raw_buffer_store_b32(v, ry, offset(p0 + p, e, n + 1 < N ? col : kStreamOob), 0, 0);
            if (n0 + BN >= N) store_b16(v, offset(p0 + p, e, n + 1 == N ? col : kStreamOob));
          }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
  });
}

namespace {

template <int BITS, int TM, int TN, int CW, int G, int PROD, int KA, int KM, int NM, bool TILED, int MODE, bool SV>
bool launch_stream(const Problem& p, int ksplit, const SplitSpace& space) {
  using C = StreamShape<BITS, TM, TN, CW, G, PROD, KA, KM, NM, SV>;
  const int tiles_m = (int)((p.m + C::kBM - 1) / C::kBM), tiles_n = (int)((p.n + C::kBN - 1) / C::kBN);
  static std::atomic<bool> lds_ok[kMaxDevices];
  const auto kernel = wq_gemm_stream_kernel<BITS, TM, TN, CW, G, PROD, KA, KM, NM, TILED, MODE, SV>;
  if (!ensure_dynamic_lds((const void*)kernel, C::kLds, lds_ok)) return false;
  int group_log2 = 0;
  while ((1 << group_log2) < p.group) ++group_log2;
  unsigned int* const counters = static_cast<unsigned int*>(space.base);
  float* const partials = space.base == nullptr ? nullptr : reinterpret_cast<float*>(static_cast<char*>(space.base) + kSplitCounterBytes);
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n * (MODE == kSplit ? ksplit : 1)), dim3(C::kThreads), C::kLds, p.stream,
                     (const half_t*)p.x, (const uint32_t*)p.wq, (const half_t*)p.scales, (int)p.m, (int)p.n, (int)p.k,
                     group_log2 | (p.zero_point << 8) | (p.activation == kActGated ? 1 << 16 : 0), tiles_m, tiles_n, ksplit,
                     (half_t*)p.y, Epilogue{(const half_t*)p.bias, (const half_t*)p.residual, p.activation}, partials, counters, space.done, space.launch, space.looks);
  return true;
}

// The builds a tile has.  The two largest fill the chip without a split; the running total of 128 x 128 beside its
// accumulators would not fit the registers.
enum { kWholeOnly, kWholeAndSplit, kAllBuilds, kSerialOnly };

template <int BITS, int MODE, int... SHAPE>
bool launch_stream_mode(const Problem& p, int ksplit, const SplitSpace& ws) {
  if (p.tiled) return launch_stream<BITS, SHAPE..., true, MODE, false>(p, ksplit, ws);
  constexpr int shape[] = {SHAPE...}, rows = shape[0] * 32, columns = shape[1] * shape[2] * 32;
  if constexpr (stream_pieces_built(BITS, rows, columns)) {
    if (stream_scale_pieces(p, rows, columns, shape[6])) return launch_stream<BITS, SHAPE..., false, MODE, true>(p, ksplit, ws);
  }
  return launch_stream<BITS, SHAPE..., false, MODE, false>(p, ksplit, ws);
}

template <int BITS, int BUILDS, int... SHAPE>
bool launch_stream_any(const Problem& p, int ksplit, const SplitSpace& ws) {
  if constexpr (BUILDS == kWholeAndSplit || BUILDS == kAllBuilds) {
    if (ksplit > 1 && ws.base != nullptr) return launch_stream_mode<BITS, kSplit, SHAPE...>(p, ksplit, ws);
  }
  if constexpr (BUILDS == kAllBuilds || BUILDS == kSerialOnly) {
    if (ksplit > 1) return launch_stream_mode<BITS, kSerial, SHAPE...>(p, ksplit, ws);
  }
  if constexpr (BUILDS != kSerialOnly) {
    if (ksplit == 1) return launch_stream_mode<BITS, kWhole, SHAPE...>(p, 1, ws);
  }
  return false;
}

}  // namespace

// The tiles of this object's bit width (the file is compiled once for each: WQ_STREAM_BITS).
template <int BITS>
bool launch_gemm_stream_bits(const Problem& p, int variant, int ksplit, const SplitSpace& space) {
#define WQ_STREAM(V, BUILDS, ...) \
  case V: return launch_stream_any<BITS, BUILDS, __VA_ARGS__>(p, ksplit, space);
  // 128 x 128 tiles' windows one after the other: in 64 x 128 tiles of the same K groups, stages and macro steps, which add up
  // every output in the same order
  if (variant == kStream128x128 && ksplit > 1 && space.base == nullptr)
    return launch_stream_any<BITS, kSerialOnly, 2, 2, 2, 2, 4, 64, BITS == 4 ? 256 : 128, BITS == 4 ? 3 : 4>(p, ksplit, space);
  if constexpr (BITS == 4) {
    switch (variant) {
      WQ_STREAM(kStream128x256, kWholeOnly, 4, 2, 4, 1, 4, 64, 256, 2)
      WQ_STREAM(kStream128x128, kWholeAndSplit, 4, 2, 2, 2, 4, 64, 256, 2)
      WQ_STREAM(kStream256x256, kWholeOnly, 8, 2, 4, 1, 0, 32, 128, 3)
      WQ_STREAM(kStream64x128, kAllBuilds, 2, 2, 2, 2, 4, 128, 256, 3)
      WQ_STREAM(kStream64x64, kAllBuilds, 2, 1, 2, 4, 4, 128, 256, 3)
      WQ_STREAM(kStream32x64, kAllBuilds, 1, 1, 2, 4, 4, 128, 256, 3)
      WQ_STREAM(kStream32x128, kAllBuilds, 1, 2, 2, 4, 4, 128, 256, 3)
      WQ_STREAM(kStream64x96, kWholeOnly, 2, 1, 3, 4, 4, 128, 256, 3)
      WQ_STREAM(kStream32x96, kWholeOnly, 1, 1, 3, 4, 4, 128, 256, 3)
    }
  } else {
    switch (variant) {
      WQ_STREAM(kStream128x256, kWholeOnly, 4, 2, 4, 1, 4, 32, 128, 3)
      WQ_STREAM(kStream128x128, kWholeAndSplit, 4, 2, 2, 2, 4, 64, 128, 3)
      WQ_STREAM(kStream256x256, kWholeOnly, 8, 2, 4, 1, 0, 32, 128, 2)
      WQ_STREAM(kStream64x128, kAllBuilds, 2, 2, 2, 2, 4, 64, 128, 4)
      WQ_STREAM(kStream64x64, kAllBuilds, 2, 1, 2, 4, 4, 128, 256, 3)
      WQ_STREAM(kStream32x64, kAllBuilds, 1, 1, 2, 4, 4, 128, 256, 3)
      WQ_STREAM(kStream32x128, kAllBuilds, 1, 2, 2, 4, 4, 128, 256, 3)
      WQ_STREAM(kStream64x96, kWholeOnly, 2, 1, 3, 4, 4, 128, 256, 3)
      WQ_STREAM(kStream32x96, kWholeOnly, 1, 1, 3, 4, 4, 128, 256, 3)
    }
  }
  return false;
#undef WQ_STREAM
}
template bool launch_gemm_stream_bits<WQ_STREAM_BITS>(const Problem&, int, int, const SplitSpace&);

}  // namespace wq
