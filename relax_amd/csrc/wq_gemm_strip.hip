// MFMA kernel for a batch's rows (17 - 256): y[M,N] = x[M,K] @ dequant(Wq,S)^T.
//
// What bounds it, by requests sent out of range (12288 x 4096 int4 at 37 rows, three column tiles, launches back to back; us, weights from memory /
// in the last-level cache): 13.7 / 10.7; without the activations 12.0 / 9.8, without the weights 9.7 / 9.6, without either 9.1 / 9.0, without the
// K loop 3.8 / 3.9.  So it is start, exchange and tail, then the wavefronts' own chain of requests, LDS reads, conversion and MFMAs (5.2), and
// then the CU's vector L1, which returns what all of its wavefronts ask for in order and holds 32 KB in flight: weights at what memory gives a CU
// (25 KB/us), activations behind them.  Deeper rings, wavefronts of their own for the weights' requests and another order of K in each workgroup
// are level; more steps of weights in the rings are 1 - 4 % behind, 64-byte pieces of a weight row instead of its whole lines 5 - 10 %.
//
// A workgroup owns all rows (above 64: a slice of them) of a strip of T column tiles of 16, so that one round of workgroups
// covers the matrix and every CU has the same share of it: 12288 columns are 256 strips of 48, where 64-column tiles are 192.  Its eight
// wavefronts split K and share nothing until the end: each has its own rings in LDS, filled by buffer loads with the lds modifier, and
// waits for its own requests only, without a barrier in the loop; each weight is converted once and each fragment read once, for
// T column tiles.  MFMAs are 16 x 16 x 32, so that 37 rows pay for 48 and not for 64.  The partial sums meet in LDS, in the order of the wavefronts.
//
// Measured against the kernels it takes over from, us, weights from memory: int4 4096 x 4096 at 20 / 37 rows 8.1 / 10.5 -> 7.3 / 9.1, 12288 x 4096
// 12.1 / 14.5 -> 11.3 / 13.7 (with the weights in the last-level cache 4096 x 4096 6.7 / 10.2 -> 5.3 / 6.6).  int8 by pieces of scales, which with two
// bytes a step were half of the lines that weights and scales touch: 0.94 of the time on 406 timings of 131 problems.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "wq_device.h"
#include "wq_internal.h"

namespace wq {

namespace {

template <int B, int E, class F>
__device__ __forceinline__ void static_for_p(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for_p<B + 1, E>(f);
  }
}

// Requests straight into LDS and the wait for them, as in the streamed GEMM.  The compiler does not see the wait states that a request
// needs behind a vector instruction which writes its scalar operands, so `lds`, `r` and `soff` have to be computed by scalar instructions
// alone (a branch on the way, and it refuses or moves one over right in front).  The built objects are read for that
// (tests/test_lds_requests_cpu.py): five wait states in every request instead cost 1 - 3 %.
__device__ __forceinline__ void dma_b128(uint32_t lds, uint32_t voff, rsrc_t r, uint32_t soff) {
  asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"{m0}"(lds), "v"(voff), "s"(r), "s"(soff) : "memory");
}
[[maybe_unused]] __device__ __forceinline__ void dma_u16(uint32_t lds, uint32_t voff, rsrc_t r, uint32_t soff) {
  asm volatile("s_nop 0\n\tbuffer_load_ushort %1, %2, %3 offen lds" ::"{m0}"(lds), "v"(voff), "s"(r), "s"(soff) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_dma() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
}  // namespace

// R8 blocks of 8 rows, T tiles of 16 columns.  Scales are asked for with every step's weights, but for int8 on canonical weights, whose
// rows have one of two bytes a step and a line to be touched for it: 16 bytes, eight steps, at a time.
template <int BITS, int R8, int T, bool TILED>
struct StripShape {
  static constexpr bool kPieces = BITS == 8 && !TILED;
  static constexpr int MB = (R8 + 1) / 2;                         // MFMA row blocks
  static constexpr int kStep = 1024 / BITS;                       // k of a row's 128-byte line of weights
  static constexpr int kSPS = kStep / 64;                         // stages (64 k, 128 bytes of an activation row) per step
  static constexpr int kNA = R8, kNWS = 2 * T + (kPieces ? 0 : 1);                // requests a stage / step
  static constexpr int kABytes = R8 * 1024, kSBase = T * 2048, kWBytes = kSBase + 1024;
  static constexpr int kWBase = 2 * kABytes;                      // two stages of activations in the ring
  static constexpr int kWaveBytes = std::max(kWBase + kWBytes, MB * T * 1024);  // (a wavefront's partial sums at the end)
  static constexpr int kLds = kStripWaves * kWaveBytes;
  static_assert(kWBase + kWBytes == strip_ring_bytes(R8, T) && kLds <= 160 * 1024, "shape");
  // Weights and scales of the next step are requested in a step's first stage (int8) or its first two (int4), ahead of the
  // stage's activations.
  static constexpr int kWsStages = kSPS / 2;
  static constexpr int ws_begin(int h) { return h >= kWsStages ? kNWS : h * kNWS / kWsStages; }
  static constexpr int requests(int h) { return kNA + ws_begin(h + 1) - ws_begin(h); }
};

template <int BITS, int R8, int T, bool TILED>
__global__ __launch_bounds__(kStripWaves * 64, 1) void wq_gemm_strip_kernel(
    const half_t* __restrict__ x, const uint32_t* __restrict__ wq, const half_t* __restrict__ scales, int M, int N, int K,
    int zero_and_gated, half_t* y, const Epilogue ep) {
  using C = StripShape<BITS, R8, T, TILED>;
  using std::integral_constant;
  constexpr int MB = C::MB, SPS = C::kSPS, UNITS = 2 * T;
  const int zero_point = zero_and_gated & 0xFF, gated = (zero_and_gated >> 8) & 1;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  const int lane = threadIdx.x & 63, col = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * (T * 16), m0 = blockIdx.y * (R8 * 8);

  // this wavefront's steps
  const int steps = (int)((uint32_t)K / C::kStep), per = steps / kStripWaves, more = steps % kStripWaves;
  const int count = per + (wave < more ? 1 : 0), k_begin = (wave * per + min(wave, more)) * C::kStep;
  const int k_end = k_begin + count * C::kStep;

  const uint32_t row_bytes = (uint32_t)K * BITS / 8, groups = (uint32_t)K / (BITS == 4 ? 32 : 128), nsuper = row_bytes / 128u;
  const uint32_t n_stored = TILED ? ((uint32_t)N + 15u) / 16u * 16u : (uint32_t)N;
  const rsrc_t rx = make_rsrc(x, (uint32_t)M * (uint32_t)K * 2u);
  const rsrc_t rw = make_rsrc(wq, n_stored * row_bytes);
  const rsrc_t rs = make_rsrc(scales, n_stored * groups * 2u);
  const uint32_t ring0 = lds0 + (uint32_t)wave * C::kWaveBytes;

  // ---- requests: offsets of this lane.  Request P of a 128-byte-row operand covers rows 8 P + lane / 8, chunk
  // (lane % 8) ^ (row / 2 % 8): sixteen rows reading the same chunk cover all LDS banks once.  Rows past M or N are out of the
  // buffer's range; so is, past the wavefront's k, the lane's offset.
  uint32_t av[2], wv[2], sv;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int r = e * 8 + lane / 8, chunk = (lane & 7) ^ ((r >> 1) & 7), n = n0 + r;
    av[e] = (uint32_t)r * (uint32_t)K * 2u + (uint32_t)chunk * 16u;
    if constexpr (TILED) wv[e] = ((uint32_t)n0 >> 4) * nsuper * 2048u + e * 1024u + (uint32_t)lane * 16u;
    else wv[e] = (uint32_t)(gated ? gated_physical_row(n, N) : n) * row_bytes + (uint32_t)chunk * 16u;
  }
  // (row and tile strides by shifts: a branch would leave them in vector registers)
  const uint32_t w_tile = TILED ? nsuper * 2048u : row_bytes << (4 - gated);
  if constexpr (!TILED) sv = (uint32_t)(gated ? gated_physical_row(n0 + lane, N) : n0 + lane) * groups * 2u;
  else if constexpr (BITS == 4) sv = (((uint32_t)n0 >> 4) + ((uint32_t)lane >> 4)) * nsuper * 256u + ((uint32_t)lane & 15u) * 16u;
  else sv = (((uint32_t)n0 >> 4) + ((uint32_t)lane >> 4)) * nsuper * 32u + ((uint32_t)lane & 15u) * 2u;
  // request P of the activations of the stage from k0 on, into the stage at `buf`
  auto issue_a = [&](auto pc, int k0, uint32_t buf) __attribute__((always_inline)) {
    constexpr int P = decltype(pc)::value;
    const bool in = k0 < k_end && P / 2 * 16 < M - m0;
    dma_b128(ring0 + buf + P * 1024u, in ? av[P & 1] : kOobOffset, rx, in ? (uint32_t)k0 * 2u + (uint32_t)(m0 + P / 2 * 16) * (uint32_t)K * 2u : 0u);
  };
  // request P of the weights and scales of the step from k0 on
  auto issue_ws = [&](auto pc, int k0) __attribute__((always_inline)) {
    constexpr int P = decltype(pc)::value;
    const bool in = k0 < k_end;
    if constexpr (P < 2 * T) {
      const uint32_t byte = in ? (uint32_t)k0 * BITS / 8u : 0u;
      dma_b128(ring0 + C::kWBase + P * 1024u, in ? wv[P & 1] : kOobOffset, rw, (TILED ? byte * 16u : byte) + P / 2 * w_tile);
    } else if constexpr (BITS == 4) {
      dma_b128(ring0 + C::kWBase + C::kSBase, in ? sv : kOobOffset, rs, in ? (TILED ? (uint32_t)k0 : (uint32_t)k0 / 16u) : 0u);
    } else {
      dma_u16(ring0 + C::kWBase + C::kSBase, in ? sv : kOobOffset, rs, in ? (uint32_t)k0 / 4u : 0u);
    }
  };
  // the first step's, and what the stages before the first would have issued, in their order
  // (int8, canonical: eight scales of every row from an even group on, 4-byte words)
  int s_first = 0;
  auto issue_piece = [&](int k0) __attribute__((always_inline)) {
    s_first = (k0 >> 7) & ~1;
    dma_b128(ring0 + C::kWBase + C::kSBase, sv, rs, (uint32_t)s_first * 2u);
  };
  if constexpr (C::kPieces) {
    if (count > 0) issue_piece(k_begin);
  }
  static_for_p<0, C::kNWS>([&](auto pc) __attribute__((always_inline)) { issue_ws(pc, k_begin); });
  static_for_p<0, 2>([&](auto tc) __attribute__((always_inline)) {
    static_for_p<0, C::kNA>([&](auto pc) __attribute__((always_inline)) { issue_a(pc, k_begin + decltype(tc)::value * 64, decltype(tc)::value * C::kABytes); });
  });

  // what the tail needs of bias and residual (nothing of an absent one: an empty buffer), a trip to memory that would stand alone at the end
  constexpr int QUADS = MB * T, MINE = (QUADS + kStripWaves - 1) / kStripWaves;  // a wavefront's share of the 16 x 16 tiles
  const int m_end = min(M, m0 + R8 * 8);
  const uint32_t pitch = (uint32_t)(gated ? N >> 1 : N) * 2u;
  auto element = [&](int i, int e) __attribute__((always_inline)) {  // offset of row e of four in this lane's column of the wavefront's i-th tile
    const int q = wave + i * kStripWaves, n = n0 + q % T * 16 + col, m = m0 + q / T * 16 + kq * 4 + e;
    const bool in = (q < QUADS) & (n < N) & (m < m_end);  // (not a chain of branches, with a wait at each)
    return in ? (uint32_t)m * pitch + (uint32_t)n * 2u : kOobOffset;
  };
  uint32_t res[MINE][4], bias[MINE];
  {
    const rsrc_t rr = make_rsrc(ep.residual, ep.residual != nullptr ? (uint32_t)M * pitch : 0u), rb = make_rsrc(ep.bias, ep.bias != nullptr ? (uint32_t)N * 2u : 0u);
#pragma unroll
    for (int i = 0; i < MINE; ++i) {
      bias[i] = load_b16(rb, (uint32_t)(n0 + (wave + i * kStripWaves) % T * 16 + col) * 2u);
#pragma unroll
      for (int e = 0; e < 4; ++e) res[i][e] = load_b16(rr, element(i, e));
    }
  }

  // ---- LDS reads of this lane: 16 k of a stage, from 16 kq on ---------------------------------------------------------
  const unsigned char* const my = smem + wave * C::kWaveBytes;
  constexpr int WORDS = BITS == 4 ? 2 : 4;  // packed words of a tile's 16 k
  uint32_t a_rd[2], w_rd[SPS];
#pragma unroll
  for (int j = 0; j < 2; ++j) a_rd[j] = (uint32_t)(col * 128 + (((kq * 2 + j) ^ ((col >> 1) & 7)) << 4));
#pragma unroll
  for (int h = 0; h < SPS; ++h) {
    const int chunk = BITS == 4 ? h * 2 + (kq >> 1) : h * 4 + kq, inner = BITS == 4 ? (kq & 1) * 8 : 0;
    w_rd[h] = (TILED ? (chunk & 1) * 1024 + ((chunk >> 1) * 16 + col) * 16 : col * 128 + ((chunk ^ ((col >> 1) & 7)) << 4)) + inner;
  }
  const uint32_t s_rd = C::kSBase + (TILED ? col * 4 : col * 16);
  const uint32_t s_shift = BITS == 4 ? (kq >> 1) * 16 : 0;

  const Q4Consts qc = make_q4_consts(zero_point);
  float4_t acc[MB][T];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

  half8_t a[2][2][MB];  // of this stage and the next: k half, row block
  uint32_t words[SPS][T][WORDS], sc[T][4];  // of the step
  uint32_t b[2][4];     // converted weights of this unit and the next: unit q is column tile q % T of k half q / T
  auto read_a = [&](auto to) __attribute__((always_inline)) {
    constexpr int h = decltype(to)::value;  // of two: place in the ring and in the registers
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < MB; ++i) a[h][j][i] = *reinterpret_cast<const half8_t*>(my + h * C::kABytes + a_rd[j] + i * 2048);
  };
  auto read_step = [&](int k0) __attribute__((always_inline)) {
    const unsigned char* const wb = my + C::kWBase;
#pragma unroll
    for (int j = 0; j < T; ++j) {
#pragma unroll
      for (int h = 0; h < SPS; ++h) {
        if constexpr (BITS == 4) {
          const u32x2 q = *reinterpret_cast<const u32x2*>(wb + w_rd[h] + j * 2048);
          words[h][j][0] = q[0], words[h][j][1] = q[1];
        } else {
          const u32x4 q = *reinterpret_cast<const u32x4*>(wb + w_rd[h] + j * 2048);
#pragma unroll
          for (int e = 0; e < 4; ++e) words[h][j][e] = q[e];
        }
      }
      if constexpr (BITS == 4 && TILED) {
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[j][e] = *reinterpret_cast<const uint32_t*>(wb + s_rd + j * 256 + e * 64);
      } else if constexpr (BITS == 4) {
        const u32x4 q = *reinterpret_cast<const u32x4*>(wb + s_rd + j * 256);
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[j][e] = q[e];
      } else {
        sc[j][0] = *reinterpret_cast<const uint16_t*>(C::kPieces ? wb + s_rd + j * 256 + ((k0 >> 7) - s_first) * 2 : wb + s_rd + j * 64);
      }
    }
  };
  // weight pair PR (of four) of unit Q of stage H
  auto convert = [&](auto hc, auto qc_, auto pc) __attribute__((always_inline)) -> uint32_t {
    constexpr int H = decltype(hc)::value, Q = decltype(qc_)::value, PR = decltype(pc)::value, J = Q % T, KH = Q / T;
    const half2_t s2 = bcast_h2(__builtin_bit_cast(half_t, (uint16_t)(BITS == 4 ? sc[J][H] >> s_shift : sc[J][0])));
    if constexpr (BITS == 4) {
      const uint32_t t = __builtin_amdgcn_perm(0u, words[H][J][KH], 0x0c000c00u | PR | (PR << 16));
      return as_u32(__builtin_elementwise_fma(as_h2(and_or(t, 0x00F0000Fu, qc.magic)), qc.mix_mul, -qc.mix_sub) * s2);
    } else {
      const uint32_t w = words[H][J][KH * 2 + PR / 2];
      return as_u32(as_h2(cvt_i8_hi<PR % 2 * 2 + 1>(cvt_i8_lo<PR % 2 * 2>(w), w)) * s2);
    }
  };

  wait_dma<C::kNA>();
  read_step(k_begin);
  read_a(integral_constant<int, 0>{});
  static_for_p<0, 4>([&](auto pc) __attribute__((always_inline)) { b[0][decltype(pc)::value] = convert(integral_constant<int, 0>{}, integral_constant<int, 0>{}, pc); });
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);

  // ---- K loop (program order is issue order: sched_barrier after every MFMA).  A stage multiplies what has been read, sends the
  // requests of later ones over its MFMAs, and before its last unit waits for and reads the next stage's operands.
  for (int k0 = k_begin; k0 < k_end; k0 += C::kStep) {
    if constexpr (C::kPieces) {
      // (not among the requests that are counted: where it is sent, the first wait is for it as well)
      if (k0 + C::kStep < k_end && ((k0 + C::kStep) >> 7) - s_first > 7) issue_piece(k0 + C::kStep);
    }
    static_for_p<0, SPS>([&](auto hc) __attribute__((always_inline)) {
      constexpr int h = decltype(hc)::value, h1 = (h + 1) % SPS;
      static_for_p<0, UNITS>([&](auto qc_) __attribute__((always_inline)) {
        constexpr int q = decltype(qc_)::value;
        if constexpr (q == UNITS - 1) {
          wait_dma<C::requests(h)>();
          read_a(integral_constant<int, (h + 1) & 1>{});
          if constexpr (h1 == 0) read_step(k0 + C::kStep);
          __builtin_amdgcn_sched_barrier(0);
        }
        static_for_p<0, MB>([&](auto ic) __attribute__((always_inline)) {
          constexpr int i = decltype(ic)::value;
          acc[i][q % T] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[h & 1][q / T][i], __builtin_bit_cast(half8_t, *reinterpret_cast<const u32x4*>(b[q & 1])),
                                                                  acc[i][q % T], 0, 0, 0);
          if constexpr (q < UNITS - 1) {
            // requests, evenly over the MFMAs of all units but the last: weights and scales first
            constexpr int slot = q * MB + i, SLOTS = (UNITS - 1) * MB, WS = C::ws_begin(h + 1) - C::ws_begin(h), ALL = WS + C::kNA;
            static_for_p<slot * ALL / SLOTS, (slot + 1) * ALL / SLOTS>([&](auto pc) __attribute__((always_inline)) {
              constexpr int P = decltype(pc)::value;
              if constexpr (P < WS) issue_ws(integral_constant<int, C::ws_begin(h) + P>{}, k0 + C::kStep);
              else issue_a(integral_constant<int, P - WS>{}, k0 + (h + 2) * 64, (h & 1) * C::kABytes);
            });
            static_for_p<i * 4 / MB, (i + 1) * 4 / MB>([&](auto pc) __attribute__((always_inline)) {
              b[(q + 1) & 1][decltype(pc)::value] = convert(hc, integral_constant<int, q + 1>{}, pc);
            });
          } else {
            static_for_p<i * 4 / MB, (i + 1) * 4 / MB>([&](auto pc) __attribute__((always_inline)) {
              b[(q + 1) & 1][decltype(pc)::value] = convert(integral_constant<int, h1>{}, integral_constant<int, 0>{}, pc);
            });
          }
          __builtin_amdgcn_sched_barrier(0);
        });
      });
      // (what has been read may be written again)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    });
  }

  // ---- the wavefronts' sums, in their order ---------------------------------------------------------------------
  wait_dma<0>();  // (the last requests, all out of range, have landed)
  {
    float4_t* const dst = reinterpret_cast<float4_t*>(smem + wave * C::kWaveBytes) + lane;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < T; ++j) dst[(i * T + j) * 64] = acc[i][j];
  }
  __syncthreads();
  const rsrc_t ry = make_rsrc(y, (uint32_t)M * pitch);
  auto as_half = [](uint32_t v) __attribute__((always_inline)) { return __builtin_bit_cast(half_t, (uint16_t)v); };
#pragma unroll
  for (int i = 0; i < MINE; ++i) {
    const int q = wave + i * kStripWaves;
    if (q >= QUADS) break;
    float4_t f = *(reinterpret_cast<const float4_t*>(smem) + q * 64 + lane);
#pragma unroll
    for (int g = 1; g < kStripWaves; ++g) f += *(reinterpret_cast<const float4_t*>(smem + g * C::kWaveBytes) + q * 64 + lane);
    half_t h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = (half_t)f[e];
    if (gated) {
      // columns 2 c (gate) and 2 c + 1 (up) of the interleaved order are in a lane and the next
      const int n = n0 + q % T * 16 + col;
      const uint32_t c = (n & 1) == 0 && n + 1 < N ? (uint32_t)(n >> 1) * 2u : kOobOffset;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + q / T * 16 + kq * 4 + e;
        const half_t t = silu_mul(h[e], (half_t)__shfl_down(f[e], 1));
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, t), ry, m < m_end && c != kOobOffset ? (uint32_t)m * pitch + c : kOobOffset, 0, 0);
      }
      continue;
    }
    if (ep.bias != nullptr) {
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = h[e] + as_half(bias[i]);
    }
    if (ep.activation == 1) {
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = h[e] > (half_t)0 ? h[e] : (half_t)0;
    }
    if (__builtin_expect(ep.activation == kActGelu, 0)) {
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = gelu_f16(h[e]);
    }
    if (ep.residual != nullptr) {
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = h[e] + as_half(res[i][e]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, h[e]), ry, element(i, e), 0, 0);
  }
}

namespace {

template <int BITS, int R8, int T, bool TILED>
bool launch_strip(const Problem& p) {
  using C = StripShape<BITS, R8, T, TILED>;
  static std::atomic<bool> lds_ok[kMaxDevices];
  const auto kernel = wq_gemm_strip_kernel<BITS, R8, T, TILED>;
  if (!ensure_dynamic_lds((const void*)kernel, C::kLds, lds_ok)) return false;
  const dim3 grid((unsigned)((p.n + T * 16 - 1) / (T * 16)), (unsigned)((p.m + R8 * 8 - 1) / (R8 * 8)));
  hipLaunchKernelGGL(kernel, grid, dim3(kStripWaves * 64), C::kLds, p.stream, (const half_t*)p.x,
                     (const uint32_t*)p.wq, (const half_t*)p.scales, (int)p.m, (int)p.n, (int)p.k,
                     p.zero_point | (p.activation == kActGated ? 1 << 8 : 0), (half_t*)p.y,
                     Epilogue{(const half_t*)p.bias, (const half_t*)p.residual, p.activation});
  return true;
}

template <int BITS, int R8, int T>
bool launch_strip_layout(const Problem& p) {
  if constexpr (strip_fits(R8, T)) return p.tiled ? launch_strip<BITS, R8, T, true>(p) : launch_strip<BITS, R8, T, false>(p);
  return false;
}

template <int BITS, int R8>
bool launch_strip_tiles(const Problem& p, int tiles) {
  switch (tiles) {
    case 1: return launch_strip_layout<BITS, R8, 1>(p);
    case 2: return launch_strip_layout<BITS, R8, 2>(p);
    case 3: return launch_strip_layout<BITS, R8, 3>(p);
    case 4: return launch_strip_layout<BITS, R8, 4>(p);
  }
  return false;
}

}  // namespace

// (rows above 64 in slices of equal height, which read the weights once each)
template <int BITS>
bool launch_gemm_strip_bits(const Problem& p, int tiles) {
  switch (strip_row_blocks(p.m)) {
    case 3: return launch_strip_tiles<BITS, 3>(p, tiles);
    case 4: return launch_strip_tiles<BITS, 4>(p, tiles);
    case 5: return launch_strip_tiles<BITS, 5>(p, tiles);
    case 6: return launch_strip_tiles<BITS, 6>(p, tiles);
    case 8: return launch_strip_tiles<BITS, 8>(p, tiles);
  }
  return false;
}
template bool launch_gemm_strip_bits<WQ_STRIP_BITS>(const Problem&, int);

}  // namespace wq
