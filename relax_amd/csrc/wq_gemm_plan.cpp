// Which kernel a call runs on from 17 rows on (and, at the end of the file, two rules of the decode kernel up to 16): the streamed GEMM (wq_gemm_stream.hip) with which tile and how many windows
// of K, the direct-weight GEMM (wq_gemm_direct.hip) or the register-activation kernel (wq_skinny.hip).  Host arithmetic only.
//
// Each kernel's time is a sum of terms of the problem's tiles, fitted per bit width and weight layout -- the layouts differ
// by up to a third: int8 15360 x 5120 at 512 rows takes 95.6 us streamed and 92.9 direct on canonical weights, 104.0 and 80.2
// on tile-major ones -- to 30,000 timings of 2,200 random problems (17 - 2048 rows, N 512 - 28000, four in ten no multiple of
// 256, K 1024 - 14336, weights from memory, launches back to back).  The fits are good to 3 - 8 % (streamed), 5 - 7 % (direct)
// and 8 - 10 % (register-activation).  Taking what they call the fastest costs 0.1 - 1.2 % on average against always taking
// the fastest; one table for both layouts, without the direct kernel and without the tail of odd N, cost 3 - 8 %.
#include <algorithm>

#include "../../include/mi355x_wq.h"
#include "wq_internal.h"

namespace wq {

namespace {

constexpr float kNever = 1e30f;

// (every call from 17 rows on plans, so the divisions are of 32 bits, which extents are within, and the device is asked once)
int ceil_div(int64_t a, int b) { return (int)(((uint32_t)a + (uint32_t)b - 1u) / (uint32_t)b); }

// One tile shape, in us: start + rounds of tiles * (tile start and end + 256-k steps * its loop alone on the chip + on odd N
// the tail) + steps * tiles per CU * what a full chip adds, and with K split into windows the exchange.
//
// The tail of odd N, timed on 5,000 random problems.  Streamed: rows that begin between two 4-byte boundaries; against the even N beside it,
// 8.6 us a round in 128 x 256 tiles (with a residual 10.8), 4.15 (5.0) in 128 x 128, 20 (23) in 256 x 256, 2.0 (2.3) in 64 x 128 and nothing in
// 64 x 64.  The other kernels store and read an element at a time: a plain call's 3 - 7 us a round (pipeline: none), with a
// bias 10 - 20 and with a residual 14 - 31.  A call's kernel does not depend on its tail, so their terms here are a plain call's and a
// third of what a bias adds.  Against always taking the fastest, calls of odd N lose 0.4 % (plain; tile-major 0.7), 0.4 (bias; 0.5), 0.5 (gelu;
// 0.8) and 0.4 (residual; 1.8) on 2,100 problems that were not fitted to; before, with a plain call's alone and the streamed tail's of one
// element at a time, 0.6 (0.6), 1.4 (1.9), 0.4 (0.9) and 1.8 (4.1).
struct TileCost {
  int variant, bm, bn;
  float start, tile, loop, loaded, odd, split, window, spread;
};

// (The tiles of 96 columns, fitted to 1,700 timings of up to 256 rows, are the fastest on 16400 - 24576 columns, where 64-column tiles are more than
// a round and 128-column ones much less: 17 - 64 rows 0.82 - 0.93 of the time there.  K is not split in them.)
// (int8 128 x 256: refitted with its ring of 32-k stages, 320 timings of 130 - 2048 rows, within 3 %.  int4 256 x 256 likewise, with scales in pieces where they
// run, by 1,300 timings of 321 problems of 129 - 2048 rows, odd N among them: so that it is to its neighbour 128 x 256 as measured.)
constexpr TileCost kStreamCost[2][2][9] = {
    {{  // int4, canonical
         {kStream128x256, 128, 256, 0.00f, 5.47f, 2.244f, 1.157f, 8.60f, 0.f, 0.f, 0.f},
         {kStream128x128, 128, 128, 0.00f, 5.68f, 1.212f, 0.494f, 4.15f, 4.12f, 1.383f, 0.31f},
         {kStream256x256, 256, 256, 0.00f, 8.60f, 4.459f, 2.142f, 31.2f, 0.f, 0.f, 0.f},
         {kStream64x128, 64, 128, 1.14f, 3.71f, 0.836f, 0.291f, 2.00f, 2.45f, 0.747f, 1.16f},
         {kStream64x64, 64, 64, 1.47f, 3.12f, 0.520f, 0.181f, 0.00f, 1.75f, 0.450f, 0.19f},
         {kStream32x64, 32, 64, 1.10f, 2.44f, 0.459f, 0.065f, 0.03f, 1.75f, 0.275f, 0.24f},
         {kStream32x128, 32, 128, 1.12f, 3.11f, 0.742f, 0.152f, 0.52f, 1.99f, 0.461f, 0.35f},
         {kStream64x96, 64, 96, 0.00f, 5.00f, 0.650f, 0.338f, 0.00f, 0.f, 0.f, 0.f},
         {kStream32x96, 32, 96, 1.18f, 3.16f, 0.584f, 0.146f, 0.03f, 0.f, 0.f, 0.f}},
     {  // int4, tile-major
         {kStream128x256, 128, 256, 0.00f, 6.00f, 2.483f, 1.013f, 10.16f, 0.f, 0.f, 0.f},
         {kStream128x128, 128, 128, 0.29f, 5.37f, 1.339f, 0.471f, 3.49f, 3.97f, 1.275f, 0.65f},
         {kStream256x256, 256, 256, 0.00f, 9.69f, 4.270f, 2.057f, 33.8f, 0.f, 0.f, 0.f},
         {kStream64x128, 64, 128, 1.11f, 3.78f, 0.902f, 0.262f, 1.90f, 2.52f, 0.802f, 0.53f},
         {kStream64x64, 64, 64, 1.53f, 2.96f, 0.577f, 0.176f, 0.00f, 1.86f, 0.453f, 0.06f},
         {kStream32x64, 32, 64, 1.45f, 2.23f, 0.490f, 0.069f, 0.15f, 1.62f, 0.246f, 0.36f},
         {kStream32x128, 32, 128, 1.21f, 3.22f, 0.786f, 0.108f, 0.63f, 1.96f, 0.473f, 0.22f},
         {kStream64x96, 64, 96, 1.65f, 3.01f, 0.774f, 0.284f, 0.00f, 0.f, 0.f, 0.f},
         {kStream32x96, 32, 96, 2.12f, 2.40f, 0.608f, 0.170f, 0.03f, 0.f, 0.f, 0.f}}},
    {{  // int8, canonical
         {kStream128x256, 128, 256, 1.29f, 5.25f, 2.456f, 1.368f, 8.60f, 0.f, 0.f, 0.f},
         {kStream128x128, 128, 128, 0.00f, 4.75f, 1.419f, 0.474f, 4.15f, 4.03f, 1.378f, 1.04f},
         {kStream256x256, 256, 256, 0.00f, 7.50f, 5.039f, 1.840f, 20.0f, 0.f, 0.f, 0.f},
         {kStream64x128, 64, 128, 1.79f, 1.69f, 1.201f, 0.192f, 2.00f, 2.61f, 0.798f, 1.83f},
         {kStream64x64, 64, 64, 1.79f, 2.47f, 0.608f, 0.161f, 0.00f, 1.87f, 0.479f, 0.57f},
         {kStream32x64, 32, 64, 1.43f, 2.01f, 0.519f, 0.063f, 0.03f, 1.74f, 0.324f, 0.47f},
         {kStream32x128, 32, 128, 1.21f, 2.71f, 0.907f, 0.097f, 0.52f, 1.99f, 0.458f, 1.00f},
         {kStream64x96, 64, 96, 0.31f, 4.29f, 0.754f, 0.692f, 0.00f, 0.f, 0.f, 0.f},
         {kStream32x96, 32, 96, 1.68f, 2.64f, 0.582f, 0.289f, 0.03f, 0.f, 0.f, 0.f}},
     {  // int8, tile-major
         {kStream128x256, 128, 256, 0.91f, 5.22f, 3.007f, 0.881f, 10.07f, 0.f, 0.f, 0.f},
         {kStream128x128, 128, 128, 0.00f, 6.12f, 1.392f, 0.518f, 3.27f, 3.28f, 1.206f, 0.46f},
         {kStream256x256, 256, 256, 0.00f, 9.99f, 4.983f, 1.781f, 25.92f, 0.f, 0.f, 0.f},
         {kStream64x128, 64, 128, 1.65f, 3.14f, 1.186f, 0.223f, 1.87f, 2.27f, 0.609f, 1.04f},
         {kStream64x64, 64, 64, 1.91f, 2.95f, 0.698f, 0.191f, 0.00f, 1.70f, 0.422f, 0.19f},
         {kStream32x64, 32, 64, 1.52f, 2.32f, 0.625f, 0.047f, 0.01f, 1.54f, 0.288f, 0.44f},
         {kStream32x128, 32, 128, 1.90f, 2.67f, 1.236f, 0.000f, 0.59f, 1.32f, 0.402f, 1.29f},
         {kStream64x96, 64, 96, 1.06f, 3.78f, 1.129f, 0.376f, 0.00f, 0.f, 0.f, 0.f},
         {kStream32x96, 32, 96, 1.23f, 3.34f, 0.825f, 0.138f, 0.03f, 0.f, 0.f, 0.f}}},
};

// The direct-weight kernel's 128 x 256 (variant 2), 64 x 256 (4) and 64 x 128 (5) tiles in the same terms (from 65 rows on).
constexpr TileCost kDirectCost[2][2][3] = {
    {{{2, 128, 256, 0.36f, 9.29f, 2.13f, 1.23f, 10.62f}, {4, 64, 256, 1.52f, 4.53f, 1.58f, 0.79f, 6.37f}, {5, 64, 128, 2.30f, 5.61f, 0.91f, 0.44f, 6.17f}},
     {{2, 128, 256, 0.56f, 9.34f, 2.10f, 1.10f, 10.24f}, {4, 64, 256, 1.27f, 5.18f, 1.46f, 0.62f, 5.89f}, {5, 64, 128, 1.63f, 6.66f, 0.82f, 0.34f, 5.81f}}},
    {{{2, 128, 256, 1.98f, 5.53f, 3.45f, 0.58f, 11.25f}, {4, 64, 256, 2.76f, 3.40f, 1.91f, 0.60f, 6.23f}, {5, 64, 128, 2.42f, 5.91f, 1.05f, 0.35f, 5.89f}},
     {{2, 128, 256, 0.00f, 9.64f, 2.40f, 0.93f, 10.35f}, {4, 64, 256, 3.18f, 2.34f, 1.92f, 0.62f, 6.10f}, {5, 64, 128, 2.70f, 4.59f, 1.11f, 0.33f, 6.40f}}},
};

// The LDS-staged pipeline's 256 x 128 and 128 x 128 tiles (canonical weights only; odd N hardly costs a plain call anything: int8, group
// 32, 1123 x 5165 x 1024 25.0 us against 30.1 streamed).
constexpr TileCost kPipeCost[2][2] = {
    {{1, 256, 128, 1.45f, 4.48f, 3.43f, 1.12f, 2.68f}, {2, 128, 128, 0.63f, 3.18f, 2.65f, 0.65f, 3.27f}},
    {{1, 256, 128, 0.36f, 5.60f, 3.80f, 0.97f, 2.62f}, {2, 128, 128, 1.68f, 2.30f, 2.85f, 0.77f, 3.25f}},
};

int layout_of(const Problem& p) { return p.tiled && p.choose_by_layout ? 1 : 0; }

// `tiles` of this shape on `cu` CUs, `steps` of 256 k each, in so many windows of K
float tile_cost(const TileCost& c, int64_t tiles, int steps, int windows, bool odd, int cu) {
  const float rounds = (float)(tiles <= cu ? 1 : tiles <= 2 * cu ? 2 : (tiles + cu - 1) / cu), per_cu = (float)tiles / (float)cu;
  float us = c.start + rounds * (c.tile + (float)steps * c.loop + (odd ? c.odd : 0.f)) + (float)steps * per_cu * c.loaded;
  if (windows > 1) us += c.split + (c.window * (float)windows + c.spread) * per_cu / rounds;
  return us;
}

// all `n` columns of the problem's rows, K in one piece
float tile_cost(const TileCost& c, const Problem& p, int64_t n, int cu) {
  return tile_cost(c, (int64_t)ceil_div(p.m, c.bm) * ceil_div(n, c.bn), ceil_div(p.k, 256), 1, p.n % 2 != 0, cu);
}

// The register-activation kernel: its start, a 256-k step, what every 16 rows of a slice add to a step -- for up to one row
// tile per CU, two, four and (per four) more, which are different builds -- and what they add to a launch.
struct SkinnyCost {
  struct {
    float start, step, rows;
  } by_tiles[4];
  float block;
};
constexpr SkinnyCost kSkinnyCost[2][3] = {
    {{{{1.45f, 0.106f, 0.087f}, {2.39f, 0.248f, 0.084f}, {3.20f, 0.296f, 0.186f}, {7.33f, 0.000f, 0.337f}}, 1.10f},    // int4, canonical
     {{{2.23f, 0.035f, 0.100f}, {3.29f, 0.086f, 0.115f}, {3.81f, 0.000f, 0.242f}, {8.15f, 0.222f, 0.173f}}, 0.88f},    // tile-major
     {{{1.56f, 0.000f, 0.228f}, {1.60f, 0.155f, 0.223f}, {3.01f, 0.383f, 0.226f}, {8.27f, 0.693f, 0.171f}}, 0.61f}},   // other groups
    {{{{1.80f, 0.151f, 0.099f}, {2.30f, 0.403f, 0.086f}, {3.99f, 0.881f, 0.043f}, {5.69f, 1.213f, 0.007f}}, 0.43f},    // int8
     {{{2.20f, 0.072f, 0.103f}, {2.81f, 0.237f, 0.096f}, {4.52f, 0.440f, 0.098f}, {7.55f, 0.686f, 0.052f}}, 0.38f},
     {{{1.63f, 0.053f, 0.244f}, {1.89f, 0.399f, 0.229f}, {2.61f, 1.032f, 0.172f}, {4.74f, 1.886f, 0.008f}}, 0.37f}},
};

bool standard_group(const Problem& p) { return p.group == (p.bits == 4 ? 32 : 128); }

}  // namespace

float skinny_cost(const Problem& p) {
  if (p.m > kSkinnyMaxM) return kNever;
  const int cu = cu_count(), slices = p.m > 64 ? ceil_div(p.m, 64) : 1, blocks = ceil_div(ceil_div(p.m, 16), slices);
  const int64_t tiles = (int64_t)ceil_div(p.n, 16) * slices;
  const int r = tiles <= cu ? 0 : tiles <= 2 * cu ? 1 : tiles <= 4 * cu ? 2 : 3;
  // (what the kernel's staged loads of weights and scales need, else it runs in the direct form)
  const bool staged = standard_group(p) && (p.bits == 8 || p.k % 128 == 0);
  const SkinnyCost& c = kSkinnyCost[p.bits == 8][layout_of(p) != 0 ? 1 : staged ? 0 : 2];
  const float steps = (float)p.k / 256.f * (r < 3 ? 1.f : (float)tiles / (float)(4 * cu)), rb = (float)blocks;
  return c.by_tiles[r].start + steps * (c.by_tiles[r].step + c.by_tiles[r].rows * rb) + c.block * rb;
}

// The standard groups and whole steps of K: a request for weights covers a row's whole line, one for scales 16 bytes of a row that begins
// on a 4-byte word, and no step is past a row's end.  (A workgroup's column tiles are within the matrix from its 128 columns on.)
bool gemm_strip_applicable(const Problem& p) {
  return p.m <= kStripMaxM && p.n >= 128 && p.n <= (4 << 20) && standard_group(p) && p.k % 256 == 0;
}

int strip_row_blocks(int64_t m) {
  const int slices = ceil_div(m, 64), blocks = ceil_div(ceil_div(m, slices), 8);
  return blocks < 3 ? 3 : blocks == 7 ? 8 : blocks;
}

// The strip kernel's time for one round of workgroups: start; what a block of eight rows adds, and the exchange of the sums of more than one column
// tile; per 512 of K what it costs by itself and per MFMA block of 16 rows and column tile; the same on the busiest SIMD, whose two
// wavefronts have a quarter of the steps of K between them, rounded up to a whole one, per block of rows and column tile (3840 x 1280 int4 at 57 rows has
// five steps and takes 6.3 us, with four 5.4, with eight 6.5); per megabyte of weights; and, past 4096 of K, the wavefronts' drifting apart.
// Fitted to 9,500 timings of 6,800 problems (17 - 256 rows, N 512 - 28000, K 1024 - 11000, weights from memory) within 4.4 %, and two per cent
// below them: the other kernels' tables lie between their times with weights from memory and with weights in the last-level cache.
//
// Why the line lies where these costs put it: a CU reads all of its rows' activations once per strip, so the kernel is ahead where
// one round of workgroups covers the matrix and K is short, and behind where K is long: then K split over workgroups reads a part of them.
// us before and now: int4 4096 x 4096 at 20 / 37 rows 8.1 / 10.5 -> 7.3 / 9.1, 12288 x 4096 12.1 / 14.5 -> 11.3 / 13.7; not 4096 x 11008 at
// 37 rows (15.3, here 20.9), nor more than a round.  Four column tiles in slices of rows are too few strips that read the weights twice
// (int8 7424 x 3072 at 70 rows 14.0 us, 64 x 64 streamed tiles 12.6).
namespace {
struct StripCost {
  float start, rows, exchange, stage, stage_mfma, busy_rows, busy_tiles, megabyte, drift;
};
constexpr StripCost kStripCost[2][2] = {
    {{1.976f, 0.152f, 0.142f, 0.259f, 0.027f, 0.051f, 0.043f, 0.102f, 0.087f},   // int4, canonical
     {2.369f, 0.122f, 0.159f, 0.118f, 0.025f, 0.057f, 0.037f, 0.100f, 0.011f}},  // tile-major
    {{2.279f, 0.161f, 0.087f, 0.180f, 0.032f, 0.057f, 0.067f, 0.071f, 0.030f},   // int8
     {2.177f, 0.174f, 0.087f, 0.193f, 0.029f, 0.052f, 0.066f, 0.079f, 0.000f}},
};
}  // namespace

// (every column tile costs something: the fewest with which one round covers the matrix)
GemmPlan plan_strip(const Problem& p) {
  GemmPlan none;
  none.us = none.both_us = kNever;
  if (p.m <= 16 || !gemm_strip_applicable(p)) return none;
  const int blocks = strip_row_blocks(p.m), slices = ceil_div(p.m, blocks * 8), columns = ceil_div(p.n, 16), strips = cu_count() / slices;
  const int t = strips > 0 ? ceil_div(columns, strips) : kStripMaxTiles + 1;
  if (t > (slices > 1 ? 3 : kStripMaxTiles) || !strip_fits(blocks, t)) return none;
  const int shift = p.bits == 4 ? 8 : 7, steps = (int)(p.k >> shift);
  const float rows = (float)blocks, tiles = (float)t, mfma = (float)((blocks + 1) / 2) * tiles, stages = (float)p.k / 512.f;
  const float busy = (float)((steps + 3) >> 2 << shift) / 128.f, megabytes = (float)(p.n * p.k) * (float)p.bits / 8e6f, past = std::max(0.f, stages - 8.f);
  auto cost = [&](const StripCost& c) {
    return c.start + c.rows * rows + c.exchange * tiles * (tiles - 1.f) + stages * (c.stage + c.stage_mfma * mfma) + busy * (c.busy_rows * rows + c.busy_tiles * tiles) +
           c.megabyte * megabytes + c.drift * past;
  };
  const int layout = layout_of(p);
  const float us = cost(kStripCost[p.bits == 8][layout]);
  return GemmPlan{t, 1, us, us + cost(kStripCost[p.bits == 8][1 - layout]), (int64_t)ceil_div(p.n, t * 16) * slices, 0};
}

// By both layouts' times together, as the streamed kernel's tile, so that the sums are the same on either.  Level cost up to 32 rows, 4 % to
// spare up to 64 and 7 % above: every strip reads all of its rows, so the more rows, the more it loses where they come from another XCD's
// kernel or from memory and not from its own L2.  The lines by 720 problems around them, strips against what runs otherwise, canonical weights from
// memory, activations in L2 / from memory: 17 - 32 rows up to 4 % below the line 0.95 / 0.94, above it 1.00 / 0.98; 33 - 64 rows 0.97 / 0.99 and 1.02 / 1.03;
// more rows 0.94 / 1.03 and 0.99 / 1.05 (tile-major 0.86 / 0.91 and 0.90 / 0.96; with the weights in the last-level cache, whose gain K split
// over workgroups does not have, 0.76 - 0.86).  From 4096 of K on, where both kernels' times scatter most, half a per cent more for every 512.
bool strip_ahead(const Problem& p, const GemmPlan& strip, const GemmPlan& stream) {
  const float level = p.m <= 32 ? 1.f : p.m <= 64 ? 0.96f : 0.93f;
  return strip.both_us < (level - 0.005f * std::max(0.f, (float)p.k / 512.f - 8.f)) * stream.both_us;
}

// The layouts' joint choice of the two, unless the other kernel is faster than what that would run.  (What is ahead of a split is ahead of the slower whole
// K as well, so a captured call without memory for the split runs the strips that the eager one does.)
StreamedChoice choose_streamed(const Problem& p, const GemmPlan& strip, const GemmPlan& stream, float other_us) {
  const bool ahead = strip_ahead(p, strip, stream);
  if (other_us < (ahead ? strip.us : stream.us)) return kOtherKernel;
  return ahead ? kStrips : kStreamedTiles;
}

bool gemm_direct_applicable(const Problem& p) { return p.k % 256 == 0 && standard_group(p) && gemm_pipe_applicable(p); }

// Columns of 128 x 256 tiles that fill whole rounds of the CUs where the rest, at most half a round, is worth 64-row tiles
// in a launch of its own: the last, partly filled round then takes about half as long (2048 x 22016: 1376 tiles = 5.4
// rounds of 256 -> five rounds and 192 half tiles: 372 -> 346 us when launches come with pauses, no difference when they run
// back to back for milliseconds -- the part is power limited then, and CUs that idle in a last round let the others clock
// higher; 512 x 22016: 2 - 7 % either way).  0 where that does not apply.
int64_t gemm_full_round_cols(const Problem& p) {
  const int64_t cu = cu_count(), tm128 = ceil_div(p.m, 128), tm64 = ceil_div(p.m, 64), tn = ceil_div(p.n, 256);
  const int64_t full_cols = (tm128 * tn / cu) * cu / tm128, rest_cols = tn - full_cols;
  if (p.k < 512 || full_cols < 1 || rest_cols < 1 || rest_cols * tm128 * 2 > cu || rest_cols * tm64 > cu) return 0;
  return full_cols;
}

// Measured at M = 128 .. 4096 on the Llama shapes: two K groups wherever K has room for them -- with 64-row tiles while
// 128-row tiles would leave half of the CUs without one, 64 x 128 tiles with four K groups while even those fit the CUs in
// one round, and whole rounds of 128-row tiles plus 64-row ones where that applies.
int choose_gemm_direct(const Problem& p) {
  const int64_t cu = cu_count();
  if ((int64_t)ceil_div(p.m, 64) * ceil_div(p.n, 128) <= cu && p.k >= 1024) return 5;
  const int tile = (int64_t)ceil_div(p.m, 128) * ceil_div(p.n, 256) <= cu / 2 ? 4 : 2;
  if (tile == 2 && gemm_full_round_cols(p) > 0) return 6;
  return p.k >= 512 ? tile : tile - 1;
}

int choose_gemm_pipe(const Problem& p) { return p.m >= 1024 ? 1 : 2; }

// Of the direct-weight kernel where it applies, else of the pipeline.
float other_gemm_cost(const Problem& p) {
  if (p.m <= 64 || !gemm_pipe_applicable(p)) return kNever;
  const int cu = cu_count();
  float us;
  if (gemm_direct_applicable(p)) {
    const TileCost(&c)[3] = kDirectCost[p.bits == 8][layout_of(p)];
    const int variant = choose_gemm_direct(p);
    const int64_t full = variant == 6 ? gemm_full_round_cols(p) * 256 : 0;
    // (two launches: 7 % above their sum on 106 problems)
    us = full > 0 ? 1.07f * (tile_cost(c[0], p, full, cu) + tile_cost(c[1], p, p.n - full, cu))
                  : tile_cost(c[variant == 5 ? 2 : variant > 2 ? 1 : 0], p, p.n, cu);
  } else if (!p.tiled) {
    us = tile_cost(kPipeCost[p.bits == 8][choose_gemm_pipe(p) - 1], p, p.n, cu);
  } else {
    return kNever;
  }
  // gelu is a pass of its own behind these kernels: the output read and written, a residual read, a launch
  if (p.activation == MI355X_WQ_ACT_GELU) us += 3.f + (float)(p.m * p.n) * (p.residual != nullptr ? 6.f : 4.f) / 5.1e6f;
  return us;
}

// Tile and windows by both layouts' times together, so that the streamed kernel's sums are the same on either (that costs 0.1 %
// against each layout's own choice); `us` by the problem's layout.
GemmPlan plan_stream(const Problem& p, bool may_split) {
  GemmPlan best;
  best.both_us = kNever;
  const int layout = layout_of(p);
  const int cu = cu_count(), macros = ceil_div(p.k, 256);
  const bool odd = p.n % 2 != 0;
  for (int i = 0; i < 9; ++i) {
    const TileCost &own = kStreamCost[p.bits == 8][layout][i], &other = kStreamCost[p.bits == 8][1 - layout][i];
    // (heights and widths are powers of two but for 96 columns: no division by what only the table knows)
    const int64_t tiles = (int64_t)((p.m + own.bm - 1) >> __builtin_ctz(own.bm)) * (own.bn == 96 ? ceil_div(p.n, 96) : (int)((p.n + own.bn - 1) >> __builtin_ctz(own.bn)));
    // (96 columns above 64 rows, in several row tiles, only by a clear margin: 141 x 7680 x 1536 int4, 240 of them for 180 tiles of 64 x 128, was
    // called 3 % faster and took a layer of such projections 68.9 -> 70.3 us; where it is called 6 % faster it mostly is, 0.86 - 0.91)
    // (int4 in 256 x 256 tiles by as clear a margin: ahead mostly on tile-major weights, 2048 x 22016 x 4096 335.8 -> 327.5 canonical and 346 -> 324, and behind
    // canonically where a round is not full or N odd -- at level cost 1087 x 12288 x 3840 had become 101 -> 107, 1945 x 6461 x 3072 89 -> 105.  Of the 321
    // problems its costs are by none is more than 1.2 % slower than with the costs before the shorter stages; of 91 that level cost moved to it 51 stay, at 0.998 and 0.970)
    const float spare = own.bn == 96 && p.m > 64 ? 1.05f : own.bm == 256 && p.bits == 4 ? 1.07f : 1.f;
    // a window has at least two steps of 256 k; up to an eighth more windows than CUs
    const int most = may_split && own.split > 0.f && 2 * tiles <= cu + cu / 8 && tiles <= kSplitMaxTiles / kStreamCounterWords ? std::min({kMaxWindows, (cu + cu / 8) / (int)tiles, macros}) : 1;
    for (int s = 1; s <= most; ++s) {
      const int per = s == 1 ? macros : ceil_div(macros, s);
      if (s > 1 && (per < 2 || (s - 1) * per >= macros)) continue;  // (windows that would be empty are dropped)
      const float us = tile_cost(own, tiles * s, per, s, odd, cu), other_us = tile_cost(other, tiles * s, per, s, odd, cu), both = spare * (us + other_us);
      if (both < best.both_us) {
        best = GemmPlan{own.variant, s, us, both, tiles, s > 1 ? kSplitCounterBytes + tiles * s * own.bm * own.bn * 4 : 0, stream_split_shares(own.bm, own.bn), other_us};
      }
    }
  }
  return best;
}

// Whether a call of more than 256 rows that brings no workspace splits on the library's.  Level cost is not enough: the split's costs scatter most where
// little is gained, the call without memory for it takes up to twice as long (wq_gemm_stream_host.hip), and captured it runs whole with other bits.  Ahead by 3 % and
// 1 us on both layouts (so that their sums are the same), or calls of 29 us and more, where the costs call the split 5 % dearer than it is.
// By 170 problems of 257 - 1456 rows for which plan_stream splits, weights from memory: the 130 taken 0.875 of the time whole (four are 2 - 3 % slower),
// the 40 left would be 1.012 (0.88 - 1.11); 150 others: 124 at 0.863 (none slower), 26 that would be 1.028 (up to 1.15).
bool split_clearly_ahead(const GemmPlan& split, const GemmPlan& whole) {
  if (std::min(whole.us, whole.other_us) >= 29.f) return true;
  auto ahead = [](float a, float b) { return a <= 0.97f * b && a + 1.f <= b; };
  return ahead(split.us, whole.us) && ahead(split.other_us, whole.other_us);
}

// The streamed kernel's scales in pieces of eight groups: their rows have to be whole 4-byte words (an even number of groups), and no macro step may reach
// past a row's end, where the next row's scales, not zeros, would follow.  Where a piece lasts for more than one macro step the rows'
// lines are asked for that much less often: a scale request touches as many lines as one for eight times the weights, and the L1
// has room for 32 KB of lines in flight.  us, with two bytes a request and with pieces: int8 99 x 27648 x 5120 47.6 -> 45.9,
// 256 x 15360 x 5120 / 5120 x 13824 47.0 / 49.6 -> 46.1 / 48.5; means over 2,300 problems, weights from memory and in the last-level
// cache: int8 64 x 128 tiles 0.94 / 1.01, 128 x 128 0.98 / 0.99, int4 groups of 64 and 128 0.97 - 0.99 from 64 x 128 on, 64 x 64 tiles of either 0.99 / 1.0.
// Not on 32 x 64 tiles, whose rows of scales are one request for four wavefronts that all send one: int4 groups of 64 and 128 1.03 / 1.03
// (20 x 2304 x 5632 8.8 -> 9.2 us), int8 up to 40 MB 1.0 / 1.015; above, where memory is the limit, int8 0.97 / 1.0 (20 x 14592 x 5632, 0.95), and so those have them.
// Where a piece does not last -- int4 groups of 32 in macro steps of 256 -- the lines are as many and seven of 32 requests go, which pays where
// 128 x 256 tiles fill the chip and its power is the limit (a 4096 / 11008 layer at 2048 rows 747.6 -> 737.6; 192 - 255 tiles of 256 CUs 0.988 / 0.985
// on 96 problems, more 0.985), and not where a launch waits for few tiles' requests (333 x 3712 x 4608 22.2 -> 24.0, 1183 x 1536 x 12288 58.3 -> 60.7).
bool stream_scale_pieces(const Problem& p, int rows, int columns, int macro_step) {
  if (!stream_pieces_built(p.bits, rows, columns) || p.tiled || p.k % 256 != 0 || (p.k / p.group) % 2 != 0) return false;
  if (rows == 32 && columns == 64 && p.n * p.k <= 40000000) return false;
  const int64_t tiles = (int64_t)ceil_div(p.m, rows) * ceil_div(p.n, columns);
  return 8 * p.group > macro_step || (columns == 256 && 4 * tiles >= 3 * cu_count());
}

// Up to 16 rows of canonical weights: where the streamed kernel's 32-row tiles, K split over workgroups, are ahead of the decode
// kernel and the register-activation kernel.  Those have every CU walk all of K for its 16 columns, so each stages all of
// the activations, in phases once they exceed the LDS; a split CU reads a part of them for more columns.  The lines by 9,500 timings
// (K 3072 - 60000, N 128 - 14000, 1 - 16 rows, all groups from 32 on, weights from memory; the streamed kernel's time against the other's, means).
// Where the rule takes it: 0.79 on 726 problems of up to 17000 of K, 0.72 on 1859 others of K up to 60000 and near the lines; 2 % of these
// are slower, by up to 9 %.  Activations (rows x K) from 4 - 10 % below a line to 10 % above it, by row tiles of 16 per CU:
//   up to one, int8 88000: 0.88 / 0.84, from K 9728 (0.87 - 0.94 / 0.90; below 7800 1.07); int4 110000: 0.89 / 0.84, from 10752 (0.85 / 0.79);
//   more, up to three windows of 64-column tiles on the CUs at once (N <= 5440 of 256), which divide worst among 16-row tiles, int8 80000:
//   0.91 / 0.90, int4 96000: 0.92 / 0.88, from K 8192 (0.99 / 0.89); N 5136 - 5376 like 5120 (0.83 - 0.90), beyond 1.0 - 1.05 and so
//   in the next class;
//   up to two (int8: one and a half), int8 138000: 0.87 / 0.90 and 0.97 - 1.05 at less, from K 13056 (0.95 / 0.91); int4 110000: 1.0 / 0.95, from 10752.
bool decode_streams(const Problem& p) {
  if (p.m > 16 || p.tiled || p.k < 8192 || p.group < 32) return false;
  const int64_t tiles = ceil_div(p.n, 16), cu = cu_count(), x = p.m * p.k;
  if (tiles <= cu) return p.bits == 8 ? p.k >= 9728 && x >= 88000 : p.k >= 10752 && x >= 110000;
  if (3 * ceil_div(p.n, 64) <= cu) return x >= (p.bits == 8 ? 80000 : 96000);
  if (tiles <= 2 * cu) return p.bits == 8 ? p.k >= 13056 && x >= 138000 && 2 * tiles <= 3 * cu : p.k >= 10752 && x >= 110000;
  return false;
}

// That split as one of up to 16 rows has it on any memory: within the library's scratch array, which a call on it must not exceed.
// `split` 1: the call is not the streamed kernel's.  (A workspace that the call brings, or the array, is the decode kernel's where that
// splits K too.  Means over 850 problems of the rule above that have both, this split's time on a workspace against the decode kernel's: int8
// up to a quarter of a tile per CU 1.11 - 1.20, a half 1.03 - 1.10, from there to one and a quarter 0.85 - 1.0 (5120 x 13312 at 12 / 16
// rows 20.0 / 21.1 and 18.6 / 19.1 us), int4 1.02 - 1.20 up to half a tile and level above.  Where it is ahead callers' workspaces have no
// room for it: its windows of 32 rows take up to twice the memory that they are sized for.)
GemmPlan plan_decode_stream(const Problem& p) {
  if (!decode_streams(p)) return {};
  const GemmPlan plan = plan_stream(p, true);
  return plan.bytes <= kDecodeSplitBytes ? plan : GemmPlan{};
}

// How the decode kernel reads its weights, by 23,000 timings (M 1 - 16, K 1536 - 14336, 4 - 256 MB, all group sizes and both layouts; means over
// a class of problems against a lane's own chunks, "from memory" through 0.9 GB of matrices and "kept" where one or two stay in the
// 256 MB last-level cache).
//
// Canonical int8 by pairs of lanes, whose requests cover whole lines: 10 - 20 MB from memory 0.92 - 0.97, above level, kept 0.96 - 1.0
// (12288 x 4096 at 2 rows 11.0 -> 9.9 us).  Not matrices of up to 10 MB and super steps fewer than two a wavefront, launches that are
// mostly their start, nor tiles of 8 .. 13 rows, whose vector work per byte is up to half as much again (5120 x 13824 at 4 rows
// 18.0 -> 19.0, 9472 x 3712 at 14 rows 11.6 -> 12.1).  int4, which has twice the vector work per byte, is level or behind.
//
// Whole lines that are not kept, int8 above a quarter of that cache: canonical from memory 0.92 - 0.95 (15360 x 5120 at 1 / 8 / 16 rows
// 15.8 / 17.7 / 19.9 -> 14.8 / 16.5 / 18.6, pairs 15.6 / 17.5 / 19.2), kept 0.98 - 1.03 up to 10 rows and 1.0 - 1.05 at 12 and 16 (the
// same matrix 13.8 / 15.6 / 17.3 -> 14.4 / 16.0 / 18.0, pairs 13.3 / 15.1 / 16.7); tile-major from memory 0.91 - 0.94, kept 0.96 - 1.06.
// The line stands for weights that come from memory: a matrix of 64 MB is found in the cache only by a program whose whole working set
// is below 256 MB.  int4 above a third: tile-major from memory 0.93 - 0.98, kept 1.0 - 1.04; canonical, which pays for the swap of the pairs, at
// 1 - 2 rows only -- from memory 0.92 - 0.97 (33792 x 5120 at 1 row 21.3 -> 19.1), kept 1.05 -- and not from 3 rows on: from memory 1.01 - 1.05
// (33792 x 5120 at 16 rows 27.7 -> 28.9), kept 1.08 - 1.11 (25.1 -> 28.8).  Nor canonical int4 in rounds (152064 x 4096 at 3 rows 76.2 -> 76.7).
int weight_reads(const Problem& p, int tile_rows, bool rounds) {
  const int64_t bytes = p.n * p.k * p.bits / 8;
  if (tile_rows < 14) return kReadOwn;
  if (p.bits == 4) return bytes > 85000000 && (p.tiled || (p.m <= 2 && !rounds)) ? kReadOnce : kReadOwn;
  if (bytes > 64000000) return kReadOnce;
  return !p.tiled && !rounds && bytes > 10000000 && p.k >= 2048 ? kReadPairs : kReadOwn;
}

}  // namespace wq
