// Per-shape tile selection: closed-form rules of (kind, m, n, k, dtype) for a 256-CU, 8-XCD MI355X.
// Host code only; no timing and no device queries, so the answer is the same at load time and at run time.
#include <algorithm>
#include <atomic>
#include <cmath>

#include "fp8_stream.h"
#include "ksq_common.h"
#include "tile_select.h"

namespace ksq {

static constexpr int kNumCU = 256;

// ksq_set_small_problem_rule: 1 (default) lets small problems of more than 32 rows run the decode-form kernels
static std::atomic<int> g_small_problem_rule{1};

// Split-K wavefront kernel (decode regime, HBM-bound).  Measured on MI355X the kernel runs fastest with few, long
// lived wavefronts, each streaming a deep ring of loads, and with every workgroup resident from the first cycle:
// - 4 wavefronts per workgroup, wavefront w taking every 4th k-tile;
// - NT, the column tiles a wavefront streams per k-tile, as wide as the register file allows (8 for one 16-row tile
//   of x, 4 for two) while the grid still has about one workgroup per CU: the x fragments and the sum-of-x MFMA are
//   shared by the NT tiles, which also divides the x traffic out of L2 by NT.
// Dense form only: with a long K and few columns (k >= 2n: down / o projections) the grid-fill rule ends at narrow
// workgroups, every one of which fetches all of x - more bytes out of the L2 than the weights out of HBM once there are
// several rows.  Then 4 column tiles share the x fragments and K is cut over 2..8 workgroups to bring the workgroup
// count back to 160 or more (fp32 partial sums through the workspace, one small second pass).  The same helps when a
// wavefront's share of K is very long (k > 16384).  Measured on MI355X, e.g. n=4096 k=14336 m=32: 28 -> 16 us.
SplitKChoice select_splitk(size_t m, size_t n, size_t k) {
  const int mt = m <= 16 ? 1 : 2;
  const size_t m_blocks = div_up(m, 16 * mt);
  SplitKChoice c = select_splitk_blocks(mt, m_blocks, n, k);
  const size_t strips = n / 16;
  // several row blocks, and four column tiles per workgroup would put a second workgroup on some CUs only (those then
  // finish last): eight column tiles when that still leaves half the CUs a workgroup (n = k = 5120 at 128 rows)
  if (m_blocks >= 2 && c.nt == 4 && strips % 8 == 0 && strips / 4 * m_blocks > static_cast<size_t>(kNumCU) &&
      strips / 8 * m_blocks >= static_cast<size_t>(kNumCU) / 2)
    c.nt = 8;
  if (strips % 4 == 0 && c.nt < 4) {
    const size_t rows = m < static_cast<size_t>(16 * mt) ? m : static_cast<size_t>(16 * mt);
    const size_t x_bytes = rows * k * 2 * (strips / c.nt) * m_blocks;  // what all workgroups together read of x
    // K the long side: whenever x outweighs the weights.  Otherwise from 48 MB of x re-reads: below that the second
    // pass costs more than the traffic it saves (n = k = 5120: 16 tokens 13.8 -> 9.4 us, 32 tokens 22.1 -> 12.6 us;
    // n = k = 4096 at 8 tokens, 17 MB of re-reads, would go 5.5 -> 7.0 us)
    const bool long_k = k >= 2 * n && (x_bytes > k * n / 2 || k > 16384);
    const bool heavy_x = x_bytes >= (size_t(48) << 20);
    if (m_blocks >= 2 && !long_k && heavy_x) {
      // several row blocks: four column tiles with x through LDS (below) rather than a cut along K - the blocks already
      // fill the chip (n = k = 5120 at 64 rows: 19.2 -> 12 us; n = k = 4096: 10.7 -> 10.0 us)
      c.nt = 4;
    } else if (long_k || heavy_x) {
      int parts = 2;
      while (parts < 8 && strips / 4 * m_blocks * parts < 160) parts *= 2;
      while (parts > 1 && k / 128 / parts < 8) parts /= 2;
      if (parts > 1) {
        c.nt = 4;
        c.parts = parts;
      }
    }
  }
  // x through LDS (group 128 only; the caller falls back to the register form otherwise).  Measured on MI355X:
  // - 17..32 rows: the x fragments are twice the weights' bytes, and fetched as 64-byte pieces of 32 rows they cost
  //   more than the weights (n = 25600, k = 5120: 27.4 -> 21.7 us; n = 14336, k = 4096: 12.8 -> 11.5 us);
  // - up to 16 rows: pays from about 48 MB of weights (n = 57344, k = 8192: 1 row 41.9 -> 40.7 us, 16 rows
  //   47.8 -> 46.3 us; n = 25600, k = 5120 at 16 rows 15.9 -> 15.0 us), not below (n = 14336, k = 4096 at 8 rows:
  //   7.9 us in registers, 8.4 us through LDS), and with up to 8 rows four column tiles per wavefront beat eight
  //   (n = 57344, k = 8192, 1 row: 40.7 against 43.1 us).
  // - K cut over workgroups, 17 rows and more: x outweighs the weights there by construction (n = 4096, k = 14336: 20 rows
  //   13.2 -> 12.9 us, 32 rows 15.8 -> 14.3..15.2, 64 rows 21.6 -> 19.0; n = k = 5120 at 32 rows
  //   12.7 -> 11.6; n = 5120, k = 25600 at 32 rows 34.4 -> 29.0; n = 2048, k = 8192 at 32 rows 11.5 -> 11.0).  Eight
  //   wavefronts are one workgroup per CU where the register form holds two, so with more workgroups than CUs a second
  //   round begins and takes back what the traffic gave (n = 2112, k = 17024, 264 workgroups: 17 rows 16.6 -> 18.2 us,
  //   26 rows 18.1 -> 18.9; n = 4544, k = 9600, 284: 20 rows 17.9 -> 18.9) until a workgroup has rows and k-tiles enough
  //   (32 rows: n = 2112 19.4 -> 19.4, n = 4544 20.6 -> 20.3, n = 4992, k = 20480 30.9 -> 28.0; n = 2432, k = 9600 at 160 rows
  //   30.3 -> 26.6; n = 1600, k = 5760 at 90 rows, 12 k-tiles a part: 15.8 -> 16.3).
  //   With fewer than 32 rows a part of 9 to 11 k-tiles stays there too: two turns of eight wavefronts, the second one
  //   nearly empty, against three turns of four (n = 1024, 64 workgroups, 9 k-tiles: 17 rows 8.2 -> 8.5 us, 24 rows 8.9 -> 9.2,
  //   32 rows 9.5 -> 9.5; 10 and 11 at 32 rows 9.6 -> 9.4, 9.8 -> 9.5; 8 and 12 at 24 rows 7.8 -> 7.6, 9.4 -> 9.2).
  if (c.parts > 1 && mt == 2) {
    const size_t kt = div_up(k / 128, c.parts);
    const bool resident = strips / 4 * m_blocks * c.parts <= static_cast<size_t>(kNumCU);
    const bool empty_turn = m < 32 && kt > 8 && kt < 12;
    if (resident ? !empty_turn : m >= 32 && kt >= 16) {
      c.waves = 8;
      c.xc = 8;
    }
  }
  if (c.parts == 1 && strips % 4 == 0) {
    if (mt == 2 && c.nt == 8) {
      c.waves = 4;
      c.xc = 4;
    } else if (mt == 2 && c.nt == 4) {
      c.waves = 8;
      c.xc = 8;
    } else if (mt == 1 && c.nt >= 4 && n * k / 2 >= (size_t(48) << 20)) {
      if (m <= 8) c.nt = 4;
      c.waves = 8;
      c.xc = 8;
    }
  }
  return c;
}

SplitKChoice select_splitk_blocks(int mt, size_t m_blocks, size_t n, size_t k) {
  SplitKChoice c;
  c.mt = mt;
  c.waves = 4;
  c.nt = 1;
  c.parts = 1;
  c.xc = 0;
  const size_t n_tiles = n / 16;
  // (eight column tiles also with two row tiles: n = 25600, k = 5120 at 32 rows 29.0 -> 22.4 us - half the x re-reads)
  for (int nt = 8; nt > 1; nt >>= 1) {
    if (n_tiles % nt == 0 && n_tiles / nt * m_blocks >= static_cast<size_t>(kNumCU) * 3 / 4) {
      c.nt = nt;
      break;
    }
  }
  (void)k;
  return c;
}

// Activations through LDS (w4a16_splitk.h) as in the dense form: 2-3 % at E = 256, hidden 7168, inter 2048 from a few
// tokens per expert on (64 tokens 813 -> 788 us, 512 tokens 1353 -> 1316 us for the whole block), not for a handful of
// blocks (1 token: 50.1 -> 52.6 us).
SplitKChoice select_splitk_grouped(size_t block_m, size_t blocks, size_t numel, size_t n, size_t k) {
  SplitKChoice c = select_splitk_blocks(static_cast<int>(block_m / 16), blocks, n, k);
  if ((n / 16) % 4 == 0 && numel >= 32) {
    if (c.mt == 2 && c.nt == 8) {
      c.waves = 4;
      c.xc = 4;
    } else if (c.mt == 2 && c.nt == 4) {
      c.waves = 8;
      c.xc = 8;
    } else if (c.mt == 1 && c.nt >= 4) {
      c.waves = 8;
      c.xc = 8;
    }
  }
  return c;
}

// Row blocks of block_m slots that numel slots fill where the router prefers none of the E experts, on average: c slots of an expert
// fill ceil(c / block_m), and c is about normal.
static double expected_row_blocks(size_t numel, size_t E, size_t block_m) {
  const double mean = static_cast<double>(numel) / E, deviation = std::sqrt(mean * (1.0 - 1.0 / E));
  if (mean > 8.0 * block_m) return E * (mean / block_m + 0.5);
  double blocks = 0;
  for (double least = 0.5; least < mean + 6.0 * deviation + 1.0; least += block_m)
    blocks += deviation > 0 ? 0.5 * std::erfc((least - mean) / (deviation * std::sqrt(2.0))) : least < mean;
  return E * blocks;
}

size_t grouped_row_blocks(size_t numel, size_t E, size_t block_m) {
  return std::min((numel + E * (block_m - 1)) / block_m, numel / block_m + E / 2 + 1);
}

// 32-slot blocks: the streaming kernel, where its workgroups of 256 columns come to three quarters of the CUs.  Whole int4 block,
// decode kernel / streaming kernel in us (experts, top-k, hidden, inter, tokens): 256, 8, 7168, 2048 at 512 tokens 1140 / 1066, at
// 1024 tokens 1690 / 1542; 128, 8, 4480, 640 at 352 210 / 177; 64, 8, 6656, 512 at 128 110 / 101; 32, 8, 3328, 512 at 124 (192
// workgroups in the first GEMM) 65.6 / 59.4; 16, 2, 4096, 1792 at 128 (224) 59.5 / 59.0.  Fewer leave the chip to a few long
// workgroups: 8, 2, 4096, 1536 at 96 (120) 44.6 / 50.8; 16, 2, 1024, 512 at 300 (108) 30.4 / 33.2; 16, 2, 2432, 512 at 144 (68)
// 33.1 / 39.4.  (Workgroups of 128 columns instead: 44.5, 30.0 and 35.8, and slower than the decode kernel above.)
//
// A little more than one round of its workgroups over the CUs leaves it behind too, where the decode kernel has eight strips to a
// workgroup (n a multiple of 128, its fastest form) and k is long.  Decode kernel / streaming kernel over 217 GEMMs of 2 to 64 experts, by
// the workgroups that even routing is expected to give: 140-192 1.05 in the mean (0.96-1.19), 192-256 1.04 (0.93-1.22), 256-320 0.96
// (0.76-1.10), 320-372 0.99 (0.88-1.15), 372-400 1.03.  Whole int4 block, streaming / decode kernel in such launches: 8, 2, 4480,
// 4736 at 17 rows per expert 90.3 / 83.6, 16, 4, 2432, 5888 at 35 151 / 130, 16, 1, 3584, 2176 at 19 73.0 / 68.7; and, k below
// 4096, where it does not hold: 16, 4, 2816, 1280 at 41 67.0 / 71.5, 8, 8, 2688, 4096 at 24 52.4 / 55.5.
bool use_w4a16_stream(size_t block_m, size_t blocks, size_t numel, size_t E, size_t n, size_t k) {
  const size_t tiles = div_up(n, 256);
  if (block_m != 32 || blocks * tiles < static_cast<size_t>(kNumCU) * 3 / 4) return false;
  if (n * k > (size_t(1) << 36)) return false;  // 32-bit offsets into an expert's scales
  if (n % 128 == 0 && k >= 4096 && blocks * tiles < 2 * static_cast<size_t>(kNumCU)) {
    const double wgs = expected_row_blocks(numel, E, block_m) * static_cast<double>(tiles);
    if (wgs > kNumCU * 1.03 && wgs <= kNumCU * 1.25) return false;  // (a handful more than 256 make no second round)
  }
  return true;
}

// Regime switch.  Up to 32 rows the split-K (decode) kernel; above, the MFMA tile kernel - except while the problem is
// small: the tile kernel has a floor of 17-22 us (a workgroup's prologue, the fp32 partial tiles of the cut along K and
// the pass that sums them), and the decode kernel run over blocks of 32 rows, each streaming the weights again (out of
// the L2: the blocks of one column group run on one XCD at the same time), stays below it while
// ceil(m / 32) * n * k <= 2^28, or 2^27 when K is the long side by four times or more (every block then re-reads a long
// row of x per column group).  Measured on MI355X over twelve shapes and 48..512 rows, decode / tile kernel in us:
// n = k = 4096 at 64 rows 10.9 / 19.2, at 128 rows 10.8 / 25.6, at 512 rows 27.0 / 29.5; n = 8192, k = 2048 at 128 rows
// 11.3 / 26.4, at 512 rows 29.2 / 40.1; n = k = 8192 at 64 rows 18.1 / 24.1, at 128 rows 30.6 / 32.0, at 192 rows
// 44.4 / 41.3; n = 14336, k = 4096 at 64 rows 17.9 / 23.1, at 128 rows 26.4 / 30.3, at 384 rows 75.1 / 56.3; n = 4096,
// k = 14336 at 128 rows 27.9 / 32.1, at 192 rows 48.4 / 38.9; n = 25600, k = 5120 at 64 rows 33.5 / 37.6, at 96 rows
// 48.6 / 46.1; n = 4096, k = 28672 at 64 rows 35.8 / 34.4; n = 5120, k = 25600 at 64 rows 61.7 / 36.6.  With the tile kernel's
// instances per number of live row tiles the line stays: n = k = 8192 at 128 rows 32.6 / 32.0, n = 25600, k = 5120 at 64 rows
// 35.1 / 36.1, n = 14336, k = 4096 at 128 rows 28.5 / 30.3, n = 4096, k = 14336 at 128 rows 29.4 / 32.1.
// (Group 128 only: the wide decode instances exist for that group.)
bool small_w4a16_problem(size_t m, size_t n, size_t k, size_t group) {
  const size_t limit = k >= 4 * n ? (size_t(1) << 27) : (size_t(1) << 28);
  return group == 128 && m <= kRowBlockMaxM && div_up(m, 32) * n * k <= limit;
}
bool use_mfma_tile(size_t m, size_t n, size_t k, size_t group) {
  if (m <= 32 || !(group == 128 || group == 64 || group == 32)) return false;
  if (g_small_problem_rule.load(std::memory_order_relaxed) && small_w4a16_problem(m, n, k, group)) return false;
  return true;
}

// 256-row tiles halve the weight traffic per output row, 128-row tiles waste less when m sits just above a multiple
// of 256.  With fewer than 192 output tiles the k range is cut into up to 256/tiles pieces of at least 4 k-tiles (512 k)
// each; the fp32 partial tiles are summed by a second, bandwidth-bound kernel.
// How to spread `tiles` output tiles of `kt` k-steps over the CUs.  Costs are in k-steps of one workgroup:
//   fixed    prologue + epilogue of a workgroup
//   partial  storing an fp32 partial tile instead of the output tile (and reading it back in the reduction)
//   reduce   launch of the reduction pass, plus per_unit for every partial tile it reads
// Candidates: every tile whole (ceil(tiles/CUs) rounds), or the full rounds whole and the tiles of the last, partly
// filled round cut into s parts of K.  A part is at least 4 k-steps and at most 512 partial tiles are written.
struct SpreadCost {
  double fixed, partial, reduce, per_unit;
};

void spread_tiles(unsigned tiles, unsigned kt, const SpreadCost& c, TilePlan* t) {
  const unsigned cus = static_cast<unsigned>(kNumCU);
  const unsigned full = tiles / cus * cus, rem = tiles - full;
  double best = div_up(tiles, cus) * (kt + c.fixed);
  t->main_items = 0;
  t->splits = 1;
  t->kt_per_split = kt;
  if (rem == 0) return;
  for (unsigned s = 2; s <= 16; ++s) {
    const unsigned per = static_cast<unsigned>(div_up(kt, s));
    if (per < 4) break;
    if (div_up(kt, per) != s) continue;  // the same parts as a smaller s
    const unsigned units = rem * s;
    if (units > 512) break;
    const double cost = (full / cus) * (kt + c.fixed) + div_up(units, cus) * (per + c.fixed + c.partial) + c.reduce + units * c.per_unit;
    if (cost < best) {
      best = cost;
      t->main_items = full;
      t->splits = s;
      t->kt_per_split = per;
    }
  }
}

void finish_plan(TilePlan* t) {
  const unsigned tiles = t->tiles_m * t->tiles_n;
  const unsigned cut = t->splits > 1 ? tiles - t->main_items : 0;
  t->grid = t->main_items + (tiles - t->main_items) * t->splits;
  t->workspace_bytes = static_cast<size_t>(cut) * t->splits * t->block_m * 256 * sizeof(float);
}

TilePlan plan_mfma_tile(size_t m, size_t n, size_t k) {
  TilePlan t{};
  const size_t rem = (m - 1) % 256;
  t.block_m = (m <= 128 || (m < 1024 && rem < 128)) ? 128 : 256;
  t.tiles_n = static_cast<unsigned>(div_up(n, 256));
  // where 256-row tiles leave more than half of the CUs idle but 128-row tiles fill the grid, take those (the weights are then fetched
  // twice as often, out of the L2 / Infinity Cache) rather than split K: fp32 partial tiles cost 8 bytes of HBM
  // traffic per output element and split.  Where neither fills it, 256-row tiles with a deeper split measured faster.
  const unsigned fill = static_cast<unsigned>(kNumCU) * 3 / 4;
  if (t.block_m == 256 && div_up(m, 256) * t.tiles_n < static_cast<unsigned>(kNumCU) / 2 && div_up(m, 128) * t.tiles_n >= fill)
    t.block_m = 128;
  // very few 256-row tiles (at most 32) are cut so finely along K that their fp32 partial tiles outweigh what the
  // larger tile saves: 128-row tiles need half the cut (n = k = 4096: 256 rows 34 -> 27 us, 512 rows 42 -> 33 us;
  // n = 4096, k = 14336 at 256 rows 52 -> 45 us; with K beyond 16384 the larger tile stays 1-3 % ahead)
  if (t.block_m == 256 && div_up(m, 256) * t.tiles_n <= 32 && k <= 16384) t.block_m = 128;
  t.tiles_m = static_cast<unsigned>(div_up(m, t.block_m));
  static const SpreadCost cost{3.0, 3.0, 2.0, 0.02};
  spread_tiles(t.tiles_m * t.tiles_n, static_cast<unsigned>(k / 128), cost, &t);
  finish_plan(&t);
  return t;
}

// Above two 16-token tiles the MFMA tile kernel (with split-K) - except, as for W4A16, while the problem is small enough
// for the streaming kernel over blocks of 32 tokens (four strips per workgroup sharing a block's activation fragments)
// to stay below the tile kernel's floor (15-22 us): ceil(m / 32) * n * k <= 5 * 2^24, and not with a K so short that a
// workgroup's life is its prologue (n > 4 k).  Measured on MI355X over eleven shapes and 48..512 tokens, streaming / tile
// kernel in us: n = k = 4096 at 64 tokens 11.3 / 17.5, at 128 tokens 11.2 / 22.4, at 256 tokens 20.1 / 23.0, at 384
// tokens 28.5 / 23.8; n = 2048, k = 7168 at 128 tokens 16.0 / 23.1, at 256 tokens 16.0 / 22.2, at 384 tokens 29.2 / 23.4;
// n = 7168, k = 2048 at 192 tokens 18.9 / 23.6, at 256 tokens 24.0 / 23.6; n = 4608, k = 7168 at 64 tokens 17.1 / 18.7, at
// 128 tokens 31.9 / 22.3; n = 7168, k = 4608 at 64 tokens 13.6 / 18.0, at 96 tokens 25.0 / 20.0; n = k = 7168 at 64 tokens
// 18.2 / 20.5, at 96 tokens 33.6 / 23.1; n = 24576, k = 1536 at 64 tokens 22.0 / 16.6; n = 18432, k = 7168 at 48 tokens
// 52.9 / 31.8.
bool use_fp8_tile(size_t m, size_t n, size_t k) {
  if (m <= 32) return false;
  if (g_small_problem_rule.load(std::memory_order_relaxed) && m <= kRowBlockMaxM && n <= 4 * k &&
      div_up(m, 32) * n * k <= (size_t(5) << 24))
    return false;
  return true;
}

// W4A8: the same, with the limit where its two kernels cross: ceil(m / 32) * n * k <= 5 * 2^25 (n <= 4 k).  Measured on
// MI355X over nine shapes and 48..512 tokens, streaming / tile kernel in us: n = k = 4096 at 64 tokens 9.5 / 16.9, at 128
// tokens 10.5 / 24.1, at 256 tokens 15.3 / 24.1, at 512 tokens 35.0 / 26.0; n = k = 5120 at 96 tokens 11.7 / 22.8, at 192
// tokens 18.7 / 23.6, at 256 tokens 28.5 / 24.6; n = 8192, k = 2048 at 128 tokens 10.3 / 23.6; n = 2048, k = 7168 at 256
// tokens 16.4 / 22.0; n = k = 8192 at 64 tokens 18.1 / 20.0, at 96 tokens 26.1 / 24.7; n = 14336, k = 4096 at 64 tokens
// 15.6 / 18.6, at 96 tokens 23.7 / 23.4; n = 25600, k = 5120 at 48 tokens 32.8 / 25.6.
bool use_w4a8_tile(size_t m, size_t n, size_t k) {
  if (m <= 32) return false;
  if (g_small_problem_rule.load(std::memory_order_relaxed) && m <= kRowBlockMaxM && n <= 4 * k &&
      div_up(m, 32) * n * k <= (size_t(5) << 25))
    return false;
  return true;
}

// Blockwise FP8, decode form: strips of 16 columns per workgroup.
// One strip up to 32 tokens while every workgroup has a CU to itself: halving their number leaves CUs idle.  GEMM alone in us, two
// strips / one: n = 4096, k = 14336 at 2, 16, 32 rows 13.4 / 12.2, 16.8 / 13.4, 22.0 / 19.1; n = k = 4096 at 16 6.4 / 5.8; n = 2048,
// k = 7168 at 16 9.0 / 7.6; n = 4224 (264 strips), k = 4096 at 16 6.4 / 8.4.
// Above, the activation fragments are as large as the weight fragments: two strips share them once there are several
// tokens, or when K is the long dimension (few strips, long streams).  With up to 8 tokens and no long K it is the last round
// of the CUs that tells: n = 13312, k = 4096 (416 workgroups of two strips) at 1 and 8 rows 10.9 / 11.3, 11.5 / 12.6, n = 24576,
// k = 1536 (768) at 8 9.8 / 10.9, but n = 18432, k = 7168 (576) 24.4 / 22.7, 25.4 / 25.0 and n = 28672, k = 4096 (896) 21.1 / 19.7;
// n = 8192, k = 4096, one round, 7.3 / 6.9 at one row, 7.3 / 7.6 at 8; n = 5120, k = 5120 6.6 / 6.8, 7.0 / 8.2.
int fp8_decode_strips(size_t m, size_t n, size_t k) {
  const size_t pairs = n / 32, rounds = div_up(pairs, kNumCU);
  int nt;
  if (m <= 32 && n <= 16 * static_cast<size_t>(kNumCU))
    nt = 1;
  else if (m > 8 || k > n)
    nt = 2;
  else if (rounds == 1)
    nt = m >= 5 ? 2 : 1;
  else
    nt = pairs * 10 >= rounds * kNumCU * (rounds == 2 ? 8 : 9) ? 2 : 1;
  // several blocks of 32 tokens (small problems above 32 tokens): four strips share a block's activation fragments while
  // the blocks together still give every other CU a workgroup
  if (m > 32 && n % 64 == 0 && n / 64 * div_up(m, 32) >= 128) nt = 4;
  return n % (16 * nt) == 0 ? nt : 1;
}

TilePlan plan_fp8_tile(size_t m, size_t n, size_t k) {
  TilePlan t{};
  // 128-token tiles where 256-token ones would be half padding (the weights are then fetched once per 128 tokens);
  // with full tiles the 256-token form is faster (M = 4096: 509 against 641 us)
  t.block_m = (m <= 128 || (m < 1024 && (m - 1) % 256 < 128)) ? 128 : 256;
  // as in plan_mfma_tile: at most 32 tiles of 256 tokens are better served by 128-token tiles and half the cut along K
  // (n = k = 5120 at 256 tokens: 31 -> 25 us; n = k = 4096 at 512 tokens: 33 -> 27 us)
  if (t.block_m == 256 && div_up(m, 256) * div_up(n, 256) <= 32 && k <= 16384) t.block_m = 128;
  t.tiles_m = static_cast<unsigned>(div_up(m, t.block_m));
  t.tiles_n = static_cast<unsigned>(div_up(n, 256));
  // fitted over five shapes at 64..2048 tokens; costlier cuts had left n = 25600, k = 5120 at 64..256 tokens on 100
  // of the 256 CUs (48 / 50 / 78 us against 36 / 43 / 65 us cut in two)
  static const SpreadCost cost{6.0, 4.0, 3.0, 0.035};
  spread_tiles(t.tiles_m * t.tiles_n, static_cast<unsigned>(k / 128), cost, &t);
  finish_plan(&t);
  return t;
}

size_t fp8_plan_kb(const TilePlan& plan, size_t k) { return plan.splits == 1 ? k / 128 : plan.kt_per_split; }

// One 256-row block of 129..240 rows: every weight is read once, by one workgroup, and the streaming tile kernel takes the tile
// kernel's plan with three (to 13 row tiles) or two k-blocks of weights in flight, activation slots for the row tiles that hold
// rows alone and eight wavefronts that share no weights.  fp8_tile.h / fp8_stream.h in us, GEMM alone, same bits: n = 18432,
// k = 7168 at 129, 150, 200, 224 rows 50.7 / 44.3, 55.7 / 47.3, 59.8 / 55.2, 61.6 / 59.8; n = 7168, k = 18432 49.5 / 41.7, 51.8 /
// 44.2, 55.3 / 52.3, 58.5 / 54.7; n = 24576, k = 1536, six k-blocks a workgroup, 27.9 / 22.2, 28.9 / 23.7, 30.7 / 27.7, 31.5 / 28.2;
// n = k = 14336 68.8 / 58.0, 73.6 / 61.3, 78.8 / 75.7, 81.1 / 77.2.  With all sixteen row tiles the two cross (n = 28672, k = 4096
// at 256 rows 60.5 / 62.8, n = k = 14336 84.9 / 84.9, n = 24576, k = 1536 33.4 / 30.7), and a few column tiles cut very often spend
// their time on partial sums (n = 1040, k = 28672: 129 rows 31.6 / 32.6, 150 36.4 / 33.7, 200 37.5 / 38.2); n = 5120, k = 25600, 20
// column tiles, at 129 and 200 rows 48.8 / 41.0, 55.1 / 50.6.  Workgroups of fewer than six k-blocks are not measured.
// Blocks of 128 rows stay on fp8_tile.h: n = 28672, k = 4096 at 33 and 100 rows 29.1 / 30.9, 35.8 / 39.0, n = 4096, k = 7168 at
// 100 rows 19.2 / 26.0; ahead by 4 to 6 % at n = k = 14336 only.
bool use_fp8_stream_dense(const TilePlan& plan, size_t m, size_t k) {
  const size_t kb_max = (plan.main_items || plan.splits == 1) ? k / 128 : plan.kt_per_split;
  return plan.tiles_m == 1 && plan.block_m == 256 && m <= 16 * kFp8StreamDenseTiles && plan.tiles_n >= 20 && fp8_plan_kb(plan, k) >= 6 &&
         fp8_stream_lds_bytes(16, kb_max) <= static_cast<size_t>(kFp8StreamLdsMax);
}

// W4A8: the blockwise-FP8 tile shapes; a k-step moves three quarters of the bytes and its prologue is shorter, so a
// cut along K pays earlier (measured at n = 25600, k = 5120: with the FP8 costs 64 / 128 / 256 tokens ran whole tiles
// on 100 of the 256 CUs in 38 / 51 / 83 us, with these they are cut in two or three: 28 / 38 / 60 us)
// Up to 64 tokens, 64-token tiles where K is whole or cut into parts of at least 32 k-blocks: the two wavefront rows share
// the row tiles (of a 128-token tile the lower one stands idle) and a barrier comes every two k-blocks.  Whole tiles, 128-
// against 64-token: n = 28672, k = 1024 at 64 tokens 13.1 / 12.4 us, n = 25600, k = 3072 24.4 / 23.2, n = 8192, k = 1024
// 12.0 / 10.8.  Shorter parts run on 128-token tiles: K is cut until (nearly) every CU has a workgroup, all of them fill
// their rings out of HBM at once, and a form that begins, and goes on, only when two k-blocks have landed starts later than
// one that waits for one (n = 16224, k = 3968 at 40 tokens, parts of 8: 17.3 / 18.0 us; n = 8192, k = 14336, parts of 14:
// 22.5 / 23.8; n = 4352, k = 20480 at 64 tokens, parts of 11: 23.8 / 24.7; parts of 20..24 at 40 tokens 27.4 / 28.4 and
// 29.7 / 30.3; parts of 32 at 64 tokens 38.2 / 37.2, 35.3 / 35.3 and 37.1 / 36.6).
TilePlan plan_w4a8_tile(size_t m, size_t n, size_t k) {
  TilePlan t{};
  t.block_m = (m <= 128 || (m < 1024 && (m - 1) % 256 < 128)) ? 128 : 256;
  // as in plan_mfma_tile: at most 32 tiles of 256 tokens are better served by 128-token tiles and half the cut along K
  // (n = k = 5120 at 256 tokens: 31 -> 25 us; n = k = 4096 at 512 tokens: 33 -> 27 us)
  if (t.block_m == 256 && div_up(m, 256) * div_up(n, 256) <= 32 && k <= 16384) t.block_m = 128;
  t.tiles_m = static_cast<unsigned>(div_up(m, t.block_m));
  t.tiles_n = static_cast<unsigned>(div_up(n, 256));
  static const SpreadCost cost{6.0, 4.0, 3.0, 0.03};
  spread_tiles(t.tiles_m * t.tiles_n, static_cast<unsigned>(k / 128), cost, &t);
  if (m <= 64 && (t.splits == 1 || t.kt_per_split >= 32)) t.block_m = 64;  // (one row block either way)
  finish_plan(&t);
  return t;
}

// One row block, 33..128 tokens.  Tile kernel / streaming kernel in us, GEMM with its reduction, same bits:
// - 65..112 tokens: n = 25600, k = 5120 at 80 33.4 / 27.9, n = 12384, k = 14592 at 70 38.6 / 31.6, n = 23872, k = 2816, whole K, at 69
//   28.4 / 20.7, n = 8896, k = 17920 at 82 35.9 / 31.8; the least n = 5120, k = 25600 at 100 36.0 / 33.1 and, parts of 6 to 8
//   k-blocks, n = 3424, k = 12288 at 108 23.7 / 23.4.  113..128, all eight row tiles: 25600, 5120 at 128 35.9 / 34.9, parts of 12 at
//   121 30.3 / 29.3, of 8 level to 2 % behind (n = 4128, k = 15360 at 115 25.6 / 26.1).
// - 33..64 tokens, parts of 20 k-blocks and more: 25600, 5120 at 33 and 64 26.0 / 22.5, 26.0 / 25.6, n = 14336, k = 8192 21.5 / 20.1,
//   23.7 / 23.2; shorter ones are over before the ring runs: parts of 8, 16224, 3968 at 64 18.5 / 19.6, of 11, 4352, 20480 23.9 / 25.0.
// - ... and whole K: workgroups of 128 columns while that is one round of them, tile kernel / 256 / 128 columns: n = 28672, k = 1024 at
//   33 and 64 10.8 / 9.5 / 8.5, 11.7 / 11.2 / 9.7, n = 8192, k = 1024 at 64 10.4 / 10.6 / 8.2.
// - ... and K that the plan cuts, where those workgroups come to three quarters of the CUs and K is not long, for no partial sums: 25600,
//   5120 (200 workgroups) at 33 and 64 26.0 / 22.5 / 21.4, 26.0 / 25.6 / 25.0, n = 28672, k = 4096 (224) 21.5 / 20.7 / 18.2, 23.4 / 23.9 /
//   20.9; but n = 20480, k = 8192 (160) at 64 29.0 / 29.1 / 36.0.
// - From 97 tokens on not with parts of up to 16 k-blocks of a K whose strips, and its parts, lie whole numbers of 16 KiB apart and
//   start on the same HBM channels: n = 4096, k = 16384 (parts of 8) at 80, 97, 112 level, 27.3 / 28.6, 27.9 / 29.3, n = 8192 (of 16) at
//   116 and 128 35.5 / 37.5, 36.2 / 37.9, n = 4096, k = 32768 at 128 37.0 / 38.5; k = 12288, 16256, 20480 ahead or level.
int w4a8_stream_strips(const TilePlan& plan, size_t m, size_t k) {
  if (plan.tiles_m != 1 || m <= 32 || m > 128) return 0;
  const unsigned narrow = 2 * plan.tiles_n;  // workgroups of 128 columns
  if (m <= 64 && narrow <= static_cast<unsigned>(kNumCU) && (plan.splits == 1 || (narrow >= static_cast<unsigned>(kNumCU) * 3 / 4 && k <= 6144)))
    return 1;
  const size_t kb = plan.splits == 1 ? k / 128 : plan.kt_per_split;
  if (m > 96 && plan.splits > 1 && kb <= 16 && k % 16384 == 0) return 0;
  return kb >= (m <= 64 ? 20u : m > 112 ? 10u : 1u) ? 2 : 0;
}

// W4A8 decode: a workgroup takes as many 16-column strips (up to 4) as still leave 128 workgroups - counting the row
// blocks of a problem of more than 32 tokens: n = k = 5120 at 64 tokens 16.8 -> 11.4 us with four strips instead of
// two -, and splits K over 8 wavefronts instead of 4 when fewer than 256 workgroups are left.
SplitKChoice select_w4a8_splitk(size_t m, size_t n) {
  SplitKChoice c{};
  c.mt = m <= 16 ? 1 : 2;
  c.nt = 4;
  const size_t m_blocks = div_up(m, 16 * c.mt);
  while (c.nt > 1 && (n % (16 * c.nt) != 0 || n / (16 * c.nt) * m_blocks < 128)) c.nt /= 2;
  c.waves = n / (16 * c.nt) * m_blocks < 256 ? 8 : 4;
  c.parts = 1;
  c.xc = 0;
  return c;
}

}  // namespace ksq

using namespace ksq;

// Row blocks of block-fp8 experts (ksq_moe_fp8_blockwise_gemm) where their sizes are not known: 16- and 32-row blocks stream
// through the split-K kernel, 128- and 256-row blocks run a tile kernel.  The lines were measured with the MFMA tile kernel
// (fp8_tile.h) for all of the latter; up to a mean of 15/16 of a block the streaming one (fp8_stream.h) runs there now, a sixth
// faster in the mean at 16 slots per expert, a tenth at 64, and the lines hold for it (ksq_moe_fp8_row_block).  With fp8_tile.h: from
// 16 rows per expert it is faster even with most of a 128-row block padding (each of its wavefronts multiplies the row tiles that
// hold rows), and 256-row blocks take over from 104 rows per expert, where experts begin to need a second block of 128 and their
// weights a second pass.  E = 256, hidden 7168, inter 2048, top-8, whole call with 16- / 32- / 128- / 256-row blocks: 1.50 / 1.49 /
// 1.61 / - ms at 2 rows per expert, 1.85 / 1.84 / 1.95 / - at 8, - / 1.95 / 1.98 / 2.02 at 12, - / 2.06 / 2.00 / 2.04 at 16, - /
// 3.18 / 2.12 / 2.12 at 32, - / - / 2.31 / 2.33 at 64, - / - / 2.56 / 2.60 at 96, - / - / 2.85 / 2.75 at 112, - / - / 3.22 / 2.87
// at 125, - / - / 3.29 / 2.91 at 128, - / - / 3.85 / 3.40 at 160, - / - / 5.45 / 4.92 at 256.
KSQ_EXPORT size_t ksq_moe_fp8_block_m(size_t numel, size_t E) {
  if (E == 0) return 16;
  const size_t per_expert = numel / E;
  if (per_expert >= 104) return 256;
  if (per_expert >= 16) return 128;
  return per_expert < 2 ? 16 : 32;
}

// The same where the experts' sizes are known.  Between 104 and 127 slots per expert the larger block pays by the rounds of
// workgroups that it saves: in 128-slot blocks, experts of more than 128 slots bring a second row block - their expected
// number under even routing, 128.5 - mean in standard deviations of a binomial -, and where those start another round of the
// 256 CUs in either GEMM, 256-slot blocks are up to a quarter faster; where they do not, a block of up to 160 slots is a
// longer chain than two of 128 and 1-7 % slower.  Whole call with 128- / 256-slot blocks, us, the faster one chosen: 32
// experts, hidden 2048, inter 1024 (256 workgroups) at 112 slots 122.9 / 92.9; 64, 1024, 512 (256) at 120 97.8 / 79.1; 16,
// 7168, 2048 at 112 266.7 / 231.9; 24, 2048, 1024 (192) at 120 86.2 / 90.7, at 127 104.4 / 90.4; 32, 1024, 512 (128) at
// 120 61.4 / 65.0; 16, 1152, 512 at 120 78.9 / 82.2; 8, 7168, 2048 at 112 134.9 / 138.6, at 127 156.1 / 143.1.  Over 92
// sizes of 4 to 160 experts the choice was at most 4.5 % behind the other one, the constant line at 104 slots 7 %.
// (From 128 slots on every second expert has a second row block, and the line is the one above.)
// These are times of the MFMA tile kernel; with the streaming one the choice was ahead or level at 104 and 116 slots in ten
// sizes, 128- / 256-slot blocks at 116: 16 experts, hidden 4096, inter 2048 198 / 142 us, 32, 4096, 2048 274 / 225, 64, 2048, 1408
// 221 / 191, where it takes 256; 8, 4096, 1536 86 / 92, 16, 2048, 1408 100 / 104, 32, 1024, 512 62 / 64.5, where it takes 128.
KSQ_EXPORT size_t ksq_moe_fp8_block_m_sized(size_t numel, size_t E, size_t hidden, size_t inter) {
  const size_t block_m = ksq_moe_fp8_block_m(numel, E);
  if (block_m != 256 || numel / E >= 128) return block_m;
  const double mean = static_cast<double>(numel) / E, variance = mean * (1.0 - 1.0 / E);
  const double share = variance > 0 ? 0.5 * std::erfc((128.5 - mean) / std::sqrt(2.0 * variance)) : 0.0;
  const size_t blocks = E + static_cast<size_t>(std::ceil(share * E));
  for (size_t n : {2 * inter, hidden}) {
    const size_t tiles = div_up(n, 256);
    if (div_up(blocks * tiles, kNumCU) > div_up(E * tiles, kNumCU)) return 256;
  }
  return 128;
}

// The block size of a whole block-fp8 expert block (both GEMMs and their alignment), the streaming tile kernel
// (fp8_stream.h) counted in.  From four slots per expert on its row blocks beat the 32-row blocks of the decode form where
// 16 experts or more give at least every other CU a 256-column tile in both GEMMs, us in 32-slot / 128-slot blocks at 4 and
// 8 slots, even routing: 256 experts, hidden 7168, inter 2048 1786 / 1653 and 1831 / 1695; 256, 1024, 512 132 / 100 and 148
// / 106; 64, 1024, 512 51 / 43 and 54 / 39; 16, 7168, 2048 132 / 125 and 136 / 126; 24, 2048, 768 (144 tiles) 48.7 / 38.3 and
// 50.5 / 38.8; 32, 1024, 512 (128 tiles) 32.5 / 31.4 and 34.2 / 32.5; 16, 2048, 1408 (128) 47.5 / 45.3 and 49.5 / 46.2; but
// 8, 7168, 2048 (128) 78 / 82 and 80 / 83, with uneven routing 71 / 76 and 76 / 82; 8, 4096, 1536 (96) 48.2 / 51.2 and 49.9
// / 52.2, 16, 1024, 512 (64) 25.2 / 28.9 and 25.6 / 29.2.  (Below four: 32, 4096, 2048 at 1 and 2 slots 106 / 118 and 138 /
// 139, 128, 2944, 768 at 1 118 / 122.)  Over 44 sizes drawn between 16 and 160 experts, hidden 1024 to 7168, inter 512 to
// 2048, at 4 to 12 slots, the row blocks are 0.98 to 1.44 times as fast as the decode form under even routing, 1.20 in the
// mean, and 0.87 to 1.54, 1.21 in the mean, where routing prefers some experts (logits with a spread of 0.7 per expert);
// where every token takes the same top-k of 16 or 32 experts too few tiles are left (16, 7168, 2048, top-2, at 8 slots 54 /
// 79, 16, 5120, 2048, top-1, at 6 40 / 75), of 48 or more experts rarely (128, 1024, 512, top-8, at 4 32 / 39; 160, 5120,
// 1536, top-6, 144 / 84).
//
// From 16 slots on the lines are those of ksq_moe_fp8_block_m_sized, for both tile kernels: 256-slot blocks gain nothing at
// 64 slots where the routing is even (16, 4096, 2048 97.8 / 97.8) and leave half as many workgroups where it is not (logits
// with a spread of 0.7 per expert, 128- / 256-slot blocks at 64 slots: 16, 2048, 1408 69 / 94; 8, 4096, 1536 81 / 105).
KSQ_EXPORT size_t ksq_moe_fp8_row_block(size_t numel, size_t E, size_t hidden, size_t inter) {
  if (E == 0) return 16;
  const size_t per_expert = numel / E, tiles = E * div_up(2 * inter < hidden ? 2 * inter : hidden, 256);
  // (the row blocks of 128 slots hold 32-bit offsets into the activations, and the weight scales of all of K in the LDS)
  const size_t longest = hidden > inter ? hidden : inter;
  const bool fits = longest <= (size_t(1) << 20) && numel * longest <= 0xffffffffull;
  if (per_expert >= 4 && per_expert < 16 && E >= 16 && tiles >= static_cast<size_t>(kNumCU) / 2 && fits) return 128;
  return ksq_moe_fp8_block_m_sized(numel, E, hidden, inter);
}

// Rows per expert block for numel routed (token, slot) pairs over E experts.  Replaces the M thresholds of
// InvokeFusedMoe (16 / 32 / 64 rows by token count): with few rows per expert the weights are streamed once per
// 16- or 32-row block (HBM-bound); above, the MFMA tile kernel takes 256-row blocks, of which it multiplies the row
// tiles that hold rows (an instance of its main loop per count), so that an expert's weights are dequantized once
// however many of the 256 rows it fills.  Few experts make few 256-row workgroups: the line lies the higher, the fewer there
// are.  Whole block, time in 32-row blocks over time in 256-row blocks at 48 / 64 / 80 / 100 / 128 rows per expert (hidden, inter), where
// routing prefers no expert and, in brackets, where it prefers some (logits with a spread of 0.7 per expert):
//   8 experts   7168, 2048 0.74 0.96 0.78 0.81 0.89 (0.81 0.67 0.71 0.63 0.68)   4096, 4096 0.75 at 60, 0.77 at 84, 0.78 at 105, 0.90
//   16          7168, 2048 0.66 0.71 0.71 0.80 0.77 (0.63 0.71 0.70 0.64 0.76)   2048, 1408 0.86 0.94 0.92 1.02 1.16 (0.78 0.67 0.73 0.71 0.87)
//   32          7168, 2048 0.68 0.74 0.80 0.99 1.00 (0.67 0.72 0.75 0.81 0.86)   2048, 1408 0.85 0.99 1.08 1.14 1.15 (0.62 0.73 0.85 0.84 0.80)
//   64          4096, 1536 0.80 0.86 0.95 1.21 1.27 (0.63 0.68 0.75 0.82 0.84)   1024, 512  1.16 1.14 1.16 1.19 1.22 (0.69 0.78 0.63 0.67 0.76)
//   128         4096, 1536 0.92 1.02 1.08 1.23 1.29 (0.70 0.83 0.87 0.96 0.99)   2048, 768  0.94 1.04 1.15 1.27 1.29 (0.67 0.81 0.81 0.77 0.91)
//   256         4096, 2048 0.89 at 50, 0.99 1.11 (0.75 at 50, 0.82 0.97)
// With 9 experts and more a line lies where the first of the sizes that were timed with so many nears its crossing without
// preferences, so that none is behind; larger ones would bear a higher line (7168, 2048 with 16 experts 0.77 at 128 rows, with 32 0.80 at
// 80; 4096, 1536 with 64 0.86 at 64), and uneven routing nearly all.  Up to 8 it lies at the end of what was timed: 0.6 to 1.0 before it,
// but for hidden 4480 with inter 6144 to 12032 from 105 rows on, 1.01-1.12 (0.82-0.91), and the sizes that
// ksq_moe_w4a16_row_block takes out.
// 16- and 32-row blocks: half-empty blocks of 32 run one row tile of the streaming kernel, which keeps more in flight than the
// decode kernel over 16-row blocks, and an expert with more than 16 rows reads its weights once (under uneven routing 32-row blocks are
// ahead sooner, by 5 to 15 %).  Time in 32-row blocks over time in 16-row blocks, no preferences, at 3 / 5 / 7 / 9 / 11 / 13 / 15 rows per expert:
//   16 experts  4096, 1536 1.01 1.02 0.99 1.00 1.01 0.99 0.99   4096, 768 1.12 1.14 1.12 1.15 1.13 1.08 1.02
//   32          7168, 2048 1.06 1.05 1.06 1.01 0.98 0.95 0.89   1024, 512 1.30 1.23 1.07 0.99 1.01 0.98 0.96
//   64          4096, 1536 0.98 0.99 0.99 1.01 0.94 0.92 0.89   7168, 2048 1.05 1.05 1.03 1.03 0.99 0.96 0.88
//   128         4096, 768  0.93 0.92 0.95 0.91 0.91 0.85 0.81   7168, 2048 1.03 1.02 1.01 1.01 0.98 0.92 0.85
//   256         7168, 2048 1.02 1.01 0.99 0.98 0.96 0.90 0.83   1024, 512 0.82 0.83 0.81 0.81 0.81 0.80 0.77
// 128-row blocks are not ahead of 256-row ones anywhere (256 experts, 128 rows 4.40 against 3.57 ms).
KSQ_EXPORT size_t ksq_moe_block_m(size_t numel, size_t E) {
  if (E == 0) return 16;
  const size_t per_expert = numel / E;
  if (per_expert >= (E <= 8 ? 129u : E <= 16 ? 72u : E <= 32 ? 56u : 44u)) return 256;
  return per_expert < (E >= 128 ? 7u : E >= 32 ? 10u : 16u) ? 16 : 32;
}

// The block size of a whole int4 expert block (both GEMMs and their alignment).  Up to 8 experts whose first GEMM has four rounds of
// 256-row workgroups (1024 of them) give the tile kernel its workgroups: its line is that of 16 experts.  Whole block, even routing,
// 32- / 256-row blocks in us at 68 / 72 / 80 / 90 / 100 / 128 rows per expert: 8 experts, hidden 6144, inter 16384 534 / 555, 595 / 561, 631 /
// 573, 693 / 600, 762 / 752, 950 / 849; 8, 8192, 28672 1346 / 1443, 1421 / 1470, 1478 / 1501, 1646 / 1574, 1828 / 1640, 2231 / 1875; 8,
// 4096, 28672 712 / 766, 739 / 801, 767 / 813, 845 / 846, 927 / 875, 1165 / 982.  With fewer 32-row blocks are ahead, or level at the
// end: 8, 4096, 14336 (896 workgroups) at 80, 100, 128 372 / 423, 435 / 511, 566 / 569, 8, 8192, 14336 702 / 794, 894 / 941, 1085 / 1065.
// Where routing prefers some experts (logits with a spread of 0.7 per expert) 32-row blocks are ahead longer, up to a quarter.  (The tile
// kernel rounds dequantized weights to T, where 16- and 32-row blocks keep them exact: 2.2e-3 and 1.7e-3 off in bf16.)
//
// With hidden a multiple of 4096 and inter of 4096 and more the gate / up projection's strips share their HBM channels (w4a16_stream.h)
// and the streaming kernel does not make up for half-empty blocks before 11 rows per expert.  Even routing, 16- / 32-row blocks at 7, 10,
// 11, 13 rows: 128 experts, hidden 4096, inter 4096 525 / 577, 549 / 586, 566 / 591, 603 / 590 us; 64, 8192, 4096 529 / 592, 536 / 594,
// 551 / 604, 602 / 618; 64, 4096, 14336 882 / 938, 913 / 951, 966 / 958, 1055 / 972; inter 2048, 128, 4096 291 / 296, 296 / 298.  (Uneven
// as above: 471 / 460, 535 / 457, 599 / 511 for the first.)
//
// From 40 rows each on, activations of 1 GiB, which the launches of 16- and 32-row blocks refuse (32-bit offsets), run the tile kernel,
// which takes 4 GiB.  (As many rows as slots: the second GEMM's, and the first one's behind a gather.)
KSQ_EXPORT size_t ksq_moe_w4a16_row_block(size_t numel, size_t E, size_t hidden, size_t inter) {
  const size_t block_m = ksq_moe_block_m(numel, E);
  const size_t longest = hidden > inter ? hidden : inter;
  if (E != 0 && numel / E >= 40 && numel > 0x3fffffffull / 2 / (longest ? longest : 1)) return 256;
  if (block_m == 32 && numel / E < 11 && hidden % 4096 == 0 && inter >= 4096) return 16;
  if (E != 0 && E <= 8 && numel / E >= 72 && E * div_up(2 * inter, 256) >= 4 * static_cast<size_t>(kNumCU)) return 256;
  return block_m;
}

KSQ_EXPORT int ksq_moe_w4a16_kernel(size_t numel, size_t E, size_t n, size_t k, size_t block_m) {
  if (block_m >= 128) return KSQ_KERNEL_MFMA_TILE;
  if (block_m == 0 || E == 0) return KSQ_KERNEL_SPLITK_WAVE;
  return use_w4a16_stream(block_m, grouped_row_blocks(numel, E, block_m), numel, E, n, k) ? KSQ_KERNEL_STREAM_TILE : KSQ_KERNEL_SPLITK_WAVE;
}

KSQ_EXPORT int ksq_w4a8_kernel(size_t m, size_t n, size_t k) {
  if (n == 0 || k == 0 || !use_w4a8_tile(m, n, k)) return KSQ_KERNEL_SPLITK_WAVE;
  return w4a8_stream_strips(plan_w4a8_tile(m, n, k), m, k) ? KSQ_KERNEL_STREAM_TILE : KSQ_KERNEL_MFMA_TILE;
}

KSQ_EXPORT int ksq_set_small_problem_rule(int enabled) { return g_small_problem_rule.exchange(enabled ? 1 : 0); }

KSQ_EXPORT int ksq_select_tile(int kind, size_t m, size_t n, size_t k, int dtype, ksq_tile_desc* d) {
  if (!d) return fail(KSQ_ERR_INVALID_ARGUMENT, "ksq_select_tile: null descriptor");
  if (m == 0 || n == 0 || k == 0) return fail(KSQ_ERR_INVALID_ARGUMENT, "ksq_select_tile: empty problem");
  if (dtype != KSQ_F16 && dtype != KSQ_BF16) return fail(KSQ_ERR_UNSUPPORTED, "ksq_select_tile: dtype %d has no kernel", dtype);
  if (k % 128 != 0 || n % 16 != 0)
    return fail(KSQ_ERR_UNSUPPORTED, "ksq_select_tile: no kernel for n=%zu k=%zu (k must be a multiple of 128, n of 16)", n, k);
  *d = ksq_tile_desc{};
  switch (kind) {
    case KSQ_KIND_W4A16:
    case KSQ_KIND_MOE_W4A16: {
      if (kind == KSQ_KIND_W4A16 && use_mfma_tile(m, n, k, 128)) {
        const TilePlan t = plan_mfma_tile(m, n, k);
        d->kernel = KSQ_KERNEL_MFMA_TILE;
        d->block_m = t.block_m;
        d->block_n = 256;
        d->block_k = 64;
        d->waves = 8;
        d->split_k = static_cast<int32_t>(t.splits);
        d->grid = static_cast<int32_t>(t.grid);
        return KSQ_OK;
      }
      const size_t slots = m <= 16 ? 16 : 32;
      const SplitKChoice c = kind == KSQ_KIND_W4A16 ? select_splitk(m, n, k) : select_splitk_grouped(slots, div_up(m, slots), m, n, k);
      d->kernel = KSQ_KERNEL_SPLITK_WAVE;
      d->block_m = 16 * c.mt;
      d->block_n = 16 * c.nt;
      d->block_k = 128;
      d->waves = c.waves;
      d->split_k = c.waves * c.parts;
      d->grid = static_cast<int32_t>((n / 16 / c.nt) * div_up(m, 16 * c.mt) * c.parts);
      d->x_chunk = c.xc;
      return KSQ_OK;
    }
    case KSQ_KIND_FP8_BLOCKWISE: {
      if (use_fp8_tile(m, n, k)) {
        const TilePlan t = plan_fp8_tile(m, n, k);
        d->kernel = use_fp8_stream_dense(t, m, k) ? KSQ_KERNEL_STREAM_TILE : KSQ_KERNEL_MFMA_TILE;
        d->block_m = t.block_m;
        d->block_n = 256;
        d->block_k = 128;
        d->waves = 8;
        d->split_k = static_cast<int32_t>(t.splits);
        d->grid = static_cast<int32_t>(t.grid);
        return KSQ_OK;
      }
      // decode: 16 weight rows x (16|32|64) tokens per workgroup, the wavefronts split K between them
      const int mt = m <= 16 ? 1 : 2;
      const int waves = 4;
      d->kernel = KSQ_KERNEL_SPLITK_WAVE;
      const int nt = fp8_decode_strips(m, n, k);
      d->block_m = 16 * mt;
      d->block_n = 16 * nt;
      d->block_k = 128;
      d->waves = waves;
      d->split_k = waves;
      d->grid = static_cast<int32_t>(div_up(m, 16 * mt) * (n / (16 * nt)));
      return KSQ_OK;
    }
    case KSQ_KIND_W4A8: {
      if (use_w4a8_tile(m, n, k)) {
        const TilePlan t = plan_w4a8_tile(m, n, k);
        d->kernel = KSQ_KERNEL_MFMA_TILE;
        const bool narrow = w4a8_stream_strips(t, m, k) == 1;  // 128 columns per workgroup, K whole
        d->block_m = narrow ? 64 : t.block_m;
        d->block_n = narrow ? 128 : 256;
        d->block_k = 128;
        d->waves = 8;
        d->split_k = narrow ? 1 : static_cast<int32_t>(t.splits);
        d->grid = static_cast<int32_t>(narrow ? 2 * t.tiles_n : t.grid);
        return KSQ_OK;
      }
      const SplitKChoice c = select_w4a8_splitk(m, n);
      d->kernel = KSQ_KERNEL_SPLITK_WAVE;
      d->block_m = 16 * c.mt;
      d->block_n = 16 * c.nt;
      d->block_k = 128;
      d->waves = c.waves;
      d->split_k = c.waves;
      d->grid = static_cast<int32_t>(div_up(m, 16 * c.mt) * (n / (16 * c.nt)));
      return KSQ_OK;
    }
    default:
      return fail(KSQ_ERR_INVALID_ARGUMENT, "ksq_select_tile: unknown kind %d", kind);
  }
}
