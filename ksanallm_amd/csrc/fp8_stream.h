// Blockwise-FP8 kernel for row blocks of at most 256 tokens whose time is the stream of their weights (the experts of a MoE
// block): a workgroup of 8 wavefronts side by side along N computes up to 256 tokens x 256 output columns.
//
// What bounds it is the stream of the weights out of HBM and what stands in its way in each CU's one vector memory path:
//   - weights never touch LDS: every fragment belongs to one wavefront (two strips of 16 columns each), which loads it from
//     its packed 2 KiB form (ksq_fp8_repack_weight) straight into a register ring of D k-blocks, non-temporally unless the
//     block is full or, dense, K is short: they are read once, and cached they turn the L2 over (256 experts, hidden 7168,
//     inter 2048, 512 tokens, whole block: 2.05 -> 1.88 ms, 6.0 TB/s of weights).
//   - activations go global -> LDS (global_load_lds_dwordx4, whole 128-byte lines) into D slots that hold only the row tiles
//     with tokens; all eight wavefronts read them from there.  Four wavefronts and 128 columns, two workgroups to a CU,
//     overlap a workgroup's ends with the other's stream but fetch the activations twice as often: 4000 tokens 2.79 against
//     2.67 ms.  D = 3 and D = 4 measure the same.
//   - a row's scales of four k-blocks are one 16-byte piece, fetched once: a load of one scale per row touches 64 lines for
//     256 bytes, and one per k-block was 7 % of the call.
//   - results leave through LDS as whole rows of the tile, non-temporally (8-byte stores of 32 bytes a row: 2.71 against 2.60 ms).
//   - a loop instance per number of row tiles, chosen once per workgroup; full 256-slot blocks run fp8_tile.h's code.
// Whole block at 4000 tokens, bf16: 2.87 ms with fp8_tile.h's grouped form, 2.60 with this one.  The sums run over k in one order,
// as fp8_tile.h's do: the same bits.  (The decode form of 16- and 32-row blocks adds four partial sums, one of each wavefront.)
#pragma once

#include "fp8_encode.h"
#include "fp8_tile.h"
#include "ksq_common.h"
#include "tile_work.h"

namespace ksq {

struct Fp8StreamParams {
  const uint8_t* a;   // [rows, k]
  const float* a_s;   // a_s[row, kb] at row * as_row_bytes + kb * as_kb_bytes
  const uint8_t* b;   // [E, n, k] in packed 2 KiB fragments (ksq_fp8_repack_weight)
  const float* b_s;   // [E, ceil(n/128), k/128]
  void* out;          // [numel, n]
  uint32_t N, K;
  uint32_t block;             // slots of a row block: tile_m holds sorted_ids[tile_m * block ..] of expert expert_ids[tile_m]
  uint32_t tiles_m, tiles_n;  // tiles_m: the most row blocks an alignment can make
  uint32_t as_row_bytes, as_kb_bytes;
  uint32_t scales4;           // the scales of four k-blocks are 16 aligned bytes of a row
  const int32_t* sorted_ids;
  const int32_t* expert_ids;
  const int32_t* num_post_pad;
  const float* topk_w;
  uint32_t numel, top_k, scale_rows;  // scale_rows = ceil(N/128): rows of one expert's b_s
  float* out_s;               // PAIRED: scales [numel, N / 256] of the codes out [numel, N / 2]
  // DENSE: a plain GEMM of numel rows (top_k 1, no slot ids), whose tiles may be cut along K
  float* out32;               // verification only: the fp32 sums go here, [numel, N], and nothing is rounded to TO
  float* partial;             // [slot][part][block][256] fp32 tiles of the workgroups that compute a part of K
  uint32_t main_items, splits, kb_per_split;  // tile_work.h
  uint32_t tile_full;         // full 256-slot blocks run the code of fp8_tile.h (0: its stages do not fit beside K's weight scales)
};

constexpr int kFp8StreamLdsMax = 160 * 1024;
// k-blocks in the weight ring and activation slots, by the registers that the accumulators leave
constexpr int fp8_stream_depth(int rt) { return rt <= 8 ? 4 : rt <= 13 ? 3 : 2; }
// activation scales: two slots of 16 bytes (four k-blocks) a row, or a slot of 256 floats per k-block in the ring
constexpr int fp8_stream_scale_slot4(int rt) { return (rt + 3) / 4 * 1024; }
constexpr int fp8_stream_area(int rt) {
  const int d = fp8_stream_depth(rt);
  return d * rt * 2048 + (2 * fp8_stream_scale_slot4(rt) > d * 1024 ? 2 * fp8_stream_scale_slot4(rt) : d * 1024);
}
constexpr int kFp8StreamDenseTiles = 15;          // row tiles of a dense block, at most
constexpr int kFp8StreamOutTiles = 8;             // row tiles whose results pass through LDS at a time
constexpr int kFp8StreamOutPitch = 256 * 2 + 16;  // bytes of a row of them
constexpr int fp8_stream_area_max(int rt_max) {
  int most = (rt_max < kFp8StreamOutTiles ? rt_max : kFp8StreamOutTiles) * 16 * kFp8StreamOutPitch;
  for (int rt = 1; rt <= rt_max; ++rt) most = fp8_stream_area(rt) > most ? fp8_stream_area(rt) : most;
  return most;
}
// ... then the block's slot ids, then the weight scales of the tile's two 128-column blocks
constexpr size_t fp8_stream_lds_bytes(int rt_max, size_t kb_max) { return fp8_stream_area_max(rt_max) + 1024 + 2 * kb_max * 4; }

// PAIRED: gate / up weights [2 * inter, K], and the result is the second GEMM's quantized input: a wavefront's strips are a
// gate strip and the matching up strip, a workgroup covers 128 channels of the activation, one quantization group, and stores
// e4m3(T(silu(T(gate)) * T(up)) / scale) with the group's scale - the bits of the plain GEMM followed by the quantizer with
// the activation in front, without [numel, 2 * inter] through memory and without the quantizer's launch (256 experts, hidden
// 7168, inter 2048, whole block: 512 tokens 1.86 -> 1.78 ms, 4000 tokens, where the activation of a tile stands for 5 us at
// the end of its workgroup, 2.58 -> 2.55; 64 experts, hidden 2048, inter 1408, 48 tokens 115 -> 111 us).
//
// DENSE: tile m holds rows m * block .., results go to their rows or, from a workgroup that computes a part of K, to fp32
// partial tiles (splitk_reduce.h).  200 rows, n = 18432, k = 7168: 59.8 us with fp8_tile.h, 55.2 with this form (2.4 TB/s of
// weights; 150 rows 55.7 -> 47.3): the MFMAs of 13 row tiles in whole waves of 32 columns and the partial sums are the rest.
// SHORT_K: a workgroup multiplies fewer than 16 k-blocks; the weights are loaded cached (fp8_blockwise_gemm.hip).
template <typename TO, int RT_MAX, bool PAIRED, bool DENSE = false, bool SHORT_K = false>
__global__ void __launch_bounds__(512, 1) fp8_stream_tile_kernel(Fp8StreamParams p) {
  extern __shared__ __attribute__((aligned(16))) char lds[];  // fp8_stream_lds_bytes
  constexpr int WAVES = 8;
  constexpr int BN = 32 * WAVES;
  constexpr int FRAG = 2048;
  constexpr int IDS_BASE = fp8_stream_area_max(RT_MAX);
  constexpr int BS_BASE = IDS_BASE + 1024;

  const int lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lrow = lane & 15, lq = lane >> 4;
  const uint32_t k_blocks = p.K / 128;

  // ---- work item (tile_work.h): over the row blocks that hold slots, those past them leave
  uint32_t tiles_m = p.tiles_m;
  if constexpr (!DENSE) {
    const uint32_t filled = (static_cast<uint32_t>(p.num_post_pad[0]) + p.block - 1) / p.block;
    tiles_m = __builtin_amdgcn_readfirstlane(filled < p.tiles_m ? filled : p.tiles_m);
    if (blockIdx.x >= tiles_m * p.tiles_n) return;  // uniform: the whole workgroup leaves
  }
  const TileWork work = tile_work(blockIdx.x, tiles_m, p.tiles_n, DENSE ? p.main_items : 0, DENSE ? p.splits : 1, !DENSE);
  const uint32_t tile_m = __builtin_amdgcn_readfirstlane(work.tile_m), tile_n = __builtin_amdgcn_readfirstlane(work.tile_n);
  const uint32_t m0 = tile_m * p.block, n0 = tile_n * BN;
  const uint32_t part = __builtin_amdgcn_readfirstlane(work.part), out_slot = __builtin_amdgcn_readfirstlane(work.slot);
  const bool direct = !DENSE || __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(work.direct)) != 0;
  // the k-blocks of this workgroup: kb0 .. kb0 + KB - 1
  const uint32_t kb0 = __builtin_amdgcn_readfirstlane(direct ? 0 : part * p.kb_per_split);
  const uint32_t KB = __builtin_amdgcn_readfirstlane(direct || k_blocks - kb0 < p.kb_per_split ? k_blocks - kb0 : p.kb_per_split);

  // ---- slots of this block: their ids go to LDS (rows past the block hold no slot)
  const size_t expert = DENSE ? 0 : static_cast<size_t>(__builtin_amdgcn_readfirstlane(p.expert_ids[tile_m]));
  constexpr int CHUNKS = RT_MAX / 4;  // of 64 slots
  uint32_t sids[CHUNKS], rows = 0;
#pragma unroll
  for (int h = 0; h < CHUNKS; ++h) {
    const uint32_t r = m0 + h * 64 + lane;
    if constexpr (DENSE)
      sids[h] = r < p.numel ? r : p.numel;
    else
      sids[h] = static_cast<uint32_t>(p.sorted_ids[r]);
    rows += static_cast<uint32_t>(__builtin_popcountll(__builtin_amdgcn_ballot_w64(sids[h] < p.numel)));
  }
  const uint32_t live_tiles = __builtin_amdgcn_readfirstlane((rows + 15) / 16);
  // A full 256-slot block is bound by the LDS here (eight wavefronts that each read all sixteen activation fragments keep it
  // busy as long as the MFMAs take) and runs the tile kernel's code, 2 x 4 wavefronts, in the same launch with the same bits.  us,
  // whole block in 256-slot blocks, fp8_tile.h alone / fp8_stream.h alone / this: logits with a spread of 1.5 per expert, 256
  // experts, hidden 7168, inter 2048 at 160 slots 3198 / 3287 / 3114; 64, 2048, 1408 257 / 271 / 250; 32, 4096, 2048 at 208 365 / 372 /
  // 361; every token on the same sixteenth of the experts, 64, 7168, 2048 at 128 452 / 473 / 449; 8, 4096, 1536 108 / 126 / 106.  Even
  // routing at 208 slots 3777 / 3497 / 3501, 261 / 249 / 249.  Blocks of 209 to 240 slots stay here, for the even routing: with
  // few experts that most tokens prefer they are up to 5 % behind (8, 4096, 1536 at 232, the latter routing, 141 / 159 / 150).
  if constexpr (!DENSE && RT_MAX == 16) {
    if (live_tiles == RT_MAX && p.tile_full) {  // uniform: the whole workgroup
      Fp8TileParams t{};
      t.a = p.a;
      t.a_s = p.a_s;
      t.b = p.b;
      t.b_s = p.b_s;
      t.out = p.out;
      t.out_s = p.out_s;
      t.M = p.tiles_m * p.block;
      t.N = p.N;
      t.K = p.K;
      t.tiles_m = p.tiles_m;
      t.tiles_n = p.tiles_n;
      t.splits = 1;
      t.kb_per_split = k_blocks;
      t.as_row_bytes = p.as_row_bytes;
      t.as_kb_bytes = p.as_kb_bytes;
      t.sorted_ids = p.sorted_ids;
      t.expert_ids = p.expert_ids;
      t.num_post_pad = p.num_post_pad;
      t.topk_w = p.topk_w;
      t.numel = p.numel;
      t.top_k = p.top_k;
      t.scale_rows = p.scale_rows;
      fp8_tile_body<TO, true, 8, 256, true, PAIRED>(t, lds);
      return;
    }
  }
  uint32_t* ids = reinterpret_cast<uint32_t*>(lds + IDS_BASE);
#pragma unroll
  for (int h = 0; h < 4; ++h)
    if (wave == static_cast<uint32_t>(h)) ids[h * 64 + lane] = h < CHUNKS ? sids[h < CHUNKS ? h : 0] : p.numel;
  // the weight scales of the tile's two blocks of 128 weight rows
  for (uint32_t t = threadIdx.x; t < 2 * KB; t += 512) {
    const uint32_t blk = t / KB, kb = t - blk * KB, nb_last = (p.N - 1) / 128;
    const uint32_t nb = PAIRED ? tile_n + blk * (p.N / 256) : n0 / 128 + blk < nb_last ? n0 / 128 + blk : nb_last;
    reinterpret_cast<float*>(lds + BS_BASE)[t] = p.b_s[(expert * p.scale_rows + nb) * k_blocks + kb0 + kb];
  }
  __syncthreads();
  auto row_of = [&](uint32_t r) -> uint32_t {  // activation row of slot r of the block; a row without a slot reads some valid one
    uint32_t sid = ids[r];
    sid = sid < p.numel ? sid : p.numel - 1;
    return DENSE ? sid : sid / p.top_k;
  };

  const uint8_t* a_base = scalar_ptr(p.a + static_cast<size_t>(kb0) * 128);
  const char* s_base = scalar_ptr(reinterpret_cast<const char*>(p.a_s) + static_cast<size_t>(kb0) * p.as_kb_bytes);
  const uint32_t s_voff = row_of((wave & 3) * 64 + lane) * p.as_row_bytes;
  const uint32_t w_voff = lane * 16;
  const uint32_t strips = p.N / 16;
  const uint8_t* w_base[2];  // (strips past N repeat the last one; their results are not stored)
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const uint32_t strip = PAIRED ? tile_n * 8 + wave + t * (strips / 2) : n0 / 16 + wave * 2 + t;
    w_base[t] = scalar_ptr(p.b + ((expert * strips + (strip < strips ? strip : strips - 1)) * k_blocks + kb0) * FRAG);
  }
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<size_t>((__attribute__((address_space(3))) char*)lds));
  // An activation fragment (16 rows x 128 bytes) is two loads of 8 rows: eight lanes take the eight 16-byte pieces of a
  // row, one whole cache line (as two loads of 64 bytes a row the same fragment is twice the requests to the L2).  Load lane
  // j lands at 16j = 128*(j/8) + 16*(j%8) and fetches piece (j%8) ^ (j/8) of its row, so that MFMA lane (row r, k slot q)
  // finds its pieces 2q and 2q+1 at 128r + 16*(piece ^ (r%8)): eight lanes that read together cover all banks.
  const uint32_t rd_lo = 128 * lrow + 16 * ((2 * lq) ^ (lrow & 7));
  const uint32_t rd_hi = rd_lo ^ 16;
  const float* bs_lds = reinterpret_cast<const float*>(lds + BS_BASE) + (PAIRED ? 0 : wave / 4 * KB);

  auto run = [&](auto rt_c) {
    constexpr int RT = decltype(rt_c)::value;
    constexpr int D = fp8_stream_depth(RT);  // k-blocks in the weight ring = activation slots
    constexpr int AL = (2 * RT + WAVES - 1) / WAVES;  // activation loads per wavefront and k-block: 2 * RT groups of 8 rows
    // loads of a wavefront per k-block that the waits count: with the four of the weights.  The scale loads, which not every
    // wavefront issues and not for every k-block, are not counted: a wait then covers one load more than it has to.
    constexpr int GROUP_LOADS = AL + 4;
    constexpr int SLOT = RT * FRAG;
    constexpr int SC_BASE = D * SLOT;
    constexpr int SC4 = fp8_stream_scale_slot4(RT);
    // A full block's expert most likely has another block, which reads the same weights: cached.  us, whole block in 128-slot
    // blocks, logits with a spread of 1.5 per expert, non-temporally / cached (and with fp8_tile.h): 256 experts, hidden 7168,
    // inter 2048 at 80 slots 2190 / 1928 (2107); 64, 7168, 2048 at 104 663 / 597 (626); 128, 2944, 768 at 80 291 / 257 (274).
    // Even routing, where a full block is its expert's only one: level (2182 / 2198, 610 / 625, 261 / 261).  (Full 256-slot blocks
    // come here where tile_full is 0.)
    constexpr bool CACHED = DENSE ? SHORT_K : RT == RT_MAX;
    const uint32_t sv = s_voff, wv = w_voff;  // (an assembly operand in a lambda inside a generic lambda is no capture)
    static_assert(D * (GROUP_LOADS + 1) < 64, "vmcnt is a 6-bit counter");

    uint32_t a_voff[AL], a_dst[AL];
#pragma unroll
    for (int i = 0; i < AL; ++i) {
      uint32_t hh = wave + WAVES * i;
      // wavefronts without a group left fetch one that is fetched anyway, so that all issue the same number
      if (hh >= 2 * RT) hh = i ? hh - WAVES : hh % (2 * RT);
      a_voff[i] = row_of(hh * 8 + (lane >> 3)) * p.K + 16 * ((lane & 7) ^ (lane >> 3));
      a_dst[i] = __builtin_amdgcn_readfirstlane(lds_base + hh * (FRAG / 2));
    }
    const uint32_t s_dst = __builtin_amdgcn_readfirstlane(lds_base + SC_BASE + wave * 256);
    const uint32_t s4_dst = __builtin_amdgcn_readfirstlane(lds_base + SC_BASE + wave * 1024);

    f32x4 acc[2][RT];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < RT; ++i) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    i32x4 ring[D][2][2];  // [k-block % D][strip][half]

    // (every group of loads is one assembly statement that opens with s_nop 4: see fp8_tile.h)
    auto load_a = [&](uint32_t kb, int slot) {
      const uint8_t* src = a_base + static_cast<size_t>(kb) * 128;
      if (p.scales4) {
        if (kb % 4 == 0 && wave < 4 && wave * 64 < 16 * RT) {
          const char* sp = s_base + kb * 4;
          const uint32_t d = s4_dst + (kb & 4 ? SC4 : 0);
          asm volatile("s_nop 4\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" ::"v"(sv), "s"(d), "s"(sp) : "memory", "m0");
        }
      } else if (wave < 4) {
        const char* sp = s_base + static_cast<size_t>(kb) * p.as_kb_bytes;
        asm volatile("s_nop 4\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, %2" ::"v"(sv), "s"(s_dst + slot * 1024), "s"(sp)
                     : "memory", "m0");
      }
#pragma unroll
      for (int i = 0; i < AL; ++i)
        asm volatile("s_nop 4\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" ::"v"(a_voff[i]), "s"(a_dst[i] + slot * SLOT),
                     "s"(src)
                     : "memory", "m0");
    };
    auto load_w = [&](uint32_t kb, i32x4 (&dst)[2][2]) {
      const uint8_t* w0 = w_base[0] + static_cast<size_t>(kb) * FRAG;
      const uint8_t* w1 = w_base[1] + static_cast<size_t>(kb) * FRAG;
      if constexpr (CACHED)
        asm volatile(
            "s_nop 4\n\t"
            "global_load_dwordx4 %0, %4, %5\n\t"
            "global_load_dwordx4 %1, %4, %5 offset:1024\n\t"
            "global_load_dwordx4 %2, %4, %6\n\t"
            "global_load_dwordx4 %3, %4, %6 offset:1024"
            : "=&v"(dst[0][0]), "=&v"(dst[0][1]), "=&v"(dst[1][0]), "=&v"(dst[1][1])
            : "v"(wv), "s"(w0), "s"(w1)
            : "memory");
      else
        asm volatile(
            "s_nop 4\n\t"
            "global_load_dwordx4 %0, %4, %5 nt\n\t"
            "global_load_dwordx4 %1, %4, %5 offset:1024 nt\n\t"
            "global_load_dwordx4 %2, %4, %6 nt\n\t"
            "global_load_dwordx4 %3, %4, %6 offset:1024 nt"
            : "=&v"(dst[0][0]), "=&v"(dst[0][1]), "=&v"(dst[1][0]), "=&v"(dst[1][1])
            : "v"(wv), "s"(w0), "s"(w1)
            : "memory");
    };
    auto wait = [&](auto n) { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(n)::value) : "memory"); };
    // the registers of k-block h became valid with the wait in front of this statement (volatile statements keep their order)
    auto tie = [&](i32x4 (&w)[2][2]) { asm volatile("" : "+v"(w[0][0]), "+v"(w[0][1]), "+v"(w[1][0]), "+v"(w[1][1])::"memory"); };

    auto compute = [&](const i32x4 (&w)[2][2], uint32_t kb, int slot) {
      const char* act = lds + slot * SLOT;
      // (per k-block: row r at float r of its slot; by four: row r at float 4r + kb % 4)
      const bool by4 = p.scales4;
      const float* as = reinterpret_cast<const float*>(lds + SC_BASE + (by4 ? (kb & 4 ? SC4 : 0) + (kb & 3) * 4 : slot * 1024)) + (by4 ? 4 * lrow : lrow);
      const uint32_t as_step = by4 ? 64 : 16;
      auto read_frag = [&](int i) {
        const i32x4 lo = *reinterpret_cast<const i32x4*>(act + i * FRAG + rd_lo);
        const i32x4 hi = *reinterpret_cast<const i32x4*>(act + i * FRAG + rd_hi);
        return i32x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      };
      constexpr int PF = 2;  // fragments read ahead
      i32x8 af[PF + 1];
#pragma unroll
      for (int i = 0; i < PF && i < RT; ++i) af[i] = read_frag(i);
      float sc[RT];
      const float bs = bs_lds[kb], bs_up = PAIRED ? bs_lds[KB + kb] : bs;
#pragma unroll
      for (int i = 0; i < RT; ++i) sc[i] = PAIRED ? as[i * as_step] : as[i * as_step] * bs;
      const i32x8 wf[2] = {
          {w[0][0].x, w[0][0].y, w[0][0].z, w[0][0].w, w[0][1].x, w[0][1].y, w[0][1].z, w[0][1].w},
          {w[1][0].x, w[1][0].y, w[1][0].z, w[1][0].w, w[1][1].x, w[1][1].y, w[1][1].z, w[1][1].w}};
      __builtin_amdgcn_sched_barrier(0x4);
      f32x4 tmp[3];
      const f32x4 zero{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 2 * RT + 2; ++j) {
        const int i = j / 2, t = j % 2;
        if (j < 2 * RT) {
          if (t == 0 && i + PF < RT) af[(i + PF) % (PF + 1)] = read_frag(i + PF);
          tmp[j % 3] = mfma_fp8_k128(wf[t], af[i % (PF + 1)], zero);
        }
        __builtin_amdgcn_sched_barrier(0x4);
        if (j >= 2) {  // the MFMA issued two places earlier has left the pipeline by now
          const int pi = (j - 2) / 2, pt = (j - 2) % 2;
          const f32x4 r = tmp[(j - 2) % 3];
          const float f = PAIRED ? sc[pi] * (pt ? bs_up : bs) : sc[pi];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[pt][pi][e] = __builtin_fmaf(r[e], f, acc[pt][pi][e]);
          // (stays here: sunk behind the branches of the schedule below, the FMAs would keep every result of the stage alive)
          asm volatile("" : "+v"(acc[pt][pi]));
        }
        __builtin_amdgcn_sched_barrier(0x4);
      }
    };

    // ---- schedule.  Stage c multiplies k-block c; then the weights of k-block c+D are loaded into the registers it leaves,
    // then this wavefront's activation loads of k-block c+1 have to have landed, and behind the barrier those of k-block c+D
    // go out into the slot that every wavefront has left.  Loads are issued in the order w(0) a(0) w(1) a(1) ...; what may
    // be outstanding when a(c+1) has to be in is w(c+2) a(c+2) .. w(c+D), the last D k-blocks short of what was not issued.
    const uint32_t first = KB < static_cast<uint32_t>(D) ? KB : D;
#pragma unroll
    for (int h = 0; h < D; ++h) {
      if (static_cast<uint32_t>(h) < first) {
        load_w(h, ring[h]);
        load_a(h, h);
      }
    }
    using Full = std::integral_constant<int, (D - 1) * GROUP_LOADS>;       // k-blocks 1 .. D-1 may be outstanding
    using Steady = std::integral_constant<int, (D - 2) * GROUP_LOADS + 4>;
    using Tail = std::integral_constant<int, (D - 2) * GROUP_LOADS>;
    using None = std::integral_constant<int, 0>;
    if (first == D) wait(Full{}); else wait(None{});
    tie(ring[0]);
    __builtin_amdgcn_s_barrier();
    for (uint32_t c0 = 0; c0 < KB; c0 += D) {
#pragma unroll
      for (int h = 0; h < D; ++h) {
        const uint32_t c = c0 + h;
        if (c < KB) {
          compute(ring[h], c, h);
          if (c + D < KB) {
            load_w(c + D, ring[h]);
            wait(Steady{});
          } else if (c + D == KB) {
            wait(Tail{});
          } else {
            wait(None{});
          }
          tie(ring[(h + 1) % D]);
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wavefront's reads of the slot have returned
          __builtin_amdgcn_s_barrier();
          if (c + D < KB) load_a(c + D, h);
        }
      }
    }
    // nothing is outstanding here: the last stages waited for everything

    // ---- store: lane holds token m = l%16 of the tile and weight rows (output columns) 4*(l/16) .. +3
    if constexpr (PAIRED) {
      // LDS: the largest value of each row in each wavefront's 16 channels, then the codes, 128 to a row
      float* const row_max = reinterpret_cast<float*>(lds);
      char* const codes = lds + RT * 16 * WAVES * 4;
      constexpr int PITCH = 128 + 16;
      auto pair = [&](int i, float (&v)[4]) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[e] = TO::to_float(TO::from_float(silu_mul_f32(TO::to_float(TO::from_float(acc[0][i][e])), TO::to_float(TO::from_float(acc[1][i][e])))));
      };
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        float v[4];
        pair(i, v);
        float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
        amax = fmaxf(amax, __shfl_xor(amax, 16));
        amax = fmaxf(amax, __shfl_xor(amax, 32));
        if (lq == 0) row_max[(i * 16 + lrow) * WAVES + wave] = amax;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[0][i][e] = v[e];
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        float amax = 1e-10f;
        const f32x4* const m = reinterpret_cast<const f32x4*>(row_max + (i * 16 + lrow) * WAVES);
#pragma unroll
        for (int e = 0; e < 4; ++e) amax = fmaxf(amax, fmaxf(m[0][e], m[1][e]));
        const float scale = fp8_group_scale<false>(amax);
        const float v[4] = {acc[0][i][0], acc[0][i][1], acc[0][i][2], acc[0][i][3]};
        *reinterpret_cast<uint32_t*>(codes + (i * 16 + lrow) * PITCH + wave * 16 + 4 * lq) = fp8_encode4<false>(ExactDiv(scale), v);
        const uint32_t row = ids[i * 16 + lrow];
        if (wave == (static_cast<uint32_t>(i) & 7) && lq == 0 && row < p.numel) p.out_s[static_cast<size_t>(row) * (p.N / 256) + tile_n] = scale;
      }
      __syncthreads();
      for (uint32_t e = threadIdx.x; e < RT * 16 * 8; e += 512) {
        const uint32_t r = e / 8, c = e % 8, row = ids[r];
        if (row < p.numel)
          *reinterpret_cast<u32x4*>(static_cast<uint8_t*>(p.out) + static_cast<size_t>(row) * (p.N / 2) + tile_n * 128 + c * 16) =
              *reinterpret_cast<const u32x4*>(codes + r * PITCH + c * 16);
      }
      return;
    }
    if constexpr (DENSE) {
      if (!direct || p.out32) {
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          const uint32_t r = i * 16 + lrow;
          if (ids[r] < p.numel) {
            float* const dst = direct ? p.out32 + static_cast<size_t>(m0 + r) * p.N + n0
                                      : p.partial + ((static_cast<size_t>(out_slot) * p.splits + part) * p.block + r) * BN;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
              const uint32_t col = wave * 32 + t * 16 + 4 * lq;
              if (n0 + col < p.N) *reinterpret_cast<f32x4*>(dst + col) = acc[t][i];
            }
          }
        }
        return;
      }
    }
    // Rounded results go through LDS (whose slots nothing reads any more), so that a row's 256 columns leave in
    // 16-byte pieces of consecutive lanes.
    float rws[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const uint32_t sid = ids[i * 16 + lrow];
      rws[i] = (!DENSE && sid < p.numel && p.topk_w) ? p.topk_w[sid] : 1.0f;
    }
    constexpr int PITCH = kFp8StreamOutPitch;
    constexpr int PIECES = BN / 8;  // 16-byte pieces of a row
#pragma unroll
    for (int i0 = 0; i0 < RT; i0 += kFp8StreamOutTiles) {
      if (i0) __syncthreads();
#pragma unroll
      for (int j = 0; j < kFp8StreamOutTiles && i0 + j < RT; ++j) {
        const int i = i0 + j;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const f32x4 v = acc[t][i] * rws[i];
          u32x2 o;
          o.x = pack2(TO::from_float(v[0]), TO::from_float(v[1]));
          o.y = pack2(TO::from_float(v[2]), TO::from_float(v[3]));
          *reinterpret_cast<u32x2*>(lds + (j * 16 + lrow) * PITCH + (wave * 32 + t * 16 + 4 * lq) * 2) = o;
        }
      }
      __syncthreads();
      const uint32_t out_rows = (RT - i0 < kFp8StreamOutTiles ? RT - i0 : kFp8StreamOutTiles) * 16;
      for (uint32_t e = threadIdx.x; e < out_rows * PIECES; e += 512) {
        const uint32_t r = e / PIECES, c = e % PIECES;
        const uint32_t row = ids[i0 * 16 + r];
        if (row < p.numel && n0 + c * 8 < p.N)
          __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(lds + r * PITCH + c * 16),
                                      reinterpret_cast<u32x4*>(static_cast<uint16_t*>(p.out) + static_cast<size_t>(row) * p.N + n0 + c * 8));
      }
    }
  };
  for_tile_count<DENSE ? 9 : 1, DENSE ? kFp8StreamDenseTiles : RT_MAX>(live_tiles, run);  // (dense: 129..240 rows)
}

}  // namespace ksq
