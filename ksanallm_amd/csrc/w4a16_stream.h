// W4A16 kernel for the 32-slot row blocks of int4 experts, whose time is the stream of their weights out of HBM: a workgroup of
// eight wavefronts side by side along N computes up to 32 rows x 256 columns over all of K.
//
//   - every weight tile belongs to one wavefront (two strips of 16 columns each), which loads it straight into a register ring
//     of four k-tiles: 64 KiB in flight per workgroup, two workgroups to a CU.  Non-temporally, for a weight is read once,
//     unless its expert has several blocks, which run at the same time and share a cached copy: the L2's where the columns are a
//     multiple of eight workgroups (the same columns of the next block are then on the same XCD), the Infinity Cache's otherwise.
//     32 / 48 slots each, non-temporal / cached, us: 256 experts, n = 4096, k = 7168 (16 column workgroups) 1002 / 942, 1410 / 1273, n =
//     7168, k = 2048 (28) 569 / 526, 777 / 707; 64, n = k = 5120 (20) 250 / 226, 352 / 305; n = 3072, k = 4096 (12) 125 / 125, 173 / 168.
//   - x goes global -> LDS (global_load_lds_dwordx4) by halves of two k-tiles, three halves ahead; all wavefronts read it from
//     there.  A strip's scales of a half are 64 contiguous bytes and come the same way, one load for a wavefront's strips.
//   - the sums of x that make up for the codes' offset are taken once per workgroup, a half ahead, and handed round through
//     LDS (each wavefront for itself they are a third of the MFMAs: 1-3 %).
//   - all loads are issued from inline assembly in a fixed order and number, so that every wait has a constant count and leaves
//     the ring in flight, also across the one barrier per half.
// The decode kernel (w4a16_splitk.h), four wavefronts that divide K among them, keeps 64 KiB per CU in flight at best, waits for
// more of it than it needs (the compiler's counts do not know the staging loads) and fetches x twice as often.  512 tokens,
// 256 experts, hidden 7168, inter 2048, bf16, GEMMs alone: the first 663 -> 618 us (6.3 TB/s), the second 415 -> 362 us, whole block 1140 ->
// 1066 (single launches behind a write of 600 MiB, in one session: 841 -> 816 and 475 -> 420);
// with weights out of the L2 484 -> 400 and 326 -> 222 (one row tile), 634 -> 562 and 417 -> 326 (two): what the SIMDs take to
// issue it, about 1.4 times the unpacking (28 instructions a tile), scaling and MFMAs added up.  Measured against it and not
// kept: four strips to a wavefront and four wavefronts, 594 / 369 us; eight of those, one workgroup to a CU, 603 / 388; two
// strips, four wavefronts 664 / 393; 64 rows to a workgroup, one to a CU, ahead at 32 slots a block (1.47 ms) and behind elsewhere.
//
// The arithmetic is that of w4a16_splitk.h (codes as exact integers, the scale on the fp32 result of a group, the offset
// through an MFMA against a constant operand); the sums run over k in one order instead of one per wavefront.
#pragma once

#include "ksq_common.h"
#include "w4a16_splitk.h"

namespace ksq {

constexpr int kW4StreamRows = 32;              // slots of a row block
constexpr int kW4StreamPairPitch = 1024 + 16;  // two rows of x, two k-tiles each, in LDS (the padding spreads rows over the banks)
// four slots of x and of every wavefront's scales, sums of x, slot ids
constexpr int kW4StreamLds = 4 * (kW4StreamRows / 2 * kW4StreamPairPitch + 8 * 256) + 512 + kW4StreamRows * 4;

int launch_w4a16_stream(const SplitKParams& p, bool paired, uint32_t m_blocks, int dtype, hipStream_t s);

// PAIRED: gate / up weights [2 * inter, K]; a wavefront holds a gate strip and the matching up strip, and
// out[s, c] = T(silu(T(gate)) * T(up)) is [numel, N / 2].
template <typename T, bool PAIRED>
__global__ void __launch_bounds__(512, 4) w4a16_stream_tile_kernel(SplitKParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];  // kW4StreamLds
  constexpr int NS = 2, WAVES = 8;  // strips of a wavefront, wavefronts
  constexpr int PITCH = kW4StreamPairPitch;
  constexpr int SLOT = kW4StreamRows / 2 * PITCH;
  constexpr int SC_BASE = 4 * SLOT;
  constexpr int SC_SLOT = WAVES * 256;
  constexpr int SX_BASE = SC_BASE + 4 * SC_SLOT;
  constexpr int IDS_BASE = SX_BASE + 512;
  constexpr int OS = PAIRED ? NS / 2 : NS;  // output strips of a wavefront
  const int lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lrow = lane & 15, lq = lane >> 4;
  const uint32_t KT = p.K / 128, strips = p.N / 16;
  const uint32_t out_strips = PAIRED ? strips / 2 : strips;

  const uint32_t pos0 = blockIdx.y * kW4StreamRows, slots = static_cast<uint32_t>(p.num_post_pad[0]);
  if (pos0 >= slots) return;  // uniform: the whole workgroup leaves
  const uint32_t e = __builtin_amdgcn_readfirstlane(p.expert_ids[blockIdx.y]);
  const size_t expert = e;
  // slots of the block (they come first, pad slots behind them): lane l holds slot l % 32
  const uint32_t sid = static_cast<uint32_t>(p.sorted_ids[pos0 + (lane & 31)]);
  const uint32_t nrows = __builtin_amdgcn_readfirstlane(__builtin_popcountll(__builtin_amdgcn_ballot_w64(lane < 32 && sid < p.numel)));
  if (nrows == 0) return;
  if (threadIdx.x < kW4StreamRows) reinterpret_cast<uint32_t*>(smem + IDS_BASE)[threadIdx.x] = sid;
  const uint32_t src_row_v = sid < p.numel ? sid / p.top_k : 0;

  // strips of this wavefront; those past the end repeat the last one, and their results are not stored
  const uint32_t ostrip0 = (blockIdx.x * WAVES + wave) * OS;
  uint32_t strip[NS];
#pragma unroll
  for (int t = 0; t < NS; ++t) {
    const uint32_t o = ostrip0 + t % OS;
    strip[t] = (o < out_strips ? o : out_strips - 1) + (t / OS) * out_strips;
  }
  const char* w_base[NS];
#pragma unroll
  for (int t = 0; t < NS; ++t)
    w_base[t] = scalar_ptr(static_cast<const char*>(p.w) + (expert * strips + strip[t]) * static_cast<size_t>(KT) * 1024);
  const char* const s_base = scalar_ptr(static_cast<const char*>(p.scales) + expert * strips * static_cast<size_t>(KT) * 32);
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<size_t>((__attribute__((address_space(3))) char*)smem));
  const uint32_t w_voff = lane * 16;
  const char* const x_base = static_cast<const char*>(p.x);

  // an expert with several blocks (they run side by side and share a cached copy of the weights)
  const bool several = (pos0 + kW4StreamRows < slots && static_cast<uint32_t>(p.expert_ids[blockIdx.y + 1]) == e) ||
                       (blockIdx.y > 0 && static_cast<uint32_t>(p.expert_ids[blockIdx.y - 1]) == e);
  // A strip is K / 128 KiB, so where K is a multiple of 4096 the strips of all workgroups start on the same HBM channels, where it is
  // one of 2048 on one of two sets of them, and the workgroups walk over the channels in step.  There an expert starts at a place
  // of its own and goes round (the same one for all its columns, which share x in the L2, and for all its blocks).  us, from k-tile 0
  // by all / with this: 64 experts of n = k = 4096 at 8, 16, 20, 32 rows 118 / 98, 121 / 108, 131 / 118, 146 / 142 (decode kernel 107,
  // 114, 122, 168); n = 4096, k = 2048 at 8 and 20 61 / 53, 70 / 66; gate / up with n = k = 4096, 256 experts at 8 393 / 371, 16 at 16
  // 34 / 31; whole int4 block, 16 experts of hidden 4096, inter 2048 at 16 66 / 59 (decode kernel 58).  With k = 2048 and several blocks to
  // an expert it is 3-5 % behind (256 experts, n = 7168 at 32 rows 529 / 547); per workgroup instead of per expert it
  // loses 3-9 % from 20 rows on, as every column then reads x at another place.
  const bool spread = KT % 32 == 0 || (KT % 16 == 0 && !several);
  const uint32_t first_kt = __builtin_amdgcn_readfirstlane(spread ? 2 * (5 * e % (KT / 2)) : 0);
  auto k_tile = [&](uint32_t i) { return i + first_kt < KT ? i + first_kt : i + first_kt - KT; };  // k-tile of place i

  uint32_t magic2 = p.magic2;
  asm volatile("" : "+v"(magic2));  // no instruction: keeps the value in a VGPR so that and / or fold into one instruction
  const uint32_t nmask = p.nibble_mask;
  auto run = [&](auto rt_c, auto cached_c) __attribute__((always_inline)) {
    constexpr int RT = decltype(rt_c)::value;
    constexpr bool CACHED = decltype(cached_c)::value;
    constexpr int XL = 8 * RT / WAVES;  // pairs of rows of x that a wavefront stages per half
    constexpr int S = XL + 1;           // staging loads of a wavefront per half: those and the scales
    // x load i: lanes 0-31 take row 2r of the pair r = wave + WAVES * i, lanes 32-63 row 2r + 1; 16-byte piece q of an odd row
    // lies at place q ^ 8, so that sixteen rows read at once touch sixteen different bank groups
    const uint32_t x_piece = (lane & 31) ^ (lane < 32 ? 0 : 8);
    uint32_t x_off[XL], x_dst[XL];
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const uint32_t r = wave + WAVES * i, r0 = 2 * r < nrows ? 2 * r : 0, r1 = 2 * r + 1 < nrows ? 2 * r + 1 : 0;
      // rows without a slot repeat the block's first
      const uint32_t row0 = __builtin_amdgcn_readlane(static_cast<int>(src_row_v), static_cast<int>(r0));
      const uint32_t row1 = __builtin_amdgcn_readlane(static_cast<int>(src_row_v), static_cast<int>(r1));
      x_off[i] = (lane < 32 ? row0 : row1) * p.K * 2;  // (x spans less than 1 GiB)
      x_dst[i] = __builtin_amdgcn_readfirstlane(lds_base + r * PITCH);
    }
    // scale load: 64 bytes (two k-tiles) of each strip to sixteen lanes (with two strips the upper lanes repeat them)
    const uint32_t st = (lane >> 4) % NS, so = ostrip0 + st % OS;
    const uint32_t s_strip = (so < out_strips ? so : out_strips - 1) + st / OS * out_strips;
    const uint32_t s_off = s_strip * KT * 32;
    const uint32_t s_byte = (lane & 15) * 4, s_last = (KT - 1) * 32 + (lane & 7) * 4;
    const uint32_t s_dst = __builtin_amdgcn_readfirstlane(lds_base + SC_BASE + wave * 256);

    // half h -> LDS slot h % 4 (assembly statements open with s_nop 4: scalar operands that a v_readfirstlane produced need
    // five wait states before a vector memory instruction reads them, and the compiler inserts none inside a statement)
    auto stage = [&](uint32_t to) __attribute__((always_inline)) {
      const uint32_t kt = k_tile(2 * to < KT ? 2 * to : 0);  // (a half past the end, of a short K, repeats the first; nothing uses it)
      const uint32_t left = (KT - kt) * 16;  // pieces of a row from this half on; lanes past them re-read the first
      const uint32_t xv = (x_piece < left ? x_piece : 0) * 16 + kt * 256;
      const char* const xs = x_base;
      const char* const sb = s_base;
#pragma unroll
      for (int i = 0; i < XL; ++i)
        asm volatile("s_nop 4\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" ::"v"(x_off[i] + xv), "s"(x_dst[i] + (to & 3) * SLOT),
                     "s"(xs)
                     : "memory", "m0");
      const uint32_t o = kt * 32 + s_byte;
      asm volatile("s_nop 4\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, %2" ::"v"(s_off + (o < s_last ? o : s_last)),
                   "s"(s_dst + (to & 3) * SC_SLOT), "s"(sb)
                   : "memory", "m0");
    };
    u32x4 ring[4][NS];
    auto load_w = [&](uint32_t kt, u32x4 (&dst)[NS]) __attribute__((always_inline)) {  // (k-tiles past the end: 16 bytes of the last one)
      const uint32_t o = k_tile(kt < KT ? kt : KT - 1) * 1024, wv = kt < KT ? w_voff : 0;
#pragma unroll
      for (int t = 0; t < NS; t += 2) {
        const char *const w0 = w_base[t] + o, *const w1 = w_base[t + 1] + o;
        if constexpr (CACHED)
          asm volatile(
              "s_nop 4\n\t"
              "global_load_dwordx4 %0, %2, %3\n\t"
              "global_load_dwordx4 %1, %2, %4"
              : "=&v"(dst[t]), "=&v"(dst[t + 1])
              : "v"(wv), "s"(w0), "s"(w1)
              : "memory");
        else
          asm volatile(
              "s_nop 4\n\t"
              "global_load_dwordx4 %0, %2, %3 nt\n\t"
              "global_load_dwordx4 %1, %2, %4 nt"
              : "=&v"(dst[t]), "=&v"(dst[t + 1])
              : "v"(wv), "s"(w0), "s"(w1)
              : "memory");
      }
    };
    auto wait = [&](auto n) { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(n)::value) : "memory"); };
    // the registers of a k-tile became valid with the wait in front of this statement (volatile statements keep their order)
    auto tie = [&](u32x4 (&w)[NS]) {
#pragma unroll
      for (int t = 0; t < NS; t += 2) asm volatile("" : "+v"(w[t]), "+v"(w[t + 1])::"memory");
    };

    f32x4 acc[NS][RT];
#pragma unroll
    for (int t = 0; t < NS; ++t)
#pragma unroll
      for (int i = 0; i < RT; ++i) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    // fragment d of row tile i of the half's k-tile j: lane (row, quarter) reads 16 bytes
    const uint32_t rd = (lrow >> 1) * PITCH + (lrow & 1) * (512 + 128) + lq * 16, rd_hi = rd + 128 - (lrow & 1) * 256;
    auto read_x = [&](uint32_t h, int j, int d0, u32x4 (&f)[RT][2]) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int d = 0; d < 2; ++d)
          f[i][d] = *reinterpret_cast<const u32x4*>(smem + (h & 3) * SLOT + i * 8 * PITCH + j * 256 + (d0 < 2 ? rd : rd_hi) + d * 64);
    };
    // -(magic + 8) * sum(x) of the half's rows and k-tiles, which all wavefronts start a group's sum from: each computes one
    // row tile and k-tile and hands it round through LDS
    auto sum_x = [&](uint32_t h) __attribute__((always_inline)) {
      const uint32_t cb = wave % (2 * RT);  // (without a branch: a loop of several basic blocks does not fit the registers)
      const char* const b = smem + (h & 3) * SLOT + (cb >> 1) * (8 * PITCH) + (cb & 1) * 256;
      const typename T::frag neg = as_frag<T>(u32x4{T::kNegSym2, T::kNegSym2, T::kNegSym2, T::kNegSym2});
      f32x4 r{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < 4; ++d) r = T::mfma(as_frag<T>(*reinterpret_cast<const u32x4*>(b + (d < 2 ? rd : rd_hi) + (d & 1) * 64)), neg, r);
      // (all sixteen columns hold the same: the lanes of a row quarter, and two or more wavefronts, store one value to one place)
      *reinterpret_cast<f32x4*>(smem + SX_BASE + ((h & 1) * 4 + cb) * 64 + lq * 16) = r;
    };
    // (two of a k-tile's four k-steps at a time: the registers hold no more)
    auto multiply = [&](const u32x4 (&w)[NS], const u32x4 (&xf)[RT][2], int d0, f32x4 (&r)[NS][RT]) __attribute__((always_inline)) {
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int t = 0; t < NS; ++t) {
          const typename T::frag wf = dequant_magic_fast<T>(w[t][d0 + d], nmask, magic2);
#pragma unroll
          for (int i = 0; i < RT; ++i) r[t][i] = T::mfma(as_frag<T>(xf[i][d]), wf, r[t][i]);
        }
    };
    auto compute = [&](const u32x4 (&w)[NS], uint32_t h, int j, const u32x4 (&x_lo)[RT][2]) __attribute__((always_inline)) {
      f32x4 r[NS][RT];
      u32x4 x_hi[RT][2];
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const f32x4 sx = *reinterpret_cast<const f32x4*>(smem + SX_BASE + ((h & 1) * 4 + i * 2 + j) * 64 + lq * 16);
#pragma unroll
        for (int t = 0; t < NS; ++t) r[t][i] = sx;
      }
      read_x(h, j, 2, x_hi);
      multiply(w, x_lo, 0, r);
      multiply(w, x_hi, 2, r);
      const char* const sb = smem + SC_BASE + (h & 3) * SC_SLOT + wave * 256 + j * 32 + lrow * 2;
#pragma unroll
      for (int t = 0; t < NS; ++t) {
        const float s = T::lo_to_float(*reinterpret_cast<const uint16_t*>(sb + t * 64));
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[t][i][e] = __builtin_fmaf(s, r[t][i][e], acc[t][i][e]);
      }
    };

    // ---- schedule, by halves of two k-tiles.  Half h: x and scales of half h + 1 have landed (its sums of x are taken behind
    // the barrier), those of half h + 3 are issued into the slot that half h - 1 left, and w(2h + 4 + j) goes into the
    // registers that k-tile 2h + j leaves.  Loads are issued in the order stage(1) w(0) w(1) stage(2) w(2) w(3) stage(3) ..:
    // behind stage(h + 1) are w(2h) w(2h+1) stage(h+2) w(2h+2) w(2h+3), behind w(2h + j) three k-tiles and two stages.
    // The last three halves issue less and count less.
    auto half = [&](auto parity_c, auto step_c, uint32_t h) __attribute__((always_inline)) {
      constexpr int PAR = decltype(parity_c)::value;
      constexpr int STEP = decltype(step_c)::value;  // 0: steady; 1, 2, 3: the last three
      constexpr int AT_BARRIER = STEP < 2 ? 4 * NS + S : 4 * NS;
      if constexpr (STEP < 3) wait(std::integral_constant<int, AT_BARRIER>{});
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if constexpr (STEP == 0) stage(h + 3);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        u32x4(&w)[NS] = ring[2 * PAR + j];
        if constexpr (STEP == 0) {
          u32x4 x_lo[RT][2];
          read_x(h, j, 0, x_lo);
          wait(std::integral_constant<int, 3 * NS + 2 * S>{});
          tie(w);
          compute(w, h, j, x_lo);
        } else {
          if constexpr (STEP == 1) wait(std::integral_constant<int, 3 * NS + S>{});
          if constexpr (STEP == 2) {
            if (j == 0) wait(std::integral_constant<int, 3 * NS>{}); else wait(std::integral_constant<int, 2 * NS>{});
          }
          if constexpr (STEP == 3) {
            if (j == 0) wait(std::integral_constant<int, NS>{}); else wait(std::integral_constant<int, 0>{});
          }
          tie(w);
          if (2 * h + j < KT) {
            u32x4 x_lo[RT][2];
            read_x(h, j, 0, x_lo);
            compute(w, h, j, x_lo);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (STEP < 2) load_w(2 * h + 4 + j, w);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (STEP < 3) sum_x(h + 1);
    };
    using Even = std::integral_constant<int, 0>;
    using Odd = std::integral_constant<int, 1>;
    stage(0);
    stage(1);
    load_w(0, ring[0]);
    load_w(1, ring[1]);
    stage(2);
    load_w(2, ring[2]);
    load_w(3, ring[3]);
    wait(std::integral_constant<int, 2 * S + 4 * NS>{});
    __syncthreads();  // (the slot ids too)
    sum_x(0);
    // (an odd number of halves, so that the ring's registers have one way through the loop; the halves and k-tiles past the
    // end are loaded, in part, but not used)
    const uint32_t halves = (KT + 1) / 2 > 3 ? (KT + 1) / 2 | 1 : 3;
    uint32_t h = 0;
    for (; h + 3 < halves; h += 2) {
      half(Even{}, Even{}, h);
      half(Odd{}, Even{}, h + 1);
    }
    half(Even{}, std::integral_constant<int, 1>{}, h);
    half(Odd{}, std::integral_constant<int, 2>{}, h + 1);
    half(Even{}, std::integral_constant<int, 3>{}, h + 2);

    // ---- store: lane holds column l % 16 of a strip and rows 4 * (l / 16) .. +3
    u32x4 ids[RT];
    f32x4 rw[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) ids[i] = *reinterpret_cast<const u32x4*>(smem + IDS_BASE + (i * 16 + 4 * lq) * 4);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) rw[i][e] = (!PAIRED && ids[i][e] < p.numel && p.topk_w) ? p.topk_w[ids[i][e]] : 1.0f;
    const uint32_t out_n = out_strips * 16;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (ids[i][e] >= p.numel) continue;
        uint16_t* const dst = static_cast<uint16_t*>(p.y) + static_cast<size_t>(ids[i][e]) * out_n + ostrip0 * 16 + lrow;
#pragma unroll
        for (int t = 0; t < OS; ++t) {
          if (ostrip0 + t >= out_strips) continue;
          if constexpr (PAIRED)
            dst[t * 16] = T::from_float(silu_mul_f32(T::to_float(T::from_float(acc[t][i][e])), T::to_float(T::from_float(acc[t + OS][i][e]))));
          else
            dst[t * 16] = T::from_float(acc[t][i][e] * rw[i][e]);
        }
      }
  };
  if (several)
    for_tile_count<1, 2>((nrows + 15) / 16, [&](auto rt_c) __attribute__((always_inline)) { run(rt_c, std::true_type{}); });
  else
    for_tile_count<1, 2>((nrows + 15) / 16, [&](auto rt_c) __attribute__((always_inline)) { run(rt_c, std::false_type{}); });
}

}  // namespace ksq
