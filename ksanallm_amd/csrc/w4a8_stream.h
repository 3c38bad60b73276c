// W4A8 kernel for one row block of 33 to 128 tokens: a workgroup of eight wavefronts side by side along N computes up to 128 tokens x
// 128 * NS columns over a range of 128-deep k-blocks.  NS = 2 runs under the tile kernel's plan (w4a8_tile.h) and with its bits; NS = 1, up
// to 64 tokens, has workgroups of 128 columns over all of K, whatever that plan cuts, and so its own grid and one order of the sums.
//
//   - weights and their scales go straight into a register ring of D k-blocks, each fragment to the one wavefront that
//     multiplies it (NS strips of 16 columns each); activations (whole 128-byte lines) and group sums go global -> LDS into D
//     slots that hold the row tiles with tokens alone.  The weights are loaded cached: one round of workgroups is over in a
//     few ring lengths, and non-temporal loads come back later (n = 25600, k = 5120 at 40 and 64 tokens 27.1 / 30.1 us, cached
//     22.5 / 25.6).
//   - all loads are issued from inline assembly in a fixed order, so every wait has a constant count.
//   - NS = 1 is for a single round of workgroups: no partial sums, no workspace, no second launch.
// What bounds it: a launch, the ramp, and per k-block the chain of LDS reads, code expansion, MFMAs and scale FMAs in two wavefronts per
// SIMD; with NS = 2 also the pass over the partial sums where the plan cuts K, 4.4 us behind the kernel.  n = 25600, k = 5120 at 64 tokens,
// which takes NS = 1 (40 k-blocks on 200 CUs): 25.6 us as NS = 2 (20 k-blocks, reduction included), 25.0 as NS = 1; single launches behind a
// write of 600 MiB 34.5 + 4.4 (tile kernel and reduction) -> 33.4.  As NS = 2 a row tile more costs 2.5 us over 20 k-blocks; the tile kernel
// pays for all eight row tiles of its 128-token form in two of four wavefronts' time.  80 tokens (NS = 2) 33.4 -> 27.9 us, 33 tokens 26.0 ->
// 22.5, as NS = 1 21.4.  Of NS = 2 at 64 tokens: fragments read four ahead instead of two 26.9 us (25.6); the group sums read behind the
// first fragments instead of in front of them 25.6 -> 26.
#pragma once

#include "fp8_stream.h"
#include "ksq_common.h"
#include "tile_work.h"
#include "w4a8_tile.h"

namespace ksq {

constexpr int kW4A8StreamTiles = 8;  // row tiles, at most
constexpr int w4a8_stream_depth(int ns, int rt) { return ns == 1 ? 12 : rt <= 4 ? 8 : 5; }
constexpr int w4a8_stream_area(int ns, int rt) { return w4a8_stream_depth(ns, rt) * (rt * 2048 + 512); }
constexpr int w4a8_stream_lds_bytes(int ns) {
  int most = 0;
  for (int rt = 1; rt <= (ns == 1 ? 4 : kW4A8StreamTiles); ++rt) most = w4a8_stream_area(ns, rt) > most ? w4a8_stream_area(ns, rt) : most;
  return most;
}

template <typename TO, int NS>
__global__ void __launch_bounds__(512, 1) w4a8_stream_tile_kernel(W4A8TileParams p, uint32_t block) {
  extern __shared__ __attribute__((aligned(16))) char lds[];  // w4a8_stream_lds_bytes
  constexpr int WAVES = 8, BN = 16 * NS * WAVES, FRAG = 2048;
  const int lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lrow = lane & 15, lq = lane >> 4;
  const uint32_t k_blocks = p.K / 128;

  const TileWork work = tile_work(blockIdx.x, p.tiles_m, p.tiles_n, p.main_items, p.splits);
  const uint32_t tile_m = __builtin_amdgcn_readfirstlane(work.tile_m), tile_n = __builtin_amdgcn_readfirstlane(work.tile_n);
  const uint32_t part = __builtin_amdgcn_readfirstlane(work.part), out_slot = __builtin_amdgcn_readfirstlane(work.slot);
  const bool direct = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(work.direct)) != 0;
  const uint32_t m0 = tile_m * block, n0 = tile_n * BN;
  const uint32_t rows = p.M - m0 < block ? p.M - m0 : block;
  // the k-blocks of this workgroup: kb0 .. kb0 + KB - 1
  const uint32_t kb0 = __builtin_amdgcn_readfirstlane(direct ? 0 : part * p.kb_per_split);
  const uint32_t KB = __builtin_amdgcn_readfirstlane(direct || k_blocks - kb0 < p.kb_per_split ? k_blocks - kb0 : p.kb_per_split);

  const uint8_t* a_base = scalar_ptr(p.a + static_cast<size_t>(m0) * p.K + static_cast<size_t>(kb0) * 128);
  const float* x_base = scalar_ptr(p.xsum + static_cast<size_t>(kb0) * p.M + m0);
  const uint32_t strips = p.N / 16;
  const uint8_t* w_base[NS];  // (strips past N repeat the last one; their results are not stored)
  const uint16_t* sc_base[NS];
#pragma unroll
  for (int t = 0; t < NS; ++t) {
    const uint32_t s = n0 / 16 + wave * NS + t, strip = s < strips ? s : strips - 1;
    w_base[t] = scalar_ptr(p.w + (static_cast<size_t>(strip) * k_blocks + kb0) * 1024);
    sc_base[t] = scalar_ptr(p.sc + static_cast<size_t>(kb0) * p.N + strip * 16);
  }
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<size_t>((__attribute__((address_space(3))) char*)lds));
  // An activation fragment (16 rows x 128 bytes) is two loads of 8 rows, eight lanes a row; piece q of row r lies at 128r + 16 *
  // (q ^ (r % 8)), so that eight lanes that read together cover all banks (fp8_stream.h).
  const uint32_t rd_lo = 128 * lrow + 16 * ((2 * lq) ^ (lrow & 7));
  const uint32_t rd_hi = rd_lo ^ 16;

  auto run = [&](auto rt_c) __attribute__((always_inline)) {
    constexpr int RT = decltype(rt_c)::value;
    constexpr int D = w4a8_stream_depth(NS, RT);
    constexpr int AL = (2 * RT + WAVES - 1) / WAVES;  // activation loads per wavefront and k-block
    // loads of a wavefront per k-block that the waits count: with two of weights and two of scales.  The group sums, which not
    // every wavefront loads, are not counted: a wait then covers one load more than it has to.
    constexpr int GROUP_LOADS = AL + 2 * NS;
    constexpr int SLOT = RT * FRAG;
    constexpr int XS_BASE = D * SLOT;
    static_assert(D * (GROUP_LOADS + 1) < 64, "vmcnt is a 6-bit counter");
    const uint32_t wv = lane * 16, scv = lq * 8;
    const uint32_t xr = (wave & 1) * 64 + lane, xv = (xr < rows ? xr : rows - 1) * 4;

    uint32_t a_voff[AL], a_dst[AL];
#pragma unroll
    for (int i = 0; i < AL; ++i) {
      uint32_t hh = wave + WAVES * i;
      // wavefronts without a group left fetch one that is fetched anyway, so that all issue the same number
      if (hh >= 2 * RT) hh = i ? hh - WAVES : hh % (2 * RT);
      const uint32_t r = hh * 8 + (lane >> 3);  // (rows past the block repeat its last; their results are not stored)
      a_voff[i] = (r < rows ? r : rows - 1) * p.K + 16 * ((lane & 7) ^ (lane >> 3));
      a_dst[i] = __builtin_amdgcn_readfirstlane(lds_base + hh * (FRAG / 2));
    }
    const uint32_t x_dst = __builtin_amdgcn_readfirstlane(lds_base + XS_BASE + (wave & 1) * 256);

    f32x4 acc[NS][RT];
#pragma unroll
    for (int t = 0; t < NS; ++t)
#pragma unroll
      for (int i = 0; i < RT; ++i) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    struct Stage {
      i32x4 w[NS];
      u32x2 sc[NS];
    };
    Stage ring[D];

    // (every group of loads is one assembly statement that opens with s_nop 4: see fp8_tile.h)
    auto load_a = [&](uint32_t kb, int slot) __attribute__((always_inline)) {
      const uint8_t* src = a_base + static_cast<size_t>(kb) * 128;
      if (wave * 64 < 16 * RT) {
        const float* xp = x_base + static_cast<size_t>(kb) * p.M;
        asm volatile("s_nop 4\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, %2" ::"v"(xv), "s"(x_dst + slot * 512), "s"(xp)
                     : "memory", "m0");
      }
#pragma unroll
      for (int i = 0; i < AL; ++i)
        asm volatile("s_nop 4\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" ::"v"(a_voff[i]), "s"(a_dst[i] + slot * SLOT),
                     "s"(src)
                     : "memory", "m0");
    };
    auto load_w = [&](uint32_t kb, Stage& s) __attribute__((always_inline)) {
      if constexpr (NS == 1) {
        const uint8_t* w0 = w_base[0] + static_cast<size_t>(kb) * 1024;
        const uint16_t* s0 = sc_base[0] + static_cast<size_t>(kb) * p.N;
        asm volatile(
            "s_nop 4\n\t"
            "global_load_dwordx4 %0, %2, %4\n\t"
            "global_load_dwordx2 %1, %3, %5"
            : "=&v"(s.w[0]), "=&v"(s.sc[0])
            : "v"(wv), "v"(scv), "s"(w0), "s"(s0)
            : "memory");
      } else {
        const uint8_t *w0 = w_base[0] + static_cast<size_t>(kb) * 1024, *w1 = w_base[NS - 1] + static_cast<size_t>(kb) * 1024;
        const uint16_t *s0 = sc_base[0] + static_cast<size_t>(kb) * p.N, *s1 = sc_base[NS - 1] + static_cast<size_t>(kb) * p.N;
        asm volatile(
            "s_nop 4\n\t"
            "global_load_dwordx4 %0, %4, %6\n\t"
            "global_load_dwordx4 %1, %4, %7\n\t"
            "global_load_dwordx2 %2, %5, %8\n\t"
            "global_load_dwordx2 %3, %5, %9"
            : "=&v"(s.w[0]), "=&v"(s.w[NS - 1]), "=&v"(s.sc[0]), "=&v"(s.sc[NS - 1])
            : "v"(wv), "v"(scv), "s"(w0), "s"(w1), "s"(s0), "s"(s1)
            : "memory");
      }
    };
    auto wait = [&](auto n) { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(n)::value) : "memory"); };
    // the registers of a k-block became valid with the wait in front of this statement (volatile statements keep their order)
    auto tie = [&](Stage& s) {
#pragma unroll
      for (int t = 0; t < NS; ++t) asm volatile("" : "+v"(s.w[t]), "+v"(s.sc[t])::"memory");
    };

    auto compute = [&](const Stage& s, int slot) __attribute__((always_inline)) {
      const char* act = lds + slot * SLOT;
      const float* xs = reinterpret_cast<const float*>(lds + XS_BASE + slot * 512) + lrow;
      auto read_frag = [&](int i) {
        const i32x4 lo = *reinterpret_cast<const i32x4*>(act + i * FRAG + rd_lo);
        const i32x4 hi = *reinterpret_cast<const i32x4*>(act + i * FRAG + rd_hi);
        return i32x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      };
      constexpr int PF = 2;  // fragments read ahead
      i32x8 af[PF + 1];
      float cs[RT];
#pragma unroll
      for (int i = 0; i < RT; ++i) cs[i] = xs[i * 16] * -0.015625f;  // -8 * 2^-9 * xsum
#pragma unroll
      for (int i = 0; i < PF && i < RT; ++i) af[i] = read_frag(i);
      float sc[NS][4];
      i32x8 wf[NS];
#pragma unroll
      for (int t = 0; t < NS; ++t) {
        sc[t][0] = F16::lo_to_float(s.sc[t].x);
        sc[t][1] = F16::hi_to_float(s.sc[t].x);
        sc[t][2] = F16::lo_to_float(s.sc[t].y);
        sc[t][3] = F16::hi_to_float(s.sc[t].y);
        wf[t] = w4a8_expand(s.w[t]);
      }
      __builtin_amdgcn_sched_barrier(0x4);
      f32x4 tmp[3];
#pragma unroll
      for (int j = 0; j < NS * RT + 2; ++j) {
        const int i = j / NS, t = j % NS;
        if (j < NS * RT) {
          if (t == 0 && i + PF < RT) af[(i + PF) % (PF + 1)] = read_frag(i + PF);
          tmp[j % 3] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[t], af[i % (PF + 1)], f32x4{cs[i], cs[i], cs[i], cs[i]}, 0, 0, 0, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0x4);
        if (j >= 2) {  // the MFMA issued two places earlier has left the pipeline by now
          const int pi = (j - 2) / NS, pt = (j - 2) % NS;
          const f32x4 r = tmp[(j - 2) % 3];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[pt][pi][e] = __builtin_fmaf(r[e], sc[pt][e], acc[pt][pi][e]);
          asm volatile("" : "+v"(acc[pt][pi]));  // (stays here: see fp8_stream.h)
        }
        __builtin_amdgcn_sched_barrier(0x4);
      }
    };

    // ---- schedule, as fp8_stream.h's: loads are issued in the order w(0) a(0) w(1) a(1) ..; behind stage c the weights of
    // k-block c + D go into the registers that it leaves, a(c + 1) has to have landed, and a(c + D) goes into its slot.  What may be
    // outstanding then is w(c+2) a(c+2) .. w(c+D), at the end the k-blocks that are left, in steps.
    const uint32_t first = KB < static_cast<uint32_t>(D) ? KB : D;
#pragma unroll
    for (int h = 0; h < D; ++h) {
      if (static_cast<uint32_t>(h) < first) {
        load_w(h, ring[h]);
        load_a(h, h);
      }
    }
    using None = std::integral_constant<int, 0>;
    if (first == D) wait(std::integral_constant<int, (D - 1) * GROUP_LOADS>{}); else wait(None{});
    tie(ring[0]);
    __builtin_amdgcn_s_barrier();
    for (uint32_t c0 = 0; c0 < KB; c0 += D) {
#pragma unroll
      for (int h = 0; h < D; ++h) {
        const uint32_t c = c0 + h;
        if (c < KB) {
          compute(ring[h], h);
          if (c + D < KB) {
            load_w(c + D, ring[h]);
            wait(std::integral_constant<int, (D - 2) * GROUP_LOADS + 2 * NS>{});
          } else if (c + 2 + (D - 2) / 2 < KB) {
            wait(std::integral_constant<int, (D - 2) / 2 * GROUP_LOADS>{});  // (at least (D - 2) / 2 whole k-blocks behind a(c + 1))
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

    // ---- store: lane holds token m = l%16 of the tile and output columns 4*(l/16) .. +3
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const uint32_t r = i * 16 + lrow;
      if (r < rows) {
#pragma unroll
        for (int t = 0; t < NS; ++t) {
          const uint32_t col = (wave * NS + t) * 16 + 4 * lq;
          if (n0 + col < p.N) {
            const f32x4 v = acc[t][i] * p.alpha512;
            if (direct) {
              u32x2 o;
              o.x = pack2(TO::from_float(v[0]), TO::from_float(v[1]));
              o.y = pack2(TO::from_float(v[2]), TO::from_float(v[3]));
              *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(p.out) + static_cast<size_t>(m0 + r) * p.N + n0 + col) = o;
            } else {
              *reinterpret_cast<f32x4*>(p.partial + ((static_cast<size_t>(out_slot) * p.splits + part) * block + r) * BN + col) = v;
            }
          }
        }
      }
    }
  };
  for_tile_count<3, NS == 1 ? 4 : kW4A8StreamTiles>((rows + 15) / 16, run);  // (33..128 tokens)
}

}  // namespace ksq
