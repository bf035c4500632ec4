// Dense W8A8 GEMM over many rows: a 256 x 256 output tile per block of eight waves and CU, operands through LDS by direct loads.
// Arithmetic of k_w8a8_tile (tile_gemm.cuh), instruction for instruction, so the same bits.
//
// What bounds it: a K block of a tile is 256 matrix instructions = 2048 cycles per SIMD with four scale fmas behind each (an
// instruction and its fmas issue in 35 cycles), next to 196 KB of operand reads and 64 KB of direct loads in the CU's LDS. A tile of
// 128 x 128 reads 256 KB for the same work, and its requests drain at every K block. Here
//  - a wave multiplies 128 weight rows x 64 tokens (128 totals per lane; a larger tile does not fit next to its operands),
//  - the four waves of the second weight half run half a K block behind those of the first: each SIMD holds one of either, so one
//    multiplies while the other fills its token registers, and a half's weights are requested again as soon as that half is through;
//    requests stay in flight across every boundary (waits by count, one boundary per half K block),
//  - a product meets its fmas three instructions later, so no wait states sit in between,
//  - token scales come for eight K blocks at a time, results leave through LDS in whole rows.
// Measured, steady clocks (1.9 GHz under this load): 4096 x 7168 -> 4096 122 us on 128 x 128 tiles, 102 here = 2.35 PFLOP/s (3260 cycles
// per K block; 2716 without the loads); 2048 x 2048 -> 7168 41 -> 32.5. Not faster: both halves in step (110), requests prefetched into
// L2 by loads of single words (114), all requests of a boundary at once (the same).
#pragma once
#include "w8a8_gemm.cuh"
#include "lds_load.cuh"

namespace ffmoe {

struct WideStage { uint8_t w[2][128 * 128]; uint8_t t[256 * 128]; };
struct WideLds { WideStage stage[2]; float sx[2][256][8]; };  // sx: the scales of eight K blocks
constexpr int WIDE_LDS = int(sizeof(WideLds));

constexpr int WIDE_LAG = 3;  // matrix instructions between a product and its fmas

template <int MODE>
__global__ __launch_bounds__(512, 2) void k_w8a8_wide(const GemmParams p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = uni(tid >> 6);
  const int wr = wave >> 2, wt = wave & 3;  // weight half (128 rows), token quarter (64 tokens)
  const int K = p.K, N = p.N, KB = K >> 7;
  const uint32_t total = p.total_units;
  const int ntiles = (N + (MODE == 0 ? 127 : 255)) / (MODE == 0 ? 128 : 256);
  const int groups = (p.rows_total + 255) / 256;
  const uint32_t xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3, per_xcd = gridDim.x >> 3;
  const uint32_t span = (total + 7u) >> 3;
  const uint32_t span_end = min(total, (xcd + 1u) * span);
  const uint32_t lds0 = lds_address(lds);
  const int r16 = lane & 15, c = lane >> 4;
  const uint32_t piece = uint32_t(((lane & 7) ^ lds_key(lane >> 3)) << 4);  // odd requests: piece ^ 4
  const uint32_t woff = uint32_t(lane >> 3) * uint32_t(K) + piece;
  const int rd_lo = r16 * 128 + (((2 * c) ^ lds_key(r16)) << 4), rd_hi = r16 * 128 + (((2 * c + 1) ^ lds_key(r16)) << 4);

  for (uint32_t u = xcd * span + slot; u < span_end; u += per_xcd) {
    const int tb = int(u) / (groups * 4), v = int(u) - tb * groups * 4;
    const int width = min(4, ntiles - tb * 4);
    const int t = tb * 4 + v % width, start = (v / width) * 256, n = min(256, p.rows_total - start);
    const uint64_t wc[2] = {p.w0_codes, MODE == 0 ? p.w1_codes : p.w0_codes}, ws[2] = {p.w0_scales, MODE == 0 ? p.w1_scales : p.w0_scales};
    // MODE 0: fragments 0 .. 3 of a half are gate rows, 4 .. 7 the up rows of the same columns
    auto column = [&](int half, int f) { return MODE == 0 ? t * 128 + half * 64 + (f & 3) * 16 : t * 256 + half * 128 + f * 16; };
    uint64_t wbase[2];  // rows of fragment `wave` of either half
#pragma unroll
    for (int h = 0; h < 2; ++h) wbase[h] = uni64((MODE == 0 ? wc[wave >> 2] : wc[0]) + uint64_t(min(column(h, wave), N - 16)) * uint64_t(K));
    uint32_t toff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) toff[i] = uint32_t(start + min(wave * 32 + i * 8 + (lane >> 3), n - 1)) * uint32_t(K) + (piece ^ (64u * (i & 1)));
    const uint64_t tbase = uint64_t(uintptr_t(p.a_codes));
    const float* sw0 = reinterpret_cast<const float*>(ws[0]) + size_t(min(column(wr, 0), N - 16) >> 7) * KB;
    const float* sw1 = reinterpret_cast<const float*>(ws[1]) + size_t(min(column(wr, 0), N - 16) >> 7) * KB;

    auto request_w = [&](int kb, int half, int i) {
      lds_load16(lds0 + uint32_t(kb & 1) * uint32_t(sizeof(WideStage)) + uint32_t(half) * 16384u + uint32_t(wave) * 2048u + i * 1024u,
                 wbase[half] + uint64_t(uint32_t(kb) * 128u) + (i ? 8u * uint64_t(K) : 0u), woff ^ (64u * i));
    };
    auto request_t = [&](int kb, int i) {
      lds_load16(lds0 + uint32_t(kb & 1) * uint32_t(sizeof(WideStage)) + uint32_t(offsetof(WideStage, t)) + uint32_t(wave) * 4096u + i * 1024u,
                 tbase + uint64_t(uint32_t(kb) * 128u), toff[i]);
    };
    auto request_s = [&](int g) {  // scales of K blocks 8 g .. 8 g + 7
      const uint32_t at = lds0 + uint32_t(offsetof(WideLds, sx)) + uint32_t(g & 1) * 8192u + uint32_t(wave) * 1024u;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        lds_load4(at + i * 256u, p.a_scales + size_t(start + min(wave * 32 + i * 8 + (lane >> 3), n - 1)) * KB + min(8 * g + (lane & 7), KB - 1));
    };
    const auto scales_with = [&](int q) { return (q & 7) == 4 && (q & ~7) + 8 < KB; };  // K block q's tokens bring the next eight scales
    // the requests of an even boundary (tokens and first weight half of K block q) and of an odd one (second weight half), in parts that
    // the steps behind the boundary take one by one: a wave that issues them in one go finds the memory pipeline full
    auto request_even = [&](int q, int i) {
      if (q < KB) {
        if (i == 0 && scales_with(q)) request_s((q >> 3) + 1);
        request_t(q, i);
        if (i >= 2) request_w(q, 0, i - 2);
      }
    };
    auto request_odd = [&](int q, int i) { if (q < KB && i < 2) request_w(q, 1, i); };
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    request_s(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) request_even(0, i);
    request_odd(0, 0);
    request_odd(0, 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) request_even(1, i);

    float acc[4][8][4];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int f = 0; f < 8; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[m][f][r] = 0.0f;

    auto read = [&](const uint8_t* base) {
      const u32x4 lo = *reinterpret_cast<const u32x4*>(base + rd_lo), hi = *reinterpret_cast<const u32x4*>(base + rd_hi);
      return v8i{int(lo[0]), int(lo[1]), int(lo[2]), int(lo[3]), int(hi[0]), int(hi[1]), int(hi[2]), int(hi[3])};
    };
    const uint8_t* const wl0 = lds + wr * 16384;
    const uint8_t* const tl0 = lds + offsetof(WideStage, t) + wt * 8192;
    const uint8_t* const sl0 = lds + offsetof(WideLds, sx) + (wt * 64 + r16) * 32;

    // half K block boundaries, the same sequence for all waves. In front of an even one (the first weight half starts K block kb): its
    // tokens and weights, requested two boundaries ago, have landed, younger are the two requests of the odd boundary between
    auto even_boundary = [&](int kb) {
      if (kb < KB) asm volatile("s_waitcnt vmcnt(2)" ::: "memory"); else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      asm volatile("s_barrier" ::: "memory");
    };
    // odd (the second half starts kb): younger are the requests of K block kb + 1
    auto odd_boundary = [&](int kb) {
      if (kb + 1 >= KB) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      else if (scales_with(kb + 1)) asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
      asm volatile("s_barrier" ::: "memory");
    };

    auto run = [&](auto grp_) {
      constexpr int G = decltype(grp_)::value;
      if constexpr (G == 1) {
        odd_boundary(0);
        request_odd(1, 0);
        request_odd(1, 1);
      }
      v8i tok[4], wf[3];
      float sx[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) { tok[m] = read(tl0 + m * 2048); sx[m] = *reinterpret_cast<const float*>(sl0 + m * 512); }
      wf[0] = read(wl0);
      wf[1] = read(wl0 + 2048);
      v4f pr[WIDE_LAG + 1];
      float s0 = 0.0f, s1 = 0.0f;
      // K block kb in buffer b; its token fragments and its weight fragments 0, 1 are in registers or on their way
      auto block = [&](int kb, auto b_) {
        constexpr int b = decltype(b_)::value;
        const uint8_t* wl = wl0 + b * sizeof(WideStage);
        const uint8_t* wn = wl0 + (b ^ 1) * sizeof(WideStage);
        const uint8_t* tn = tl0 + (b ^ 1) * sizeof(WideStage);
        const uint8_t* sn = sl0 + (((kb + 1) >> 3) & 1) * 8192 + ((kb + 1) & 7) * 4;
        float sc[4][MODE == 0 ? 2 : 1];
        static_for<32 + WIDE_LAG>([&](auto step_) {
          constexpr int step = decltype(step_)::value;
          constexpr int f = step >> 2, m = step & 3;
          if constexpr (step < 32) {
            if constexpr (m == 0 && f < 6) wf[(f + 2) % 3] = read(wl + (f + 2) * 2048);
            if constexpr (m == 0 && f == 3) {
              if constexpr (G == 0) odd_boundary(kb); else even_boundary(kb + 1);
            }
            if constexpr (m == 0 && f == 7) {
              asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this half of buffer b has been read
              if constexpr (G == 0) even_boundary(kb + 1); else odd_boundary(kb + 1);
              wf[0] = read(wn);  // past the last K block: whatever is there
            }
            if constexpr (f == 3) {
              if constexpr (G == 0) request_odd(kb + 1, m); else request_even(kb + 2, m);
            }
            if constexpr (f == 7) {
              if constexpr (G == 0) request_even(kb + 2, m); else request_odd(kb + 2, m);
            }
            if constexpr (f == 5) sx[m] = *reinterpret_cast<const float*>(sn + m * 512);
            pr[step % (WIDE_LAG + 1)] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[f % 3], tok[m], v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0, 0, 0, 0);
            if constexpr (f == 7) {
              tok[m] = read(tn + m * 2048);
              if constexpr (m == 3) wf[1] = read(wn + 2048);
            }
          }
          if constexpr (step + 1 >= WIDE_LAG && step + 1 < WIDE_LAG + 4) {
            constexpr int qm = step + 1 - WIDE_LAG;
            sc[qm][0] = __fmul_rn(s0, sx[qm]);
            if constexpr (MODE == 0) sc[qm][1] = __fmul_rn(s1, sx[qm]);
          }
          if constexpr (step >= WIDE_LAG) {
            constexpr int q = step - WIDE_LAG, qf = q >> 2, qm = q & 3;
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[qm][qf][r] = __fmaf_rn(pr[q % (WIDE_LAG + 1)][r], sc[qm][MODE == 0 && qf >= 4 ? 1 : 0], acc[qm][qf][r]);
#pragma unroll
            for (int r = 0; r < 4; ++r) asm volatile("" ::"v"(acc[qm][qf][r]));
          }
          __builtin_amdgcn_sched_barrier(0);
        });
      };
      for (int kb0 = 0; kb0 < KB; kb0 += 64) {
        const int kl = min(kb0 + lane, KB - 1);
        const float swl0 = landed(load_global<float>(sw0 + kl));
        const float swl1 = MODE == 0 ? landed(load_global<float>(sw1 + kl)) : swl0;
        const int kend = min(KB, kb0 + 64);
        auto scale = [&](float v_, int kb) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v_), kb - kb0)); };
        for (int kb = kb0; kb < kend; kb += 2) {
          s0 = scale(swl0, kb); s1 = scale(swl1, kb);
          block(kb, std::integral_constant<int, 0>{});
          if (kb + 1 < kend) {
            s0 = scale(swl0, kb + 1); s1 = scale(swl1, kb + 1);
            block(kb + 1, std::integral_constant<int, 1>{});
          }
        }
      }
      if constexpr (G == 0) asm volatile("s_barrier" ::: "memory");
    };
    if (KB > 1) asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); else asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    if (wr == 0) run(std::integral_constant<int, 0>{});
    else run(std::integral_constant<int, 1>{});

    // through LDS, so that a store covers whole rows of the wave's columns: a wave owns 64 tokens x ROW bytes, 16-byte pieces swizzled by
    // the token (straight from the accumulators a store touches 16 rows for 32 bytes each: 2048 x 2048 -> 7168 38 us instead of 32.5)
    constexpr int ROW = MODE == 0 ? 128 : 256, LPR = ROW / 16;
    uint8_t* const mine = lds + wave * (64 * ROW);
    auto key = [](int row) { return MODE == 0 ? (row >> 1) & 7 : row & 15; };
    int el = lane;  // its own copy: addresses derived from it are not computed ahead of the K loop, where they would spill
    asm volatile("s_barrier" : "+v"(el)::"memory");  // nobody reads operands any more, and no request is in flight
    {
      const int er = el & 15, ec = el >> 4;
      uint8_t* const mw = mine + er * ROW + (ec & 1) * 8;
      const int k0 = (ec >> 1) ^ key(er);
#pragma unroll
      for (int f = 0; f < (MODE == 0 ? 4 : 8); ++f) {
        uint8_t* const at = mw + ((k0 ^ (2 * f)) << 4);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          u32x2 o;
          if (MODE == 0) {
            uint32_t h[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) h[r] = swiglu_bf16_two_branch(bround(acc[m][f][r]), bround(acc[m][f + 4][r]), p.swiglu, p.limit);
            o = u32x2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
          } else {
            o = u32x2{pack_bf16x2(acc[m][f][0], acc[m][f][1]), pack_bf16x2(acc[m][f][2], acc[m][f][3])};
          }
          *reinterpret_cast<u32x2*>(at + 16 * m * ROW) = o;
        }
      }
    }
    wave_lds_fence();
    {
      const int pl = el & (LPR - 1), col = column(wr, 0) + pl * 8;
#pragma unroll 1
      for (int row = el / LPR; row < 64; row += 64 / LPR) {
        const int token = wt * 64 + row;
        if (token < n && col + 8 <= N)
          *reinterpret_cast<u32x4*>(p.out + size_t(start + token) * N + col) = *reinterpret_cast<const u32x4*>(mine + row * ROW + ((pl ^ key(row)) << 4));
      }
    }
  }
}

}  // namespace ffmoe
