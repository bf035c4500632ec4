// Dense W8A8 GEMM over many rows: a 256 x 256 output tile per block of eight waves and CU, operands through LDS by direct loads.
// Arithmetic of k_dense_tile (tile_gemm.cuh), instruction for instruction, so the same bits.
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

// One tile by all eight waves of a block. GROUPED: the tokens are positions start .. start + n - 1 of the permuted order (MODE 0 gathers
// their rows, MODE 1 weights its results and scatters them to their assignments).
template <int MODE, bool GROUPED>
__device__ __forceinline__ void wide_tile(const GemmParams& p, uint8_t* lds, int t, int start, int n, const uint64_t (&wc)[2], const uint64_t (&ws)[2]) {
    // What follows from the thread's index is worked out again for every unit: kept from unit to unit it spilled, and a launch with a scratch
    // segment starts later (cohort kernel, 36 bytes per lane: a layer of 64 small groups at 4096 / 1536 253 us, 248 without)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int wave = uni(tid >> 6);
    const int wr = wave >> 2, wt = wave & 3;  // weight half (128 rows), token quarter (64 tokens)
    const int K = p.K, N = p.N, KB = K >> 7;
    const uint32_t lds0 = lds_address(lds);
    const int r16 = lane & 15, c = lane >> 4;
    const uint32_t piece = uint32_t(((lane & 7) ^ lds_key(lane >> 3)) << 4);  // odd requests: piece ^ 4
    const uint32_t woff = uint32_t(lane >> 3) * uint32_t(K) + piece;
    const int rd_lo = r16 * 128 + (((2 * c) ^ lds_key(r16)) << 4), rd_hi = r16 * 128 + (((2 * c + 1) ^ lds_key(r16)) << 4);
    // MODE 0: fragments 0 .. 3 of a half are gate rows, 4 .. 7 the up rows of the same columns
    auto column = [&](int half, int f) { return MODE == 0 ? t * 128 + half * 64 + (f & 3) * 16 : t * 256 + half * 128 + f * 16; };
    uint64_t wbase[2];  // rows of fragment `wave` of either half
#pragma unroll
    for (int h = 0; h < 2; ++h) wbase[h] = uni64((MODE == 0 ? wc[wave >> 2] : wc[0]) + uint64_t(min(column(h, wave), N - 16)) * uint64_t(K));
    uint32_t toff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int pos = start + min(wave * 32 + i * 8 + (lane >> 3), n - 1);
      const int row = GROUPED && MODE == 0 ? load_global<int>(p.perm + pos) / p.top_k : pos;
      toff[i] = uint32_t(row) * uint32_t(K) + (piece ^ (64u * (i & 1)));
    }
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
        lds_load4(at + i * 256u, p.a_scales + (toff[i] >> 7) + min(8 * g + (lane & 7), KB - 1));  // a row of 128 KB codes has KB scales
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
    int to = start + wt * 64 + el;  // lane l: where token l of the wave's 64 goes, and its routing weight
    float rwl = 1.0f;
    if constexpr (MODE == 1) {
      to = load_global<int>(p.perm + start + min(wt * 64 + el, n - 1));
      if (p.weights)
        rwl = p.weights_f32 ? load_global<float>(reinterpret_cast<const float*>(p.weights) + to) : bf16_to_f32(load_global<uint16_t>(reinterpret_cast<const uint16_t*>(p.weights) + to));
    }
    {
      const int er = el & 15, ec = el >> 4;
      float rw[4];
      if constexpr (MODE == 1) {
#pragma unroll
        for (int m = 0; m < 4; ++m) rw[m] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((16 * m + er) << 2, __builtin_bit_cast(int, rwl)));
      }
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
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = MODE == 1 && p.weights ? w8a8_weighted(acc[m][f][r], rw[m], p.routed_weight) : acc[m][f][r];
            o = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
          }
          *reinterpret_cast<u32x2*>(at + 16 * m * ROW) = o;
        }
      }
    }
    wave_lds_fence();
    {
      const int pl = el & (LPR - 1), col = column(wr, 0) + pl * 8;
#pragma unroll 1
      for (int row0 = el / LPR; row0 < 64; row0 += 4 * 64 / LPR) {  // four rows' reads in flight
        u32x4 v[4];
        int at[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = row0 + i * (64 / LPR);
          v[i] = *reinterpret_cast<const u32x4*>(mine + row * ROW + ((pl ^ key(row)) << 4));
          at[i] = MODE == 1 ? __builtin_amdgcn_ds_bpermute(row << 2, to) : start + wt * 64 + row;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (wt * 64 + row0 + i * (64 / LPR) < n && col + 8 <= N) {
            *reinterpret_cast<u32x4*>(p.out + size_t(at[i]) * N + col) = v[i];
            if (MODE == 1 && p.done && t == 0 && wr == 0 && pl == 0) p.done[at[i]] = 1u;
          }
      }
    }
}

template <int MODE>
__global__ __launch_bounds__(512, 2) void k_w8a8_wide(const GemmParams p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const uint32_t total = p.total_units;
  const int ntiles = (p.N + (MODE == 0 ? 127 : 255)) / (MODE == 0 ? 128 : 256);
  const int groups = (p.rows_total + 255) / 256;
  const uint32_t xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3, per_xcd = gridDim.x >> 3;
  const uint32_t span = (total + 7u) >> 3;
  const uint32_t span_end = min(total, (xcd + 1u) * span);
  for (uint32_t u = xcd * span + slot; u < span_end; u += per_xcd) {
    const int tb = int(u) / (groups * 4), v = int(u) - tb * groups * 4;  // the blocks of an XCD run a window of 4 x 8 tiles
    const int width = min(4, ntiles - tb * 4);
    const int t = tb * 4 + v % width, start = (v / width) * 256, n = min(256, p.rows_total - start);
    const uint64_t wc[2] = {p.w0_codes, MODE == 0 ? p.w1_codes : p.w0_codes}, ws[2] = {p.w0_scales, MODE == 0 ? p.w1_scales : p.w0_scales};
    wide_tile<MODE, false>(p, lds, t, start, n, wc, ws);
  }
}

// ---- cohorts: token groups of a routed layer ---------------------------------------------------------------------------
// Popular experts come in groups of up to 256 tokens, which run the tile above; the rest of an expert's tokens, up to 128, are one group, which
// streams the expert's weights past its live 16-token fragments (k_w8a8_cohort). 4096 tokens, top-8 of 256 experts at hidden 7168 /
// intermediate 2048, Zipf-like: gate/up 2197 -> 1800 us, down 1280 -> 1080 us against 64-row groups throughout; 65 tokens, all stream: a
// layer 1022 -> 935 us. What bounds it: a tile is at 3500 of 2048 cycles per K block, a stream's share of memory gives it a K block of 32 KB
// every 2200 cycles; between units a block waits for claims, descriptors and first operands (6000 cycles) and drains (a gate/up tile's SwiGLU 20000).
// Two groups of 64 for the rest fetch the weights twice, too far apart to share them: evenly routed chunks of 64 to 128 tokens per expert were 10 to
// 25 % behind the 64-row kernel, whose two groups run side by side. us per call, that one / two groups / one, even: 1024 tokens, top-6 of 64
// at 4096 / 1536 360 / 456 / 338; 2048, top-8 of 256 at 7168 / 2048 2485 / 2761 / 2229; Zipf-like, 4096 of the latter 3424 / 3003 / 2835. The
// larger groups in one list with the tiles, so that they start first: 2973 there.
// Stage of a group of up to 16 MF tokens: a K block of 256 weight rows (32 per wave) and of the tokens; a ring of STAGES of them.
template <int MF> struct StreamStage { uint8_t w[256 * 128]; uint8_t t[MF * 16 * 128]; };
template <int MF> constexpr int stream_stages() { return MF > 2 ? 3 : 4; }
constexpr int COHORT_SX = 4 * int(sizeof(StreamStage<2>)), STREAM_SX = 128 * 8 * 4, COHORT_LDS = COHORT_SX + 2 * STREAM_SX + 16;  // the scales of eight K blocks, twice; the claim
static_assert(WIDE_LDS <= COHORT_SX && 3 * int(sizeof(StreamStage<8>)) <= COHORT_SX && 4 * int(sizeof(StreamStage<1>)) <= COHORT_SX && COHORT_LDS <= 160 * 1024, "one block per CU");

template <int MODE, int MF>
__device__ __forceinline__ void stream_tile(const GemmParams& p, uint8_t* lds, int t, int start, int n, const uint64_t (&wc)[2], const uint64_t (&ws)[2]) {
  using Stage = StreamStage<MF>;
  constexpr int NS = stream_stages<MF>();
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // as in wide_tile
  const int lane = tid & 63;
  const int wave = uni(tid >> 6);
  const int K = p.K, N = p.N, KB = K >> 7;
  const uint32_t lds0 = lds_address(lds);
  const int r16 = lane & 15, c = lane >> 4;
  const uint32_t piece = uint32_t(((lane & 7) ^ lds_key(lane >> 3)) << 4);  // odd requests: piece ^ 4
  const uint32_t woff = uint32_t(lane >> 3) * uint32_t(K) + piece;
  const int rd_lo = r16 * 128 + (((2 * c) ^ lds_key(r16)) << 4), rd_hi = r16 * 128 + (((2 * c + 1) ^ lds_key(r16)) << 4);
  // fragment f of this wave; MODE 0: gate rows and the up rows of the same columns. Past N: clamped and dropped at the store
  auto column = [&](int f) { return MODE == 0 ? t * 128 + wave * 16 : t * 256 + wave * 32 + f * 16; };
  uint64_t wbase[2];
#pragma unroll
  for (int f = 0; f < 2; ++f) wbase[f] = uni64(wc[f] + uint64_t(min(column(f), N - 16)) * uint64_t(K));
  // block scales, lane l keeps K block l (+ 64); a wave's columns sit inside one 128-row block
  const float* sw0 = reinterpret_cast<const float*>(ws[0]) + size_t(min(column(0), N - 16) >> 7) * KB;
  const float* sw1 = reinterpret_cast<const float*>(ws[1]) + size_t(min(column(0), N - 16) >> 7) * KB;
  float swl0 = load_global<float>(sw0 + min(lane, KB - 1)), swl1 = MODE == 0 ? load_global<float>(sw1 + min(lane, KB - 1)) : 0.0f;
  constexpr int TR = MF > 4 ? 2 : 1;  // token requests of a wave, of eight tokens each
  const bool mover = wave * TR < 2 * MF;  // the waves that make them
  uint32_t toff[TR];
#pragma unroll
  for (int i = 0; i < TR; ++i) {
    toff[i] = 0;
    if (mover) {
      const int q = wave * TR + i, pos = start + min(q * 8 + (lane >> 3), n - 1);
      const int row = MODE == 0 ? load_global<int>(p.perm + pos) / p.top_k : pos;
      toff[i] = uint32_t(row) * uint32_t(K) + (piece ^ (64u * (q & 1)));
    }
  }
  swl0 = landed(swl0);
  if (MODE == 0) swl1 = landed(swl1);
  auto request = [&](int q, uint32_t b) {
    const uint32_t at = lds0 + b * uint32_t(sizeof(Stage));
#pragma unroll
    for (int i = 0; i < 4; ++i)
      lds_load16_nt(at + uint32_t(wave) * 4096u + i * 1024u, wbase[i >> 1] + uint64_t(uint32_t(q) * 128u) + ((i & 1) ? 8u * uint64_t(K) : 0u), woff ^ (64u * (i & 1)));
    if (mover) {
#pragma unroll
      for (int i = 0; i < TR; ++i) {
        const uint32_t t8 = uint32_t(wave) * TR + i;
        if ((q & 7) == 0) lds_load4(lds0 + uint32_t(COHORT_SX) + uint32_t((q >> 3) & 1) * uint32_t(STREAM_SX) + t8 * 256u, p.a_scales + (toff[i] >> 7) + min(q + (lane & 7), KB - 1));
        lds_load16(at + uint32_t(offsetof(Stage, t)) + t8 * 1024u, uint64_t(uintptr_t(p.a_codes)) + uint64_t(uint32_t(q) * 128u), toff[i]);
      }
    }
  };
  float acc[MF][2][4];
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[m][f][r] = 0.0f;
  // the previous unit's last reads are done and nothing is in flight
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int b = 0; b < NS - 1; ++b)
    if (b < KB) request(b, b);
  uint32_t b = 0;
  for (int kb = 0; kb < KB; ++kb) {
    // K block kb has landed: behind it the requests of NS - 2 later ones (and scales now and then: the wait is one request stricter then)
    if (kb + NS - 2 < KB) {
      if (mover) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * (4 + TR)) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * 4) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // for every wave, and the K block before it has been read
    if (kb + NS - 1 < KB) request(kb + NS - 1, b == 0 ? NS - 1 : b - 1);
    const uint8_t* st = lds + b * sizeof(Stage);
    b = b == NS - 1 ? 0 : b + 1;
    if ((kb & 63) == 0 && kb > 0) {
      swl0 = landed(load_global<float>(sw0 + min(kb + lane, KB - 1)));
      if (MODE == 0) swl1 = landed(load_global<float>(sw1 + min(kb + lane, KB - 1)));
    }
    const float s0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, swl0), kb & 63));
    const float s1 = MODE == 0 ? __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, swl1), kb & 63)) : s0;
    auto read = [&](const uint8_t* base) {
      const u32x4 lo = *reinterpret_cast<const u32x4*>(base + rd_lo), hi = *reinterpret_cast<const u32x4*>(base + rd_hi);
      return v8i{int(lo[0]), int(lo[1]), int(lo[2]), int(lo[3]), int(hi[0]), int(hi[1]), int(hi[2]), int(hi[3])};
    };
    const float* sl = reinterpret_cast<const float*>(lds + COHORT_SX + ((kb >> 3) & 1) * STREAM_SX) + r16 * 8 + (kb & 7);
    v8i wf[2];
#pragma unroll
    for (int f = 0; f < 2; ++f) wf[f] = read(st + wave * 4096 + f * 2048);
    v4f pr[MF][2];
    float sx[MF];
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      sx[m] = sl[16 * 8 * m];
      const v8i tok = read(st + offsetof(Stage, t) + m * 2048);
#pragma unroll
      for (int f = 0; f < 2; ++f) pr[m][f] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[f], tok, v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0, 0, 0, 0);
    }
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      const float sc0 = __fmul_rn(s0, sx[m]), sc1 = MODE == 0 ? __fmul_rn(s1, sx[m]) : sc0;
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[m][f][r] = __fmaf_rn(pr[m][f][r], MODE == 0 && f == 1 ? sc1 : sc0, acc[m][f][r]);
    }
  }
#pragma unroll
  for (int m = 0; m < MF; ++m) {
    const int token = 16 * m + r16;
    if (token >= n) continue;
    const int pos = start + token;
    if (MODE == 0) {
      const int col = column(0);
      if (col + 16 <= N) {
        uint32_t o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = swiglu_bf16_two_branch(bround(acc[m][0][r]), bround(acc[m][1][r]), p.swiglu, p.limit);
        *reinterpret_cast<u32x2*>(p.out + size_t(pos) * N + col + 4 * c) = u32x2{o[0] | (o[1] << 16), o[2] | (o[3] << 16)};
      }
    } else {
      const int a = load_global<int>(p.perm + pos);
      float rw = 1.0f;
      if (p.weights) rw = p.weights_f32 ? load_global<float>(reinterpret_cast<const float*>(p.weights) + a) : bf16_to_f32(load_global<uint16_t>(reinterpret_cast<const uint16_t*>(p.weights) + a));
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        const int col = column(f);
        if (col + 16 <= N) {
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = p.weights ? w8a8_weighted(acc[m][f][r], rw, p.routed_weight) : acc[m][f][r];
          *reinterpret_cast<u32x2*>(p.out + size_t(a) * N + col + 4 * c) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        }
      }
      if (p.done && t == 0 && wave == 0 && lane < 16) p.done[a] = 1u;
    }
  }
}

// Units of the two kinds are two lists, each cut into eight spans, one per XCD (prefill's unit order: neighbours share weights). Half of an
// XCD's blocks start on its tiles, half on its streams: the tiles bound by the matrix cores and the streams by memory share the chip, and
// tiles that share operands run side by side (in one list, in expert order, an expert's tiles start at different times, lose each other in
// L2 and the launch takes 1950 us instead of 1815). A unit's cost is not known ahead, so blocks claim units one by one and go on
// to the other kind and to other XCDs' spans when theirs are through. queue[x] counts the claims on span x behind the first unit of each of
// its own blocks; every block makes one claim too many on each span, and the last of those puts the counter back to zero for the next launch.
template <int MODE>
__global__ __launch_bounds__(512, 2) void k_w8a8_cohort(const GemmParams p, const uint32_t* big_groups, uint32_t* queue) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  uint32_t* const s_claim = reinterpret_cast<uint32_t*>(lds + COHORT_SX + 2 * STREAM_SX);
  const int tid = threadIdx.x;
  const uint32_t tiles = uint32_t(p.N + (MODE == 0 ? 127 : 255)) / (MODE == 0 ? 128u : 256u);
  const uint32_t split = load_uniform<uint32_t>(big_groups) * tiles, total = load_uniform<uint32_t>(p.unit_total);
  const uint32_t home = blockIdx.x & 7u, slot = blockIdx.x >> 3, per_xcd = gridDim.x >> 3;
  uint32_t j = 0;  // spans this block is through with
  uint32_t x, first, len, owners;
  auto enter = [&]() {  // the j-th span: kinds alternate, XCDs advance
    const uint32_t kind = (slot ^ j) & 1u, s = (home + (j >> 1)) & 7u;
    const uint32_t lo = kind ? split : 0u, count = kind ? total - split : split, span = (count + 7u) >> 3;
    x = kind * 8u + s;
    first = lo + min(count, s * span);
    len = lo + min(count, (s + 1u) * span) - first;
    owners = kind ? per_xcd >> 1 : (per_xcd + 1u) >> 1;  // blocks that start here
  };
  enter();
  uint32_t u = first + (slot >> 1);
  bool have = (slot >> 1) < len;
  for (;;) {
    while (len <= owners) {  // nothing left to claim
      if (++j == 16u) break;
      enter();
    }
    if (j == 16u && !have) return;
    uint32_t claim = 0;
    if (tid == 0 && j < 16u) claim = atomicAdd(queue + x, 1u);  // has landed when the unit's first requests go out
    if (have) {
      const u32x2 un = load_uniform<u32x2>(p.units + u);
      const int* gd = reinterpret_cast<const int*>(p.groups + int(un.x));
      const int t = int(un.y), expert = load_uniform<int>(gd), start = load_uniform<int>(gd + 1), n = load_uniform<int>(gd + 2);
      const uint64_t* sl = p.slots + size_t(expert) * 6 + (MODE == 0 ? 0 : 4);
      const uint64_t wc[2] = {load_uniform<uint64_t>(sl), load_uniform<uint64_t>(sl + (MODE == 0 ? 2 : 0))};
      const uint64_t ws[2] = {load_uniform<uint64_t>(sl + 1), load_uniform<uint64_t>(sl + (MODE == 0 ? 3 : 1))};
      if (n > 128) wide_tile<MODE, true>(p, lds, t, start, n, wc, ws);
      else if (n > 96) stream_tile<MODE, 8>(p, lds, t, start, n, wc, ws);
      else if (n > 64) stream_tile<MODE, 6>(p, lds, t, start, n, wc, ws);
      else if (n > 32) stream_tile<MODE, 4>(p, lds, t, start, n, wc, ws);
      else if (n > 16) stream_tile<MODE, 2>(p, lds, t, start, n, wc, ws);
      else stream_tile<MODE, 1>(p, lds, t, start, n, wc, ws);
    }
    if (j == 16u) return;
    if (tid == 0) *s_claim = claim;
    __syncthreads();
    const uint32_t v = uint32_t(uni(int(*s_claim)));
    __syncthreads();
    have = v < len - owners;
    u = first + owners + v;
    if (!have) {
      if (tid == 0 && v == len - owners + gridDim.x - 1u) queue[x] = 0u;
      if (++j < 16u) enter(); else return;
    }
  }
}

}  // namespace ffmoe
