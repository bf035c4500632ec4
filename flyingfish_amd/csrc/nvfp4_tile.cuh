// Grouped W4A16 GEMM of NVFP4 experts with K a multiple of 256: 128 weight rows x up to 64 tokens per block of four waves,
// both operands through LDS by direct loads, three blocks per CU. Arithmetic (dequantization to the decode path's BF16 effective
// weights, operand order, epilogue) is that of k_w16_grouped<FmtNvfp4>, results equal bit for bit.
//
// What bounds it: the weight stream next to two VALU instructions of dequantization per weight and row group, which want
// several waves per SIMD: three blocks share a CU's LDS (two blocks with a third weight buffer instead: 1021 tokens 2537 us
// a layer, three blocks 2414, k_w16_nvfp4_lines 3136). Whole 128-byte lines of codes (256 columns of a row) and the row's 16
// scale bytes are requested one stage ahead, token tiles of 64 or 128 columns two steps ahead (64 tokens: one); nothing
// passes through registers on its way in, so the wait of a step covers only what the step needs, and a group moves and
// multiplies only its live 16-token fragments.
#pragma once
#include "w16_gemm.cuh"
#include "lds_load.cuh"

namespace ffmoe {

struct NvWeights {
  uint8_t w[128 * 128];  // row r of the tile: 256 columns, 16-byte piece c at c ^ (r / 2 & 7)
  uint8_t s[128 * 16];   // its 16 scale bytes
};
// token tiles: MF x 16 rows of COLS columns; 16-byte piece c of row r at c ^ (r & 15) (256-byte rows) or c ^ (r / 2 & 7) (128)
template <int MF> struct NvTokens {
  static constexpr int COLS = MF == 1 ? 128 : 64, RING = MF > 2 ? 2 : 3, BYTES = MF * 16 * COLS * 2, REQUESTS = BYTES / 4096;
};
template <int MF> constexpr int nv_lds() { return 2 * int(sizeof(NvWeights)) + NvTokens<MF>::RING * NvTokens<MF>::BYTES; }
constexpr int NV_TILE_LDS = nv_lds<4>();
static_assert(nv_lds<2>() <= NV_TILE_LDS && nv_lds<1>() <= NV_TILE_LDS && 3 * NV_TILE_LDS <= 160 * 1024, "three blocks per CU");

// A unit of the list is 128 activation (MODE 0) or 256 output columns of one row group; a block takes it in two halves.
template <int MODE>
__global__ __launch_bounds__(256, 3) void k_nvfp4_tile(const W16Params p) {
  using F = W16<FmtNvfp4>;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = uni(tid >> 6);
  const int K = p.K, N = p.N, stages = K >> 8;
  const uint32_t total = 2u * load_uniform<uint32_t>(p.unit_total);
  const int ntiles = (N + gemm_tile_cols<MODE>() - 1) / gemm_tile_cols<MODE>();
  const uint32_t xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3, per_xcd = gridDim.x >> 3;
  const uint32_t span = (total + 7u) >> 3;
  const uint32_t span_end = min(total, (xcd + 1u) * span);
  const uint32_t lds0 = lds_address(lds);
  const int r16 = lane & 15, c = lane >> 4;
  // code requests: eight lanes per row, rows 0 .. 7 (even request) or 8 .. 15 (odd) of a fragment
  const uint32_t wrow = uint32_t(lane >> 3) * uint32_t(K >> 1);
  const uint32_t wpiece = uint32_t((lane & 7) ^ (lane >> 4));
  const uint32_t woff[2] = {wrow + (wpiece << 4), wrow + ((wpiece ^ 4u) << 4)};

  for (uint32_t u = xcd * span + slot; u < span_end; u += per_xcd) {
    const W16Unit d = w16_unit<MODE>(p, u >> 1, ntiles, 64);
    const int t = 2 * d.t + int(u & 1u);
    // fragments of this wave; MODE 0: gate rows and the up rows of the same columns. Past N: clamped and dropped at the store
    const int col0[2] = {MODE == 0 ? t * 64 + wave * 16 : t * 128 + wave * 32, MODE == 0 ? t * 64 + wave * 16 : t * 128 + wave * 32 + 16};
    if ((MODE == 0 ? t * 64 : t * 128) >= N) continue;
    uint64_t wbase[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) wbase[i] = uni64(d.wc[i >> 1] + uint64_t(min(col0[i >> 1], N - 16) + (i & 1) * 8) * uint64_t(K >> 1));
    // lanes 0 .. 31: the scale bytes of the wave's 32 rows
    const int sf = (lane >> 4) & 1;
    const uint8_t* ssrc = reinterpret_cast<const uint8_t*>(sf ? d.ws[1] : d.ws[0]) + size_t(min(sf ? col0[1] : col0[0], N - 16) + r16) * (K >> 4);
    typename F::Row wrow_of[2];  // only the global scale is read: the bytes come from LDS
    wrow_of[0].global = d.gl[0];
    wrow_of[1].global = d.gl[1];

    auto run = [&](auto mfc) {
      constexpr int MF = decltype(mfc)::value;
      using T = NvTokens<MF>;
      constexpr int SPS = 256 / T::COLS;     // token steps per weight stage
      constexpr int WL = 5, TL = T::REQUESTS;  // requests of a wave per weight stage and per token tile
      constexpr int RPR = 1024 / (2 * T::COLS);  // token rows per request
      const int steps = stages * SPS;
      uint8_t* const tiles = lds + 2 * sizeof(NvWeights);
      const uint8_t* tsrc[TL];
#pragma unroll
      for (int i = 0; i < TL; ++i) {
        const int r = (4 * i + wave) * RPR + (RPR == 4 ? lane >> 4 : lane >> 3);
        const int piece = RPR == 4 ? (lane & 15) ^ (r & 15) : (lane & 7) ^ ((r >> 1) & 7);
        const int pos = d.start + min(r, d.n - 1);
        const int row = MODE == 0 && p.perm && !d.ride ? load_global<int>(p.perm + pos) / p.top_k : pos;
        tsrc[i] = reinterpret_cast<const uint8_t*>(d.ride ? p.a_sh : p.a) + size_t(row) * K * 2 + piece * 16;
      }
      auto request_weights = [&](int ks, int b) {
        const uint32_t base = lds0 + uint32_t(b) * uint32_t(sizeof(NvWeights));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t at = base + uint32_t(wave) * 4096u + i * 1024u;
          // a short group's codes are read once: the streaming hint keeps the lines of scale bytes, which a row comes back to for
          // eight stages, in L2
          if constexpr (MF <= 2) lds_load16_nt(at, wbase[i] + uint64_t(uint32_t(ks) * 128u), woff[i & 1]);
          else lds_load16(at, wbase[i] + uint64_t(uint32_t(ks) * 128u), woff[i & 1]);
        }
        if (lane < 32) lds_load16(base + offsetof(NvWeights, s) + uint32_t(wave) * 512u, ssrc + uint32_t(ks) * 16u);
      };
      auto request_tokens = [&](int step, int b) {
        const uint32_t base = lds0 + uint32_t(2 * sizeof(NvWeights)) + uint32_t(b) * T::BYTES + uint32_t(wave) * 1024u;
#pragma unroll
        for (int i = 0; i < TL; ++i) lds_load16(base + i * 4096u, tsrc[i] + uint32_t(step) * (2u * T::COLS));
      };
      v4f acc[MF][2];
#pragma unroll
      for (int m = 0; m < MF; ++m) acc[m][0] = acc[m][1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      // the previous unit's last step has been read, and what was requested has landed
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      request_weights(0, 0);
#pragma unroll
      for (int b = 0; b < T::RING - 1; ++b) request_tokens(b, b);  // at least two steps: K >= 256
      int tr = 0;  // token buffer of the step at hand
      for (int step = 0; step < steps; ++step) {
        const int phase = step % SPS, ks = step / SPS;
        // A step requests a token tile (RING - 1 ahead), then, in phase 0, the next weight stage. Needed now: token tile `step`,
        // requested RING - 1 steps ago, and in phase 0 weight stage ks, requested SPS steps ago. Requested behind both: with three
        // token buffers tile step + 1; the next weight stage in phase 1, and in phase 2 where its tile was asked for in phase 0.
        const bool weights_behind = (phase == 1 || (SPS == 4 && T::RING == 3 && phase == 2)) && ks + 1 < stages;
        if (weights_behind) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(WL + (T::RING == 3 ? TL : 0)) : "memory");
        else if (T::RING == 3 && step + 1 < steps) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(TL) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // there for every wave, and the buffers of the step before are free
        if (step + T::RING - 1 < steps) request_tokens(step + T::RING - 1, tr == 0 ? T::RING - 1 : tr - 1);
        if (phase == 0 && ks + 1 < stages) request_weights(ks + 1, (ks + 1) & 1);
        const NvWeights& st = *reinterpret_cast<const NvWeights*>(lds + (ks & 1) * int(sizeof(NvWeights)));
        const uint8_t* tl = tiles + tr * T::BYTES;
        tr = tr == T::RING - 1 ? 0 : tr + 1;
#pragma unroll
        for (int h = 0; h < T::COLS / 64; ++h) {  // K blocks of 64 columns
          const int q = phase * (T::COLS / 64) + h;
          w16_bf16x8 a0[2], a1[2];
#pragma unroll
          for (int f = 0; f < 2; ++f) {
            const int row = wave * 32 + f * 16 + r16;
            typename F::Frag wm;
            wm.codes = *reinterpret_cast<const u32x2*>(st.w + row * 128 + (((2 * q + (c >> 1)) ^ (r16 >> 1)) << 4) + (c & 1) * 8);
            wm.scale = st.s[row * 16 + q * 4 + c];
            uint32_t wd[8];
            F::dequant(wm, wrow_of[f], wd);
            a0[f] = __builtin_bit_cast(w16_bf16x8, u32x4{wd[0], wd[1], wd[2], wd[3]});
            a1[f] = __builtin_bit_cast(w16_bf16x8, u32x4{wd[4], wd[5], wd[6], wd[7]});
          }
#pragma unroll
          for (int m = 0; m < MF; ++m) {
            const uint8_t* tb = tl + (16 * m + r16) * (2 * T::COLS);
            const int key = T::COLS == 128 ? r16 : r16 >> 1;
            const u32x4 lo = *reinterpret_cast<const u32x4*>(tb + (((8 * h + 2 * c) ^ key) << 4)), hi = *reinterpret_cast<const u32x4*>(tb + (((8 * h + 2 * c + 1) ^ key) << 4));
            const w16_bf16x8 b0 = __builtin_bit_cast(w16_bf16x8, lo), b1 = __builtin_bit_cast(w16_bf16x8, hi);
#pragma unroll
            for (int f = 0; f < 2; ++f) {
              acc[m][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[f], b0, acc[m][f], 0, 0, 0);
              acc[m][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[f], b1, acc[m][f], 0, 0, 0);
            }
          }
        }
      }
      w16_store<MF, MODE, 2>(acc, p, d.ride, d.start, d.n, t, col0, wave, lane);
    };
    if (d.n <= 16) run(std::integral_constant<int, 1>{});
    else if (d.n <= 32) run(std::integral_constant<int, 2>{});
    else run(std::integral_constant<int, 4>{});
  }
}

}  // namespace ffmoe
