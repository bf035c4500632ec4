// Grouped GEMM of E2M1 / E8M0 experts against E4M3 / E8M0 activations: 128 weight rows x up to 64 tokens per block of four
// waves, both operands through LDS by direct loads, two blocks per CU.
//
// MODE as in mx_gemm.cuh; one v_mfma_scale_f32_16x16x128_f8f6f4 per fragment pair and K block, K blocks in ascending order.
//
// What bounds it: a cohort is many experts of a few rows, which stream their weights, and a few popular ones, which run from
// cache. A stage is 256 columns, whole 128-byte lines of the weight rows; requests for groups of up to 32 tokens run two stages
// ahead in a ring of three (64 tokens: one stage, two buffers), scales come for two or four stages at a time, a group moves and multiplies only its live 16-token
// fragments, and the second block of the CU works while this one waits. Against 64-byte pieces of the weight rows moved through registers
// and a transposition buffer, 64 tokens multiplied whatever the group holds (top-8 of 256 experts, hidden 7168, Zipf-like): 1500
// tokens gate/up 1532 -> 1157 us, down 663 -> 600; a layer of 200 tokens, nearly all of it weight stream, 1464 -> 1052 us = 5.3 TB/s. (Those figures are without the scales' grouping.)
// Not faster: the next unit's first stages requested behind this one's last (1180 / 605 us), the two blocks of a CU on
// different halves of their XCD's units (1183 / 602).
#pragma once
#include "mx_gemm.cuh"
#include "lds_load.cuh"

namespace ffmoe {

template <int MF> struct MxStage {
  uint8_t w[128 * 128];                     // row r of the tile: 256 columns, 16-byte piece c at c ^ (r / 2 & 7)
  uint8_t t[MF * 16 * 256];                 // token row r: 256 columns, 16-byte piece c at c ^ (r & 15)
};
template <int MF> constexpr int mx_stages() { return MF > 2 ? 2 : 3; }
// The scale bytes of SG stages at a time, 8 SG per row, double-buffered. A stage's eight bytes of every row, fetched by each wave for its
// rows and for all tokens, touch a line per row: more line look-ups than the operands (1500 tokens gate/up 1187 -> 991 us, down 615 -> 540).
template <int MF> struct MxScales {
  static constexpr int SG = MF == 2 ? 2 : 4;  // four do not fit next to three stages of 32 tokens
  uint32_t w[2][128][2 * SG], t[2][MF * 16][2 * SG];
};
template <int MF> constexpr int mx_lds() { return mx_stages<MF>() * int(sizeof(MxStage<MF>)) + int(sizeof(MxScales<MF>)); }
constexpr int MX_TILE_LDS = mx_lds<2>();
static_assert(mx_lds<4>() <= MX_TILE_LDS && mx_lds<1>() <= MX_TILE_LDS && 2 * MX_TILE_LDS <= 160 * 1024, "two blocks per CU");

// A unit of the list is 128 activation (MODE 0) or 256 output columns of one row group; a block takes it in two halves.
template <int MODE>
__global__ __launch_bounds__(256, 2) void k_mx_tile(const MxParams p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = uni(tid >> 6);
  const int K = p.K, N = p.N, SB = K >> 5, KS = (K + 255) >> 8;
  const bool ragged = (K & 255) != 0;  // the last stage holds 128 columns
  const uint32_t total = 2u * load_uniform<uint32_t>(p.unit_total);
  const uint32_t xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3, per_xcd = gridDim.x >> 3;
  const uint32_t span = (total + 7u) >> 3;
  const uint32_t span_end = min(total, (xcd + 1u) * span);
  const uint32_t lds0 = lds_address(lds);
  const int r16 = lane & 15, c = lane >> 4;
  // weight requests: eight lanes per row, rows 0 .. 7 (even request) or 8 .. 15 (odd) of a fragment
  const uint32_t wrow = uint32_t(lane >> 3) * uint32_t(K >> 1);
  const uint32_t wpiece = uint32_t((lane & 7) ^ (lane >> 4));
  const uint32_t woff[2] = {wrow + (wpiece << 4), wrow + ((wpiece ^ 4u) << 4)};
  const uint32_t woff_half = wrow + ((wpiece & 3u) << 4);  // a last stage of 128 columns: the upper pieces repeat the lower ones
  const int tpiece = (lane & 15) ^ (wave * 4 + (lane >> 4));
  const int tback = (tpiece & 8) * 16;
  const int wrd0 = r16 * 128 + ((c ^ (r16 >> 1)) << 4), wrd1 = r16 * 128 + (((4 + c) ^ (r16 >> 1)) << 4);

  struct Desc { int start, n, t; uint64_t wc[2], ws[2]; };
  auto fetch_unit = [&](uint32_t u) {
    Desc d;
    const u32x2 un = load_uniform<u32x2>(p.units + (u >> 1));
    const int* gd = reinterpret_cast<const int*>(p.groups + int(un.x));
    d.t = 2 * int(un.y) + int(u & 1u);
    d.start = load_uniform<int>(gd + 1);
    d.n = load_uniform<int>(gd + 2);
    const uint64_t* sl = p.slots + size_t(load_uniform<int>(gd)) * 6 + (MODE == 0 ? 0 : 4);
    d.wc[0] = load_uniform<uint64_t>(sl); d.ws[0] = load_uniform<uint64_t>(sl + 1);
    d.wc[1] = MODE == 0 ? load_uniform<uint64_t>(sl + 2) : d.wc[0]; d.ws[1] = MODE == 0 ? load_uniform<uint64_t>(sl + 3) : d.ws[0];
    return d;
  };
  const uint32_t u_first = xcd * span + slot;
  Desc next = {};
  if (u_first < span_end) next = fetch_unit(u_first);
  for (uint32_t u = u_first; u < span_end; u += per_xcd) {
    const Desc d = next;
    if (u + per_xcd < span_end) next = fetch_unit(u + per_xcd);  // three dependent loads, under this unit's work
    // fragment f of this wave; MODE 0: gate rows and the up rows of the same columns. Past N: clamped and dropped at the store
    auto column = [&](int f) { return MODE == 0 ? d.t * 64 + wave * 16 : d.t * 128 + wave * 32 + f * 16; };
    if ((MODE == 0 ? d.t * 64 : d.t * 128) >= N) continue;
    uint64_t wbase[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) wbase[i] = uni64(d.wc[i >> 1] + uint64_t(min(column(i >> 1), N - 16) + (i & 1) * 8) * uint64_t(K >> 1));
    // the slots promise no alignment of scale bytes, a direct load of a word needs it: other addresses go through registers
    const bool words = ((d.ws[0] | d.ws[1]) & 3u) == 0;
    auto token_row = [&](int m) {
      const int pos = d.start + min(m, d.n - 1);
      return MODE == 0 ? load_global<int>(p.perm + pos) / p.top_k : pos;
    };

    auto run = [&](auto mfc) {
      constexpr int MF = decltype(mfc)::value, NS = mx_stages<MF>();
      constexpr int LPS = 4 + MF;  // requests of a wave per stage
      using Scales = MxScales<MF>;
      constexpr int SG = Scales::SG, RPR = 64 / (2 * SG);  // rows of a scale request, 2 SG lanes each
      constexpr int WR = 32 / RPR, TR = MF * 16 / RPR;     // scale requests: of a wave for its 32 rows, of the block for the tokens
      static_assert(SG >= NS - 1 && (TR == 2 || TR == 8), "a buffer is free when the next but one group is asked for");
      const uint32_t scales0 = lds0 + uint32_t(NS * sizeof(MxStage<MF>));
      const int tq = TR == 8 ? 2 : wave < 2 ? 1 : 0;       // token scale requests of this wave: wave, wave + 4
      const uint8_t* tsrc[MF];
#pragma unroll
      for (int i = 0; i < MF; ++i) tsrc[i] = p.a_codes + size_t(token_row(16 * i + wave * 4 + (lane >> 4))) * K + tpiece * 16;
      const int srow = lane / (2 * SG), sword = lane % (2 * SG), words_row = SB >> 2;
      const uint8_t* wssrc[WR];
#pragma unroll
      for (int i = 0; i < WR; ++i) {
        const int r = i * RPR + srow, f = r >> 4;
        wssrc[i] = reinterpret_cast<const uint8_t*>(d.ws[MODE == 0 ? f : 0]) + size_t(min(column(f), N - 16) + (r & 15)) * SB;
      }
      const uint8_t* tssrc[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) tssrc[i] = p.a_scales + size_t(token_row(min((wave + 4 * i) * RPR + srow, MF * 16 - 1))) * SB;
      auto request = [&](int ks, int b) {
        const uint32_t base = lds0 + uint32_t(b) * uint32_t(sizeof(MxStage<MF>));
        const bool half = ragged && ks == KS - 1;
        if (ks % SG == 0) {
          const uint32_t sb = uint32_t(ks / SG) & 1u;
          const int at = min(2 * ks + sword, words_row - 1) * 4;  // past the row's end: its last word, which nothing reads
          const uint32_t tw = scales0 + uint32_t(offsetof(Scales, t)) + sb * uint32_t(sizeof(Scales::t) / 2) + uint32_t(wave) * 256u;
          if (tq > 0) lds_load4(tw, tssrc[0] + at);
          if (tq > 1) lds_load4(tw + 1024u, tssrc[1] + at);
          const uint32_t ww = scales0 + sb * uint32_t(sizeof(Scales::w) / 2) + uint32_t(wave) * (WR * 256u);
#pragma unroll
          for (int i = 0; i < WR; ++i) {
            if (words) {
              lds_load4(ww + i * 256u, wssrc[i] + at);
            } else {  // fewer requests in flight: stage() then waits for all of them
              uint32_t v = 0;
#pragma unroll
              for (int q = 0; q < 4; ++q) v |= uint32_t(load_global<uint8_t>(wssrc[i] + at + q)) << (8 * q);
              reinterpret_cast<Scales*>(lds + NS * sizeof(MxStage<MF>))->w[sb][wave * 32 + i * RPR + srow][sword] = v;
            }
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
          lds_load16(base + offsetof(MxStage<MF>, w) + uint32_t(wave) * 4096u + i * 1024u, wbase[i] + uint64_t(uint32_t(ks) * 128u), half ? woff_half : woff[i & 1]);
#pragma unroll
        for (int i = 0; i < MF; ++i)
          lds_load16(base + offsetof(MxStage<MF>, t) + uint32_t(i) * 4096u + uint32_t(wave) * 1024u, tsrc[i] + uint32_t(ks) * 256u - (half ? tback : 0));
      };
      v4f acc[MF][2];
#pragma unroll
      for (int m = 0; m < MF; ++m) acc[m][0] = acc[m][1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      // the previous unit's last stage has been read; whatever it requested it has waited for
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
      for (int b = 0; b < NS - 1; ++b)
        if (b < KS) request(b, b);
      auto stage = [&](int ks, int b) {
        // what this stage needs has landed; younger are the requests of the next one where there are three buffers
        if (NS == 2 || !words || ks + NS - 1 > KS) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else if ((ks + 1) % SG != 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPS) : "memory");
        else if (tq == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPS + WR) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPS + WR + 1) : "memory");
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the stage is there for every wave, the buffer before it is free
        if (ks + NS - 1 < KS) request(ks + NS - 1, (b + NS - 1) % NS);
        const MxStage<MF>& st = *reinterpret_cast<const MxStage<MF>*>(lds + b * sizeof(MxStage<MF>));
        const Scales& sc = *reinterpret_cast<const Scales*>(lds + NS * sizeof(MxStage<MF>));
        const uint8_t* wsl = reinterpret_cast<const uint8_t*>(sc.w[(ks / SG) & 1][wave * 32 + r16]) + (ks % SG) * 8 + c;
        const uint8_t* tsl = reinterpret_cast<const uint8_t*>(sc.t[(ks / SG) & 1][r16]) + (ks % SG) * 8 + c;
        auto multiply = [&](int s) {
          v8i wf[2];
          int wsc[2];
#pragma unroll
          for (int f = 0; f < 2; ++f) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(st.w + wave * 4096 + f * 2048 + (s ? wrd1 : wrd0));
            wf[f] = v8i{int(v[0]), int(v[1]), int(v[2]), int(v[3]), 0, 0, 0, 0};
            wsc[f] = wsl[f * 16 * 8 * SG + s * 4];
          }
#pragma unroll
          for (int m = 0; m < MF; ++m) {
            const uint8_t* tb = st.t + (16 * m + r16) * 256;
            const u32x4 lo = *reinterpret_cast<const u32x4*>(tb + (((8 * s + c) ^ r16) << 4)), hi = *reinterpret_cast<const u32x4*>(tb + (((8 * s + 4 + c) ^ r16) << 4));
            const int tsc = tsl[m * 16 * 8 * SG + s * 4];
            const v8i tok = {int(lo[0]), int(lo[1]), int(lo[2]), int(lo[3]), int(hi[0]), int(hi[1]), int(hi[2]), int(hi[3])};
#pragma unroll
            for (int f = 0; f < 2; ++f) acc[m][f] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[f], tok, acc[m][f], 4, 0, 0, wsc[f], 0, tsc);
          }
        };
        multiply(0);
        if (!(ragged && ks == KS - 1)) multiply(1);
      };
      for (int ks = 0; ks < KS; ks += NS) {
#pragma unroll
        for (int b = 0; b < NS; ++b)
          if (ks + b < KS) stage(ks + b, b);
      }

#pragma unroll
      for (int m = 0; m < MF; ++m) {
        const int token = 16 * m + r16;
        if (token >= d.n) continue;
        const int pos = d.start + token;
        if (MODE == 0) {
          const int col = column(0);
          if (col + 16 <= N) {
            const float wk = p.weights ? load_global<float>(p.weights + load_global<int>(p.perm + pos)) : 1.0f;
            uint32_t o[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = mx_swiglu(acc[m][0][r], acc[m][1][r], wk, p.limit);
            *reinterpret_cast<u32x2*>(p.out + size_t(pos) * N + col + 4 * c) = u32x2{o[0] | (o[1] << 16), o[2] | (o[3] << 16)};
          }
        } else {
          const int a = load_global<int>(p.perm + pos);
#pragma unroll
          for (int f = 0; f < 2; ++f) {
            const int col = column(f);
            if (col + 16 <= N)
              *reinterpret_cast<u32x2*>(p.out + size_t(a) * N + col + 4 * c) = u32x2{pack_bf16x2(acc[m][f][0], acc[m][f][1]), pack_bf16x2(acc[m][f][2], acc[m][f][3])};
          }
          if (p.done && d.t == 0 && wave == 0 && lane < 16) p.done[a] = 1u;
        }
      }
    };
    if (d.n <= 16) run(std::integral_constant<int, 1>{});
    else if (d.n <= 32) run(std::integral_constant<int, 2>{});
    else run(std::integral_constant<int, 4>{});
  }
}

}  // namespace ffmoe
