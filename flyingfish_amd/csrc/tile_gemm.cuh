// Dense W8A8 GEMM over many rows: a 128 x 128 output tile per block of four waves, both operands through
// LDS by direct loads (global_load_lds), two blocks per CU.
//
// Same arithmetic as k_w8a8_grouped (w8a8_gemm.cuh), instruction for instruction, so the same bits: one
// v_mfma_f32_16x16x128_f8f6f4 per 16 x 16 tile and K block, total = fma(block sum, sw * sx, total).
//
// What bounds it: operand traffic on its way into the CU. k_w8a8_grouped gives every wave 64 weight rows x 64 tokens, moves
// the weights through registers into a wave-private transposition buffer and so passes 24 KB through LDS per 16 matrix
// instructions; its cache-resident rate stays near 1.2 PFLOP/s. Here two waves share each operand half, nothing goes through
// registers on its way in, and a wave's 16 instructions read 16 KB; the 32 KB of a K block are requested one K block ahead
// and land while the previous one is multiplied. Two independent blocks per CU (72 KB of LDS each) cover each other's
// barriers, first loads and epilogues. Measured, steady clocks: 4096 x 7168 -> 4096 in 122 us = 1.97 PFLOP/s (129 while a wave fetched its
// 64 token scales per K block, a line look-up per token; 157 with that and bank conflicts in every operand read), 2048 x 2048 -> 7168 41 us.
#pragma once
#include "mx_gemm.cuh"
#include "w16_gemm.cuh"
#include "lds_load.cuh"

namespace ffmoe {

// Waves: wave / 2 is the weight half (64 rows), wave % 2 the token half (64 tokens). LDS rows are 128 bytes, 16-byte piece
// c of row r at c ^ lds_key(r); the swizzle is applied to the source address, since a direct load writes its lanes in order.
// MX: E4M3 weights with one E8M0 scale per 32 x 32 block against E4M3 activations with one per 32 columns (mx_gemm.cuh's dense form, the
// same bits): the matrix core applies the scales and sums over the whole contraction. 1500 tokens at hidden 7168 / intermediate 2048:
// gate/up 142 -> 88 us, down 70 -> 39 us against 64-row units with the weights requested in operand order.
// BF16: BF16 weights and activations, no scales: a stage is 64 columns, two matrix instructions, summed in one chain as in w16_gemm.cuh.
// BF16_SPLIT: the same, summed as dense_splitk.cuh does: eight partial sums over the columns that its waves take, added in their order.
// A tile walks the partial sums one behind the other: K a multiple of 1024, two stages of every sixteen, else contiguous eighths, whose
// ends may halve a stage (K a multiple of 256). So either takes over rows of its kernel with the same bits. 1021 tokens, hidden
// 7168 / intermediate 2048: 122 + 78 -> 85 + 36 us against the 64-row kernel.
enum TileForm { TILE_W8A8, TILE_MX, TILE_BF16, TILE_BF16_SPLIT };
template <int MODE, TileForm FORM>
__global__ __launch_bounds__(256, 2) void k_dense_tile(const GemmParams p) {
  constexpr bool MX = FORM == TILE_MX, SPLIT = FORM == TILE_BF16_SPLIT, BF = FORM == TILE_BF16 || SPLIT;
  struct Stage { uint8_t w[128 * 128]; uint8_t t[128 * 128]; };
  __shared__ __attribute__((aligned(16))) Stage stage[2];
  __shared__ float sx_lds[2][128][8];  // token scales of eight K blocks
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = uni(tid >> 6);
  const int wr = wave >> 1, wt = wave & 1;
  const int K = BF ? 2 * p.K : p.K, N = p.N, KB = K >> 7;  // bytes of a row, 128 per stage
  const uint32_t total = p.total_units;
  const int ntiles = (N + (MODE == 0 ? 63 : 127)) / (MODE == 0 ? 64 : 128);
  const int groups = (p.rows_total + 127) / 128;
  const uint32_t xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3, per_xcd = gridDim.x >> 3;
  const uint32_t span = (total + 7u) >> 3;
  const uint32_t span_end = min(total, (xcd + 1u) * span);
  const uint32_t lds_w[2] = {lds_address(stage[0].w) + uint32_t(wave) * 4096u, lds_address(stage[1].w) + uint32_t(wave) * 4096u};
  const uint32_t lds_t[2] = {lds_address(stage[0].t) + uint32_t(wave) * 4096u, lds_address(stage[1].t) + uint32_t(wave) * 4096u};
  const uint32_t lds_s = lds_address(sx_lds) + uint32_t(wave) * 1024u;
  const uint32_t woff = uint32_t(lane >> 3) * uint32_t(K) + uint32_t(((lane & 7) ^ lds_key(lane >> 3)) << 4);  // odd requests: piece ^ 4
  // operand reads: row lane % 16, bytes 32 c .. 32 c + 31 of the K block for lane group c
  // (MX: bytes 16 c .. 16 c + 15 and 64 + 16 c .. 64 + 16 c + 15, the operand form whose scales sit in lane group column / 32;
  // BF16: 16 columns of a lane, the first eight in the first instruction; BF16_SPLIT: 32 columns of the stage per instruction)
  const int r16 = lane & 15, c = lane >> 4, c_lo = MX || SPLIT ? c : 2 * c, c_hi = MX || SPLIT ? c + 4 : 2 * c + 1;
  const int rd_lo = r16 * 128 + ((c_lo ^ lds_key(r16)) << 4), rd_hi = r16 * 128 + ((c_hi ^ lds_key(r16)) << 4);

  for (uint32_t u = xcd * span + slot; u < span_end; u += per_xcd) {
    // blocks of eight column tiles, row groups inside: the blocks of an XCD run an 8 x 8 window of tiles (4096 x 7168 -> 4096:
    // 172 -> 158 us against row groups innermost, whose window is 2 x 32)
    const int tb = int(u) / (groups * 8), v = int(u) - tb * groups * 8;
    const int width = min(8, ntiles - tb * 8);
    const int t = tb * 8 + v % width, start = (v / width) * 128, n = min(128, p.rows_total - start);
    const uint64_t wc[2] = {p.w0_codes, MODE == 0 ? p.w1_codes : p.w0_codes}, ws[2] = {p.w0_scales, MODE == 0 ? p.w1_scales : p.w0_scales};
    // Output column of this wave's fragment f; fragments past N are clamped onto the last 16 rows and dropped at the store.
    // MODE 0: fragments 0, 1 are gate rows, 2, 3 the up rows of the same columns.
    auto column = [&](int half, int f) { return MODE == 0 ? t * 64 + half * 32 + (f & 1) * 16 : t * 128 + half * 64 + f * 16; };
    uint64_t wbase[4];  // request i of this wave: eight weight rows of fragment 2 (wave % 2) + i / 2 of weight half wave / 2
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int f = 2 * wt + (i >> 1);
      wbase[i] = uni64((MODE == 0 ? wc[f >> 1] : wc[0]) + uint64_t(min(column(wr, f), N - 16) + (i & 1) * 8) * uint64_t(K));
    }
    const uint8_t* tsrc[4];  // request i: token rows 32 wave + 8 i + lane / 8
    auto token_row = [&](int m) { return start + min(m, n - 1); };
#pragma unroll
    for (int i = 0; i < 4; ++i) tsrc[i] = p.a_codes + size_t(token_row(wave * 32 + i * 8 + (lane >> 3))) * K + (((lane & 7) ^ lds_key(lane >> 3) ^ 4 * (i & 1)) << 4);
    // Block scales, one word per K block; lane l keeps K block l (+ 64). A wave's columns sit inside one 128-row block; MX: four
    // bytes per 32 rows, which are the wave's fragments 0, 1 and its fragments 2, 3.
    [[maybe_unused]] const float* sw0 = reinterpret_cast<const float*>(ws[0]) + size_t(min(column(wr, 0), N - 16) >> (MX ? 5 : 7)) * KB;
    [[maybe_unused]] const float* sw1 = reinterpret_cast<const float*>(ws[1]) + size_t(min(column(wr, MX ? 2 : 0), N - 16) >> (MX ? 5 : 7)) * KB;

    auto request = [&](int kb, int b) {
#pragma unroll
      for (int i = 0; i < 4; ++i) lds_load16(lds_w[b] + i * 1024u, wbase[i] + uint64_t(uint32_t(kb) * 128u), woff ^ (64u * (i & 1)));
#pragma unroll
      for (int i = 0; i < 4; ++i) lds_load16(lds_t[b] + i * 1024u, tsrc[i] + uint32_t(kb) * 128u);
      // Token scales, a row of KB words per token (MX: the four scale bytes of a K block are one word): a request takes eight K blocks of
      // eight tokens. One K block of 64 tokens per request touches a line per lane, as many line look-ups as the operands themselves.
      if (!BF && (kb & 7) == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          lds_load4(lds_s + uint32_t((kb >> 3) & 1) * 4096u + i * 256u, p.a_scales + size_t(token_row(wave * 32 + i * 8 + (lane >> 3))) * KB + min(kb + (lane & 7), KB - 1));
      }
    };
    __syncthreads();  // the previous unit's last tile has been read
    request(0, 0);

    float acc[4][4][4];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[m][f][r] = 0.0f;

    // SPLIT: the sum of the partial sums so far (the first one is added to -0.0, which leaves it as it is), the stage asked for last, as the
    // j-th of partial sum w, and the 32-column steps since the last partial sum ended
    [[maybe_unused]] float tot[SPLIT ? 4 : 1][4][4];
    if constexpr (SPLIT) {
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
          for (int r = 0; r < 4; ++r) tot[m][f][r] = -0.0f;
    }
    [[maybe_unused]] const int part_steps = KB >> 2;       // of 32 columns
    [[maybe_unused]] const bool dealt = part_steps % 4 == 0;
    [[maybe_unused]] int ask_w = 0, ask_j = 0, steps = 0;
    auto next_stage = [&](int q) {  // where the q-th stage of the walk is
      if constexpr (!SPLIT) return q;
      if (!dealt) return q;
      if (++ask_j == part_steps >> 1) { ask_j = 0; ++ask_w; }
      return ((ask_j >> 1) * 8 + ask_w) * 2 + (ask_j & 1);
    };

    auto block = [&](int kb, int b, float s0, float s1) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();  // K block kb is there for every wave, and nobody reads the other buffer any more
      if (kb + 1 < KB) request(next_stage(kb + 1), b ^ 1);
      const uint8_t* wl = stage[b].w + wr * 8192;
      const uint8_t* tl = stage[b].t + wt * 8192;
      const float* sl = &sx_lds[(kb >> 3) & 1][wt * 64 + r16][kb & 7];
      v8i wf[4];
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const u32x4 lo = *reinterpret_cast<const u32x4*>(wl + f * 2048 + rd_lo), hi = *reinterpret_cast<const u32x4*>(wl + f * 2048 + rd_hi);
        wf[f] = v8i{int(lo[0]), int(lo[1]), int(lo[2]), int(lo[3]), int(hi[0]), int(hi[1]), int(hi[2]), int(hi[3])};
      }
      u32x4 tlo[2], thi[2];
      float sx[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) sx[m] = BF ? 1.0f : sl[16 * 8 * m];
      tlo[0] = *reinterpret_cast<const u32x4*>(tl + rd_lo);
      thi[0] = *reinterpret_cast<const u32x4*>(tl + rd_hi);
      if constexpr (BF) {
        auto half = [](const v8i& v, int h) { return __builtin_bit_cast(w16_bf16x8, u32x4{uint32_t(v[4 * h]), uint32_t(v[4 * h + 1]), uint32_t(v[4 * h + 2]), uint32_t(v[4 * h + 3])}); };
        auto multiply = [&](const u32x4& token, int m, int h) {
#pragma unroll
          for (int f = 0; f < 4; ++f) {
            v4f t4 = {acc[m][f][0], acc[m][f][1], acc[m][f][2], acc[m][f][3]};
            t4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(half(wf[f], h), __builtin_bit_cast(w16_bf16x8, token), t4, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[m][f][r] = t4[r];
          }
        };
        if constexpr (SPLIT) {
          u32x4 tok[4];
#pragma unroll
          for (int m = 0; m < 4; ++m) tok[m] = *reinterpret_cast<const u32x4*>(tl + m * 2048 + rd_lo);
#pragma unroll
          for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int m = 0; m < 4; ++m) {
              multiply(tok[m], m, h);
              if (h == 0) tok[m] = *reinterpret_cast<const u32x4*>(tl + m * 2048 + rd_hi);
            }
            if (++steps == part_steps) {
              steps = 0;
#pragma unroll
              for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int f = 0; f < 4; ++f)
#pragma unroll
                  for (int r = 0; r < 4; ++r) {
                    tot[m][f][r] = __fadd_rn(tot[m][f][r], acc[m][f][r]);
                    acc[m][f][r] = 0.0f;
                  }
            }
          }
        } else {
#pragma unroll
          for (int m = 0; m < 4; ++m) {
            if (m + 1 < 4) {
              tlo[(m + 1) & 1] = *reinterpret_cast<const u32x4*>(tl + (m + 1) * 2048 + rd_lo);
              thi[(m + 1) & 1] = *reinterpret_cast<const u32x4*>(tl + (m + 1) * 2048 + rd_hi);
            }
            multiply(tlo[m & 1], m, 0);
            multiply(thi[m & 1], m, 1);
          }
        }
        return;
      }
      if constexpr (MX) {
        const int w0 = int((__float_as_uint(s0) >> (8 * c)) & 0xffu), w1 = int((__float_as_uint(s1) >> (8 * c)) & 0xffu);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          if (m + 1 < 4) {
            tlo[(m + 1) & 1] = *reinterpret_cast<const u32x4*>(tl + (m + 1) * 2048 + rd_lo);
            thi[(m + 1) & 1] = *reinterpret_cast<const u32x4*>(tl + (m + 1) * 2048 + rd_hi);
          }
          const u32x4 lo = tlo[m & 1], hi = thi[m & 1];
          const v8i tok = {int(lo[0]), int(lo[1]), int(lo[2]), int(lo[3]), int(hi[0]), int(hi[1]), int(hi[2]), int(hi[3])};
          const int ts = int((__float_as_uint(sx[m]) >> (8 * c)) & 0xffu);
#pragma unroll
          for (int f = 0; f < 4; ++f) {
            v4f t4 = {acc[m][f][0], acc[m][f][1], acc[m][f][2], acc[m][f][3]};
            t4 = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[f], tok, t4, 0, 0, 0, f >= 2 ? w1 : w0, 0, ts);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[m][f][r] = t4[r];
          }
        }
        return;
      }
      v4f pr[2][4];
      // row fragment m's products are folded into the totals while fragment m + 1 is in the matrix core
#pragma unroll
      for (int m = 0; m <= 4; ++m) {
        if (m < 4) {
          if (m + 1 < 4) {
            tlo[(m + 1) & 1] = *reinterpret_cast<const u32x4*>(tl + (m + 1) * 2048 + rd_lo);
            thi[(m + 1) & 1] = *reinterpret_cast<const u32x4*>(tl + (m + 1) * 2048 + rd_hi);
          }
          const u32x4 lo = tlo[m & 1], hi = thi[m & 1];
          const v8i tok = {int(lo[0]), int(lo[1]), int(lo[2]), int(lo[3]), int(hi[0]), int(hi[1]), int(hi[2]), int(hi[3])};
#pragma unroll
          for (int f = 0; f < 4; ++f) pr[m & 1][f] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[f], tok, v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0, 0, 0, 0);
        }
        if (m > 0) {
          const float sc0 = __fmul_rn(s0, sx[m - 1]), sc1 = __fmul_rn(s1, sx[m - 1]);
#pragma unroll
          for (int f = 0; f < 4; ++f)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[m - 1][f][r] = __fmaf_rn(pr[(m - 1) & 1][f][r], (MODE == 0 && f >= 2) ? sc1 : sc0, acc[m - 1][f][r]);
          // pins the fmas in front of the fence: without it they all end up behind the last one, after the matrix work
#pragma unroll
          for (int f = 0; f < 4; ++f)
#pragma unroll
            for (int r = 0; r < 4; ++r) asm volatile("" ::"v"(acc[m - 1][f][r]));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    for (int kb0 = 0; kb0 < KB; kb0 += 64) {
      const int kl = min(kb0 + lane, KB - 1);
      const float swl0 = BF ? 1.0f : landed(load_global<float>(sw0 + kl));
      const float swl1 = !BF && (MODE == 0 || MX) ? landed(load_global<float>(sw1 + kl)) : swl0;
      const int kend = min(KB, kb0 + 64);
      auto scale = [&](float v, int kb) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), kb - kb0)); };
      for (int kb = kb0; kb < kend; kb += 2) {  // kb0 is even: buffer = parity of the K block
        block(kb, 0, scale(swl0, kb), scale(swl1, kb));
        if (kb + 1 < kend) block(kb + 1, 1, scale(swl0, kb + 1), scale(swl1, kb + 1));
      }
    }

    if constexpr (SPLIT) {
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[m][f][r] = tot[m][f][r];
    }
    const int sub = (lane >> 4) * 4;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int token = wt * 64 + 16 * m + r16;
      if (token < n) {
        const int pos = start + token;
        if (MODE == 0) {
#pragma unroll
          for (int f = 0; f < 2; ++f) {
            const int col = column(wr, f);
            if (col + 16 <= N) {
              uint32_t o[4];
#pragma unroll
              for (int r = 0; r < 4; ++r) o[r] = MX ? mx_swiglu(acc[m][f][r], acc[m][f + 2][r], 1.0f, p.limit) : BF ? swiglu_bf16(bround(acc[m][f][r]), bround(acc[m][f + 2][r]), p.swiglu, p.limit) : swiglu_bf16_two_branch(bround(acc[m][f][r]), bround(acc[m][f + 2][r]), p.swiglu, p.limit);
              *reinterpret_cast<u32x2*>(p.out + size_t(pos) * N + col + sub) = u32x2{o[0] | (o[1] << 16), o[2] | (o[3] << 16)};
            }
          }
        } else {
#pragma unroll
          for (int f = 0; f < 4; ++f) {
            const int col = column(wr, f);
            if (col + 16 <= N)
              *reinterpret_cast<u32x2*>(p.out + size_t(pos) * N + col + sub) = u32x2{pack_bf16x2(acc[m][f][0], acc[m][f][1]), pack_bf16x2(acc[m][f][2], acc[m][f][3])};
          }
        }
      }
    }
  }
}

}  // namespace ffmoe
