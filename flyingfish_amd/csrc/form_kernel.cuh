// Decode expert FFN in the reference's own reduction orders, bit for bit.
//
// The reference keeps two summation orders for an expert dot product and its CPU path reproduces both exactly
// (src/cpu/expert_ffn.rs:689-776, `Form::Lane16` and `Form::Lane8`), so that a layer may run some experts on the CPU and
// some on the GPU with identical results; on the GPU they are the "invariant" kernels moe_ffn_*_lane16
// (kernels/moe_ffn.cu:364-393) and the production kernels moe_gate_up / moe_down (kernels/moe_ffn.cu:98-302):
//
//   Lane16: 16 accumulators; element k goes to accumulator k % 16 by fused multiply-add in ascending k; the result is
//           ((l0+l1)+(l2+l3))+((l4+l5)+(l6+l7)) + the same of l8..l15  (expert_ffn.rs:681-687).
//   Lane8:  every vector of 8 consecutive elements is summed by a fused multiply-add chain starting from 0; vector v is
//           ADDED to accumulator v % 8; the result is ((l0+l4)+(l2+l6))+((l1+l5)+(l3+l7))  (expert_ffn.rs:37-41).
//
// The streaming kernels of decode_kernel.cuh use one 64-lane sum per row and match these only to tolerance. The
// kernels here keep the orders exactly: Lane16 gives two hardware lanes to a row, each holding 8 of the 16
// accumulators in registers (elements 16i .. 16i+7 and 16i+8 .. 16i+15 are contiguous, so each lane still loads whole
// words); Lane8 gives eight hardware lanes to a row, lane l taking the vectors v = l, l+8, ...; the final trees are
// lane-pair exchanges in the order above. Activation roundings are those of the streaming kernels. SiLU follows the
// reference per form: g / (1 + exp(-g)) for Lane8 and for Lane16 with one rounding, g * (1 / (1 + exp(-g))) for Lane16
// with two roundings (kernels/moe_ffn.cu:58, :201-203).
//
// Formats: BF16 and per-channel FP8 experts, the formats the reference's CPU path executes.
#pragma once
#include "decode_kernel.cuh"

namespace ffmoe {

#define FFMOE_FORM_LANE16_ 0
#define FFMOE_FORM_LANE8_ 1

// 8 consecutive effective weights of a row as FP32, from element k0 (a multiple of 8)
template <class F>
struct FormRow;

template <>
struct FormRow<FmtBf16> {
  const uint16_t* w;
  __device__ __forceinline__ FormRow(uint64_t codes, uint64_t, int j, int K) : w(reinterpret_cast<const uint16_t*>(codes) + size_t(j) * K) {}
  __device__ __forceinline__ void load8(int k0, float (&o)[8]) const {
    const u32x4 v = load16(w + k0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[2 * i] = __uint_as_float(v[i] << 16);
      o[2 * i + 1] = __uint_as_float(v[i] & 0xffff0000u);
    }
  }
};

template <>
struct FormRow<FmtFp8Channel> {
  const uint8_t* w;
  float scale;
  __device__ __forceinline__ FormRow(uint64_t codes, uint64_t scales, int j, int K)
      : w(reinterpret_cast<const uint8_t*>(codes) + size_t(j) * K), scale(bf16_to_f32(reinterpret_cast<const uint16_t*>(scales)[j])) {}
  __device__ __forceinline__ void load8(int k0, float (&o)[8]) const {
    const u32x2 v = load_global<u32x2>(w + k0);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      uint32_t w01, w23;
      dequant4_e4m3(v[i], scale, w01, w23);  // bf16(e4m3 * scale), src/fp8.rs:138-140
      o[4 * i] = __uint_as_float(w01 << 16);
      o[4 * i + 1] = __uint_as_float(w01 & 0xffff0000u);
      o[4 * i + 2] = __uint_as_float(w23 << 16);
      o[4 * i + 3] = __uint_as_float(w23 & 0xffff0000u);
    }
  }
};

// 8 consecutive BF16 activations from LDS as FP32
__device__ __forceinline__ void form_x8(const uint8_t* xs, int k0, float (&o)[8]) {
  const u32x4 v = *reinterpret_cast<const u32x4*>(xs + size_t(k0) * 2);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o[2 * i] = __uint_as_float(v[i] << 16);
    o[2 * i + 1] = __uint_as_float(v[i] & 0xffff0000u);
  }
}

__device__ __forceinline__ float lane_xor(float v, int mask) { return __shfl_xor(v, mask, 64); }

// Dot product of the LDS row xs[0..K) with one weight row in the given form. `sub` is this lane's index inside the
// row's lane group (Lane16: 0..1, Lane8: 0..7); every lane of the group returns the result.
template <class F, int FORM>
__device__ __forceinline__ float form_dot(const uint8_t* xs, const FormRow<F>& row, int K, int sub) {
  float x[8], w[8];
  if (FORM == FFMOE_FORM_LANE16_) {
    float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    // this lane owns accumulators 8*sub .. 8*sub+7: elements 16i + 8*sub + t. A last half step (K % 16 == 8) belongs
    // to accumulators 0..7, i.e. to sub 0 only.
    for (int k0 = 8 * sub; k0 < K; k0 += 16) {
      form_x8(xs, k0, x);
      row.load8(k0, w);
#pragma unroll
      for (int t = 0; t < 8; ++t) acc[t] = __fmaf_rn(x[t], w[t], acc[t]);
    }
    const float half = __fadd_rn(__fadd_rn(__fadd_rn(acc[0], acc[1]), __fadd_rn(acc[2], acc[3])),
                                 __fadd_rn(__fadd_rn(acc[4], acc[5]), __fadd_rn(acc[6], acc[7])));
    const float other = lane_xor(half, 1);
    return sub == 0 ? __fadd_rn(half, other) : __fadd_rn(other, half);  // low + high
  }
  float acc = 0.0f;
  for (int k0 = 8 * sub; k0 < K; k0 += 64) {  // vectors sub, sub + 8, ...
    form_x8(xs, k0, x);
    row.load8(k0, w);
    float inner = 0.0f;
#pragma unroll
    for (int t = 0; t < 8; ++t) inner = __fmaf_rn(x[t], w[t], inner);
    acc = __fadd_rn(acc, inner);
  }
  // ((l0+l4)+(l2+l6)) + ((l1+l5)+(l3+l7)): partners 4, 2, 1; the lower lane index is the left operand
  float o = lane_xor(acc, 4);
  acc = (sub & 4) ? __fadd_rn(o, acc) : __fadd_rn(acc, o);
  o = lane_xor(acc, 2);
  acc = (sub & 2) ? __fadd_rn(o, acc) : __fadd_rn(acc, o);
  o = lane_xor(acc, 1);
  acc = (sub & 1) ? __fadd_rn(o, acc) : __fadd_rn(acc, o);
  return acc;
}

// SwiGLU with the reference's SiLU per form (see the file comment)
__device__ __forceinline__ uint16_t form_swiglu(float g, float u, int mode, float limit, bool reciprocal) {
  if (mode == FFMOE_SWIGLU_GELU_TWICE) return f32_to_bf16(__fmul_rn(bround(gelu_tanh(g)), u));
  if (mode >= 2) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
  }
  const float den = __fadd_rn(1.0f, det_expf(-g));
  const float act = reciprocal ? __fmul_rn(g, __fdiv_rn(1.0f, den)) : __fdiv_rn(g, den);
  const float prod = (mode == 0 || mode == 2) ? __fmul_rn(bround(act), u) : __fmul_rn(act, u);
  return f32_to_bf16(prod);
}

// grid (ceil(out / ROWS), rows, top_k + 1): block z < top_k is choice z of token row y, z == top_k the shared expert
// (the reference's launch shape, src/backend/cuda/moe/decode.rs:486-514). STAGE 0: gate/up + SwiGLU -> h,
// STAGE 1: down (+ routing weight) -> contributions / shared_out.
template <class F, int FORM, int STAGE>
__global__ __launch_bounds__(256) void k_decode_form(const DecodeParams p) {
  constexpr int LPR = FORM == FFMOE_FORM_LANE16_ ? 2 : 8;  // hardware lanes per output row
  constexpr int ROWS = 256 / LPR;
  extern __shared__ __align__(16) uint8_t xs[];
  const int tid = threadIdx.x;
  const int r = blockIdx.y, z = blockIdx.z;
  const bool is_shared = z == p.top_k;
  if (is_shared && !p.has_shared) return;
  const int A = p.rows * p.top_k;
  int expert, gn, grow[1], gslot[1];
  load_group<1>(p, is_shared ? A + r : r * p.top_k + z, expert, gn, grow, gslot);
  if (gn == 0) return;  // inactive, invalid or stale choice: nothing written, done stays 0
  const int Kg = STAGE == 0 ? p.hidden : (is_shared ? p.shared_inter : p.inter);
  const int out = STAGE == 0 ? (is_shared ? p.shared_inter : p.inter) : p.hidden;
  if (int(blockIdx.x) * ROWS >= out) return;
  {
    const uint16_t* src = STAGE == 0 ? p.x + size_t(r) * p.hidden : p.h + size_t(gslot[0]) * p.h_stride;
    u32x4* d4 = reinterpret_cast<u32x4*>(xs);
    for (int v = tid; v < (Kg >> 3); v += 256) d4[v] = load16(src + size_t(v) * 8);
  }
  __syncthreads();
  const int j = blockIdx.x * ROWS + tid / LPR;
  const int sub = tid % LPR;
  if (j >= out) return;
  uint64_t sl[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) sl[i] = is_shared ? p.shared_slot[i] : p.slots[size_t(expert) * 6 + i];
  if (STAGE == 0) {
    const FormRow<F> gate(sl[0], sl[1], j, Kg), up(sl[2], sl[3], j, Kg);
    const float g = form_dot<F, FORM>(xs, gate, Kg, sub);
    const float u = form_dot<F, FORM>(xs, up, Kg, sub);
    const bool reciprocal = FORM == FFMOE_FORM_LANE16_ && (p.swiglu == FFMOE_SWIGLU_TWICE || p.swiglu == FFMOE_SWIGLU_CLAMPED_TWICE);
    if (sub == 0) p.h[size_t(gslot[0]) * p.h_stride + j] = form_swiglu(bround(g), bround(u), p.swiglu, p.swiglu_limit, reciprocal);
  } else {
    const FormRow<F> down(sl[4], sl[5], j, Kg);
    const float d = form_dot<F, FORM>(xs, down, Kg, sub);
    if (sub == 0) {
      if (is_shared) {
        p.shared_out[size_t(r) * p.hidden + j] = f32_to_bf16(d);
      } else {
        const float wk = p.weights_f32 ? reinterpret_cast<const float*>(p.weights)[gslot[0]]
                                       : bf16_to_f32(reinterpret_cast<const uint16_t*>(p.weights)[gslot[0]]);
        const float v = __fmul_rn(p.routed_weight == FFMOE_WEIGHT_AFTER_DOWN_BF16 ? bround(d) : d, wk);
        p.contributions[size_t(gslot[0]) * p.hidden + j] = f32_to_bf16(v);
        if (j == 0 && p.done) p.done[gslot[0]] = 1u;
      }
    }
  }
}

// The same dot product for up to RG activation rows at once: a weight word is loaded once and every row keeps its own
// accumulators, so each (row, column) result is the chain of form_dot bit for bit. n = live rows (uniform in the block).
template <class F, int FORM, int RG>
__device__ __forceinline__ void form_dot_rows(const uint8_t* xs, int xstride, int n, const FormRow<F>& row, int K, int sub, float (&out)[RG]) {
  float x[8], w[8];
  if (FORM == FFMOE_FORM_LANE16_) {
    float acc[RG][8];
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
      for (int t = 0; t < 8; ++t) acc[r][t] = 0.0f;
    for (int k0 = 8 * sub; k0 < K; k0 += 16) {
      row.load8(k0, w);
#pragma unroll
      for (int r = 0; r < RG; ++r) {
        if (r < n) {
          form_x8(xs + size_t(r) * xstride, k0, x);
#pragma unroll
          for (int t = 0; t < 8; ++t) acc[r][t] = __fmaf_rn(x[t], w[t], acc[r][t]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < RG; ++r) {
      const float half = __fadd_rn(__fadd_rn(__fadd_rn(acc[r][0], acc[r][1]), __fadd_rn(acc[r][2], acc[r][3])),
                                   __fadd_rn(__fadd_rn(acc[r][4], acc[r][5]), __fadd_rn(acc[r][6], acc[r][7])));
      const float other = lane_xor(half, 1);
      out[r] = sub == 0 ? __fadd_rn(half, other) : __fadd_rn(other, half);
    }
    return;
  }
  float acc[RG];
#pragma unroll
  for (int r = 0; r < RG; ++r) acc[r] = 0.0f;
  for (int k0 = 8 * sub; k0 < K; k0 += 64) {
    row.load8(k0, w);
#pragma unroll
    for (int r = 0; r < RG; ++r) {
      if (r < n) {
        form_x8(xs + size_t(r) * xstride, k0, x);
        float inner = 0.0f;
#pragma unroll
        for (int t = 0; t < 8; ++t) inner = __fmaf_rn(x[t], w[t], inner);
        acc[r] = __fadd_rn(acc[r], inner);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RG; ++r) {
    float a = acc[r];
    float o = lane_xor(a, 4);
    a = (sub & 4) ? __fadd_rn(o, a) : __fadd_rn(a, o);
    o = lane_xor(a, 2);
    a = (sub & 2) ? __fadd_rn(o, a) : __fadd_rn(a, o);
    o = lane_xor(a, 1);
    a = (sub & 1) ? __fadd_rn(o, a) : __fadd_rn(a, o);
    out[r] = a;
  }
}

// Token-sorted form of k_decode_form: grid (ceil(out / ROWS), groups). A block takes one group of up to RG assignments of
// one expert (k_group_assignments; the shared expert's rows come as groups of their own), stages their activation rows
// in LDS and streams each weight row once for all of them. The reference's grouped kernels read a weight row once per
// (row, column) and leave the reuse to the cache (kernels/moe_prefill.cu:13-71); the results are the same bits.
template <class F, int FORM, int STAGE, int RG>
__global__ __launch_bounds__(256) void k_decode_form_grouped(const DecodeParams p) {
  constexpr int LPR = FORM == FFMOE_FORM_LANE16_ ? 2 : 8;
  constexpr int ROWS = 256 / LPR;
  extern __shared__ __align__(16) uint8_t xs[];
  const int tid = threadIdx.x;
  const int g = blockIdx.y;
  const int n_routed = uni(load_global<int>(p.counters)), n_shared = uni(load_global<int>(p.counters + 1));
  if (g >= n_routed + n_shared) return;
  int expert, gn, grow[RG], gslot[RG];
  load_group<RG>(p, g, expert, gn, grow, gslot);
  if (gn == 0) return;
  const bool is_shared = expert < 0;
  const int Kg = STAGE == 0 ? p.hidden : (is_shared ? p.shared_inter : p.inter);
  const int out = STAGE == 0 ? (is_shared ? p.shared_inter : p.inter) : p.hidden;
  if (int(blockIdx.x) * ROWS >= out) return;
  const int xstride = Kg * 2;
#pragma unroll
  for (int r = 0; r < RG; ++r) {
    if (r < gn) {
      const uint16_t* src = STAGE == 0 ? p.x + size_t(grow[r]) * p.hidden : p.h + size_t(gslot[r]) * p.h_stride;
      u32x4* d4 = reinterpret_cast<u32x4*>(xs + size_t(r) * xstride);
      for (int v = tid; v < (Kg >> 3); v += 256) d4[v] = load16(src + size_t(v) * 8);
    }
  }
  __syncthreads();
  const int j = blockIdx.x * ROWS + tid / LPR;
  const int sub = tid % LPR;
  if (j >= out) return;
  uint64_t sl[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) sl[i] = is_shared ? p.shared_slot[i] : p.slots[size_t(expert) * 6 + i];
  if (STAGE == 0) {
    const FormRow<F> gate(sl[0], sl[1], j, Kg), up(sl[2], sl[3], j, Kg);
    float gv[RG], uv[RG];
    form_dot_rows<F, FORM, RG>(xs, xstride, gn, gate, Kg, sub, gv);
    form_dot_rows<F, FORM, RG>(xs, xstride, gn, up, Kg, sub, uv);
    const bool reciprocal = FORM == FFMOE_FORM_LANE16_ && (p.swiglu == FFMOE_SWIGLU_TWICE || p.swiglu == FFMOE_SWIGLU_CLAMPED_TWICE);
    if (sub == 0) {
#pragma unroll
      for (int r = 0; r < RG; ++r)
        if (r < gn) p.h[size_t(gslot[r]) * p.h_stride + j] = form_swiglu(bround(gv[r]), bround(uv[r]), p.swiglu, p.swiglu_limit, reciprocal);
    }
  } else {
    const FormRow<F> down(sl[4], sl[5], j, Kg);
    float dv[RG];
    form_dot_rows<F, FORM, RG>(xs, xstride, gn, down, Kg, sub, dv);
    if (sub == 0) {
#pragma unroll
      for (int r = 0; r < RG; ++r) {
        if (r < gn) {
          if (is_shared) {
            p.shared_out[size_t(grow[r]) * p.hidden + j] = f32_to_bf16(dv[r]);
          } else {
            const float wk = p.weights_f32 ? reinterpret_cast<const float*>(p.weights)[gslot[r]]
                                           : bf16_to_f32(reinterpret_cast<const uint16_t*>(p.weights)[gslot[r]]);
            const float v = __fmul_rn(p.routed_weight == FFMOE_WEIGHT_AFTER_DOWN_BF16 ? bround(dv[r]) : dv[r], wk);
            p.contributions[size_t(gslot[r]) * p.hidden + j] = f32_to_bf16(v);
            if (j == 0 && p.done) p.done[gslot[r]] = 1u;
          }
        }
      }
    }
  }
}

// The same sums with the weights streamed through LDS (contractions that are whole 128-byte lines of every weight row; the two
// kernels above keep the others). A wave owns 32 weight rows - 16 gate rows and the up rows beside them, or 32 down rows -
// and moves them in chunks of 128 bytes a row: eight lanes request one line, the chunk goes into the wave's own LDS buffer
// (16-byte pieces XOR-swizzled by the row; LDS operations of a wave execute in order, so nothing waits between its writes
// and reads) and every lane picks out the elements of its accumulators. Requested in accumulator order instead, a row gives
// 16 bytes per request and its line is looked up in the vector L1, and often fetched, eight times.
//   Lane16: four lanes a row, four of the sixteen accumulators each, two rows per lane.
//   Lane8:  eight lanes a row, every eighth vector of 8 elements each, four rows per lane.
// A lane's rows share its reads of the activations, the tokens of a group (up to T) share the dequantization of its rows.
// Bound by the vector ALUs next to HBM: dequantizing a per-channel FP8 weight to an FP32 operand takes 3 instructions
// (conversion, scale, BF16 rounding, unpacking; pairs where the ISA has them), a token 1.5 more.
// One token, 8 of 64 experts + shared at hidden 7168 / intermediate 2048, us before / now: per-channel FP8 Lane16 336 / 94,
// Lane8 174 / 88 (397 MB: 4.5 TB/s), BF16 Lane16 420 / 148, Lane8 194 / 147 (5.4 TB/s); 4 rows at 4096 / 1536, top-6: Lane16
// 282 / 96; 32 rows at 7168, in groups: Lane16 2305 / 920. One chunk ahead is enough for the groups of one FP8 token, two chunks
// cost them waves; three or four change nothing for BF16.
template <class F, int FORM>
struct FormShape {
  static constexpr int EB = std::is_same<F, FmtBf16>::value ? 2 : 1;  // bytes per weight
  static constexpr int CH = 128 / EB;                                 // elements of a row per chunk
  static constexpr int L = FORM == FFMOE_FORM_LANE16_ ? 4 : 8;        // lanes per row
  static constexpr int NR = FORM == FFMOE_FORM_LANE16_ ? 2 : 4;       // rows per lane
  static constexpr int EL = FORM == FFMOE_FORM_LANE16_ ? 4 : 8;  // elements of a lane per step: 4 | 8
  static constexpr int STEP = FORM == FFMOE_FORM_LANE16_ ? 16 : 64;   // elements of a row per step
  static constexpr int STEPS = CH / STEP;
};
constexpr int FFMOE_FORM_WAVE_LDS = 32 * 128;

constexpr int FFMOE_FORM_SEG = 2048;  // elements of a token in LDS at a time: longer rows would leave one or two blocks per CU

struct FormTile {
  int K, out, j0;          // contraction, output columns, first column of the wave
  bool live, is_shared;
  uint64_t sl[4];          // STAGE 0: gate codes, scales, up codes, scales; STAGE 1: down codes, scales
  int gn;
};

// N: tokens of the group as a constant (gn of them exist, the others repeat the last one and store nothing): as run-time tests inside
// the loop the tokens' branches cost a group of one 40 %
template <class F, int FORM, int STAGE, int N, int T>
__device__ __forceinline__ void form_rows_run(const DecodeParams& p, const FormTile& f, const int (&grow)[T], const int (&gslot)[T], uint8_t* lds) {
  using S = FormShape<F, FORM>;
  constexpr int NR = S::NR, L = S::L, RPL = 64 / L;
  constexpr bool L16 = FORM == FFMOE_FORM_LANE16_;
  constexpr int NACC = L16 ? 4 : 1;
  constexpr int D = N == 1 && S::EB == 1 ? 1 : 2;  // chunks on their way
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = uni(tid >> 6);
  const int K = f.K;
  const int jb = f.live ? f.j0 : 0;
  const uint32_t rowb = uint32_t(K) * S::EB;
  const int NC = int(rowb >> 7);
  // rows 8 h .. 8 h + 7 of the wave's buffer: their matrix and first weight row
  uint64_t base[4];
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    const int mat = STAGE == 1 ? 0 : (L16 ? h >> 1 : h & 1);
    const int row = jb + (STAGE == 1 ? 8 * h : 8 * (L16 ? h & 1 : h >> 1));
    base[h] = f.sl[2 * mat] + uint64_t(row) * rowb;
  }
  const uint32_t loff = uint32_t(lane >> 3) * rowb + uint32_t(lane & 7) * 16u;
  u32x4 w[D][4];
  auto request = [&](int s, int c) {  // past the end: one line with every lane, nothing reads it
    const uint32_t off = c < NC ? loff + uint32_t(c) * 128u : 0u;
#pragma unroll
    for (int h = 0; h < 4; ++h) w[s][h] = load16_stream(reinterpret_cast<const uint8_t*>(base[h]) + off);
  };
#pragma unroll
  for (int s = 0; s < D; ++s) request(s, s);
  // per-channel scales of this lane's rows
  const int r = lane / L, sub = lane % L;
  float scale[NR];
#pragma unroll
  for (int n = 0; n < NR; ++n) {
    scale[n] = 1.0f;
    if constexpr (S::EB == 1) {
      const int mat = STAGE == 1 ? 0 : n & 1;
      const int row = jb + (STAGE == 1 ? n * RPL : (n >> 1) * RPL) + r;
      scale[n] = bf16_to_f32(load_global<uint16_t>(reinterpret_cast<const uint16_t*>(f.sl[2 * mat + 1]) + row));
    }
  }
  uint8_t* wl = lds + size_t(wave) * FFMOE_FORM_WAVE_LDS;
  uint8_t* xs = lds + 4 * FFMOE_FORM_WAVE_LDS;
  auto key = [](int row) { return (row ^ (row >> 3)) & 7; };
  float acc[NR][N][NACC];
#pragma unroll
  for (int n = 0; n < NR; ++n)
#pragma unroll
    for (int t = 0; t < N; ++t)
#pragma unroll
      for (int a = 0; a < NACC; ++a) acc[n][t][a] = 0.0f;
  for (int k0 = 0; k0 < K; k0 += FFMOE_FORM_SEG) {
    const int len = K - k0 < FFMOE_FORM_SEG ? K - k0 : FFMOE_FORM_SEG;
    if (k0 > 0) __syncthreads();  // the previous segment has been read
#pragma unroll
    for (int t = 0; t < N; ++t) {
      const int tt = t < f.gn ? t : f.gn - 1;
      int row = grow[0], slot = gslot[0];
#pragma unroll
      for (int q = 1; q < (N < T ? N : T); ++q) { row = tt == q ? grow[q] : row; slot = tt == q ? gslot[q] : slot; }
      const uint16_t* src = (STAGE == 0 ? p.x + size_t(row) * p.hidden : p.h + size_t(slot) * p.h_stride) + k0;
      u32x4* d4 = reinterpret_cast<u32x4*>(xs + size_t(t) * FFMOE_FORM_SEG * 2);
      if (tid < (len >> 3)) d4[tid] = load16(src + size_t(tid) * 8);
    }
    __syncthreads();
    const int c_end = f.live ? (k0 + len) / S::CH : 0;
    for (int c0 = k0 / S::CH; c0 < c_end; c0 += D) {
#pragma unroll
      for (int s = 0; s < D; ++s) {
        const int c = c0 + s;
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const int row = 8 * h + (lane >> 3);
          *reinterpret_cast<u32x4*>(wl + row * 128 + (((lane & 7) ^ key(row)) << 4)) = w[s][h];
        }
        request(s, c + D);
        __builtin_amdgcn_wave_barrier();
        if (c < c_end) {  // only the last segment can hold an odd number of chunks
          const uint8_t* xc = xs + size_t(c * S::CH - k0) * 2 + sub * (S::EL * 2);
#pragma unroll
          for (int st = 0; st < S::STEPS; ++st) {
            float wf[NR][S::EL];
#pragma unroll
            for (int n = 0; n < NR; ++n) {
              const int row = n * RPL + r;
              const int byte = (st * S::STEP + sub * S::EL) * S::EB;  // inside the row's chunk
              const uint8_t* at = wl + row * 128 + (((byte >> 4) ^ key(row)) << 4) + (byte & 15);
              if constexpr (S::EB == 1) {
                uint32_t d[S::EL / 4];
                if constexpr (S::EL == 4) d[0] = *reinterpret_cast<const uint32_t*>(at);
                else { const u32x2 v = *reinterpret_cast<const u32x2*>(at); d[0] = v.x; d[1] = v.y; }
#pragma unroll
                for (int q = 0; q < S::EL / 4; ++q) {
                  uint32_t w01, w23;
                  dequant4_e4m3(d[q], scale[n], w01, w23);  // bf16(e4m3 * scale), src/fp8.rs:138-140
                  wf[n][4 * q] = __uint_as_float(w01 << 16); wf[n][4 * q + 1] = __uint_as_float(w01 & 0xffff0000u);
                  wf[n][4 * q + 2] = __uint_as_float(w23 << 16); wf[n][4 * q + 3] = __uint_as_float(w23 & 0xffff0000u);
                }
              } else {
                uint32_t d[S::EL / 2];
                if constexpr (S::EL == 4) { const u32x2 v = *reinterpret_cast<const u32x2*>(at); d[0] = v.x; d[1] = v.y; }
                else { const u32x4 v = *reinterpret_cast<const u32x4*>(at); d[0] = v[0]; d[1] = v[1]; d[2] = v[2]; d[3] = v[3]; }
#pragma unroll
                for (int q = 0; q < S::EL / 2; ++q) { wf[n][2 * q] = __uint_as_float(d[q] << 16); wf[n][2 * q + 1] = __uint_as_float(d[q] & 0xffff0000u); }
              }
            }
#pragma unroll
            for (int t = 0; t < N; ++t) {
              const uint8_t* xa = xc + t * (FFMOE_FORM_SEG * 2) + st * (S::STEP * 2);
              float xf[S::EL];
              uint32_t d[S::EL / 2];
              if constexpr (S::EL == 4) { const u32x2 v = *reinterpret_cast<const u32x2*>(xa); d[0] = v.x; d[1] = v.y; }
              else { const u32x4 v = *reinterpret_cast<const u32x4*>(xa); d[0] = v[0]; d[1] = v[1]; d[2] = v[2]; d[3] = v[3]; }
#pragma unroll
              for (int q = 0; q < S::EL / 2; ++q) { xf[2 * q] = __uint_as_float(d[q] << 16); xf[2 * q + 1] = __uint_as_float(d[q] & 0xffff0000u); }
#pragma unroll
              for (int n = 0; n < NR; ++n) {
                if constexpr (L16) {
#pragma unroll
                  for (int a = 0; a < 4; ++a) acc[n][t][a] = __fmaf_rn(xf[a], wf[n][a], acc[n][t][a]);
                } else {
                  float inner = 0.0f;
#pragma unroll
                  for (int e = 0; e < S::EL; ++e) inner = __fmaf_rn(xf[e], wf[n][e], inner);
                  acc[n][t][0] = __fadd_rn(acc[n][t][0], inner);
                }
              }
            }
          }
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
  }
  if (!f.live) return;
#pragma unroll
  for (int t = 0; t < N; ++t) {
    if (t >= f.gn || t >= T) break;
    const int row = grow[t < T ? t : 0], slot = gslot[t < T ? t : 0];
    float total[NR];  // in every lane of the row: the trees of form_dot, whose additions commute
#pragma unroll
    for (int n = 0; n < NR; ++n) {
      if constexpr (L16) {
        float v = __fadd_rn(__fadd_rn(acc[n][t][0], acc[n][t][1]), __fadd_rn(acc[n][t][2], acc[n][t][3]));
        v = __fadd_rn(v, dpp_or<DPP_QUAD_SWAP1, 0xf>(0.0f, v));
        total[n] = __fadd_rn(v, dpp_or<DPP_QUAD_SWAP2, 0xf>(0.0f, v));
      } else {
        float v = acc[n][t][0];
        v = __fadd_rn(v, lane_xor(v, 4));
        v = __fadd_rn(v, dpp_or<DPP_QUAD_SWAP2, 0xf>(0.0f, v));
        total[n] = __fadd_rn(v, dpp_or<DPP_QUAD_SWAP1, 0xf>(0.0f, v));
      }
    }
    if (sub != (t & (L - 1))) continue;  // the tokens' epilogues go to different lanes
    if (STAGE == 0) {
      const bool reciprocal = L16 && (p.swiglu == FFMOE_SWIGLU_TWICE || p.swiglu == FFMOE_SWIGLU_CLAMPED_TWICE);
#pragma unroll
      for (int n = 0; n < NR; n += 2)
        p.h[size_t(slot) * p.h_stride + f.j0 + (n >> 1) * RPL + r] =
            form_swiglu(bround(total[n]), bround(total[n + 1]), p.swiglu, p.swiglu_limit, reciprocal);
    } else {
      float wk = 1.0f;
      if (!f.is_shared)
        wk = p.weights_f32 ? reinterpret_cast<const float*>(p.weights)[slot] : bf16_to_f32(reinterpret_cast<const uint16_t*>(p.weights)[slot]);
#pragma unroll
      for (int n = 0; n < NR; ++n) {
        const int j = f.j0 + n * RPL + r;
        if (f.is_shared) {
          p.shared_out[size_t(row) * p.hidden + j] = f32_to_bf16(total[n]);
        } else {
          const float v = __fmul_rn(p.routed_weight == FFMOE_WEIGHT_AFTER_DOWN_BF16 ? bround(total[n]) : total[n], wk);
          p.contributions[size_t(slot) * p.hidden + j] = f32_to_bf16(v);
          if (j == 0 && p.done) p.done[slot] = 1u;
        }
      }
    }
  }
}

// grid: (group, tile of output columns) pairs, the shared expert's first
template <class F, int FORM, int STAGE, int T>
__global__ __launch_bounds__(256) void k_decode_form_rows(const DecodeParams p) {
  extern __shared__ __align__(16) uint8_t lds[];
  constexpr int COLS = STAGE == 0 ? 64 : 128;  // output columns per block
  const int wave = uni(int(threadIdx.x) >> 6);
  const int A = p.rows * p.top_k;
  const int tiles_s = ((STAGE == 0 ? p.shared_inter : p.hidden) + COLS - 1) / COLS, tiles_r = ((STAGE == 0 ? p.inter : p.hidden) + COLS - 1) / COLS;
  const int n_routed = p.groups ? load_uniform<int>(p.counters) : A;
  const int n_shared = p.groups ? load_uniform<int>(p.counters + 1) : (p.has_shared ? p.rows : 0);
  int group, tile;
  {
    const uint32_t b = flat_block(), bs = uint32_t(n_shared) * uint32_t(tiles_s);
    if (b < bs) {
      group = int(b / uint32_t(tiles_s));
      tile = int(b) - group * tiles_s;
      group += n_routed;
    } else {
      group = int((b - bs) / uint32_t(tiles_r));
      if (group >= n_routed) return;
      tile = int(b - bs) - group * tiles_r;
    }
  }
  int expert, grow[T], gslot[T];
  FormTile f;
  load_group<T>(p, group, expert, f.gn, grow, gslot);
  if (f.gn == 0) return;  // inactive, invalid or stale choice: nothing written, done stays 0
  f.is_shared = expert < 0;
  f.K = STAGE == 0 ? p.hidden : (f.is_shared ? p.shared_inter : p.inter);
  f.out = STAGE == 0 ? (f.is_shared ? p.shared_inter : p.inter) : p.hidden;
  f.j0 = tile * COLS + wave * (COLS / 4);
  f.live = f.j0 < f.out;  // columns come in multiples of 64: a wave is inside or outside as a whole
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = STAGE == 0 ? i : 4 + (i & 1);
    f.sl[i] = f.is_shared ? p.shared_slot[e] : load_uniform<uint64_t>(p.slots + size_t(expert) * 6 + e);
  }
  if (T == 1 || f.gn == 1) form_rows_run<F, FORM, STAGE, 1, T>(p, f, grow, gslot, lds);
  else if (T == 2 || f.gn == 2) form_rows_run<F, FORM, STAGE, 2, T>(p, f, grow, gslot, lds);
  else if (f.gn == 3) form_rows_run<F, FORM, STAGE, 3, T>(p, f, grow, gslot, lds);
  else if (T == 4 || f.gn == 4) form_rows_run<F, FORM, STAGE, 4, T>(p, f, grow, gslot, lds);
  else if (f.gn <= 6) form_rows_run<F, FORM, STAGE, 6, T>(p, f, grow, gslot, lds);
  else form_rows_run<F, FORM, STAGE, 8, T>(p, f, grow, gslot, lds);
}

// whole lines of every row: the streaming form of the kernels applies
template <class F>
bool form_rows_fit(const DecodeParams& p) {
  constexpr int CH = FormShape<F, FFMOE_FORM_LANE16_>::CH;
  return p.hidden % CH == 0 && p.inter % CH == 0 && (!p.has_shared || p.shared_inter % CH == 0);
}

template <class F, int FORM, int T>
int launch_form_rows(const DecodeParams& p, long long routed, long long shared, int stage_mask, hipStream_t st) {
  const long long b0 = routed * ((p.inter + 63) / 64) + shared * ((p.shared_inter + 63) / 64), b1 = (routed + shared) * ((p.hidden + 127) / 128);
  if (b0 > FLAT_BLOCKS_MAX || b1 > FLAT_BLOCKS_MAX) return ff_fail(FFMOE_ERR_SHAPE, "%lld groups exceed the launch grid", routed + shared);
  constexpr size_t lds = 4 * FFMOE_FORM_WAVE_LDS + size_t(T) * FFMOE_FORM_SEG * 2;
  if (stage_mask & 1) {
    hipLaunchKernelGGL((k_decode_form_rows<F, FORM, 0, T>), flat_grid(b0, 256), dim3(256), lds, st, p);
    FF_TRY(ff_launch_status());
  }
  if (stage_mask & 2) {
    hipLaunchKernelGGL((k_decode_form_rows<F, FORM, 1, T>), flat_grid(b1, 256), dim3(256), lds, st, p);
    FF_TRY(ff_launch_status());
  }
  return 0;
}

template <class F, int FORM, int RG>
int launch_form_grouped(const DecodeParams& p, unsigned max_groups, int stage_mask, hipStream_t st) {
  constexpr int ROWS = 256 / (FORM == FFMOE_FORM_LANE16_ ? 2 : 8);
  const int imax = p.inter > p.shared_inter ? p.inter : p.shared_inter;
  if (stage_mask & 1) {
    hipLaunchKernelGGL((k_decode_form_grouped<F, FORM, 0, RG>), dim3((imax + ROWS - 1) / ROWS, max_groups), dim3(256), size_t(RG) * p.hidden * 2, st, p);
    FF_TRY(ff_launch_status());
  }
  if (stage_mask & 2) {
    hipLaunchKernelGGL((k_decode_form_grouped<F, FORM, 1, RG>), dim3((p.hidden + ROWS - 1) / ROWS, max_groups), dim3(256), size_t(RG) * imax * 2, st, p);
    FF_TRY(ff_launch_status());
  }
  return 0;
}

template <class F, int FORM>
int launch_form(const DecodeParams& p, int stage_mask, hipStream_t st) {
  constexpr int ROWS = 256 / (FORM == FFMOE_FORM_LANE16_ ? 2 : 8);
  const int imax = p.inter > p.shared_inter ? p.inter : p.shared_inter;
  if (stage_mask & 1) {
    hipLaunchKernelGGL((k_decode_form<F, FORM, 0>), dim3((imax + ROWS - 1) / ROWS, p.rows, p.top_k + 1), dim3(256), size_t(p.hidden) * 2, st, p);
    FF_TRY(ff_launch_status());
  }
  if (stage_mask & 2) {
    hipLaunchKernelGGL((k_decode_form<F, FORM, 1>), dim3((p.hidden + ROWS - 1) / ROWS, p.rows, p.top_k + 1), dim3(256), size_t(imax) * 2, st, p);
    FF_TRY(ff_launch_status());
  }
  return 0;
}

}  // namespace ffmoe
