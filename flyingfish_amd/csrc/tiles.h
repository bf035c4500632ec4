// Launch functions of tiles.hip
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ffmoe {
struct GemmParams;
struct MxParams;
struct W16Params;
// W8A8 on 128 x 128 tiles (MODE of w8a8_gemm.cuh; a gate/up tile is 64 activation columns): units of a dense call
inline uint32_t tile_units(int mode, int rows, int n) { return uint32_t((rows + 127) / 128) * uint32_t(mode == 0 ? (n + 63) / 64 : (n + 127) / 128); }
int launch_w8a8_tile(int mode, const GemmParams& p, unsigned blocks, hipStream_t stream);
// the same on 256 x 256 tiles (128 activation columns): units of a dense call
inline uint32_t wide_units(int mode, int rows, int n) { return uint32_t((rows + 255) / 256) * uint32_t(mode == 0 ? (n + 127) / 128 : (n + 255) / 256); }
int launch_w8a8_wide(int mode, const GemmParams& p, unsigned blocks, hipStream_t stream);
// routed row groups of at most 256 rows (mode 0 gate/up, 1 down), units of 128 activation or 256 output columns, those of
// the *big_groups groups of more than 128 rows first; queue: sixteen words, zero
int launch_w8a8_cohort(int mode, const GemmParams& p, const uint32_t* big_groups, uint32_t* queue, unsigned blocks, hipStream_t stream);
// 128 x 128 tiles for BF16 weights and activations (a_codes holds BF16 rows, K counts elements; no scales): in one chain, or split, with K a
// multiple of 256, in the eight partial sums of dense_splitk.cuh
int launch_bf16_tile(int mode, bool split, const GemmParams& p, unsigned blocks, hipStream_t stream);
// and for E4M3 / E8M0 block-32 weights and activations (a_scales and w*_scales hold scale bytes)
int launch_mx_dense_tile(int mode, const GemmParams& p, unsigned blocks, hipStream_t stream);
// E2M1 / E8M0 row groups of at most 64 tokens (mode 0 gate/up, 1 down), units of 128 activation or 256 output columns
int launch_mx_tile(int mode, const MxParams& p, unsigned blocks, hipStream_t stream);
// NVFP4 W4A16 row groups of at most 64 tokens, K a multiple of 256 (mode 0 gate/up, 1 down), the same units
int launch_nvfp4_tile(int mode, const W16Params& p, unsigned blocks, hipStream_t stream);
}  // namespace ffmoe
