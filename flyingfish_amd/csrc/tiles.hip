// Launches of the kernels whose operand tiles go straight to LDS (tile_gemm.cuh, wide_gemm.cuh, mx_tile.cuh, nvfp4_tile.cuh)
#include "tile_gemm.cuh"
#include "wide_gemm.cuh"
#include "mx_tile.cuh"
#include "nvfp4_tile.cuh"
#include "tiles.h"
#include "api.h"

namespace ffmoe {

int launch_w8a8_tile(int mode, const GemmParams& p, unsigned blocks, hipStream_t stream) {
  if (mode == 0) hipLaunchKernelGGL((k_dense_tile<0, TILE_W8A8>), dim3(blocks), dim3(256), 0, stream, p);
  else hipLaunchKernelGGL((k_dense_tile<2, TILE_W8A8>), dim3(blocks), dim3(256), 0, stream, p);
  return ff_launch_status();
}
int launch_mx_dense_tile(int mode, const GemmParams& p, unsigned blocks, hipStream_t stream) {
  if (mode == 0) hipLaunchKernelGGL((k_dense_tile<0, TILE_MX>), dim3(blocks), dim3(256), 0, stream, p);
  else hipLaunchKernelGGL((k_dense_tile<2, TILE_MX>), dim3(blocks), dim3(256), 0, stream, p);
  return ff_launch_status();
}

int launch_bf16_tile(int mode, bool split, const GemmParams& p, unsigned blocks, hipStream_t stream) {
  const auto kernel = split ? (mode == 0 ? k_dense_tile<0, TILE_BF16_SPLIT> : k_dense_tile<2, TILE_BF16_SPLIT>)
                            : (mode == 0 ? k_dense_tile<0, TILE_BF16> : k_dense_tile<2, TILE_BF16>);
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, stream, p);
  return ff_launch_status();
}

template <int MODE>
static int launch_wide(const GemmParams& p, unsigned blocks, hipStream_t stream) {
  static const hipError_t ok = hipFuncSetAttribute(reinterpret_cast<const void*>(k_w8a8_wide<MODE>), hipFuncAttributeMaxDynamicSharedMemorySize, WIDE_LDS);
  if (ok != hipSuccess) return ff_fail(FFMOE_ERR_UNSUPPORTED, "%d bytes of LDS per block: %s", WIDE_LDS, hipGetErrorString(ok));
  hipLaunchKernelGGL(k_w8a8_wide<MODE>, dim3(blocks), dim3(512), WIDE_LDS, stream, p);
  return ff_launch_status();
}
int launch_w8a8_wide(int mode, const GemmParams& p, unsigned blocks, hipStream_t stream) {
  return mode == 0 ? launch_wide<0>(p, blocks, stream) : launch_wide<2>(p, blocks, stream);
}

template <int MODE>
static int launch_cohort(const GemmParams& p, const uint32_t* big_groups, uint32_t* queue, unsigned blocks, hipStream_t stream) {
  static const hipError_t ok = hipFuncSetAttribute(reinterpret_cast<const void*>(k_w8a8_cohort<MODE>), hipFuncAttributeMaxDynamicSharedMemorySize, COHORT_LDS);
  if (ok != hipSuccess) return ff_fail(FFMOE_ERR_UNSUPPORTED, "%d bytes of LDS per block: %s", COHORT_LDS, hipGetErrorString(ok));
  hipLaunchKernelGGL(k_w8a8_cohort<MODE>, dim3(blocks), dim3(512), COHORT_LDS, stream, p, big_groups, queue);
  return ff_launch_status();
}
int launch_w8a8_cohort(int mode, const GemmParams& p, const uint32_t* big_groups, uint32_t* queue, unsigned blocks, hipStream_t stream) {
  return mode == 0 ? launch_cohort<0>(p, big_groups, queue, blocks, stream) : launch_cohort<1>(p, big_groups, queue, blocks, stream);
}

template <int MODE>
static int launch_mx(const MxParams& p, unsigned blocks, hipStream_t stream) {
  static const hipError_t ok = hipFuncSetAttribute(reinterpret_cast<const void*>(k_mx_tile<MODE>), hipFuncAttributeMaxDynamicSharedMemorySize, MX_TILE_LDS);
  if (ok != hipSuccess) return ff_fail(FFMOE_ERR_UNSUPPORTED, "%d bytes of LDS per block: %s", MX_TILE_LDS, hipGetErrorString(ok));
  hipLaunchKernelGGL(k_mx_tile<MODE>, dim3(blocks), dim3(256), MX_TILE_LDS, stream, p);
  return ff_launch_status();
}
int launch_mx_tile(int mode, const MxParams& p, unsigned blocks, hipStream_t stream) {
  return mode == 0 ? launch_mx<0>(p, blocks, stream) : launch_mx<1>(p, blocks, stream);
}

template <int MODE>
static int launch_nvfp4(const W16Params& p, unsigned blocks, hipStream_t stream) {
  static const hipError_t ok = hipFuncSetAttribute(reinterpret_cast<const void*>(k_nvfp4_tile<MODE>), hipFuncAttributeMaxDynamicSharedMemorySize, NV_TILE_LDS);
  if (ok != hipSuccess) return ff_fail(FFMOE_ERR_UNSUPPORTED, "%d bytes of LDS per block: %s", NV_TILE_LDS, hipGetErrorString(ok));
  hipLaunchKernelGGL(k_nvfp4_tile<MODE>, dim3(blocks), dim3(256), NV_TILE_LDS, stream, p);
  return ff_launch_status();
}
int launch_nvfp4_tile(int mode, const W16Params& p, unsigned blocks, hipStream_t stream) {
  return mode == 0 ? launch_nvfp4<0>(p, blocks, stream) : launch_nvfp4<1>(p, blocks, stream);
}

}  // namespace ffmoe
