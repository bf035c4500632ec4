// Launches of the 128 x 128 tile kernels (tile_gemm.cuh)
#include "tile_gemm.cuh"
#include "tiles.h"
#include "api.h"

namespace ffmoe {

int launch_w8a8_tile(int mode, const GemmParams& p, unsigned blocks, hipStream_t stream) {
  if (mode == 0) hipLaunchKernelGGL(k_w8a8_tile<0>, dim3(blocks), dim3(256), 0, stream, p);
  else hipLaunchKernelGGL(k_w8a8_tile<2>, dim3(blocks), dim3(256), 0, stream, p);
  return ff_launch_status();
}

}  // namespace ffmoe
