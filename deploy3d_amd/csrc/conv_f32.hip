// Instantiates the MFMA convolutions for fp32 storage: the resident-weight kernel for layers of at most 16 -> 32 or
// 32 -> 16 channels, the software-pipelined kernel for the rest.  Built with -mllvm -amdgpu-mfma-vgpr-form like the
// other instantiations of the pipelined kernel.  Bound by the fp32 MFMA rate (the fp32 vector rate without packed
// math is half of it, and the vector kernels also pass every operand through LDS): the layers of an encoder-decoder
// on 40 000 voxels went from 60 / 315 / 630 us (16 -> 16, 32 -> 32, 64 -> 64) to 10 / 72 / 285.
#include "conv_pipe.h"

namespace d3d {

// 16 -> 16, 16 -> 32 and 32 -> 16 run with resident weights or not at all; the pipelined kernel takes the rest up to 64 taps
// (conv_pipe.h).  Beyond that the vector kernels run on the rows as stored: the layer is neither widened nor packed for an
// MFMA.
bool floatMfmaFits(int kVol, int cin, int cout) {
  return cin * cout <= 512 ? convk::residentFits(kVol, cin, cout, sizeof(float)) : kVol <= 64;
}

int32_t launchMfmaFloat(const ConvArgs& a, hipStream_t stream) {
  const int32_t rc = convk::launchFloatResident<>(a, stream);
  if (rc != D3D_ERR_UNSUPPORTED || a.rowChannels > 0) return rc;
  return convk::launchPipe<float>(a, stream);
}

}  // namespace d3d
