// Instantiates the software-pipelined MFMA convolution (conv_pipe.h) for one storage type.  Built with
// -mllvm -amdgpu-mfma-vgpr-form: the kernel keeps its accumulators in ordinary VGPRs (it fits 256 of them), and
// without the switch the compiler moves them through AGPRs with four copies per MFMA.
#include "conv_solo.h"

namespace d3d {

int32_t launchPipeBf16(const ConvArgs& a, hipStream_t stream) {
  const int32_t rc = convk::launchSolo<__bf16>(a, stream);
  return rc != D3D_ERR_UNSUPPORTED ? rc : convk::launchPipe<__bf16>(a, stream);
}

}  // namespace d3d
