// Instantiates the MFMA convolution kernels (conv_kernels.h) for one storage type.
#include "conv_taps.h"

namespace d3d {

int32_t launchMfmaInt8(const ConvArgs& a, hipStream_t stream) { return convk::launchInt8<>(a, stream); }

bool convReadsNarrowRows(int32_t dtype, int kVol, int cin, int cout, int64_t inRows) {
  if (cout != 16 && cout != 32) return false;
  // int8: rows of 16 channels, and of up to 8 where convTaps reads them (a 5 -> 16 layer on 120 000 rows: 8 us against 4.5 for
  // the widening pass and 9.6 on the widened rows); others are widened (read byte by byte: 19 us against 17), and so are those
  // whose rows' offsets convTaps cannot hold
  if (dtype == D3D_INT8)
    return (cin == 16 || (cin <= 8 && convk::tapsFit(kVol, 16, cout) && convk::tapsReach(inRows, cin))) && convk::residentFits(kVol, 32, cout, 1);
  // two-byte types: rows below 16 channels as stored (that layer: 8 us in convTaps, up to 8 channels; 16.3 element by
  // element against 17.6 with the widening pass)
  if (dtype == D3D_HALF || dtype == D3D_BF16) return cin < 16 && convk::residentFits(kVol, 16, cout, 2);
  if (dtype == D3D_FLOAT) return cin < 16 && convk::residentFits(kVol, 16, cout, 4);
  return false;
}

}  // namespace d3d
