// stream_minmax.hip -- MIN / MAX over a whole square mask (erode, dilate:
// Kernel::reduce(Domain, MIN / MAX) without weights, samples-public/
// 1_Local_Operators/Erode, Dilate) through the row-streaming kernel of
// hh_stream.hpp, pixels in and out of one type.
//
// The generic kernel evaluated mask_w * mask_h taps per pixel with a typed
// load each.  The extreme of a window is the extreme of its row extremes, so
// a streamed row costs ceil(log2 K) picks per pixel for its row extreme and
// one pick per mask row; each pixel is loaded once per wave row.
#include "hh_stream.hpp"

namespace hh {

int dispatch_stream_minmax(const LocalArgs& a, int acc_is_float, int seg, hipStream_t s) {
  const Geom& g = a.g;
  if ((a.reduce != HIPACC_REDUCE_MIN && a.reduce != HIPACC_REDUCE_MAX) || a.use_weights ||
      a.mask_w != a.mask_h || g.in_dtype != g.out_dtype ||
      (acc_is_float != 0) != (g.in_dtype == HIPACC_F32))
    return HIPACC_ERR_UNSUPPORTED;
  for (int t = 0; t < a.mask_w * a.mask_h; ++t)
    if (!a.domain[t]) return HIPACC_ERR_UNSUPPORTED;
  const bool mn = a.reduce == HIPACC_REDUCE_MIN;
#define HH_SMM(T, DT, ACC, K)                                                                    \
  if (g.in_dtype == DT && a.mask_w == K)                                                         \
    return mn ? launch_stream<T, T, ACC, 4, K, K, HH_PF(K), false, kStreamMin, false>(a, seg, s) \
              : launch_stream<T, T, ACC, 4, K, K, HH_PF(K), false, kStreamMax, false>(a, seg, s);
#define HH_SMMK(T, DT, ACC) HH_SMM(T, DT, ACC, 3) HH_SMM(T, DT, ACC, 5) HH_SMM(T, DT, ACC, 7) HH_SMM(T, DT, ACC, 9)
  HH_SMMK(uint8_t, HIPACC_U8, int32_t)
  HH_SMMK(uint16_t, HIPACC_U16, int32_t)
  HH_SMMK(int16_t, HIPACC_I16, int32_t)
  HH_SMMK(float, HIPACC_F32, float)
#undef HH_SMMK
#undef HH_SMM
  return HIPACC_ERR_UNSUPPORTED;
}

}  // namespace hh
