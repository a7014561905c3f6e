// stream_vec4.hip -- local operators on 4-wide pixels (the RGBA samples)
// through the row-streaming kernel of hh_stream.hpp: the image is its
// interleaved channels, a lane holds the four channels of one pixel, and the
// horizontal taps are CH = 4 elements apart, i.e. whole lanes.
//
// Square 3x3 .. 7x7 masks: weighted sums of uchar4 (float or integer) and
// float4, and MIN / MAX over whole masks.  The other shapes stay with
// local_vec4_kernel, which evaluates every tap from an LDS tile of 16-byte
// pixels with run-time types and mask. 1920x1080 uchar4 5x5: 107 us there,
// 18.9 us here, where a tap is one FMA per channel (100 FMA per pixel, 5.3 us
// of VALU issue, and a third more rows for the segments' halo).
#include "hh_stream.hpp"

namespace hh {

int dispatch_stream_vec4(const LocalArgs& a0, int acc_is_float, hipStream_t s) {
  const Geom& g0 = a0.g;
  if (a0.wdev || a0.mask_w != a0.mask_h) return HIPACC_ERR_UNSUPPORTED;
  const int ti = dtype_base(g0.in_dtype), to = dtype_base(g0.out_dtype);
  // row elements are counted in 32 bits
  const long long most = 1ll << 28;
  if (g0.in_stride >= most || g0.out_stride >= most || g0.in_imgw >= most)
    return HIPACC_ERR_UNSUPPORTED;
  const bool f32 = ti == HIPACC_F32;
  // the constant as a pixel: vector views keep it as given
  if (g0.boundary == HIPACC_BOUNDARY_CONSTANT && !f32 &&
      (float)(uint8_t)g0.const_i != g0.const_f)
    return HIPACC_ERR_UNSUPPORTED;
  LocalArgs a = a0;
  const int n = a.mask_w * a.mask_h;
  const bool sum = a.reduce == HIPACC_REDUCE_SUM;
  for (int t = 0; t < n; ++t) {
    // a hole is a zero weight for byte pixels; for floats (0 * inf) and
    // extremes it is not
    if (!a.domain[t] && (f32 || !sum)) return HIPACC_ERR_UNSUPPORTED;
    if (acc_is_float) a.w.f[t] = a.domain[t] ? (a.use_weights ? a.w.f[t] : 1.0f) : 0.0f;
    else a.w.i[t] = a.domain[t] ? (a.use_weights ? a.w.i[t] : 1) : 0;
  }
  a.g.in_dtype = ti;
  a.g.out_dtype = to;
  a.g.in_plane *= 4;
  a.g.out_plane *= 4;
  a.g.in_stride *= 4;
  a.g.out_stride *= 4;
  a.g.in_imgw *= 4;
  a.g.lo_x *= 4;
  a.g.hi_x *= 4;
  a.g.in_ox *= 4;
  a.g.out_ox *= 4;
  a.g.is_w *= 4;
#define HH_SV4F(T, DT, K)                                                                       \
  if (acc_is_float && ti == DT && to == DT && a.mask_w == K)                                    \
    return a.fma ? launch_stream<T, T, float, 4, K, K, HH_PF(K), true, kStream2D, false, 4>(a, 0, s) \
                 : launch_stream<T, T, float, 4, K, K, HH_PF(K), false, kStream2D, false, 4>(a, 0, s);
#define HH_SV4I(TO, DT, K)                                                                      \
  if (!acc_is_float && ti == HIPACC_U8 && to == DT && a.mask_w == K)                            \
    return launch_stream<uint8_t, TO, int32_t, 4, K, K, HH_PF(K), false, kStream2D, false, 4>(a, 0, s);
#define HH_SV4M(T, DT, ACC, K)                                                                  \
  if (acc_is_float == (DT == HIPACC_F32) && ti == DT && to == DT && a.mask_w == K)              \
    return a.reduce == HIPACC_REDUCE_MIN                                                        \
               ? launch_stream<T, T, ACC, 4, K, K, HH_PF(K), false, kStreamMin, false, 4>(a, 0, s) \
               : launch_stream<T, T, ACC, 4, K, K, HH_PF(K), false, kStreamMax, false, 4>(a, 0, s);
  if (sum) {
    HH_SV4F(uint8_t, HIPACC_U8, 3) HH_SV4F(uint8_t, HIPACC_U8, 5) HH_SV4F(uint8_t, HIPACC_U8, 7)
    HH_SV4F(float, HIPACC_F32, 3) HH_SV4F(float, HIPACC_F32, 5) HH_SV4F(float, HIPACC_F32, 7)
    HH_SV4I(uint8_t, HIPACC_U8, 3) HH_SV4I(uint8_t, HIPACC_U8, 5) HH_SV4I(uint8_t, HIPACC_U8, 7)
    HH_SV4I(int32_t, HIPACC_I32, 3) HH_SV4I(int32_t, HIPACC_I32, 5)
  } else if ((a.reduce == HIPACC_REDUCE_MIN || a.reduce == HIPACC_REDUCE_MAX) && !a.use_weights &&
             a.g.post_div == 0.0f) {
    HH_SV4M(uint8_t, HIPACC_U8, int32_t, 3) HH_SV4M(uint8_t, HIPACC_U8, int32_t, 5)
    HH_SV4M(uint8_t, HIPACC_U8, int32_t, 7)
    HH_SV4M(float, HIPACC_F32, float, 3) HH_SV4M(float, HIPACC_F32, float, 5)
    HH_SV4M(float, HIPACC_F32, float, 7)
  }
#undef HH_SV4F
#undef HH_SV4I
#undef HH_SV4M
  return HIPACC_ERR_UNSUPPORTED;
}

}  // namespace hh
