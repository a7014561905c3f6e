// point.hip -- point operators (Kernel::execute with a per-pixel output()).
//
// Each thread produces N adjacent pixels of one row, N such that the wider of
// the input and output vectors is 16 bytes (uint8 to uint8: 16 pixels), and
// the operator is decoded once per thread, not per pixel.  Images whose rows
// are back to back are one long row.  HBM bound: 4096^2 float AFFINE 20 us
// (6.6 TB/s).  The Sobel combine at 4032x3024 (int16 x 2 -> uint8) took 28 us
// with an integer division per input and pixel and 4 pixels per thread; here
// 13 us.
#include "hh_tile.hpp"
#include "hh_point.hpp"

namespace hh {

template <typename T, int N> __device__ __forceinline__ void load_word(const T* p, T* v) {
  constexpr int B = N * (int)sizeof(T);
#define HH_LOAD_WORD(W)                                \
  {                                                    \
    const W w = *reinterpret_cast<const W*>(p);        \
    __builtin_memcpy(v, &w, B);                        \
  }
  if constexpr (B == 16) HH_LOAD_WORD(u32x4_any)
  else if constexpr (B == 8) HH_LOAD_WORD(u32x2_any)
  else HH_LOAD_WORD(u32_any)
#undef HH_LOAD_WORD
}

// N pixels at any alignment as one load of up to 16 bytes; where only n < N of
// them exist, by fours as far as they go (a wave that holds a row's end waits
// for these too: u8 magnitude at 712x2050, pitched, 5.4 us pixel by pixel).
template <typename T, int N> __device__ __forceinline__ void load_n(const T* p, T (&v)[N], int n) {
  if (n == N) {
    load_word<T, N>(p, v);
    return;
  }
#pragma unroll
  for (int g = 0; g < N; g += 4) {
    if (g + 4 <= n) {
      load_word<T, 4>(p + g, v + g);
    } else {
#pragma unroll
      for (int k = g; k < g + 4; ++k) v[k] = k < n ? p[k] : T(0);
    }
  }
}

template <typename T, typename TO> constexpr int point_pixels() {
  return 16 / (int)(sizeof(T) > sizeof(TO) ? sizeof(T) : sizeof(TO));
}

// MAGNITUDE of 8- and 16-bit integers into an integer type.  The quotients
// enter squared, so their signs do not matter, and |a| / |norm| truncated is
// (|a| + 1/2) / |norm| truncated: that is at least 1 / (2 |norm|) away from
// any integer, more than the float product with the reciprocal is off for
// |a| < 2^22.  The sum of squares x is a (wrapping) 32-bit integer as before.
// truncate(sqrt(x)) is truncate(sqrt(x + 1/2)), again away from the integers
// by more than the one unit in the last place the instruction may be off (up
// to 255, where the result saturates), and round(sqrt(x)) has no ties.
template <typename TO>
__device__ __forceinline__ TO magnitude_small(int32_t a, int32_t b, float rinv, bool div, int cvt) {
  int32_t qa = a, qb = b;
  if (div) {
    const float half = 0.5f * rinv;
    qa = (int32_t)__builtin_fmaf(__builtin_fabsf((float)a), rinv, half);
    qb = (int32_t)__builtin_fmaf(__builtin_fabsf((float)b), rinv, half);
  }
  const int32_t x = (int32_t)((uint32_t)__mul24(qa, qa) + (uint32_t)__mul24(qb, qb));
  const float xf = (float)x;
  float f = __builtin_amdgcn_sqrtf(cvt == HIPACC_CVT_ROUND ? xf : xf + 0.5f);
  f = f < 255.0f ? f : 255.0f;
  f = f > 0.0f ? f : 0.0f;
  return convert_f<TO>(f, cvt, 0.0f);
}

template <typename T, typename TO, bool FLOAT_MATH, int OP, int N>
__device__ __forceinline__ void point_row(const PointArgs& a, const T (&v0)[N], const T (&v1)[N],
                                          TO (&r)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k)
    r[k] = point_pixel<TO, FLOAT_MATH>(OP, (float)v0[k], (float)v1[k], (int32_t)v0[k],
                                       (int32_t)v1[k], a.alpha, a.beta, a.cvt);
}

// Both inputs of one pixel type.  Integer inputs: int arithmetic except
// AFFINE (float) and MAGNITUDE (int division by the norm, int sum of squares,
// float sqrt and clamp).
template <typename T, typename TO>
__global__ __launch_bounds__(256) void point_kernel(const PointArgs a) {
  constexpr int N = point_pixels<T, TO>();
  constexpr bool FM = std::is_same<T, float>::value;
  // 2^lanes threads of the block side by side, 256 >> lanes rows
  const int x = ((int)(blockIdx.x << a.lanes) + (int)(threadIdx.x & ((1 << a.lanes) - 1))) * N;
  const int y = (int)(blockIdx.y << (8 - a.lanes)) + (int)(threadIdx.x >> a.lanes);
  if (x >= a.w || y >= a.h) return;
  const int n = a.w - x < N ? a.w - x : N;
  const long long b = blockIdx.z;
  T v0[N], v1[N];
  load_n<T, N>(static_cast<const T*>(a.in0) + b * a.plane0 + (long long)(a.oy0 + y) * a.stride0 +
                   a.ox0 + x, v0, n);
  if (a.in1) {
    load_n<T, N>(static_cast<const T*>(a.in1) + b * a.plane1 + (long long)(a.oy1 + y) * a.stride1 +
                     a.ox1 + x, v1, n);
  } else {
#pragma unroll
    for (int k = 0; k < N; ++k) v1[k] = T(0);
  }
  TO r[N];
  switch (a.op) {
    case HIPACC_POINT_AFFINE: point_row<T, TO, FM, HIPACC_POINT_AFFINE, N>(a, v0, v1, r); break;
    case HIPACC_POINT_ADD: point_row<T, TO, FM, HIPACC_POINT_ADD, N>(a, v0, v1, r); break;
    case HIPACC_POINT_SUB: point_row<T, TO, FM, HIPACC_POINT_SUB, N>(a, v0, v1, r); break;
    case HIPACC_POINT_MUL: point_row<T, TO, FM, HIPACC_POINT_MUL, N>(a, v0, v1, r); break;
    case HIPACC_POINT_ABSDIFF: point_row<T, TO, FM, HIPACC_POINT_ABSDIFF, N>(a, v0, v1, r); break;
    case HIPACC_POINT_MIN: point_row<T, TO, FM, HIPACC_POINT_MIN, N>(a, v0, v1, r); break;
    case HIPACC_POINT_MAX: point_row<T, TO, FM, HIPACC_POINT_MAX, N>(a, v0, v1, r); break;
    case HIPACC_POINT_MAGNITUDE:
      if constexpr (sizeof(T) <= 2 && !std::is_same<TO, float>::value) {
        const int32_t nrm = (int32_t)a.alpha;
        const float rinv = 1.0f / __builtin_fabsf((float)nrm);   // unused for norm 0
#pragma unroll
        for (int k = 0; k < N; ++k)
          r[k] = magnitude_small<TO>((int32_t)v0[k], (int32_t)v1[k], rinv, nrm != 0, a.cvt);
      } else {
        point_row<T, TO, FM, HIPACC_POINT_MAGNITUDE, N>(a, v0, v1, r);
      }
      break;
    default: point_row<T, TO, FM, HIPACC_POINT_COPY, N>(a, v0, v1, r); break;
  }
  TO* po = static_cast<TO*>(a.out) + b * a.plane_out + (long long)(a.oyo + y) * a.stride_out +
           a.oxo + x;
  if (n == N) {
    store_vec<TO, N>(po, r, a.vec_ok);
  } else {
#pragma unroll
    for (int g = 0; g < N; g += 4) {
      const TO q[4] = {r[g], r[g + 1], r[g + 2], r[g + 3]};
      if (g + 4 <= n) {
        store_vec<TO, 4>(po + g, q, false);
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (g + k < n) po[g + k] = q[k];
      }
    }
  }
}

template <typename T0, typename T1, typename TO>
static int launch_point_t(const PointArgs& a0, hipStream_t s) {
  static_assert(std::is_same<T0, T1>::value, "inputs of one pixel type");
  constexpr int N = point_pixels<T0, TO>();
  PointArgs a = a0;
  // rows back to back in every image: one row
  const long long n = (long long)a.w * a.h;
  if (a.h > 1 && a.stride0 == a.w && a.stride_out == a.w && (!a.in1 || a.stride1 == a.w) &&
      n < (1ll << 30)) {
    a.w = (int)n;
    a.h = 1;
  }
  const uintptr_t po = reinterpret_cast<uintptr_t>(static_cast<TO*>(a.out) +
                                                   (long long)a.oyo * a.stride_out + a.oxo);
  const long long align = N * (long long)sizeof(TO);
  a.vec_ok = po % align == 0 && (a.h == 1 || (a.stride_out * (long long)sizeof(TO)) % align == 0) &&
             (a.batch == 1 || (a.plane_out * (long long)sizeof(TO)) % align == 0);
  // blocks of several rows where a row has less than 256 vectors (int8
  // magnitude, 2 x 128x1840: 7.2 us with 8 of a block's threads in use)
  while (a.lanes < 8 && (N << a.lanes) < a.w) ++a.lanes;
  dim3 grid(ceil_div(a.w, N << a.lanes), ceil_div(a.h, 256 >> a.lanes), a.batch);
  hipLaunchKernelGGL((point_kernel<T0, TO>), grid, dim3(256), 0, s, a);
  return hip_status(hipGetLastError(), "point_kernel launch");
}

template <typename T0, typename T1>
static int launch_point_out(const PointArgs& a, int dto, hipStream_t s) {
  switch (dto) {
    case HIPACC_U8: return launch_point_t<T0, T1, uint8_t>(a, s);
    case HIPACC_I8: return launch_point_t<T0, T1, int8_t>(a, s);
    case HIPACC_U16: return launch_point_t<T0, T1, uint16_t>(a, s);
    case HIPACC_I16: return launch_point_t<T0, T1, int16_t>(a, s);
    case HIPACC_U32: return launch_point_t<T0, T1, uint32_t>(a, s);
    case HIPACC_I32: return launch_point_t<T0, T1, int32_t>(a, s);
    case HIPACC_F32: return launch_point_t<T0, T1, float>(a, s);
  }
  return HIPACC_ERR_INVALID_ARG;
}

// Both inputs share one pixel type (the second input, when present, must
// have the first one's type).
int launch_point(const PointArgs& a, int dt0, int dt1, int dto, hipStream_t s) {
  if (a.in1 && dt1 != dt0) return set_error(HIPACC_ERR_UNSUPPORTED, "point: inputs of different pixel types");
  switch (dt0) {
    case HIPACC_U8: return launch_point_out<uint8_t, uint8_t>(a, dto, s);
    case HIPACC_I8: return launch_point_out<int8_t, int8_t>(a, dto, s);
    case HIPACC_U16: return launch_point_out<uint16_t, uint16_t>(a, dto, s);
    case HIPACC_I16: return launch_point_out<int16_t, int16_t>(a, dto, s);
    case HIPACC_U32: return launch_point_out<uint32_t, uint32_t>(a, dto, s);
    case HIPACC_I32: return launch_point_out<int32_t, int32_t>(a, dto, s);
    case HIPACC_F32: return launch_point_out<float, float>(a, dto, s);
  }
  return HIPACC_ERR_INVALID_ARG;
}

}  // namespace hh
