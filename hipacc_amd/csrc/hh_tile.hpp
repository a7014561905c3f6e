// hh_tile.hpp -- LDS staging of an input tile plus halo, and vector I/O.
//
// A block of 256 threads (4 waves) owns a tile of 64*VEC columns by 4*PPT rows
// of the iteration space; VEC = 16 / sizeof(pixel), so every lane moves one
// 16-byte vector per row.  The tile plus HV vectors of halo on each side and
// RY rows above and below is staged in LDS:
//  - interior tiles (the whole staged region lies where raw reads are valid)
//    are loaded with aligned 16-byte global loads and no index arithmetic;
//  - border tiles resolve the boundary mode per staged element.
// This is the "boundary handling only in border blocks" split of the
// reference (runtime/hipacc_cu_standalone.hpp:66-103, lib/AST/
// ASTTranslate.cpp:787-980), applied once while staging instead of per tap.
#pragma once

#include <type_traits>

#include "hh_local.hpp"

namespace hh {

// Words of row pixels at any pixel's alignment: global accesses of 4 to 16
// bytes need none on this device (a wave's row costs at most one more cache
// line), so rows of odd pitch move as whole vectors too.
typedef unsigned int u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
typedef unsigned int u32x2_any __attribute__((ext_vector_type(2), aligned(1)));
typedef unsigned int u32_any __attribute__((aligned(1)));
typedef unsigned short u16_any __attribute__((aligned(1)));

// Stores VEC values of TO at dst: with nontemporal stores (operator outputs
// are not re-read by the kernel) where dst is aligned to min(16, VEC *
// sizeof(TO)), else with plain ones, so that the L2 joins the cache lines that
// neighbouring tiles write in parts.
template <typename TO, int VEC>
__device__ __forceinline__ void store_vec(TO* dst, const TO (&v)[VEC], bool aligned = true) {
  constexpr int BYTES = VEC * (int)sizeof(TO);
  // (a macro: a template parameter would drop the types' alignment; with an
  // empty asm on either side of it the plain store can neither be hoisted nor
  // sunk to join the nontemporal one, which would make both plain)
#define HH_STORE_WORD(W, p, src)                                    \
  {                                                                 \
    W w;                                                            \
    __builtin_memcpy(&w, src, sizeof(W));                           \
    if (aligned) {                                                  \
      __builtin_nontemporal_store(w, (W*)(p));                      \
    } else {                                                        \
      asm volatile("" ::: "memory");                                \
      *(W*)(p) = w;                                                 \
      asm volatile("" ::: "memory");                                \
    }                                                               \
  }
  if constexpr (BYTES >= 16) {
#pragma unroll
    for (int k = 0; k < BYTES / 16; ++k)
      HH_STORE_WORD(u32x4_any, reinterpret_cast<char*>(dst) + 16 * k,
                    reinterpret_cast<const char*>(v) + 16 * k)
  } else if constexpr (BYTES == 8) {
    HH_STORE_WORD(u32x2_any, dst, v)
  } else if constexpr (BYTES == 4) {
    HH_STORE_WORD(u32_any, dst, v)
  } else if constexpr (BYTES == 2) {
    HH_STORE_WORD(u16_any, dst, v)
  } else {
    static_assert(BYTES == 1, "pixel vector");
    HH_STORE_WORD(unsigned char, dst, v)
  }
#undef HH_STORE_WORD
}

template <typename TI> __device__ __forceinline__ TI const_pixel(const Geom& g);
template <> __device__ __forceinline__ float const_pixel<float>(const Geom& g) { return g.const_f; }
template <> __device__ __forceinline__ uint8_t const_pixel<uint8_t>(const Geom& g) { return (uint8_t)g.const_i; }
template <> __device__ __forceinline__ int8_t const_pixel<int8_t>(const Geom& g) { return (int8_t)g.const_i; }
template <> __device__ __forceinline__ uint16_t const_pixel<uint16_t>(const Geom& g) { return (uint16_t)g.const_i; }
template <> __device__ __forceinline__ int16_t const_pixel<int16_t>(const Geom& g) { return (int16_t)g.const_i; }
template <> __device__ __forceinline__ uint32_t const_pixel<uint32_t>(const Geom& g) { return (uint32_t)g.const_i; }
template <> __device__ __forceinline__ int32_t const_pixel<int32_t>(const Geom& g) { return (int32_t)g.const_i; }

// Region where raw (unmapped) reads return what the boundary mode would: the
// accessor window, or the whole allocation for UNDEFINED.
__device__ __forceinline__ void raw_region(const Geom& g, int& lx, int& hx, int& ly, int& hy) {
  if (g.boundary == HIPACC_BOUNDARY_UNDEFINED) {
    lx = 0; hx = g.in_imgw; ly = 0; hy = g.in_imgh;
  } else {
    lx = g.lo_x; hx = g.hi_x; ly = g.lo_y; hy = g.hi_y;
  }
}

// Whether rows [iy0, iy0+lh) x columns [ix0, ix0+lw) all read raw pixels.
__device__ __forceinline__ bool raw_tile(const Geom& g, int ix0, int iy0, int lw, int lh) {
  int lx, hx, ly, hy;
  raw_region(g, lx, hx, ly, hy);
  return ix0 >= lx && ix0 + lw <= hx && iy0 >= ly && iy0 + lh <= hy;
}

// Stages rows [iy0, iy0+LH) x columns [ix0, ix0+NV*VEC) of the input into
// tile (row pitch NV*VEC elements).
template <typename TI, int VEC, int NV, int LH>
__device__ __forceinline__ void stage_tile(TI* __restrict__ tile, const TI* __restrict__ in,
                                           const Geom& g, int ix0, int iy0) {
  constexpr int LW = NV * VEC;
  const int tid = threadIdx.x;
  if (raw_tile(g, ix0, iy0, LW, LH)) {
    // Every load of the thread is issued before the first LDS write, so all
    // of them are in flight together.  Threads past the last vector load it
    // again: with the loads under a condition the staging array was placed in
    // LDS and the loads waited for one by one, and the kernel read the
    // workgroup size from the dispatch packet in host memory (7 us at the
    // start of every launch).
    constexpr int N = LH * NV, NL = (N + 255) / 256;
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    const TI* src = in + (long long)iy0 * g.in_stride + ix0;
    u32x4 w[NL];
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      const int i = min(tid + k * 256, N - 1);
      const int r = i / NV;
      const int c = i - r * NV;
      w[k] = *reinterpret_cast<const u32x4_any*>(src + (long long)r * g.in_stride + c * VEC);
    }
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      const int i = tid + k * 256;
      if (i < N) *reinterpret_cast<u32x4*>(tile + i * VEC) = w[k];
    }
  } else {
    const bool cmode = g.boundary == HIPACC_BOUNDARY_CONSTANT;
    const TI cval = const_pixel<TI>(g);
    for (int i = tid; i < LH * LW; i += 256) {
      const int r = i / LW;
      const int c = i - r * LW;
      int x = ix0 + c;
      int y = iy0 + r;
      TI v;
      if (cmode) {
        if (x < g.lo_x || x >= g.hi_x || y < g.lo_y || y >= g.hi_y)
          v = cval;
        else
          v = in[(long long)y * g.in_stride + x];
      } else {
        x = bh_map(g.boundary, x, g.lo_x, g.hi_x, g.in_imgw);
        y = bh_map(g.boundary, y, g.lo_y, g.hi_y, g.in_imgh);
        v = in[(long long)y * g.in_stride + x];
      }
      tile[r * LW + c] = v;
    }
  }
}

// Loads NW consecutive 16-byte vectors of LDS and widens them to ACC.
template <typename TI, typename ACC, int VEC, int NW>
__device__ __forceinline__ void load_window(ACC (&win)[NW * VEC], const TI* __restrict__ p) {
#pragma unroll
  for (int k = 0; k < NW; ++k) {
    TI t[VEC];
    const uint4 w = *reinterpret_cast<const uint4*>(p + k * VEC);
    __builtin_memcpy(t, &w, 16);
#pragma unroll
    for (int v = 0; v < VEC; ++v) win[k * VEC + v] = (ACC)t[v];
  }
}

// Writes one output row segment of VEC pixels (iteration-space-relative
// column ox, row oy) of a tile.
template <typename TO, typename ACC, int VEC>
__device__ __forceinline__ void store_row(TO* __restrict__ out, const Geom& g, int out_vec_ok,
                                          int ox, int oy, const ACC (&acc)[VEC]) {
  if (oy >= g.is_h || ox >= g.is_w) return;
  TO* dst = out + (long long)(g.out_oy + oy) * g.out_stride + g.out_ox + ox;
  TO vals[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    if constexpr (std::is_same<ACC, float>::value)
      vals[v] = convert_f<TO>((float)acc[v], g.cvt, g.post_div);
    else
      vals[v] = convert_i<TO>((int32_t)acc[v], g.cvt, g.post_div);
  }
  if (ox + VEC <= g.is_w) {
    store_vec<TO, VEC>(dst, vals, out_vec_ok);
  } else {
#pragma unroll
    for (int v = 0; v < VEC; ++v)
      if (ox + v < g.is_w) dst[v] = vals[v];
  }
}

}  // namespace hh
