// Shared helpers for the TensorMol-AMD HIP library (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define TM_WAVE 64

// status codes returned by every extern "C" entry point
enum {
  TM_OK = 0,
  TM_ERR_ARG = -1,
  TM_ERR_HIP = -2,
  TM_ERR_CAPACITY = -3,
};

// flag word layout written by kernels (int32 device array, caller-zeroed)
enum {
  TM_FLAG_NB_OVERFLOW = 0,   // a row of the 4.6 A list exceeded its stride
  TM_FLAG_ANG_OVERFLOW = 1,  // a row of the 3.1 A sub-list exceeded its stride
  TM_FLAG_CELL_OVERFLOW = 2, // an atom fell outside the open-boundary cell grid (clamped)
  TM_FLAG_NONFINITE = 3,     // a non-finite coordinate was seen
  TM_NFLAGS = 8,
};

void tm_set_error(const char* fmt, ...);

#define TM_HIP_CHECK(expr)                                                     \
  do {                                                                         \
    hipError_t _e = (expr);                                                    \
    if (_e != hipSuccess) {                                                    \
      tm_set_error("%s:%d %s: %s", __FILE__, __LINE__, #expr,                  \
                   hipGetErrorString(_e));                                     \
      return TM_ERR_HIP;                                                       \
    }                                                                          \
  } while (0)

#define TM_LAUNCH_CHECK()                                                      \
  do {                                                                         \
    hipError_t _e = hipGetLastError();                                         \
    if (_e != hipSuccess) {                                                    \
      tm_set_error("%s:%d launch: %s", __FILE__, __LINE__,                     \
                   hipGetErrorString(_e));                                     \
      return TM_ERR_HIP;                                                       \
    }                                                                          \
  } while (0)

#define TM_REQUIRE(cond, ...)                                                  \
  do {                                                                         \
    if (!(cond)) {                                                             \
      tm_set_error(__VA_ARGS__);                                               \
      return TM_ERR_ARG;                                                       \
    }                                                                          \
  } while (0)

static inline unsigned tm_div_up(long a, long b) { return (unsigned)((a + b - 1) / b); }

// Maximum number of elements a model may carry (descriptor offsets are sized by it).
#define TM_MAX_ELE 8

// Minimum-image displacement along one axis for an orthorhombic box edge L
// (L <= 0 means open boundary).  Evaluated in float64 with the product and
// the difference rounded separately (no fused multiply-add), as the host
// restatement of the neighbour predicate does.
__device__ __forceinline__ double tm_min_image(double d, double L) {
#pragma clang fp contract(off)
  if (L > 0.0) d = d - L * rint(d / L);
  return d;
}

// wave-level sum of a float (butterfly over 64 lanes)
__device__ __forceinline__ float tm_wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
// Sum over the wave, in every lane, in the order of a butterfly over lane ^ 32,
// ^ 16, ^ 8, ^ 4, ^ 2, ^ 1, without a trip through LDS.  The halves and the rows
// of 16 lanes are exchanged by swaps; after that lanes that differ by 16 or 32
// hold the same sum, after the step of 8 also lanes that differ by 8, and so on,
// so a rotation of the row by 8, 4, 2, 1 reads what lane ^ 8, 4, 2, 1 holds.
struct tm_d2 {
  double a, b;
};
template <int ROWS>
__device__ __forceinline__ tm_d2 tm_swap_d(double v) {
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  const u2 x = __builtin_bit_cast(u2, v);
  auto swap = [](unsigned u) {
    if constexpr (ROWS == 32) return __builtin_amdgcn_permlane32_swap(u, u, false, false);
    else return __builtin_amdgcn_permlane16_swap(u, u, false, false);
  };
  const auto lo = swap(x.x), hi = swap(x.y);
  return {__builtin_bit_cast(double, u2{(unsigned)lo[0], (unsigned)hi[0]}),
          __builtin_bit_cast(double, u2{(unsigned)lo[1], (unsigned)hi[1]})};
}
template <int N>
__device__ __forceinline__ double tm_row_ror_d(double v) {
  typedef int i2 __attribute__((ext_vector_type(2)));
  const i2 x = __builtin_bit_cast(i2, v);
  return __builtin_bit_cast(double, i2{__builtin_amdgcn_update_dpp(0, x.x, 0x120 + N, 0xf, 0xf, true),
                                       __builtin_amdgcn_update_dpp(0, x.y, 0x120 + N, 0xf, 0xf, true)});
}
__device__ __forceinline__ double tm_wave_sum_d(double v) {
  const tm_d2 h = tm_swap_d<32>(v);
  v = h.a + h.b;
  const tm_d2 r = tm_swap_d<16>(v);
  v = r.a + r.b;
  v += tm_row_ror_d<8>(v);
  v += tm_row_ror_d<4>(v);
  v += tm_row_ror_d<2>(v);
  v += tm_row_ror_d<1>(v);
  return v;
}
