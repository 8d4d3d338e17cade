// A wave's strip of a one-layer grid, shared by the explicit step (adr.hip) and
// the implicit sweeps (implicit.hip): one column per lane, H columns either
// side held for their levels only, the wave walking x on its own. Neighbours
// in x come from registers, neighbours in y from the next lanes.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "adr_site.hpp"
#include "common.hpp"
#include "internal.hpp"

namespace msim {

constexpr int kStripBlock = 256;  // four waves, each its own strip
constexpr int kStripWaves = kStripBlock / kWave;

// Launch shape of a walk: strips of one wave, four waves per block, 12 x-rows
// per wave, or 8 or 4 on smaller grids for at least 4096 waves (one round of 16
// per compute unit). The explicit step at 4096x2048 with three signals (FP64
// upwind, FP32 upwind, FP32 van Leer): 12 rows take 131, 74 and 109 us, 8 rows
// 135, 77 and 111, 16 rows 138, 84 and 111, 20 rows 128, 91 and 121, 28 rows
// 151, 78 and 111: longer walks read fewer rows twice but leave a last round of
// waves nearly empty.
// FP32 walks take 2 rows where 4 leave less than 3072 waves, and 1 where 2 leave
// less than 2048: on small grids a walk is a chain of rows, and one of a single
// row, whose three rows are read at once, the latency of a thread per site. FP64
// walks stay at 4, since with three signals their bytes count sooner: two rows
// lose 5 % at 790x512, one 6 % at 420x350. us with 1, 2 and 4 rows, three signals:
//             FP32 upwind       FP32 van Leer     a Crank-Nicolson step   FP64 upwind
//   256x128    5.3  6.2  8.4     9.7 10.8 13.5    190  359  418             6.8  8.2 10.6
//   400x300    6.3  6.8  9.0    11.1 11.8 14.4    198  210  262            10.3  9.3 11.3
//   768x512    8.4  8.2  9.2    14.3 13.9 15.0    237  228  256            15.7 12.9 12.9
//   1024x512   9.7  9.3 10.3    16.4 15.5 17.2    277  261  290            18.8 16.2 15.9
//   1531x769  18.1 17.2 15.4    28.9 27.5 25.2    411  398  354            35.4 29.1 25.8
// (the 256x128 Crank-Nicolson steps are bimodal: 185 to 333 with one row).
struct AdrShape {
  uint32_t strips, rows, blocks;
};

inline AdrShape adr_shape(uint32_t strips, uint32_t nx, uint32_t rows) {
  return AdrShape{strips, rows, (strips * ((nx + rows - 1) / rows) + kStripWaves - 1) / kStripWaves};
}

inline AdrShape adr_shape(uint32_t nx, uint32_t ny, bool limited, uint32_t precision) {
  const uint32_t width = static_cast<uint32_t>(kWave) - (limited ? 4 : 2);
  const uint32_t strips = (ny + width - 1) / width;
  uint32_t rows = 12;
  auto waves = [&] { return static_cast<uint64_t>(strips) * ((nx + rows - 1) / rows); };
  while (rows > 4 && waves() < 4096) rows -= 4;
  if (precision == 32) {
    if (rows == 4 && waves() < 3072) rows = 2;
    if (rows == 2 && waves() < 2048) rows = 1;
  }
  return adr_shape(strips, nx, rows);
}

// What one lane holds of one x-row of its column: the S levels, the velocities
// of the site's lower faces, and what of the site a face next to it needs
// (kOpen: a flux may cross it; kLimit: the limited correction may read it).
// Beyond a fixed face stands a ghost site, open and holding the reservoir's
// level; beyond a closed face a site that is neither.
constexpr uint32_t kOpen = 1, kLimit = 2;

template <typename T, int S>
struct StripRow {
  T c[S];
  float ux, uy;
  uint32_t site;
};

// A value from the lane below or above (columns col - 1, col + 1); lanes 0
// and 63 get zero from beyond the wave.
__device__ inline float lane_below(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ inline float lane_above(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}
template <int kControl>
__device__ inline double lane_shift(double v) {
  const uint64_t bits = static_cast<uint64_t>(__double_as_longlong(v));
  const uint32_t lo = static_cast<uint32_t>(
      __builtin_amdgcn_update_dpp(0, static_cast<int>(bits), kControl, 0xf, 0xf, true));
  const uint32_t hi = static_cast<uint32_t>(
      __builtin_amdgcn_update_dpp(0, static_cast<int>(bits >> 32), kControl, 0xf, 0xf, true));
  return __longlong_as_double(
      static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
}
__device__ inline double lane_below(double v) { return lane_shift<0x138>(v); }
__device__ inline double lane_above(double v) { return lane_shift<0x130>(v); }

// The lane's place in the strip that wave `walk` walks, x-rows [xa, xb).
template <bool kLimited, bool kPatched>
struct Strip {
  static constexpr int kHalo = kLimited ? 2 : 1;
  static constexpr int kWidth = kWave - 2 * kHalo;
  const AdrParams& P;
  uint32_t nx, ny, y;
  size_t n;
  int xa, xb, col;
  // This lane's column is on the grid or (periodic) stands for its partner;
  // the wave updates it.
  bool loads, owns;
  int ghost_y;    // the fixed y face this column lies beyond, or -1
  bool limits_y;  // the column's sites serve the limiter
  bool on_y, xper, yper, field;

  __device__ Strip(const AdrParams& params, uint32_t walk, uint32_t strips, uint32_t rows)
      : P(params), nx(params.nx), ny(params.ny), n(static_cast<size_t>(params.nx) * params.ny) {
    const int lane = threadIdx.x & (kWave - 1);
    walk = __builtin_amdgcn_readfirstlane(walk);
    xa = static_cast<int>(min(nx, (walk / strips) * rows));
    xb = static_cast<int>(min(nx, static_cast<uint32_t>(xa) + rows));
    xper = P.kind[0] == MSIM_PERIODIC;
    yper = P.kind[2] == MSIM_PERIODIC;
    field = P.has_field != 0;
    col = static_cast<int>((walk % strips) * kWidth) + lane - kHalo;
    on_y = col >= 0 && col < static_cast<int>(ny);
    int src_col = col;
    if (!on_y && yper) src_col = col < 0 ? col + static_cast<int>(ny) : col - static_cast<int>(ny);
    loads = src_col >= 0 && src_col < static_cast<int>(ny) && (on_y || (yper && ny > 1));
    ghost_y = ny == 1                                                              ? -1
              : col == -1 && P.kind[2] == MSIM_FIXED                               ? 2
              : col == static_cast<int>(ny) && P.kind[3] == MSIM_FIXED             ? 3
                                                                                   : -1;
    limits_y = on_y || ny >= 3;
    owns = on_y && lane >= kHalo && lane < kHalo + kWidth;
    y = static_cast<uint32_t>(src_col);
  }

  // Row xx of the walk, xx in [-H, nx + H - 1]; `full` rows are the ones the
  // wave updates.
  template <typename T, int S>
  __device__ StripRow<T, S> load(int xx, bool full, const uint8_t* __restrict__ solid,
                                 const float* __restrict__ xf, const float* __restrict__ yf,
                                 const T* __restrict__ in) const {
    StripRow<T, S> w{};
    const bool on_x = xx >= 0 && xx < static_cast<int>(nx);
    if (field && owns && xx >= 0 && xx <= static_cast<int>(nx))
      w.ux = xf[static_cast<size_t>(xx) * ny + y];
    int row = xx;
    if (!on_x) {
      if (xper && nx > 1) {
        row = xx < 0 ? xx + static_cast<int>(nx) : xx - static_cast<int>(nx);
      } else {
        const int face = xx == -1 ? 0 : xx == static_cast<int>(nx) ? 1 : -1;
        if (nx > 1 && on_y && face >= 0 && P.kind[face] == MSIM_FIXED) {
          w.site = kOpen;
#pragma unroll
          for (int s = 0; s < S; ++s)
            w.c[s] = static_cast<T>(reservoir<kPatched>(P, face, s, y));
        }
        return w;
      }
    }
    if (row < 0 || row >= static_cast<int>(nx)) return w;
    if (loads) {
      const size_t i = static_cast<size_t>(row) * ny + y;
      const uint32_t limit = limits_y && (on_x || nx >= 3) ? kOpen | kLimit : kOpen;
      w.site = solid[i] != 0 ? 0u : limit;
#pragma unroll
      for (int s = 0; s < S; ++s) w.c[s] = in[s * n + i];
    } else if (ghost_y >= 0 && on_x) {
      w.site = kOpen;
#pragma unroll
      for (int s = 0; s < S; ++s)
        w.c[s] = static_cast<T>(reservoir<kPatched>(P, ghost_y, s, static_cast<uint32_t>(row)));
    }
    if (full && field && col >= 0 && col <= static_cast<int>(ny))
      w.uy = yf[static_cast<size_t>(row) * (ny + 1) + static_cast<uint32_t>(col)];
    return w;
  }
};

// What crosses a face from the lower site (level a) to the upper one (b):
// FP64 the flux, FP32 its advective part (the diffusive one is the site's)
// and, under van Leer, the correction; zero where the face is closed. far_a
// and far_b are the levels one further out, `lim` the sites a and b, lim_a
// and lim_b those further out.
template <typename T>
struct StripFace {
  T flux;
  T extra;  // FP32 van Leer
};

template <bool kLimited, typename T>
__device__ inline StripFace<T> strip_face(T a, T b, float velocity, [[maybe_unused]] float diffusion,
                                          [[maybe_unused]] T ih, bool open,
                                          [[maybe_unused]] T far_a, [[maybe_unused]] T far_b,
                                          [[maybe_unused]] uint32_t lim,
                                          [[maybe_unused]] uint32_t lim_a,
                                          [[maybe_unused]] uint32_t lim_b) {
  constexpr bool kF64 = sizeof(T) == 8;
  const T u = static_cast<T>(velocity);
  const bool forward = u >= T(0);
  T f = u * (forward ? a : b);
  if constexpr (kF64) f -= static_cast<T>(diffusion) * (b - a) * ih;
  T extra = T(0);
  if constexpr (kLimited) {
    const T inc = van_leer_increment<T>(forward ? a : b, forward ? b : a, forward ? far_a : far_b);
    const bool corrected = (lim & (forward ? lim_a : lim_b) & kLimit) != 0;
    if constexpr (kF64) {
      if (corrected) f += u * inc;
    } else {
      if (corrected) extra = u * inc;
    }
  }
  return StripFace<T>{open ? f : T(0), extra};
}

// The FP32 transport rate of a site (transport_rates_into,
// signals.cpp:1145-1291; transport_rate_f32 spells it out) from its level,
// its neighbours' and its faces, in the reference's order.
template <bool kLimited>
__device__ inline float strip_rate(const AdrParams& P, float D, float c, float xl, float xu,
                                   float yl, float yu, const StripFace<float>& xlo,
                                   const StripFace<float>& xhi, const StripFace<float>& ylo,
                                   const StripFace<float>& yhi, bool open_xlo, bool open_xhi,
                                   bool open_ylo, bool open_yhi, float ihx, float ihy) {
  float rate = 0.0f;
  if (P.nx != 1) {
    const float l = open_xlo ? xl : c, u = open_xhi ? xu : c;
    rate += D * (l - (2.0f * c) + u) * ihx * ihx;
    rate -= (xhi.flux - xlo.flux) * ihx;
    if constexpr (kLimited) rate -= (xhi.extra - xlo.extra) * ihx;
  }
  if (P.ny != 1) {
    const float l = open_ylo ? yl : c, u = open_yhi ? yu : c;
    rate += D * (l - (2.0f * c) + u) * ihy * ihy;
    rate -= (yhi.flux - ylo.flux) * ihy;
    if constexpr (kLimited) rate -= (yhi.extra - ylo.extra) * ihy;
  }
  return rate;
}

// The sites of a row's y neighbours, from the next lanes.
__device__ inline uint32_t site_below(uint32_t site) {
  return __float_as_uint(lane_below(__uint_as_float(site)));
}
__device__ inline uint32_t site_above(uint32_t site) {
  return __float_as_uint(lane_above(__uint_as_float(site)));
}

}  // namespace msim
