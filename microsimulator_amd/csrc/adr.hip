// Explicit advection-diffusion-reaction step on the device, one layer.
//
// One marching kernel, k_adr_step, in two arithmetic forms: a wave owns a
// strip of columns and walks x, each lane advancing every signal of its
// site, so levels, faces, mask and occupancy are read from memory once.
//  * FP32 levels: the reference's per-site rate in its own float order
//    (cpp/core/signals.cpp:1145-1291 transport, 305-320 affine reaction,
//    1109-1134 forward Euler), Monod uptake as the affine loss
//    vmax*phi/(K+c) it equals under forward Euler.
//  * FP64 levels in face-flux form: every face flux is one expression of the
//    two sites it joins, so what leaves one site enters the other bit for
//    bit; the step's mass, boundary supply and uptake are tallied in FP64 for
//    the conservation ledger.
// A site whose update is negative or non-finite raises a flag (the reference
// throws, signals.cpp:1124-1130); the step is then refused as a whole.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "adr_site.hpp"
#include "adr_strip.hpp"
#include "common.hpp"
#include "internal.hpp"

namespace msim {
namespace {

constexpr int kAdrBlock = kStripBlock;

// The ledger of a step lives as per-block partial sums (mass after, boundary
// supply rate, uptake rate, for each signal) in two generations by step
// parity. 3S further blocks of the next step's launch each add one partial of
// the previous step (in a fixed order) into its ledger row, so no grid-wide
// fence is needed; a last small launch adds the final step's.
struct LedgerParts {
  double* parts;   // [2][3 * kMaxSignals][blocks]
  double* ledger;  // [steps][S][4]
  uint32_t blocks;
};

template <int S, int NT>
__device__ inline void fold_ledger(const AdrParams& P, LedgerParts L, uint32_t step, float dt,
                                   uint32_t j, double* lds) {
  // Partial j of `step` into ledger row `step`.
  const double* v =
      L.parts + (static_cast<size_t>(step & 1) * (3 * kMaxSignals) + j) * L.blocks;
  double total = 0.0;
  for (uint32_t b = threadIdx.x; b < L.blocks; b += NT) total += v[b];
  total = block_sum<NT>(total, lds);
  if (threadIdx.x == 0) {
    const double volume =
        static_cast<double>(P.dx) * static_cast<double>(P.dy) * static_cast<double>(P.dz);
    const uint32_t s = j / 3, what = j % 3;
    double* row = L.ledger + (static_cast<size_t>(step) * S + s) * 4;
    row[1 + what] = what == 0 ? total * volume : static_cast<double>(dt) * total * volume;
  }
}

// Sums of K values over a block in one pass: every wave reduces its K values,
// then thread 0 adds the waves in order. Only thread 0's result is meaningful.
template <int NT, int K>
__device__ inline void block_sums(double (&v)[K], double* lds) {
  constexpr int kWaves = NT / kWave;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = wave_sum(v[k]);
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < K; ++k) lds[k * kWaves + wave] = v[k];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      double t = 0.0;
      for (int w = 0; w < kWaves; ++w) t += lds[k * kWaves + w];
      v[k] = t;
    }
  }
}

// One forward-Euler step for S signals, marching: each wave owns a strip of
// 64 - 2H columns and `rows` x-rows and walks x on its own, one column per
// lane, so each level is read from memory once; its x neighbours come from
// registers and its y neighbours from the next lanes (H = 1 for the upwind
// scheme, 2 under van Leer, whose correction reads the site two away: the
// strip's first and last H lanes only hold the columns outside it, their
// periodic partners or their ghosts). The next row's loads are issued a row
// ahead.
//  * Every face's flux (and limited correction) is computed once: the upper
//    x face's is kept for the next row, the upper y face's comes from the
//    lane above. The two sites of a face have the same expression for it, so
//    this changes no bit.
//  * T = float: the reference's per-site rate in its float order
//    (signals.cpp:1145-1291, 305-320, 1109-1134; transport_rate_f32 and
//    fe_update_f32 spell it out), so every site matches its CPU step.
//  * T = double: face-flux form; the step's mass, boundary supply and uptake
//    go to the ledger partials.
// A site whose update is non-finite, or negative under upwind, raises a flag
// (the reference throws, signals.cpp:1119-1131); the step is then refused as
// a whole. Under van Leer each block also leaves the largest level it wrote,
// and flags[2] says whether any was negative, for the settle that follows.
// The step was bound by instructions and barriers, not memory: every face
// computed from both sides with a branch per case, an LDS row and a barrier
// per x-row. 4096x2048, three signals with Monod, before and after: FP64
// upwind 161 and 130 us (3.9 TB/s of its 61 B per site), FP32 upwind 86 and 74
// us (4.2 TB/s), FP32 van Leer with its settle 207 and 109 us; 1531x769, two
// signals, FP32 van Leer 40.5 and 20.8 us.
template <typename T, int S, bool kAffine, bool kLimited, bool kPatched>
__global__ __launch_bounds__(kAdrBlock) void k_adr_step(
    AdrParams P, const uint8_t* __restrict__ solid, const float* __restrict__ xf,
    const float* __restrict__ yf, const float* __restrict__ phi, const float* __restrict__ source,
    const float* __restrict__ loss, const T* __restrict__ in, T* __restrict__ out, float dt,
    uint32_t* flags, uint32_t step, uint32_t rows, uint32_t strips, LedgerParts L,
    double* largest) {
  constexpr bool kF64 = sizeof(T) == 8;
  using Lane = Strip<kLimited, kPatched>;
  using Row = StripRow<T, S>;
  using Face = StripFace<T>;
  __shared__ double s_red[(kF64 ? 3 * S : 1) * kStripWaves];
  // An earlier step failed: the run stops there. (flags[1] holds the first
  // failed step; a failure of this step may be seen here half-published, and
  // then the previous step's ledger row is still folded, as it is valid.)
  if (flags[0] != 0 && flags[1] < step) return;
  if constexpr (kF64) {
    // The blocks past the walking ones add the previous step's ledger.
    if (blockIdx.x >= L.blocks) {
      if (step > 0)
        fold_ledger<S, kAdrBlock>(P, L, step - 1, dt, blockIdx.x - L.blocks, s_red);
      return;
    }
  }
  if (flags[0] != 0) return;  // this step already failed elsewhere
  const Lane at(P, xcd_tile(blockIdx.x, L.blocks) * kStripWaves + threadIdx.x / kWave, strips,
                rows);
  const int xa = at.xa, xb = at.xb, col = at.col;
  const uint32_t nx = at.nx, ny = at.ny, y = at.y;
  const size_t n = at.n;
  const bool owns = at.owns, field = at.field, monod = P.has_monod != 0;
  auto load = [&](int xx, bool full) {
    return at.template load<T, S>(xx, full, solid, xf, yf, in);
  };
  // What a site's own update reads besides, for rows the wave updates.
  struct Extra {
    float src[kAffine ? S : 1], los[kAffine ? S : 1], phi;
  };
  auto load_extra = [&](int xx) {
    Extra w{};
    if (xx >= xb || !owns) return w;
    const size_t i = static_cast<size_t>(xx) * ny + y;
    if (monod) w.phi = phi[i];
    if constexpr (kAffine) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        w.src[s] = source[s * n + i];
        w.los[s] = loss[s * n + i];
      }
    }
    return w;
  };
  const T ihx = T(1) / static_cast<T>(P.dx), ihy = T(1) / static_cast<T>(P.dy);
  auto face = [&](T a, T b, float velocity, int s, T ih, bool open, T far_a, T far_b, uint32_t lim,
                  uint32_t lim_a, uint32_t lim_b) {
    return strip_face<kLimited, T>(a, b, velocity, P.diffusion[s], ih, open, far_a, far_b, lim,
                                   lim_a, lim_b);
  };
  double acc[kF64 ? 3 * S : 1] = {};
  T top = T(0);  // largest level written (van Leer)
  bool bad = false, negative = false;
  if (xa < xb) {
    // Rows xx - 1 .. xx + 1 (and xx + 2 under van Leer).
    Row prev = load(xa - 1, false);
    Row cur = load(xa, true);
    Row next = load(xa + 1, xa + 1 < xb);
    Row n2 = kLimited ? load(xa + 2, xa + 2 < xb) : Row{};
    Extra own = load_extra(xa), own_next = load_extra(xa + 1);
    Face below[S];  // across the lower x face of the current row
    {
      const Row p2 = kLimited ? load(xa - 2, false) : Row{};
#pragma unroll
      for (int s = 0; s < S; ++s) {
        below[s] = face(prev.c[s], cur.c[s], field ? cur.ux : P.advection[s][0], s, ihx,
                        (prev.site & cur.site & kOpen) != 0, p2.c[s], next.c[s],
                        prev.site & cur.site, p2.site, next.site);
      }
    }
    for (int xx = xa; xx < xb; ++xx) {
      constexpr int kAhead = kLimited ? 3 : 2;
      const Row ahead =
          xx + kAhead < xb + Lane::kHalo ? load(xx + kAhead, xx + kAhead < xb) : Row{};
      const Extra own_ahead = load_extra(xx + 2);
      const size_t i = static_cast<size_t>(xx) * ny + y;
      // The y neighbours' sites, and whether the four faces are open.
      const uint32_t site_lo = site_below(cur.site), site_hi = site_above(cur.site);
      const bool open_xlo = (prev.site & cur.site & kOpen) != 0;
      const bool open_xhi = (cur.site & next.site & kOpen) != 0;
      const bool open_ylo = (site_lo & cur.site & kOpen) != 0;
      const bool open_yhi = (cur.site & site_hi & kOpen) != 0;
      [[maybe_unused]] uint32_t site_lo2 = 0;
      if constexpr (kLimited) site_lo2 = site_below(site_lo);
      const bool fluid = (cur.site & kOpen) != 0;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const T c = cur.c[s];
        const T ylo_v = lane_below(c), yhi_v = lane_above(c);
        [[maybe_unused]] T far_lo = T(0);
        if constexpr (kLimited) far_lo = lane_below(ylo_v);
        const Face xlo = below[s];
        const Face xhi = face(c, next.c[s], field ? next.ux : P.advection[s][0], s, ihx, open_xhi,
                              prev.c[s], n2.c[s], cur.site & next.site, prev.site, n2.site);
        below[s] = xhi;
        const Face ylo = face(ylo_v, c, field ? cur.uy : P.advection[s][1], s, ihy, open_ylo,
                              far_lo, yhi_v, site_lo & cur.site, site_lo2, site_hi);
        Face yhi;
        yhi.flux = lane_above(ylo.flux);
        if constexpr (kLimited && !kF64) yhi.extra = lane_above(ylo.extra);
        T v;
        if constexpr (!kF64) {
          float rate = strip_rate<kLimited>(P, P.diffusion[s], c, prev.c[s], next.c[s], ylo_v,
                                            yhi_v, xlo, xhi, ylo, yhi, open_xlo, open_xhi,
                                            open_ylo, open_yhi, ihx, ihy);
          if constexpr (kAffine) rate += own.src[s] - (own.los[s] * c);
          if (monod) {
            const float uptake = P.vmax[s] * own.phi / (P.monod_k[s] + c);
            rate += 0.0f - (uptake * c);
          }
          v = c + (dt * rate);
        } else {
          double rate = 0.0, supply = 0.0;
          // A flux through an edge of the grid is supplied from outside.
          if (nx != 1) {
            if (xx == 0 && !at.xper) supply += xlo.flux * ihx;
            if (xx + 1 == static_cast<int>(nx) && !at.xper) supply -= xhi.flux * ihx;
            rate -= (xhi.flux - xlo.flux) * ihx;
          }
          if (ny != 1) {
            if (col == 0 && !at.yper) supply += ylo.flux * ihy;
            if (col + 1 == static_cast<int>(ny) && !at.yper) supply -= yhi.flux * ihy;
            rate -= (yhi.flux - ylo.flux) * ihy;
          }
          double lossr = 0.0;
          if constexpr (kAffine) {
            rate += static_cast<double>(own.src[s]);
            supply += static_cast<double>(own.src[s]);
            lossr += static_cast<double>(own.los[s]);
          }
          if (monod) {
            lossr += static_cast<double>(P.vmax[s]) * static_cast<double>(own.phi) /
                     (static_cast<double>(P.monod_k[s]) + c);
          }
          rate -= lossr * c;
          v = c + static_cast<double>(dt) * rate;
          // Solid sites hold their (zero) level; the mass counts only what moved.
          if (owns && fluid) {
            acc[3 * s + 0] += v;
            acc[3 * s + 1] += supply;
            acc[3 * s + 2] += lossr * c;
          }
        }
        if (owns) {
          if (fluid) {
            bad = bad || !isfinite(v) || (!kLimited && v < T(0));
          } else {
            v = c;
          }
          if constexpr (kLimited) {
            top = max(top, v);
            negative = negative || v < T(0);
          }
          out[s * n + i] = v;
        }
      }
      own = own_next;
      own_next = own_ahead;
      prev = cur;
      cur = next;
      if constexpr (kLimited) {
        next = n2;
        n2 = ahead;
      } else {
        next = ahead;
      }
    }
  }
  if (bad) {
    atomicOr(&flags[0], kFlagNegative);
    atomicMin(&flags[1], step);
  }
  if constexpr (kLimited) {
    if (negative) flags[2] = step + 1;
    const double m = block_max<kAdrBlock>(static_cast<double>(top), s_red);
    if (threadIdx.x == 0) largest[blockIdx.x] = m;
  }
  if constexpr (kF64) {
    block_sums<kAdrBlock, 3 * S>(acc, s_red);
    if (threadIdx.x == 0) {
#pragma unroll
      for (int k = 0; k < 3 * S; ++k) {
        L.parts[(static_cast<size_t>(step & 1) * (3 * kMaxSignals) + k) * L.blocks + blockIdx.x] =
            acc[k];
      }
    }
  }
}

// settle_step_levels then validate_signal_levels (signals.cpp:979-1001,
// 754-784) after a van Leer step, in place over the S*N levels it wrote:
// levels below zero by no more than 16 epsilon (of the level type) times the
// largest level become zero; a level still negative or not finite refuses
// the step. Every block takes the largest level from the step's block
// maxima. `marked`: the step said in flags[2] whether it wrote a negative
// level (a level that is not finite has already refused it), and there is
// nothing to do where it did not: 3 us in place of a pass over the levels.
template <typename T>
__global__ __launch_bounds__(kAdrBlock) void k_adr_settle(T* __restrict__ levels, size_t count,
                                                          const double* __restrict__ largest,
                                                          uint32_t parts, uint32_t* flags,
                                                          uint32_t step, uint32_t marked) {
  __shared__ double s_red[kAdrBlock / kWave];
  __shared__ double s_top;
  if (flags[0] != 0) return;
  if (marked != 0 && flags[2] != step + 1) return;
  double m = 0.0;
  for (uint32_t b = threadIdx.x; b < parts; b += kAdrBlock) m = fmax(m, largest[b]);
  m = block_max<kAdrBlock>(m, s_red);
  if (threadIdx.x == 0) s_top = m;
  __syncthreads();
  const T top = static_cast<T>(s_top);
  const T eps = sizeof(T) == 8 ? static_cast<T>(DBL_EPSILON) : static_cast<T>(FLT_EPSILON);
  const T rounding = T(-16) * eps * top;
  bool bad = false;
  for (size_t i = static_cast<size_t>(blockIdx.x) * kAdrBlock + threadIdx.x; i < count;
       i += static_cast<size_t>(gridDim.x) * kAdrBlock) {
    const T v = levels[i];
    if (v < T(0)) {
      if (v >= rounding) {
        levels[i] = T(0);
      } else {
        bad = true;
      }
    } else if (!isfinite(v)) {
      bad = true;
    }
  }
  if (bad) {
    atomicOr(&flags[0], kFlagLevels);
    atomicMin(&flags[1], step);
  }
}

// Adds the final step's ledger partials.
template <int S>
__global__ __launch_bounds__(kAdrBlock) void k_adr_ledger_tail(AdrParams P, LedgerParts L,
                                                               uint32_t step, float dt,
                                                               const uint32_t* flags) {
  __shared__ double s_red[kAdrBlock / kWave];
  if (flags[0] != 0) return;
  fold_ledger<S, kAdrBlock>(P, L, step, dt, blockIdx.x, s_red);
}

// Sum of levels per signal (FP64), and the greatest outflow rate over fluid
// sites (SignalGrid::transport_cache, signals.cpp:870-896) for the explicit
// bound. On a small grid the reductions are all there is: every quantity's wave
// sums meet in one barrier, and signals that are not there take no part (64x48
// with one signal: 14.3 to 7.9 us).
template <typename T>
__global__ __launch_bounds__(kAdrBlock) void k_adr_survey(
    AdrParams P, const uint8_t* __restrict__ solid, const float* __restrict__ xf,
    const float* __restrict__ yf, const T* __restrict__ levels, double* partials, CgState* st,
    double* mass) {
  constexpr int kWaves = kAdrBlock / kWave;
  __shared__ double s_red[kMaxSignals + 1][kWaves];
  __shared__ double s_total[kMaxSignals + 1];
  __shared__ bool s_last;
  const size_t n = static_cast<size_t>(P.nx) * P.ny;
  double acc[kMaxSignals + 1];
#pragma unroll
  for (int k = 0; k <= kMaxSignals; ++k) acc[k] = 0.0;
  const size_t stride = static_cast<size_t>(gridDim.x) * kAdrBlock;
  for (size_t i = static_cast<size_t>(blockIdx.x) * kAdrBlock + threadIdx.x; i < n; i += stride) {
    for (uint32_t s = 0; s < P.signals && s < kMaxSignals; ++s)
      acc[s] += static_cast<double>(levels[s * n + i]);
    if (P.has_field != 0 && solid[i] == 0) {
      const uint32_t x = static_cast<uint32_t>(i / P.ny), y = static_cast<uint32_t>(i % P.ny);
      double outflow = 0.0;
      if (P.nx > 1) {
        outflow += (fmax(static_cast<double>(xf[i + P.ny]), 0.0) -
                    fmin(static_cast<double>(xf[i]), 0.0)) *
                   (1.0 / static_cast<double>(P.dx));
      }
      if (P.ny > 1) {
        const size_t yfi = static_cast<size_t>(x) * (P.ny + 1) + y;
        outflow += (fmax(static_cast<double>(yf[yfi + 1]), 0.0) -
                    fmin(static_cast<double>(yf[yfi]), 0.0)) *
                   (1.0 / static_cast<double>(P.dy));
      }
      acc[kMaxSignals] = fmax(acc[kMaxSignals], outflow);
    }
  }
  const uint32_t signals = min(P.signals, static_cast<uint32_t>(kMaxSignals));
  // The block's total of each quantity, in wave order, in s_total.
  auto reduce = [&](double (&v)[kMaxSignals + 1]) {
    const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
#pragma unroll
    for (int k = 0; k < kMaxSignals; ++k) {
      if (static_cast<uint32_t>(k) < signals) {
        const double w = wave_sum(v[k]);
        if (lane == 0) s_red[k][wave] = w;
      }
    }
    const double w = wave_max(v[kMaxSignals]);
    if (lane == 0) s_red[kMaxSignals][wave] = w;
    __syncthreads();
    if (threadIdx.x < signals) {
      double t = 0.0;
      for (int j = 0; j < kWaves; ++j) t += s_red[threadIdx.x][j];
      s_total[threadIdx.x] = t;
    } else if (threadIdx.x == kMaxSignals) {
      double t = s_red[kMaxSignals][0];
      for (int j = 1; j < kWaves; ++j) t = fmax(t, s_red[kMaxSignals][j]);
      s_total[kMaxSignals] = t;
    }
    __syncthreads();
  };
  reduce(acc);
  if (threadIdx.x == 0) {
    for (uint32_t k = 0; k < signals; ++k)
      partials[static_cast<size_t>(k) * gridDim.x + blockIdx.x] = s_total[k];
    partials[static_cast<size_t>(kMaxSignals) * gridDim.x + blockIdx.x] = s_total[kMaxSignals];
    __threadfence();
    s_last = atomicAdd(&st->ticket[kTicketMisc], 1u) + 1 == gridDim.x;
  }
  __syncthreads();
  if (!s_last) return;
  __threadfence();
#pragma unroll
  for (int k = 0; k <= kMaxSignals; ++k) {
    double v = 0.0;
    if (static_cast<uint32_t>(k) < signals || k == kMaxSignals) {
      for (uint32_t b = threadIdx.x; b < gridDim.x; b += kAdrBlock) {
        const double p = partials[static_cast<size_t>(k) * gridDim.x + b];
        v = k == kMaxSignals ? fmax(v, p) : v + p;
      }
    }
    acc[k] = v;
  }
  reduce(acc);
  if (threadIdx.x == 0) {
    st->ticket[kTicketMisc] = 0;
    const double volume =
        static_cast<double>(P.dx) * static_cast<double>(P.dy) * static_cast<double>(P.dz);
    for (uint32_t k = 0; k < kMaxSignals; ++k) mass[k] = k < signals ? s_total[k] * volume : 0.0;
    st->peak = s_total[kMaxSignals];
  }
}

double* survey_mass(AdrDevice& a) { return reinterpret_cast<double*>(a.state.data() + 1); }

uint32_t site_blocks(size_t n) { return static_cast<uint32_t>((n + kAdrBlock - 1) / kAdrBlock); }

}  // namespace

// The kernels' parameters of a signal grid (one layer): shape, spacing,
// boundary kinds and values, diffusion, Monod constants, the scheme and
// which optional arrays it has. The velocity field and patches are set by
// the caller.
AdrParams transport_params(const msim_signal_grid& grid) {
  AdrParams P;
  std::memset(&P, 0, sizeof(P));
  P.nx = grid.grid.nx;
  P.ny = grid.grid.ny;
  P.nz = grid.grid.nz;
  P.signals = grid.signal_count;
  P.dx = grid.grid.dx;
  P.dy = grid.grid.dy;
  P.dz = grid.grid.dz;
  for (int f = 0; f < 6; ++f) P.kind[f] = grid.grid.boundary[f];
  for (uint32_t s = 0; s < grid.signal_count; ++s) {
    P.diffusion[s] = grid.diffusion[s];
    for (int f = 0; f < 6; ++f)
      P.boundary[s][f] = grid.boundary_values != nullptr ? grid.boundary_values[6 * s + f] : 0.0f;
    if (grid.monod_vmax != nullptr) {
      P.vmax[s] = grid.monod_vmax[s];
      P.monod_k[s] = grid.monod_k[s];
    }
    for (int a = 0; a < 3; ++a)
      P.advection[s][a] = grid.advection != nullptr ? grid.advection[3 * s + a] : 0.0f;
  }
  P.has_field = grid.x_faces != nullptr ? 1 : 0;
  P.limited = grid.advection_scheme == MSIM_VAN_LEER ? 1 : 0;
  P.has_affine = grid.loss_rates != nullptr ? 1 : 0;
  P.has_monod = grid.phi != nullptr ? 1 : 0;
  return P;
}

void adr_upload(Context& ctx, const msim_signal_grid& grid, const void* levels,
                uint32_t precision, bool use_flow_field) {
  // Coupled state belongs to the grid it was uploaded with.
  ctx.coupled.uploaded = false;
  auto& a = ctx.adr;
  auto& P = a.params;
  const uint32_t nz = grid.grid.nz;
  const size_t n = static_cast<size_t>(grid.grid.nx) * grid.grid.ny * nz;
  const uint32_t S = grid.signal_count;
  const bool same_spec = a.uploaded && grid.revision != 0 && grid.revision == a.revision &&
                         P.nx == grid.grid.nx && P.ny == grid.grid.ny && P.nz == nz &&
                         P.signals == S && !use_flow_field && !a.flow_field;
  P = transport_params(grid);
  a.integration = grid.integration;
  a.max_iterations = grid.solver_max_iterations;
  a.absolute_tolerance = grid.solver_absolute_tolerance;
  a.relative_tolerance = grid.solver_relative_tolerance;
  a.last_report = msim_signal_report{1, 0, 0.0f};
  a.predicted_iterations = kPredictedIterations;
  P.has_field = (use_flow_field || grid.x_faces != nullptr) ? 1 : 0;
  const bool patched = grid.patches != nullptr && grid.patch_count > 0;
  a.precision = precision;
  const size_t bytes = S * n * (precision == 64 ? sizeof(double) : sizeof(float));
  a.levels_a.reserve(bytes);
  a.levels_b.reserve(bytes);
  a.current = 0;
  a.flags.reserve(3);
  a.state.reserve(2);  // the second holds the survey's masses
  // Ledger partials [2][3 * kMaxSignals][blocks], then the van Leer block
  // maxima [blocks]; the survey's partials reuse the front. FP32's shape has
  // the more blocks.
  const uint32_t step_parts = adr_shape(P.nx, P.ny, P.limited != 0, 32).blocks;
  a.partials.reserve(std::max<size_t>(
      static_cast<size_t>(3 * kMaxSignals * 2 + 1) * step_parts,
      static_cast<size_t>(kMaxSignals + 1) * 2048));
  if (!same_spec) {
    a.has_edge = patched;
    if (patched && nz > 1) {
      // GridBoundary::values_at (signals.cpp:439-447) for every boundary site
      // of the six faces, in each face's (first, second) order: the last
      // patch holding the site, else the face's value.
      const uint32_t extent[6][2] = {{P.ny, nz}, {P.ny, nz}, {P.nx, nz},
                                     {P.nx, nz}, {P.nx, P.ny}, {P.nx, P.ny}};
      size_t offset[7] = {0};
      for (int f = 0; f < 6; ++f)
        offset[f + 1] = offset[f] + static_cast<size_t>(extent[f][0]) * extent[f][1];
      const size_t row = offset[6];
      std::vector<float> edge(S * row);
      for (uint32_t s = 0; s < S; ++s) {
        for (int f = 0; f < 6; ++f) {
          for (uint32_t first = 0; first < extent[f][0]; ++first) {
            for (uint32_t second = 0; second < extent[f][1]; ++second) {
              float v = P.boundary[s][f];
              for (uint32_t k = grid.patch_count; k-- > 0;) {
                const msim_boundary_patch& pt = grid.patches[k];
                if (static_cast<int>(pt.face) == f && first >= pt.begin[0] && first < pt.end[0] &&
                    second >= pt.begin[1] && second < pt.end[1]) {
                  v = pt.values[s];
                  break;
                }
              }
              edge[s * row + offset[f] + static_cast<size_t>(first) * extent[f][1] + second] = v;
            }
          }
        }
      }
      a.edge.reserve(edge.size());
      check(hipMemcpyAsync(a.edge.data(), edge.data(), edge.size() * sizeof(float),
                           hipMemcpyHostToDevice, ctx.stream),
            "upload boundary patches");
      check(hipStreamSynchronize(ctx.stream), "upload boundary patches");
    } else if (patched) {
      // GridBoundary::values_at (signals.cpp:439-447) for every boundary site
      // of the four in-plane faces (second in-plane index z = 0): the last
      // patch holding the site, else the face's value.
      const size_t row = 2 * static_cast<size_t>(P.ny) + 2 * static_cast<size_t>(P.nx);
      std::vector<float> edge(S * row);
      const uint32_t extent[4] = {P.ny, P.ny, P.nx, P.nx};
      const size_t offset[4] = {0, P.ny, 2 * static_cast<size_t>(P.ny),
                                2 * static_cast<size_t>(P.ny) + P.nx};
      for (uint32_t s = 0; s < S; ++s) {
        for (int f = 0; f < 4; ++f) {
          for (uint32_t along = 0; along < extent[f]; ++along) {
            float v = P.boundary[s][f];
            for (uint32_t k = grid.patch_count; k-- > 0;) {
              const msim_boundary_patch& pt = grid.patches[k];
              if (static_cast<int>(pt.face) == f && along >= pt.begin[0] && along < pt.end[0] &&
                  0 >= pt.begin[1] && 0 < pt.end[1]) {
                v = pt.values[s];
                break;
              }
            }
            edge[s * row + offset[f] + along] = v;
          }
        }
      }
      a.edge.reserve(edge.size());
      check(hipMemcpyAsync(a.edge.data(), edge.data(), edge.size() * sizeof(float),
                           hipMemcpyHostToDevice, ctx.stream),
            "upload boundary patches");
      check(hipStreamSynchronize(ctx.stream), "upload boundary patches");
    }
    a.solid.reserve(n);
    if (grid.grid.obstacles != nullptr) {
      check(hipMemcpyAsync(a.solid.data(), grid.grid.obstacles, n, hipMemcpyHostToDevice,
                           ctx.stream),
            "upload mask");
    } else {
      check(hipMemsetAsync(a.solid.data(), 0, n, ctx.stream), "clear mask");
    }
    if (use_flow_field) {
      a.xf.release();
      a.yf.release();
    } else if (grid.x_faces != nullptr) {
      a.xf.reserve(static_cast<size_t>(P.nx + 1) * P.ny * nz);
      a.yf.reserve(static_cast<size_t>(P.nx) * (P.ny + 1) * nz);
      check(hipMemcpyAsync(a.xf.data(), grid.x_faces, a.xf.size() * sizeof(float),
                           hipMemcpyHostToDevice, ctx.stream),
            "upload x faces");
      check(hipMemcpyAsync(a.yf.data(), grid.y_faces, a.yf.size() * sizeof(float),
                           hipMemcpyHostToDevice, ctx.stream),
            "upload y faces");
      if (nz > 1) {
        a.zf.reserve(static_cast<size_t>(P.nx) * P.ny * (nz + 1));
        check(hipMemcpyAsync(a.zf.data(), grid.z_faces, a.zf.size() * sizeof(float),
                             hipMemcpyHostToDevice, ctx.stream),
              "upload z faces");
      }
    }
    if (grid.phi != nullptr) {
      a.phi.reserve(n);
      check(hipMemcpyAsync(a.phi.data(), grid.phi, n * sizeof(float), hipMemcpyHostToDevice,
                           ctx.stream),
            "upload phi");
    }
    if (grid.loss_rates != nullptr) {
      a.source.reserve(S * n);
      a.loss.reserve(S * n);
      check(hipMemcpyAsync(a.loss.data(), grid.loss_rates, S * n * sizeof(float),
                           hipMemcpyHostToDevice, ctx.stream),
            "upload loss");
      check(hipMemcpyAsync(a.source.data(), grid.source_rates, S * n * sizeof(float),
                           hipMemcpyHostToDevice, ctx.stream),
            "upload source");
    }
  }
  P.edge = a.has_edge ? a.edge.data() : nullptr;
  a.flow_field = use_flow_field;
  a.flow_generation = use_flow_field ? ctx.flow.generation : 0;
  a.revision = grid.revision;
  check(hipMemcpyAsync(a.levels_a.data(), levels, bytes, hipMemcpyHostToDevice, ctx.stream),
        "upload levels");
  check(hipMemsetAsync(a.state.data(), 0, sizeof(CgState), ctx.stream), "clear state");
  const float* xf = use_flow_field ? ctx.flow.faces.data() : a.xf.data();
  const float* yf = use_flow_field ? ctx.flow.faces.data() + ctx.flow.x_faces() : a.yf.data();
  const uint32_t blocks = std::min<uint32_t>(site_blocks(n), 2048);
  if (nz > 1) {
    adr3_survey(ctx, xf, yf, a.zf.data(), reinterpret_cast<const float*>(a.levels_a.data()),
                a.state.data(), a.partials.data(), survey_mass(a));
  } else if (precision == 64) {
    k_adr_survey<double><<<blocks, kAdrBlock, 0, ctx.stream>>>(
        P, a.solid.data(), xf, yf, reinterpret_cast<const double*>(a.levels_a.data()),
        a.partials.data(), a.state.data(), survey_mass(a));
  } else {
    k_adr_survey<float><<<blocks, kAdrBlock, 0, ctx.stream>>>(
        P, a.solid.data(), xf, yf, reinterpret_cast<const float*>(a.levels_a.data()),
        a.partials.data(), a.state.data(), survey_mass(a));
  }
  check(hipGetLastError(), "launch k_adr_survey");
  CgState host[2];
  check(hipMemcpyAsync(host, a.state.data(), sizeof(host), hipMemcpyDeviceToHost, ctx.stream),
        "read survey");
  check(hipStreamSynchronize(ctx.stream), "survey");
  a.greatest_outflow = P.has_field != 0 ? host[0].peak : 0.0;
  static_assert(sizeof(a.host_mass) <= sizeof(CgState));
  std::memcpy(a.host_mass, host + 1, sizeof(a.host_mass));
  a.uploaded = true;
}

// The device arrays one transport step reads and writes besides the levels:
// the context's buffers, or the static scratch of the allocation-free step.
struct AdrView {
  const AdrParams* P;
  const uint8_t* solid;
  const float *phi, *source, *loss;
  uint32_t* flags;
};

AdrView view_of(Context& ctx) {
  auto& a = ctx.adr;
  return AdrView{&a.params, a.solid.data(), a.phi.data(), a.source.data(), a.loss.data(),
                 a.flags.data()};
}

template <typename T, int S, bool kAffine, bool kLimited>
void launch_step(hipStream_t stream, const AdrView& v, const AdrShape& sh, const float* xf,
                 const float* yf, const uint8_t* src, uint8_t* dst, float dt, uint32_t k,
                 LedgerParts L, double* largest) {
  const AdrParams& P = *v.P;
  const T* in = reinterpret_cast<const T*>(src);
  T* out = reinterpret_cast<T*>(dst);
  const uint32_t blocks = sh.blocks + (sizeof(T) == 8 ? 3 * S : 0);
  if (P.edge != nullptr) {
    k_adr_step<T, S, kAffine, kLimited, true><<<blocks, kAdrBlock, 0, stream>>>(
        P, v.solid, xf, yf, v.phi, v.source, v.loss, in, out, dt, v.flags, k, sh.rows, sh.strips,
        L, largest);
  } else {
    k_adr_step<T, S, kAffine, kLimited, false><<<blocks, kAdrBlock, 0, stream>>>(
        P, v.solid, xf, yf, v.phi, v.source, v.loss, in, out, dt, v.flags, k, sh.rows, sh.strips,
        L, largest);
  }
}

template <typename T, int S, bool kLimited>
void launch_typed(hipStream_t stream, const AdrView& v, const AdrShape& sh, const float* xf,
                  const float* yf, const uint8_t* src, uint8_t* dst, float dt, uint32_t k,
                  LedgerParts L, double* largest, bool settle = true) {
  const AdrParams& P = *v.P;
  if (P.has_affine != 0) {
    launch_step<T, S, true, kLimited>(stream, v, sh, xf, yf, src, dst, dt, k, L, largest);
  } else {
    launch_step<T, S, false, kLimited>(stream, v, sh, xf, yf, src, dst, dt, k, L, largest);
  }
  if (kLimited && settle) {
    const size_t count = static_cast<size_t>(S) * P.nx * P.ny;
    const uint32_t blocks = static_cast<uint32_t>(
        std::min<size_t>((count + kAdrBlock - 1) / kAdrBlock, 2048));
    k_adr_settle<T><<<blocks, kAdrBlock, 0, stream>>>(reinterpret_cast<T*>(dst), count, largest,
                                                      sh.blocks, v.flags, k, 1);
  }
}

// The explicit candidate of one FP32 step, unsettled.
template <int S>
void launch_candidate(Context& ctx, float dt, const float* in, float* out, uint32_t step,
                      const float* xf, const float* yf) {
  auto& a = ctx.adr;
  const bool limited = a.params.limited != 0;
  AdrShape sh = adr_shape(a.params.nx, a.params.ny, limited, 32);
  LedgerParts L{a.partials.data(), a.ledger.data(), sh.blocks};
  double* largest = a.partials.data() + static_cast<size_t>(3 * kMaxSignals * 2) * sh.blocks;
  const auto* src = reinterpret_cast<const uint8_t*>(in);
  auto* dst = reinterpret_cast<uint8_t*>(out);
  const AdrView v = view_of(ctx);
  if (limited) {
    launch_typed<float, S, true>(ctx.stream, v, sh, xf, yf, src, dst, dt, step, L, largest, false);
  } else {
    launch_typed<float, S, false>(ctx.stream, v, sh, xf, yf, src, dst, dt, step, L, largest,
                                  false);
  }
}

template <int S>
void launch_steps(Context& ctx, float dt, uint32_t steps, const float* xf, const float* yf) {
  auto& a = ctx.adr;
  const auto& P = a.params;
  const bool limited = P.limited != 0;
  AdrShape sh = adr_shape(P.nx, P.ny, limited, a.precision);
  LedgerParts L{a.partials.data(), a.ledger.data(), sh.blocks};
  double* largest = a.partials.data() + static_cast<size_t>(3 * kMaxSignals * 2) * sh.blocks;
  const AdrView v = view_of(ctx);
  for (uint32_t k = 0; k < steps; ++k) {
    const uint8_t* src = a.current == 0 ? a.levels_a.data() : a.levels_b.data();
    uint8_t* dst = a.current == 0 ? a.levels_b.data() : a.levels_a.data();
    if (a.precision == 64) {
      if (limited) {
        launch_typed<double, S, true>(ctx.stream, v, sh, xf, yf, src, dst, dt, k, L, largest);
      } else {
        launch_typed<double, S, false>(ctx.stream, v, sh, xf, yf, src, dst, dt, k, L, largest);
      }
    } else {
      if (limited) {
        launch_typed<float, S, true>(ctx.stream, v, sh, xf, yf, src, dst, dt, k, L, largest);
      } else {
        launch_typed<float, S, false>(ctx.stream, v, sh, xf, yf, src, dst, dt, k, L, largest);
      }
    }
    check(hipGetLastError(), "launch transport step");
    a.current ^= 1;
  }
  if (a.precision == 64 && steps > 0) {
    k_adr_ledger_tail<S><<<3 * S, kAdrBlock, 0, ctx.stream>>>(P, L, steps - 1, dt,
                                                             a.flags.data());
    check(hipGetLastError(), "launch ledger tail");
  }
}

void fe_candidate_f32(Context& ctx, float dt, const float* in, float* out, uint32_t step,
                      const float* xf, const float* yf) {
  switch (ctx.adr.params.signals) {
    case 1: launch_candidate<1>(ctx, dt, in, out, step, xf, yf); break;
    case 2: launch_candidate<2>(ctx, dt, in, out, step, xf, yf); break;
    case 3: launch_candidate<3>(ctx, dt, in, out, step, xf, yf); break;
    case 4: launch_candidate<4>(ctx, dt, in, out, step, xf, yf); break;
    case 5: launch_candidate<5>(ctx, dt, in, out, step, xf, yf); break;
    case 6: launch_candidate<6>(ctx, dt, in, out, step, xf, yf); break;
    case 7: launch_candidate<7>(ctx, dt, in, out, step, xf, yf); break;
    default: launch_candidate<8>(ctx, dt, in, out, step, xf, yf); break;
  }
  check(hipGetLastError(), "launch transport candidate");
}

void launch_settle_f32(Context& ctx, float* levels, size_t count, const double* largest,
                       uint32_t parts, uint32_t step) {
  const uint32_t blocks =
      static_cast<uint32_t>(std::min<size_t>((count + kAdrBlock - 1) / kAdrBlock, 2048));
  k_adr_settle<float><<<blocks, kAdrBlock, 0, ctx.stream>>>(levels, count, largest, parts,
                                                            ctx.adr.flags.data(), step, 0);
  check(hipGetLastError(), "launch k_adr_settle");
}

void adr_run(Context& ctx, float dt, uint32_t steps, double* ledger) {
  auto& a = ctx.adr;
  const auto& P = a.params;
  const float* xf = a.flow_field ? ctx.flow.faces.data() : a.xf.data();
  const float* yf = a.flow_field ? ctx.flow.faces.data() + ctx.flow.x_faces() : a.yf.data();
  const uint32_t init_flags[3] = {0u, 0xffffffffu, 0u};
  check(hipMemcpyAsync(a.flags.data(), init_flags, sizeof(init_flags), hipMemcpyHostToDevice,
                       ctx.stream),
        "clear flags");
  if (a.integration != MSIM_FORWARD_EULER || P.nz > 1) {
    // Implicit steps (FP32 levels, each step's solve judged on the host),
    // and every step on a grid of several layers.
    check(hipEventRecord(ctx.start, ctx.stream), "event");
    if (a.integration != MSIM_FORWARD_EULER) {
      implicit_run(ctx, dt, steps, xf, yf);
    } else {
      adr3_run(ctx, dt, steps, xf, yf, a.zf.data());
    }
    check(hipEventRecord(ctx.stop, ctx.stream), "event");
    check(hipEventSynchronize(ctx.stop), "event sync");
    float ms = 0.0f;
    check(hipEventElapsedTime(&ms, ctx.start, ctx.stop), "event time");
    a.seconds = ms * 1.0e-3;
    return;
  }
  if (a.precision == 64) a.ledger.reserve(static_cast<size_t>(steps) * P.signals * 4 + 1);
  check(hipEventRecord(ctx.start, ctx.stream), "event");
  switch (P.signals) {
    case 1: launch_steps<1>(ctx, dt, steps, xf, yf); break;
    case 2: launch_steps<2>(ctx, dt, steps, xf, yf); break;
    case 3: launch_steps<3>(ctx, dt, steps, xf, yf); break;
    case 4: launch_steps<4>(ctx, dt, steps, xf, yf); break;
    case 5: launch_steps<5>(ctx, dt, steps, xf, yf); break;
    case 6: launch_steps<6>(ctx, dt, steps, xf, yf); break;
    case 7: launch_steps<7>(ctx, dt, steps, xf, yf); break;
    default: launch_steps<8>(ctx, dt, steps, xf, yf); break;
  }
  check(hipEventRecord(ctx.stop, ctx.stream), "event");
  uint32_t flags[2] = {0, 0};
  check(hipMemcpyAsync(flags, a.flags.data(), sizeof(flags), hipMemcpyDeviceToHost, ctx.stream),
        "read flags");
  std::vector<double> rows;
  if (a.precision == 64 && steps > 0) {
    rows.resize(static_cast<size_t>(steps) * P.signals * 4);
    check(hipMemcpyAsync(rows.data(), a.ledger.data(), rows.size() * sizeof(double),
                         hipMemcpyDeviceToHost, ctx.stream),
          "read ledger");
  }
  check(hipStreamSynchronize(ctx.stream), "transport steps");
  float ms = 0.0f;
  check(hipEventElapsedTime(&ms, ctx.start, ctx.stop), "event time");
  a.seconds = ms * 1.0e-3;
  if (flags[0] != 0) {
    // Levels stay those before the failed step: step k read buffer (k even ?
    // the starting one : the other).
    const uint32_t failed = flags[1];
    a.current = static_cast<int>((a.current ^ (steps & 1u)) ^ (failed & 1u));
    // The steps before it stand: their ledger rows carry the mass on, and go
    // to the caller.
    if (!rows.empty()) {
      const uint32_t kept = std::min(failed, steps);
      for (uint32_t k = 0; k < kept; ++k) {
        for (uint32_t s = 0; s < P.signals; ++s) {
          double* row = rows.data() + (static_cast<size_t>(k) * P.signals + s) * 4;
          row[0] = a.host_mass[s];
          a.host_mass[s] = row[1];
        }
      }
      if (ledger != nullptr && kept > 0) {
        std::memcpy(ledger, rows.data(),
                    static_cast<size_t>(kept) * P.signals * 4 * sizeof(double));
      }
    }
    if ((flags[0] & kFlagNegative) != 0) {
      throw Error(MSIM_DOMAIN_ERROR,
                  "signal grid update produced a non-finite or negative concentration (step " +
                      std::to_string(failed) + ")");
    }
    // The settle refused the step (accept_step, signals.cpp:1003-1011).
    throw Error(MSIM_INVALID_ARGUMENT, "signal grid levels must be finite and non-negative (step " +
                                           std::to_string(failed) + ")");
  }
  if (!rows.empty()) {
    // Mass before each step: the mass after the previous one.
    for (uint32_t k = 0; k < steps; ++k) {
      for (uint32_t s = 0; s < P.signals; ++s) {
        double* row = rows.data() + (static_cast<size_t>(k) * P.signals + s) * 4;
        row[0] = a.host_mass[s];
        a.host_mass[s] = row[1];
      }
    }
    if (ledger != nullptr) std::memcpy(ledger, rows.data(), rows.size() * sizeof(double));
  }
}

double adr_refresh_outflow(Context& ctx) {
  auto& a = ctx.adr;
  const auto& P = a.params;
  if (P.has_field == 0) return 0.0;
  const float* xf = a.flow_field ? ctx.flow.faces.data() : a.xf.data();
  const float* yf = a.flow_field ? ctx.flow.faces.data() + ctx.flow.x_faces() : a.yf.data();
  const uint8_t* levels = a.current == 0 ? a.levels_a.data() : a.levels_b.data();
  const size_t n = a.sites();
  const uint32_t blocks = std::min<uint32_t>(site_blocks(n), 2048);
  // The survey's mass goes to survey_mass only; the ledger's running mass
  // (host_mass) is left to the steps' own rows.
  if (P.nz > 1) {
    adr3_survey(ctx, xf, yf, a.zf.data(), reinterpret_cast<const float*>(levels),
                a.state.data(), a.partials.data(), survey_mass(a));
  } else if (a.precision == 64) {
    k_adr_survey<double><<<blocks, kAdrBlock, 0, ctx.stream>>>(
        P, a.solid.data(), xf, yf, reinterpret_cast<const double*>(levels), a.partials.data(),
        a.state.data(), survey_mass(a));
  } else {
    k_adr_survey<float><<<blocks, kAdrBlock, 0, ctx.stream>>>(
        P, a.solid.data(), xf, yf, reinterpret_cast<const float*>(levels), a.partials.data(),
        a.state.data(), survey_mass(a));
  }
  check(hipGetLastError(), "launch k_adr_survey");
  CgState host{};
  check(hipMemcpyAsync(&host, a.state.data(), sizeof(CgState), hipMemcpyDeviceToHost, ctx.stream),
        "read survey");
  check(hipStreamSynchronize(ctx.stream), "survey");
  a.greatest_outflow = host.peak;
  return host.peak;
}

void adr_download(Context& ctx, void* levels) {
  auto& a = ctx.adr;
  const size_t bytes =
      a.params.signals * a.sites() * (a.precision == 64 ? sizeof(double) : sizeof(float));
  const uint8_t* src = a.current == 0 ? a.levels_a.data() : a.levels_b.data();
  download(ctx, levels, src, bytes, "download levels");
}

// ---------------------------------------------------------------------------
// The allocation-free step (msim_hip_advance_signal_grid_static)
// ---------------------------------------------------------------------------
// Everything one FP32 forward-Euler step needs on the device besides the
// caller's host arrays lives in one file-scope array: the staged mask, faces,
// occupancy and reaction rates, both level buffers, the ledger and survey
// partials, the flags and the survey's state. Each device holds its own copy
// of the array for the life of the process; host code reaches it only through
// the address hipGetSymbolAddress gives on that device (the array's name is a
// host-side stand-in, not a device address).

namespace {

constexpr size_t kStaticScratchBytes = size_t(64) << 20;
constexpr int kStaticDevices = 64;

static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

void* g_scratch[kStaticDevices] = {};
std::mutex g_scratch_lock[kStaticDevices];

// The scratch holds 49 doubles for each of these blocks: strips of 62, 126 or
// 254 columns (60, 124 or 252 under van Leer; whichever takes the fewest threads)
// by 16 x-rows, or fewer down to 4 for 2048 blocks. A formula of its own, so
// that the grids that fit the scratch stay the same whatever shape a step is
// launched in (of which it needs one double a block).
uint32_t static_blocks(const AdrParams& P) {
  uint64_t best = ~0ull, strips = 1;
  for (uint32_t threads : {256u, 128u, 64u}) {
    const uint64_t width = threads - (P.limited != 0 ? 4 : 2);
    const uint64_t count = (P.ny + width - 1) / width;
    if (count * threads < best) {
      best = count * threads;
      strips = count;
    }
  }
  uint32_t rows = 16;
  while (rows > 4 && strips * ((P.nx + rows - 1) / rows) < 2048) rows /= 2;
  return std::max(static_cast<uint32_t>(strips * ((P.nx + rows - 1) / rows)), 3u * kMaxSignals);
}

// Carves 256-byte aligned regions out of the scratch array, in order.
struct ScratchLayout {
  size_t used = 0;
  size_t take(size_t bytes) {
    const size_t at = used;
    used += (bytes + 255) & ~size_t(255);
    return at;
  }
};

__global__ void k_fill_bytes(uint8_t* __restrict__ out, size_t count, uint8_t value) {
  for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < count;
       i += static_cast<size_t>(gridDim.x) * blockDim.x) {
    out[i] = value;
  }
}

template <int S>
void launch_static_step(hipStream_t stream, const AdrView& v, const AdrShape& sh, const float* xf,
                        const float* yf, const uint8_t* src, uint8_t* dst, float dt,
                        LedgerParts L, double* largest) {
  if (v.P->limited != 0) {
    launch_typed<float, S, true>(stream, v, sh, xf, yf, src, dst, dt, 0, L, largest);
  } else {
    launch_typed<float, S, false>(stream, v, sh, xf, yf, src, dst, dt, 0, L, largest);
  }
}

}  // namespace

size_t static_scratch_bytes() { return kStaticScratchBytes; }

void bind_static_scratch(int device) {
  if (device < 0 || device >= kStaticDevices) return;
  std::lock_guard<std::mutex> hold(g_scratch_lock[device]);
  if (g_scratch[device] != nullptr) return;
  void* ptr = nullptr;
  check(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
  g_scratch[device] = ptr;
}

void adr_step_static(Context& ctx, const msim_signal_grid& grid, float dt, float* levels) {
  if (ctx.device < 0 || ctx.device >= kStaticDevices || g_scratch[ctx.device] == nullptr) {
    throw Error(MSIM_DEVICE_ERROR, "the static scratch of this device is not set up");
  }
  if (grid.integration != MSIM_FORWARD_EULER) {
    throw Error(MSIM_UNSUPPORTED, "the allocation-free transport step takes forward Euler only");
  }
  if (grid.patches != nullptr && grid.patch_count > 0) {
    throw Error(MSIM_UNSUPPORTED,
                "the allocation-free transport step takes no boundary patches");
  }
  if (grid.grid.nz != 1) {
    throw Error(MSIM_UNSUPPORTED, "the allocation-free transport step takes a grid of one layer");
  }
  AdrParams P = transport_params(grid);
  const uint32_t S = P.signals;
  const size_t n = static_cast<size_t>(P.nx) * P.ny;
  const AdrShape sh = adr_shape(P.nx, P.ny, P.limited != 0, 32);
  const uint32_t survey_blocks = std::min<uint32_t>(site_blocks(n), 2048);
  ScratchLayout at;
  const size_t o_state = at.take(sizeof(CgState));
  const size_t o_flags = at.take(3 * sizeof(uint32_t));
  const size_t o_mass = at.take(kMaxSignals * sizeof(double));
  const size_t o_parts = at.take(
      std::max({static_cast<size_t>(3 * kMaxSignals * 2 + 1) * static_blocks(P),
                static_cast<size_t>(kMaxSignals + 1) * survey_blocks,
                static_cast<size_t>(sh.blocks)}) *
      sizeof(double));
  const size_t o_solid = at.take(n);
  const size_t nxf = static_cast<size_t>(P.nx + 1) * P.ny, nyf = static_cast<size_t>(P.nx) * (P.ny + 1);
  const size_t o_xf = P.has_field != 0 ? at.take(nxf * sizeof(float)) : 0;
  const size_t o_yf = P.has_field != 0 ? at.take(nyf * sizeof(float)) : 0;
  const size_t o_phi = P.has_monod != 0 ? at.take(n * sizeof(float)) : 0;
  const size_t o_loss = P.has_affine != 0 ? at.take(S * n * sizeof(float)) : 0;
  const size_t o_source = P.has_affine != 0 ? at.take(S * n * sizeof(float)) : 0;
  const size_t o_a = at.take(S * n * sizeof(float));
  const size_t o_b = at.take(S * n * sizeof(float));
  if (at.used > kStaticScratchBytes) {
    throw Error(MSIM_INVALID_ARGUMENT,
                "the allocation-free transport step needs " + std::to_string(at.used) +
                    " bytes of device scratch for this grid; its limit is " +
                    std::to_string(kStaticScratchBytes) + " bytes");
  }
  // One call at a time per device in this process: every call shares the
  // device's array.
  std::lock_guard<std::mutex> hold(g_scratch_lock[ctx.device]);
  uint8_t* base_ptr = static_cast<uint8_t*>(g_scratch[ctx.device]);
  auto* state = reinterpret_cast<CgState*>(base_ptr + o_state);
  auto* flags = reinterpret_cast<uint32_t*>(base_ptr + o_flags);
  auto* mass = reinterpret_cast<double*>(base_ptr + o_mass);
  auto* parts = reinterpret_cast<double*>(base_ptr + o_parts);
  uint8_t* solid = base_ptr + o_solid;
  float* xf = P.has_field != 0 ? reinterpret_cast<float*>(base_ptr + o_xf) : nullptr;
  float* yf = P.has_field != 0 ? reinterpret_cast<float*>(base_ptr + o_yf) : nullptr;
  float* phi = P.has_monod != 0 ? reinterpret_cast<float*>(base_ptr + o_phi) : nullptr;
  float* loss = P.has_affine != 0 ? reinterpret_cast<float*>(base_ptr + o_loss) : nullptr;
  float* source = P.has_affine != 0 ? reinterpret_cast<float*>(base_ptr + o_source) : nullptr;
  uint8_t* lv_a = base_ptr + o_a;
  uint8_t* lv_b = base_ptr + o_b;
  hipStream_t stream = ctx.stream;
  // The array keeps the last call's contents: the state (with its tickets),
  // the flags and every staged array are written afresh.
  const CgState zero_state{};
  const uint32_t init_flags[3] = {0u, 0xffffffffu, 0u};
  check(hipMemcpyAsync(state, &zero_state, sizeof(CgState), hipMemcpyHostToDevice, stream),
        "clear state");
  check(hipMemcpyAsync(flags, init_flags, sizeof(init_flags), hipMemcpyHostToDevice, stream),
        "clear flags");
  if (grid.grid.obstacles != nullptr) {
    check(hipMemcpyAsync(solid, grid.grid.obstacles, n, hipMemcpyHostToDevice, stream),
          "upload mask");
  } else {
    k_fill_bytes<<<std::min<uint32_t>(site_blocks(n), 1024), kAdrBlock, 0, stream>>>(solid, n, 0);
    check(hipGetLastError(), "launch k_fill_bytes");
  }
  if (P.has_field != 0) {
    check(hipMemcpyAsync(xf, grid.x_faces, nxf * sizeof(float), hipMemcpyHostToDevice, stream),
          "upload x faces");
    check(hipMemcpyAsync(yf, grid.y_faces, nyf * sizeof(float), hipMemcpyHostToDevice, stream),
          "upload y faces");
  }
  if (P.has_monod != 0) {
    check(hipMemcpyAsync(phi, grid.phi, n * sizeof(float), hipMemcpyHostToDevice, stream),
          "upload phi");
  }
  if (P.has_affine != 0) {
    check(hipMemcpyAsync(loss, grid.loss_rates, S * n * sizeof(float), hipMemcpyHostToDevice,
                         stream),
          "upload loss");
    check(hipMemcpyAsync(source, grid.source_rates, S * n * sizeof(float), hipMemcpyHostToDevice,
                         stream),
          "upload source");
  }
  check(hipMemcpyAsync(lv_a, levels, S * n * sizeof(float), hipMemcpyHostToDevice, stream),
        "upload levels");
  // The greatest outflow for the explicit bound (transport_cache).
  k_adr_survey<float><<<survey_blocks, kAdrBlock, 0, stream>>>(
      P, solid, xf, yf, reinterpret_cast<const float*>(lv_a), parts, state, mass);
  check(hipGetLastError(), "launch k_adr_survey");
  CgState host{};
  check(hipMemcpyAsync(&host, state, sizeof(CgState), hipMemcpyDeviceToHost, stream),
        "read survey");
  check(hipStreamSynchronize(stream), "survey");
  double max_loss[kMaxSignals] = {};
  max_losses(grid, max_loss);
  validate_explicit_bound(P, MSIM_FORWARD_EULER, P.has_field != 0 ? host.peak : 0.0, max_loss,
                          dt);
  if (dt == 0.0f) return;
  const AdrView v{&P, solid, phi, source, loss, flags};
  // FP32 levels keep no ledger: the block maxima are all the step leaves.
  LedgerParts L{nullptr, nullptr, sh.blocks};
  double* largest = parts;
  switch (S) {
    case 1: launch_static_step<1>(stream, v, sh, xf, yf, lv_a, lv_b, dt, L, largest); break;
    case 2: launch_static_step<2>(stream, v, sh, xf, yf, lv_a, lv_b, dt, L, largest); break;
    case 3: launch_static_step<3>(stream, v, sh, xf, yf, lv_a, lv_b, dt, L, largest); break;
    case 4: launch_static_step<4>(stream, v, sh, xf, yf, lv_a, lv_b, dt, L, largest); break;
    case 5: launch_static_step<5>(stream, v, sh, xf, yf, lv_a, lv_b, dt, L, largest); break;
    case 6: launch_static_step<6>(stream, v, sh, xf, yf, lv_a, lv_b, dt, L, largest); break;
    case 7: launch_static_step<7>(stream, v, sh, xf, yf, lv_a, lv_b, dt, L, largest); break;
    default: launch_static_step<8>(stream, v, sh, xf, yf, lv_a, lv_b, dt, L, largest); break;
  }
  check(hipGetLastError(), "launch transport step");
  uint32_t result[2] = {0, 0};
  check(hipMemcpyAsync(result, flags, sizeof(result), hipMemcpyDeviceToHost, stream),
        "read flags");
  check(hipStreamSynchronize(stream), "transport step");
  if ((result[0] & kFlagNegative) != 0) {
    throw Error(MSIM_DOMAIN_ERROR,
                "signal grid update produced a non-finite or negative concentration (step 0)");
  }
  if (result[0] != 0) {
    throw Error(MSIM_INVALID_ARGUMENT, "signal grid levels must be finite and non-negative (step 0)");
  }
  check(hipMemcpyAsync(levels, lv_b, S * n * sizeof(float), hipMemcpyDeviceToHost, stream),
        "download levels");
  check(hipStreamSynchronize(stream), "download levels");
}

}  // namespace msim
