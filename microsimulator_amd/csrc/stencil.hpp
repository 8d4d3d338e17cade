// Device helpers shared by the pressure-solve kernels: the harmonic mean of
// the assembly, the marching-tile geometry, and the per-block partial sums of
// the Krylov kernels with the fixed-order sum every block re-computes.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.hpp"
#include "internal.hpp"

namespace msim {

constexpr int kStream = 256;  // threads per block of the streaming kernels

// cpp/core/flow_system.hpp:171-174.
__device__ __host__ inline float harmonic(float a, float b) {
  const float sum = a + b;
  return sum > 0.0f ? 2.0f * a * b / sum : 0.0f;
}

// Whether the exterior face `side` (0 x lower, 1 x upper, 2 y lower, 3 y
// upper) at in-plane index `along` is open, and the pressure held half a
// spacing outside it.
__device__ __forceinline__ bool open_edge(const FlowEdges& e, uint32_t side, uint32_t along,
                                          uint32_t nx, uint32_t ny, float& pressure) {
  if (e.open == nullptr) {
    pressure = (side & 1u) != 0 || e.held_zero != 0 ? 0.0f : 1.0f;
    return (side >> 1) == e.axis;
  }
  const uint32_t slot =
      along + (side == 0 ? 0u : side == 1 ? ny : side == 2 ? 2u * ny : 2u * ny + nx);
  pressure = e.held_zero != 0 ? 0.0f : e.pressure[slot];
  return e.open[slot] != 0;
}

// Assembly (flow_system.hpp:549-599) of site i: diagonal, right-hand side and
// boundary conductance in the reference's float order (x lower, x upper, y
// lower, y upper), and the lower-face conductances the operator uses. Each
// open exterior face adds 2m/h^2 toward the pressure held outside it.
__device__ inline void assemble_site(const float* __restrict__ cond, float* __restrict__ diag,
                                     float* __restrict__ rhs, float* __restrict__ bc,
                                     float* __restrict__ cxl, float* __restrict__ cyl, size_t i,
                                     uint32_t nx, uint32_t ny, float dx, float dy,
                                     const FlowEdges& edges) {
  const uint32_t x = static_cast<uint32_t>(i / ny);
  const uint32_t y = static_cast<uint32_t>(i % ny);
  const float m = cond[i];
  cxl[i] = x > 0 ? harmonic(m, cond[i - ny]) : 0.0f;
  cyl[i] = y > 0 ? harmonic(m, cond[i - 1]) : 0.0f;
  float d = 0.0f, r = 0.0f, b = 0.0f;
  if (m != 0.0f) {
    const float isx = 1.0f / (dx * dx);
    const float isy = 1.0f / (dy * dy);
    float held = 0.0f;
    auto open = [&](uint32_t side, uint32_t along, float is) {
      if (!open_edge(edges, side, along, nx, ny, held)) return;
      const float c = 2.0f * m * is;
      d += c;
      b += c;
      r += c * held;
    };
    if (x > 0) {
      d += harmonic(m, cond[i - ny]) * isx;
    } else {
      open(0, y, isx);
    }
    if (x + 1 < nx) {
      d += harmonic(m, cond[i + ny]) * isx;
    } else {
      open(1, y, isx);
    }
    if (y > 0) {
      d += harmonic(m, cond[i - 1]) * isy;
    } else {
      open(2, x, isy);
    }
    if (y + 1 < ny) {
      d += harmonic(m, cond[i + 1]) * isy;
    } else {
      open(3, x, isy);
    }
  }
  diag[i] = d;
  rhs[i] = r;
  bc[i] = b;
}

// Inverse diagonal of a level's operator at cell i.
__device__ inline float level_dinv(const float* __restrict__ wx, const float* __restrict__ wy,
                                   const float* __restrict__ bc, size_t i, uint32_t nx,
                                   uint32_t ny) {
  const uint32_t x = static_cast<uint32_t>(i / ny), y = static_cast<uint32_t>(i % ny);
  float d = bc[i] + wx[i] + wy[i];
  if (x + 1 < nx) d += wx[i + ny];
  if (y + 1 < ny) d += wy[i + 1];
  return d > 0.0f ? 1.0f / d : 0.0f;
}

// Galerkin coarse operator of 2x2 aggregation at coarse cell c, from the
// fine level's couplings and boundary terms (fnx x fny).
__device__ inline void coarsen_cell(const float* __restrict__ fwx, const float* __restrict__ fwy,
                                    const float* __restrict__ fbc, uint32_t fnx, uint32_t fny,
                                    float* __restrict__ wx, float* __restrict__ wy,
                                    float* __restrict__ bc, size_t c, uint32_t nyc) {
  const uint32_t X = static_cast<uint32_t>(c / nyc), Y = static_cast<uint32_t>(c % nyc);
  const uint32_t fx = 2 * X, fy = 2 * Y;
  const bool x1 = fx + 1 < fnx, y1 = fy + 1 < fny;
  const size_t i = static_cast<size_t>(fx) * fny + fy;
  float cx = 0.0f, cy = 0.0f;
  if (X > 0) cx = fwx[i] + (y1 ? fwx[i + 1] : 0.0f);
  if (Y > 0) cy = fwy[i] + (x1 ? fwy[i + fny] : 0.0f);
  float b = fbc[i];
  if (y1) b += fbc[i + 1];
  if (x1) b += fbc[i + fny];
  if (x1 && y1) b += fbc[i + fny + 1];
  wx[c] = cx;
  wy[c] = cy;
  bc[c] = b;
}

struct Tile {
  uint32_t ty, x0, x1, y;
  bool valid, lo_halo, hi_halo;
  size_t ylo, yhi;
};

template <int TY>
__device__ inline Tile tile_of(uint32_t nx, uint32_t ny, uint32_t rows) {
  const uint32_t t = xcd_tile(blockIdx.x, gridDim.x);
  const uint32_t nty = (ny + TY - 1) / TY;
  Tile tile;
  tile.ty = t % nty;
  tile.x0 = (t / nty) * rows;
  tile.x1 = min(nx, tile.x0 + rows);
  tile.y = tile.ty * TY + threadIdx.x;
  tile.valid = tile.y < ny;
  // Thread 0 also carries the site below the tile, thread TY-1 the one above.
  tile.lo_halo = threadIdx.x == 0 && tile.ty > 0;
  tile.hi_halo = threadIdx.x == TY - 1 && tile.ty * TY + TY < ny;
  tile.ylo = tile.ty * TY - 1;
  tile.yhi = static_cast<size_t>(tile.ty) * TY + TY;
  return tile;
}

// Per-block partial sums of the Krylov kernels, two generations of each
// (indexed by iteration parity): p . A p from the operator kernel (p1 blocks),
// r . r and r . M^-1 r from the update kernel and the set-up (p2 blocks).
struct CgPartials {
  double* pq;
  double* rz;
  double* rr;
  uint32_t p1, p2;
};

// Sum of `count` partials in a fixed order, the same in every thread of every
// block that calls it: thread t adds t, t+NT, ... in order, then the block
// combines waves in order.
template <int NT>
__device__ inline double fixed_sum(const double* v, uint32_t count, double* lds, double* bcast) {
  double s = 0.0;
  for (uint32_t i = threadIdx.x; i < count; i += NT) s += v[i];
  s = block_sum<NT>(s, lds);
  if (threadIdx.x == 0) *bcast = s;
  __syncthreads();
  const double out = *bcast;
  __syncthreads();
  return out;
}

}  // namespace msim
