// Batched sweep: many independent depth-averaged devices of uneven sizes
// (a parameter sweep), each with its own geometry, mobility, occupancy,
// inlet pressure and solute diffusivity, advanced together. No counterpart
// in the reference, which runs one job per invocation
// (docs/architecture/0005-batch-execution.md:30); each instance follows the
// reference's single-grid algorithms:
//   pressure  -- the assembled operator (flow_system.hpp:522-695) solved by
//                FP32 conjugate-gradient corrections (cpp/cpu/cpu_flow.cpp:65-140; FP64
//                dot products) inside FP64 iterative refinement of an FP64
//                pressure, warm-started, to an FP64 true relative residual;
//   velocity  -- face velocities and lift (flow_system.hpp:711-736, 424-445)
//                for the Dirichlet inlet pressure, unscaled;
//   transport -- one FP32 forward-Euler step of one solute with Monod uptake,
//                every site in the single-grid kernel's float operations
//                (adr_site.hpp), with FP64 mass tallies.
//
// A step runs over work items (instance, block of rows) of a few thousand
// sites, spread over the whole chip, in one launch. Each item
// recomputes its rows' FP64 pressure residual (the step's flow check), writes
// the face velocities it owns, and advances its sites, so no item waits on
// another. Instances up to 256 columns wide take a marching kernel: one
// thread per column walks the item's rows, neighbours from registers and an
// LDS row, each array read once and each x face computed once; wider ones a
// general sweep. Per-item FP64 partials (residual, masses, uptake) are added
// per instance in a fixed order on the host. A run of steps is captured once
// into a HIP graph and replayed.
//
// The pressure solve takes one of two forms: one launch with one workgroup per
// instance (largest first), or launches in which every instance's iteration
// advances together over the whole chip. Each FP32 correction is conjugate
// gradient preconditioned by the instance's own multilevel cycle (2x2
// aggregation, V(1,1) damped Jacobi, the coarse correction weighted by 1.8, the
// coarsest level of <= 64 cells inverted densely): the cycle of the
// single-grid multilevel form. It is
// linear and symmetric positive definite, so plain CG applies.
//
// The launch shapes (sites per item; workgroup size and sweep row width of
// the general sweep) are chosen by timing each candidate on the uploaded
// batch: the autotuner.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <numeric>
#include <vector>

#include "adr_site.hpp"
#include "common.hpp"
#include "internal.hpp"
#include "stencil.hpp"

namespace msim {
namespace {

struct BatchDesc {
  uint32_t nx, ny;
  uint64_t site, xface, yface;  // first site / x face / y face of the instance
  float dx, dy, dz;
  float inlet;      // pressure at x = 0 (0 at x = nx)
  float diffusion;  // of the solute
  float reservoir;  // solute level beyond x = 0 (0 beyond x = nx)
};

struct BatchItem {
  uint32_t inst, x0, x1, pad;
};

// The multilevel hierarchy of one instance: level l has nx[l] x ny[l] cells
// at offset off[l] of the level arrays (level 0 at the instance's own first
// site); the coarsest level's dense inverse is coarse_n x coarse_n floats, transposed, at
// offset cinv of the inverse pool.
constexpr uint32_t kBatchLevels = 16;
constexpr uint32_t kBatchCoarse = 64;
struct BatchLevels {
  uint32_t count, coarse_n;
  uint64_t cinv;
  uint64_t off[kBatchLevels];
  uint32_t nx[kBatchLevels], ny[kBatchLevels];
};

struct BatchData {
  const BatchDesc* desc;
  const uint32_t* order;
  const uint8_t* solid;
  const float* cond;
  const float* cxl;
  const float* cyl;
  const float* bc;
  const float* rhs;
  const float* phi;
  double* x64;  // pressure
  float* x;     // FP32 correction of one refinement
  float* r;
  float* p;
  float* p2;  // the direction before or after p, by turns
  float* q;
  float* xf;
  float* yf;
  float* la;
  float* lb;
  uint32_t* iterations;  // [instance]: FP32 CG iterations of the last flow solve
  float* residual;       // [instance]: FP64 true relative residual after it
  double* bnorm2;        // [instance]: ||b||^2
  uint32_t* flags;       // [instance]: 1 CG breakdown, 2 not converged, 4 bad level
  float* z;              // preconditioned residual
  const BatchLevels* levels;
  const float* lwx;      // level couplings to the lower x / y cell (over h^2),
  const float* lwy;      // boundary term and inverse diagonal
  const float* lbc;
  const float* ldinv;
  float* lr;             // level residual and correction (coarse levels)
  float* le;
  const float* cinv;     // dense inverses of the coarsest levels, each transposed
};

struct BatchParams {
  float tolerance;
  uint32_t max_iterations;
  float vmax, monod_k;
};

// FP64 sums over the workgroup, broadcast to every thread.
template <int NT, int K>
__device__ inline void block_sums(double (&v)[K], double* lds) {
  __shared__ double s_out[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const double t = block_sum<NT>(v[k], lds);
    if (threadIdx.x == 0) s_out[k] = t;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = s_out[k];
  __syncthreads();
}

// b - A x in FP64 at site i, b = inlet * (the assembled Dirichlet-1 rhs).
__device__ inline double residual_f64(const double* __restrict__ x, const float* __restrict__ cxl,
                                      const float* __restrict__ cyl, const float* __restrict__ bc,
                                      const float* __restrict__ rhs, float inlet, uint32_t xx,
                                      uint32_t y, uint32_t nx, uint32_t ny, size_t i, double isx,
                                      double isy) {
  const double c = x[i];
  double a = static_cast<double>(bc[i]) * c;
  if (xx > 0) a += (static_cast<double>(cxl[i]) * isx) * (c - x[i - ny]);
  if (xx + 1 < nx) a += (static_cast<double>(cxl[i + ny]) * isx) * (c - x[i + ny]);
  if (y > 0) a += (static_cast<double>(cyl[i]) * isy) * (c - x[i - 1]);
  if (y + 1 < ny) a += (static_cast<double>(cyl[i + 1]) * isy) * (c - x[i + 1]);
  return static_cast<double>(inlet) * static_cast<double>(rhs[i]) - a;
}

// Face velocities (flow_system.hpp:711-736 with the lift of 424-445) from the
// FP64 pressure: x face fx (0..nx) of row y, y face fy (0..ny) of column x.
__device__ inline float face_x(const BatchDesc& I, const double* __restrict__ p,
                               const float* __restrict__ cond, const uint8_t* __restrict__ solid,
                               uint32_t fx, uint32_t y) {
  const uint32_t nx = I.nx, ny = I.ny;
  const bool has_lower = fx > 0, has_upper = fx < nx;
  const size_t upper = static_cast<size_t>(fx) * ny + y;
  const size_t lower = upper - ny;
  double value;
  if (has_lower && has_upper) {
    const float fm = harmonic(cond[lower], cond[upper]);
    value = -static_cast<double>(fm) * (p[upper] - p[lower]) / static_cast<double>(I.dx);
  } else {
    const size_t site = has_upper ? upper : lower;
    const float m = cond[site];
    float fc = 0.0f, fp = 0.0f;
    if (m != 0.0f) {
      fc = (has_upper ? 2.0f : -2.0f) * m / I.dx;
      fp = has_upper ? I.inlet : 0.0f;
    }
    value = static_cast<double>(fc) * (static_cast<double>(fp) - p[site]);
  }
  const float flux = static_cast<float>(value);
  if ((has_lower && solid[lower] != 0) || (has_upper && solid[upper] != 0)) return 0.0f;
  return flux / I.dz;
}

__device__ inline float face_y(const BatchDesc& I, const double* __restrict__ p,
                               const float* __restrict__ cond, const uint8_t* __restrict__ solid,
                               uint32_t x, uint32_t fy) {
  const uint32_t ny = I.ny;
  const bool has_lower = fy > 0, has_upper = fy < ny;
  const size_t upper = static_cast<size_t>(x) * ny + fy;
  const size_t lower = upper - 1;
  double value;
  if (has_lower && has_upper) {
    const float fm = harmonic(cond[lower], cond[upper]);
    value = -static_cast<double>(fm) * (p[upper] - p[lower]) / static_cast<double>(I.dy);
  } else {
    const size_t site = has_upper ? upper : lower;
    value = static_cast<double>(0.0f) * (static_cast<double>(0.0f) - p[site]);
  }
  const float flux = static_cast<float>(value);
  if ((has_lower && solid[lower] != 0) || (has_upper && solid[upper] != 0)) return 0.0f;
  return flux / I.dz;
}

// One level of an instance's hierarchy as the cycle sees it.
struct LevelRef {
  const float* wx;
  const float* wy;
  const float* bc;
  const float* dinv;
  float* r;
  float* e;
  uint32_t nx, ny;
};

__device__ inline LevelRef level_ref(const BatchData& D, const BatchLevels& V, uint32_t l,
                                     size_t site) {
  const size_t o = V.off[l];
  return LevelRef{D.lwx + o,
                  D.lwy + o,
                  D.lbc + o,
                  D.ldinv + o,
                  l == 0 ? D.r + site : D.lr + o,
                  l == 0 ? D.z + site : D.le + o,
                  V.nx[l],
                  V.ny[l]};
}

constexpr float kCycleOmega = 0.8f;
constexpr float kCycleCorrection = 1.8f;

// A workgroup's pass over the cells [lo, hi): each thread takes U of them, NT
// apart, and issues all their loads before it uses any, so a pass of few cells
// per thread is one memory latency and not U of them.
template <int NT, int U, class Load, class Use>
__device__ inline void sweep_cells(uint32_t lo, uint32_t hi, Load&& load, Use&& use) {
  for (uint32_t i0 = lo + threadIdx.x; i0 < hi; i0 += U * NT) {
    decltype(load(0u)) v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = i0 + static_cast<uint32_t>(u * NT);
      if (i < hi) v[u] = load(i);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = i0 + static_cast<uint32_t>(u * NT);
      if (i < hi) use(i, v[u]);
    }
  }
}

// The operator at a cell of a level: its couplings to the four neighbours and
// its boundary term. The lower couplings are zero on the first row and column
// (and the first column's are the last column's upper ones), so the neighbours
// are taken by index alone, clamped to the grid.
struct CellOp {
  float xl, xu, yl, yu, b;
  uint32_t ixl, ixu, iyl, iyu;
};

__device__ inline CellOp cell_op(const float* wx, const float* wy, const float* bc, uint32_t i,
                                 uint32_t cells, uint32_t ny) {
  CellOp o;
  o.ixl = i >= ny ? i - ny : i;
  o.ixu = i + ny < cells ? i + ny : i;
  o.iyl = i >= 1 ? i - 1 : i;
  o.iyu = i + 1 < cells ? i + 1 : i;
  o.xl = wx[i];
  o.xu = i + ny < cells ? wx[i + ny] : 0.0f;
  o.yl = wy[i];
  o.yu = i + 1 < cells ? wy[i + 1] : 0.0f;
  o.b = bc[i];
  return o;
}

__device__ inline float cell_apply(const CellOp& o, float c, float xl, float xu, float yl,
                                   float yu) {
  float a = o.b * c;
  a += o.xl * (c - xl);
  a += o.xu * (c - xu);
  a += o.yl * (c - yl);
  a += o.yu * (c - yu);
  return a;
}

// The cycle's passes over a range of a level's cells. The finest level's
// x = omega D^-1 r stands in x0 (the pass that leaves r leaves it too); a
// coarser level's (x0 null) is formed where it is read.
//
// Down: the residual of x, restricted to the cells [lo, hi) of the next level.
template <int NT>
__device__ inline void cycle_down(const LevelRef& F, const LevelRef& C, const float* x0,
                                  uint32_t lo, uint32_t hi) {
  const uint32_t fine = F.nx * F.ny;
  auto pre = [&](uint32_t j) { return x0 != nullptr ? x0[j] : kCycleOmega * F.dinv[j] * F.r[j]; };
  struct Quad {
    float r[4], c[4], n[4][4];
    CellOp o[4];
    uint32_t in;
  };
  sweep_cells<NT, 1>(
      lo, hi,
      [&](uint32_t c) {
        Quad q;
        const uint32_t X = c / C.ny, Y = c - X * C.ny;
        q.in = 0;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
          const uint32_t fx = 2 * X + (k >> 1), fy = 2 * Y + (k & 1);
          if (fx < F.nx && fy < F.ny) {
            const uint32_t i = fx * F.ny + fy;
            q.in |= 1u << k;
            q.o[k] = cell_op(F.wx, F.wy, F.bc, i, fine, F.ny);
            q.r[k] = F.r[i];
            q.c[k] = pre(i);
            q.n[k][0] = pre(q.o[k].ixl);
            q.n[k][1] = pre(q.o[k].ixu);
            q.n[k][2] = pre(q.o[k].iyl);
            q.n[k][3] = pre(q.o[k].iyu);
          }
        }
        return q;
      },
      [&](uint32_t c, const Quad& q) {
        float sum = 0.0f;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
          if ((q.in >> k) & 1u)
            sum += q.r[k] - cell_apply(q.o[k], q.c[k], q.n[k][0], q.n[k][1], q.n[k][2], q.n[k][3]);
        }
        C.r[c] = sum;
      });
}

// Up: x + 1.8 P e_c, post-smoothed, on the cells [lo, hi); their share of z.r
// joins rz.
template <int NT>
__device__ inline void cycle_up(const LevelRef& F, const LevelRef& C, const float* x0, uint32_t lo,
                                uint32_t hi, double& rz) {
  const uint32_t cells = F.nx * F.ny;
  struct Cell {
    CellOp o;
    float r, d, c, xl, xu, yl, yu;
  };
  sweep_cells<NT, 2>(
      lo, hi,
      [&](uint32_t i) {
        Cell v;
        const uint32_t x = i / F.ny, y = i - x * F.ny;
        // The cells over a clamped neighbour: its coupling is zero there.
        const uint32_t xl = (x > 0 ? x - 1 : 0) / 2, xu = min(x + 1, F.nx - 1) / 2;
        const uint32_t yl = (y > 0 ? y - 1 : 0) / 2, yu = min(y + 1, F.ny - 1) / 2;
        auto corrected = [&](uint32_t j, uint32_t X, uint32_t Y) {
          return (x0 != nullptr ? x0[j] : kCycleOmega * F.dinv[j] * F.r[j]) +
                 kCycleCorrection * C.e[X * C.ny + Y];
        };
        v.o = cell_op(F.wx, F.wy, F.bc, i, cells, F.ny);
        v.r = F.r[i];
        v.d = F.dinv[i];
        v.c = corrected(i, x / 2, y / 2);
        v.xl = corrected(v.o.ixl, xl, y / 2);
        v.xu = corrected(v.o.ixu, xu, y / 2);
        v.yl = corrected(v.o.iyl, x / 2, yl);
        v.yu = corrected(v.o.iyu, x / 2, yu);
        return v;
      },
      [&](uint32_t i, const Cell& v) {
        const float z =
            v.c + kCycleOmega * v.d * (v.r - cell_apply(v.o, v.c, v.xl, v.xu, v.yl, v.yu));
        F.e[i] = z;
        rz += static_cast<double>(z) * static_cast<double>(v.r);
      });
}

// The cycle from level `from` down to the coarsest level's dense inverse and
// back, by the whole workgroup: from level 0 it is z = M r and returns r.z
// (this thread's share of it).
template <int NT>
__device__ double batch_cycle(const BatchData& D, const BatchLevels& V, size_t site,
                              uint32_t from) {
  const uint32_t K = V.count - 1;
  const float* x0 = D.q + site;
  for (uint32_t l = from; l < K; ++l) {
    const LevelRef F = level_ref(D, V, l, site), C = level_ref(D, V, l + 1, site);
    cycle_down<NT>(F, C, l == 0 ? x0 : nullptr, 0, C.nx * C.ny);
    __syncthreads();
  }
  double rz = 0.0;
  {
    const LevelRef B = level_ref(D, V, K, site);
    // The inverse is stored transposed; each row's columns are split into
    // NT / n contiguous ranges, one thread each (the rows of a wave adjacent,
    // so a step reads the inverse coalesced), added in range order.
    static_assert(NT >= static_cast<int>(kBatchCoarse), "one thread per row at least");
    __shared__ float s_r[kBatchCoarse];
    __shared__ float s_part[NT];
    const uint32_t n = V.coarse_n;
    const float* inv = D.cinv + V.cinv;
    for (uint32_t j = threadIdx.x; j < n; j += NT) s_r[j] = B.r[j];
    __syncthreads();
    const uint32_t parts = NT / n;
    const uint32_t span = (n + parts - 1) / parts;
    if (threadIdx.x < parts * n) {
      const uint32_t row = threadIdx.x % n, part = threadIdx.x / n;
      const uint32_t j1 = min(n, part * span + span);
      float v = 0.0f;
      for (uint32_t j = part * span; j < j1; ++j) v += inv[static_cast<size_t>(j) * n + row] * s_r[j];
      s_part[part * n + row] = v;
    }
    __syncthreads();
    for (uint32_t row = threadIdx.x; row < n; row += NT) {
      float v = 0.0f;
      for (uint32_t part = 0; part < parts; ++part) v += s_part[part * n + row];
      B.e[row] = v;
      if (K == 0) rz += static_cast<double>(v) * static_cast<double>(s_r[row]);
    }
    __syncthreads();
  }
  for (uint32_t l = K; l-- > from;) {
    const LevelRef F = level_ref(D, V, l, site), C = level_ref(D, V, l + 1, site);
    rz = 0.0;
    cycle_up<NT>(F, C, l == 0 ? x0 : nullptr, 0, F.nx * F.ny, rz);
    __syncthreads();
  }
  return rz;
}

// What the setup writes of an instance.
struct BatchSetup {
  const uint8_t* solid;
  const float* mobility;
  float *cond, *diag, *rhs, *bc, *cxl, *cyl;
  float *lwx, *lwy, *lbc, *ldinv, *cinv;
};

// Every instance's system and hierarchy, one workgroup per instance (order[b],
// largest first): conductance, assembly, the level operators, and the dense
// inverse of the coarsest (<= 64 cells) by FP64 Cholesky in LDS, rows and
// columns of cells without a diagonal, or whose pivot vanishes (a fluid pocket
// with no open boundary), left zero. Two launches for each of some 2000 levels
// and a host factorisation per instance took 47 of the 72 ms of a 256-instance
// upload; this takes 1.0 ms.
template <int NT>
__global__ __launch_bounds__(NT) void k_batch_setup(const BatchDesc* __restrict__ desc,
                                                    const uint32_t* __restrict__ order,
                                                    const BatchLevels* __restrict__ levels,
                                                    BatchSetup D) {
  constexpr uint32_t kC = kBatchCoarse;
  __shared__ double s_l[kC * (kC + 1) / 2];  // Cholesky factor, rows packed
  __shared__ double s_col[kC][kC];           // inverse: row, column
  __shared__ double s_diag[kC];
  __shared__ uint32_t s_act[kC], s_m;
  __shared__ uint8_t s_dead[kC];
  const uint32_t inst = order[blockIdx.x];
  const BatchDesc I = desc[inst];
  const BatchLevels& V = levels[inst];
  const uint32_t t = threadIdx.x;
  const size_t o = I.site, sites = static_cast<size_t>(I.nx) * I.ny;
  float* cond = D.cond + o;
  for (size_t i = t; i < sites; i += NT)
    cond[i] = D.solid[o + i] != 0 ? 0.0f : I.dz * D.mobility[o + i];
  __syncthreads();
  const FlowEdges edges{};
  const float isx = 1.0f / (I.dx * I.dx), isy = 1.0f / (I.dy * I.dy);
  for (size_t i = t; i < sites; i += NT) {
    assemble_site(cond, D.diag + o, D.rhs + o, D.bc + o, D.cxl + o, D.cyl + o, i, I.nx, I.ny, I.dx,
                  I.dy, edges);
    D.lwx[o + i] = D.cxl[o + i] * isx;
    D.lwy[o + i] = D.cyl[o + i] * isy;
    D.lbc[o + i] = D.bc[o + i];
  }
  __syncthreads();
  for (uint32_t l = 0; l < V.count; ++l) {
    const size_t at = V.off[l], cells = static_cast<size_t>(V.nx[l]) * V.ny[l];
    if (l > 0) {
      const size_t f = V.off[l - 1];
      for (size_t c = t; c < cells; c += NT) {
        coarsen_cell(D.lwx + f, D.lwy + f, D.lbc + f, V.nx[l - 1], V.ny[l - 1], D.lwx + at,
                     D.lwy + at, D.lbc + at, c, V.ny[l]);
      }
      __syncthreads();
    }
    for (size_t i = t; i < cells; i += NT)
      D.ldinv[at + i] = level_dinv(D.lwx + at, D.lwy + at, D.lbc + at, i, V.nx[l], V.ny[l]);
    __syncthreads();
  }
  // The coarsest operator's inverse, in the order of operations of a plain
  // column-by-column factorisation.
  const uint32_t n = V.coarse_n, last = V.count - 1, ny = V.ny[last];
  const float* wx = D.lwx + V.off[last];
  const float* wy = D.lwy + V.off[last];
  const float* bc = D.lbc + V.off[last];
  float* inv = D.cinv + V.cinv;
  for (uint32_t i = t; i < n * n; i += NT) inv[i] = 0.0f;
  if (t < n) {
    double d = static_cast<double>(bc[t]);
    if (t >= ny) d += static_cast<double>(wx[t]);
    if (t % ny != 0) d += static_cast<double>(wy[t]);
    if ((t + 1) % ny != 0) d += static_cast<double>(wy[t + 1]);
    if (t + ny < n) d += static_cast<double>(wx[t + ny]);
    s_diag[t] = d;
  }
  __syncthreads();
  if (t == 0) {
    uint32_t m = 0;
    for (uint32_t i = 0; i < n; ++i) {
      if (s_diag[i] > 0.0) s_act[m++] = i;
    }
    s_m = m;
  }
  __syncthreads();
  const uint32_t m = s_m;
  double scale = 0.0;
  for (uint32_t i = 0; i < n; ++i) scale = fmax(scale, s_diag[i]);
  auto entry = [&](uint32_t i, uint32_t j) -> double {  // rows i >= j of the active cells
    const uint32_t a = s_act[i], b = s_act[j];
    if (a == b) return s_diag[a];
    double v = 0.0;
    if (a - b == ny) v -= static_cast<double>(wx[a]);
    if (a - b == 1 && a % ny != 0) v -= static_cast<double>(wy[a]);
    return v;
  };
  auto at = [](uint32_t i, uint32_t j) { return i * (i + 1) / 2 + j; };
  for (uint32_t j = 0; j < m; ++j) {
    double v = 0.0;
    if (t >= j && t < m) {
      v = entry(t, j);
      for (uint32_t k = 0; k < j; ++k) v -= s_l[at(t, k)] * s_l[at(j, k)];
    }
    if (t == j) {
      s_dead[j] = v <= 1e-12 * scale ? 1 : 0;
      s_l[at(j, j)] = s_dead[j] != 0 ? 0.0 : sqrt(v);
    }
    __syncthreads();
    if (t > j && t < m) s_l[at(t, j)] = s_dead[j] != 0 ? 0.0 : v / s_l[at(j, j)];
    __syncthreads();
  }
  if (t < m && s_dead[t] == 0) {
    for (uint32_t i = 0; i < m; ++i) {
      double v = i == t ? 1.0 : 0.0;
      for (uint32_t k = 0; k < i; ++k) v -= s_l[at(i, k)] * s_col[k][t];
      s_col[i][t] = s_dead[i] != 0 ? 0.0 : v / s_l[at(i, i)];
    }
    for (uint32_t i = m; i-- > 0;) {
      double v = s_col[i][t];
      for (uint32_t k = i + 1; k < m; ++k) v -= s_l[at(k, i)] * s_col[k][t];
      s_col[i][t] = s_dead[i] != 0 ? 0.0 : v / s_l[at(i, i)];
    }
    // Stored transposed: entry (row, j) at j * n + row.
    for (uint32_t i = 0; i < m; ++i)
      inv[static_cast<size_t>(s_act[t]) * n + s_act[i]] = static_cast<float>(s_col[i][t]);
  }
}

// The pressure solve's passes over a range of an instance's sites, and what
// decides between them. A solve is FP64 refinement around FP32 corrections by
// conjugate gradient with the instance's multilevel cycle.
constexpr uint32_t kRefinements = 16;
constexpr double kInner = 1.0e-4;  // relative tolerance of each FP32 correction

// An instance's vectors.
struct FlowRef {
  const float *cxl, *cyl, *bc, *rhs, *wx, *wy, *dinv;
  double* x64;
  float *x, *r, *q, *z;
  float inlet;
  uint32_t nx, ny, sites;
  double isx, isy;
};

__device__ inline FlowRef flow_ref(const BatchData& D, const BatchDesc& I) {
  const size_t o = I.site;
  // The finest level's couplings (over the spacing squared), boundary term and
  // inverse diagonal are the operator's own.
  return FlowRef{D.cxl + o,  D.cyl + o, D.bc + o, D.rhs + o, D.lwx + o,
                 D.lwy + o,  D.ldinv + o, D.x64 + o, D.x + o, D.r + o,
                 D.q + o,    D.z + o,   I.inlet,  I.nx,      I.ny,
                 I.nx * I.ny, 1.0 / (static_cast<double>(I.dx) * I.dx),
                 1.0 / (static_cast<double>(I.dy) * I.dy)};
}

// FP64 true residual; its FP32 copy starts the correction x = 0, with the
// cycle's first sweep beside it. s[0], s[1]: r.r (FP64) and b.b.
template <int NT>
__device__ inline void flow_residual(const FlowRef& A, uint32_t lo, uint32_t hi, double (&s)[2]) {
  struct Cell {
    double res, b;
    float d;
  };
  sweep_cells<NT, 2>(
      lo, hi,
      [&](uint32_t i) {
        const uint32_t x = i / A.ny, y = i - x * A.ny;
        return Cell{residual_f64(A.x64, A.cxl, A.cyl, A.bc, A.rhs, A.inlet, x, y, A.nx, A.ny, i,
                                 A.isx, A.isy),
                    static_cast<double>(A.inlet) * static_cast<double>(A.rhs[i]), A.dinv[i]};
      },
      [&](uint32_t i, const Cell& v) {
        const float ri = static_cast<float>(v.res);
        A.r[i] = ri;
        A.q[i] = kCycleOmega * v.d * ri;
        A.x[i] = 0.0f;
        s[0] += v.res * v.res;
        s[1] += v.b * v.b;
      });
}

// p = z + beta p (beta = 0 and no old p at the first), q = A p; p.q joins pq.
// Neighbours' new directions are formed where they are read, so the old and
// the new direction are two vectors.
template <int NT, int U, bool kFirst>
__device__ inline void flow_direction(const FlowRef& A, const float* p, float* pn, float beta,
                                      uint32_t lo, uint32_t hi, double& pq) {
  struct Cell {
    CellOp o;
    float c, xl, xu, yl, yu;
  };
  auto at = [&](uint32_t j) { return kFirst ? A.z[j] : A.z[j] + beta * p[j]; };
  sweep_cells<NT, U>(
      lo, hi,
      [&](uint32_t i) {
        Cell v;
        v.o = cell_op(A.wx, A.wy, A.bc, i, A.sites, A.ny);
        v.c = at(i);
        v.xl = at(v.o.ixl);
        v.xu = at(v.o.ixu);
        v.yl = at(v.o.iyl);
        v.yu = at(v.o.iyu);
        return v;
      },
      [&](uint32_t i, const Cell& v) {
        const float qi = cell_apply(v.o, v.c, v.xl, v.xu, v.yl, v.yu);
        pn[i] = v.c;
        A.q[i] = qi;
        pq += static_cast<double>(v.c) * static_cast<double>(qi);
      });
}

// x += alpha p, r -= alpha q, the cycle's first sweep; r.r joins rr.
template <int NT>
__device__ inline void flow_update(const FlowRef& A, const float* p, float alpha, uint32_t lo,
                                   uint32_t hi, double& rr) {
  struct Cell {
    float x, p, r, q, d;
  };
  sweep_cells<NT, 4>(
      lo, hi, [&](uint32_t i) { return Cell{A.x[i], p[i], A.r[i], A.q[i], A.dinv[i]}; },
      [&](uint32_t i, const Cell& v) {
        A.x[i] = v.x + alpha * v.p;
        const float ri = v.r - alpha * v.q;
        A.r[i] = ri;
        A.q[i] = kCycleOmega * v.d * ri;
        rr += static_cast<double>(ri) * static_cast<double>(ri);
      });
}

template <int NT>
__device__ inline void flow_correct(const FlowRef& A, uint32_t lo, uint32_t hi) {
  struct Cell {
    double x;
    float e;
  };
  sweep_cells<NT, 4>(
      lo, hi, [&](uint32_t i) { return Cell{A.x64[i], A.x[i]}; },
      [&](uint32_t i, const Cell& v) { A.x64[i] = v.x + static_cast<double>(v.e); });
}

// The face velocities of the sites [lo, hi): their lower faces, and the last
// row's and column's upper ones.
template <int NT>
__device__ inline void flow_faces(const BatchData& D, const BatchDesc& I, uint32_t lo,
                                  uint32_t hi) {
  const size_t o = I.site;
  const double* x64 = D.x64 + o;
  const float* cond = D.cond + o;
  const uint8_t* solid = D.solid + o;
  float* xf = D.xf + I.xface;
  float* yf = D.yf + I.yface;
  for (uint32_t i = lo + threadIdx.x; i < hi; i += NT) {
    const uint32_t x = i / I.ny, y = i - x * I.ny;
    xf[i] = face_x(I, x64, cond, solid, x, y);
    if (x + 1 == I.nx) xf[i + I.ny] = face_x(I, x64, cond, solid, x + 1, y);
    yf[i + x] = face_y(I, x64, cond, solid, x, y);
    if (y + 1 == I.ny) yf[i + x + 1] = face_y(I, x64, cond, solid, x, y + 1);
  }
}

__device__ inline bool flow_breaks(double product) {
  return !(product > 0.0) || !isfinite(product);
}

__device__ inline double flow_threshold(const BatchParams& P, double bb) {
  const double bound = static_cast<double>(P.tolerance) * sqrt(bb);
  return bound * bound;
}

__device__ inline void flow_result(const BatchData& D, uint32_t inst, uint32_t it, double rr64,
                                   double bb, bool failed, bool short_of) {
  D.iterations[inst] = it;
  D.residual[inst] = bb > 0.0 ? static_cast<float>(sqrt(rr64 / bb)) : 0.0f;
  D.bnorm2[inst] = bb;
  if (failed) D.flags[inst] |= 1u;
  if (short_of && !failed) D.flags[inst] |= 2u;
}

// One workgroup per instance (order[b]) solves it alone: one launch, barriers
// in place of launches. A compute unit moves about 20 GB/s of a 512x256
// instance (its 6 MB are past its L2's share), so this is the form of small
// instances, and of batches that keep every unit busy (solve_alone).
template <int NT>
__global__ __launch_bounds__(NT) void k_batch_flow(BatchData D, BatchParams P) {
  __shared__ double s_red[NT / kWave];
  const uint32_t inst = D.order[blockIdx.x];
  const BatchDesc I = D.desc[inst];
  const BatchLevels& V = D.levels[inst];
  const FlowRef A = flow_ref(D, I);
  const uint32_t n = A.sites;
  uint32_t it = 0;
  bool failed = false;
  double rr64 = 0.0, bb = 0.0, threshold = 0.0;
  for (uint32_t ref = 0;; ++ref) {
    double s2[2] = {0.0, 0.0};
    flow_residual<NT>(A, 0, n, s2);
    block_sums<NT, 2>(s2, s_red);
    rr64 = s2[0];
    bb = s2[1];
    threshold = flow_threshold(P, bb);
    if (rr64 <= threshold || ref == kRefinements || it >= P.max_iterations) break;
    double rr = rr64, rz_old = 0.0;
    const double inner = kInner * kInner * rr64;
    // The first is taken also where the residual is not finite: its product
    // then is not either, and the instance is flagged.
    for (uint32_t k = 0; (k == 0 || rr > inner) && it < P.max_iterations; ++k, ++it) {
      float* p = (k & 1u) != 0 ? D.p2 + I.site : D.p + I.site;
      float* pn = (k & 1u) != 0 ? D.p + I.site : D.p2 + I.site;
      double rz[1] = {batch_cycle<NT>(D, V, I.site, 0)};
      block_sums<NT, 1>(rz, s_red);
      failed = flow_breaks(rz[0]);
      if (failed) break;
      double pq[1] = {0.0};
      if (k == 0) {
        flow_direction<NT, 2, true>(A, p, pn, 0.0f, 0, n, pq[0]);
      } else {
        flow_direction<NT, 2, false>(A, p, pn, static_cast<float>(rz[0] / rz_old), 0, n, pq[0]);
      }
      block_sums<NT, 1>(pq, s_red);
      failed = flow_breaks(pq[0]);
      if (failed) break;
      rz_old = rz[0];
      double s[1] = {0.0};
      flow_update<NT>(A, pn, static_cast<float>(rz[0] / pq[0]), 0, n, s[0]);
      block_sums<NT, 1>(s, s_red);
      rr = s[0];
    }
    if (failed) break;
    flow_correct<NT>(A, 0, n);
    __syncthreads();
  }
  if (threadIdx.x == 0) flow_result(D, inst, it, rr64, bb, failed, rr64 > threshold);
  flow_faces<NT>(D, I, 0, n);
}

// The same solve over the whole chip: every instance's iteration advances
// together, each pass one launch over tiles of all instances,
//   down (finest levels) - tail (one workgroup per instance: its levels of at
//   most kTailCells, and the decision of what comes next) - up - direction -
//   update,
// and an instance whose correction is done adds it and takes its FP64 residual
// in the up and direction launches of the same body. Each tile leaves its share
// of a product; whoever needs the product adds the instance's shares in tile
// order. Nothing waits inside a launch, and the host looks at the number of
// finished instances a few bodies behind.
enum FlowPhase : uint32_t { kFlowCorrect, kFlowIterate, kFlowDone };

struct FlowState {
  double rz, rr64, bb, inner;
  uint32_t phase, first, it, ref;
};

// A range of an instance's cells of one level, and the instance's tiles of the
// finest level.
struct FlowTile {
  uint32_t inst, lo, hi, slot;
};
struct FlowSpan {
  uint32_t first, count, tail, pad;  // tail: the level the tail starts at
};

struct FlowWork {
  BatchData D;
  BatchParams P;
  const FlowSpan* span;
  FlowState* state;
  double* share;  // [3][tiles]: r.z | p.q, FP64 r.r | r.r, b.b
  uint32_t tiles;
  uint32_t* done;
};

constexpr int kFlowTileThreads = 256;
constexpr uint32_t kFlowTile = 1024;  // sites of a tile (512: 20.6 ms, 2048: 18.6)

// The instance's shares of product k in tile order, the same in every wave.
__device__ inline double flow_sum(const FlowWork& W, const FlowSpan& s, uint32_t k) {
  const double* at = W.share + static_cast<size_t>(k) * W.tiles + s.first;
  double v = 0.0;
  for (uint32_t j = threadIdx.x % kWave; j < s.count; j += kWave) v += at[j];
  return wave_sum(v);
}

__device__ inline void flow_share(const FlowWork& W, uint32_t slot, uint32_t k, double v,
                                  double* lds) {
  const double t = block_sum<kFlowTileThreads>(v, lds);
  if (threadIdx.x == 0) W.share[static_cast<size_t>(k) * W.tiles + slot] = t;
}

// What follows the last body: the state after it, from its shares.
__device__ inline FlowState flow_next(const FlowWork& W, const FlowSpan& s, FlowState S,
                                      bool& failed) {
  failed = false;
  S.first = 0;
  if (S.phase == kFlowIterate) {
    const double rz = flow_sum(W, s, 0), pq = flow_sum(W, s, 1), rr = flow_sum(W, s, 2);
    failed = flow_breaks(rz) || flow_breaks(pq);
    S.rz = rz;
    if (failed) {
      S.phase = kFlowDone;
    } else {
      ++S.it;
      if (!(rr > S.inner) || S.it >= W.P.max_iterations) S.phase = kFlowCorrect;
    }
  } else if (S.phase == kFlowCorrect) {
    S.rr64 = flow_sum(W, s, 1);
    S.bb = flow_sum(W, s, 2);
    if (S.rr64 <= flow_threshold(W.P, S.bb) || S.ref == kRefinements ||
        S.it >= W.P.max_iterations) {
      S.phase = kFlowDone;
    } else {
      S.phase = kFlowIterate;
      S.first = 1;
      S.inner = kInner * kInner * S.rr64;
      ++S.ref;
    }
  }
  return S;
}

__global__ __launch_bounds__(kFlowTileThreads) void k_flow_down(FlowWork W, const FlowTile* tiles,
                                                                uint32_t level) {
  const FlowTile t = tiles[blockIdx.x];
  const FlowState S = W.state[t.inst];
  if (S.phase == kFlowDone) return;
  bool failed;
  if (flow_next(W, W.span[t.inst], S, failed).phase != kFlowIterate) return;
  const BatchLevels& V = W.D.levels[t.inst];
  const size_t site = W.D.desc[t.inst].site;
  cycle_down<kFlowTileThreads>(level_ref(W.D, V, level, site), level_ref(W.D, V, level + 1, site),
                               level == 0 ? W.D.q + site : nullptr, t.lo, t.hi);
}

template <int NT>
__global__ __launch_bounds__(NT) void k_flow_tail(FlowWork W) {
  const uint32_t inst = W.D.order[blockIdx.x];
  const FlowState S = W.state[inst];
  if (S.phase == kFlowDone) return;
  const FlowSpan s = W.span[inst];
  bool failed;
  const FlowState next = flow_next(W, s, S, failed);
  __syncthreads();
  if (threadIdx.x == 0) {
    W.state[inst] = next;
    if (next.phase == kFlowDone) {
      flow_result(W.D, inst, next.it, next.rr64, next.bb, failed,
                  next.rr64 > flow_threshold(W.P, next.bb));
      atomicAdd(W.done, 1u);
    }
  }
  if (next.phase == kFlowIterate)
    batch_cycle<NT>(W.D, W.D.levels[inst], W.D.desc[inst].site, s.tail);
}

__global__ __launch_bounds__(kFlowTileThreads) void k_flow_up(FlowWork W, const FlowTile* tiles,
                                                              uint32_t level) {
  __shared__ double s_red[kFlowTileThreads / kWave];
  const FlowTile t = tiles[blockIdx.x];
  const FlowState S = W.state[t.inst];
  if (S.phase == kFlowDone) return;
  const BatchDesc I = W.D.desc[t.inst];
  if (S.phase == kFlowCorrect) {
    if (level == 0) flow_correct<kFlowTileThreads>(flow_ref(W.D, I), t.lo, t.hi);
    return;
  }
  const BatchLevels& V = W.D.levels[t.inst];
  double rz = 0.0;
  if (V.count > 1) {
    cycle_up<kFlowTileThreads>(level_ref(W.D, V, level, I.site),
                               level_ref(W.D, V, level + 1, I.site),
                               level == 0 ? W.D.q + I.site : nullptr, t.lo, t.hi, rz);
  } else {  // one level: the tail's dense inverse left z
    const FlowRef A = flow_ref(W.D, I);
    for (uint32_t i = t.lo + threadIdx.x; i < t.hi; i += kFlowTileThreads)
      rz += static_cast<double>(A.z[i]) * static_cast<double>(A.r[i]);
  }
  if (level == 0) flow_share(W, t.slot, 0, rz, s_red);
}

__global__ __launch_bounds__(kFlowTileThreads) void k_flow_direction(FlowWork W,
                                                                     const FlowTile* tiles) {
  __shared__ double s_red[kFlowTileThreads / kWave];
  const FlowTile t = tiles[blockIdx.x];
  const FlowState S = W.state[t.inst];
  if (S.phase == kFlowDone) return;
  const BatchDesc I = W.D.desc[t.inst];
  const FlowRef A = flow_ref(W.D, I);
  if (S.phase == kFlowCorrect) {
    double s[2] = {0.0, 0.0};
    flow_residual<kFlowTileThreads>(A, t.lo, t.hi, s);
    flow_share(W, t.slot, 1, s[0], s_red);
    flow_share(W, t.slot, 2, s[1], s_red);
    return;
  }
  const double rz = flow_sum(W, W.span[t.inst], 0);
  if (flow_breaks(rz)) return;
  float* p = ((S.it & 1u) != 0 ? W.D.p2 : W.D.p) + I.site;
  float* pn = ((S.it & 1u) != 0 ? W.D.p : W.D.p2) + I.site;
  double pq = 0.0;
  if (S.first != 0) {
    flow_direction<kFlowTileThreads, 4, true>(A, p, pn, 0.0f, t.lo, t.hi, pq);
  } else {
    flow_direction<kFlowTileThreads, 4, false>(A, p, pn, static_cast<float>(rz / S.rz), t.lo,
                                               t.hi, pq);
  }
  flow_share(W, t.slot, 1, pq, s_red);
}

__global__ __launch_bounds__(kFlowTileThreads) void k_flow_update(FlowWork W,
                                                                  const FlowTile* tiles) {
  __shared__ double s_red[kFlowTileThreads / kWave];
  const FlowTile t = tiles[blockIdx.x];
  const FlowState S = W.state[t.inst];
  if (S.phase != kFlowIterate) return;
  const FlowSpan span = W.span[t.inst];
  const double rz = flow_sum(W, span, 0), pq = flow_sum(W, span, 1);
  if (flow_breaks(rz) || flow_breaks(pq)) return;
  const BatchDesc I = W.D.desc[t.inst];
  const float* pn = ((S.it & 1u) != 0 ? W.D.p : W.D.p2) + I.site;
  double rr = 0.0;
  flow_update<kFlowTileThreads>(flow_ref(W.D, I), pn, static_cast<float>(rz / pq), t.lo, t.hi, rr);
  flow_share(W, t.slot, 2, rr, s_red);
}

__global__ __launch_bounds__(kFlowTileThreads) void k_flow_faces(BatchData D,
                                                                 const FlowTile* tiles) {
  const FlowTile t = tiles[blockIdx.x];
  flow_faces<kFlowTileThreads>(D, D.desc[t.inst], t.lo, t.hi);
}

__global__ void k_flow_begin(FlowState* state, uint32_t count, uint32_t* done) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < count) state[k] = FlowState{0.0, 0.0, 0.0, 0.0, kFlowCorrect, 0, 0, 0};
  if (k == 0) *done = 0;
}

// One step for work item blockIdx.x (rows [x0, x1) of an instance): the FP64
// residual of the rows, their face velocities, and the forward-Euler step of
// their sites. partials[(step * items + item) * 4 + k]: residual r.r, mass
// before, mass after, uptake rate (FP64, before the volume factor).
template <int NT, int TY>
__global__ __launch_bounds__(NT) void k_batch_step(BatchData D, BatchParams P,
                                                   const BatchItem* __restrict__ items,
                                                   double* __restrict__ partials, uint32_t step,
                                                   float dt, uint32_t base, uint32_t total) {
  __shared__ double s_red[NT / kWave];
  constexpr int RX = NT / TY;
  const BatchItem item = items[base + blockIdx.x];
  const uint32_t inst = item.inst;
  const BatchDesc I = D.desc[inst];
  const uint32_t nx = I.nx, ny = I.ny;
  const size_t o = I.site;
  const uint8_t* solid = D.solid + o;
  const float* cond = D.cond + o;
  const double* x64 = D.x64 + o;
  float* xf = D.xf + I.xface;
  float* yf = D.yf + I.yface;
  const float* in = ((step & 1) == 0 ? D.la : D.lb) + o;
  float* out = ((step & 1) == 0 ? D.lb : D.la) + o;
  const float* phi = D.phi != nullptr ? D.phi + o : nullptr;
  const double isx = 1.0 / (static_cast<double>(I.dx) * I.dx);
  const double isy = 1.0 / (static_cast<double>(I.dy) * I.dy);
  AdrParams A{};
  A.nx = nx;
  A.ny = ny;
  A.signals = 1;
  A.dx = I.dx;
  A.dy = I.dy;
  A.dz = I.dz;
  A.kind[0] = A.kind[1] = MSIM_FIXED;
  A.kind[2] = A.kind[3] = A.kind[4] = A.kind[5] = MSIM_NO_FLUX;
  A.has_field = 0;  // velocities are set per site below
  A.has_affine = 0;
  A.has_monod = phi != nullptr ? 1 : 0;
  A.diffusion[0] = I.diffusion;
  A.boundary[0][0] = I.reservoir;
  A.vmax[0] = P.vmax;
  A.monod_k[0] = P.monod_k;
  const uint32_t tx = threadIdx.x / TY, ty = threadIdx.x % TY;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  uint32_t bad = 0;
  for (uint32_t xr = item.x0; xr < item.x1; xr += RX) {
    const uint32_t x = xr + tx;
    if (x >= item.x1) continue;
    for (uint32_t y = ty; y < ny; y += TY) {
      const size_t i = static_cast<size_t>(x) * ny + y;
      const double res = residual_f64(x64, D.cxl + o, D.cyl + o, D.bc + o, D.rhs + o, I.inlet, x,
                                      y, nx, ny, i, isx, isy);
      acc[0] += res * res;
      // This site's four faces; the lower x and y faces (and the upper ones
      // at the grid's end) are this item's to store.
      const float uxl = face_x(I, x64, cond, solid, x, y);
      const float uxu = face_x(I, x64, cond, solid, x + 1, y);
      const float uyl = face_y(I, x64, cond, solid, x, y);
      const float uyu = face_y(I, x64, cond, solid, x, y + 1);
      xf[i] = uxl;
      if (x + 1 == nx) xf[i + ny] = uxu;
      const size_t yi = static_cast<size_t>(x) * (ny + 1) + y;
      yf[yi] = uyl;
      if (y + 1 == ny) yf[yi + 1] = uyu;
      const float current = in[i];
      if (solid[i] != 0) {
        out[i] = current;
        continue;
      }
      SiteGeometry g = geometry(A, solid, xf, yf, x, y, 0);
      g.ulo[0] = uxl;
      g.uup[0] = uxu;
      g.ulo[1] = uyl;
      g.uup[1] = uyu;
      const float candidate = fe_candidate_f32(A, g, in, x, y, 0, dt, 0.0f, 0.0f, phi);
      if (!isfinite(candidate) || candidate < 0.0f) bad = 1;
      out[i] = candidate;
      acc[1] += static_cast<double>(current);
      acc[2] += static_cast<double>(candidate);
      if (phi != nullptr) {
        acc[3] += static_cast<double>(P.vmax) * static_cast<double>(phi[i]) *
                  static_cast<double>(current) / (static_cast<double>(P.monod_k) + current);
      }
    }
  }
  if (bad) atomicOr(&D.flags[inst], 4u);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const double t = block_sum<NT>(acc[k], s_red);
    if (threadIdx.x == 0) {
      partials[(static_cast<size_t>(step) * total + base + blockIdx.x) * 4 + k] = t;
    }
  }
}

// The same step for instances at most 256 columns wide, marching, every
// width class in one launch. A workgroup of 256 threads holds 256 / W groups
// of W threads (W = 64, 128 or 256: the width class), each group one work
// item (rows [x0, x1) of an instance), one thread per column. A group walks
// x, so each array is read once; the x neighbours come from registers, the y
// neighbours from the group's segment of an LDS row, and each x face is
// computed once (the upper face of a row is the next row's lower face). The
// groups of a workgroup walk the same number of rows (the most any of them
// has; a group past its own rows idles), so the row barriers are uniform.
// Every site's arithmetic is the general kernel's, so the two agree bit for
// bit.
constexpr int kMarchThreads = 256;
constexpr int kMarchGroups = 4;  // groups per workgroup at the narrowest width

struct MarchBlock {
  uint32_t width;                 // W
  uint32_t rows;                  // rows every group walks
  uint32_t item[kMarchGroups];    // work items; 0xffffffff: none
};

__global__ __launch_bounds__(kMarchThreads) void k_batch_march(
    BatchData D, BatchParams P, const BatchItem* __restrict__ items,
    const MarchBlock* __restrict__ blocks, double* __restrict__ partials, uint32_t step, float dt,
    uint32_t total) {
  struct Row {
    double p;
    float cond, c, cxl, cyl, bc, rhs, phi;
    bool solid;
  };
  __shared__ double s_p[2][kMarchThreads];
  __shared__ float s_cond[2][kMarchThreads], s_c[2][kMarchThreads], s_cyl[2][kMarchThreads];
  __shared__ uint8_t s_s[2][kMarchThreads];
  __shared__ double s_red[4][kMarchThreads / kWave];
  const MarchBlock blk = blocks[blockIdx.x];
  const uint32_t W = blk.width;
  const uint32_t group = threadIdx.x / W;
  const uint32_t y = threadIdx.x % W;
  const uint32_t seg = group * W;  // the group's segment of the LDS rows
  const uint32_t item_index = blk.item[group];
  const bool has_item = item_index != 0xffffffffu;
  const BatchItem item = has_item ? items[item_index] : BatchItem{0, 0, 0, 0};
  const uint32_t inst = item.inst;
  const BatchDesc I = D.desc[inst];
  const uint32_t nx = I.nx, ny = I.ny;
  const size_t o = I.site;
  const bool valid = has_item && y < ny;
  const float* in = ((step & 1) == 0 ? D.la : D.lb) + o;
  float* out = ((step & 1) == 0 ? D.lb : D.la) + o;
  const bool monod = D.phi != nullptr;
  float* xf = D.xf + I.xface;
  float* yf = D.yf + I.yface;
  const double isx = 1.0 / (static_cast<double>(I.dx) * I.dx);
  const double isy = 1.0 / (static_cast<double>(I.dy) * I.dy);
  AdrParams A{};
  A.nx = nx;
  A.ny = ny;
  A.signals = 1;
  A.dx = I.dx;
  A.dy = I.dy;
  A.dz = I.dz;
  A.kind[0] = A.kind[1] = MSIM_FIXED;
  A.kind[2] = A.kind[3] = A.kind[4] = A.kind[5] = MSIM_NO_FLUX;
  A.has_field = 1;
  A.has_monod = monod ? 1 : 0;
  A.diffusion[0] = I.diffusion;
  A.boundary[0][0] = I.reservoir;
  A.vmax[0] = P.vmax;
  A.monod_k[0] = P.monod_k;
  const int x0 = static_cast<int>(item.x0), x1 = static_cast<int>(item.x1);
  auto load = [&](int xx, bool full) {
    Row w{};
    if (!valid || xx < 0 || xx >= static_cast<int>(nx) || xx > x1) return w;
    const size_t i = o + static_cast<size_t>(xx) * ny + y;
    w.p = D.x64[i];
    w.cond = D.cond[i];
    w.c = in[i - o];
    w.solid = D.solid[i] != 0;
    w.cxl = D.cxl[i];  // also the upper x coupling of the row before
    if (!full) return w;
    w.cyl = D.cyl[i];
    w.bc = D.bc[i];
    w.rhs = D.rhs[i];
    if (monod) w.phi = D.phi[i];
    return w;
  };
  // Face x fx of this column from the rows either side (face_x's arithmetic).
  auto face_x_of = [&](const Row& lo, const Row& up, int fx) -> float {
    const bool has_lower = fx > 0, has_upper = fx < static_cast<int>(nx);
    double value;
    if (has_lower && has_upper) {
      const float fm = harmonic(lo.cond, up.cond);
      value = -static_cast<double>(fm) * (up.p - lo.p) / static_cast<double>(I.dx);
    } else {
      const Row& site = has_upper ? up : lo;
      float fc = 0.0f, fp = 0.0f;
      if (site.cond != 0.0f) {
        fc = (has_upper ? 2.0f : -2.0f) * site.cond / I.dx;
        fp = has_upper ? I.inlet : 0.0f;
      }
      value = static_cast<double>(fc) * (static_cast<double>(fp) - site.p);
    }
    const float flux = static_cast<float>(value);
    if ((has_lower && lo.solid) || (has_upper && up.solid)) return 0.0f;
    return flux / I.dz;
  };
  // Face y fy of row buf from the group's LDS row (face_y's arithmetic).
  auto face_y_of = [&](int buf, uint32_t fy) -> float {
    const bool has_lower = fy > 0, has_upper = fy < ny;
    double value;
    if (has_lower && has_upper) {
      const float fm = harmonic(s_cond[buf][seg + fy - 1], s_cond[buf][seg + fy]);
      value = -static_cast<double>(fm) * (s_p[buf][seg + fy] - s_p[buf][seg + fy - 1]) /
              static_cast<double>(I.dy);
    } else {
      const double ps = has_upper ? s_p[buf][seg + fy] : s_p[buf][seg + fy - 1];
      value = static_cast<double>(0.0f) * (static_cast<double>(0.0f) - ps);
    }
    const float flux = static_cast<float>(value);
    if ((has_lower && s_s[buf][seg + fy - 1] != 0) || (has_upper && s_s[buf][seg + fy] != 0))
      return 0.0f;
    return flux / I.dz;
  };
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  uint32_t bad = 0;
  Row prev = load(x0 - 1, false);
  Row cur = load(x0, true);
  Row next = load(x0 + 1, x0 + 1 < x1);
  float uxl = face_x_of(prev, cur, x0);
  for (uint32_t r = 0; r < blk.rows; ++r) {
    const int xx = x0 + static_cast<int>(r);
    const bool live = valid && xx < x1;
    const Row ahead = xx + 2 <= x1 ? load(xx + 2, xx + 2 < x1) : Row{};
    const int buf = static_cast<int>(r & 1);
    s_p[buf][threadIdx.x] = cur.p;
    s_cond[buf][threadIdx.x] = cur.cond;
    s_c[buf][threadIdx.x] = cur.c;
    s_cyl[buf][threadIdx.x] = cur.cyl;
    s_s[buf][threadIdx.x] = cur.solid ? 1 : 0;
    __syncthreads();
    const float uxu = face_x_of(cur, next, xx + 1);
    if (live) {
      const size_t i = static_cast<size_t>(xx) * ny + y;
      // residual_f64's arithmetic.
      const double c = cur.p;
      double a = static_cast<double>(cur.bc) * c;
      if (xx > 0) a += (static_cast<double>(cur.cxl) * isx) * (c - prev.p);
      if (xx + 1 < static_cast<int>(nx)) a += (static_cast<double>(next.cxl) * isx) * (c - next.p);
      if (y > 0) a += (static_cast<double>(cur.cyl) * isy) * (c - s_p[buf][seg + y - 1]);
      if (y + 1 < ny)
        a += (static_cast<double>(s_cyl[buf][seg + y + 1]) * isy) * (c - s_p[buf][seg + y + 1]);
      const double res = static_cast<double>(I.inlet) * static_cast<double>(cur.rhs) - a;
      acc[0] += res * res;
      const float uyl = face_y_of(buf, y);
      const float uyu = face_y_of(buf, y + 1);
      xf[i] = uxl;
      if (xx + 1 == static_cast<int>(nx)) xf[i + ny] = uxu;
      const size_t yi = static_cast<size_t>(xx) * (ny + 1) + y;
      yf[yi] = uyl;
      if (y + 1 == ny) yf[yi + 1] = uyu;
      const float current = cur.c;
      if (cur.solid) {
        out[i] = current;
      } else {
        const bool xlo_edge = xx == 0, xhi_edge = xx + 1 == static_cast<int>(nx);
        const bool ylo_edge = y == 0, yhi_edge = y + 1 == ny;
        SiteGeometry g;
        g.clo[0] = xlo_edge ? false : prev.solid;
        g.cup[0] = xhi_edge ? false : next.solid;
        g.clo[1] = ylo_edge ? true : s_s[buf][seg + y - 1] != 0;
        g.cup[1] = yhi_edge ? true : s_s[buf][seg + y + 1] != 0;
        g.ulo[0] = uxl;
        g.uup[0] = uxu;
        g.ulo[1] = uyl;
        g.uup[1] = uyu;
        const float l0 = xlo_edge ? exterior(A, 0, 0, current, 0.0f, y) : prev.c;
        const float u0 = xhi_edge ? exterior(A, 1, 0, current, 0.0f, y) : next.c;
        const float l1 = ylo_edge ? exterior(A, 2, 0, current, 0.0f, static_cast<uint32_t>(xx))
                                  : s_c[buf][seg + y - 1];
        const float u1 = yhi_edge ? exterior(A, 3, 0, current, 0.0f, static_cast<uint32_t>(xx))
                                  : s_c[buf][seg + y + 1];
        const float candidate =
            fe_update_f32(A, g, current, l0, u0, l1, u1, 0, dt, 0.0f, 0.0f, cur.phi);
        if (!isfinite(candidate) || candidate < 0.0f) bad = 1;
        out[i] = candidate;
        acc[1] += static_cast<double>(current);
        acc[2] += static_cast<double>(candidate);
        if (monod) {
          acc[3] += static_cast<double>(P.vmax) * static_cast<double>(cur.phi) *
                    static_cast<double>(current) / (static_cast<double>(P.monod_k) + current);
        }
      }
    }
    uxl = uxu;
    prev = cur;
    cur = next;
    next = ahead;
  }
  if (bad) atomicOr(&D.flags[inst], 4u);
  // Per group: wave sums, then the group's waves in order.
  const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const double v = wave_sum(acc[k]);
    if (lane == 0) s_red[k][wave] = v;
  }
  __syncthreads();
  if (has_item && y == 0) {
    const uint32_t first = seg / kWave, waves = W / kWave;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      double t = 0.0;
      for (uint32_t w = 0; w < waves; ++w) t += s_red[k][first + w];
      partials[(static_cast<size_t>(step) * total + item_index) * 4 + k] = t;
    }
  }
}

using StepKernel = void (*)(BatchData, BatchParams, const BatchItem*, double*, uint32_t, float,
                            uint32_t, uint32_t);

// A launch shape of the step: sites per work item, and for instances wider
// than 256 columns (the general kernel) the workgroup size and sweep row
// width.
struct Shape {
  int threads, row, chunk;
  StepKernel step;
};

const Shape kShapes[] = {
    {256, 64, 512, k_batch_step<256, 64>},    {256, 64, 1024, k_batch_step<256, 64>},
    {256, 64, 2048, k_batch_step<256, 64>},   {256, 64, 4096, k_batch_step<256, 64>},
    {512, 64, 8192, k_batch_step<512, 64>},   {256, 128, 16384, k_batch_step<256, 128>},
};
constexpr int kShapeCount = static_cast<int>(sizeof(kShapes) / sizeof(kShapes[0]));
constexpr int kDefaultShape = 1;
// Instance classes by width: the marching kernel's groups of 64, 128 and 256
// threads for at most that many columns, then the general kernel.
constexpr int kClasses = 4;
constexpr uint32_t kClassWidth[kClasses - 1] = {64, 128, 256};

int class_of(uint32_t ny) {
  for (int c = 0; c < kClasses - 1; ++c) {
    if (ny <= kClassWidth[c]) return c;
  }
  return kClasses - 1;
}
constexpr int kSetupThreads = 1024;
constexpr int kFlowThreads = 1024;  // of k_batch_flow and k_flow_tail
// Levels of at most this many cells are the tail's: a 256-instance sweep solves
// in 17.6 ms with 2048, 17.9 with 4096, 18.0 with 8192.
constexpr uint64_t kTailCells = 2048;
constexpr uint32_t kFlowBodies = 4;  // bodies between two looks at the finished instances

// Whether a batch is solved one workgroup per instance. An iteration then takes
// what the largest instance takes one compute unit; over the whole chip it
// takes some 45 us of launches and dependent reads, and the sites of all. In us
// per iteration, alone and together: 1 x 64x64 31 and 46, 1 x 96x80 52 and 54,
// 1 x 128x96 67 and 58, 64 x 128x96 78 and 81, 256 x 128x96 92 and 144,
// 64 x 256x128 187 and 121, 256 x 256x128 291 and 328, 64 x 512x256 903 and 344
// (256 compute units).
constexpr uint64_t kAloneSites = 8192;
bool solve_alone(uint64_t units, uint64_t sites, uint64_t largest) {
  return largest <= kAloneSites || units * sites >= largest * largest;
}

}  // namespace

// Device state of an uploaded batch.
struct BatchDevice {
  uint32_t count = 0;
  uint64_t sites = 0, xfaces = 0, yfaces = 0;
  std::vector<BatchDesc> desc;
  std::vector<uint32_t> order;
  std::vector<std::vector<BatchItem>> items;  // per shape, grouped by instance class
  std::vector<std::array<uint32_t, 5>> class_begin;  // per shape: first item of each class, end
  std::vector<std::unique_ptr<DeviceBuffer<BatchItem>>> d_items;
  std::vector<std::vector<MarchBlock>> march;  // per shape: workgroups of the marching launch
  std::vector<std::unique_ptr<DeviceBuffer<MarchBlock>>> d_march;
  DeviceBuffer<BatchDesc> d_desc;
  DeviceBuffer<uint32_t> d_order, iterations, flags;
  DeviceBuffer<uint8_t> solid;
  DeviceBuffer<float> mobility, cond, cxl, cyl, bc, diag, rhs, phi, x, r, p, p2, q, z, xf, yf, la, lb,
      residual, saved;
  std::vector<BatchLevels> levels;  // per instance
  DeviceBuffer<BatchLevels> d_levels;
  DeviceBuffer<float> lwx, lwy, lbc, ldinv, lr, le, cinv;
  DeviceBuffer<double> x64, bnorm2, partials;
  // The solve over the whole chip: tiles per level (down: of the level below),
  // shares of the products, the host's view of the finished instances.
  std::vector<std::unique_ptr<DeviceBuffer<FlowTile>>> flow_down, flow_up;
  DeviceBuffer<FlowSpan> flow_span;
  DeviceBuffer<FlowState> flow_state;
  DeviceBuffer<double> flow_share;
  DeviceBuffer<uint32_t> flow_done;
  uint32_t* host_done = nullptr;  // pinned, two by turns
  hipEvent_t looked[2] = {};
  BatchParams params{};
  bool has_phi = false;
  bool solved = false;
  int shape = -1;   // chosen by the autotuner; -1: the default
  int current = 0;  // 0: levels in la, 1: in lb
  hipGraphExec_t graph = nullptr;  // the captured run and what it was captured with
  uint32_t graph_steps = 0;
  float graph_dt = 0.0f;
  int graph_shape = -1;
  BatchData graph_data{};
  const double* graph_partials = nullptr;
  ~BatchDevice() {
    for (hipEvent_t e : looked) {
      if (e != nullptr) static_cast<void>(hipEventDestroy(e));
    }
    if (host_done != nullptr) static_cast<void>(hipHostFree(host_done));
    if (graph != nullptr) static_cast<void>(hipGraphExecDestroy(graph));
  }
};

namespace {

BatchData batch_data(BatchDevice& B) {
  BatchData D{};
  D.desc = B.d_desc.data();
  D.order = B.d_order.data();
  D.solid = B.solid.data();
  D.cond = B.cond.data();
  D.cxl = B.cxl.data();
  D.cyl = B.cyl.data();
  D.bc = B.bc.data();
  D.rhs = B.rhs.data();
  D.phi = B.has_phi ? B.phi.data() : nullptr;
  D.x64 = B.x64.data();
  D.x = B.x.data();
  D.r = B.r.data();
  D.p = B.p.data();
  D.p2 = B.p2.data();
  D.q = B.q.data();
  D.xf = B.xf.data();
  D.yf = B.yf.data();
  D.la = B.la.data();
  D.lb = B.lb.data();
  D.iterations = B.iterations.data();
  D.residual = B.residual.data();
  D.bnorm2 = B.bnorm2.data();
  D.flags = B.flags.data();
  D.z = B.z.data();
  D.levels = B.d_levels.data();
  D.lwx = B.lwx.data();
  D.lwy = B.lwy.data();
  D.lbc = B.lbc.data();
  D.ldinv = B.ldinv.data();
  D.lr = B.lr.data();
  D.le = B.le.data();
  D.cinv = B.cinv.data();
  return D;
}

int shape_of(const BatchDevice& B) { return B.shape >= 0 ? B.shape : kDefaultShape; }

void launch_step(Context& ctx, BatchDevice& B, const BatchData& D, int shape, uint32_t step,
                 float dt) {
  const Shape& s = kShapes[shape];
  const auto& begin = B.class_begin[shape];
  const uint32_t total = static_cast<uint32_t>(B.items[shape].size());
  // Every instance at most 256 columns wide: one launch.
  const uint32_t marching = static_cast<uint32_t>(B.march[shape].size());
  if (marching > 0) {
    k_batch_march<<<marching, kMarchThreads, 0, ctx.stream>>>(
        D, B.params, B.d_items[shape]->data(), B.d_march[shape]->data(), B.partials.data(), step,
        dt, total);
    check(hipGetLastError(), "launch batch step");
  }
  // Wider instances: the general sweep.
  const uint32_t base = begin[kClasses - 1], n = begin[kClasses] - begin[kClasses - 1];
  if (n > 0) {
    hipLaunchKernelGGL(s.step, dim3(n), dim3(static_cast<uint32_t>(s.threads)), 0, ctx.stream, D,
                       B.params, B.d_items[shape]->data(), B.partials.data(), step, dt, base,
                       total);
    check(hipGetLastError(), "launch batch step");
  }
}

// Runs `steps` steps from the current levels, in a graph or eagerly.
void run_steps(Context& ctx, BatchDevice& B, int shape, float dt, uint32_t steps, bool graph) {
  const BatchData D = batch_data(B);
  if (B.current != 0) {
    check(hipMemcpyAsync(B.la.data(), B.lb.data(), B.sites * sizeof(float),
                         hipMemcpyDeviceToDevice, ctx.stream),
          "levels to the first buffer");
    B.current = 0;
  }
  size_t most = 0;
  for (const auto& it : B.items) most = std::max(most, it.size());
  B.partials.reserve(static_cast<size_t>(steps) * most * 4);
  if (!graph) {
    for (uint32_t s = 0; s < steps; ++s) launch_step(ctx, B, D, shape, s, dt);
  } else {
    // A captured graph holds every pointer: capture again when any changed.
    if (B.graph == nullptr || B.graph_steps != steps || B.graph_dt != dt ||
        B.graph_shape != shape || std::memcmp(&B.graph_data, &D, sizeof(D)) != 0 ||
        B.graph_partials != B.partials.data()) {
      if (B.graph != nullptr) {
        check(hipGraphExecDestroy(B.graph), "destroy graph");
        B.graph = nullptr;
      }
      hipGraph_t g = nullptr;
      check(hipStreamBeginCapture(ctx.stream, hipStreamCaptureModeThreadLocal), "begin capture");
      for (uint32_t s = 0; s < steps; ++s) launch_step(ctx, B, D, shape, s, dt);
      check(hipStreamEndCapture(ctx.stream, &g), "end capture");
      const hipError_t e = hipGraphInstantiate(&B.graph, g, nullptr, nullptr, 0);
      static_cast<void>(hipGraphDestroy(g));
      check(e, "instantiate graph");
      B.graph_steps = steps;
      B.graph_dt = dt;
      B.graph_shape = shape;
      B.graph_data = D;
      B.graph_partials = B.partials.data();
    }
    check(hipGraphLaunch(B.graph, ctx.stream), "launch graph");
  }
  B.current = static_cast<int>(steps & 1);
}

}  // namespace

namespace {

// Each instance's system and multilevel hierarchy: level shapes and offsets
// here, the operators and the coarsest inverses on the device.
void build_systems(Context& ctx, BatchDevice& B) {
  B.levels.assign(B.count, BatchLevels{});
  uint64_t pool = B.sites, inverses = 0;
  for (uint32_t k = 0; k < B.count; ++k) {
    const BatchDesc& d = B.desc[k];
    BatchLevels& L = B.levels[k];
    uint32_t nx = d.nx, ny = d.ny;
    L.off[0] = d.site;
    L.nx[0] = nx;
    L.ny[0] = ny;
    L.count = 1;
    while (static_cast<uint64_t>(nx) * ny > kBatchCoarse) {
      if (L.count == kBatchLevels) throw Error(MSIM_OVERFLOW, "batch instance needs too many levels");
      nx = (nx + 1) / 2;
      ny = (ny + 1) / 2;
      L.off[L.count] = pool;
      L.nx[L.count] = nx;
      L.ny[L.count] = ny;
      pool += static_cast<uint64_t>(nx) * ny;
      ++L.count;
    }
    L.coarse_n = nx * ny;
    L.cinv = inverses;
    inverses += static_cast<uint64_t>(L.coarse_n) * L.coarse_n;
  }
  for (auto* b : {&B.lwx, &B.lwy, &B.lbc, &B.ldinv, &B.lr, &B.le}) b->reserve(pool);
  B.cinv.reserve(std::max<uint64_t>(inverses, 1));
  B.d_levels.reserve(B.count);
  check(hipMemcpyAsync(B.d_levels.data(), B.levels.data(), B.count * sizeof(BatchLevels),
                       hipMemcpyHostToDevice, ctx.stream),
        "upload hierarchies");
  const BatchSetup D{B.solid.data(), B.mobility.data(), B.cond.data(), B.diag.data(),
                     B.rhs.data(),   B.bc.data(),       B.cxl.data(),  B.cyl.data(),
                     B.lwx.data(),   B.lwy.data(),      B.lbc.data(),  B.ldinv.data(),
                     B.cinv.data()};
  k_batch_setup<kSetupThreads><<<B.count, kSetupThreads, 0, ctx.stream>>>(
      B.d_desc.data(), B.d_order.data(), B.d_levels.data(), D);
  check(hipGetLastError(), "launch k_batch_setup");
}

// Tiles of the solve over the whole chip; none for a batch of small instances.
void plan_flow(Context& ctx, BatchDevice& B) {
  B.flow_down.clear();
  B.flow_up.clear();
  const BatchDesc& largest = B.desc[B.order[0]];
  if (solve_alone(ctx.compute_units, B.sites, static_cast<uint64_t>(largest.nx) * largest.ny)) return;
  std::vector<FlowSpan> span(B.count);
  std::vector<std::vector<FlowTile>> down, up;
  auto cut = [](std::vector<FlowTile>& to, uint32_t inst, uint32_t cells, uint32_t tile) {
    for (uint32_t lo = 0; lo < cells; lo += tile)
      to.push_back(FlowTile{inst, lo, std::min(cells, lo + tile), static_cast<uint32_t>(to.size())});
  };
  for (uint32_t k : B.order) {
    const BatchLevels& L = B.levels[k];
    uint32_t tail = 0;
    do {
      if (up.size() <= tail) {
        up.emplace_back();
        down.emplace_back();
      }
      const uint32_t first = static_cast<uint32_t>(up[tail].size());
      cut(up[tail], k, L.nx[tail] * L.ny[tail], kFlowTile);
      if (tail == 0) span[k] = FlowSpan{first, static_cast<uint32_t>(up[0].size()) - first, 0, 0};
      if (L.count == 1) break;
      cut(down[tail], k, L.nx[tail + 1] * L.ny[tail + 1], kFlowTile / 4);
      ++tail;
    } while (tail + 1 < L.count && static_cast<uint64_t>(L.nx[tail]) * L.ny[tail] > kTailCells);
    span[k].tail = tail;
  }
  auto upload = [&](const std::vector<FlowTile>& tiles) {
    auto buf = std::make_unique<DeviceBuffer<FlowTile>>();
    buf->reserve(tiles.size());
    check(hipMemcpyAsync(buf->data(), tiles.data(), tiles.size() * sizeof(FlowTile),
                         hipMemcpyHostToDevice, ctx.stream),
          "upload flow tiles");
    return buf;
  };
  for (const auto& t : up) B.flow_up.push_back(upload(t));
  for (const auto& t : down) B.flow_down.push_back(upload(t));
  B.flow_span.reserve(B.count);
  check(hipMemcpyAsync(B.flow_span.data(), span.data(), B.count * sizeof(FlowSpan),
                       hipMemcpyHostToDevice, ctx.stream),
        "upload flow spans");
  B.flow_state.reserve(B.count);
  B.flow_share.reserve(3 * up[0].size());
  B.flow_done.reserve(1);
  if (B.host_done == nullptr) {
    void* ptr = nullptr;
    check(hipHostMalloc(&ptr, 2 * sizeof(uint32_t), hipHostMallocDefault), "hipHostMalloc");
    B.host_done = static_cast<uint32_t*>(ptr);
    for (hipEvent_t& e : B.looked)
      check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
  }
  // The host vectors end here.
  check(hipStreamSynchronize(ctx.stream), "flow tiles");
}

void solve_together(Context& ctx, BatchDevice& B) {
  const uint32_t levels = static_cast<uint32_t>(B.flow_up.size());
  const uint32_t tiles = static_cast<uint32_t>(B.flow_up[0]->size());
  const FlowWork W{batch_data(B),        B.params, B.flow_span.data(), B.flow_state.data(),
                   B.flow_share.data(), tiles,    B.flow_done.data()};
  k_flow_begin<<<(B.count + 255) / 256, 256, 0, ctx.stream>>>(W.state, B.count, W.done);
  k_flow_direction<<<tiles, kFlowTileThreads, 0, ctx.stream>>>(W, B.flow_up[0]->data());
  auto body = [&]() {
    for (uint32_t l = 0; l < levels; ++l) {
      const uint32_t n = static_cast<uint32_t>(B.flow_down[l]->size());
      if (n > 0)
        k_flow_down<<<n, kFlowTileThreads, 0, ctx.stream>>>(W, B.flow_down[l]->data(), l);
    }
    k_flow_tail<kFlowThreads><<<B.count, kFlowThreads, 0, ctx.stream>>>(W);
    for (uint32_t l = levels; l-- > 0;) {
      k_flow_up<<<static_cast<uint32_t>(B.flow_up[l]->size()), kFlowTileThreads, 0, ctx.stream>>>(
          W, B.flow_up[l]->data(), l);
    }
    k_flow_direction<<<tiles, kFlowTileThreads, 0, ctx.stream>>>(W, B.flow_up[0]->data());
    k_flow_update<<<tiles, kFlowTileThreads, 0, ctx.stream>>>(W, B.flow_up[0]->data());
    check(hipGetLastError(), "launch batch flow");
  };
  // An instance takes one body per iteration and per refinement, and one to
  // find that it is done.
  const uint64_t most = static_cast<uint64_t>(B.params.max_iterations) + kRefinements + 2;
  const uint64_t looks = (most + kFlowBodies - 1) / kFlowBodies;
  for (uint64_t k = 0; k <= looks; ++k) {
    if (k < looks) {
      for (uint32_t j = 0; j < kFlowBodies; ++j) body();
      check(hipMemcpyAsync(B.host_done + (k & 1), B.flow_done.data(), sizeof(uint32_t),
                           hipMemcpyDeviceToHost, ctx.stream),
            "look at finished instances");
      check(hipEventRecord(B.looked[k & 1], ctx.stream), "event");
    }
    if (k == 0) continue;
    check(hipEventSynchronize(B.looked[(k - 1) & 1]), "batch flow");
    if (B.host_done[(k - 1) & 1] == B.count) break;
  }
  k_flow_faces<<<tiles, kFlowTileThreads, 0, ctx.stream>>>(W.D, B.flow_up[0]->data());
  check(hipGetLastError(), "launch k_flow_faces");
}

}  // namespace

BatchDevice& batch_of(Context& ctx) {
  if (ctx.batch == nullptr) ctx.batch = std::make_shared<BatchDevice>();
  return *ctx.batch;
}

void batch_upload(Context& ctx, uint32_t count, const msim_batch_instance* inst,
                  const msim_batch_params& params) {
  ctx.batch.reset();
  BatchDevice& B = batch_of(ctx);
  B.count = count;
  B.desc.resize(count);
  uint64_t site = 0, xface = 0, yface = 0;
  B.has_phi = false;
  for (uint32_t k = 0; k < count; ++k) {
    const msim_batch_instance& in = inst[k];
    BatchDesc& d = B.desc[k];
    d.nx = in.nx;
    d.ny = in.ny;
    d.site = site;
    d.xface = xface;
    d.yface = yface;
    d.dx = in.dx;
    d.dy = in.dy;
    d.dz = in.dz;
    d.inlet = in.inlet_pressure;
    d.diffusion = in.diffusion;
    d.reservoir = in.reservoir;
    site += static_cast<uint64_t>(in.nx) * in.ny;
    xface += static_cast<uint64_t>(in.nx + 1) * in.ny;
    yface += static_cast<uint64_t>(in.nx) * (in.ny + 1);
    if (in.phi != nullptr) B.has_phi = true;
  }
  B.sites = site;
  B.xfaces = xface;
  B.yfaces = yface;
  // Largest instances first: they are dispatched first.
  B.order.resize(count);
  std::iota(B.order.begin(), B.order.end(), 0u);
  std::stable_sort(B.order.begin(), B.order.end(), [&](uint32_t a, uint32_t b) {
    return static_cast<uint64_t>(B.desc[a].nx) * B.desc[a].ny >
           static_cast<uint64_t>(B.desc[b].nx) * B.desc[b].ny;
  });
  // Work items of each shape: blocks of whole rows of about `chunk` sites.
  B.items.assign(kShapeCount, {});
  B.class_begin.assign(kShapeCount, {});
  B.d_items.clear();
  B.march.clear();
  B.d_march.clear();
  for (int s = 0; s < kShapeCount; ++s) {
    for (int c = 0; c < kClasses; ++c) {
      B.class_begin[s][c] = static_cast<uint32_t>(B.items[s].size());
      for (uint32_t k : B.order) {
        const BatchDesc& d = B.desc[k];
        if (class_of(d.ny) != c) continue;
        const uint32_t rows =
            std::max<uint32_t>(1, static_cast<uint32_t>(kShapes[s].chunk) / d.ny);
        for (uint32_t x0 = 0; x0 < d.nx; x0 += rows)
          B.items[s].push_back(BatchItem{k, x0, std::min(d.nx, x0 + rows), 0});
      }
    }
    B.class_begin[s][kClasses] = static_cast<uint32_t>(B.items[s].size());
    if (B.items[s].size() > 0x7FFFFFFFu) throw Error(MSIM_OVERFLOW, "too many batch work items");
    // Workgroups of the marching launch: 256 / W consecutive items of a
    // class of width W, walking the most rows any of them has.
    std::vector<MarchBlock> blocks;
    for (int c = 0; c < kClasses - 1; ++c) {
      const uint32_t width = kClassWidth[c];
      const uint32_t per = static_cast<uint32_t>(kMarchThreads) / width;
      for (uint32_t j = B.class_begin[s][c]; j < B.class_begin[s][c + 1]; j += per) {
        MarchBlock b{};
        b.width = width;
        for (uint32_t g = 0; g < static_cast<uint32_t>(kMarchGroups); ++g) {
          const uint32_t it = j + g;
          if (g < per && it < B.class_begin[s][c + 1]) {
            b.item[g] = it;
            b.rows = std::max(b.rows, B.items[s][it].x1 - B.items[s][it].x0);
          } else {
            b.item[g] = 0xffffffffu;
          }
        }
        blocks.push_back(b);
      }
    }
    auto mbuf = std::make_unique<DeviceBuffer<MarchBlock>>();
    mbuf->reserve(std::max<size_t>(blocks.size(), 1));
    check(hipMemcpyAsync(mbuf->data(), blocks.data(), blocks.size() * sizeof(MarchBlock),
                         hipMemcpyHostToDevice, ctx.stream),
          "upload marching workgroups");
    B.d_march.push_back(std::move(mbuf));
    B.march.push_back(std::move(blocks));
    auto buf = std::make_unique<DeviceBuffer<BatchItem>>();
    buf->reserve(B.items[s].size());
    check(hipMemcpyAsync(buf->data(), B.items[s].data(), B.items[s].size() * sizeof(BatchItem),
                         hipMemcpyHostToDevice, ctx.stream),
          "upload work items");
    B.d_items.push_back(std::move(buf));
  }
  const size_t n = site;
  B.solid.reserve(n);
  for (auto* b : {&B.mobility, &B.cond, &B.cxl, &B.cyl, &B.bc, &B.diag, &B.rhs, &B.phi, &B.x,
                  &B.r, &B.p, &B.p2, &B.q, &B.z, &B.la, &B.lb, &B.saved})
    b->reserve(n);
  B.x64.reserve(n);
  B.xf.reserve(xface);
  B.yf.reserve(yface);
  B.d_desc.reserve(count);
  B.d_order.reserve(count);
  B.iterations.reserve(count);
  B.flags.reserve(count);
  B.residual.reserve(count);
  B.bnorm2.reserve(count);
  check(hipMemcpyAsync(B.d_desc.data(), B.desc.data(), count * sizeof(BatchDesc),
                       hipMemcpyHostToDevice, ctx.stream),
        "upload batch");
  check(hipMemcpyAsync(B.d_order.data(), B.order.data(), count * sizeof(uint32_t),
                       hipMemcpyHostToDevice, ctx.stream),
        "upload batch order");
  check(hipMemsetAsync(B.flags.data(), 0, count * sizeof(uint32_t), ctx.stream), "clear flags");
  check(hipMemsetAsync(B.x64.data(), 0, n * sizeof(double), ctx.stream), "clear pressure");
  for (uint32_t k = 0; k < count; ++k) {
    const msim_batch_instance& in = inst[k];
    const BatchDesc& d = B.desc[k];
    const size_t m = static_cast<size_t>(d.nx) * d.ny;
    if (in.obstacles != nullptr) {
      check(hipMemcpyAsync(B.solid.data() + d.site, in.obstacles, m, hipMemcpyHostToDevice,
                           ctx.stream),
            "upload obstacles");
    } else {
      check(hipMemsetAsync(B.solid.data() + d.site, 0, m, ctx.stream), "clear obstacles");
    }
    check(hipMemcpyAsync(B.mobility.data() + d.site, in.mobility, m * sizeof(float),
                         hipMemcpyHostToDevice, ctx.stream),
          "upload mobility");
    if (B.has_phi) {
      if (in.phi != nullptr) {
        check(hipMemcpyAsync(B.phi.data() + d.site, in.phi, m * sizeof(float),
                             hipMemcpyHostToDevice, ctx.stream),
              "upload phi");
      } else {
        check(hipMemsetAsync(B.phi.data() + d.site, 0, m * sizeof(float), ctx.stream),
              "clear phi");
      }
    }
    if (in.levels != nullptr) {
      check(hipMemcpyAsync(B.la.data() + d.site, in.levels, m * sizeof(float),
                           hipMemcpyHostToDevice, ctx.stream),
            "upload levels");
    } else {
      check(hipMemsetAsync(B.la.data() + d.site, 0, m * sizeof(float), ctx.stream),
            "clear levels");
    }
  }
  build_systems(ctx, B);
  plan_flow(ctx, B);
  B.params.tolerance = params.relative_tolerance;
  B.params.max_iterations = params.max_iterations;
  B.params.vmax = params.monod_vmax;
  B.params.monod_k = params.monod_k;
  B.current = 0;
  B.solved = false;
  check(hipStreamSynchronize(ctx.stream), "batch upload");
}

// Solves every instance's pressure from its current one and rebuilds its
// velocities.
void batch_solve_flow(Context& ctx, uint32_t* iterations, float* residual, uint32_t* flags) {
  BatchDevice& B = batch_of(ctx);
  if (B.count == 0) throw Error(MSIM_INVALID_ARGUMENT, "no batch is uploaded");
  if (B.flow_up.empty()) {
    k_batch_flow<kFlowThreads>
        <<<B.count, kFlowThreads, 0, ctx.stream>>>(batch_data(B), B.params);
    check(hipGetLastError(), "launch k_batch_flow");
  } else {
    solve_together(ctx, B);
  }
  B.solved = true;
  if (iterations != nullptr) {
    check(hipMemcpyAsync(iterations, B.iterations.data(), B.count * sizeof(uint32_t),
                         hipMemcpyDeviceToHost, ctx.stream),
          "download iterations");
  }
  if (residual != nullptr) {
    check(hipMemcpyAsync(residual, B.residual.data(), B.count * sizeof(float),
                         hipMemcpyDeviceToHost, ctx.stream),
          "download residuals");
  }
  if (flags != nullptr) {
    check(hipMemcpyAsync(flags, B.flags.data(), B.count * sizeof(uint32_t),
                         hipMemcpyDeviceToHost, ctx.stream),
          "download flags");
  }
  check(hipStreamSynchronize(ctx.stream), "batch flow");
}

int batch_autotune(Context& ctx, float dt, uint32_t steps, double* seconds) {
  BatchDevice& B = batch_of(ctx);
  if (B.count == 0) throw Error(MSIM_INVALID_ARGUMENT, "no batch is uploaded");
  if (!B.solved) throw Error(MSIM_INVALID_ARGUMENT, "solve the batch's flow first");
  // Every candidate starts from the same levels, and the batch is left as it was.
  float* levels = B.current == 0 ? B.la.data() : B.lb.data();
  check(hipMemcpyAsync(B.saved.data(), levels, B.sites * sizeof(float), hipMemcpyDeviceToDevice,
                       ctx.stream),
        "save levels");
  auto restore = [&]() {
    check(hipMemcpyAsync(B.la.data(), B.saved.data(), B.sites * sizeof(float),
                         hipMemcpyDeviceToDevice, ctx.stream),
          "restore levels");
    B.current = 0;
  };
  double best = 0.0;
  int choice = 0;
  for (int c = 0; c < kShapeCount; ++c) {
    restore();
    run_steps(ctx, B, c, dt, 1, false);  // warm
    restore();
    check(hipEventRecord(ctx.start, ctx.stream), "event");
    run_steps(ctx, B, c, dt, steps, false);
    check(hipEventRecord(ctx.stop, ctx.stream), "event");
    check(hipEventSynchronize(ctx.stop), "autotune");
    float ms = 0.0f;
    check(hipEventElapsedTime(&ms, ctx.start, ctx.stop), "event time");
    const double t = ms * 1.0e-3 / steps;
    if (seconds != nullptr) seconds[c] = t;
    if (c == 0 || t < best) {
      best = t;
      choice = c;
    }
  }
  restore();
  check(hipMemsetAsync(B.flags.data(), 0, B.count * sizeof(uint32_t), ctx.stream), "clear flags");
  check(hipStreamSynchronize(ctx.stream), "autotune");
  B.shape = choice;
  return choice;
}

void batch_shape(int index, int* threads, int* row, int* chunk) {
  *threads = kShapes[index].threads;
  *row = kShapes[index].row;
  *chunk = kShapes[index].chunk;
}

int batch_shape_count() { return kShapeCount; }

void batch_run(Context& ctx, float dt, uint32_t steps, bool graph, double* ledger,
               double* seconds) {
  BatchDevice& B = batch_of(ctx);
  if (B.count == 0) throw Error(MSIM_INVALID_ARGUMENT, "no batch is uploaded");
  if (!B.solved) throw Error(MSIM_INVALID_ARGUMENT, "solve the batch's flow first");
  const int shape = shape_of(B);
  check(hipEventRecord(ctx.start, ctx.stream), "event");
  run_steps(ctx, B, shape, dt, steps, graph);
  check(hipEventRecord(ctx.stop, ctx.stream), "event");
  check(hipEventSynchronize(ctx.stop), "batch run");
  float ms = 0.0f;
  check(hipEventElapsedTime(&ms, ctx.start, ctx.stop), "event time");
  if (seconds != nullptr) *seconds = ms * 1.0e-3;
  if (ledger == nullptr) return;
  // Per-instance rows from the per-item partials, added in item order.
  const auto& items = B.items[shape];
  std::vector<double> parts(static_cast<size_t>(steps) * items.size() * 4);
  std::vector<double> bb(B.count);
  check(hipMemcpyAsync(parts.data(), B.partials.data(), parts.size() * sizeof(double),
                       hipMemcpyDeviceToHost, ctx.stream),
        "download partials");
  check(hipMemcpyAsync(bb.data(), B.bnorm2.data(), B.count * sizeof(double),
                       hipMemcpyDeviceToHost, ctx.stream),
        "download norms");
  check(hipStreamSynchronize(ctx.stream), "ledger");
  std::fill(ledger, ledger + static_cast<size_t>(steps) * B.count * 4, 0.0);
  for (uint32_t s = 0; s < steps; ++s) {
    for (size_t j = 0; j < items.size(); ++j) {
      const double* pj = &parts[(static_cast<size_t>(s) * items.size() + j) * 4];
      double* row = ledger + (static_cast<size_t>(s) * B.count + items[j].inst) * 4;
      row[0] += pj[1];
      row[1] += pj[2];
      row[2] += pj[3];
      row[3] += pj[0];
    }
    for (uint32_t k = 0; k < B.count; ++k) {
      const BatchDesc& d = B.desc[k];
      const double volume = static_cast<double>(d.dx) * d.dy * d.dz;
      double* row = ledger + (static_cast<size_t>(s) * B.count + k) * 4;
      row[0] *= volume;
      row[1] *= volume;
      row[2] *= static_cast<double>(dt) * volume;
      row[3] = bb[k] > 0.0 ? std::sqrt(row[3] / bb[k]) : 0.0;
    }
  }
}

void batch_flags(Context& ctx, uint32_t* flags) {
  BatchDevice& B = batch_of(ctx);
  if (B.count == 0) throw Error(MSIM_INVALID_ARGUMENT, "no batch is uploaded");
  check(hipMemcpyAsync(flags, B.flags.data(), B.count * sizeof(uint32_t), hipMemcpyDeviceToHost,
                       ctx.stream),
        "download flags");
  check(hipStreamSynchronize(ctx.stream), "flags");
}

void batch_download(Context& ctx, uint32_t index, double* pressure, float* x_faces,
                    float* y_faces, float* levels) {
  BatchDevice& B = batch_of(ctx);
  if (index >= B.count) throw Error(MSIM_INVALID_ARGUMENT, "instance index out of range");
  const BatchDesc& d = B.desc[index];
  const size_t m = static_cast<size_t>(d.nx) * d.ny;
  if (pressure != nullptr) {
    check(hipMemcpyAsync(pressure, B.x64.data() + d.site, m * sizeof(double),
                         hipMemcpyDeviceToHost, ctx.stream),
          "download pressure");
  }
  if (x_faces != nullptr) {
    check(hipMemcpyAsync(x_faces, B.xf.data() + d.xface,
                         static_cast<size_t>(d.nx + 1) * d.ny * sizeof(float),
                         hipMemcpyDeviceToHost, ctx.stream),
          "download faces");
  }
  if (y_faces != nullptr) {
    check(hipMemcpyAsync(y_faces, B.yf.data() + d.yface,
                         static_cast<size_t>(d.nx) * (d.ny + 1) * sizeof(float),
                         hipMemcpyDeviceToHost, ctx.stream),
          "download faces");
  }
  if (levels != nullptr) {
    const float* src = (B.current == 0 ? B.la.data() : B.lb.data()) + d.site;
    check(hipMemcpyAsync(levels, src, m * sizeof(float), hipMemcpyDeviceToHost, ctx.stream),
          "download levels");
  }
  check(hipStreamSynchronize(ctx.stream), "batch download");
}

}  // namespace msim
