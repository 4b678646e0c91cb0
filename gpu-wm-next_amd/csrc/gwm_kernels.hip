// gwm_kernels.hip -- gfx950 kernels of the dry + warm-rain time step.
//
// Each kernel states the reference operator(s) it covers.  Semantics are the
// reference's 1x1 layout: a neighbour outside the owned range is the value
// the reference's halo exchange places there (map_cell / map_face), so no
// kernel depends on halo storage.  Periodic wrap faces (face 0 and face n of
// a face field) are kept equal as a state invariant, which makes the
// reference's owned-interface averaging (halo_exchange.cpp:217-285) an
// identity inside the step; gwm_sync_interfaces() establishes it on entry.
#include "gwm_kernels.hpp"
#include "gwm_micro.hpp"

#include <mutex>

namespace gwm {

namespace {

// Deterministic block sum of a double (256 threads).
__device__ inline double block_sum(double v, double* sh) {
  const int t = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
  const int n = blockDim.x * blockDim.y * blockDim.z;
  sh[t] = v;
  __syncthreads();
  for (int s = n / 2; s > 0; s >>= 1) {
    if (t < s) sh[t] += sh[t + s];
    __syncthreads();
  }
  const double r = sh[0];
  __syncthreads();
  return r;
}

}  // namespace

// ===========================================================================
// Level sums (deterministic).  mode 0: theta = rho_theta/max(rho,1e-6) of a
// state (dry_core.cu:462-490); mode 1: rho and p(rho, rho*theta_fixed) of the
// fast subcycle (dry_fast_modes.cu:42-67, FP32 atomics replaced by FP64
// partials in fixed order).  Block = 256 threads over a chunk of rows of one
// level; partials[(k*nchunk + c)*2 + {0,1}].
// ===========================================================================
constexpr int kPartialRows = 8;  // rows of one level per work-group

template <class R>
__device__ __forceinline__ void level_partials_body(const Geo& g, const R* rho, const R* aux,
                                                    int mode, double* partials,
                                                    const Base<R>& base, const VBlock& vb) {
  __shared__ double sh[256];
  const int k = vb.y;
  const int c = vb.x;
  const int nchunk = vb.gx;
  const int j0 = c * kPartialRows;
  const int t = threadIdx.x;
  double s0 = 0.0, s1 = 0.0;
  const bool pert = base.rho != nullptr;
  const R rb = pert ? base.rho[k] : R(0), thb = pert ? base.th[k] : R(0);
  const R rtb = pert ? base.rt[k] : R(0), pb = pert ? base.p[k] : R(0);
  // Each thread loads a column segment of the chunk's rows at once (all
  // loads in flight), then accumulates in row order.
  for (int i = t; i < g.nx; i += 256) {
    R rv[kPartialRows], av[kPartialRows];
#pragma unroll
    for (int q = 0; q < kPartialRows; ++q) {
      rv[q] = R(0);
      av[q] = R(0);
      if (j0 + q < g.ny) {
        const size_t c0 = g.cell(i, j0 + q, k);
        rv[q] = rho[c0];
        av[q] = aux[c0];
      }
    }
#pragma unroll
    for (int q = 0; q < kPartialRows; ++q) {
      if (j0 + q >= g.ny) break;
      const R r = rv[q];
      if (pert && base.drho) {
        // terrain form: theta relative to the level's base value (the
        // cell's base deviation plus its departure), for theta_ref
        const size_t c0 = g.cell(i, j0 + q, k);
        const R dt = base.dth[c0];
        s0 += static_cast<double>(dt + theta_pert(r, av[q], rb + base.drho[c0], thb + dt));
      } else if (pert) {
        // departures: theta' of (rho', (rho theta)'), or rho' and p' of
        // (rho', theta' fixed)
        if (mode == 0) {
          s0 += static_cast<double>(theta_pert(r, av[q], rb, thb));
        } else {
          const R tp = av[q];
          s0 += static_cast<double>(r);
          s1 += static_cast<double>(p_pert(rb * tp + r * (thb + tp), rtb, pb));
        }
      } else if (mode == 0) {
        s0 += static_cast<double>(q_theta(r, av[q]));
      } else {
        s0 += static_cast<double>(r);
        s1 += static_cast<double>(q_pressure(r, r * av[q]));
      }
    }
  }
  s0 = block_sum(s0, sh);
  s1 = block_sum(s1, sh);
  if (t == 0) {
    partials[(static_cast<size_t>(k) * nchunk + c) * 2 + 0] = s0;
    partials[(static_cast<size_t>(k) * nchunk + c) * 2 + 1] = s1;
  }
}

template <class R>
__global__ __launch_bounds__(256) void k_level_partials(Geo g, const R* rho, const R* aux,
                                                         int mode, double* partials,
                                                         Base<R> base) {
  level_partials_body(g, rho, aux, mode, partials, base, hw_block());
}
template <class R>
__global__ __launch_bounds__(256) void k_level_partials_batch(const PartialsItem<R>* items,
                                                               BatchMap bm) {
  VBlock vb;
  const PartialsItem<R>* it = batch_member(items, bm, vb);
  if (!it) return;
  const PartialsItem<R> a = *it;
  level_partials_body(a.g, a.rho, a.aux, a.mode, a.partials, a.base, vb);
}

// One 1024-thread block per level: thread t sums partials t, t+1024, ... in
// order over four interleaved accumulators (a level's 4096 partials of the
// 512 x 512 grid in one round of four loads per thread: the kernel is bound
// by load latency, not bytes), a fixed DPP reduction adds each wave's lanes
// (total in lane 63) and thread 0 adds the sixteen waves in a fixed tree, so
// the result does not depend on scheduling.  The kernel runs between every
// two fast substeps, so its length is the round trips it waits for.
constexpr int kFinalizeThreads = 1024;
constexpr int kFinalizeAcc = 4;

template <class R>
__device__ __forceinline__ void level_finalize_body(int nchunk, const double* partials, int mode,
                                                    double count, R* out0, R* out1,
                                                    const VBlock& vb) {
  __shared__ double sh[2][kFinalizeThreads / 64];
  const int k = vb.x;
  const int t = threadIdx.x;
  const double2* p = reinterpret_cast<const double2*>(partials) + static_cast<size_t>(k) * nchunk;
  constexpr int A = kFinalizeAcc;
  double a0[A], a1[A];
#pragma unroll
  for (int q = 0; q < A; ++q) a0[q] = a1[q] = 0.0;
  int c = t;
  for (; c + (A - 1) * kFinalizeThreads < nchunk; c += A * kFinalizeThreads) {
    double2 v[A];
#pragma unroll
    for (int q = 0; q < A; ++q) v[q] = p[c + q * kFinalizeThreads];
#pragma unroll
    for (int q = 0; q < A; ++q) {
      a0[q] += v[q].x;
      a1[q] += v[q].y;
    }
  }
#pragma unroll
  for (int q = 0; q < A; ++q) {
    if (c + q * kFinalizeThreads < nchunk) {
      const double2 v = p[c + q * kFinalizeThreads];
      a0[q] += v.x;
      a1[q] += v.y;
    }
  }
  const double s0 = wave_sum_to63((a0[0] + a0[1]) + (a0[2] + a0[3]));
  const double s1 = wave_sum_to63((a1[0] + a1[1]) + (a1[2] + a1[3]));
  if ((t & 63) == 63) {
    sh[0][t >> 6] = s0;
    sh[1][t >> 6] = s1;
  }
  __syncthreads();
  if (t != 0) return;
  // sixteen waves, pairwise
  auto tree = [](const double* x) {
    const double q0 = (x[0] + x[1]) + (x[2] + x[3]), q1 = (x[4] + x[5]) + (x[6] + x[7]);
    const double q2 = (x[8] + x[9]) + (x[10] + x[11]), q3 = (x[12] + x[13]) + (x[14] + x[15]);
    return (q0 + q1) + (q2 + q3);
  };
  static_assert(kFinalizeThreads == 1024 && kFinalizeAcc == 4, "tree sizes");
  const double S0 = tree(sh[0]);
  const double S1 = tree(sh[1]);
  if (mode == 0) {
    out0[k] = static_cast<R>(S0 / count);  // dry_core.cu:485-490
  } else {
    const R inv = R(1) / static_cast<R>(count);  // dry_fast_modes.cu:481-482
    out0[k] = static_cast<R>(S0) * inv;
    out1[k] = static_cast<R>(S1) * inv;
  }
}

template <class R>
__global__ __launch_bounds__(kFinalizeThreads) void k_level_finalize(int nz, int nchunk,
                                                                     const double* partials,
                                                                     int mode, double count,
                                                                     R* out0, R* out1) {
  (void)nz;
  level_finalize_body(nchunk, partials, mode, count, out0, out1, hw_block());
}
template <class R>
__global__ __launch_bounds__(kFinalizeThreads) void k_level_finalize_batch(
    const FinalizeItem<R>* items, BatchMap bm) {
  VBlock vb;
  const FinalizeItem<R>* it = batch_member(items, bm, vb);
  if (!it) return;
  const FinalizeItem<R> a = *it;
  level_finalize_body(a.nchunk, a.partials, a.mode, a.count, a.out0, a.out1, vb);
}

// ===========================================================================
// Pressure over the full storage (halo included) of the halo-filled state:
// compute_dry_pressure_fields (dry_pressure_gradient.cu:177-202, K20).
// ===========================================================================
template <class R>
__global__ void k_pressure(Geo g, const R* rho, const R* rt, R* p) {
  const size_t n = g.cell_total();
  const size_t a = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (a >= n) return;
  const int pi = static_cast<int>(a % g.pxc);
  const int pj = static_cast<int>((a / g.pxc) % g.pyc);
  const int k = static_cast<int>(a / (static_cast<size_t>(g.pxc) * g.pyc));
  Loader<R> L{g};
  const R r = L.cell(rho, pi - g.h, pj - g.h, k);
  const R t = L.cell(rt, pi - g.h, pj - g.h, k);
  p[a] = d_pressure(r, t);
}

template <class R>
__global__ void k_theta(Geo g, const R* rho, const R* rt, R* th, Base<R> base) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  const int k = blockIdx.z;
  if (i >= g.nx || j >= g.ny || k >= g.nz) return;
  const size_t c = g.cell(i, j, k);
  if (base.drho)  // terrain form: the cell's base
    th[c] = theta_pert(rho[c], rt[c], base.rho[k] + base.drho[c], base.th[k] + base.dth[c]);
  else
    th[c] = base.rho ? theta_pert(rho[c], rt[c], base.rho[k], base.th[k]) : q_theta(rho[c], rt[c]);
}

template <class R>
__global__ void k_rebuild_rt(Geo g, const R* rho, const R* th, R* rt, Base<R> base) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  const int k = blockIdx.z;
  if (i >= g.nx || j >= g.ny) return;
  const size_t c = g.cell(i, j, k);
  if (base.drho) {  // terrain form: the cell's base
    const R rb = base.rho[k] + base.drho[c], tb = base.th[k] + base.dth[c];
    rt[c] = rb * th[c] + rho[c] * (tb + th[c]);
  } else {
    rt[c] = base.rho ? base.rho[k] * th[c] + rho[c] * (base.th[k] + th[c]) : rho[c] * th[c];
  }
}

// ===========================================================================
// Warm rain + fallout, marching columns top-down: K24 (warm_rain.cu:36-120)
// on cell k, then the fallout sweep on the same cell (K25 nominal,
// warm_rain.cu:122-154, or K26 metric, 156-191), which reads the
// post-microphysics rain exactly like the reference's qr_old copy.
//
// A wave is 64 columns, and the waves of a work-group share them, each with a
// chunk of the levels (blockDim.y chunks; blockDim.z rows of such waves: one,
// but in the widest batched members): what falls into a chunk depends on
// the level above it only, which the wave adjusts a second time for itself.
// The update is in place, so every wave reads that level before any writes
// (they are all in the work-group).  One thread per column leaves too few
// waves to cover the loads of small and deep grids (figures at the launcher's
// rule).  CHUNKED: more chunks than one; whole columns take a kernel of their
// own, which the second adjustment's code made 3 to 5 % slower.
// ===========================================================================
template <class R, bool TERRAIN, bool CHUNKED>
__device__ __forceinline__ void warm_rain_body(const WarmRainArgs<R>& a, const VBlock& vb) {
  const Geo g = a.g;
  int bx, by;
  xcd_block2d(vb, bx, by);
  const int ic = bx * 64 + static_cast<int>(threadIdx.x);
  const int jc = by * static_cast<int>(blockDim.z) + static_cast<int>(threadIdx.z);
  const bool in = ic < g.nx && jc < g.ny;
  const int i = ic < g.nx ? ic : g.nx - 1, j = jc < g.ny ? jc : g.ny - 1;
  const int nch = CHUNKED ? static_cast<int>(blockDim.y) : 1;
  const int chunk = CHUNKED ? static_cast<int>(threadIdx.y) : 0;
  const int k0 = (g.nz * chunk) / nch, k1 = (g.nz * (chunk + 1)) / nch;
  const R dt = a.dt;
  R inc = 0;
  const R dz_nom = rmax(a.depth, R(1.0e-3));
  const R frac_nom = rmin(rmax(a.vt * dt / dz_nom, R(0)), R(1));
  // The nominal sweep leaves the column alone when nothing falls out
  // (warm_rain.cu:134-136); the metric sweep has no such exit.
  const bool nominal = a.fallout == 1 && frac_nom > R(0), metric = a.fallout == 2;
  const R rdz_nom = R(1) / dz_nom;
  const MicroCfg<R> mc{dt, a.relax, a.thr, a.krate, a.erate, a.kacc, a.heat};
  const size_t plane = static_cast<size_t>(g.pxc) * g.pyc;
  struct Lv {
    R rho, rt, qv, qc, qr;
  };
  auto load = [&](size_t cc) -> Lv { return {a.rho[cc], a.rt[cc], a.qv[cc], a.qc[cc], a.qr[cc]}; };
  const bool pert = a.base.rho != nullptr;
  // The adjusted cell: perturbation form: full rho and rho*theta for the
  // microphysics; the stored departure of rho*theta then changes by rho *
  // dtheta only.
  struct Adjusted {
    R rt, rqv, rqc, rqr;
  };
  auto adjust = [&](const Lv& cur, int k) -> Adjusted {
    const R rho = rmax(pert ? cur.rho + a.base.rho[k] : cur.rho, R(1.0e-6));
    const R rt0 = pert ? cur.rt + a.base.rt[k] : cur.rt;
    MicroCell<R> m = micro_prepare(rho, rt0, cur.qv, cur.qc, cur.qr);
    const R th0 = m.th;
    micro_apply(m, mc);
    return {pert ? cur.rt + rho * (m.th - th0) : rho * m.th, rho * m.qv, rho * m.qc, rho * m.qr};
  };
  // What stays of a cell's rain, and what it lets fall (into inc).
  auto fall = [&](R rqr, int k) -> R {
    if (nominal) {
      const R old = rmax(rqr, R(0)) * dz_nom;
      const R out = frac_nom * old;
      rqr = qdivc(old - out + inc, dz_nom, rdz_nom);
      inc = out;
    } else if (metric) {
      const R idz = rmax(TERRAIN ? a.idz_c[g.metric(i, j, k)] : a.lev_idz_c[k], R(1.0e-6));
      const R dz = qrcp(idz);
      const R frac = rmin(rmax(a.vt * dt * idz, R(0)), R(1));
      const R old = rmax(rqr, R(0)) * dz;
      const R out = frac * old;
      rqr = (old - out + inc) * idz;
      inc = out;
    }
    return rqr;
  };
  // The loads of the level three below are issued before the current level's
  // arithmetic.
  size_t c = g.cell(i, j, k1 - 1);
  Lv l1{}, l2{}, l3{}, above{};
  if (CHUNKED && k1 < g.nz) above = load(c + plane);
  if (k1 > k0) l1 = load(c);
  if (k1 - 1 > k0) l2 = load(c - plane);
  if (k1 - 2 > k0) l3 = load(c - 2 * plane);
  if constexpr (CHUNKED) {
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the level above has been read
    __syncthreads();
  }
  if (!in) return;
  if (CHUNKED && k1 < g.nz && (nominal || metric)) fall(adjust(above, k1).rqr, k1);
  for (int k = k1 - 1; k >= k0; --k) {
    const Lv cur = l1;
    l1 = l2;
    l2 = l3;
    if (k - 3 >= k0) l3 = load(c - 3 * plane);
    const Adjusted n = adjust(cur, k);
    a.qv[c] = n.rqv;
    a.qc[c] = n.rqc;
    a.rt[c] = n.rt;
    a.qr[c] = fall(n.rqr, k);
    c -= plane;
  }
  if (k0 > 0) return;
  if (nominal || metric) a.precip[static_cast<size_t>(j) * g.nx + i] += inc;
}

template <class R, bool TERRAIN, bool CHUNKED>
__global__ __launch_bounds__(512) void k_warm_rain(WarmRainArgs<R> a) {
  // (a row of 64-column waves after the other in x: the launch's y extent
  // would limit the rows)
  const int gx = (a.g.nx + 63) / 64, b = static_cast<int>(blockIdx.x);
  const int rows = static_cast<int>(blockDim.z);
  warm_rain_body<R, TERRAIN, CHUNKED>(a, VBlock{b % gx, b / gx, gx, (a.g.ny + rows - 1) / rows});
}
template <class R, bool TERRAIN, bool CHUNKED>
__global__ __launch_bounds__(512) void k_warm_rain_batch(const WarmRainItem<R>* items, BatchMap bm) {
  VBlock vb;
  const WarmRainItem<R>* it = batch_member(items, bm, vb);
  if (!it) return;
  const WarmRainArgs<R> a = it->a;
  warm_rain_body<R, TERRAIN, CHUNKED>(a, vb);
}

// ===========================================================================
// Halo fill / interface averaging (1x1 layout) and the multi-rank exchange.
// ===========================================================================
template <class R>
__global__ void k_halo_fill(Geo g, int orient, R* f) {
  // orient: 0 cell, 1 x-face, 2 y-face, 3 z-face
  const int fx = g.nx + (orient == 1), fy = g.ny + (orient == 2), fz = g.nz + (orient == 3);
  const int px = fx + 2 * g.h, py = fy + 2 * g.h;
  const size_t n = static_cast<size_t>(px) * py * fz;
  const size_t a = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (a >= n) return;
  const int ii = static_cast<int>(a % px) - g.h;
  const int jj = static_cast<int>((a / px) % py) - g.h;
  const int k = static_cast<int>(a / (static_cast<size_t>(px) * py));
  if (ii >= 0 && ii < fx && jj >= 0 && jj < fy) return;
  const int si = orient == 1 ? map_face(ii, g.nx, g.per_x) : map_cell(ii, g.nx, g.per_x);
  const int sj = orient == 2 ? map_face(jj, g.ny, g.per_y) : map_cell(jj, g.ny, g.per_y);
  f[a] = (si < 0 || sj < 0) ? R(0)
                            : f[(static_cast<size_t>(k) * py + (sj + g.h)) * px + (si + g.h)];
}

template <class R>
__global__ void k_sync_interfaces(Geo g, int orient, R* f) {
  // synchronize_face_owned_interfaces_impl for a 1x1 periodic layout
  // (halo_exchange.cpp:255-283): face n and face 0 both take their average.
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (orient == 1) {
    if (a >= g.ny * g.nz) return;
    const int j = a % g.ny, k = a / g.ny;
    const size_t e = g.xf(g.nx, j, k), w = g.xf(0, j, k);
    const R avg = R(0.5) * (f[e] + f[w]);
    f[e] = avg;
    f[w] = avg;
  } else {
    if (a >= g.nx * g.nz) return;
    const int i = a % g.nx, k = a / g.nx;
    const size_t nn = g.yf(i, g.ny, k), s = g.yf(i, 0, k);
    const R avg = R(0.5) * (f[nn] + f[s]);
    f[nn] = avg;
    f[s] = avg;
  }
}

// Multi-rank exchange (halo_exchange.cpp:32-116, 148-215, 313-373, 563-620):
// phase 0 fills the x ghosts of owned rows, phase 1 the y ghost rows (which
// include the x ghosts).  d: 13 ints per rank + 4 neighbour ranks.
template <class R>
__global__ void k_exchange_layout(int phase, int orient, int nranks, const int* d, R* const* F,
                                  int maxn) {
  const int rank = blockIdx.y;
  if (rank >= nranks) return;
  const int* D = d + rank * 17;
  const int h = D[8], nxl = D[10] - D[9], nyl = D[12] - D[11];
  const int fx = nxl + (orient == 1), fy = nyl + (orient == 2), fz = D[7] + (orient == 3);
  const int px = fx + 2 * h, py = fy + 2 * h;
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  R* f = F[rank];
  auto at = [&](R* base, int ppx, int ppy, int i, int j, int k) -> R& {
    return base[(static_cast<size_t>(k) * ppy + (j + h)) * ppx + (i + h)];
  };
  if (phase == 0) {
    // x phase: for k < fz, j < fy, hh < h: west ghost (-h+hh) and east ghost (fx+hh)
    const int total = fz * fy * h;
    if (a >= total) return;
    const int hh = a % h, j = (a / h) % fy, k = a / (h * fy);
    const int west = D[13], east = D[14];
    // west ghost <- west neighbour's east send
    if (west >= 0) {
      const int* W = d + west * 17;
      const int wnxl = W[10] - W[9], wnyl = W[12] - W[11];
      const int wfx = wnxl + (orient == 1), wfy = wnyl + (orient == 2);
      const int ei = orient == 1 ? wnxl - h + hh : wfx - h + hh;
      at(f, px, py, -h + hh, j, k) = at(F[west], wfx + 2 * h, wfy + 2 * h, ei, j, k);
    } else {
      at(f, px, py, -h + hh, j, k) = R(0);
    }
    if (east >= 0) {
      const int* E = d + east * 17;
      const int enxl = E[10] - E[9], enyl = E[12] - E[11];
      const int efx = enxl + (orient == 1), efy = enyl + (orient == 2);
      const int wi = orient == 1 ? 1 + hh : hh;
      at(f, px, py, fx + hh, j, k) = at(F[east], efx + 2 * h, efy + 2 * h, wi, j, k);
    } else {
      at(f, px, py, fx + hh, j, k) = R(0);
    }
  } else {
    const int total = fz * h * (fx + 2 * h);
    if (a >= total) return;
    const int i = a % (fx + 2 * h) - h, hh = (a / (fx + 2 * h)) % h, k = a / ((fx + 2 * h) * h);
    const int south = D[15], north = D[16];
    if (south >= 0) {
      const int* S = d + south * 17;
      const int snxl = S[10] - S[9], snyl = S[12] - S[11];
      const int sfx = snxl + (orient == 1), sfy = snyl + (orient == 2);
      const int nj = orient == 2 ? snyl - h + hh : sfy - h + hh;
      at(f, px, py, i, -h + hh, k) = at(F[south], sfx + 2 * h, sfy + 2 * h, i, nj, k);
    } else {
      at(f, px, py, i, -h + hh, k) = R(0);
    }
    if (north >= 0) {
      const int* N = d + north * 17;
      const int nnxl = N[10] - N[9], nnyl = N[12] - N[11];
      const int nfx = nnxl + (orient == 1), nfy = nnyl + (orient == 2);
      const int sj = orient == 2 ? 1 + hh : hh;
      at(f, px, py, i, fy + hh, k) = at(F[north], nfx + 2 * h, nfy + 2 * h, i, sj, k);
    } else {
      at(f, px, py, i, fy + hh, k) = R(0);
    }
  }
  (void)maxn;
}

// ===========================================================================
// Boundary strips / relaxation on the outermost owned strips of one field
// (boundary_conditions.cpp:9-161; relaxation is the extension documented in
// the header).  orient as in k_halo_fill.  Threads cover the frame of
// cells within wx (wy) of the open x (y) sides when it is narrower than the
// field (wx = 0: the whole field): x strips of every row, then y strips of
// the columns between them; each cell's test and update are the same
// either way.
// ===========================================================================
template <class R>
__global__ void k_boundary(Geo g, int orient, R* f, const R* ref, int mode, R width, int wx,
                           int wy) {
  const int fx = g.nx + (orient == 1), fy = g.ny + (orient == 2), fz = g.nz + (orient == 3);
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  int i, j, k;
  if (wx > 0 || wy > 0) {
    const int wx0 = wx > 0 ? wx : 0;
    const int nxs = wx > 0 ? 2 * wx * fy : 0;
    const int nys = wy > 0 ? 2 * wy * (fx - 2 * wx0) : 0;
    const int per = nxs + nys;
    if (a >= per * fz) return;
    k = a / per;
    int r = a % per;
    if (r < nxs) {
      const int ii = r % (2 * wx);
      j = r / (2 * wx);
      i = ii < wx ? ii : fx - 2 * wx + ii;
    } else {
      r -= nxs;
      const int jj = r % (2 * wy);
      i = wx0 + r / (2 * wy);
      j = jj < wy ? jj : fy - 2 * wy + jj;
    }
  } else {
    if (a >= fx * fy * fz) return;
    i = a % fx;
    j = (a / fx) % fy;
    k = a / (fx * fy);
  }
  const bool w = !g.per_x, e = !g.per_x, s = !g.per_y, n = !g.per_y;
  const int px = fx + 2 * g.h, py = fy + 2 * g.h;
  const size_t idx = (static_cast<size_t>(k) * py + (j + g.h)) * px + (i + g.h);
  if (mode == 1) {
    if ((w && i == 0) || (e && i == fx - 1) || (s && j == 0) || (n && j == fy - 1)) f[idx] = ref[idx];
    return;
  }
  double dmin = 1e30;
  if (w) dmin = fmin(dmin, static_cast<double>(i));
  if (e) dmin = fmin(dmin, static_cast<double>(fx - 1 - i));
  if (s) dmin = fmin(dmin, static_cast<double>(j));
  if (n) dmin = fmin(dmin, static_cast<double>(fy - 1 - j));
  if (dmin >= static_cast<double>(width)) return;
  const double a0 = 1.0 - dmin / static_cast<double>(width);
  const R wgt = static_cast<R>(a0 * a0);
  f[idx] = f[idx] + wgt * (ref[idx] - f[idx]);
}

// ===========================================================================
// Metric construction (grid_metrics.hpp:184-236): one thread per column,
// FP64 arithmetic without contraction so the stored values match a host
// build of the same formulas.
// ===========================================================================
template <class R>
__global__ void k_metrics(Geo g, const double* zif, const double* zc, const double* wif,
                          const double* wc, const float* terrain, R* zif_m, R* zc_m, R* idz_c,
                          R* idz_f, R* slope_x, R* slope_y, R* terr_out) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= g.nx || j >= g.ny) return;
  auto tr = [&](int ii, int jj) -> float { return terrain ? terrain[static_cast<size_t>(jj) * g.nx + ii] : 0.0f; };
  auto wi = [&](int ii) { return g.per_x ? map_cell(ii, g.nx, 1) : min(max(ii, 0), g.nx - 1); };
  auto wj = [&](int jj) { return g.per_y ? map_cell(jj, g.ny, 1) : min(max(jj, 0), g.ny - 1); };
  const float th = tr(i, j);
  const size_t c2 = static_cast<size_t>(j) * g.nx + i;
  terr_out[c2] = static_cast<R>(th);
  const double ddx = (static_cast<double>(tr(wi(i + 1), j)) - static_cast<double>(tr(wi(i - 1), j))) /
                     (g.per_x || (i > 0 && i + 1 < g.nx) ? 2.0 * g.dx : g.dx);
  const double ddy = (static_cast<double>(tr(i, wj(j + 1))) - static_cast<double>(tr(i, wj(j - 1)))) /
                     (g.per_y || (j > 0 && j + 1 < g.ny) ? 2.0 * g.dy : g.dy);
  slope_x[c2] = static_cast<R>(ddx);
  slope_y[c2] = static_cast<R>(ddy);
  const double thd = static_cast<double>(th);
  for (int k = 0; k <= g.nz; ++k) {
    const double prod = wif[k] * thd;
    zif_m[g.metric(i, j, k)] = static_cast<R>(zif[k] + prod);
    if (k == 0 || k == g.nz) {
      idz_f[g.metric(i, j, k)] = R(0);
    } else {
      const double hi = zc[k] + wc[k] * thd;
      const double lo = zc[k - 1] + wc[k - 1] * thd;
      const double dzf = hi - lo;
      idz_f[g.metric(i, j, k)] = static_cast<R>(1.0 / fmax(dzf, 1.0e-6));
    }
  }
  for (int k = 0; k < g.nz; ++k) {
    const double prod = wc[k] * thd;
    zc_m[g.metric(i, j, k)] = static_cast<R>(zc[k] + prod);
    const double dzc = static_cast<double>(zif_m[g.metric(i, j, k + 1)]) -
                       static_cast<double>(zif_m[g.metric(i, j, k)]);
    idz_c[g.metric(i, j, k)] = static_cast<R>(1.0 / fmax(dzc, 1.0e-6));
  }
}

// The FP32 arithmetic helpers, elementwise (gwm_fp32_math).
__global__ void k_fp32_math(int fn, const float* x, float* y, size_t n) {
  const size_t t = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const float v = x[t];
  float r;
  switch (fn) {
    case 0: r = qpow(v, 1.0f / (1.0f - Phys<float>::kappa)); break;
    case 1: r = qpow(v, Phys<float>::kappa); break;
    case 2: r = qexp(v); break;
    case 3: r = qlog1p(v); break;
    case 4: r = qexpm1(v); break;
    case 6: r = p_pert(v, 1.0f, 1.0f); break;  // (1 + x)^gamma - 1
    default: r = qrcp(v); break;
  }
  y[t] = r;
}

template <class R>
__global__ void k_copy(const R* src, R* dst, size_t n) {
  const size_t a = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (a < n) dst[a] = src[a];
}
// Several buffers in one launch: chunks of 16 KiB, four 16-byte loads of each
// thread in flight, dealt round robin to at most 1024 work-groups.  A copy per
// buffer costs a state's copy nine launches, four to five us each where the
// fields are small: a subcycle of 331 x 203 x 50 from a copied state 226 -> 214
// us, a surrogate call of 256 x 256 x 64 414 -> 384 us.
constexpr unsigned kCopyWords = 4096;  // of a chunk
__global__ __launch_bounds__(256) void k_copy_jobs(CopyJobs J) {
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  const unsigned t = threadIdx.x, total = J.chunk0[J.n];
  int q = 0;
  for (unsigned b = blockIdx.x; b < total; b += gridDim.x) {
    while (b >= J.chunk0[q + 1]) ++q;
    const size_t w0 = static_cast<size_t>(b - J.chunk0[q]) * kCopyWords;
    const size_t left = J.words[q] - w0;
    const unsigned* s = static_cast<const unsigned*>(J.src[q]) + w0;
    unsigned* d = static_cast<unsigned*>(J.dst[q]) + w0;
    const bool wide =
        ((reinterpret_cast<uintptr_t>(s) | reinterpret_cast<uintptr_t>(d)) & 15) == 0;
    if (wide && left >= kCopyWords) {
      u4 v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = reinterpret_cast<const u4*>(s)[t + 256 * e];
#pragma unroll
      for (int e = 0; e < 4; ++e) reinterpret_cast<u4*>(d)[t + 256 * e] = v[e];
    } else {
      const unsigned n = static_cast<unsigned>(left < kCopyWords ? left : kCopyWords);
      for (unsigned e = t; e < n; e += 256) d[e] = s[e];
    }
  }
}
template <class R>
__global__ void k_fill(R* dst, size_t n, R v) {
  const size_t a = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (a < n) dst[a] = v;
}

// ===========================================================================
// Launchers
// ===========================================================================
namespace {
inline dim3 cell_grid(const Geo& g, dim3 b) {
  return dim3((g.nx + b.x - 1) / b.x, (g.ny + b.y - 1) / b.y, g.nz);
}
inline unsigned blocks_for(size_t n, unsigned b) { return static_cast<unsigned>((n + b - 1) / b); }
}  // namespace

template <class R>
void launch_level_partials(hipStream_t st, const Geo& g, const R* rho, const R* aux, int mode,
                           double* partials, int* nchunk_out, Base<R> base) {
  const int nchunk = level_partials_chunks(g.ny);
  *nchunk_out = nchunk;
  if (recorder()) {
    record_launch(reinterpret_cast<const void*>(&k_level_partials_batch<R>), dim3(256), 0,
                  PartialsItem<R>{g, rho, aux, mode, partials, base, 0, 0}, nchunk, g.nz);
    return;
  }
  hipLaunchKernelGGL(k_level_partials<R>, dim3(nchunk, g.nz), dim3(256), 0, st, g, rho, aux, mode,
                     partials, base);
}
int level_partials_chunks(int ny) { return (ny + kPartialRows - 1) / kPartialRows; }
template <class R>
void launch_level_finalize(hipStream_t st, int nz, int nchunk, const double* partials, int mode,
                           double count, R* o0, R* o1) {
  if (recorder()) {
    record_launch(reinterpret_cast<const void*>(&k_level_finalize_batch<R>),
                  dim3(kFinalizeThreads), 0,
                  FinalizeItem<R>{nz, nchunk, partials, mode, count, o0, o1, 0, 0}, nz, 1);
    return;
  }
  hipLaunchKernelGGL(k_level_finalize<R>, dim3(nz), dim3(kFinalizeThreads), 0, st, nz, nchunk, partials,
                     mode, count, o0, o1);
}
template <class R>
void launch_pressure(hipStream_t st, const Geo& g, const R* rho, const R* rt, R* p) {
  if (refuse_record("pressure")) return;
  hipLaunchKernelGGL(k_pressure<R>, dim3(blocks_for(g.cell_total(), 256)), dim3(256), 0, st, g,
                     rho, rt, p);
}
template <class R>
void launch_theta(hipStream_t st, const Geo& g, const R* rho, const R* rt, R* th, Base<R> base) {
  if (refuse_record("theta")) return;
  const dim3 b(64, 4, 1);
  hipLaunchKernelGGL(k_theta<R>, cell_grid(g, b), b, 0, st, g, rho, rt, th, base);
}
template <class R>
void launch_rebuild_rt(hipStream_t st, const Geo& g, const R* rho, const R* th, R* rt,
                       Base<R> base) {
  if (refuse_record("rebuild_rt")) return;
  const dim3 b(64, 4, 1);
  hipLaunchKernelGGL(k_rebuild_rt<R>, cell_grid(g, b), b, 0, st, g, rho, th, rt, base);
}
template <class R>
void launch_warm_rain(hipStream_t st, const WarmRainArgs<R>& a, bool terrain) {
  // Enough waves to cover the loads, and no more than that: each chunk costs a
  // second adjustment of a level, so chunks keep some levels too.  By the
  // number of 64-column waves (of a batched launch, the member's).  Measured
  // with 1 / 2 / 4 / 8 chunks (us, nominal fallout):
  //   waves x levels   FP32                     FP64
  //   64 x 40          34, 21, 13, 11           46, 28, 17, 17
  //   1024 x 16        20, 16, 16, 17           26.6, 26.1, 28.5, 36
  //   1024 x 64        59, 44, 40, 41           86, 78, 78, 88
  //   4096 x 8         22, 24, 28, 28           42, 49, 60, 59
  //   4096 x 24        54, 56                   112, 113
  //   4096 x 64        144, 138, 146, 155       294, 297, 317, 342
  //   16384 x 8        65, 76, 91, 91           154, 183, 217, 219
  //   16384 x 32       285, 285, 284, 307       558, 586, 623, 759
  // and eight FP32 members of 192 to 896 waves in one batched launch 152, 124,
  // 119, 126.
  constexpr bool f64 = sizeof(R) == 8;
  const dim3 gr((a.g.nx + 63) / 64, a.g.ny);
  const long waves = static_cast<long>(gr.x) * gr.y;
  int chunks = waves >= 2048 ? (f64 ? 1 : 2) : waves >= 128 ? 4 : 8;
  const int levels = waves >= 2048 ? 16 : f64 && waves >= 128 ? 8 : 4;  // of a chunk
  while (chunks > 1 && a.g.nz < levels * chunks) chunks /= 2;
  // (a batched launch numbers a member's work-groups in kBatchBlockBits bits)
  const int rows = recorder() && waves >= (1L << kBatchBlockBits) ? 4 : 1;
  const dim3 b(64, chunks, rows);
  const unsigned gy = (gr.y + rows - 1) / rows;
  auto go = [&](auto t, auto c) {
    constexpr bool T = decltype(t)::value, C = decltype(c)::value;
    if (recorder())
      record_launch(reinterpret_cast<const void*>(&k_warm_rain_batch<R, T, C>), b, 0,
                    WarmRainItem<R>{a, 0, 0}, static_cast<int>(gr.x), static_cast<int>(gy));
    else
      hipLaunchKernelGGL((k_warm_rain<R, T, C>), dim3(gr.x * gy), b, 0, st, a);
  };
  using std::false_type;
  using std::true_type;
  if (terrain) chunks > 1 ? go(true_type{}, true_type{}) : go(true_type{}, false_type{});
  else chunks > 1 ? go(false_type{}, true_type{}) : go(false_type{}, false_type{});
}
template <class R>
void launch_halo_fill(hipStream_t st, const Geo& g, int orient, R* f) {
  if (refuse_record("halo_fill")) return;
  const int fx = g.nx + (orient == 1), fy = g.ny + (orient == 2), fz = g.nz + (orient == 3);
  const size_t n = static_cast<size_t>(fx + 2 * g.h) * (fy + 2 * g.h) * fz;
  hipLaunchKernelGGL(k_halo_fill<R>, dim3(blocks_for(n, 256)), dim3(256), 0, st, g, orient, f);
}
template <class R>
void launch_sync_interfaces(hipStream_t st, const Geo& g, int orient, R* f) {
  if (refuse_record("sync_interfaces")) return;
  const int n = orient == 1 ? g.ny * g.nz : g.nx * g.nz;
  hipLaunchKernelGGL(k_sync_interfaces<R>, dim3(blocks_for(n, 256)), dim3(256), 0, st, g, orient, f);
}
template <class R>
void launch_exchange_layout(hipStream_t st, int phase, int orient, int nranks, const int* d,
                            R* const* F, int max_elems) {
  hipLaunchKernelGGL(k_exchange_layout<R>, dim3(blocks_for(max_elems, 256), nranks), dim3(256), 0,
                     st, phase, orient, nranks, d, F, max_elems);
}
template <class R>
void launch_boundary(hipStream_t st, const Geo& g, int orient, R* f, const R* ref, int mode,
                     double width) {
  if (refuse_record("boundary")) return;
  const int fx = g.nx + (orient == 1), fy = g.ny + (orient == 2), fz = g.nz + (orient == 3);
  // frame widths: the cells a side can reach (the outermost one for strips,
  // distance < width for relaxation); the whole field when a frame would
  // cover it
  const int reach = mode == 1 ? 1 : (width > 0.0 ? static_cast<int>(std::ceil(width)) : 0);
  int wx = g.per_x ? 0 : reach, wy = g.per_y ? 0 : reach;
  size_t n = static_cast<size_t>(fx) * fy * fz;
  if ((wx > 0 || wy > 0) && 2 * wx < fx && 2 * wy < fy) {
    const size_t nxs = wx > 0 ? 2 * static_cast<size_t>(wx) * fy : 0;
    const size_t nys = wy > 0 ? 2 * static_cast<size_t>(wy) * (fx - 2 * wx) : 0;
    n = (nxs + nys) * fz;
  } else {
    wx = wy = 0;
  }
  if (n == 0) return;
  hipLaunchKernelGGL(k_boundary<R>, dim3(blocks_for(n, 256)), dim3(256), 0, st, g, orient, f, ref,
                     mode, static_cast<R>(width), wx, wy);
}
Recorder*& recorder() {
  static thread_local Recorder* r = nullptr;
  return r;
}

// Block partials of the allocation-free budget entry point
// (gwm_budget_sums_noalloc): a file-scope array, one copy per GPU, whose
// device address is resolved once per device by noalloc_scratch_setup.  The
// name is a host-side stand-in; host code uses only the resolved address.
static __device__ __align__(256) double scratch[kNoAllocScratchDoubles];

hipError_t noalloc_scratch_setup(int device, double** out) {
  static std::mutex mu;
  static double* addr[kNoAllocMaxDevices] = {};
  std::lock_guard<std::mutex> lock(mu);
  *out = nullptr;
  if (device < 0 || device >= kNoAllocMaxDevices) return hipErrorInvalidDevice;
  if (addr[device] == nullptr) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    addr[device] = static_cast<double*>(p);
  }
  *out = addr[device];
  return hipSuccess;
}
template <class R>
void launch_metrics(hipStream_t st, const Geo& g, const double* zif, const double* zc,
                    const double* wif, const double* wc, const float* terrain, R* zif_m, R* zc_m,
                    R* idz_c, R* idz_f, R* sx, R* sy, R* terr) {
  const dim3 b(64, 4, 1);
  hipLaunchKernelGGL(k_metrics<R>, dim3((g.nx + 63) / 64, (g.ny + 3) / 4), b, 0, st, g, zif, zc,
                     wif, wc, terrain, zif_m, zc_m, idz_c, idz_f, sx, sy, terr);
}
void launch_fp32_math(hipStream_t st, int fn, const float* x, float* y, size_t n) {
  hipLaunchKernelGGL(k_fp32_math, dim3(blocks_for(n, 256)), dim3(256), 0, st, fn, x, y, n);
}
template <class R>
void launch_copy(hipStream_t st, const R* src, R* dst, size_t n) {
  if (refuse_record("copy")) return;
  hipLaunchKernelGGL(k_copy<R>, dim3(blocks_for(n, 256)), dim3(256), 0, st, src, dst, n);
}
void launch_copy_jobs(hipStream_t st, CopyJobs j) {
  unsigned c = 0;
  for (int q = 0; q < j.n; ++q) {
    j.chunk0[q] = c;
    c += static_cast<unsigned>((j.words[q] + kCopyWords - 1) / kCopyWords);
  }
  j.chunk0[j.n] = c;
  if (c) hipLaunchKernelGGL(k_copy_jobs, dim3(c < 1024 ? c : 1024), dim3(256), 0, st, j);
}
template <class R>
void launch_fill(hipStream_t st, R* dst, size_t n, R v) {
  if (refuse_record("fill")) return;
  hipLaunchKernelGGL(k_fill<R>, dim3(blocks_for(n, 256)), dim3(256), 0, st, dst, n, v);
}

#define GWM_INSTANTIATE(R)                                                                          \
  template void launch_level_partials<R>(hipStream_t, const Geo&, const R*, const R*, int,        \
                                         double*, int*, Base<R>);                                 \
  template void launch_level_finalize<R>(hipStream_t, int, int, const double*, int, double, R*,   \
                                         R*);                                                     \
  template void launch_pressure<R>(hipStream_t, const Geo&, const R*, const R*, R*);             \
  template void launch_theta<R>(hipStream_t, const Geo&, const R*, const R*, R*, Base<R>);       \
  template void launch_rebuild_rt<R>(hipStream_t, const Geo&, const R*, const R*, R*, Base<R>);  \
  template void launch_warm_rain<R>(hipStream_t, const WarmRainArgs<R>&, bool);                  \
  template void launch_halo_fill<R>(hipStream_t, const Geo&, int, R*);                           \
  template void launch_sync_interfaces<R>(hipStream_t, const Geo&, int, R*);                     \
  template void launch_exchange_layout<R>(hipStream_t, int, int, int, const int*, R* const*, int); \
  template void launch_boundary<R>(hipStream_t, const Geo&, int, R*, const R*, int, double);     \
  template void launch_metrics<R>(hipStream_t, const Geo&, const double*, const double*,         \
                                  const double*, const double*, const float*, R*, R*, R*, R*, R*, \
                                  R*, R*);                                                        \
  template void launch_copy<R>(hipStream_t, const R*, R*, size_t);                               \
  template void launch_fill<R>(hipStream_t, R*, size_t, R);

GWM_INSTANTIATE(float)
GWM_INSTANTIATE(double)

}  // namespace gwm
