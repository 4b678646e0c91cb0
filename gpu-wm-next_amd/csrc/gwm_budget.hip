// gwm_budget.hip -- the budget sums of a state in one launch: compensated
// FP64 sums, extremes and non-finite counts of every prognostic field
// (summarize_dry_states, src/dycore/dry_diagnostics.cpp:11-96;
// summarize_runtime_state, src/core/runtime_summary.cpp:27-178).
//
// Work-groups are divided among jobs: the cell job reads rho and rho*theta
// (sums of both, extremes of rho and theta), one job per face field, the
// tracer job reads rho and up to three tracers (column paths and mixing-ratio
// extremes), the bucket job the precipitation bucket.  Every field is read
// once (rho twice), so the kernel is bound by those bytes: the 512 x 512 x 64
// FP32 state with three tracers (604 MB) takes 146 us (4.1 TB/s; the call
// 166 us), where fourteen reductions, each with its own pass, copy to the host
// and wait, took 2.2 ms.
// A wave takes whole rows (level and row index are scalar, no division per
// element) with several independent loads in flight per lane; 256 work-groups
// of 1024 threads keep the block records within 4096 doubles, the static
// array that the allocation-free entry point has.
#include "gwm_kernels.hpp"

namespace gwm {

namespace {

constexpr int kThreads = 1024, kWaves = kThreads / 64;

// Running sum with its compensation, extremes and non-finite count.
struct Acc {
  double s = 0.0, c = 0.0, mn = 1e300, mx = -1e300;
  int bad = 0;
  // TwoSum: the rounding error of every addition joins the compensation.
  __device__ void sum(double v) {
    const double t = s + v;
    const double b = t - s;
    c += (s - (t - b)) + (v - b);
    s = t;
  }
  __device__ void ext(double v) {
    mn = fmin(mn, v);
    mx = fmax(mx, v);
  }
  __device__ void join(const Acc& o) {
    sum(o.s);
    c += o.c;
    mn = fmin(mn, o.mn);
    mx = fmax(mx, o.mx);
    bad += o.bad;
  }
};

// One step of the wave reduction (the moves of wave_sum_to63: lane 63 ends
// with the whole wave, in a fixed order).
template <int CTRL, int ROWS>
__device__ inline void wave_step(Acc& a) {
  Acc o;
  o.s = dpp_f64<CTRL, ROWS>(a.s);
  o.c = dpp_f64<CTRL, ROWS>(a.c);
  o.mn = dpp_f64<CTRL, ROWS>(a.mn);
  o.mx = dpp_f64<CTRL, ROWS>(a.mx);
  o.bad = __builtin_amdgcn_mov_dpp(a.bad, CTRL, ROWS, 0xF, false);
  a.join(o);
}

// Block total of one accumulator (valid in thread 0).
typedef double Shared[5][kWaves];
__device__ inline Acc block_join(Acc a, Shared& sh) {
  wave_step<0xB1, 0xF>(a);
  wave_step<0x4E, 0xF>(a);
  wave_step<0x141, 0xF>(a);
  wave_step<0x140, 0xF>(a);
  wave_step<0x142, 0xA>(a);
  wave_step<0x143, 0xC>(a);
  const int t = threadIdx.x, w = t >> 6;
  __syncthreads();  // the last call's records have been read
  if ((t & 63) == 63) {
    sh[0][w] = a.s;
    sh[1][w] = a.c;
    sh[2][w] = a.mn;
    sh[3][w] = a.mx;
    sh[4][w] = static_cast<double>(a.bad);
  }
  __syncthreads();
  Acc r;
  if (t == 0) {
    for (int q = 0; q < kWaves; ++q) {
      Acc o;
      o.s = sh[0][q];
      o.c = sh[1][q];
      o.mn = sh[2][q];
      o.mx = sh[3][q];
      o.bad = static_cast<int>(sh[4][q]);
      r.join(o);
    }
  }
  return r;
}

__device__ inline void put(double* out, const Acc& a) {
  if (threadIdx.x != 0) return;
  out[0] = a.s;
  out[1] = a.c;
  out[2] = a.mn;
  out[3] = a.mx;
  out[4] = static_cast<double>(a.bad);
}

// Quotients by a shared reciprocal (rcp_newton of a positive normal b): the
// product corrected with its exact residual, which are the division's own
// steps without its scaling of the operands (identical results for 7001
// quotients as near to a tie as there are); an operand that is not finite
// gives a quotient that is not.  Five instructions for b and three a quotient
// against about thirteen each.
__device__ inline double quot(double a, double b, double r) {
  const double q = a * r;
  return __builtin_fma(__builtin_fma(-q, b, a), r, q);
}

// A value that is not finite is counted, and kept out of the sums and
// extremes, which then describe the finite values.  CHECK = false leaves the
// test out: a NaN or infinity then shows in the totals, and the work-group
// goes over its rows again with it (k_budget).
template <bool CHECK>
__device__ inline bool finite2(double a, double b) {
  return !CHECK || (isfinite(a) && isfinite(b));
}

// Rows of a field with fx x fy x fz owned elements, taken wave by wave:
// row(k, j, offset of element 0).  px, py: row pitch and rows of a level of
// the storage, h the halo.
template <class F>
__device__ inline void for_rows(int wave, int waves, int fy, int fz, int px, int py, int h, F row) {
  const int rows = fy * fz;
  for (int r = wave; r < rows; r += waves) {
    const int k = r / fy, j = r - k * fy;
    row(k, j, static_cast<unsigned>((k * py + (j + h)) * px + h));
  }
}

// Elements i = lane, lane + 64, ... of a row in batches of U independent
// loads.  A whole batch is straight-line code (a test per element would put
// each load behind a branch, and a wait behind each load); the rest of the
// row takes batches of half the size, down to single elements.
template <int U, class L, class F>
__device__ inline void along(int fx, L load, F use, int i0 = 0) {
  const int lane = threadIdx.x & 63;
  if constexpr (U == 1) {
    for (int i = i0 + lane; i < fx; i += 64) use(load(i));
  } else {
    for (; i0 + 64 * U <= fx; i0 += 64 * U) {
      decltype(load(0)) v[U];
#pragma unroll
      for (int q = 0; q < U; ++q) v[q] = load(i0 + lane + 64 * q);
#pragma unroll
      for (int q = 0; q < U; ++q) use(v[q]);
    }
    along<U / 2>(fx, load, use, i0);
  }
}

}  // namespace

// One pass of work-group blk of nblk over its job's rows, the records to
// out.  Returns (thread 0) whether every total is finite.
// TERRAIN: 1 / dz per cell, and per-cell bases in the perturbation form.
// NTR: tracers (at most 3); reading rho in the place of missing ones, their
// results unused, made one tracer dearer than three (512 x 512 x 64 FP32: 184,
// 153 and 163 us for one, two and three tracers; now 131, 150 and 163).
template <class R, bool CHECK, bool TERRAIN, int NTR>
__device__ __forceinline__ bool budget_pass(const BudgetArgs<R>& a, int job, int blk, int nblk,
                                            double* out, Shared& sh) {
  const Geo& g = a.g;
  const int wave = __builtin_amdgcn_readfirstlane(blk * kWaves + static_cast<int>(threadIdx.x >> 6));
  const int waves = nblk * kWaves;
  const bool pert = a.base.rho != nullptr;
  const bool pert3 = TERRAIN && a.base.drho != nullptr;

  if (job == 0) {
    struct V {
      R r, t, dr, dt;
    };
    Acc ar, at, ath;
    for_rows(wave, waves, g.ny, g.nz, g.pxc, g.pyc, g.h, [&](int k, int, unsigned o) {
      // perturbation form: extremes of the full values, sums of the departures
      const double rb = pert ? static_cast<double>(a.base.rho[k]) : 0.0;
      const double tb = pert ? static_cast<double>(a.base.rt[k]) : 0.0;
      const double thb = pert3 ? static_cast<double>(a.base.th[k]) : 0.0;
      along<4>(
          g.nx,
          [&](int i) {
            V v{ld32(a.rho, o + i), ld32(a.rt, o + i), R(0), R(0)};
            if (TERRAIN && pert3) {
              v.dr = ld32(a.base.drho, o + i);
              v.dt = ld32(a.base.dth, o + i);
            }
            return v;
          },
          [&](const V& v) {
            const double r = static_cast<double>(v.r), t = static_cast<double>(v.t);
            const double cb = pert3 ? rb + static_cast<double>(v.dr) : rb;
            const double cbt = pert3 ? cb * (thb + static_cast<double>(v.dt)) : tb;
            const double fr = pert ? r + cb : r, ft = pert ? t + cbt : t;
            if (finite2<CHECK>(fr, r)) {
              ar.sum(r);
              ar.ext(fr);
            } else {
              ++ar.bad;
            }
            if (finite2<CHECK>(ft, t)) at.sum(t);
            else ++at.bad;
            const double d = fmax(fr, 1.0e-12);
            const double th = CHECK ? ft / d : quot(ft, d, rcp_newton(d));
            if (finite2<CHECK>(ft, th)) ath.ext(th);
            else ++ath.bad;
            if (!CHECK) ath.s += th;  // shows a theta that is not finite
          });
    });
    ar = block_join(ar, sh);
    at = block_join(at, sh);
    ath = block_join(ath, sh);
    put(out, ar);
    put(out + 5, at);
    put(out + 10, ath);
    return isfinite(ar.s) && isfinite(at.s) && isfinite(ath.s);
  } else if (job <= 3) {
    const R* f = a.face[job - 1];
    const int fx = g.nx + (job == 1), fy = g.ny + (job == 2), fz = g.nz + (job == 3);
    Acc x;
    for_rows(wave, waves, fy, fz, fx + 2 * g.h, fy + 2 * g.h, g.h, [&](int, int, unsigned o) {
      along<8>(
          fx, [&](int i) { return ld32(f, o + i); },
          [&](R u) {
            const double v = static_cast<double>(u);
            if (finite2<CHECK>(v, v)) {
              x.sum(v);
              x.ext(v);
            } else {
              ++x.bad;
            }
          });
    });
    x = block_join(x, sh);
    put(out, x);
    return isfinite(x.s);
  } else if (job == 4 && NTR > 0) {
    constexpr int N = NTR > 0 ? NTR : 1;
    struct V {
      R r, dr, z, q[N];
    };
    Acc path[N], mix[N];
    for_rows(wave, waves, g.ny, g.nz, g.pxc, g.pyc, g.h, [&](int k, int j, unsigned o) {
      const double rb = pert ? static_cast<double>(a.base.rho[k]) : 0.0;
      const unsigned m = static_cast<unsigned>((k * g.ny + j) * g.nx);
      const R idz = TERRAIN ? R(1) : a.idz_lev[k];
      const double dz = 1.0 / static_cast<double>(idz);
      along<(N < 3 ? 4 : 2)>(
          g.nx,
          [&](int i) {
            V v{};
            v.r = ld32(a.rho, o + i);
            if (TERRAIN && pert3) v.dr = ld32(a.base.drho, o + i);
            if (TERRAIN) v.z = ld32(a.idz3, m + i);
#pragma unroll
            for (int t = 0; t < N; ++t) v.q[t] = ld32(a.q[t], o + i);
            return v;
          },
          [&](const V& v) {
            double r = static_cast<double>(v.r);
            if (pert) r += rb + (pert3 ? static_cast<double>(v.dr) : 0.0);
            const double d = TERRAIN ? 1.0 / static_cast<double>(v.z) : dz;
            r = fmax(r, 1.0e-12);
            const double ir = rcp_newton(r);
#pragma unroll
            for (int t = 0; t < N; ++t) {
              const double q = static_cast<double>(v.q[t]);
              const double p = q * d, x = CHECK ? q / r : quot(q, r, ir);
              if (finite2<CHECK>(q, p)) path[t].sum(p);
              else ++path[t].bad;
              if (finite2<CHECK>(q, x)) mix[t].ext(x);
              else ++mix[t].bad;
              if (!CHECK) mix[t].s += x;  // shows a ratio that is not finite
            }
          });
    });
    bool ok = true;
#pragma unroll
    for (int t = 0; t < N; ++t) {
      // the path's extremes are not reported: its record carries the mixing
      // ratio's instead, and the ratio's non-finite count follows
      Acc p = block_join(path[t], sh);
      const Acc x = block_join(mix[t], sh);
      p.mn = x.mn;
      p.mx = x.mx;
      put(out + 6 * t, p);
      if (threadIdx.x == 0) out[6 * t + 5] = static_cast<double>(x.bad);
      ok = ok && isfinite(p.s) && isfinite(x.s);
    }
    return ok;
  } else {
    Acc x;
    int wet = 0;
    const int n = g.nx * g.ny;
    for (int e = blk * kThreads + static_cast<int>(threadIdx.x); e < n; e += nblk * kThreads) {
      const double v = static_cast<double>(a.precip[e]);
      if (finite2<CHECK>(v, v)) {
        x.sum(v);
        x.ext(v);
        wet += v > 0.0;
      } else {
        ++x.bad;
      }
    }
    // the count of positive columns travels as the count of another record
    Acc w;
    w.bad = wet;
    x = block_join(x, sh);
    w = block_join(w, sh);
    put(out, x);
    if (threadIdx.x == 0) out[5] = static_cast<double>(w.bad);
    return isfinite(x.s);
  }
}

template <class R, bool TERRAIN, int NTR>
__global__ __launch_bounds__(kThreads) void k_budget(BudgetArgs<R> a) {
  __shared__ Shared sh;
  __shared__ int again;
  int job = 0;
  while (job + 1 < kBudgetJobs && static_cast<int>(blockIdx.x) >= a.block0[job + 1]) ++job;
  const int blk = static_cast<int>(blockIdx.x) - a.block0[job];
  const int nblk = a.block0[job + 1] - a.block0[job];
  double* out = a.part + a.part0[job] + static_cast<size_t>(blk) * a.record[job];
  const bool ok = budget_pass<R, false, TERRAIN, NTR>(a, job, blk, nblk, out, sh);
  if (threadIdx.x == 0) again = !ok;
  __syncthreads();
  if (again) budget_pass<R, true, TERRAIN, NTR>(a, job, blk, nblk, out, sh);
}

// Work-groups of the jobs (of 256 in all) about in proportion to the bytes
// and divisions of each: the cell job reads two fields and divides once per
// cell, a face job reads one field, the tracer job one more than it has
// tracers and divides once for each.
template <class R>
int budget_layout(BudgetArgs<R>& a) {
  const int weight[kBudgetJobs] = {28, 12, 12, 12, a.ntr > 0 ? 10 + 14 * a.ntr : 0, 2};
  const int record[kBudgetJobs] = {15, 5, 5, 5, 6 * a.ntr, 6};
  int total = 0, blocks = 0, doubles = 0;
  for (int w : weight) total += w;
  for (int q = 0; q < kBudgetJobs; ++q) {
    a.block0[q] = blocks;
    a.part0[q] = doubles;
    a.record[q] = record[q];
    const int nb = weight[q] == 0 ? 0 : (256 * weight[q]) / total > 0 ? (256 * weight[q]) / total : 1;
    blocks += nb;
    doubles += nb * record[q];
  }
  a.block0[kBudgetJobs] = blocks;
  a.part0[kBudgetJobs] = doubles;
  return blocks;
}

template <class R>
void launch_budget(hipStream_t st, const BudgetArgs<R>& a) {
  if (refuse_record("budget")) return;
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(a.block0[kBudgetJobs]), dim3(kThreads), 0, st, a);
  };
  auto form = [&](auto terrain) {
    constexpr bool T = decltype(terrain)::value;
    switch (a.ntr) {
      case 0: go(k_budget<R, T, 0>); break;
      case 1: go(k_budget<R, T, 1>); break;
      case 2: go(k_budget<R, T, 2>); break;
      default: go(k_budget<R, T, 3>); break;
    }
  };
  if (a.idz3) form(std::true_type{});
  else form(std::false_type{});
}

template int budget_layout<float>(BudgetArgs<float>&);
template int budget_layout<double>(BudgetArgs<double>&);
template void launch_budget<float>(hipStream_t, const BudgetArgs<float>&);
template void launch_budget<double>(hipStream_t, const BudgetArgs<double>&);

}  // namespace gwm
