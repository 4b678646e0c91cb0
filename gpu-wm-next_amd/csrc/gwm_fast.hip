// gwm_fast.hip -- column-marching fast substep for gfx950.
//
// One substep of apply_local_split_explicit_fast_modes
// (src/dycore/dry_fast_modes.cu:495-652): K10 + K20 pressure from rho and the
// fixed theta, K11 column hydrostatic reference (terrain), K12/K13
// horizontal pressure gradient, K14 vertical perturbation branch, K15
// density from the divergence of (m - m_base), and K10 rho*theta rebuild on
// the last substep.  Arithmetic is the step kernels' q* forms
// (gwm_internal.hpp).
//
// Mapping.  A work-group of 64 x 4 threads owns a 64 x 4 column tile and
// marches it upwards over a chunk of levels [k0, k1), one level per
// iteration.  Pressure of the tile plus a one-cell ring is computed once per
// cell and level into an LDS ring of four planes (levels k-1 .. k+2); the
// plane two levels ahead and the face momenta one level ahead are loaded into
// registers an iteration early, so their global loads overlap the current
// level's arithmetic.  The w face above the cell is carried in registers, so
// each face is computed once.  One barrier per level.  Splitting the column
// into chunks (chosen by the autotuner) gives the chip more independent
// work-groups; a chunk recomputes its bottom w face from the level below.
// Terrain has a march of its own below, with the column hydrostatic reference
// (a recurrence from the ground) in a kernel before it.  Work-group b is
// remapped so that each XCD (which receives every eighth work-group) owns a
// contiguous band of tiles and the ring rows shared by neighbouring tiles hit
// the same L2.
//
// Faces as departures.  Inside a subcycle the kernel carries the face
// momenta as departures m - m_base from the subcycle's entry faces (K15
// needs only the divergence of m - m_base, and m - m_base starts at zero), so
// a middle substep reads rho, theta and three departure fields and writes
// rho and three departures -- 9 fields instead of the 12 of the full faces
// and their bases.  The first substep reads no faces; the last reads the
// base faces and writes full faces (m_base + departure) and rho*theta.
//
// Flat terrain: the level means of rho and p for the next substep are
// emitted as per-wave FP64 partial sums of the new rho (fixed order: a DPP
// reduction, lane 63 writes), replacing a separate pass over the state.
#include "gwm_kernels.hpp"

namespace gwm {

namespace {

// Tile width: one wave per tile row.  The tile height TY (8 or 4) is a
// template parameter chosen per launch shape by the autotuner.
constexpr int TX = 64, PX = TX + 2;

}  // namespace

// Per-level values of a chunk (levels k0-1 .. k1+1), staged in LDS once per
// work-group so the level loop issues no global loads besides the pipelined
// planes and faces.
enum { LV_PREF = 0, LV_RREF, LV_IDZF, LV_IDZC, LV_BRHO, LV_BTH, LV_BRT, LV_BP, NLV };

// Level sums of the next substep (flat references, K6/K7) of one level, or of
// theta for the next stage: one partial per wave (a 64-column row segment), at
// (level, tile column, row), so the layout and with it the finalize's
// summation order do not depend on the tile height, and a work-group's waves
// write consecutive slots.  A row's 64 values are summed in FP64, except in
// the FP32 perturbation form: its values are departures from the level means,
// small and of either sign, whose FP32 sum (error below 4e-7 of the sum of
// their magnitudes) leaves the mean's error far below the departures' own
// rounding; the partial is stored in FP64.
template <class R, bool PERT, class Press>
__device__ __forceinline__ void emit_part(const FastArgs<R>& a, double* part_out, int k, int tile_x,
                                          int tiles_x, int j, int lx, bool active, R rho_new,
                                          R rt_new, R brho, R bth, Press&& press) {
  using S = typename std::conditional<PERT && sizeof(R) == 4, float, double>::type;
  S sr = S(0), spp = S(0);
  if (active) {
    if (a.part_theta) {  // theta_ref of the next stage (dry_core.cu:462-490)
      sr = static_cast<S>(PERT ? theta_pert(rho_new, rt_new, brho, bth) : q_theta(rho_new, rt_new));
    } else {
      sr = static_cast<S>(rho_new);
      spp = static_cast<S>(press());
    }
  }
  sr = wave_sum_to63(sr);
  spp = wave_sum_to63(spp);
  if (lx == TX - 1 && j < a.g.ny) {
    const size_t nw = static_cast<size_t>(a.g.ny) * tiles_x;
    const size_t slot = (static_cast<size_t>(k) * nw + static_cast<size_t>(tile_x) * a.g.ny +
                         static_cast<size_t>(j)) * 2;
    gstore(part_out, slot, static_cast<double>(sr));
    gstore(part_out, slot + 1, static_cast<double>(spp));
  }
}

// KIND: bit 0 first substep of the subcycle, bit 1 last substep.  DOWN:
// march the columns from the top down (whole columns of flat grids only),
// so that a substep reads first the levels the previous substep, marching
// up, wrote last; every cell's arithmetic is the upward march's, in the
// same order, so the results are identical.
template <class R, bool PERT, int KIND, int TYV, bool DOWN, bool SUMS>
__device__ __forceinline__ void fast_body(const FastArgs<R>& a, int tiles_x, int tiles, int nkc,
                                          double* part_out, const VBlock& vb) {
  constexpr int TY = TYV, PY = TY + 2, PN = PX * PY;
  constexpr int NHALO = PN - TX * TY;  // ring cells (148 at TY 8, 140 at TY 4)
  static_assert(NHALO <= TX * TY, "one thread per ring cell");
  constexpr bool FIRST = (KIND & 1) != 0, LAST = (KIND & 2) != 0;
  __shared__ R sp[4][PN];
  extern __shared__ __align__(16) unsigned char lev_raw[];
  R* const lev = reinterpret_cast<R*>(lev_raw);
  const Geo g = a.g;
  const int nz = g.nz;

  // XCD-aware order (work-group b runs on XCD b % 8), then (chunk, tile).
  const int nb = tiles * nkc;
  int b = vb.x;
  if ((nb & 7) == 0) b = (b & 7) * (nb >> 3) + (b >> 3);
  const int chunk = b / tiles, tile = b % tiles;
  const int k0 = (nz * chunk) / nkc, k1 = (nz * (chunk + 1)) / nkc;
  const int ti0 = (tile % tiles_x) * TX, tj0 = (tile / tiles_x) * TY;
  const int lx = threadIdx.x, ly = threadIdx.y;
  const int t = lx + TX * ly;
  const int i = ti0 + lx, j = tj0 + ly;
  const bool active = i < g.nx && j < g.ny;
  const int ci = (lx + 1) + PX * (ly + 1);

  // Ring cell of this thread (t < NHALO): rows -1 and TY, then columns -1 and TX.
  int hx = 0, hy = 0;
  if (t < 2 * PX) {
    hx = (t % PX) - 1;
    hy = t < PX ? -1 : TY;
  } else if (t < NHALO) {
    const int q = t - 2 * PX;
    hx = (q & 1) ? TX : -1;
    hy = q >> 1;
  }
  const int hci = (hx + 1) + PX * (hy + 1);

  // Per-level values of levels k0-1 .. k1+1 (indices clamped to the arrays).
  for (int q = t; q < k1 - k0 + 3; q += TX * TY) {
    const int kk = k0 - 1 + q;
    const int kc = kk < 0 ? 0 : (kk >= nz ? nz - 1 : kk), kf = kk < 0 ? 0 : (kk > nz ? nz : kk);
    R* e = lev + q * NLV;
    if constexpr (!SUMS) {
      e[LV_PREF] = a.pref_lev[kc];
      e[LV_RREF] = a.rref_lev[kc];
    }
    e[LV_IDZF] = a.m.lev_idz_f[kf];
    e[LV_IDZC] = a.m.lev_idz_c[kc];
    if (PERT) {
      e[LV_BRHO] = a.base.rho[kc];
      e[LV_BTH] = a.base.th[kc];
      e[LV_BRT] = a.base.rt[kc];
      e[LV_BP] = a.base.p[kc];
    }
  }
  if constexpr (SUMS) {  // level means, one level per wave
#pragma unroll 2
    for (int q = ly; q < k1 - k0 + 3; q += TY) {
      const int kk = k0 - 1 + q;
      double s0, s1;
      level_sums(a.lev_part, a.lev_nparts, kk < 0 ? 0 : (kk >= nz ? nz - 1 : kk), lx, s0, s1);
      if (lx == 63) {
        lev[q * NLV + LV_RREF] = static_cast<R>(s0) * a.lev_inv;
        lev[q * NLV + LV_PREF] = static_cast<R>(s1) * a.lev_inv;
      }
    }
  }
  auto LV = [&](int kk, int q) -> R { return lev[(kk - k0 + 1) * NLV + q]; };
  __syncthreads();

  const R dx = static_cast<R>(g.dx), dy = static_cast<R>(g.dy);
  const R rdx = R(1) / dx, rdy = R(1) / dy;
  const R dtf = a.dtf, grav = a.gravity;

  // Loads are unconditional (threads without a ring cell, or outside the
  // domain, read a valid stand-in and discard it), so the level loop is
  // straight-line code and each wait covers exactly the loads it needs:
  // the loads of level k+3 planes and k+1 faces stay in flight while level
  // k is computed.
  const unsigned pc = static_cast<unsigned>(g.pxc) * g.pyc;
  const int oc = stage_pos(g, i, j).c;
  const int hc = t < NHALO ? stage_pos(g, ti0 + hx, tj0 + hy).c : oc;
  auto ldc = [&](const R* f, int off, int k) -> R {
    const R v = ld32(f, static_cast<unsigned>(off < 0 ? 0 : off) + static_cast<unsigned>(k) * pc);
    return off < 0 ? R(0) : v;
  };
  struct Plane {
    R rc, tc, rh, th;
  };
  auto load_plane = [&](int k) -> Plane {
    return Plane{ldc(a.rho, oc, k), ldc(a.theta, oc, k), ldc(a.rho, hc, k), ldc(a.theta, hc, k)};
  };
  // Perturbation form: rho' and theta' in, p' out (K10 rho*theta = rho*theta_fixed
  // written for the departures: rho_b theta' + rho' (theta_b + theta')).
  auto press = [&](R r, R th, int k) -> R {
    if (!PERT) return q_pressure(r, r * th);
    const R rb = LV(k, LV_BRHO), tb = LV(k, LV_BTH);
    return p_pert(rb * th + r * (tb + th), LV(k, LV_BRT), LV(k, LV_BP));
  };
  auto stage_plane = [&](const Plane& P, int k) {
    sp[k & 3][ci] = press(P.rc, P.tc, k);
    if (t < NHALO) sp[k & 3][hci] = press(P.rh, P.th, k);
  };

  // Face departures m - m_base of one level of the own cell: none on the
  // first substep (the faces are the base faces), the previous substep's
  // output otherwise; the base faces on the last substep only, which writes
  // full faces.  Indices clamped into the domain for threads outside it.
  const int ic = i < g.nx ? i : g.nx - 1, jc = j < g.ny ? j : g.ny - 1;
  // Offsets of level k are the level-0 offset plus k times the field's level
  // stride (k is uniform, so the product is scalar work).
  const unsigned sxk = static_cast<unsigned>(g.pyc) * g.pxu;  // x faces
  const unsigned syk = static_cast<unsigned>(g.pyv) * g.pxc;  // y faces
  const unsigned xf_c = static_cast<unsigned>(g.xf(ic, jc, 0));
  const unsigned yf_c = static_cast<unsigned>(g.yf(ic, jc, 0));
  const unsigned zf_c = static_cast<unsigned>(g.zf(ic, jc, 0));
  const unsigned c_o = static_cast<unsigned>(g.cell(i, j, 0));
  const unsigned xf_o = static_cast<unsigned>(g.xf(i, j, 0));
  const unsigned yf_o = static_cast<unsigned>(g.yf(i, j, 0));
  // w1 / wb1: the z face the level computes, k+1 marching up, k marching
  // down (its departure and its base).
  struct Faces {
    R u0, u1, v0, v1, w1, ub0, ub1, vb0, vb1, wb1;
  };
  auto load_faces = [&](int k) -> Faces {
    Faces F{};
    const unsigned xf0 = xf_c + static_cast<unsigned>(k) * sxk;
    const unsigned yf0 = yf_c + static_cast<unsigned>(k) * syk;
    const unsigned yf1 = yf0 + static_cast<unsigned>(g.pxc);
    const unsigned zf1 = zf_c + static_cast<unsigned>(DOWN ? k : k + 1) * pc;
    if constexpr (!FIRST) {
      F.u0 = ld32(a.u, xf0);
      F.u1 = ld32(a.u, xf0 + 1);
      F.v0 = ld32(a.v, yf0);
      F.v1 = ld32(a.v, yf1);
      F.w1 = ld32(a.w, zf1);
    }
    if constexpr (LAST) {
      F.ub0 = ld32(a.ub, xf0);
      F.ub1 = ld32(a.ub, xf0 + 1);
      F.vb0 = ld32(a.vb, yf0);
      F.vb1 = ld32(a.vb, yf1);
      F.wb1 = ld32(a.wb, zf1);
    }
    return F;
  };

  // ---- prologue: planes k0-1 .. k0+1 staged, plane k0+2 and faces of k0
  // in flight, bottom w face.
  const int kmax = nz - 1 < k1 ? nz - 1 : k1;  // highest plane a chunk stages
  // rho_k1 / th_k1 hold the next level of the march (k+1 up, k-1 down);
  // w0 / wb0 the z face carried from the level before (the bottom face k
  // marching up, the top face k+1 marching down).
  R rho_km1 = R(0);
  R rho_k, th_k, rho_k1 = R(0), th_k1 = R(0);
  Plane P2;
  Faces F;
  R w0, wb0;
  if constexpr (DOWN) {
    // whole columns: planes nz-1 and nz-2 staged, plane nz-3 and the faces
    // of level nz-1 in flight, the top w face (left as it is).
    {
      const Plane P = load_plane(nz - 1);
      stage_plane(P, nz - 1);
      rho_k = P.rc;
      th_k = P.tc;
    }
    if (nz > 1) {
      const Plane P = load_plane(nz - 2);
      stage_plane(P, nz - 2);
      rho_k1 = P.rc;
      th_k1 = P.tc;
    }
    P2 = load_plane(nz - 3 > 0 ? nz - 3 : 0);
    F = load_faces(nz - 1);
    const size_t zft = g.zf(ic, jc, nz);
    w0 = FIRST ? R(0) : a.w[zft];
    wb0 = LAST ? a.wb[zft] : R(0);
  } else {
    if (k0 > 0) {
      const Plane P = load_plane(k0 - 1);
      stage_plane(P, k0 - 1);
      rho_km1 = P.rc;
    }
    {
      const Plane P = load_plane(k0);
      stage_plane(P, k0);
      rho_k = P.rc;
      th_k = P.tc;
    }
    if (k0 + 1 < nz) {
      const Plane P = load_plane(k0 + 1);
      stage_plane(P, k0 + 1);
      rho_k1 = P.rc;
      th_k1 = P.tc;
    }
    P2 = load_plane(k0 + 2 < kmax ? k0 + 2 : kmax);
    F = load_faces(k0);
    const size_t zf0 = g.zf(ic, jc, k0);
    w0 = FIRST ? R(0) : a.w[zf0];
    wb0 = LAST ? a.wb[zf0] : R(0);
  }
  __syncthreads();

  const bool ow = !g.per_x, os = !g.per_y;
  if (!DOWN && active && k0 > 0) {
    // K14 at face k0 from levels k0-1 and k0.
    const R ppl = sp[(k0 - 1) & 3][ci] - LV(k0 - 1, LV_PREF);
    const R ppu = sp[k0 & 3][ci] - LV(k0, LV_PREF);
    const R rpf = R(0.5) * ((rho_km1 - LV(k0 - 1, LV_RREF)) + (rho_k - LV(k0, LV_RREF)));
    const R tend = -(ppu - ppl) * LV(k0, LV_IDZF) - grav * rpf;
    w0 = w0 + dtf * tend;
  }

  // Level k: P2 / F hold plane k+2 and the faces of level k (loaded an
  // iteration ago); the loads of plane k+3 and of the faces of level k+1 go
  // into P3 / Fn first.  The loop is unrolled by two with the buffers
  // swapped, so no register copy waits for loads in flight.
  auto level = [&](int k, const Plane& P2, const Faces& F, Plane& P3, Faces& Fn) {
    // Stage the plane two levels ahead in the march (k+2 up, k-2 down).
    if constexpr (DOWN) {
      P3 = load_plane(k - 3 > 0 ? k - 3 : 0);
      Fn = load_faces(k - 1 > 0 ? k - 1 : 0);
      if (k - 2 >= 0) stage_plane(P2, k - 2);
    } else {
      P3 = load_plane(k + 3 < kmax ? k + 3 : kmax);
      Fn = load_faces(k + 1 < k1 ? k + 1 : k1 - 1);
      if (k + 2 <= kmax) stage_plane(P2, k + 2);
    }
    const R rho_k2 = P2.rc, th_k2 = P2.tc;

    const R* pk = sp[k & 3];
    const R* pdn = sp[(k + 3) & 3];  // level k-1
    const R* pup = sp[(k + 1) & 3];  // level k+1

    R rho_new = R(0), rt_new = R(0);
    if (active) {
      // K12 / K13: faces i, i+1 and j, j+1 of the cell.
      R u0 = F.u0, u1 = F.u1, v0 = F.v0, v1 = F.v1;
      if (a.horizontal) {
        if (!(i == 0 && ow)) u0 = F.u0 + (-dtf * qdivc(pk[ci] - pk[ci - 1], dx, rdx));
        if (!(i + 1 == g.nx && ow))
          u1 = F.u1 + (-dtf * qdivc(pk[ci + 1] - pk[ci], dx, rdx));
        if (!(j == 0 && os)) v0 = F.v0 + (-dtf * qdivc(pk[ci] - pk[ci - PX], dy, rdy));
        if (!(j + 1 == g.ny && os))
          v1 = F.v1 + (-dtf * qdivc(pk[ci + PX] - pk[ci], dy, rdy));
      }
      // K14 (faces 0 and nz are left as they are): marching up, w face k+1
      // from levels k and k+1; marching down, w face k from levels k-1 and
      // k (the same arithmetic for a face either way).
      auto k14 = [&](R wf, R p_lo, R p_hi, R pl, R pu, R r_lo, R r_hi, R rl, R ru, R idz) -> R {
        const R ppl = p_lo - pl;
        const R ppu = p_hi - pu;
        const R rpf = R(0.5) * ((r_lo - rl) + (r_hi - ru));
        const R tend = -(ppu - ppl) * idz - grav * rpf;
        return wf + dtf * tend;
      };
      R w1 = F.w1;  // the face this level computes
      if constexpr (DOWN) {
        if (k > 0)
          w1 = k14(F.w1, pdn[ci], pk[ci], LV(k - 1, LV_PREF), LV(k, LV_PREF), rho_k1, rho_k,
                   LV(k - 1, LV_RREF), LV(k, LV_RREF), LV(k, LV_IDZF));
      } else if (k + 1 < nz) {
        w1 = k14(F.w1, pk[ci], pup[ci], LV(k, LV_PREF), LV(k + 1, LV_PREF), rho_k, rho_k1,
                 LV(k, LV_RREF), LV(k + 1, LV_RREF), LV(k + 1, LV_IDZF));
      }
      // the bottom and top w faces of the cell
      const R wlo = DOWN ? w1 : w0, whi = DOWN ? w0 : w1;
      // K15
      rho_new = rho_k;
      if (a.density) {
        const R idz = LV(k, LV_IDZC);
        // divergence of (m - m_base): the faces are departures already
        const R div = qdivc(u1 - u0, dx, rdx) + qdivc(v1 - v0, dy, rdy) + (whi - wlo) * idz;
        const R floor = PERT ? R(1.0e-6) - LV(k, LV_BRHO) : R(1.0e-6);
        rho_new = rmax(floor, rho_new - dtf * div);
      }
      const unsigned c0 = c_o + static_cast<unsigned>(k) * pc;
      const unsigned xf0 = xf_o + static_cast<unsigned>(k) * sxk;
      const unsigned yf0 = yf_o + static_cast<unsigned>(k) * syk;
      st32(a.rho_out, c0, rho_new);
      rt_new = PERT ? LV(k, LV_BRHO) * th_k + rho_new * (LV(k, LV_BTH) + th_k) : rho_new * th_k;
      if (a.rt_out) st32(a.rt_out, c0, rt_new);
      // departures, or full faces base + departure on the last substep
      st32(a.u_out, xf0, LAST ? F.ub0 + u0 : u0);
      st32(a.v_out, yf0, LAST ? F.vb0 + v0 : v0);
      // w face k (and face nz on the top level), with its base on the last
      // substep: the carried face marching up, the computed one marching down
      const R wb_lo = DOWN ? F.wb1 : wb0, wb_hi = DOWN ? wb0 : F.wb1;
      st32(a.w_out, c0, LAST ? wb_lo + wlo : wlo);
      if (i == g.nx - 1) st32(a.u_out, xf0 + 1, LAST ? F.ub1 + u1 : u1);
      if (j == g.ny - 1) st32(a.v_out, yf0 + static_cast<unsigned>(g.pxc), LAST ? F.vb1 + v1 : v1);
      if (k == nz - 1) st32(a.w_out, c0 + pc, LAST ? wb_hi + whi : whi);
      w0 = w1;
    }
    wb0 = F.wb1;

    if (part_out)
      emit_part<R, PERT>(a, part_out, k, tile % tiles_x, tiles_x, j, lx, active, rho_new, rt_new,
                         LV(k, LV_BRHO), LV(k, LV_BTH), [&] { return press(rho_new, th_k, k); });

    rho_k = rho_k1;
    th_k = th_k1;
    rho_k1 = rho_k2;
    th_k1 = th_k2;
    __syncthreads();
  };
  Plane P3;
  Faces Fn;
  if constexpr (DOWN) {
    for (int k = nz - 1; k >= 0; k -= 2) {
      level(k, P2, F, P3, Fn);
      if (k - 1 >= 0) level(k - 1, P3, Fn, P2, F);
    }
    return;
  }
  for (int k = k0; k < k1; k += 2) {
    level(k, P2, F, P3, Fn);
    if (k + 1 < k1) level(k + 1, P3, Fn, P2, F);
  }
}

// ===========================================================================
// Terrain.  The same march over a grid whose heights vary within a level:
// K12 / K13 take the pressure gradient along the sloping levels,
//   dp/dx - dz/dx (dp/dz_l + dp/dz_r) / 2,
// so a face needs p, dp/dz and z of the columns on its two sides.  A thread
// forms dp/dz once for its own and once for its ring cell, from the pressures
// and heights of three levels it carries in registers, and stages p, dp/dz
// and z of one level ahead in LDS (two slots, one barrier a level): 1.3
// quotients a cell, and each height is loaded once, with the plane it belongs
// to, two levels early.  Reading the five columns' heights at each level from
// global memory instead (17 dependent loads a cell behind no prefetch) is
// what bound this kernel before: FP32 perturbation substep of 192 x 192 x 60
// 67.5 -> 35.0 us, FP64 substep of 151 x 97 x 40 257 -> 28 us and the column reference.
//
// REF: where K14's reference state comes from -- the level means (heights
// all below 1e-6 m), the column's hydrostatic reference (K11, in memory,
// k_column_reference below), or none (the perturbation form: the column
// reference's terms cancel between its recurrence and K14 up to the
// recurrence's residual, which the z-face base forcing carries; K14 acts on
// the departures and adds that forcing; per-cell bases).
// ===========================================================================
enum { REF_LEVEL = 0, REF_COLUMN, REF_BASE };

template <class R, int REF, int KIND, int TYV>
__device__ __forceinline__ void fast_terrain_body(const FastArgs<R>& a, int tiles_x, int tiles,
                                                  int nkc, double* part_out, const VBlock& vb) {
  constexpr bool TP = REF == REF_BASE;
  constexpr int TY = TYV, PY = TY + 2, PN = PX * PY;
  constexpr int NHALO = PN - TX * TY;
  static_assert(NHALO <= TX * TY, "one thread per ring cell");
  constexpr bool FIRST = (KIND & 1) != 0, LAST = (KIND & 2) != 0;
  __shared__ R sp[2][PN], sg[2][PN], sz[2][PN];
  extern __shared__ __align__(16) unsigned char lev_raw[];
  R* const lev = reinterpret_cast<R*>(lev_raw);
  const Geo g = a.g;
  const Loader<R> L{g};
  const int nz = g.nz;

  const int nb = tiles * nkc;
  int b = vb.x;
  if ((nb & 7) == 0) b = (b & 7) * (nb >> 3) + (b >> 3);
  const int chunk = b / tiles, tile = b % tiles;
  const int k0 = (nz * chunk) / nkc, k1 = (nz * (chunk + 1)) / nkc;
  const int ti0 = (tile % tiles_x) * TX, tj0 = (tile / tiles_x) * TY;
  const int lx = threadIdx.x, ly = threadIdx.y;
  const int t = lx + TX * ly;
  const int i = ti0 + lx, j = tj0 + ly;
  const bool active = i < g.nx && j < g.ny;
  const int ci = (lx + 1) + PX * (ly + 1);
  int hx = lx, hy = ly;
  if (t < 2 * PX) {
    hx = (t % PX) - 1;
    hy = t < PX ? -1 : TY;
  } else if (t < NHALO) {
    const int q = t - 2 * PX;
    hx = (q & 1) ? TX : -1;
    hy = q >> 1;
  }
  const int hci = (hx + 1) + PX * (hy + 1);
  const bool ring = t < NHALO;

  // Per-level values of levels k0-1 .. k1+1 (indices clamped to the arrays).
  if constexpr (REF != REF_COLUMN) {
    for (int q = t; q < k1 - k0 + 3; q += TX * TY) {
      const int kk = k0 - 1 + q;
      const int kc = kk < 0 ? 0 : (kk >= nz ? nz - 1 : kk);
      R* e = lev + q * NLV;
      if constexpr (TP) {
        e[LV_BRHO] = a.base.rho[kc];
        e[LV_BTH] = a.base.th[kc];
        e[LV_BP] = a.base.p[kc];
      } else {
        e[LV_PREF] = a.pref_lev[kc];
        e[LV_RREF] = a.rref_lev[kc];
      }
    }
    __syncthreads();
  }
  auto LV = [&](int kk, int q) -> R { return lev[(kk - k0 + 1) * NLV + q]; };

  const R dx = static_cast<R>(g.dx), dy = static_cast<R>(g.dy);
  const R rdx = R(1) / dx, rdy = R(1) / dy;
  const R dtf = a.dtf, grav = a.gravity;

  // Cell offsets of the own and the ring position (-1 outside an open
  // domain: zero, read from a stand-in), and their metric columns (periodic
  // wrap, or the edge column: dry_fast_modes.cu:24-30).
  const unsigned pc = static_cast<unsigned>(g.pxc) * g.pyc;
  const unsigned pm = static_cast<unsigned>(g.nx) * g.ny;
  const int oc = stage_pos(g, i, j).c;
  const int hc = ring ? stage_pos(g, ti0 + hx, tj0 + hy).c : oc;
  const unsigned om = static_cast<unsigned>(L.mj(j) * g.nx + L.mi(i));
  const unsigned hm = ring ? static_cast<unsigned>(L.mj(tj0 + hy) * g.nx + L.mi(ti0 + hx)) : om;
  auto ldb = [&](const R* f, int off, int k) -> R {
    return ld32(f, static_cast<unsigned>(off < 0 ? 0 : off) + static_cast<unsigned>(k) * pc);
  };
  auto ldc = [&](const R* f, int off, int k) -> R {
    const R v = ldb(f, off, k);
    return off < 0 ? R(0) : v;
  };
  struct Cell {
    R r, th, z, br, bt, bp;  // rho, theta, height; base deviations (REF_BASE)
  };
  struct Plane {
    Cell o, h;    // own, ring
    R pref, rref;  // column reference of the own cell (REF_COLUMN)
  };
  auto load_cell = [&](int off, unsigned m, int k) -> Cell {
    Cell c{ldc(a.rho, off, k), ldc(a.theta, off, k), ld32(a.m.zc, m + static_cast<unsigned>(k) * pm),
           R(0), R(0), R(0)};
    if constexpr (TP) {
      c.br = ldb(a.base.drho, off, k);
      c.bt = ldb(a.base.dth, off, k);
      c.bp = ldb(a.base.dp, off, k);
    }
    return c;
  };
  auto load_plane = [&](int k) -> Plane {
    Plane P{load_cell(oc, om, k), load_cell(hc, hm, k), R(0), R(0)};
    if constexpr (REF == REF_COLUMN) {
      P.pref = ld32(a.pref3, om + static_cast<unsigned>(k) * pm);
      P.rref = ld32(a.rref3, om + static_cast<unsigned>(k) * pm);
    }
    return P;
  };
  // p of a cell, or p' against its base: rho_b theta' + rho' (theta_b + theta').
  auto press = [&](const Cell& c, int k) -> R {
    if constexpr (TP) {
      const R rb = LV(k, LV_BRHO) + c.br, tb = LV(k, LV_BTH) + c.bt;
      return p_pert(rb * c.th + c.r * (tb + c.th), rb * tb, LV(k, LV_BP) + c.bp);
    }
    return q_pressure(c.r, c.r * c.th);
  };
  // dp/dz between two levels of a column (dry_pressure_gradient.cu:37-73).
  auto grad = [&](R p_lo, R p_hi, R z_lo, R z_hi) -> R {
    return qdiv(p_hi - p_lo, rmax(z_hi - z_lo, R(1.0e-6)));
  };

  const int ic = i < g.nx ? i : g.nx - 1, jc = j < g.ny ? j : g.ny - 1;
  const unsigned sxk = static_cast<unsigned>(g.pyc) * g.pxu;  // x faces
  const unsigned syk = static_cast<unsigned>(g.pyv) * g.pxc;  // y faces
  const unsigned xf_c = static_cast<unsigned>(g.xf(ic, jc, 0));
  const unsigned yf_c = static_cast<unsigned>(g.yf(ic, jc, 0));
  const unsigned zf_c = static_cast<unsigned>(g.zf(ic, jc, 0));
  const unsigned c_o = static_cast<unsigned>(g.cell(i, j, 0));
  const unsigned xf_o = static_cast<unsigned>(g.xf(i, j, 0));
  const unsigned yf_o = static_cast<unsigned>(g.yf(i, j, 0));
  struct Faces {
    R u0, u1, v0, v1, w1, ub0, ub1, vb0, vb1, wb1;
    R fu0, fu1, fv0, fv1, fw1;  // base forcing (REF_BASE)
    R idz_f1, idz_c;            // of z face k+1 and of the cell
  };
  auto load_faces = [&](int k) -> Faces {
    Faces F{};
    const unsigned xf0 = xf_c + static_cast<unsigned>(k) * sxk;
    const unsigned yf0 = yf_c + static_cast<unsigned>(k) * syk;
    const unsigned yf1 = yf0 + static_cast<unsigned>(g.pxc);
    const unsigned zf1 = zf_c + static_cast<unsigned>(k + 1) * pc;
    if constexpr (!FIRST) {
      F.u0 = ld32(a.u, xf0);
      F.u1 = ld32(a.u, xf0 + 1);
      F.v0 = ld32(a.v, yf0);
      F.v1 = ld32(a.v, yf1);
      F.w1 = ld32(a.w, zf1);
    }
    if constexpr (LAST) {
      F.ub0 = ld32(a.ub, xf0);
      F.ub1 = ld32(a.ub, xf0 + 1);
      F.vb0 = ld32(a.vb, yf0);
      F.vb1 = ld32(a.vb, yf1);
      F.wb1 = ld32(a.wb, zf1);
    }
    if constexpr (TP) {
      F.fu0 = ld32(a.base.fu, xf0);
      F.fu1 = ld32(a.base.fu, xf0 + 1);
      F.fv0 = ld32(a.base.fv, yf0);
      F.fv1 = ld32(a.base.fv, yf1);
      F.fw1 = ld32(a.base.fw, zf1);
    }
    F.idz_f1 = ld32(a.m.idz_f, om + static_cast<unsigned>(k + 1) * pm);
    F.idz_c = ld32(a.m.idz_c, om + static_cast<unsigned>(k) * pm);
    return F;
  };

  // What a thread carries of a level: pressure and height of the own and the
  // ring cell; of the own cell also rho, theta, its base and its reference.
  struct Lev {
    R p, z, ph, zh, r, th, br, bt, pref, rref;
  };
  auto level_of = [&](const Plane& P, int k) -> Lev {
    Lev v{press(P.o, k), P.o.z, R(0), P.h.z, P.o.r, P.o.th, P.o.br, P.o.bt, P.pref, P.rref};
    if (ring) v.ph = press(P.h, k);
    if constexpr (REF == REF_LEVEL) {
      v.pref = LV(k, LV_PREF);
      v.rref = LV(k, LV_RREF);
    }
    return v;
  };
  // Stages level k given the levels whose difference gives its dp/dz.
  auto stage = [&](int k, const Lev& v, const Lev& lo, const Lev& hi) {
    const int s = k & 1;
    sp[s][ci] = v.p;
    sz[s][ci] = v.z;
    sg[s][ci] = nz == 1 ? R(0) : grad(lo.p, hi.p, lo.z, hi.z);
    if (ring) {
      sp[s][hci] = v.ph;
      sz[s][hci] = v.zh;
      sg[s][hci] = nz == 1 ? R(0) : grad(lo.ph, hi.ph, lo.zh, hi.zh);
    }
  };
  // K14 at a z face between levels lo and hi.
  auto k14 = [&](R wf, const Lev& lo, const Lev& hi, R idz, R fw) -> R {
    if constexpr (TP) {
      const R rpf = R(0.5) * (lo.r + hi.r);
      const R tend = -(hi.p - lo.p) * idz - grav * rpf;
      return wf + dtf * (tend + fw);
    }
    const R ppl = lo.p - lo.pref, ppu = hi.p - hi.pref;
    const R rpf = R(0.5) * ((lo.r - lo.rref) + (hi.r - hi.rref));
    const R tend = -(ppu - ppl) * idz - grav * rpf;
    return wf + dtf * tend;
  };

  // ---- prologue: level k0 staged, levels k0 and k0+1 carried, plane k0+2
  // and the faces of k0 in flight.
  const int kmax = nz - 1 < k1 ? nz - 1 : k1;  // highest plane a chunk needs
  Lev c, n;  // levels k and k+1
  Plane P2;
  Faces F;
  R w0, wb0;
  {
    const Plane Pm = load_plane(k0 > 0 ? k0 - 1 : 0);
    const Plane Pc = load_plane(k0);
    const Plane Pn = load_plane(k0 + 1 < nz ? k0 + 1 : k0);
    P2 = load_plane(k0 + 2 < kmax ? k0 + 2 : kmax);
    F = load_faces(k0);
    const unsigned zf0 = zf_c + static_cast<unsigned>(k0) * pc;
    w0 = FIRST ? R(0) : ld32(a.w, zf0);
    wb0 = LAST ? ld32(a.wb, zf0) : R(0);
    const Lev m = level_of(Pm, k0 > 0 ? k0 - 1 : 0);
    c = level_of(Pc, k0);
    n = level_of(Pn, k0 + 1 < nz ? k0 + 1 : k0);
    // (k0 == 0: m is level 0; k0 == nz-1: n is level nz-1)
    stage(k0, c, m, n);
    if (k0 > 0) {
      const R idz = ld32(a.m.idz_f, om + static_cast<unsigned>(k0) * pm);
      R fw = R(0);
      if constexpr (TP) fw = ld32(a.base.fw, zf0);
      w0 = k14(w0, m, c, idz, fw);
    }
  }
  __syncthreads();

  const bool ow = !g.per_x, os = !g.per_y;
  // Level k: P2 / F hold plane k+2 and the faces of level k (loaded an
  // iteration ago); the loop is unrolled by two with the buffers swapped, so
  // no register copy waits for loads in flight.
  auto level = [&](int k, const Plane& P2, const Faces& F, Plane& P3, Faces& Fn) {
    P3 = load_plane(k + 3 < kmax ? k + 3 : kmax);
    Fn = load_faces(k + 1 < k1 ? k + 1 : k1 - 1);
    Lev n2 = n;  // level k+2, or k+1 where there is none
    if (k + 2 <= kmax) n2 = level_of(P2, k + 2);
    // (written here, read in the next iteration: the barrier is between)
    if (k + 1 < k1) stage(k + 1, n, c, n2);

    const R* pk = sp[k & 1];
    const R* gk = sg[k & 1];
    const R* zk = sz[k & 1];
    R rho_new = R(0), rt_new = R(0);
    if (active) {
      const R g_own = gk[ci];
      // pressure gradient at the face between the own cell and a neighbour
      auto pgf_lo = [&](int nb, R d, R rd) -> R {  // the neighbour is the lower one
        return qdivc(c.p - pk[nb], d, rd) - qdivc(c.z - zk[nb], d, rd) * (R(0.5) * (gk[nb] + g_own));
      };
      auto pgf_hi = [&](int nb, R d, R rd) -> R {
        return qdivc(pk[nb] - c.p, d, rd) - qdivc(zk[nb] - c.z, d, rd) * (R(0.5) * (g_own + gk[nb]));
      };
      // (the perturbation form adds the base's forcing of the face)
      auto fb = [&](R pg, R f) -> R {
        if constexpr (TP) return pg + f;
        return pg;
      };
      R u0 = F.u0, u1 = F.u1, v0 = F.v0, v1 = F.v1;
      if (a.horizontal) {
        if (!(i == 0 && ow)) u0 = F.u0 + (-dtf * fb(pgf_lo(ci - 1, dx, rdx), F.fu0));
        if (!(i + 1 == g.nx && ow)) u1 = F.u1 + (-dtf * fb(pgf_hi(ci + 1, dx, rdx), F.fu1));
        if (!(j == 0 && os)) v0 = F.v0 + (-dtf * fb(pgf_lo(ci - PX, dy, rdy), F.fv0));
        if (!(j + 1 == g.ny && os)) v1 = F.v1 + (-dtf * fb(pgf_hi(ci + PX, dy, rdy), F.fv1));
      }
      // K14 at face k+1 (faces 0 and nz are left as they are)
      const R w1 = k + 1 < nz ? k14(F.w1, c, n, F.idz_f1, F.fw1) : F.w1;
      // K15: divergence of (m - m_base), the faces are departures already
      R rb = R(0), tb = R(0);
      if constexpr (TP) {
        rb = LV(k, LV_BRHO) + c.br;
        tb = LV(k, LV_BTH) + c.bt;
      }
      rho_new = c.r;
      if (a.density) {
        const R div = qdivc(u1 - u0, dx, rdx) + qdivc(v1 - v0, dy, rdy) + (w1 - w0) * F.idz_c;
        rho_new = rmax(TP ? R(1.0e-6) - rb : R(1.0e-6), rho_new - dtf * div);
      }
      rt_new = TP ? rb * c.th + rho_new * (tb + c.th) : rho_new * c.th;
      const unsigned c0 = c_o + static_cast<unsigned>(k) * pc;
      const unsigned xf0 = xf_o + static_cast<unsigned>(k) * sxk;
      const unsigned yf0 = yf_o + static_cast<unsigned>(k) * syk;
      st32(a.rho_out, c0, rho_new);
      if (a.rt_out) st32(a.rt_out, c0, rt_new);
      // departures, or full faces base + departure on the last substep
      st32(a.u_out, xf0, LAST ? F.ub0 + u0 : u0);
      st32(a.v_out, yf0, LAST ? F.vb0 + v0 : v0);
      st32(a.w_out, c0, LAST ? wb0 + w0 : w0);
      if (i == g.nx - 1) st32(a.u_out, xf0 + 1, LAST ? F.ub1 + u1 : u1);
      if (j == g.ny - 1) st32(a.v_out, yf0 + static_cast<unsigned>(g.pxc), LAST ? F.vb1 + v1 : v1);
      if (k == nz - 1) st32(a.w_out, c0 + pc, LAST ? F.wb1 + w1 : w1);
      w0 = w1;
    }
    wb0 = F.wb1;
    if constexpr (REF == REF_LEVEL) {
      if (part_out)
        emit_part<R, false>(a, part_out, k, tile % tiles_x, tiles_x, j, lx, active, rho_new, rt_new,
                            R(0), R(0), [&] { return q_pressure(rho_new, rho_new * c.th); });
    }
    c = n;
    n = n2;
    __syncthreads();
  };
  Plane P3;
  Faces Fn;
  for (int k = k0; k < k1; k += 2) {
    level(k, P2, F, P3, Fn);
    if (k + 1 < k1) level(k + 1, P3, Fn, P2, F);
  }
}

// ===========================================================================
// Column hydrostatic reference (K11, dry_fast_modes.cu:120-178): a recurrence
// up each column of (p, rho), four fixed-point iterations of p_{k+1} = p_k -
// g dz (rho_k + rho(p_{k+1}, theta)) / 2 a level, each with the density of a
// trial pressure at the cell's theta.
//
// The chain of dependent operations is what bounds it: five powers and ten
// quotients a level, carried in the substep's own whole-column march, made an
// FP64 substep of 151 x 97 x 40 take 257 us; this kernel takes 18 of the 47
// it takes now.  Here each density is a series about the cell's own state,
// which needs no power: with p_a = EOS(rho_a, theta), rho(p, theta) = rho_a
// (p / p_a)^(1 - kappa), and u = p / p_a - 1 is small as the reference
// follows the column (the first trial, an Euler step, is off by about
// (dz / H)^2 / 2); the four trials run in u, five dependent operations each.
// The terms kept leave 2^-66 of the result at |u| = 2^-5 in FP64 and 2^-31 in
// FP32; a level with a trial further out, or a state on one of the EOS's
// floors, is done with the power.  p_a and 1 / p_a do not depend on the chain:
// wave 0 of a work-group marches 64 columns, and the other seven prepare the
// next seven levels, one each, in LDS meanwhile.  p_{k+1} is rounded once from
// p_k: K14 takes the difference of neighbouring levels, which then holds that
// one rounding (a compensated sum holds two, its levels being rounded apart).
// ===========================================================================
constexpr int kRefWaves = 8, kRefSeg = kRefWaves - 1;

// (1 + u)^(1 - kappa), |u| <= 2^-5: the binomial series to u^11 (FP64) or u^4
// (FP32), in Estrin's order (half the depth of Horner's).
template <class R>
struct RhoSeries {
  R c[12];
  constexpr RhoSeries() : c{} {
    const double e = 1.0 - static_cast<double>(Phys<R>::kappa);
    double v = 1.0;
    c[0] = R(1);
    for (int q = 1; q < 12; ++q) {
      v *= (e - (q - 1)) / q;
      c[q] = static_cast<R>(v);
    }
  }
};
__device__ inline float rho_series(float u) {
  constexpr RhoSeries<float> C;
  const float u2 = u * u;
  const float hi = __builtin_fmaf(__builtin_fmaf(C.c[4], u, C.c[3]), u, C.c[2]);
  return __builtin_fmaf(hi, u2, __builtin_fmaf(C.c[1], u, 1.0f));
}
__device__ inline double rho_series(double u) {
  constexpr RhoSeries<double> C;
  const double u2 = u * u, u4 = u2 * u2;
  auto pair = [&](int q) { return __builtin_fma(C.c[q + 1], u, C.c[q]); };
  auto quad = [&](int q) { return __builtin_fma(pair(q + 2), u2, pair(q)); };
  return __builtin_fma(__builtin_fma(quad(8), u4, quad(4)), u4, quad(0));
}

template <class R>
__device__ __forceinline__ void column_reference_body(const FastArgs<R>& a, const VBlock& vb) {
  __shared__ R s_pa[2][kRefSeg][64], s_ra[2][kRefSeg][64], s_rho[2][kRefSeg][64],
      s_h[2][kRefSeg][64];
  const Geo g = a.g;
  const int nz = g.nz;
  const unsigned n2 = static_cast<unsigned>(g.nx) * g.ny;
  const int lane = threadIdx.x, wave = threadIdx.y;
  const unsigned col = static_cast<unsigned>(vb.x) * 64u + lane;
  const bool in = col < n2;
  const unsigned m0 = in ? col : n2 - 1;
  const unsigned c0 = static_cast<unsigned>(g.cell(m0 % g.nx, m0 / g.nx, 0));
  const unsigned pc = static_cast<unsigned>(g.pxc) * g.pyc;
  const R grav = a.gravity;
  // level k >= 1 of the column: its pressure (and reciprocal), density, and
  // half the weight of the layer below it per density
  auto fill = [&](int k, int buf) {
    const unsigned c = c0 + static_cast<unsigned>(k) * pc, m = m0 + static_cast<unsigned>(k) * n2;
    const R r = ld32(a.rho, c), th = ld32(a.theta, c);
    const R dz = ld32(a.m.zc, m) - ld32(a.m.zc, m - n2);
    const R pa = q_pressure(r, r * th);
    // away from the floors of rho, p, p / p0 and R_d theta Exner, each with
    // room for the series' range; else u is NaN and the power is taken
    const bool series = r >= R(2.0e-6) && pa >= R(2) && pa >= R(2.0e-6) * r;
    const int q = k % kRefSeg;
    s_pa[buf][q][lane] = pa;
    s_ra[buf][q][lane] = series ? qrcp(pa) : static_cast<R>(__builtin_nanf(""));
    s_rho[buf][q][lane] = r;
    s_h[buf][q][lane] = grav * R(0.5) * dz;
  };
  const int nseg = (nz + kRefSeg - 1) / kRefSeg;
  // segment s: levels s * kRefSeg + 0 .. kRefSeg - 1 (level 0 starts the march)
  auto fill_seg = [&](int s) {
    const int k = s * kRefSeg + wave - 1;
    if (k >= 1 && k < nz) fill(k, s & 1);
  };
  R p = R(0), r = R(0);
  if (wave > 0) {
    fill_seg(0);
  } else {
    const R rho0 = ld32(a.rho, c0), rt0 = rho0 * ld32(a.theta, c0);
    p = q_pressure(rho0, rt0);
    r = q_rho_from_p_theta(p, q_theta(rho0, rt0));
    if (in) {
      st32(a.pref3, m0, p);
      st32(a.rref3, m0, r);
    }
  }
  __syncthreads();
  struct Prep {
    R pa, ra, rho, h;
  };
  for (int s = 0; s < nseg; ++s) {
    if (wave > 0) {
      fill_seg(s + 1);
    } else {
      const int kb = s * kRefSeg, ke = kb + kRefSeg < nz ? kb + kRefSeg : nz;
      auto prep = [&](int k) -> Prep {
        const int q = k - kb;
        return Prep{s_pa[s & 1][q][lane], s_ra[s & 1][q][lane], s_rho[s & 1][q][lane],
                    s_h[s & 1][q][lane]};
      };
      const int kf = kb > 0 ? kb : 1;
      Prep nx{};
      if (kf < ke) nx = prep(kf);
      for (int k = kf; k < ke; ++k) {
        const Prep c = nx;
        nx = prep(k + 1 < ke ? k + 1 : k);  // in flight during this level
        // p_{k+1} less the layer's weight, in one rounding
        auto weigh = [&](R sum) -> R { return static_cast<R>(fma(-c.h, sum, p)); };
        // (a NaN is not near: no series at this level, an infinite pressure,
        // or an overflow on the way)
        bool near = true;
        auto shape = [&](R u) -> R {  // rho(pa (1 + u)) / rho
          near &= (u < R(0) ? -u : u) <= R(0.03125);
          return rho_series(u);
        };
        // the trials run in u: the recurrence p - h (r + rho f(u)) is u =
        // (p - pa) / pa - h (r + rho f(u)) / pa
        const R u0 = (p - c.pa) * c.ra, hr = c.h * c.ra;
        const R A = hr * c.rho, B = static_cast<R>(fma(-hr, r, u0));
        R u = static_cast<R>(fma(-hr, r, B)), f = R(0);
#pragma unroll
        for (int it = 0; it < 4; ++it) {
          f = shape(u);
          if (it < 3) u = static_cast<R>(fma(-A, f, B));
        }
        R pn = weigh(static_cast<R>(fma(c.rho, f, r)));
        R rn = c.rho * shape((pn - c.pa) * c.ra);
        if (!near) {
          const R th = q_theta(c.rho, c.rho * ld32(a.theta, c0 + static_cast<unsigned>(k) * pc));
          pn = rmax(weigh(r + r), R(1));
#pragma unroll 1
          for (int it = 0; it < 4; ++it) pn = rmax(weigh(r + q_rho_from_p_theta(pn, th)), R(1));
          rn = q_rho_from_p_theta(pn, th);
        }
        p = pn;
        r = rn;
        if (in) {
          const unsigned m = m0 + static_cast<unsigned>(k) * n2;
          st32(a.pref3, m, p);
          st32(a.rref3, m, r);
        }
      }
    }
    __syncthreads();
  }
}

template <class R>
__global__ __launch_bounds__(64 * kRefWaves) void k_column_reference(FastArgs<R> a) {
  column_reference_body(a, hw_block());
}
template <class R>
__global__ __launch_bounds__(64 * kRefWaves) void k_column_reference_batch(
    const ColumnRefItem<R>* __restrict__ items, BatchMap bm) {
  VBlock vb;
  const ColumnRefItem<R>* it = batch_member(items, bm, vb);
  if (!it) return;
  const FastArgs<R> a = it->a;
  column_reference_body(a, vb);
}
template <class R>
void launch_column_reference(hipStream_t st, const FastArgs<R>& a) {
  const unsigned n2 = static_cast<unsigned>(a.g.nx) * a.g.ny;
  const dim3 grid((n2 + 63) / 64), blk(64, kRefWaves);
  if (recorder()) {
    record_launch(reinterpret_cast<const void*>(&k_column_reference_batch<R>), blk, 0,
                  ColumnRefItem<R>{a, 0, 0}, static_cast<int>(grid.x), 1);
    return;
  }
  hipLaunchKernelGGL(k_column_reference<R>, grid, blk, 0, st, a);
}

// FORM: 0 full and 1 perturbation form on flat grids, marching up; 2 and 3 the
// same marching down; 4 + REF on terrain.  SUMS: the level means are summed
// from their partials in the prologue (a kernel of its own: the branch in the
// common one cost substeps that do not take it 1.5 %).
template <class R, int FORM, int KIND, int TYV, bool SUMS>
__device__ __forceinline__ void fast_form(const FastArgs<R>& a, int tiles_x, int tiles, int nkc,
                                          double* part_out, const VBlock& vb) {
  if constexpr (FORM >= 4)
    fast_terrain_body<R, FORM - 4, KIND, TYV>(a, tiles_x, tiles, nkc, part_out, vb);
  else
    fast_body<R, (FORM & 1) != 0, KIND, TYV, (FORM & 2) != 0, SUMS>(a, tiles_x, tiles, nkc, part_out, vb);
}

template <class R, int FORM, int KIND, int TYV, bool SUMS>
__global__ __launch_bounds__(TX * TYV) void k_fast_column(FastArgs<R> a, int tiles_x, int tiles,
                                                          int nkc, double* part_out) {
  fast_form<R, FORM, KIND, TYV, SUMS>(a, tiles_x, tiles, nkc, part_out, hw_block());
}
template <class R, int FORM, int KIND, int TYV>
__global__ __launch_bounds__(TX * TYV) void k_fast_column_batch(
    const FastItem<R>* __restrict__ items, BatchMap bm) {
  VBlock vb;
  const FastItem<R>* it = batch_member(items, bm, vb);
  if (!it) return;
  // the member's arguments, read once before the kernel stores anything
  const FastArgs<R> a = it->a;
  fast_form<R, FORM, KIND, TYV, false>(a, it->tiles_x, it->tiles, it->nkc, it->part_out, vb);
}

template <class R, int FORM, int TYV>
void launch_fast_kind(hipStream_t st, const FastArgs<R>& a, int nkc, double* part_out) {
  const int tx = (a.g.nx + TX - 1) / TX, ty = (a.g.ny + TYV - 1) / TYV;
  const int tiles = tx * ty;
  const dim3 grid(tiles * nkc), blk(TX, TYV, 1);
  // per-level LDS: the longest chunk plus the levels below and above it (the
  // column reference form has no per-level values)
  const size_t lds = FORM == 4 + REF_COLUMN
                         ? 0
                         : static_cast<size_t>((a.g.nz + nkc - 1) / nkc + 3) * NLV * sizeof(R);
  const int kind = (a.first ? 1 : 0) | (a.last ? 2 : 0);
  if (recorder()) {
    const void* fns[4] = {reinterpret_cast<const void*>(&k_fast_column_batch<R, FORM, 0, TYV>),
                          reinterpret_cast<const void*>(&k_fast_column_batch<R, FORM, 1, TYV>),
                          reinterpret_cast<const void*>(&k_fast_column_batch<R, FORM, 2, TYV>),
                          reinterpret_cast<const void*>(&k_fast_column_batch<R, FORM, 3, TYV>)};
    record_launch(fns[kind], blk, lds, FastItem<R>{a, tx, tiles, nkc, part_out, 0, 0},
                  static_cast<int>(grid.x), 1);
    return;
  }
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, blk, lds, st, a, tx, tiles, nkc, part_out);
  };
  if constexpr (FORM < 4) {
    if (a.lev_part) {
      switch (kind) {
        case 0: go(k_fast_column<R, FORM, 0, TYV, true>); break;
        case 1: go(k_fast_column<R, FORM, 1, TYV, true>); break;
        case 2: go(k_fast_column<R, FORM, 2, TYV, true>); break;
        default: go(k_fast_column<R, FORM, 3, TYV, true>); break;
      }
      return;
    }
  }
  switch (kind) {
    case 0: go(k_fast_column<R, FORM, 0, TYV, false>); break;
    case 1: go(k_fast_column<R, FORM, 1, TYV, false>); break;
    case 2: go(k_fast_column<R, FORM, 2, TYV, false>); break;
    default: go(k_fast_column<R, FORM, 3, TYV, false>); break;
  }
}

template <class R>
void launch_fast_column(hipStream_t st, const FastArgs<R>& a, bool terrain, int code,
                        double* part_out, int* nparts_out) {
  // code: level chunks (low 4 bits), tile height (bit 4 set: 4 rows, else
  // 8), bit 6 set: every substep marches upwards (a.down ignored)
  int nkc = code & 15;
  const bool down = a.down && (code & 64) == 0;
  const bool ty4 = ((code >> 4) & 1) != 0;
  if (nparts_out) *nparts_out = fast_column_parts(a.g.nx, a.g.ny);
  if (nkc < 1) nkc = 1;
  if (nkc > a.g.nz) nkc = a.g.nz;
  auto go = [&](auto form, double* part) {
    if (ty4) launch_fast_kind<R, decltype(form)::value, 4>(st, a, nkc, part);
    else launch_fast_kind<R, decltype(form)::value, 8>(st, a, nkc, part);
  };
  using std::integral_constant;
  if (terrain) {
    if (a.col_ref) {
      launch_column_reference(st, a);
      go(integral_constant<int, 4 + REF_COLUMN>{}, nullptr);
      return;
    }
    if constexpr (sizeof(R) == 4) {
      if (a.base.drho) {  // perturbation form on terrain (per-cell bases)
        go(integral_constant<int, 4 + REF_BASE>{}, nullptr);
        return;
      }
    }
    go(integral_constant<int, 4 + REF_LEVEL>{}, part_out);
    return;
  }
  const bool pert = a.base.rho != nullptr;  // flat, doubly periodic
  if (down && nkc == 1) {  // whole columns marched from the top down
    if (pert) go(integral_constant<int, 3>{}, part_out);
    else go(integral_constant<int, 2>{}, part_out);
  } else {
    if (pert) go(integral_constant<int, 1>{}, part_out);
    else go(integral_constant<int, 0>{}, part_out);
  }
}

// Level partials per level: one per 64-column row segment.
int fast_column_parts(int nx, int ny) { return ((nx + TX - 1) / TX) * ny; }

template void launch_fast_column<float>(hipStream_t, const FastArgs<float>&, bool, int, double*,
                                        int*);
template void launch_fast_column<double>(hipStream_t, const FastArgs<double>&, bool, int,
                                         double*, int*);

}  // namespace gwm
