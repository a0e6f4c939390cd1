// gd_strip.hpp -- tendency rows in registers for the rows away from the polar
// filter, in the fast and slow passes of an integrator call.
//
// A tile is a segment of kSeg longitudes (as the row tiles of gd_tend.hpp: thread
// t < W owns longitude i0 + t) by a group of rows, and marches north over the
// group.  What a point shares with its northern or western neighbour (sqrt gd,
// u, row sums, mass fluxes) is formed once per row instead of once per tile
// that reads it: one row takes one square root and one division for the winds
// where a row tile takes six and up to five, and 7 loads where it takes 22.
// Longitude neighbours come from the next lane by DPP.  A wave's end lanes
// load their outer neighbour's column themselves (lane 0 the one west, lane 63
// the one east) and form what they need of it, so the waves of a tile run
// without LDS and without a barrier; only the beta partials of phase C are
// added over the tile's four waves at its end.
//
// Every value is formed by the expressions of seg_eval (gd_tend.hpp) in their
// order, and the partials are added over the same threads as block_sum_n, so a
// strip tile gives the bits of the row tiles it replaces.  A division by a
// row constant takes its reciprocal, rounded once on the host, and a
// remainder step, which rounds as the division does.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "gd_common.hpp"
#include "gd_device.hpp"

namespace gd {

// Coefficients of one row in the compute type, with the reciprocals of the
// constants the stencils divide by.
template <typename CT>
struct StripRow {
  CT f, c, c1, c2, hc, fdlon, r_fdlon, hdlat, r_hdlat;
  CT kul, kut, kvl, kvt;
  double hcos, fcos, fdlon_d, r_fdlon_d, fdlat_d, r_fdlat_d;
};

// Row `row` of the table, through the constant address space (no kernel
// writes it): scalar loads.
template <typename CT>
__device__ __forceinline__ StripRow<CT> strip_row(const Args &a, int row) {
  const __attribute__((address_space(4))) StripRow<CT> *t =
      (const __attribute__((address_space(4))) StripRow<CT> *)a.strip_coef + min(max(row, 0), a.M - 1);
  StripRow<CT> b;
  b.f = t->f;
  b.c = t->c;
  b.c1 = t->c1;
  b.c2 = t->c2;
  b.hc = t->hc;
  b.fdlon = t->fdlon;
  b.r_fdlon = t->r_fdlon;
  b.hdlat = t->hdlat;
  b.r_hdlat = t->r_hdlat;
  b.kul = t->kul;
  b.kut = t->kut;
  b.kvl = t->kvl;
  b.kvt = t->kvt;
  b.hcos = t->hcos;
  b.fcos = t->fcos;
  b.fdlon_d = t->fdlon_d;
  b.r_fdlon_d = t->r_fdlon_d;
  b.fdlat_d = t->fdlat_d;
  b.r_fdlat_d = t->r_fdlat_d;
  return b;
}

// x / d with r = 1/d rounded to nearest: Markstein's division by a divisor known
// in advance, one product and two fused steps, which rounds as the division does
// where nothing over- or underflows (Brisebarre, Muller and Raina, IEEE
// Transactions on Computers 53(8), 2004); the fixup gives zeros, infinities and
// NaN the division's result.
__device__ __forceinline__ double divu(double x, double d, double r) {
  double q = x * r;
  q = __builtin_fma(__builtin_fma(-q, d, x), r, q);
  return __builtin_amdgcn_div_fixup(q, d, x);
}
__device__ __forceinline__ float divu(float x, float d, float r) {
  float q = x * r;
  q = __builtin_fmaf(__builtin_fmaf(-q, d, x), r, q);
  return __builtin_amdgcn_div_fixupf(q, d, x);
}

// The value of the next lane east (lane + 1) or west (lane - 1), around the
// wave.
constexpr int kDppEast = 0x134, kDppWest = 0x13C;  // wave_rol:1, wave_ror:1
__device__ __forceinline__ double east(double x) { return dpp_mov<kDppEast>(x); }
__device__ __forceinline__ float east(float x) { return dpp_mov<kDppEast>(x); }
__device__ __forceinline__ double west(double x) { return dpp_mov<kDppWest>(x); }
__device__ __forceinline__ float west(float x) { return dpp_mov<kDppWest>(x); }

// The field value at byte offset `off` (32 bits: the base stays in scalar
// registers).
__device__ __forceinline__ double ld(const double *base, unsigned off) {
  return *(const double *)((const char *)base + off);
}
__device__ __forceinline__ void st(double *base, unsigned off, double v) { *(double *)((char *)base + off) = v; }

// One row of a state in the fast pass.  Suffix e, w: the value one longitude
// east or west; Fyp, Wp: of the row before.
template <typename CT>
struct FastRow {
  double gd, gde, h, he, G, Ge, U, V, Fx, Fxw, Fyp;
  CT t, Q, Qw, W, Wp;  // f + c u, (f + c u) U, V + V(i+1)
};

// ... and in the slow pass, where gd does not change.  Y, Z: v cos,
// (v + v(i+1)) cos.
template <typename CT>
struct SlowRow {
  CT U, Ue, Uw, V, Ve, Vw, u, ue, uw, Y, Z;
};

template <typename CT>
__device__ __forceinline__ CT adv(bool upwind, CT a2, CT a1, CT x, CT xp, CT xm, CT b) {
  if (!upwind) return a2 * xp - a1 * xm;
  return a2 * (x + xp) - b * fabs(a2) * (xp - x) - a1 * (x + xm) + b * fabs(a1) * (x - xm) - (a2 - a1) * x;
}

// Rows of one group's wave sums in LDS: [row][wave][6].
__host__ __device__ constexpr size_t strip_lds_bytes(int rows) { return (size_t)rows * 4 * 6 * sizeof(double); }

// Phase a.phase (PH_A, PH_B or PH_C) of tile t = (member, group of a.strip_r
// rows, segment), segment fastest.  live = false: no stores (a spare tile).
// FOLD 1: phase A's state is s_fold + dt beta Tc, formed where a row is loaded,
// and stored to s_in.  FOLD 2: phase C's state is S0 + hdt Tb, which phase B
// then need not have stored.  `red`: 24 doubles.
template <typename CT, int PASS, bool FULL, int FOLD>
__device__ __forceinline__ void strip_tile(const Args &a, int t, bool live, unsigned char *smem, double *red) {
  const int N = a.N, nseg = a.nseg, tid = ltid(), lane = threadIdx.x & 63, wv = (threadIdx.x >> 6) & 3;
  const int seg = t % nseg, q = t / nseg, grp = q % a.strip_ngroup, m = q / a.strip_ngroup;
  const Member mb = member_at(a, a.m0 + m);
  const int r0 = a.strip_a + grp * a.strip_r, r1 = min(r0 + a.strip_r - 1, a.strip_b);
  const int i0 = seg * kSeg, W = min(N - i0, kSeg);
  const bool first = lane == 0, last = lane == 63, pc = a.phase == PH_C;
  double *sums = (double *)smem;
  const double dtb = FOLD == 1 ? fold_step(a, mb, red) : (FOLD == 2 ? a.hdt : 0.0);
  // (a wave past the segment's end has nothing to do but its zero sums)
  const bool busy = __builtin_amdgcn_readfirstlane(wv * 64) < W;
  if (busy) {
    const bool own = live && tid < W;
    auto wrap = [N](int i) { return (unsigned)(i < 0 ? i + N : (i >= N ? i - N : i)) * 8u; };
    // this column, the outer neighbour of an end lane (else this column), and
    // the one after it for lane 63
    const unsigned P8 = (unsigned)a.pitch * 8u;
    // (threads past the eastern neighbour repeat a column, so that every one
    // is inside the row)
    const int ic = i0 + min(tid, W + 1);
    const unsigned c0 = wrap(ic), cx = wrap(ic + (last ? 1 : (first ? -1 : 0)));
    const int si = FOLD == 1 ? a.s_fold : (FOLD == 2 ? a.s0 : a.s_in);
    const double *gd = mb.st(si, FGD), *Ug = mb.st(si, FU), *Vg = mb.st(si, FV), *hg = mb.ghs();
    const double *tg = FOLD == 2 ? mb.tb(CDGD) : mb.tc(CDGD), *tu = FOLD == 2 ? mb.tb(CDU) : mb.tc(CDU);
    const double *tv = FOLD == 2 ? mb.tb(CDV) : mb.tc(CDV);
    auto in = [&](const double *f, const double *tc, unsigned o) {
      if constexpr (FOLD) return ld(f, o) + dtb * ld(tc, o);
      return ld(f, o);
    };
    const double *ug = mb.st(a.s_in, Fu), *vg = mb.st(a.s_in, Fv);
    // what the epilogue reads at the point (S0, or Tb in phase C) and where it
    // writes
    const double *pu = pc ? mb.tb(CDU) : mb.st(a.s0, FU), *pv = pc ? mb.tb(CDV) : mb.st(a.s0, FV);
    const double *pg = pc ? mb.tb(CDGD) : mb.st(a.s0, FGD);
    double *ou = pc ? mb.tc(CDU) : mb.st(a.s_out, FU), *ov = pc ? mb.tc(CDV) : mb.st(a.s_out, FV);
    double *og = pc ? mb.tc(CDGD) : mb.st(a.s_out, FGD);
    auto finish = [&](int j, const StripRow<CT> &c, double du, double dv, double dg, double xu, double xv, double xg) {
      const unsigned o = (unsigned)j * P8 + c0;
      double pq[6] = {0, 0, 0, 0, 0, 0};
      if (own) {
        if (pc) {
          st(ou, o, du);
          st(ov, o, dv);
          st(og, o, dg);
          pq[0] += xu * du * c.fcos;
          pq[1] += du * du * c.fcos;
          pq[2] += xv * dv * c.hcos;
          pq[3] += dv * dv * c.hcos;
          pq[4] += xg * dg * c.fcos;
          pq[5] += dg * dg * c.fcos;
        } else {
          if (FOLD == 1) {
            st(mb.st(a.s_in, FU), o, xu);
            st(mb.st(a.s_in, FV), o, xv);
            st(mb.st(a.s_in, FGD), o, xg);
          }
          if (a.phase != PH_B || j < a.s2_lo || j > a.s2_hi) {
            st(ou, o, xu + a.hdt * du);
            st(ov, o, xv + a.hdt * dv);
            st(og, o, xg + a.hdt * dg);
          }
          if (a.phase == PH_B) {
            st(mb.tb(CDU), o, du);
            st(mb.tb(CDV), o, dv);
            st(mb.tb(CDGD), o, dg);
          }
        }
      }
      if (pc) wave_sums_to<6>(pq, sums + ((j - r0) * 4 + wv) * 6);
    };
    if constexpr (PASS == 1) {
      struct Ld {
        double g, U, V, h, gx, x, hx, u, ux;
      };
      // x: U of the western neighbour for lane 0, V of the eastern for lane 63
      const unsigned cuv = cx;
      const double *xg_ = first ? Ug : Vg, *xt_ = first ? tu : tv;
      auto load = [&](int row) {
        const unsigned o = (unsigned)row * P8;
        Ld l;
        l.g = in(gd, tg, o + c0);
        l.U = in(Ug, tu, o + c0);
        l.V = in(Vg, tv, o + c0);
        l.h = ld(hg, o + c0);
        l.gx = in(gd, tg, o + cx);
        l.x = in(xg_, xt_, o + cuv);
        l.hx = ld(hg, o + cx);
        l.u = FULL ? ld(ug, o + c0) : 0.0;
        l.ux = FULL ? ld(ug, o + cx) : 0.0;
        return l;
      };
      auto row_from = [&](const Ld &l, const StripRow<CT> &c) {
        FastRow<CT> x;
        x.gd = l.g;
        x.h = l.h;
        x.U = l.U;
        x.V = l.V;
        x.G = sqrt(l.g);
        const double Gx = sqrt(l.gx);
        const double ge = east(x.G), de = east(l.g), he = east(l.h), ve = east(l.V);
        x.Ge = last ? Gx : ge;
        x.gde = last ? l.gx : de;
        x.he = last ? l.hx : he;
        const double Ve = last ? l.x : ve;
        // update_state: u = U * 2 / (G(i) + G(i+1))  (dycore_mod.F90:636-640)
        const CT u = FULL ? (CT)l.u : ((CT)l.U * (CT)2) / ((CT)x.G + (CT)x.Ge);
        const CT ux = FULL ? (CT)l.ux : ((CT)l.x * (CT)2) / ((CT)Gx + (CT)x.G);
        x.t = c.f + c.c * u;
        x.Q = x.t * (CT)l.U;
        const CT Qx = (c.f + c.c * ux) * (CT)l.x, Qw = west(x.Q);
        x.Qw = first ? Qx : Qw;
        x.W = (CT)l.V + (CT)Ve;
        x.Fx = (x.G + x.Ge) * l.U;
        const double Fxx = (Gx + x.G) * l.x, Fw = west(x.Fx);
        x.Fxw = first ? Fxx : Fw;
        return x;
      };
      Ld l0 = load(r0 - 1), l1 = load(r0), l2 = load(r0 + 1);
      StripRow<CT> cp = strip_row<CT>(a, r0 - 1), cs = strip_row<CT>(a, r0);
      FastRow<CT> s;
      {
        const FastRow<CT> p = row_from(l0, cp);
        s = row_from(l1, cs);
        s.Fyp = (p.G + s.G) * p.V * cp.hcos;
        s.Wp = p.W;
      }
      for (int j = r0; j <= r1; ++j) {
        const unsigned o = (unsigned)j * P8 + c0;
        const double xu = FOLD == 1 ? s.U : ld(pu, o), xv = FOLD == 1 ? s.V : ld(pv, o);
        const double xg = FOLD == 1 ? s.gd : ld(pg, o);
        const Ld l = l2;
        l2 = load(min(j + 2, r1 + 1));
        const StripRow<CT> cn = strip_row<CT>(a, j + 1);
        FastRow<CT> n = row_from(l, cn);
        const double Fy = (s.G + n.G) * s.V * cs.hcos;
        n.Fyp = Fy;
        n.Wp = s.W;
        // (seg_eval's u, v and mass equations)
        const CT fv = (CT)0.25 * s.t * (cs.c1 * s.Wp + cs.c2 * s.W);
        const double dphi = s.gde + s.he - s.gd - s.h;
        const CT upgf = divu((CT)0.5 * ((CT)s.G + (CT)s.Ge), cs.fdlon, cs.r_fdlon) * (CT)dphi;
        const CT fu = (CT)0.25 * (s.Q + s.Qw + n.Q + n.Qw);
        const double dphn = n.gd + n.h - s.gd - s.h;
        const CT vpgf = divu((CT)0.5 * ((CT)s.G + (CT)n.G), cs.hdlat, cs.r_hdlat) * cs.hc * (CT)dphn;
        const double mdl = divu((s.Fx - s.Fxw) * 0.5, cs.fdlon_d, cs.r_fdlon_d);
        const double mdp = divu((Fy - s.Fyp) * 0.5, cs.fdlat_d, cs.r_fdlat_d);
        finish(j, cs, (double)(fv - upgf), (double)(-fu - vpgf), -mdl - mdp, xu, xv, xg);
        s = n;
        cs = cn;
      }
    } else {
      const bool upwind = a.upwind != 0;
      const CT bl = (CT)a.beta_lon, bt = (CT)a.beta_lat;
      const unsigned cy = last ? wrap(ic + 2) : c0;
      struct Ld {
        double g, gx, gy, U, V, Ux, Vx, u, v, ux, vx;  // g, gx, gy: of the row after
      };
      auto load = [&](int row) {
        const unsigned o = (unsigned)row * P8, on = o + P8;
        Ld l;
        l.g = in(gd, tg, on + c0);
        l.gx = in(gd, tg, on + cx);
        l.gy = FULL ? 0.0 : in(gd, tg, on + cy);
        l.U = in(Ug, tu, o + c0);
        l.V = in(Vg, tv, o + c0);
        l.Ux = in(Ug, tu, o + cx);
        l.Vx = in(Vg, tv, o + cx);
        l.u = FULL ? ld(ug, o + c0) : 0.0;
        l.v = FULL ? ld(vg, o + c0) : 0.0;
        l.ux = FULL ? ld(ug, o + cx) : 0.0;
        l.vx = FULL ? ld(vg, o + cx) : 0.0;
        return l;
      };
      const unsigned op = (unsigned)(r0 - 1) * P8;
      double G = 0, Gx = 0, Gy = 0;  // sqrt gd of the row to come
      if (!FULL) {
        G = sqrt(in(gd, tg, op + c0));
        Gx = sqrt(in(gd, tg, op + cx));
        Gy = sqrt(in(gd, tg, op + cy));
      }
      auto row_from = [&](const Ld &l, const StripRow<CT> &c) {
        CT u, v, ux, vx;
        if constexpr (FULL) {
          u = (CT)l.u;
          v = (CT)l.v;
          ux = (CT)l.ux;
          vx = (CT)l.vx;
        } else {
          const double Gn = sqrt(l.g), Gxn = sqrt(l.gx), ge = east(G);
          const double Ge = last ? Gx : ge;
          u = ((CT)l.U * (CT)2) / ((CT)G + (CT)Ge);
          v = ((CT)l.V * (CT)2) / ((CT)G + (CT)Gn);
          ux = ((CT)l.Ux * (CT)2) / ((CT)Gx + (CT)Gy);
          vx = ((CT)l.Vx * (CT)2) / ((CT)Gx + (CT)Gxn);
          G = Gn;
          Gx = Gxn;
          Gy = sqrt(l.gy);
        }
        SlowRow<CT> x;
        const CT Ux = (CT)l.Ux, Vx = (CT)l.Vx;
        auto pair = [&](CT y, CT yx, CT &e, CT &w) {
          const CT ye = east(y), yw = west(y);
          e = last ? yx : ye;
          w = first ? yx : yw;
        };
        x.U = (CT)l.U;
        x.V = (CT)l.V;
        x.u = u;
        pair(x.U, Ux, x.Ue, x.Uw);
        pair(x.V, Vx, x.Ve, x.Vw);
        pair(u, ux, x.ue, x.uw);
        const CT ve = east(v);
        x.Y = v * c.hc;
        x.Z = (v + (last ? vx : ve)) * c.hc;
        return x;
      };
      Ld l0 = load(r0 - 1), l1 = load(r0);
      StripRow<CT> cs = strip_row<CT>(a, r0 - 1);
      SlowRow<CT> p = row_from(l0, cs), s;
      l0 = load(r0 + 1);
      cs = strip_row<CT>(a, r0);
      s = row_from(l1, cs);
      CT Up = p.U, Vp = p.V, Yp = p.Y, Zp = p.Z;
      for (int j = r0; j <= r1; ++j) {
        const unsigned o = (unsigned)j * P8 + c0;
        const double xu = FOLD == 1 ? in(Ug, tu, o) : ld(pu, o), xv = FOLD == 1 ? in(Vg, tv, o) : ld(pv, o);
        const double xg = FOLD == 1 ? in(gd, tg, o) : ld(pg, o);
        const Ld l = l0;
        l0 = load(min(j + 2, r1 + 1));
        const StripRow<CT> cn = strip_row<CT>(a, j + 1);
        const SlowRow<CT> n = row_from(l, cn);
        const CT ual = cs.kul * adv<CT>(upwind, s.u + s.ue, s.u + s.uw, s.U, s.Ue, s.Uw, bl);
        const CT uat = cs.kut * adv<CT>(upwind, s.Z, Zp, s.U, n.U, Up, bt);
        const CT val = cs.kvl * adv<CT>(upwind, s.u + n.u, s.uw + n.uw, s.V, s.Ve, s.Vw, bl);
        const CT vat = cs.kvt * adv<CT>(upwind, s.Y + n.Y, s.Y + Yp, s.V, n.V, Vp, bt);
        finish(j, cs, (double)(-ual - uat), (double)(-val - vat), 0.0, xu, xv, xg);
        Up = s.U;
        Vp = s.V;
        Yp = s.Y;
        Zp = s.Z;
        s = n;
        cs = cn;
      }
    }
  } else if (pc) {
    for (int x = lane; x < (r1 - r0 + 1) * 6; x += 64) sums[((x / 6) * 4 + wv) * 6 + x % 6] = 0.0;
  }
  if (pc) {
    // ((wave 0 + wave 1) + wave 2) + wave 3, as block_sum_n
    __syncthreads();
    for (int x = tid; x < (r1 - r0 + 1) * 6 && live; x += kBlock) {
      const int row = x / 6, p = x - row * 6;
      double v = sums[row * 24 + p];
      for (int k = 1; k < 4; ++k) v += sums[row * 24 + k * 6 + p];
      mb.part()[(((size_t)(r0 + row) * 3 + p / 2) * nseg + seg) * 2 + (p & 1)] = v;
    }
  }
}

// The strip tiles of a launch: blocks from `base` on, TILES tiles side by side
// in each, every XCD a contiguous run (base and strip_blk are multiples of
// kXcd).  A spare tile past the last does the last one's work and barriers
// without its stores.
template <typename CT, int PASS, bool FULL, int TILES = 1, int FOLD = 0>
__device__ __forceinline__ void strip_block(const Args &a, int base, unsigned char *smem, double *red) {
  const int b = (int)blockIdx.x - base;
  const int t0 = ((b % kXcd) * (a.strip_blk / kXcd) + b / kXcd) * TILES;
  if (t0 >= a.nstrip) return;
  const int s = TILES > 1 ? (int)threadIdx.x / kBlock : 0, t = t0 + s;
  strip_tile<CT, PASS, FULL, FOLD>(a, __builtin_amdgcn_readfirstlane(min(t, a.nstrip - 1)), t < a.nstrip,
                                   smem + s * strip_lds_bytes(a.strip_r), red + s * 4 * 6);
}

}  // namespace gd
