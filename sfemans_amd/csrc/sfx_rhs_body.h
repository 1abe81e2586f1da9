// Right-hand-side assembly from Gauss-point values (body for gfx950 and the
// CPU emulator).
//
// rhs_3x3 (SOURCES/SOLVER/assembling_rhs.F90:5-126, without the tensor
// options) and qs_00_gauss (SOURCES/SOLVER/fem_rhs_axi.F90:940-987) scatter
// per-element contributions to the nodes with VecSetValues(ADD_VALUES), one
// element after the other.  Here each output entry is gathered by one thread
// from the node's (element, local node) list in element order, so the sums
// are formed in the reference's order, deterministically and without atomics.
// For rhs_3x3 the element contributions are formed first, one thread per
// (element, mode) reading the Gauss array once, into a work array.
//
//   wgt(e,l)     = rj(l,e) * ray(l,e)                 (assembling_rhs.F90:73)
//   vb(n, ki, m) = sum_(e,i) sum_l ww(i,l) wgt(e,l) rhs(7e+l, comp(ki), m)
// with comp = (1,4,5) for vb_145 and (2,3,6) for vb_236 (:75-95).
#pragma once
#include "sfx_gather.h"
#include "sfx_geom.h"
#include "sfx_portable.h"

namespace sfx {

struct RhsArgs {
  const int64_t* adj_ptr;   // (np+1)
  const int32_t* adj_ent;   // e*6 + i
  const double* wgt;        // (7, me): rj * ray
  const double* tab;        // ww(6,7), ...
  int64_t me, np, G;
  int M;                    // modes (or columns for the scalar assembly)
  double scale;             // multiplies the result (-1 for the -rotv_v share)
  // rhs_3x3
  const double* rhs;        // (G, 6, M)
  double* v145;             // (np, 3, M)
  double* v236;             // (np, 3, M)
  // qs_00_gauss (ncols independent right-hand sides)
  const int32_t* jj;        // (6, me)
  const double* heat_capa;  // (me)
  const double* ff;         // (np, M) nodal source
  const double* ffg;        // (G, M) Gauss source
  double* vect;             // (np, M)
  double* elo;              // per-element nodal contributions, index ((6e+i)*6 + k)*M + m
  int64_t n_rhs, n_ff, n_ffg, n_out, n_adj, n_elo;
  // full NS right-hand side (rhs_ns_tile_body); a null field counts as zero
  const double* rr;         // (2, np) node coordinates
  const int32_t* lmode;     // (M) mode numbers
  const double* v1m;        // (np, 6, M) time-derivative term
  const double* fsrc;       // (np, 6, M) nodal momentum source
  const double* pres;       // (np, 2, M) pressure on the velocity mesh
  const double* pinc;       // (np, 2, M) pressure increment on the velocity mesh
  const double* tens;       // (3, G, 6, M) opt_tensor of rhs_3x3
  double rsign;             // sign of the Gauss field rhs: -1 for -rotv_v, +1 for rhs_3x3's rhs_in
  // velocity imposed in solids by penalty (computing_rhs_gauss.F90:103-121):
  // isign * SUM(imp*ww) added to the mode slot imp_slot (-1: none)
  const double* imp;        // (np, 6) 3 u_imposed / (2 dt)
  int imp_slot;
  double isign;
  double* gout;             // (G, 6, M): with the Gauss output, rhs without fp goes here
  int64_t n_v1m, n_fsrc, n_pres, n_pinc, n_tens, n_imp, n_gout;
};

// Work item gid of the element kernels -> (element e, mode or column m).  A
// wave takes ELEM_EB consecutive elements x ELEM_MB consecutive modes, modes
// fastest: a load of one Gauss plane then touches the 7 * ELEM_EB
// consecutive points of those elements (two cache lines) for ELEM_MB planes
// instead of 64 planes, and the stores still write ELEM_MB consecutive modes
// (one whole line) of each entry.
constexpr int ELEM_EB = 4, ELEM_MB = 16;
SFX_DEV void elem_item(int64_t gid, int M, int64_t& e, int& m) {
  const int64_t w = gid / 64;
  const int lane = (int)(gid % 64);
  const int nmb = (M + ELEM_MB - 1) / ELEM_MB;
  e = (w / nmb) * ELEM_EB + lane / ELEM_MB;
  m = (int)(w % nmb) * ELEM_MB + lane % ELEM_MB;
}
inline int64_t elem_items(int64_t me, int M) {
  return ((me + ELEM_EB - 1) / ELEM_EB) * (int64_t)((M + ELEM_MB - 1) / ELEM_MB) * 64;
}

// Element share of rhs_3x3, one thread per (element, mode) (elem_item):
//   elo(6e+i, k, m) = sum_l ww(i,l) wgt(e,l) rhs(7e+l, comp k, m)
// (the values the reference adds with VecSetValues, assembling_rhs.F90:73-95).
// A thread reads the 7 consecutive Gauss values of its element per
// component; the stores of a wave cover consecutive modes.  rhs_gather_block
// then sums the entries of each node in element order.
SFX_DEV void rhs_elem_body(const RhsArgs& a, int64_t gid) {
  int64_t e;
  int m;
  elem_item(gid, a.M, e, m);
  if (e >= a.me || m >= a.M) return;
  double w[7], r[7][6];
#pragma unroll
  for (int l = 0; l < 7; ++l) {
    w[l] = a.wgt[7 * e + l];
    const int64_t gi = 7 * e + l + a.G * 6 * m;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      SFX_CHECK("rhs load", gi + a.G * k, a.n_rhs);
      r[l][k] = a.rhs[gi + a.G * k];
    }
  }
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    double loc[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int l = 0; l < 7; ++l) {
      const double c = a.tab[i + 6 * l] * w[l];
#pragma unroll
      for (int k = 0; k < 6; ++k) loc[k] = fma(c, r[l][k], loc[k]);
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const int64_t o = ((6 * e + i) * 6 + k) * a.M + m;
      SFX_CHECK("elo store", o, a.n_elo);
      a.elo[o] = loc[k];
    }
  }
}

// Full explicit NS right-hand side of rhs_ns_gauss_3x3 without the penalty
// options (SOURCES/SOLVER/computing_rhs_gauss.F90:7-146) fused with the
// element share of rhs_3x3:
//   rhs(l, :) = (ft + fp_inc + fs - rotv_v(7e+l, :)) + fp         (:100, :145)
// (rsign = -1; with rsign = +1 and the other fields absent it is rhs_3x3's
// own rhs_in, so the kernel also serves rhs_3x3 with opt_tensor)
//   ft = SUM(V1m*ww), fs = SUM(ff*ww),
//   fp = (-d_r P_c, -d_r P_s, -P_s/ray*m, P_c/ray*m, -d_z P_c, -d_z P_s) (:69-97)
// with P and P_inc the pressure injected onto the velocity mesh; then
//   elo(6e+i, k, m) = sum_l ww(i,l) wgt(e,l) rhs(l, k)   as rhs_elem_body.
// With TENSOR, rhs_3x3's opt_tensor T(3, G, 6, M) (assembling_rhs.F90:56-121):
// node i of component k adds, per Gauss point,
//   (ww(i,l) f_tensor(k) + d_r phi_i T(k/2, k%2) + d_z phi_i T(k/2, 4 + k%2)) wgt(e,l)
// with f_tensor the 1/r and mode terms (row k/2 of T, its cos columns for
// even k, sin for odd).
// The Gauss array rhs_gauss is never stored.
//
// What bounds it: HBM (rotv_v and the tensor are 192 bytes per Gauss point and
// mode).  A work-group takes RNS_E elements and MC modes of them, one mode
// at a time: one thread per Gauss point loads rotv_v and the tensor (224
// consecutive points of each plane, whole lines), one per (element, node) the
// nodal fields, which are added at the nodes (V1m + ff, P + P_inc) and
// interpolated from LDS; each point's weights of the shape values and of the
// reference derivatives (18 numbers, as in the adjoint) go to LDS, and one
// thread per (element, component) sums them for the six nodes, keeping MC
// modes so that it stores 64-byte runs (MC = RNS_MC).  (One thread per (element, mode) with all
// of its fields in registers took 418 registers, one wave per SIMD, and each of
// its loads touched 40 lines: 1.4 TB/s, 6.15 ms with the gather at 102,720
// triangles, M = 48, against 3.04 ms, 3.8 TB/s in this kernel.)
constexpr int RNS_E = 32, RNS_MC = 8, RNS_THREADS = 256;
constexpr int RNS_PT = 7 * RNS_E;              // Gauss points
constexpr int RNS_EROW = 6 * 8 + 2;            // doubles per element of the staged nodal sums (8 per node)
constexpr int RNS_SK = RNS_PT + 2;             // doubles per weight
template <bool TENSOR>
constexpr int rns_smem_doubles() { return RNS_E * RNS_EROW + (TENSOR ? 18 : 6) * RNS_SK + 128; }
inline int64_t rns_blocks(int64_t me, int M, int MC) {
  return ((me + RNS_E - 1) / RNS_E) * (int64_t)((M + MC - 1) / MC);
}
// Modes per work-group: RNS_MC, or 2 where that would leave CUs idle while the
// others work through eight modes in series (two work-groups share a CU).  With
// the gather, without the tensor, one thread per (element, mode) / 8 modes / 2
// modes: 26.5 / 28.5 / 14.9 us at 400 triangles, M = 8 (13 work-groups of 8), 107
// / 114 / 104 at M = 128 (208), 62.8 / 57.9 / 52.0 at 3,192, M = 24 (300), but 65.6
// / 65.8 at M = 32 (400) with 8 / 2 modes; with the tensor 67.8 / 61.5 (300), 77.3
// / 79.1 at 6,084, M = 15 (382) and 76.1 / 78.7 (400).
constexpr int RNS_FEW = 2, RNS_FULL = 320;
inline int rns_modes(int64_t me, int M) { return rns_blocks(me, M, RNS_MC) < RNS_FULL ? RNS_FEW : RNS_MC; }

template <bool TENSOR, int MC>
SFX_DEV void rhs_ns_tile_body(const RhsArgs& a, int tid, int64_t bid, double* smem) {
  const int nmc = (a.M + MC - 1) / MC;
  const int64_t e0 = (bid / nmc) * RNS_E;      // the mode chunks of one set of elements are neighbours
  const int m0 = (int)(bid % nmc) * MC, m1 = m0 + MC < a.M ? m0 + MC : a.M;
  // staged nodal sums: written before a mode's first barrier, read between it
  // and the second, so the next mode's writes wait for every reader
  double* nod = smem;
  double* red = nod + RNS_E * RNS_EROW;
  double* tab = red + (TENSOR ? 18 : 6) * RNS_SK;
  for (int i = tid; i < 126; i += RNS_THREADS) tab[i] = a.tab[i];

  // this thread's node slot, Gauss point and (element, component)
  const bool nslot = tid < 6 * RNS_E && e0 + tid / 6 < a.me;
  const int64_t node = nslot ? (int64_t)a.jj[6 * e0 + tid] - 1 : 0;
  const int el = tid / 7, lg = tid % 7;
  const bool point = tid < RNS_PT && e0 + el < a.me;
  const int64_t p = point ? 7 * e0 + tid : 0;
  const int ke = tid % RNS_E, kc = tid / RNS_E;
  const bool sums = tid < 6 * RNS_E && e0 + ke < a.me;
  double a11 = 0, a12 = 0, a21 = 0, a22 = 0, iray = 0, wl = 0;
  SFX_SYNC();
  const double* w = tab + 6 * (point ? lg : 0);
  const double* d = tab + 42 + 12 * (point ? lg : 0);
  if (point) {
    double rn[6], zn[6], ray = 0;
#pragma unroll
    for (int n = 0; n < 6; ++n) {
      const int64_t jn = (int64_t)a.jj[6 * (e0 + el) + n] - 1;
      SFX_CHECK("rr load", 2 * jn + 1, 2 * a.np);
      rn[n] = a.rr[2 * jn];
      zn[n] = a.rr[2 * jn + 1];
      ray = fma(rn[n], w[n], ray);
    }
    p2_inverse_jacobian(rn, zn, d, a11, a12, a21, a22);
    iray = 1.0 / ray;
    wl = a.wgt[p];
  }
  double acc[MC][6];
#pragma unroll
  for (int q = 0; q < MC; ++q)
#pragma unroll
    for (int i = 0; i < 6; ++i) acc[q][i] = 0.0;

#pragma unroll
  for (int q = 0; q < MC; ++q) {
    const int m = m0 + q;
    if (m >= m1) continue;                     // uniform over the work-group
    // ---- loads of this mode
    double rv[6], T[TENSOR ? 3 : 1][6];
    if (point) {
      const int64_t g0 = p + a.G * 6 * (int64_t)m;
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        SFX_CHECK("rotv load", g0 + a.G * k, a.rhs ? a.n_rhs : 1 << 30);
        rv[k] = a.rhs ? a.rhs[g0 + a.G * k] : 0.0;
        if constexpr (TENSOR) {
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            SFX_CHECK("tensor load", c + 3 * (g0 + a.G * k), a.n_tens);
            T[c][k] = a.tens[c + 3 * (g0 + a.G * k)];
          }
        }
      }
    }
    if (nslot) {
      double s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      const int64_t i6 = node + a.np * 6 * (int64_t)m, i2 = node + a.np * 2 * (int64_t)m;
      if (a.v1m) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          SFX_CHECK("V1m load", i6 + a.np * k, a.n_v1m);
          s[k] = a.v1m[i6 + a.np * k];
        }
      }
      if (a.fsrc) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          SFX_CHECK("ff load", i6 + a.np * k, a.n_fsrc);
          s[k] += a.fsrc[i6 + a.np * k];
        }
      }
      if (a.pres) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          SFX_CHECK("P load", i2 + a.np * k, a.n_pres);
          s[6 + k] = a.pres[i2 + a.np * k];
        }
      }
      if (a.pinc) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          SFX_CHECK("P_inc load", i2 + a.np * k, a.n_pinc);
          s[6 + k] += a.pinc[i2 + a.np * k];
        }
      }
      if (a.imp && m == a.imp_slot) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          SFX_CHECK("imposed velocity load", node + a.np * k, a.n_imp);
          s[k] += a.isign * a.imp[node + a.np * k];
        }
      }
      double2* o = reinterpret_cast<double2*>(nod + (tid / 6) * RNS_EROW + (tid % 6) * 8);
#pragma unroll
      for (int k = 0; k < 4; ++k) o[k] = make_double2(s[2 * k], s[2 * k + 1]);
    }
    SFX_SYNC();
    // ---- the right-hand side at this point: weights of the shape values and
    // of d/dx, d/dy
    if (point) {
      const double mv = (double)a.lmode[m];
      double f[6], pv[2] = {0, 0}, pr[2] = {0, 0}, pz[2] = {0, 0};
#pragma unroll
      for (int k = 0; k < 6; ++k) f[k] = 0.0;
#pragma unroll
      for (int n = 0; n < 6; ++n) {
        const double2* s = reinterpret_cast<const double2*>(nod + el * RNS_EROW + n * 8);
        const double wn = w[n], dx = d[2 * n], dy = d[2 * n + 1];
        const double dr = fma(a11, dx, a12 * dy), dz = fma(a21, dx, a22 * dy);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const double2 x = s[k];
          f[2 * k] = fma(wn, x.x, f[2 * k]);
          f[2 * k + 1] = fma(wn, x.y, f[2 * k + 1]);
        }
        const double2 x = s[3];
        pv[0] = fma(wn, x.x, pv[0]); pv[1] = fma(wn, x.y, pv[1]);
        pr[0] = fma(dr, x.x, pr[0]); pr[1] = fma(dr, x.y, pr[1]);
        pz[0] = fma(dz, x.x, pz[0]); pz[1] = fma(dz, x.y, pz[1]);
      }
      const double mr = mv * iray;
#pragma unroll
      for (int k = 0; k < 6; ++k) f[k] = f[k] + a.rsign * rv[k];
      f[0] -= pr[0]; f[1] -= pr[1];
      f[2] -= mr * pv[1]; f[3] += mr * pv[0];
      f[4] -= pz[0]; f[5] -= pz[1];
      double* o = red + tid;
      if constexpr (TENSOR) {
        f[0] += (-mv * T[0][3] + T[1][2]) * iray;
        f[1] += (mv * T[0][2] + T[1][3]) * iray;
        f[2] += (-T[0][2] - mv * T[1][3]) * iray;
        f[3] += (-T[0][3] + mv * T[1][2]) * iray;
        f[4] -= T[2][3] * mr;
        f[5] += T[2][2] * mr;
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          const double tr = T[k / 2][k % 2] * wl, tz = T[k / 2][4 + k % 2] * wl;
          o[(3 * k) * RNS_SK] = f[k] * wl;
          o[(3 * k + 1) * RNS_SK] = fma(a11, tr, a21 * tz);
          o[(3 * k + 2) * RNS_SK] = fma(a12, tr, a22 * tz);
        }
      } else {
#pragma unroll
        for (int k = 0; k < 6; ++k) o[k * RNS_SK] = f[k] * wl;
      }
    }
    SFX_SYNC();
    // ---- sums over the element's points, the tables through scalar registers
    if (sums) {
      constexpr int KW = TENSOR ? 3 : 1;
      const SFX_KARG double* tb = (const SFX_KARG double*)a.tab;
      SFX_OPAQUE_S(tb);
      const double* src = red + KW * kc * RNS_SK + 7 * ke;
#pragma unroll
      for (int l = 0; l < 7; ++l) {
        double v[KW];
#pragma unroll
        for (int j = 0; j < KW; ++j) v[j] = src[j * RNS_SK + l];
#pragma unroll
        for (int n = 0; n < 6; ++n) {
          if constexpr (TENSOR) {
            const double dx = tb[42 + 2 * (n + 6 * l)], dy = tb[42 + 2 * (n + 6 * l) + 1];
            acc[q][n] = fma(tb[n + 6 * l], v[0], fma(dx, v[1], fma(dy, v[2], acc[q][n])));
          } else {
            acc[q][n] = fma(tb[n + 6 * l], v[0], acc[q][n]);
          }
        }
      }
    }
  }
  if (sums) {
#pragma unroll
    for (int n = 0; n < 6; ++n) {
      const int64_t o = ((6 * (e0 + ke) + n) * 6 + kc) * (int64_t)a.M + m0;
#pragma unroll
      for (int q = 0; q < MC; ++q) {
        if (m0 + q >= m1) continue;
        SFX_CHECK("elo store", o + q, a.n_elo);
        a.elo[o + q] = acc[q][n];
      }
    }
  }
}

// The Gauss values ft + fp_inc + fs - rotv_v, minus the imposed velocity on its
// slot, to gout, one thread per (element, mode) (elem_item): the first step of
// the penalty branch, whose product with the penalty function mixes the modes
// at each Gauss point (computing_rhs_gauss.F90:124-129).
SFX_DEV void rhs_ns_gauss_body(const RhsArgs& a, int64_t gid) {
  int64_t e;
  int m;
  elem_item(gid, a.M, e, m);
  if (e >= a.me || m >= a.M) return;
  int64_t j[6];
  double rn[6], zn[6];
#pragma unroll
  for (int n = 0; n < 6; ++n) {
    j[n] = (int64_t)a.jj[6 * e + n] - 1;
    SFX_CHECK("rr load", 2 * j[n] + 1, 2 * a.np);
    rn[n] = a.rr[2 * j[n]];
    zn[n] = a.rr[2 * j[n] + 1];
  }
  const double mv = (double)a.lmode[m];
  double V[6][6], F[6][6], Q[6][2];
#pragma unroll
  for (int n = 0; n < 6; ++n) {
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const int64_t i6 = j[n] + a.np * (k + 6 * (int64_t)m);
      SFX_CHECK("V1m load", i6, a.v1m ? a.n_v1m : 1 << 30);
      SFX_CHECK("ff load", i6, a.fsrc ? a.n_fsrc : 1 << 30);
      V[n][k] = a.v1m ? a.v1m[i6] : 0.0;
      F[n][k] = a.fsrc ? a.fsrc[i6] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int64_t i2 = j[n] + a.np * (k + 2 * (int64_t)m);
      SFX_CHECK("P_inc load", i2, a.pinc ? a.n_pinc : 1 << 30);
      Q[n][k] = a.pinc ? a.pinc[i2] : 0.0;
    }
  }
  const bool imposed = a.imp && m == a.imp_slot;
#pragma unroll
  for (int l = 0; l < 7; ++l) {
    const double* w = a.tab + 6 * l;
    const double* d = a.tab + 42 + 12 * l;
    // isoparametric Jacobian at this Gauss point: d/dr = a11 d/dx + a12 d/dy,
    // d/dz = a21 d/dx + a22 d/dy (exact for curved elements)
    double a11, a12, a21, a22;
    p2_inverse_jacobian(rn, zn, d, a11, a12, a21, a22);
    double ray = 0, ft[6] = {0, 0, 0, 0, 0, 0}, fs[6] = {0, 0, 0, 0, 0, 0};
    double qv[2] = {0, 0}, qx[2] = {0, 0}, qy[2] = {0, 0};
#pragma unroll
    for (int n = 0; n < 6; ++n) {
      ray = fma(rn[n], w[n], ray);
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        ft[k] = fma(V[n][k], w[n], ft[k]);
        fs[k] = fma(F[n][k], w[n], fs[k]);
      }
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        qv[k] = fma(Q[n][k], w[n], qv[k]);
        qx[k] = fma(Q[n][k], d[2 * n], qx[k]);
        qy[k] = fma(Q[n][k], d[2 * n + 1], qy[k]);
      }
    }
    double fq[6];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      fq[k] = -fma(a11, qx[k], a12 * qy[k]);
      fq[4 + k] = -fma(a21, qx[k], a22 * qy[k]);
    }
    fq[2] = -qv[1] / ray * mv;
    fq[3] = qv[0] / ray * mv;
    const int64_t gi = 7 * e + l + a.G * 6 * (int64_t)m;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      SFX_CHECK("rotv load", gi + a.G * k, a.rhs ? a.n_rhs : 1 << 30);
      const double rv = a.rhs ? a.rhs[gi + a.G * k] : 0.0;
      double base = ft[k] + fq[k] + fs[k] + a.rsign * rv;
      if (imposed) {
        double iv = 0;
#pragma unroll
        for (int n = 0; n < 6; ++n) {
          const int64_t jn = (int64_t)a.jj[6 * e + n] - 1;
          SFX_CHECK("imposed velocity load", jn + a.np * k, a.n_imp);
          iv = fma(a.imp[jn + a.np * k], w[n], iv);
        }
        base = base + a.isign * iv;
      }
      SFX_CHECK("gauss store", gi + a.G * k, a.n_gout);
      a.gout[gi + a.G * k] = base;
    }
  }
}

// vb_145 / vb_236 of work-group bid: the nodes' element contributions summed
// in element order (sfx_gather.h), components (1,4,5) and (2,3,6), times scale.
SFX_DEV void rhs_gather_block(const RhsArgs& a, int64_t bid, int tid, double* tile) {
  gather_body<6>(a.adj_ptr, a.adj_ent, a.n_adj, a.elo, a.n_elo, a.np, a.M, bid, tid, tile,
                 [&](int k, int m, int64_t n, double v) {
                   // component k -> (array, column): 1,4,5 -> vb_145; 2,3,6 -> vb_236
                   const bool v145 = (k == 0 || k == 3 || k == 4);
                   const int col = (k == 0 || k == 1) ? 0 : (k == 2 || k == 3) ? 1 : 2;
                   const int64_t o = n + a.np * (col + 3 * (int64_t)m);
                   SFX_CHECK("vb store", o, a.n_out);
                   (v145 ? a.v145 : a.v236)[o] = a.scale * v;
                 });
}

// Element share of qs_00_gauss, one thread per (element, column) (elem_item):
//   fl(l)       = (hc(e) SUM(ff_loc * ww(:,l)) + ff_gauss(7e+l)) * rj * ray
//   elo(6e+i,c) = sum_l ww(i,l) fl(l)                    (fem_rhs_axi.F90:958-975)
SFX_DEV void qs00_elem_body(const RhsArgs& a, int64_t gid) {
  int64_t e;
  int c;
  elem_item(gid, a.M, e, c);
  if (e >= a.me || c >= a.M) return;
  double ffl[6];
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const int64_t fi = (int64_t)a.jj[6 * e + j] - 1 + a.np * (int64_t)c;
    SFX_CHECK("ff load", fi, a.ff ? a.n_ff : 1 << 30);
    ffl[j] = a.ff ? a.ff[fi] : 0.0;
  }
  // a null heat capacity is 1; a null nodal or Gauss source is zero (the mass
  // matrix applied to ff, or the Galerkin right-hand side of ff_gauss alone)
  const double hc = a.heat_capa ? a.heat_capa[e] : 1.0;
  double fl[7];
#pragma unroll
  for (int l = 0; l < 7; ++l) {
    double s = 0;
#pragma unroll
    for (int j = 0; j < 6; ++j) s = fma(ffl[j], a.tab[j + 6 * l], s);
    const int64_t gi = 7 * e + l + a.G * (int64_t)c;
    SFX_CHECK("ffg load", gi, a.ffg ? a.n_ffg : 1 << 30);
    fl[l] = (hc * s + (a.ffg ? a.ffg[gi] : 0.0)) * a.wgt[7 * e + l];
  }
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    double loc = 0;
#pragma unroll
    for (int l = 0; l < 7; ++l) loc = fma(a.tab[i + 6 * l], fl[l], loc);
    const int64_t o = (6 * e + i) * a.M + c;
    SFX_CHECK("elo store", o, a.n_elo);
    a.elo[o] = loc;
  }
}

// vect(n, c) of work-group bid: the nodes' element contributions summed in
// element order (sfx_gather.h).
SFX_DEV void qs00_gather_block(const RhsArgs& a, int64_t bid, int tid, double* tile) {
  gather_body<1>(a.adj_ptr, a.adj_ent, a.n_adj, a.elo, a.n_elo, a.np, a.M, bid, tid, tile,
                 [&](int, int c, int64_t n, double v) {
                   SFX_CHECK("vect store", n + a.np * c, a.n_out);
                   a.vect[n + a.np * c] = a.scale * v;
                 });
}

// ---- boundary term of rhs_3x3 (opt_tensor_scaln_bdy, assembling_rhs.F90:129-185)
// For every boundary side ms (mesh%jjs: two ends, then the midpoint) and its
// three Gauss points, smb = T_bdy(3 ms + ls, :) * ray * rjs (points on the
// axis, ray < 1e-10, skipped), added to the side's nodes with the edge shape
// values wws and the (1,4,5)/(2,3,6) packing of the volume term.  Each
// boundary node is gathered by one thread from its (side, local node) list
// in side order, after the volume sums (the reference's VecSetValues order:
// elements first, then sides).
struct BdyArgs {
  const int64_t* bptr;      // (nb+1) offsets of each boundary node's entries
  const int32_t* bent;      // 3*ms + local node, side order
  const int64_t* bnode;     // (nb) node index (0-based)
  const double* bw;         // (3, mes): ray * rjs per side Gauss point, 0 where skipped
  double wws[9];            // wws(ns, ls) at 3*ls + ns
  int64_t nb, mes, np;
  int M;
  double scale;
  const double* tb;         // (3*mes, 6, M)
  double* v145;             // (np, 3, M)
  double* v236;             // (np, 3, M)
  int64_t n_tb, n_out, n_ent;
};

// One thread per (boundary node, mode), nodes fastest.
SFX_DEV void rhs_bdy_body(const BdyArgs& a, int64_t gid) {
  if (a.nb <= 0) return;
  const int64_t b = gid % a.nb, m = gid / a.nb;
  if (m >= a.M) return;
  const int64_t n = a.bnode[b];
  // component k -> (array, column): 1,4,5 -> vb_145 columns 1,2,3; 2,3,6 -> vb_236 columns 1,2,3
  int64_t o[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const int col = (k == 0 || k == 1) ? 0 : (k == 2 || k == 3) ? 1 : 2;
    o[k] = n + a.np * (col + 3 * m);
    SFX_CHECK("vb bdy", o[k], a.n_out);
  }
  double acc[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const bool v145 = (k == 0 || k == 3 || k == 4);
    acc[k] = (v145 ? a.v145 : a.v236)[o[k]];
  }
  for (int64_t t = a.bptr[b]; t < a.bptr[b + 1]; ++t) {
    SFX_CHECK("bdy entry", t, a.n_ent);
    const int32_t en = a.bent[t];
    const int64_t ms = en / 3;
    const int ns = en % 3;
    double side[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int ls = 0; ls < 3; ++ls) {
      const double wl = a.bw[3 * ms + ls];
      if (wl == 0.0) continue;                      // a point on the axis (ray < 1e-10)
      const double c = a.wws[3 * ls + ns] * wl;
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        const int64_t it = 3 * ms + ls + 3 * a.mes * (k + 6 * m);
        SFX_CHECK("T_bdy load", it, a.n_tb);
        side[k] = fma(c, a.tb[it], side[k]);
      }
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) acc[k] = fma(a.scale, side[k], acc[k]);
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const bool v145 = (k == 0 || k == 3 || k == 4);
    (v145 ? a.v145 : a.v236)[o[k]] = acc[k];
  }
}

}  // namespace sfx
