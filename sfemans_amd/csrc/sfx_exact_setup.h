// Host-side set-up of the exact-grid products, shared by the library and the
// CPU emulator: DFT tables and the field descriptors of each product.
#pragma once
#include <math.h>
#include <string.h>

#include <vector>

#include "sfx_exact_mm_body.h"

namespace sfx {

inline int exact_nj(int K) { return (K + 1 + EXACT_NJ_ALIGN - 1) / EXACT_NJ_ALIGN * EXACT_NJ_ALIGN; }
inline int exact_mr(int M) { return (M + EXACT_MC - 1) / EXACT_MC * EXACT_MC; }
inline size_t exact_ctab_size(int M, int K) { return (size_t)2 * M * exact_nj(K); }
inline size_t exact_rtab_size(int M, int K) { return (size_t)2 * (K + 1) * exact_mr(M); }

// ctab then rtab (layouts in ExactArgs), angles 2 pi (m j mod N)/N in long double.
inline void exact_host_tables(int M, int K, std::vector<double>& h) {
  const int N = 2 * K + 1, nj = exact_nj(K), MR = exact_mr(M);
  const size_t nc = exact_ctab_size(M, K);
  h.assign(nc + exact_rtab_size(M, K), 0.0);
  const long double two_pi = 6.283185307179586476925286766559005768L;
  for (int m = 0; m < M; ++m)
    for (int j = 0; j <= K; ++j) {
      const long double t = two_pi * (long double)(((int64_t)m * j) % N) / (long double)N;
      const long double c = cosl(t), s = sinl(t);
      h[(size_t)m * nj + j] = (double)c;
      h[(size_t)(M + m) * nj + j] = (double)s;
      h[nc + (size_t)j * MR + m] = (double)((m == 0 ? 1.0L : 2.0L) / (long double)N * c);
      h[nc + (size_t)(K + 1 + j) * MR + m] = m == 0 ? 0.0 : (double)(2.0L / (long double)N * s);
    }
}

// Whether the matrix-core kernel takes these sizes: accumulators for at most
// two halves of 64 modes, and tables that stay in every L2.
inline bool exact_mm_sizes(int M, int K) { return M >= 1 && M <= EXACT_MM_MAX_M && K + 1 <= EXACT_MM_MAX_PAD; }

// Its tables (ExactMmArgs: ct then rt), from the ones of exact_host_tables.
inline void exact_mm_host_tables(int M, int K, const double* h, std::vector<double>& t) {
  const int nj = exact_nj(K), MR = exact_mr(M), MBN = exact_mm_mbn(M), JBN = exact_mm_jbn(K);
  const double* r = h + exact_ctab_size(M, K);
  const size_t nc = exact_mm_ctab_size(M, K);
  t.assign(nc + exact_mm_rtab_size(M, K), 0.0);
  for (int kb = 0; kb < 4 * MBN; ++kb)
    for (int jb = 0; jb < JBN; ++jb)
      for (int l = 0; l < 64; ++l) {
        const int j = 16 * jb + l % 16, m = 4 * kb + l / 16;
        if (j > K || m >= M) continue;
        double* d = &t[((size_t)(kb * JBN + jb) * 64 + l) * 2];
        d[0] = h[(size_t)m * nj + j];
        d[1] = h[(size_t)(M + m) * nj + j];
      }
  for (int q = 0; q < 4 * JBN; ++q)
    for (int mb = 0; mb < MBN; ++mb)
      for (int l = 0; l < 64; ++l) {
        const int m = 16 * mb + l % 16, j = 4 * q + l / 16;
        if (j > K || m >= M) continue;
        double* d = &t[nc + ((size_t)(q * MBN + mb) * 64 + l) * 2];
        d[0] = r[(size_t)j * MR + m];
        d[1] = r[(size_t)(K + 1 + j) * MR + m];
      }
}

// The matrix-core kernel reads an input while other work-groups have already
// stored outputs, so it does not take calls whose outputs overlap inputs (the
// two-pass kernels read everything before the first store).
inline bool exact_mm_disjoint(const ExactArgs& a) {
  for (int g = 0; g < a.nout; ++g) {
    const ExactOut& o = a.out[g];
    const double *o0 = o.base, *o1 = o.base + (a.np - 1) * o.sp + (a.M - 1) * o.sm + o.off + 1;
    for (int f = 0; f < a.nin; ++f) {
      const ExactField& i = a.in[f];
      if (!i.base) continue;
      if (o0 < i.base + (a.np - 1) * i.sp + (a.M - 1) * i.sm + i.off + 1 && i.base < o1) return false;
    }
    if (a.creal && o0 < a.creal + a.n_creal && a.creal < o1) return false;
  }
  return true;
}

// Products that stay on the two-pass kernels though the matrix-core kernel has
// their sizes: with M modes in whole blocks of 16 and m_max_pad angles in
// blocks of 16, the share of useful products, f = M m_max_pad / (256 blocks),
// is small for a few modes and for a mode count a little above a multiple of
// 16, and the operation runs on every padded angle (and, for the tension and
// the entropy viscosities, again for each output).  Below some number of
// points the two-pass kernels are two launches that leave the chip idle, and
// the matrix-core kernel is faster all the same; with a scratch array larger
// than the last-level cache (256 MB, which S, D and the inputs share) they
// fall behind again.  A product takes the two-pass kernels if one of its
// lines holds: more than points + slope f points, f below the line's, at most
// `scratch` MB of S and D, at least `modes` modes.  Times, two-pass /
// matrix-core kernel in us, on both sides of the lines:
//   tension   M = 2: 12 / 12 on 8,190 points, 55 / 289 on 262,136; M = 8: 33 / 23 on 16,380, 55 / 59 on 49,140;
//             M = 12: 43 / 38 on 16,380, 58 / 69 on 32,767, 297 / 266 on 131,068; M = 14: 348 / 280 on 131,068
//   compressive entropy viscosity   M = 2: 14 / 11 on 8,190, 14 / 46 on 65,534; M = 10: 130 / 110 on 131,068;
//             M = 12: 34 / 28 on 16,380, 168 / 203 on 131,068; M = 24: 91 / 108 on 32,767, 442 / 450 on 131,068
//   entropy viscosity   M = 6: 38 / 25 on 8,190, 82 / 99 on 65,534, 372 / 421 on 262,136; M = 8: 115 / 102 on 65,534
//   level-set compression   M = 17: 39 / 28 on 12,285, 136 / 174 on 131,068; M = 38: 183 / 159 on 49,140
//   Heaviside of 2 interfaces   M = 12: 45 / 38 on 131,068; M = 24: 45 / 28 on 32,767, 77 / 91 on 131,068;
//             of 4   M = 10: 30 / 21 on 49,140, 58 / 68 on 196,602
//   the others, only for a few modes   v / s M = 2: 12 / 10 on 32,767, 24 / 69 on 262,136, M = 6: 73 / 70 there;
//             gradients M = 4: 18 / 14 on 16,380, 38 / 44 on 65,534; division M = 2: 11 / 10 on 65,534, 12 / 28 on
//             262,136
struct ExactMmLine {
  int op, nin;                       // nin: 0 for any
  int modes;
  double points, slope, f, scratch;  // points and slope in units of 1024
};
constexpr double EXACT_MM_ANY = 1e30;
constexpr ExactMmLine EXACT_MM_LINES[] = {
    {EX_TENSION, 0, 1, 8, 64, 0.28, EXACT_MM_ANY},
    {EX_TENSION, 0, 1, 24, 0, 0.50, 145},
    {EX_TENSION, 0, 17, 20, 0, 0.57, 125},
    {EX_COMPR, 0, 1, 16, 0, 0.40, EXACT_MM_ANY},
    {EX_COMPR, 0, 12, 16, 0, 0.52, EXACT_MM_ANY},
    {EX_COMPR, 0, 12, 24, 0, 0.58, 80},
    {EX_COMPR, 0, 17, 22, 0, 0.61, 80},
    {EX_EVISC, 0, 1, 8, 128, 0.22, EXACT_MM_ANY},
    {EX_EVISC, 0, 1, 8, 128, 0.65, 100},
    {EX_CLS, 0, 1, 34, 120, 0.40, EXACT_MM_ANY},
    {EX_CLS, 0, 9, 56, 0, 0.58, EXACT_MM_ANY},
    {EX_CLS, 0, 17, 40, 0, 0.69, EXACT_MM_ANY},
    {EX_HEAVI, 1, 1, 96, 0, 0.10, EXACT_MM_ANY},
    {EX_HEAVI, 2, 1, 96, 0, 0.22, EXACT_MM_ANY},
    {EX_HEAVI, 2, 17, 63, 0, 0.65, EXACT_MM_ANY},
    {EX_HEAVI, 3, 1, 48, 0, 0.12, EXACT_MM_ANY},
    {EX_HEAVI, 3, 1, 100, 0, 0.25, EXACT_MM_ANY},
    {EX_HEAVI, 3, 1, 160, 0, 0.50, EXACT_MM_ANY},
    {EX_HEAVI, 3, 12, 48, 0, 0.65, EXACT_MM_ANY},
    {EX_HEAVI, 3, 17, 31, 0, 0.80, EXACT_MM_ANY},
    {EX_HEAVI, 4, 1, 40, 0, 0.12, EXACT_MM_ANY},
    {EX_HEAVI, 4, 1, 66, 0, 0.60, EXACT_MM_ANY},
    {EX_HEAVI, 4, 12, 48, 0, 0.65, EXACT_MM_ANY},
    {EX_HEAVI, 4, 17, 31, 0, 0.78, EXACT_MM_ANY},
    {EX_GRADMOM, 0, 1, 16, 96, 0.10, EXACT_MM_ANY},
    {EX_ENTRO, 0, 1, 32, 256, 0.14, EXACT_MM_ANY},
    {EX_ETA3, 0, 1, 48, 256, 0.10, EXACT_MM_ANY},
    {EX_SV2, 0, 1, 40, 128, 0.14, EXACT_MM_ANY},
    {EX_SVCLAMP, 0, 1, 40, 128, 0.14, EXACT_MM_ANY},
    {EX_DIV, 0, 1, 64, 512, 0.22, EXACT_MM_ANY},
    {EX_DIV, 0, 17, 96, 0, 0.54, 80},
    {EX_ETA, 0, 1, 96, 0, 0.05, EXACT_MM_ANY},
    {EX_SQRT, 0, 1, 96, 0, 0.05, EXACT_MM_ANY},
    {EX_CLAMP01, 0, 1, 96, 0, 0.05, EXACT_MM_ANY},
    {EX_FROMREAL, 0, 1, 300, 0, 0.03, EXACT_MM_ANY}};

inline bool exact_mm_two_pass(int op, const ExactArgs& a) {
  const double f = a.M * (double)(a.K + 1) / (256.0 * exact_mm_mbn(a.M) * exact_mm_jbn(a.K));
  const double mb = 16.0 * a.nout * (a.K + 1) * (double)a.np / (1 << 20);
  for (const ExactMmLine& l : EXACT_MM_LINES)
    if (l.op == op && (l.nin == 0 || l.nin == a.nin) && a.M >= l.modes && f < l.f && mb <= l.scratch &&
        (double)a.np > 1024.0 * (l.points + l.slope * f))
      return true;
  return false;
}

// Whether a product runs on the matrix-core kernel (EX_EVISC: its two parts).
// Its exact form (M <= 64 on a grid of 3/2 as many angle pairs) beside the
// lines above.  The general form (more modes, other grids) repeats the
// synthesis for the second half of the modes and is taken up to the number of
// points where every product still gains (M = 80, v / s 76 / 30 us, tension
// 130 / 86 on 2,044 points, but tension 137 / 164 on 4,088; v / s gains up to
// some 32,000).  The analysis alone (EX_FROMREAL) has no synthesis: 238 / 87 on
// 60,000 points at M = 80.
inline bool exact_mm_use(int op, const ExactArgs& a) {
  // EX_EVISC's products are those of EX_GRADMOM on its last nine inputs
  if (!exact_mm_has(op == EX_EVISC ? EX_GRADMOM : op) || a.np <= 0 || !exact_mm_sizes(a.M, a.K) ||
      !exact_mm_disjoint(a))
    return false;
  if (op == EX_FROMREAL) return !exact_mm_two_pass(op, a);
  const int jb = exact_mm_jb(exact_mm_mb(a.M)), jbn = exact_mm_jbn(a.K);
  if (a.M > 64 || (jbn != jb && jbn != jb - 1)) return a.np <= 2048;
  return !exact_mm_two_pass(op, a);
}

inline void exact_setup_sizes(ExactArgs& a, int64_t np, int M, int m_max_pad) {
  a.np = np; a.M = M; a.K = m_max_pad - 1;
  a.nj = exact_nj(a.K);
  a.MR = exact_mr(M);
}

inline ExactField exact_field(const double* base, int64_t sp, int64_t sm, int64_t off) {
  ExactField f;
  f.base = base; f.sp = sp; f.sm = sm; f.off = off;
  return f;
}
inline ExactOut exact_outf(double* base, int64_t sp, int64_t sm, int64_t off) {
  ExactOut f;
  f.base = base; f.sp = sp; f.sm = sm; f.off = off;
  return f;
}

// Field k of an (np, nb, M) array: cos column 2k, sin column 2k+1.
inline ExactField exact_col(const double* V, int64_t np, int nb, int k) {
  return exact_field(V + 2 * k * np, 1, (int64_t)nb * np, np);
}
inline ExactOut exact_colo(double* V, int64_t np, int nb, int k) {
  return exact_outf(V + 2 * k * np, 1, (int64_t)nb * np, np);
}

// FFT_PAR_DIV_DCL: c1, c2, c (np, 2, M).
inline void exact_setup_div(ExactArgs& a, const double* c1, const double* c2, double* c, int64_t np, int M) {
  memset(&a, 0, sizeof(a));
  a.nin = 2; a.nout = 1;
  a.in[0] = exact_col(c1, np, 2, 0);
  a.in[1] = exact_col(c2, np, 2, 0);
  a.out[0] = exact_colo(c, np, 2, 0);
  a.n_in[0] = a.n_in[1] = a.n_out[0] = np * 2 * (int64_t)M;
}

// FFT_SCALAR_VECT_DCL pb = 2: V (np, 6, M) / s (np, 2, M) -> out (np, 6, M).
inline void exact_setup_sv2(ExactArgs& a, const double* V, const double* s, double* out, int64_t np, int M) {
  memset(&a, 0, sizeof(a));
  a.nin = 4; a.nout = 3;
  for (int k = 0; k < 3; ++k) {
    a.in[k] = exact_col(V, np, 6, k);
    a.out[k] = exact_colo(out, np, 6, k);
    a.n_in[k] = a.n_out[k] = np * 6 * (int64_t)M - 2 * k * np;
  }
  a.in[3] = exact_col(s, np, 2, 0);
  a.n_in[3] = np * 2 * (int64_t)M;
}

// FFT_SCALAR_VECT_NO_OVERSHOOT: as pb = 1 / 2 with the scalar clamped to [smin, smax].
inline void exact_setup_svclamp(ExactArgs& a, const double* V, const double* s, double* out, int64_t np, int M,
                                int pb, double smin, double smax) {
  exact_setup_sv2(a, V, s, out, np, M);
  a.pb = pb; a.smin = smin; a.smax = smax;
}

// FFT_PAR_ENTRO_VISC_DCL: V (np, 6, M), c (np, 2, M), c_in_real (N, np) ->
// V_out (np, 6, M) = (coeff - c_in_real) V, c_out (np, 2, M) = MAX(0, c (1 - c)).
inline void exact_setup_entro(ExactArgs& a, const double* V, const double* c, const double* creal, double coeff,
                              double* Vout, double* cout, int64_t np, int M, int m_max_pad) {
  memset(&a, 0, sizeof(a));
  a.nin = 4; a.nout = 4;
  for (int k = 0; k < 3; ++k) {
    a.in[k] = exact_col(V, np, 6, k);
    a.out[k] = exact_colo(Vout, np, 6, k);
    a.n_in[k] = a.n_out[k] = np * 6 * (int64_t)M - 2 * k * np;
  }
  a.in[3] = exact_col(c, np, 2, 0);
  a.out[3] = exact_colo(cout, np, 2, 0);
  a.n_in[3] = a.n_out[3] = np * 2 * (int64_t)M;
  a.creal = creal;
  a.n_creal = (2 * (int64_t)m_max_pad - 1) * np;
  a.coeff = coeff;
}

// FFT_PAR_COMPR_ENTRO_VISC_DCL: grad(phi) V1, grad(phi_reg) V2 (np, 6, M), phi c (np, 2, M),
// c_in_real (N, np) -> V_out (np, 6, M), c_out (np, 2, M).
inline void exact_setup_compr(ExactArgs& a, const double* V1, const double* V2, const double* c, const double* creal,
                              double coeff, double comp, double* Vout, double* cout, int64_t np, int M,
                              int m_max_pad) {
  exact_setup_entro(a, V1, c, creal, coeff, Vout, cout, np, M, m_max_pad);
  a.nin = 7;
  a.in[6] = a.in[3];
  a.n_in[6] = a.n_in[3];
  for (int k = 0; k < 3; ++k) {
    a.in[3 + k] = exact_col(V2, np, 6, k);
    a.n_in[3 + k] = np * 6 * (int64_t)M - 2 * k * np;
  }
  a.coeff2 = comp;
}

// FFT_COMPUTE_ENTROPY_VISC_GRAD_MOM: V1, V2, V3 (np, 6, M), c_in_real (N, np) ->
// out (3, np, 6, M), out(a, :, 2f:2f+1, :) = coefficients of (c_in_real - coeff) V_a,f.
inline void exact_setup_gradmom(ExactArgs& a, const double* V1, const double* V2, const double* V3,
                                const double* creal, double coeff, double* out, int64_t np, int M, int m_max_pad) {
  memset(&a, 0, sizeof(a));
  a.nin = 9; a.nout = 9;
  const double* V[3] = {V1, V2, V3};
  for (int r = 0; r < 3; ++r)
    for (int f = 0; f < 3; ++f) {
      a.in[3 * r + f] = exact_col(V[r], np, 6, f);
      a.n_in[3 * r + f] = np * 6 * (int64_t)M - 2 * f * np;
      a.out[3 * r + f] = exact_outf(out + r + 3 * np * 2 * f, 3, 3 * np * 6, 3 * np);
      a.n_out[3 * r + f] = 3 * np * 6 * (int64_t)M - r - 3 * np * 2 * f;
    }
  a.creal = creal;
  a.n_creal = (2 * (int64_t)m_max_pad - 1) * np;
  a.coeff = coeff;
}

// FFT_COMPUTE_ENTROPY_VISC: velocity V1, residual V2, tensor rows V3, V4, V5
// (np, 6, M), hloc (np), lg points per element -> O1, O2, O3 (np, 6, M).  The
// per-element maxima array (me * N doubles) is set by the caller in a.nint.
inline void exact_setup_evisc(ExactArgs& a, const double* const (&V)[5], const double* hloc, double* const (&O)[3],
                              int64_t np, int M, int lg, double c1, double c2, double c4, double res) {
  memset(&a, 0, sizeof(a));
  a.nin = 15; a.nout = 9;
  for (int v = 0; v < 5; ++v)
    for (int k = 0; k < 3; ++k) {
      a.in[3 * v + k] = exact_col(V[v], np, 6, k);
      a.n_in[3 * v + k] = np * 6 * (int64_t)M - 2 * k * np;
    }
  for (int r = 0; r < 3; ++r)
    for (int k = 0; k < 3; ++k) {
      a.out[3 * r + k] = exact_colo(O[r], np, 6, k);
      a.n_out[3 * r + k] = np * 6 * (int64_t)M - 2 * k * np;
    }
  a.hloc = hloc;
  a.lg = lg;
  a.coeff = c1; a.coeff2 = c2; a.coeff3 = c4; a.coeff4 = res;
}

// FFT_COMPUTE_ENTROPY_VISC in two passes from its full argument set `a`: `v`
// writes the viscosity on the grid into vreal (N, np) from the velocity and
// residual; `w` multiplies the three tensor rows by it (EX_GRADMOM with no
// offset) and carries the r2c outputs.
inline void exact_evisc_split(const ExactArgs& a, double* vreal, ExactArgs& v, ExactArgs& w) {
  v = a;
  v.nin = 6; v.nout = 0;
  v.rout1 = vreal;
  v.n_nint2 = (2 * (int64_t)a.K + 1) * a.np;
  w = a;
  w.nin = 9; w.nout = 9;
  for (int f = 0; f < 9; ++f) {
    w.in[f] = a.in[6 + f];
    w.n_in[f] = a.n_in[6 + f];
  }
  w.creal = vreal;
  w.n_creal = v.n_nint2;
  w.coeff = 0.0;
}

// FFT_COMPUTE_ENTROPY_VISC_MOM: u V1, momentum V2, residual V3 (np, 6, M), mass
// residual c (np, 2, M), hloc (np); real-space outputs (N, np).  The caller sets
// the per-element arrays, pmax and the sizes.
inline void exact_setup_emom(ExactArgs& a, const double* V1, const double* V2, const double* V3, const double* c,
                             const double* hloc, double* out1, double* out2, int64_t np, int M, int lg, double c2,
                             double c4) {
  memset(&a, 0, sizeof(a));
  a.nin = 10; a.nout = 0;
  const double* V[3] = {V1, V2, V3};
  for (int v = 0; v < 3; ++v)
    for (int k = 0; k < 3; ++k) {
      a.in[3 * v + k] = exact_col(V[v], np, 6, k);
      a.n_in[3 * v + k] = np * 6 * (int64_t)M - 2 * k * np;
    }
  a.in[9] = exact_col(c, np, 2, 0);
  a.n_in[9] = np * 2 * (int64_t)M;
  a.hloc = hloc;
  a.rout1 = out1; a.rout2 = out2;
  a.lg = lg;
  a.coeff2 = c2; a.coeff3 = c4;
}

// FFT_COMPRESSION_LEVEL_SET_DCL, product pass: grad(phi) V1 (np, 6, M), phi c
// (np, 2, M) -> c_out (np, 2, M); dmax (device) the maximum of |velocity|.
inline void exact_setup_cls(ExactArgs& a, const double* V1, const double* c, double* cout, const double* dmax,
                            int64_t np, int M, double comp, double les_coeff4, double h_min_distance) {
  memset(&a, 0, sizeof(a));
  a.nin = 4; a.nout = 1;
  for (int k = 0; k < 3; ++k) {
    a.in[k] = exact_col(V1, np, 6, k);
    a.n_in[k] = np * 6 * (int64_t)M - 2 * k * np;
  }
  a.in[3] = exact_col(c, np, 2, 0);
  a.n_in[3] = np * 2 * (int64_t)M;
  a.out[0] = exact_colo(cout, np, 2, 0);
  a.n_out[0] = np * 2 * (int64_t)M;
  a.dmax = dmax;
  a.coeff = comp * 4.0 * les_coeff4;
  a.coeff2 = h_min_distance;
}

// FFT_PAR_REAL, field f of V (np, nb, M) -> its values on the N = 2K+1 grid
// angles, out(N, nb/2, np) column-major: out[j + N*(f + nb/2*p)].
inline void exact_setup_real(ExactArgs& a, const double* V, int f, int nb, double* out, int64_t np, int M, int N) {
  memset(&a, 0, sizeof(a));
  a.nin = 1; a.nout = 0;
  a.in[0] = exact_col(V, np, nb, f);
  a.n_in[0] = np * nb * (int64_t)M - 2 * (int64_t)f * np;
  a.rout1 = out + (int64_t)N * f;
  a.rstride = (int64_t)N * (nb / 2);
  a.n_nint2 = a.rstride * np - (int64_t)N * f;
}

// FFT_SQUAREROOT_SCALAR and FFT_NO_OVERSHOOT_LEVEL_SET: first scalar of c (np, nb, M)
// -> first scalar of out (np, nb, M).
inline void exact_setup_sqrt(ExactArgs& a, const double* c, double* out, int64_t np, int nb, int M) {
  memset(&a, 0, sizeof(a));
  a.nin = 1; a.nout = 1;
  a.in[0] = exact_col(c, np, nb, 0);
  a.out[0] = exact_colo(out, np, nb, 0);
  a.n_in[0] = a.n_out[0] = np * nb * (int64_t)M;
}

// FFT_HEAVISIDE_DCL: V1 (n_int, np, 2, M), values (n_int + 1) -> out (np, 2, M).
inline void exact_setup_heavi(ExactArgs& a, const double* V1, const double* values, int n_values, double* out,
                              int64_t np, int M, double eps) {
  memset(&a, 0, sizeof(a));
  const int n_int = n_values - 1;
  a.nin = n_int; a.nout = 1; a.n_int = n_int; a.eps = eps;
  for (int i = 0; i < n_values; ++i) a.vals[i] = values[i];
  for (int i = 0; i < n_int; ++i) {
    a.in[i] = exact_field(V1 + i, n_int, (int64_t)n_int * np * 2, (int64_t)n_int * np);
    a.n_in[i] = (int64_t)n_int * np * 2 * M - i;
  }
  a.out[0] = exact_colo(out, np, 2, 0);
  a.n_out[0] = np * 2 * (int64_t)M;
}

// FFT_TENSOR_DCL with opt_tension: V1, V2 (np, 6, M) -> out (3, np, 6, M), out(r, :, 2c:2c+1, :).
inline void exact_setup_tension(ExactArgs& a, const double* V1, const double* V2, double* out, int64_t np,
                                int M) {
  memset(&a, 0, sizeof(a));
  a.nin = 6; a.nout = 9;
  for (int k = 0; k < 3; ++k) {
    a.in[k] = exact_col(V1, np, 6, k);
    a.in[3 + k] = exact_col(V2, np, 6, k);
    a.n_in[k] = a.n_in[3 + k] = np * 6 * (int64_t)M - 2 * k * np;
  }
  for (int r = 0; r < 3; ++r)
    for (int c = 0; c < 3; ++c) {
      a.out[3 * r + c] = exact_outf(out + r + 3 * np * 2 * c, 3, 3 * np * 6, 3 * np);
      a.n_out[3 * r + c] = 3 * np * 6 * (int64_t)M - r - 3 * np * 2 * c;
    }
}

// FFT_MAX_VEL_DCL: V1 (np, nb, M), nb = 6 (|v|) or 2 (|c|).
inline void exact_setup_maxvel(ExactArgs& a, const double* V1, int64_t np, int nb, int M) {
  memset(&a, 0, sizeof(a));
  a.nin = nb == 6 ? 3 : 1; a.nout = 0;
  for (int k = 0; k < a.nin; ++k) {
    a.in[k] = exact_col(V1, np, nb, k);
    a.n_in[k] = np * nb * (int64_t)M - 2 * k * np;
  }
}

// FFT_PAR_VAR_ETA_PROD_T_DCL / _GAUSS_DCL: eta (N, np) on the grid angles,
// c (np, nb, M), nb = 2 or 6 -> out (np, nb, M), the coefficients of eta * c.
inline void exact_setup_eta(ExactArgs& a, const double* eta, const double* c, double* out, int64_t np, int nb,
                            int M, int m_max_pad) {
  memset(&a, 0, sizeof(a));
  a.nin = a.nout = nb / 2;
  for (int k = 0; k < a.nin; ++k) {
    a.in[k] = exact_col(c, np, nb, k);
    a.out[k] = exact_colo(out, np, nb, k);
    a.n_in[k] = a.n_out[k] = np * nb * (int64_t)M - 2 * k * np;
  }
  a.creal = eta;
  a.n_creal = (2 * (int64_t)m_max_pad - 1) * np;
}

// Analysis of values on the grid: real (N, np) -> c (np, 2, M), the
// truncated, scaled real DFT the products end with.
inline void exact_setup_fromreal(ExactArgs& a, const double* real, double* c, int64_t np, int M, int m_max_pad) {
  memset(&a, 0, sizeof(a));
  a.nin = 1; a.nout = 1;
  a.out[0] = exact_colo(c, np, 2, 0);
  a.n_out[0] = np * 2 * (int64_t)M;
  a.creal = real;
  a.n_creal = (2 * (int64_t)m_max_pad - 1) * np;
}

// FFT_CHECK_INTERFACE: V1 (n_int, np, 2, M) level sets, as for the Heaviside.
inline void exact_setup_checkif(ExactArgs& a, const double* V1, int n_int, int64_t np, int M) {
  memset(&a, 0, sizeof(a));
  a.nin = n_int; a.nout = 0; a.n_int = n_int;
  for (int i = 0; i < n_int; ++i) {
    a.in[i] = exact_field(V1 + i, n_int, (int64_t)n_int * np * 2, (int64_t)n_int * np);
    a.n_in[i] = (int64_t)n_int * np * 2 * M - i;
  }
}

}  // namespace sfx
