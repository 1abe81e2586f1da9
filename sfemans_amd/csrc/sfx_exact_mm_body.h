// Exact-grid products on the matrix cores: synthesis, pointwise operation and
// analysis in one kernel (compiled for gfx950 and for the CPU emulator).
//
// The sums of sfx_exact_body.h are matrix products with the angle pairs (j,
// N - j) folded: E = C a, O = S b (angles x modes times modes x points) and
// A = R S', B = R' D (modes x angles times angles x points).  Both run as
// v_mfma_f64_16x16x4.  A work-group owns 16 points (the columns).  In the
// synthesis wave f forms field f at JB blocks of 16 angles; in the analysis
// wave g forms output g, 16 MB modes of it, from 4 angles at a time.  The
// result layout of the f64 MFMA (lane l, element v: row l / 16 + 4 v, column
// l % 16) is the layout of its 4 x 16 operand for the four rows of element v,
// so a value needs no transposition on the way from one product to the other:
// field f's values pass through 4 KB of LDS per angle block to the waves that
// need them, and every input is read once per JB blocks.
//
// What bounds it: on gfx950 the f64 MFMA (64 cycles) and the other vector
// instructions of a SIMD do not overlap, whichever waves they come from (4
// MFMA and 64 integer operations take the sum of their times), so a kernel's
// time is MFMA time plus vector time plus what no wave covers.  The factors
// are therefore loaded in operand order at constant offsets (L1 and L2 hold
// them; stepping residues m j mod N through a table in LDS costs 7 vector
// operations per pair of MFMA, 1.70 against 1.52 ms), and the masks of the
// first and last angles and modes are applied in their own steps only.
// Measured: v / s (7 transforms) at 402,753 points, M = 64: 2.85 ms with an
// angle pass, a scratch array and an analysis pass, 1.52 ms here (45 TF; the
// MFMA alone 0.96 ms, other vector instructions 0.2 ms); entropy viscosity at
// 351,232 points, M = 32: 3.72 -> 2.30 ms.
#pragma once
#include "sfx_exact_body.h"

namespace sfx {

// Operations of the fused kernel.  The first ones are ExactOp values; the
// others are parts of products whose outputs do not depend on all inputs.
// MM_SCALE3: three fields times (creal - coeff), a third of EX_GRADMOM;
// MM_TENSROW: row r of the tension tensor, inputs u_r, v_0..v_2.
enum ExactMmOp { MM_SCALE3 = 64, MM_TENSROW };

constexpr int exact_mm_nin(int op, int nin) {
  return op == MM_SCALE3 ? 3 : op == MM_TENSROW ? 4 : op == EX_FROMREAL ? 0 : nin;
}
constexpr int exact_mm_nout(int op) { return op == MM_SCALE3 || op == MM_TENSROW ? 3 : exact_nout(op); }
// Groups of outputs, one row of the grid each (its own inputs and outputs).
constexpr int exact_mm_groups(int op) { return op == MM_SCALE3 || op == MM_TENSROW ? 3 : 1; }
// Waves of a work-group: one per field and per output.
constexpr int exact_mm_waves(int ni, int no) { return ni > no ? ni : no > 0 ? no : 1; }

// Sizes: M modes in MBN blocks of 16 (4 steps each), K + 1 angles in JBN blocks of 16.
constexpr int EXACT_MM_MAX_M = 128, EXACT_MM_MAX_PAD = 512;
inline int exact_mm_mbn(int M) { return (M + 15) / 16; }
inline int exact_mm_jbn(int K) { return (K + 16) / 16; }
inline size_t exact_mm_ctab_size(int M, int K) { return (size_t)exact_mm_jbn(K) * exact_mm_mbn(M) * 4 * 128; }
inline size_t exact_mm_rtab_size(int M, int K) { return (size_t)exact_mm_jbn(K) * 4 * exact_mm_mbn(M) * 128; }
// Mode blocks per work-group: all of them up to 64 modes, else half (their
// accumulators and those of the angles have to fit in 256 registers).
inline int exact_mm_mb(int M) { const int n = exact_mm_mbn(M); return n <= 4 ? n : (n + 1) / 2; }
// Angle blocks per pass of the general form: those of 3/2 as many angles as
// 16 MB modes.
constexpr int exact_mm_jb(int mb) { return mb == 1 ? 2 : mb == 2 ? 3 : mb == 3 ? 5 : 6; }

// Whether launch_exact_mm takes the operation.
constexpr bool exact_mm_has(int op) {
  return op == EX_DIV || op == EX_SV2 || op == EX_SVCLAMP || op == EX_SQRT || op == EX_CLAMP01 || op == EX_HEAVI ||
         op == EX_TENSION || op == EX_ENTRO || op == EX_GRADMOM || op == EX_COMPR || op == EX_CLS || op == EX_ETA ||
         op == EX_ETA3 || op == EX_FROMREAL || op == EX_EVISCV;
}

struct ExactMmArgs {
  ExactArgs a;
  const double* ct;   // cos, sin of angle 16 jb + l % 16 and mode 4 kb + l / 16 at [((kb*JBN + jb)*64 + l)*2],
                      // kb < 4 MBN, zero past M and K
  const double* rt;   // r2c factors of mode 16 mb + l % 16 and angle 4 q + l / 16 at [((q*MBN + mb)*64 + l)*2]
  int64_t n_ct, n_rt;
  int mbn, jbn;
};

// Output g of the operation at one angle: U(f) is field f there, x and y the
// real-space inputs (exact_op).
template <int OP, int NI, typename Field>
SFX_DEV double exact_mm_op(const ExactArgs& a, int grp, int g, Field U, double x, double y) {
  if constexpr (OP == MM_SCALE3 || OP == EX_GRADMOM) {
    return (x - a.coeff) * U(g);
  } else if constexpr (OP == EX_ETA || OP == EX_ETA3) {
    return x * U(g);
  } else if constexpr (OP == EX_FROMREAL) {
    return x;
  } else if constexpr (OP == EX_SV2) {
    return U(g) / U(3);
  } else if constexpr (OP == EX_SVCLAMP) {
    const double sc = fmax(a.smin, fmin(U(3), a.smax));
    return a.pb == 1 ? sc * U(g) : U(g) / sc;
  } else if constexpr (OP == EX_ENTRO) {
    const double u = U(g);
    return g == 3 ? fmax(0.0, u * (1.0 - u)) : (a.coeff - x) * u;
  } else if constexpr (OP == EX_COMPR) {
    const double u6 = U(6), c2 = fmax(0.0, u6 * (1.0 - u6));
    if (g == 3) return c2;
    const double v0 = U(3), v1 = U(4), v2 = U(5);
    const double ng = sqrt(v0 * v0 + v1 * v1 + v2 * v2) + 1.e-14;
    const double ve = -a.coeff + x, vc = x * a.coeff2 * c2 / ng;
    return -ve * U(g) + vc * U(3 + g);
  } else if constexpr (OP == MM_TENSROW) {
    const double v0 = U(1), v1 = U(2), v2 = U(3);
    const double nrm = sqrt(v0 * v0 + v1 * v1 + v2 * v2);
    return U(0) * (g == 0 ? v0 : g == 1 ? v1 : v2) / (nrm + 1.e-14) - (g == grp ? nrm : 0.0);
  } else {
    double u[NI], w[1];
#pragma unroll
    for (int f = 0; f < NI; ++f) u[f] = U(f);
    exact_op<OP, NI, (OP == EX_EVISCV ? 0 : 1)>(a, u, w, x, y);
    return w[0];
  }
}

// Whether OP reads real-space values at each angle.
constexpr bool exact_mm_creal(int op) {
  return op == MM_SCALE3 || op == EX_ENTRO || op == EX_COMPR || op == EX_ETA || op == EX_ETA3 || op == EX_FROMREAL;
}

// Argument field of input f (of output g) of group grp, through selects:
// indexing the argument array with a run-time value would copy it to scratch.
template <int OP, int NI>
SFX_DEV ExactField exact_mm_in(const ExactArgs& a, int f, int grp, int64_t& n) {
  const int k = OP == MM_SCALE3 ? 3 * grp + f : OP == MM_TENSROW ? (f == 0 ? grp : 2 + f) : f;
  ExactField r = a.in[0];
  n = a.n_in[0];
#pragma unroll
  for (int i = 1; i < (OP == MM_SCALE3 ? 9 : OP == MM_TENSROW ? 6 : NI); ++i) {
    r.base = k == i ? a.in[i].base : r.base;
    r.sm = k == i ? a.in[i].sm : r.sm;      // the point stride and the offset are the same for all
    n = k == i ? a.n_in[i] : n;
  }
  return r;
}
template <int OP, int NO>
SFX_DEV ExactOut exact_mm_out(const ExactArgs& a, int g, int grp, int64_t& n) {
  const int k = exact_mm_groups(OP) > 1 ? 3 * grp + g : g;
  ExactOut r = a.out[0];
  n = a.n_out[0];
#pragma unroll
  for (int i = 1; i < (exact_mm_groups(OP) > 1 ? 9 : NO); ++i) {
    r.base = k == i ? a.out[i].base : r.base;
    r.sm = k == i ? a.out[i].sm : r.sm;
    n = k == i ? a.n_out[i] : n;
  }
  return r;
}

// LDS doubles: two buffers of every field's values at 16 angle pairs.
constexpr int exact_mm_smem(int ni) { return 2 * ni * 512; }

// 16 points, mode blocks mb0 .. mb0 + MB - 1 of the outputs of group grp, in
// passes over JB angle blocks.  ONE: MB and JB are all the blocks there are.
template <int OP, int NIN, int MB, int JB, bool ONE>
SFX_DEV void exact_mm_body(const ExactMmArgs& A, int tid, int64_t bid, int grp, int mpart, double* smem) {
  constexpr int NI = exact_mm_nin(OP, NIN), NO = exact_mm_nout(OP), NW = exact_mm_waves(NI, NO);
  // real-space inputs per lane and angle block: 4 angles in the analysis, one without
  constexpr int XV = exact_mm_creal(OP) ? 4 : OP == EX_EVISCV ? 1 : 0;
  const ExactArgs& a = A.a;
  const int lane = tid & 63, col = lane & 15, row = lane >> 4;
  // the wave's field and output: rotated over the work-groups, so that the
  // waves without a field or output do not all sit on the same SIMD
  const int role = SFX_UNIFORM((int)(((tid >> 6) + bid) % NW));
  const int mb0 = mpart * MB;
  const int N = 2 * a.K + 1;
  const int64_t p = bid * 16 + col, pc = p < a.np ? p : a.np - 1;   // columns past the end repeat the last point
  const bool works = NO > 0 ? role < NO : role < 4;
  const double *xb = nullptr, *yb = nullptr;   // the real-space inputs of this point and row, forwards and backwards
  if constexpr (exact_mm_creal(OP)) {
    xb = a.creal + pc * N + row;
    yb = a.creal + pc * N + (N - row);
  }
  int64_t el = 0;
  double y = 0.0;
  if constexpr (OP == EX_EVISCV) {
    el = pc / a.lg;
    y = a.hloc[pc];
    xb = a.nint + el * N + row;
    yb = a.nint + el * N + (N - row);
  }
  sfx_d4 SA[MB], SB[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) SA[b] = SB[b] = sfx_d4{0, 0, 0, 0};

  for (int jb0 = 0; jb0 < (ONE ? 1 : A.jbn); jb0 += JB) {
    double xp[2][XV > 0 ? XV : 1], xm[2][XV > 0 ? XV : 1];
    // real-space inputs at angles 16 (jb0 + q) + 4 v + row and their mirrors
    auto real_in = [&](int q, int h) {
      const bool edge = ONE ? q == 0 || q == JB - 1 : jb0 + q == 0 || jb0 + q >= A.jbn - 1;   // uniform
#pragma unroll
      for (int i = 0; i < XV; ++i) {
        const int v = NO == 0 ? role : i;
        const int o = 16 * (jb0 + q) + 4 * v;
        if (edge) {
          const int jc = o + row <= a.K ? o + row : 0, jm = jc > 0 ? N - jc : 0;
          if constexpr (exact_mm_creal(OP)) {
            SFX_CHECK("exact creal", pc * N + jm, a.n_creal);
            xp[h][i] = a.creal[pc * N + jc];
            xm[h][i] = a.creal[pc * N + jm];
          } else if constexpr (OP == EX_EVISCV) {
            xp[h][i] = exact_evisc_norm(a, el, jc);
            xm[h][i] = exact_evisc_norm(a, el, jm);
          }
        } else if constexpr (exact_mm_creal(OP)) {
          SFX_CHECK("exact creal", yb - o - a.creal, a.n_creal);
          xp[h][i] = xb[o];
          xm[h][i] = yb[-o];
        } else if constexpr (OP == EX_EVISCV) {   // no wrap inside: angles 1 .. N - 2
          SFX_CHECK("exact nint", yb - o + 1 - a.nint, a.n_nint);
          xp[h][i] = fmax(fmax(xb[o - 1], xb[o]), xb[o + 1]);
          xm[h][i] = fmax(fmax(yb[-o - 1], yb[-o]), yb[-o + 1]);
        }
      }
    };
    if constexpr (XV > 0) {
      if (works) real_in(0, 0);
    }
    // ---- synthesis: E and O of field `role` at the angles of blocks jb0 .. jb0 + JB - 1
    sfx_d4 E[JB], O[JB];
#pragma unroll
    for (int q = 0; q < JB; ++q) E[q] = O[q] = sfx_d4{0, 0, 0, 0};
    if (NI > 0 && role < NI) {
      int64_t n;
      const ExactField F = exact_mm_in<OP, NI>(a, role, grp, n);
      // Loads return in order, so an input (memory) fetched between the factors
      // (L2) of two steps would hold up the second: inputs come four steps at a
      // time, the next four after the factors of the second of these steps.
      double c[2][4], s[2][4];
      const double* base = F.base + pc * F.sp;
      const double* in = base + row * F.sm;
      int m = row;                                // mode of `in`
      auto fetch = [&](int g) {
#pragma unroll
        for (int h = 0; h < 4; ++h, m += 4, in += 4 * F.sm) {
          const double* b = m < a.M ? in : base;
          SFX_CHECK("exact in", b - F.base + F.off, n);
          c[g][h] = b[0];
          s[g][h] = b[F.off];
        }
      };
      // a mode past M counts as zero; the sine of mode 0 is dropped (:241)
      auto mask = [&](int k0, int g) {
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const int mm = 4 * (k0 + h) + row;
          c[g][h] = mm < a.M ? c[g][h] : 0.0;
          s[g][h] = mm < a.M && mm > 0 ? s[g][h] : 0.0;
        }
      };
      double2 tb[2][JB];
      const double2* tp = reinterpret_cast<const double2*>(A.ct) + (int64_t)jb0 * 64 + lane;
      auto tables = [&](int h) {
#pragma unroll
        for (int q = 0; q < JB; ++q) {
          // past the last block (general form): the first one again, unused
          const double2* t = tp + (ONE || jb0 + q < A.jbn ? q : 0) * 64;
          SFX_CHECK("exact ct", 2 * (t - reinterpret_cast<const double2*>(A.ct)) + 1, A.n_ct);
          tb[h][q] = *t;
        }
        tp += (int64_t)(ONE ? JB : A.jbn) * 64;
      };
      auto step = [&](int g, int h) {
#pragma unroll
        for (int q = 0; q < JB; ++q) {
          E[q] = SFX_MFMA_F64(tb[h & 1][q].x, c[g][h], E[q]);
          O[q] = SFX_MFMA_F64(tb[h & 1][q].y, s[g][h], O[q]);
        }
      };
      auto four = [&](int k0, int g, bool more) {
        mask(k0, g);
        tables(1);
        step(g, 0);
        tables(0);
        if (more) fetch(g ^ 1);
        step(g, 1);
        tables(1);
        step(g, 2);
        if (more) tables(0);
        step(g, 3);
      };
      const int nb = ONE ? MB : A.mbn;            // groups of four steps
      fetch(0);
      tables(0);
      int b = 0;
      for (; b + 2 <= nb; b += 2) {
        four(4 * b, 0, true);
        four(4 * b + 4, 1, b + 2 < nb);
      }
      if (b < nb) four(4 * b, 0, false);
    }
    // ---- operation and analysis, one block of 16 angles after the other; the
    // real-space inputs of the next block and the factors of the next 4 angles
    // are in flight meanwhile
    double2 rt[2][MB];
    const double2* rp = reinterpret_cast<const double2*>(A.rt) + (int64_t)mb0 * 64 + lane;
    auto factors = [&](int jq, int h) {
#pragma unroll
      for (int b = 0; b < MB; ++b) {
        const int bb = ONE || mb0 + b < A.mbn ? b : 0;   // past the last block, the first one again, unused
        const double2* t = rp + ((int64_t)(jq < 4 * (ONE ? JB : A.jbn) ? jq : 0) * (ONE ? MB : A.mbn) + bb) * 64;
        SFX_CHECK("exact rt", 2 * (t - reinterpret_cast<const double2*>(A.rt)) + 1, A.n_rt);
        rt[h][b] = *t;
      }
    };
    if constexpr (NO > 0) {
      if (works) factors(4 * jb0, 0);
    }
#pragma unroll
    for (int q = 0; q < JB; ++q) {
      if (!ONE && jb0 + q >= A.jbn) continue;     // uniform over the work-group
      // buffers alternate with the block number, also from one pass to the next
      double* buf = smem + ((jb0 + q) & 1) * (NI * 512);
      if (NI > 0 && role < NI) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          buf[role * 512 + (2 * v) * 64 + lane] = E[q][v] + O[q][v];
          buf[role * 512 + (2 * v + 1) * 64 + lane] = E[q][v] - O[q][v];
        }
      }
      if (NI > 0) SFX_SYNC();
      if (works) {
        if constexpr (XV > 0) {
          if (q + 1 < JB && (ONE || jb0 + q + 1 < A.jbn)) real_in(q + 1, (q + 1) & 1);
        }
        const bool edge = ONE ? q == 0 || q == JB - 1 : jb0 + q == 0 || jb0 + q == A.jbn - 1;   // uniform
#pragma unroll
        for (int i = 0; i < (NO == 0 ? 1 : 4); ++i) {
          const int v = NO == 0 ? role : i;       // no analysis: wave v takes angles 4 v .. 4 v + 3
          const int j = 16 * (jb0 + q) + 4 * v + row;
          if constexpr (NO > 0) factors(4 * (jb0 + q) + v + 1, (v + 1) & 1);
          const double x1 = XV > 0 ? xp[q & 1][i < XV ? i : 0] : 0.0, x2 = XV > 0 ? xm[q & 1][i < XV ? i : 0] : 0.0;
          const double wp = exact_mm_op<OP, NI>(a, grp, role, [&](int f) { return buf[f * 512 + (2 * v) * 64 + lane]; }, x1, y);
          const double wm = exact_mm_op<OP, NI>(a, grp, role, [&](int f) { return buf[f * 512 + (2 * v + 1) * 64 + lane]; }, x2, y);
          if constexpr (OP == EX_EVISCV) {
            if (j <= a.K && p < a.np) {
              SFX_CHECK("exact rout", p * N + (j > 0 ? N - j : 0), a.n_nint2);
              a.rout1[p * N + j] = wp;
              if (j > 0) a.rout1[p * N + (N - j)] = wm;
            }
          } else {
            double S = wp + wm, D = wp - wm;
            if (edge) {   // angle 0 has no mirror; angles past K: zero, also where wp is not finite
              S = j > a.K ? 0.0 : j > 0 ? S : wp;
              D = j > a.K || j == 0 ? 0.0 : D;
            }
#pragma unroll
            for (int b = 0; b < MB; ++b) {
              SA[b] = SFX_MFMA_F64(rt[v & 1][b].x, S, SA[b]);
              SB[b] = SFX_MFMA_F64(rt[v & 1][b].y, D, SB[b]);
            }
          }
        }
      }
    }
  }
  if (NO > 0 && works && p < a.np) {
    int64_t n;
    const ExactOut F = exact_mm_out<OP, NO>(a, role, grp, n);
    double* o = F.base + p * F.sp + (16 * mb0 + row) * F.sm;
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
      for (int v = 0; v < 4; ++v, o += 4 * F.sm) {
        if (16 * (mb0 + b) + 4 * v + row >= a.M) continue;
        SFX_CHECK("exact out", o - F.base + F.off, n);
        o[0] = SA[b][v];
        o[F.off] = SB[b][v];
      }
  }
}

}  // namespace sfx
