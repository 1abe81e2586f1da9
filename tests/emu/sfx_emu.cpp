// CPU emulator of the libsfx kernel bodies (test infrastructure).
//
// Each work-group runs as 64*wpb std::threads sharing one LDS buffer, with a
// std::barrier standing in for __syncthreads.  Every global and LDS index the
// kernels compute is checked against its buffer (SFX_CHECK); a violation
// prints the site and aborts, so tests run the emulator in a child process.
#define SFX_EMULATE 1
#include <barrier>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <algorithm>
#include <functional>
#include <memory>
#include <thread>
#include <type_traits>
#include <vector>

#include "../../sfemans_amd/csrc/sfx_fftprod_body.h"
#include "../../sfemans_amd/csrc/sfx_twiddle.h"

static thread_local std::barrier<>* g_bar = nullptr;        // work-group barrier
static thread_local std::barrier<>* g_wave_bar = nullptr;   // barrier of the thread's wave (64 threads)
static thread_local double (*g_wave_ab)[64] = nullptr;       // the wave's matrix-core operands a, b
static thread_local int g_lane = 0;
void sfx_emu_sync() { g_bar->arrive_and_wait(); }
void sfx_emu_wave_sync() { g_wave_bar->arrive_and_wait(); }
// v_mfma_f64_16x16x4: every lane of the wave calls it together
sfx_d4 sfx_emu_mfma_f64(double a, double b, const sfx_d4& c) {
  g_wave_ab[0][g_lane] = a;
  g_wave_ab[1][g_lane] = b;
  g_wave_bar->arrive_and_wait();
  sfx_d4 d = c;
  for (int v = 0; v < 4; ++v)
    for (int k = 0; k < 4; ++k)
      d[v] = std::fma(g_wave_ab[0][16 * k + g_lane / 16 + 4 * v], g_wave_ab[1][16 * k + g_lane % 16], d[v]);
  g_wave_bar->arrive_and_wait();
  return d;
}
// transposition of (a, b) with a lane bit: every lane of the wave calls it together
void sfx_emu_lane_swap(double& a, double& b, int bit) {
  g_wave_ab[0][g_lane] = a;
  g_wave_ab[1][g_lane] = b;
  g_wave_bar->arrive_and_wait();
  const bool one = (g_lane & bit) != 0;
  const double x = one ? g_wave_ab[1][g_lane - bit] : a, y = one ? b : g_wave_ab[0][g_lane + bit];
  g_wave_bar->arrive_and_wait();
  a = x;
  b = y;
}
void sfx_emu_oob(const char* what, long long idx, long long n, const char* file, int line) {
  std::fprintf(stderr, "SFX_EMU out of bounds: %s index %lld not in [0,%lld) at %s:%d\n", what, idx, n, file, line);
  std::fflush(stderr);
  std::abort();
}

using namespace sfx;

static void run_grid(int64_t nblk, int threads, size_t smem_cplx,
                     const std::function<void(int, int64_t, double2*)>& body) {
  // LDS followed by a guard zone: a write past the end of the declared LDS
  // size changes the guard and aborts the run
  constexpr size_t GUARD = 256;
  std::vector<double2> smem(smem_cplx + GUARD);
  for (int64_t b = 0; b < nblk; ++b) {
    std::barrier<> bar(threads);
    std::vector<std::unique_ptr<std::barrier<>>> wbar;
    for (int w = 0; w < (threads + 63) / 64; ++w)
      wbar.emplace_back(new std::barrier<>(std::min(64, threads - 64 * w)));
    std::vector<double> ab((size_t)wbar.size() * 128);
    for (auto& x : smem) x = make_double2(1e300, -1e300);   // poison: stale reads show up
    std::vector<std::thread> th;
    th.reserve(threads);
    for (int t = 0; t < threads; ++t)
      th.emplace_back([&, t] { g_bar = &bar; g_wave_bar = wbar[t / 64].get();
                            g_wave_ab = reinterpret_cast<double(*)[64]>(&ab[(size_t)(t / 64) * 128]); g_lane = t % 64; body(t, b, smem.data()); });
    for (auto& x : th) x.join();
    for (size_t i = smem_cplx; i < smem.size(); ++i)
      if (smem[i].x != 1e300 || smem[i].y != -1e300) sfx_emu_oob("LDS guard", (long long)i, (long long)smem_cplx, __FILE__, __LINE__);
  }
}

template <int MP, int OP>
static void emu_fftprod_mp(const FftProdArgs& a, int wpb) {
  const int64_t pts = (int64_t)Shape<MP>::PW * wpb;
  const int64_t nblk = (a.np + pts - 1) / pts;
  run_grid(nblk, 64 * wpb, fftprod_smem_cplx<MP>(wpb),
           [&](int t, int64_t b, double2* s) { fftprod_body<MP, OP>(a, t, b, wpb, s); });
}

template <int OP>
static int emu_op(const FftProdArgs& a, int wpb) {
  switch (a.MP) {
    case 4: emu_fftprod_mp<4, OP>(a, wpb); return 0;
    case 8: emu_fftprod_mp<8, OP>(a, wpb); return 0;
    case 16: emu_fftprod_mp<16, OP>(a, wpb); return 0;
    case 32: emu_fftprod_mp<32, OP>(a, wpb); return 0;
    case 64: emu_fftprod_mp<64, OP>(a, wpb); return 0;
    case 128: emu_fftprod_mp<128, OP>(a, wpb); return 0;
    case 256: emu_fftprod_mp<256, OP>(a, wpb); return 0;
  }
  return 1;
}

extern "C" int emu_fftprod(int op, const double* V1, const double* V2, double* Vout, int64_t np, int M,
                           int nb1, int nb2, int nbout, int wpb) {
  FftProdArgs a;
  a.V1 = V1; a.V2 = V2; a.Vout = Vout;
  a.np = np; a.M = M; a.MP = mp_for(M); a.nb1 = nb1; a.nb2 = nb2;
  a.n1 = np * nb1 * (int64_t)M; a.n2 = np * nb2 * (int64_t)M; a.nout = np * nbout * (int64_t)M;
  std::vector<double2> wN, wMP;
  host_twiddles(a.MP, wN, wMP);
  a.wN = wN.data(); a.wMP = wMP.data();
  switch (op) {
    case OP_CROSS: return emu_op<OP_CROSS>(a, wpb);
    case OP_DOT: return emu_op<OP_DOT>(a, wpb);
    case OP_PROD: return emu_op<OP_PROD>(a, wpb);
    case OP_SVECT1: return emu_op<OP_SVECT1>(a, wpb);
    case OP_TENSOR: return emu_op<OP_TENSOR>(a, wpb);
  }
  return 2;
}

// ---- fused Gauss-point kernels
#include "../../sfemans_amd/csrc/sfx_gauss_body.h"
#include "../../sfemans_amd/csrc/sfx_p2tab.h"

template <int MP, int V>
static void emu_gauss_mp(const GaussArgs& a) {
  // as the GPU launcher
  const bool whole = gauss_take_whole<MP, V>(a.me) || !(gauss_point_tiles<MP, V>() || gauss_half<MP, V>());
  const int64_t nblk = whole ? gauss_whole_blocks<MP>(a.me) : gauss_blocks<MP, V>(a.me);
  if (whole) {
    constexpr int NW = gauss_waves<MP, V>();
    run_grid(nblk, 64 * NW, GaussCfg<MP, V, NW>::LY::TOTAL,
             [&](int t, int64_t b, double2* s) { gauss_body<MP, V, NW>(a, t, b, s); });
  } else if constexpr (gauss_point_tiles<MP, V>()) {
    run_grid(nblk, 64 * GAUSS_PT_WAVES, GaussPtCfg<MP, V>::LY::TOTAL, [&](int t, int64_t b, double2* s) {
      gauss_body<MP, V, GAUSS_PT_WAVES, false, false, true, gauss_pt_elems<MP>()>(a, t, b, s);
    });
  } else if constexpr (gauss_half<MP, V>()) {
    run_grid(nblk, 256, GaussHalfCfg<MP, V>::LY::TOTAL,
             [&](int t, int64_t b, double2* s) { gauss_body<MP, V, 4, false, false, false, 128 / MP>(a, t, b, s); });
  }
}

template <int V>
static int emu_gauss_v(const GaussArgs& a) {
  switch (a.MP) {
    case 4: emu_gauss_mp<4, V>(a); return 0;
    case 8: emu_gauss_mp<8, V>(a); return 0;
    case 16: emu_gauss_mp<16, V>(a); return 0;
    case 32: emu_gauss_mp<32, V>(a); return 0;
    case 64: emu_gauss_mp<64, V>(a); return 0;
    case 128: emu_gauss_mp<128, V>(a); return 0;
    case 256: emu_gauss_mp<256, V>(a); return 0;
  }
  return 1;
}

extern "C" int emu_gauss(int variant, const int32_t* jj, const double* rr, int64_t me, int64_t np,
                         const double* U, int ncU, const double* U2, int ncU2, const double* U3,
                         const double* heat_capa, const int32_t* list_mode, int M, double* Vout, int ncout,
                         double c_lorentz, double om0, double om1, double om2) {
  // variants: 0 cross-curl, 1 (curl U) x U2, 2 u.grad c, 3 MHD (U=u, U2=H, U3=B), 4 tangent (U, U2=dU)
  GaussArgs a;
  std::memset(&a, 0, sizeof(a));
  a.jj = jj; a.rr = rr; a.me = me; a.np = np; a.G = 7 * me;
  a.U = U; a.U2 = U2;
  a.nU = np * ncU * (int64_t)M; a.nU2 = np * ncU2 * (int64_t)M;
  const int64_t n6 = np * 6 * (int64_t)M;
  int kernel = GV_PAIRS;
  auto add = [&](const double* c, const double* v, double k) {
    a.pc[a.npass] = c; a.pv[a.npass] = v; a.coef[a.npass] = k; a.npc[a.npass] = a.npv[a.npass] = n6; ++a.npass;
  };
  if (variant == 0) kernel = GV_CROSS_CURL;
  else if (variant == 2) kernel = GV_UGRADC;
  else if (variant == 1) add(U, U2, 1.0);
  else if (variant == 3) { add(U2, U3, -c_lorentz); add(U, U, 1.0); }
  else if (variant == 4) { add(U, U2, 1.0); add(U2, U, 1.0); }
  a.heat_capa = heat_capa; a.list_mode = list_mode;
  double tab[126];
  p2_reference_tables(tab);
  a.tab = tab;
  a.Vout = Vout; a.nout = a.G * ncout * (int64_t)M;
  a.M = M; a.MP = mp_for(M);
  a.om[0] = om0; a.om[1] = om1; a.om[2] = om2;
  std::vector<double2> wN, wMP;
  host_twiddles(a.MP, wN, wMP);
  a.wN = wN.data(); a.wMP = wMP.data();
  if (kernel == GV_PAIRS && pairs_as_passes(a.MP)) {
    // as the library: one single-pass launch per pass, adding to the output
    const GaussArgs all = a;
    for (int i = 0; i < all.npass; ++i) {
      a.npass = 1;
      a.pc[0] = all.pc[i]; a.pv[0] = all.pv[i]; a.coef[0] = all.coef[i];
      a.npc[0] = all.npc[i]; a.npv[0] = all.npv[i];
      a.accum = i > 0;
      if (emu_gauss_v<GV_CURL_CROSS>(a)) return 1;
    }
    return 0;
  }
  switch (kernel) {
    case GV_CROSS_CURL: return emu_gauss_v<GV_CROSS_CURL>(a);
    case GV_PAIRS: return emu_gauss_v<GV_PAIRS>(a);
    case GV_UGRADC: return emu_gauss_v<GV_UGRADC>(a);
  }
  return 2;
}

// ---- right-hand-side assembly
#include "../../sfemans_amd/csrc/sfx_rhs_body.h"

static void build_adjacency(const int32_t* jj, int64_t me, int64_t np, std::vector<int64_t>& ptr,
                            std::vector<int32_t>& ent) {
  ptr.assign(np + 1, 0);
  for (int64_t e = 0; e < me; ++e)
    for (int n = 0; n < 6; ++n) ptr[jj[6 * e + n]] += 1;
  for (int64_t i = 0; i < np; ++i) ptr[i + 1] += ptr[i];
  ent.assign(ptr[np], 0);
  std::vector<int64_t> fill(ptr.begin(), ptr.end() - 1);
  for (int64_t e = 0; e < me; ++e)
    for (int n = 0; n < 6; ++n) ent[fill[jj[6 * e + n] - 1]++] = (int32_t)(6 * e + n);
}

extern "C" int emu_rhs(int which, const int32_t* jj, const double* rr, int64_t me, int64_t np, int M,
                       const double* rhs, double* v145, double* v236, const double* hc, const double* ff,
                       const double* ffg, double* vect, double scale) {
  std::vector<int64_t> ptr;
  std::vector<int32_t> ent;
  build_adjacency(jj, me, np, ptr, ent);
  double tab[126];
  p2_reference_tables(tab);
  std::vector<double> wgt(7 * me);
  p2_assembly_weights(jj, rr, me, tab, wgt.data());
  RhsArgs a;
  std::memset(&a, 0, sizeof(a));
  a.adj_ptr = ptr.data(); a.adj_ent = ent.data(); a.wgt = wgt.data(); a.tab = tab;
  a.jj = jj; a.me = me; a.np = np; a.G = 7 * me; a.M = M; a.scale = scale; a.n_adj = (int64_t)ent.size();
  if (which == 0) {
    std::vector<double> elo((size_t)36 * me * M + 1);
    a.rhs = rhs; a.v145 = v145; a.v236 = v236; a.elo = elo.data();
    a.n_rhs = a.G * 6 * (int64_t)M; a.n_out = np * 3 * (int64_t)M; a.n_elo = 36 * me * (int64_t)M;
    for (int64_t g = 0; g < elem_items(me, M); ++g) rhs_elem_body(a, g);
    run_grid((np + GATHER_NODES - 1) / GATHER_NODES, GATHER_THREADS, (gather_tile_doubles<6>() + 1) / 2,
             [&](int t, int64_t b, double2* sm) { rhs_gather_block(a, b, t, reinterpret_cast<double*>(sm)); });
  } else {
    std::vector<double> elo((size_t)6 * me * M + 1);
    a.heat_capa = hc; a.ff = ff; a.ffg = ffg; a.vect = vect; a.elo = elo.data();
    a.n_ff = np * (int64_t)M; a.n_ffg = a.G * (int64_t)M; a.n_out = np * (int64_t)M; a.n_elo = 6 * me * (int64_t)M;
    for (int64_t g = 0; g < elem_items(me, M); ++g) qs00_elem_body(a, g);
    run_grid((np + GATHER_NODES - 1) / GATHER_NODES, GATHER_THREADS, (gather_tile_doubles<1>() + 1) / 2,
             [&](int t, int64_t b, double2* sm) { qs00_gather_block(a, b, t, reinterpret_cast<double*>(sm)); });
  }
  return 0;
}

#include "../../sfemans_amd/csrc/sfx_bdy_setup.h"

// Boundary term of rhs_3x3 added to vb145/vb236 (np, 3, M).
extern "C" int emu_rhs_bdy(const int32_t* jjs, int64_t mes, const double* rr, int64_t np, int M, const double* tb,
                           double* v145, double* v236, double scale) {
  BdyTables t;
  build_boundary_tables(jjs, mes, rr, np, t);
  BdyArgs a;
  std::memset(&a, 0, sizeof(a));
  double d[9], p[3];
  p2_edge_tables(a.wws, d, p);
  a.bptr = t.ptr.data(); a.bent = t.ent.data(); a.bnode = t.node.data(); a.bw = t.bw.data();
  a.nb = (int64_t)t.node.size(); a.mes = mes; a.np = np; a.M = M; a.scale = scale;
  a.tb = tb; a.v145 = v145; a.v236 = v236;
  a.n_tb = 3 * mes * 6 * (int64_t)M; a.n_out = np * 3 * (int64_t)M; a.n_ent = (int64_t)t.ent.size();
  for (int64_t g = 0; g < a.nb * (int64_t)M; ++g) rhs_bdy_body(a, g);
  return 0;
}

// The Gauss values of the NS right-hand side (the first step of the penalty
// branch): gout(G, 6, M) = ft + fp_inc + fs - rotv_v - (imposed velocity on imp_slot).
extern "C" int emu_rhs_ns_gauss(const int32_t* jj, const double* rr, int64_t me, int64_t np, const int32_t* lm,
                                int M, const double* rotv, const double* V1m, const double* ff, const double* Pinc,
                                const double* imp, int imp_slot, double* gout) {
  std::vector<int64_t> ptr;
  std::vector<int32_t> ent;
  build_adjacency(jj, me, np, ptr, ent);
  double tab[126];
  p2_reference_tables(tab);
  std::vector<double> wgt(7 * me);
  p2_assembly_weights(jj, rr, me, tab, wgt.data());
  RhsArgs a;
  std::memset(&a, 0, sizeof(a));
  a.adj_ptr = ptr.data(); a.adj_ent = ent.data(); a.wgt = wgt.data(); a.tab = tab;
  a.jj = jj; a.me = me; a.np = np; a.G = 7 * me; a.M = M; a.scale = 1.0; a.n_adj = (int64_t)ent.size();
  a.rr = rr; a.lmode = lm;
  a.rhs = rotv; a.v1m = V1m; a.fsrc = ff; a.pinc = Pinc; a.rsign = -1.0;
  a.imp = imp; a.imp_slot = imp ? imp_slot : -1; a.isign = -1.0; a.gout = gout;
  a.n_rhs = a.G * 6 * (int64_t)M; a.n_v1m = a.n_fsrc = np * 6 * (int64_t)M; a.n_pinc = np * 2 * (int64_t)M;
  a.n_imp = np * 6; a.n_gout = a.G * 6 * (int64_t)M;
  for (int64_t g = 0; g < elem_items(me, M); ++g) rhs_ns_gauss_body(a, g);
  return 0;
}

template <int MC>
static void emu_rns_elems(const RhsArgs& a) {
  if (a.tens)
    run_grid(rns_blocks(a.me, a.M, MC), RNS_THREADS, (rns_smem_doubles<true>() + 1) / 2, [&](int t, int64_t b, double2* sm) {
      rhs_ns_tile_body<true, MC>(a, t, b, reinterpret_cast<double*>(sm));
    });
  else
    run_grid(rns_blocks(a.me, a.M, MC), RNS_THREADS, (rns_smem_doubles<false>() + 1) / 2, [&](int t, int64_t b, double2* sm) {
      rhs_ns_tile_body<false, MC>(a, t, b, reinterpret_cast<double*>(sm));
    });
}

extern "C" int emu_rns_modes(int64_t me, int M) { return rns_modes(me, M); }

extern "C" int emu_rhs_ns(const int32_t* jj, const double* rr, int64_t me, int64_t np, const int32_t* lm, int M,
                          const double* rotv, const double* V1m, const double* ff, const double* P,
                          const double* Pinc, const double* tens, double* v145, double* v236) {
  std::vector<int64_t> ptr;
  std::vector<int32_t> ent;
  build_adjacency(jj, me, np, ptr, ent);
  double tab[126];
  p2_reference_tables(tab);
  std::vector<double> wgt(7 * me);
  p2_assembly_weights(jj, rr, me, tab, wgt.data());
  RhsArgs a;
  std::memset(&a, 0, sizeof(a));
  a.adj_ptr = ptr.data(); a.adj_ent = ent.data(); a.wgt = wgt.data(); a.tab = tab;
  a.jj = jj; a.me = me; a.np = np; a.G = 7 * me; a.M = M; a.scale = 1.0; a.n_adj = (int64_t)ent.size();
  std::vector<double> elo((size_t)36 * me * M + 1);
  a.rr = rr; a.lmode = lm;
  a.rhs = rotv; a.v1m = V1m; a.fsrc = ff; a.pres = P; a.pinc = Pinc; a.tens = tens; a.rsign = -1.0;
  a.v145 = v145; a.v236 = v236; a.elo = elo.data();
  a.n_rhs = a.G * 6 * (int64_t)M; a.n_v1m = a.n_fsrc = np * 6 * (int64_t)M; a.n_pres = a.n_pinc = np * 2 * (int64_t)M;
  a.n_tens = 3 * a.n_rhs;
  a.n_out = np * 3 * (int64_t)M; a.n_elo = 36 * me * (int64_t)M;
  // both forms, whichever the rule takes; their element sums are the same bits
  emu_rns_elems<RNS_FEW>(a);
  const std::vector<double> few = elo;
  std::fill(elo.begin(), elo.end(), NAN);
  emu_rns_elems<RNS_MC>(a);
  if (std::memcmp(few.data(), elo.data(), sizeof(double) * 36 * me * M) != 0) return 1;
  run_grid((np + GATHER_NODES - 1) / GATHER_NODES, GATHER_THREADS, (gather_tile_doubles<6>() + 1) / 2,
           [&](int t, int64_t b, double2* sm) { rhs_gather_block(a, b, t, reinterpret_cast<double*>(sm)); });
  return 0;
}

// ---- adjoint of the tangent
#include "../../sfemans_amd/csrc/sfx_adjoint_body.h"

template <int MP, bool SPLIT>
static void emu_adjoint_mp(const AdjArgs& A) {
  constexpr int NW = adjoint_waves<MP, SPLIT>();
  constexpr int E = adjoint_elems<MP, SPLIT>();
  const int64_t nblk = (A.g.me + E - 1) / E;
  run_grid(nblk, 64 * NW, AdjLds<MP, SPLIT, NW>::TOTAL,
           [&](int t, int64_t b, double2* s) { adjoint_body<MP, SPLIT, NW>(A, t, b, s); });
}

template <bool SPLIT>
static void emu_adjoint_split(const AdjArgs& A) {
  switch (A.g.MP) {
    case 4: emu_adjoint_mp<4, SPLIT>(A); break;
    case 8: emu_adjoint_mp<8, SPLIT>(A); break;
    case 16: emu_adjoint_mp<16, SPLIT>(A); break;
    case 32: emu_adjoint_mp<32, SPLIT>(A); break;
    case 64: emu_adjoint_mp<64, SPLIT>(A); break;
    case 128: emu_adjoint_mp<128, SPLIT>(A); break;
    case 256: emu_adjoint_mp<256, SPLIT>(A); break;
  }
}

// UB == nullptr: convective adjoint around U into dbar.  Otherwise the split
// (Lorentz) form around (A = U, B = UB) times coef: W^T part into dbar, R^T
// part into dbar2.
extern "C" int emu_adjoint(const int32_t* jj, const double* rr, int64_t me, int64_t np, const double* U,
                           const double* ybar, const int32_t* list_mode, int M, double* dbar, const double* UB,
                           double coef, double* dbar2) {
  const bool split = UB != nullptr;
  AdjArgs A;
  std::memset(&A, 0, sizeof(A));
  GaussArgs& a = A.g;
  a.jj = jj; a.rr = rr; a.me = me; a.np = np; a.G = 7 * me;
  a.U = U; a.nU = np * 6 * (int64_t)M;
  a.list_mode = list_mode;
  double tab[126];
  p2_reference_tables(tab);
  a.tab = tab;
  a.M = M; a.MP = mp_for(M);
  std::vector<double2> wN, wMP;
  host_twiddles(a.MP, wN, wMP);
  a.wN = wN.data(); a.wMP = wMP.data();
  std::vector<double> elo((size_t)6 * me * 6 * M, -1e300), elo2(split ? elo.size() : 1, -1e300);
  A.UB = UB; A.nUB = split ? a.nU : 0; A.coef = split ? coef : 1.0;
  A.ybar = ybar; A.nybar = a.G * 6 * (int64_t)M;
  A.elo = elo.data(); A.elo2 = split ? elo2.data() : nullptr; A.nelo = (int64_t)elo.size();
  if (split) emu_adjoint_split<true>(A);
  else emu_adjoint_split<false>(A);
  std::vector<int64_t> ptr;
  std::vector<int32_t> ent;
  build_adjacency(jj, me, np, ptr, ent);
  GatherArgs ga;
  ga.adj_ptr = ptr.data(); ga.adj_ent = ent.data(); ga.elo = elo.data(); ga.out = dbar;
  ga.me = me; ga.np = np; ga.n_adj = (int64_t)ent.size(); ga.nelo = (int64_t)elo.size();
  ga.nout = np * 6 * (int64_t)M; ga.M = M;
  auto gather = [&](const GatherArgs& g) {
    run_grid((np + GATHER_NODES - 1) / GATHER_NODES, GATHER_THREADS, (gather_tile_doubles<6>() + 1) / 2,
             [&](int t, int64_t b, double2* sm) { adjoint_gather_block(g, b, t, reinterpret_cast<double*>(sm)); });
  };
  gather(ga);
  if (split) {
    ga.elo = elo2.data(); ga.out = dbar2;
    gather(ga);
  }
  return 0;
}

// ---- batched persistent launch: problems packed in flat buffers with offsets
#include "../../sfemans_amd/csrc/sfx_batch_body.h"

extern "C" int emu_batch(int n, const int32_t* jj, const int64_t* jj_off, const double* rr, const int64_t* rr_off,
                         const int64_t* me, const int64_t* np, const double* U, const int64_t* U_off,
                         const int32_t* lm, const int64_t* lm_off, const int32_t* M, double* out,
                         const int64_t* out_off, int policy, int n_wg, int32_t* n_wg_used) {
  std::vector<GaussArgs> probs(n);
  std::vector<std::vector<double2>> wN(n), wMP(n);
  double tab[126];
  p2_reference_tables(tab);
  std::vector<int64_t> mev(n);
  std::vector<int> mp(n);
  size_t smem = 0;
  for (int i = 0; i < n; ++i) {
    GaussArgs& a = probs[i];
    std::memset(&a, 0, sizeof(a));
    a.jj = jj + jj_off[i]; a.rr = rr + rr_off[i]; a.me = me[i]; a.np = np[i]; a.G = 7 * me[i];
    a.U = U + U_off[i]; a.nU = np[i] * 6 * (int64_t)M[i];
    a.list_mode = lm + lm_off[i]; a.tab = tab;
    a.Vout = out + out_off[i]; a.nout = a.G * 6 * (int64_t)M[i];
    a.M = M[i]; a.MP = mp_for(M[i]);
    host_twiddles(a.MP, wN[i], wMP[i]);
    a.wN = wN[i].data(); a.wMP = wMP[i].data();
    mev[i] = me[i];
    mp[i] = a.MP;
    if (batch_smem_cplx(a.MP) > smem) smem = batch_smem_cplx(a.MP);
  }
  std::vector<BatchTile> nat, tiles;
  std::vector<double> cost;
  std::vector<int32_t> ptr;
  batch_tiles(mev, mp, nat, cost);
  const int32_t used = batch_schedule(nat, cost, mp, policy, n_wg, tiles, ptr);
  if (used < 0) return 1;
  *n_wg_used = used;
  BatchArgs b;
  b.probs = probs.data(); b.tiles = tiles.data(); b.wg_ptr = ptr.data();
  b.n_prob = n; b.n_wg = used; b.n_tiles = (int64_t)tiles.size();
  if (policy == 3) {
    // as the library: one grid per grid size
    for (int32_t c = 0; c < used; ++c) {
      const int32_t t0 = ptr[c], nt = ptr[c + 1] - t0;
      if (nt <= 0) continue;
      auto grid = [&](auto mpc) {
        constexpr int MPC = decltype(mpc)::value;
        constexpr int NW = gauss_waves<MPC, GV_CROSS_CURL>();
        run_grid(nt, 64 * NW, GaussCfg<MPC, GV_CROSS_CURL, NW>::LY::TOTAL,
                 [&](int t, int64_t w, double2* s) { batch_class_body<MPC>(b, t0, t, w, s); });
      };
      switch (probs[tiles[t0].prob].MP) {
        case 4: grid(std::integral_constant<int, 4>()); break;
        case 8: grid(std::integral_constant<int, 8>()); break;
        case 16: grid(std::integral_constant<int, 16>()); break;
        case 32: grid(std::integral_constant<int, 32>()); break;
        case 64: grid(std::integral_constant<int, 64>()); break;
        case 128: grid(std::integral_constant<int, 128>()); break;
        case 256: grid(std::integral_constant<int, 256>()); break;
        default: return 1;
      }
    }
    return 0;
  }
  run_grid(used, 64 * BATCH_WAVES, smem,
           [&](int t, int64_t w, double2* s) { batch_body(b, t, (int)w, s); });
  return 0;
}

// ---- exact-grid products (non-polynomial FFT_PAR_*)
#include "../../sfemans_amd/csrc/sfx_exact_setup.h"

template <int OP, int NI>
static void emu_exact_grid(const ExactArgs& a, double& vmax) {
  constexpr int JC = exact_jc(OP, NI);
  const int nch = (a.K + 1 + JC - 1) / JC;
  for (int64_t p = 0; p < a.np; ++p)
    for (int jc = 0; jc < nch; ++jc) exact_grid_body<OP, NI>(a, p, jc, vmax);
}

// FFT_COMPUTE_ENTROPY_VISC: V = [V1 .. V5] (5 x np*6*M), out = [O1 | O2 | O3];
// the element maxima as exact_enorm_kernel computes them (32 elements and 16
// angle pairs per work-group, one thread per point).
static int emu_exact_mm_op(int op, ExactArgs& a);
static int emu_evisc(bool mm, int64_t np, int M, int mp, int lg, const double* V, const double* hloc, double c1,
                     double c2, double c4, double res, double* out) {
  const int64_t n6 = np * 6 * M;
  const double* Vp[5] = {V, V + n6, V + 2 * n6, V + 3 * n6, V + 4 * n6};
  double* O[3] = {out, out + n6, out + 2 * n6};
  ExactArgs a;
  exact_setup_evisc(a, Vp, hloc, O, np, M, lg, c1, c2, c4, res);
  exact_setup_sizes(a, np, M, mp);
  std::vector<double> tab;
  exact_host_tables(M, a.K, tab);
  a.ctab = tab.data();
  a.rtab = tab.data() + exact_ctab_size(M, a.K);
  const int N = 2 * a.K + 1;
  const int64_t me = np / lg;
  std::vector<double> nint((size_t)me * N + 1, -1.0);
  a.nint = nint.data();
  a.n_nint = me * N;
  constexpr int RW = 2 * EXACT_NORM_JC + 1;
  const int nch = (a.K + 1 + EXACT_NORM_JC - 1) / EXACT_NORM_JC;
  std::vector<double> red((size_t)32 * lg * RW);
  for (int64_t eb = 0; eb < (me + 31) / 32; ++eb)
    for (int jc = 0; jc < nch; ++jc) {
      const int j0 = jc * EXACT_NORM_JC;
      for (int t = 0; t < 32 * lg; ++t) {
        const int64_t p = eb * 32 * lg + t;
        double nrm[2 * EXACT_NORM_JC] = {0};
        if (p < np) exact_norm_body(a, p, j0, nrm);
        for (int v = 0; v < 2 * EXACT_NORM_JC; ++v) red[(size_t)t * RW + v] = nrm[v];
      }
      for (int le = 0; le < 32; ++le)
        for (int v = 0; v < 2 * EXACT_NORM_JC; ++v) {
          const int64_t e = eb * 32 + le;
          const int j = j0 + v % EXACT_NORM_JC;
          const bool mirror = v >= EXACT_NORM_JC;
          if (e >= me || j > a.K || (mirror && j == 0)) continue;
          double x = red[(size_t)(le * lg) * RW + v];
          for (int l = 1; l < lg; ++l) x = std::max(x, red[(size_t)(le * lg + l) * RW + v]);
          nint[(size_t)e * N + (mirror ? N - j : j)] = x;
        }
    }
  for (double x : std::vector<double>(nint.begin(), nint.begin() + me * N))
    if (x < 0) return 3;   // every (element, angle) written
  a.n_W = 2 * (int64_t)a.nout * (a.K + 1) * np;
  std::vector<double> W((size_t)a.n_W + 1);
  a.W = W.data();
  // as the library launches it: the viscosity on the grid, then the products
  std::vector<double> vreal((size_t)N * np + 1);
  ExactArgs v, w;
  exact_evisc_split(a, vreal.data(), v, w);
  double vmax = 0.0;
  if (mm) {
    const int rc = emu_exact_mm_op(EX_EVISCV, v);
    return rc ? rc : emu_exact_mm_op(EX_GRADMOM, w);
  }
  emu_exact_grid<EX_EVISCV, 6>(v, vmax);
  emu_exact_grid<EX_GRADMOM, 9>(w, vmax);
  const int nmc = (M + EXACT_MC - 1) / EXACT_MC;
  for (int64_t p = 0; p < np; ++p)
    for (int g = 0; g < w.nout; ++g)
      for (int mc = 0; mc < nmc; ++mc) exact_r2c_body(w, p, g, mc);
  return 0;
}

extern "C" int emu_exact_evisc(int64_t np, int M, int mp, int lg, const double* V, const double* hloc, double c1,
                               double c2, double c4, double res, double* out) {
  return emu_evisc(false, np, M, mp, lg, V, hloc, c1, c2, c4, res, out);
}
extern "C" int emu_exact_evisc_mm(int64_t np, int M, int mp, int lg, const double* V, const double* hloc, double c1,
                                  double c2, double c4, double res, double* out) {
  return emu_evisc(true, np, M, mp, lg, V, hloc, c1, c2, c4, res, out);
}

extern "C" int emu_exact(int op, int64_t np, int M, int mp, const double* in1, const double* in2,
                         const double* values, int n_values, double eps, int nb, double* out);

// The argument sets of emu_exact (below); cls_vmax holds EX_CLS's velocity maximum.
static int emu_exact_setup(ExactArgs& a, double& cls_vmax, int op, int64_t np, int M, int mp, const double* in1,
                           const double* in2, const double* values, int n_values, double eps, int nb, double* out) {
  switch (op) {
    case EX_DIV: exact_setup_div(a, in1, in2, out, np, M); break;
    case EX_SV2: exact_setup_sv2(a, in1, in2, out, np, M); break;
    case EX_SQRT: exact_setup_sqrt(a, in1, out, np, nb, M); break;
    case EX_HEAVI: exact_setup_heavi(a, in1, values, n_values, out, np, M, eps); break;
    case EX_TENSION: exact_setup_tension(a, in1, in2, out, np, M); break;
    case EX_MAXVEL: exact_setup_maxvel(a, in1, np, nb, M); break;
    case EX_SVCLAMP: exact_setup_svclamp(a, in1, in2, out, np, M, nb, values[0], values[1]); break;
    case EX_CLAMP01: exact_setup_sqrt(a, in1, out, np, nb, M); break;
    case EX_ENTRO:   // in2 = c (np,2,M) then c_in_real (N,np) packed after it; out = V_out then c_out
      exact_setup_entro(a, in1, in2, in2 + 2 * np * M, values[0], out, out + 6 * np * M, np, M, mp);
      break;
    case EX_GRADMOM:   // in1 = [V1 | V2 | V3] (3 x np*6*M) then c_in_real (N, np); values = {coeff}
      exact_setup_gradmom(a, in1, in1 + 6 * np * M, in1 + 12 * np * M, in1 + 18 * np * M, values[0], out, np, M, mp);
      break;
    case EX_COMPR:   // in1 = [V1 | V2] (2 x np*6*M), in2 = [c (np,2,M) | c_in_real (N,np)],
                     // values = {coeff, comp}, out = [V_out | c_out]
      exact_setup_compr(a, in1, in1 + 6 * np * M, in2, in2 + 2 * np * M, values[0], values[1], out,
                        out + 6 * np * M, np, M, mp);
      break;
    case EX_CLS: {   // in1 = [grad phi | velocity] (2 x np*6*M), in2 = phi (np,2,M),
                     // values = {level_set_comp_factor, LES_coeff4, h_min_distance}
      const int rc = emu_exact(EX_MAXVEL, np, M, mp, in1 + 6 * np * M, nullptr, nullptr, 0, 0.0, 6, &cls_vmax);
      if (rc) return rc;
      exact_setup_cls(a, in1, in2, out, &cls_vmax, np, M, values[0], values[1], values[2]);
      break;
    }
    case EX_ETA:     // 17/18 eta products: in1 = c (np, nb, M), in2 = eta (N, np)
    case EX_ETA3: exact_setup_eta(a, in2, in1, out, np, nb, M, mp); break;
    case EX_FROMREAL: exact_setup_fromreal(a, in2, out, np, M, mp); break;   // 19: in2 = values (N, np)
    default: return 1;
  }
  return 0;
}

// op: 0 DIV (in1 c1, in2 c2), 1 SV2 (in1 V, in2 s), 2 SQRT (in1 c (np,nb,M), out a copy of c),
// 3 HEAVISIDE (in1 V1 (n_int,np,2,M), values), 4 TENSION (in1, in2 (np,6,M), out (3,np,6,M)),
// 5 MAX_VEL (in1 (np,nb,M), out[0] = maximum), 6 SCALAR_VECT_NO_OVERSHOOT (in1 V, in2 s,
// nb = pb, values = {min, max}), 7 NO_OVERSHOOT_LEVEL_SET (as 2), 8 ENTRO_VISC (in1 V,
// in2 = [c (np,2,M) | c_in_real (N,np)], values = {coeff}, out = [V_out | c_out]); 9-10, 13
// below.
extern "C" int emu_exact(int op, int64_t np, int M, int mp, const double* in1, const double* in2,
                         const double* values, int n_values, double eps, int nb, double* out) {
  ExactArgs a;
  double cls_vmax = 0.0;
  if (op == EX_VELSTAT) {   // 15 FFT_MAX_MIN_VEL_DCL: in1 (np, nb, M) -> out[0] max, out[1] min
    int rc = emu_exact(EX_MAXVEL, np, M, mp, in1, nullptr, nullptr, 0, 0.0, nb, out);
    if (rc) return rc;
    exact_setup_maxvel(a, in1, np, nb, M);
    exact_setup_sizes(a, np, M, mp);
    std::vector<double> tab;
    exact_host_tables(M, a.K, tab);
    a.ctab = tab.data();
    a.rtab = tab.data() + exact_ctab_size(M, a.K);
    double r[3] = {0.0, -INFINITY, 0.0};
    const int JC = exact_jc(EX_MAXVEL, a.nin), nch = (a.K + 1 + JC - 1) / JC;
    for (int64_t p = 0; p < np; ++p)
      for (int jc = 0; jc < nch; ++jc) {
        if (a.nin == 3) exact_velstat_body<3>(a, p, jc, r);
        else exact_velstat_body<1>(a, p, jc, r);
      }
    if (r[0] != out[0]) return 3;   // the one-pass maximum equals FFT_MAX_VEL_DCL's
    out[1] = r[2] >= 1.0 ? -r[1] : 0.0;
    return 0;
  }
  if (op == EX_CHECKIF) {   // 16 FFT_CHECK_INTERFACE: in1 (nb - 1, np, 2, M), nb = nb_fluids -> out[0] = ok
    if (nb == 2) { out[0] = 1.0; return 0; }
    exact_setup_checkif(a, in1, nb - 1, np, M);
    exact_setup_sizes(a, np, M, mp);
    std::vector<double> tab;
    exact_host_tables(M, a.K, tab);
    a.ctab = tab.data();
    a.rtab = tab.data() + exact_ctab_size(M, a.K);
    double f = 0.0;
    if (a.nin == 2) emu_exact_grid<EX_CHECKIF, 2>(a, f);
    else if (a.nin == 3) emu_exact_grid<EX_CHECKIF, 3>(a, f);
    else if (a.nin == 4) emu_exact_grid<EX_CHECKIF, 4>(a, f);
    else return 2;
    out[0] = f >= 1.0 ? 0.0 : 1.0;
    return 0;
  }
  if (op == EX_REAL) {   // 14 FFT_PAR_REAL: in1 = V (np, nb, M), out = (N, nb/2, np), N = 2mp-1
    std::vector<double> tab;
    for (int f = 0; f < nb / 2; ++f) {
      exact_setup_real(a, in1, f, nb, out, np, M, 2 * mp - 1);
      exact_setup_sizes(a, np, M, mp);
      if (f == 0) exact_host_tables(M, a.K, tab);
      a.ctab = tab.data();
      a.rtab = tab.data() + exact_ctab_size(M, a.K);
      double vmax = 0.0;
      emu_exact_grid<EX_REAL, 1>(a, vmax);
    }
    return 0;
  }
  if (const int rc = emu_exact_setup(a, cls_vmax, op, np, M, mp, in1, in2, values, n_values, eps, nb, out)) return rc;
  exact_setup_sizes(a, np, M, mp);
  std::vector<double> tab;
  exact_host_tables(M, a.K, tab);
  a.ctab = tab.data();
  a.rtab = tab.data() + exact_ctab_size(M, a.K);
  a.n_W = 2 * (int64_t)a.nout * (a.K + 1) * np;
  std::vector<double> W((size_t)a.n_W + 1);
  a.W = W.data();
  double vmax = 0.0;
  switch (op) {
    case EX_DIV: emu_exact_grid<EX_DIV, 2>(a, vmax); break;
    case EX_SV2: emu_exact_grid<EX_SV2, 4>(a, vmax); break;
    case EX_SQRT: emu_exact_grid<EX_SQRT, 1>(a, vmax); break;
    case EX_TENSION: emu_exact_grid<EX_TENSION, 6>(a, vmax); break;
    case EX_SVCLAMP: emu_exact_grid<EX_SVCLAMP, 4>(a, vmax); break;
    case EX_CLAMP01: emu_exact_grid<EX_CLAMP01, 1>(a, vmax); break;
    case EX_ENTRO: emu_exact_grid<EX_ENTRO, 4>(a, vmax); break;
    case EX_GRADMOM: emu_exact_grid<EX_GRADMOM, 9>(a, vmax); break;
    case EX_COMPR: emu_exact_grid<EX_COMPR, 7>(a, vmax); break;
    case EX_CLS: emu_exact_grid<EX_CLS, 4>(a, vmax); break;
    case EX_ETA: emu_exact_grid<EX_ETA, 1>(a, vmax); break;
    case EX_ETA3: emu_exact_grid<EX_ETA3, 3>(a, vmax); break;
    case EX_FROMREAL: emu_exact_grid<EX_FROMREAL, 1>(a, vmax); break;
    case EX_HEAVI:
      if (a.nin == 1) emu_exact_grid<EX_HEAVI, 1>(a, vmax);
      else if (a.nin == 2) emu_exact_grid<EX_HEAVI, 2>(a, vmax);
      else if (a.nin == 3) emu_exact_grid<EX_HEAVI, 3>(a, vmax);
      else if (a.nin == 4) emu_exact_grid<EX_HEAVI, 4>(a, vmax);
      else return 2;
      break;
    case EX_MAXVEL:
      if (a.nin == 3) emu_exact_grid<EX_MAXVEL, 3>(a, vmax);
      else emu_exact_grid<EX_MAXVEL, 1>(a, vmax);
      out[0] = vmax;
      return 0;
  }
  const int nmc = (M + EXACT_MC - 1) / EXACT_MC;
  for (int64_t p = 0; p < np; ++p)
    for (int g = 0; g < a.nout; ++g)
      for (int mc = 0; mc < nmc; ++mc) exact_r2c_body(a, p, g, mc);
  return 0;
}

// The same products on the matrix-core kernel (sfx_exact_mm_body.h).
template <int OP, int NIN, int MB>
static void emu_exact_mm_run(const ExactMmArgs& A) {
  constexpr int NI = exact_mm_nin(OP, NIN), NO = exact_mm_nout(OP);
  for (int y = 0; y < exact_mm_groups(OP); ++y)
    for (int z = 0; z < (NO > 0 ? (A.mbn + MB - 1) / MB : 1); ++z)
      run_grid((A.a.np + 15) / 16, 64 * exact_mm_waves(NI, NO), exact_mm_smem(NI) / 2,
               [&](int t, int64_t b, double2* sm) {
                 double* d = reinterpret_cast<double*>(sm);
                 constexpr int JB = exact_mm_jb(MB);   // as the GPU launcher
                 if (A.mbn == MB && A.jbn == JB) exact_mm_body<OP, NIN, MB, JB, true>(A, t, b, y, z, d);
                 else if (A.mbn == MB && A.jbn == JB - 1) exact_mm_body<OP, NIN, MB, JB - 1, true>(A, t, b, y, z, d);
                 else exact_mm_body<OP, NIN, MB, JB, false>(A, t, b, y, z, d);
               });
}
template <int OP, int NIN>
static int emu_exact_mm_m(const ExactMmArgs& A) {
  switch (exact_mm_mb(A.a.M)) {
    case 1: emu_exact_mm_run<OP, NIN, 1>(A); return 0;
    case 2: emu_exact_mm_run<OP, NIN, 2>(A); return 0;
    case 3: emu_exact_mm_run<OP, NIN, 3>(A); return 0;
    case 4: emu_exact_mm_run<OP, NIN, 4>(A); return 0;
    }
    return 2;
}
static int emu_exact_mm_op(int op, ExactArgs& a) {
  std::vector<double> tab, mm;
  exact_host_tables(a.M, a.K, tab);
  if (!exact_mm_sizes(a.M, a.K) || !exact_mm_disjoint(a)) return 4;
  exact_mm_host_tables(a.M, a.K, tab.data(), mm);
  ExactMmArgs A;
  A.a = a;
  A.mbn = exact_mm_mbn(a.M); A.jbn = exact_mm_jbn(a.K);
  A.n_ct = (int64_t)exact_mm_ctab_size(a.M, a.K); A.n_rt = (int64_t)exact_mm_rtab_size(a.M, a.K);
  A.ct = mm.data(); A.rt = mm.data() + A.n_ct;
  switch (op) {   // as launch_exact_mm
    case EX_DIV: return emu_exact_mm_m<EX_DIV, 2>(A);
    case EX_SV2: return emu_exact_mm_m<EX_SV2, 4>(A);
    case EX_SVCLAMP: return emu_exact_mm_m<EX_SVCLAMP, 4>(A);
    case EX_SQRT: return emu_exact_mm_m<EX_SQRT, 1>(A);
    case EX_CLAMP01: return emu_exact_mm_m<EX_CLAMP01, 1>(A);
    case EX_TENSION: return emu_exact_mm_m<MM_TENSROW, 4>(A);
    case EX_ENTRO: return emu_exact_mm_m<EX_ENTRO, 4>(A);
    case EX_GRADMOM: return emu_exact_mm_m<MM_SCALE3, 3>(A);
    case EX_COMPR: return emu_exact_mm_m<EX_COMPR, 7>(A);
    case EX_CLS: return emu_exact_mm_m<EX_CLS, 4>(A);
    case EX_ETA: return emu_exact_mm_m<EX_ETA, 1>(A);
    case EX_ETA3: return emu_exact_mm_m<EX_ETA3, 3>(A);
    case EX_FROMREAL: return emu_exact_mm_m<EX_FROMREAL, 0>(A);
    case EX_EVISCV: return emu_exact_mm_m<EX_EVISCV, 6>(A);
    case EX_HEAVI:
      return a.nin == 1 ? emu_exact_mm_m<EX_HEAVI, 1>(A) : a.nin == 2 ? emu_exact_mm_m<EX_HEAVI, 2>(A)
             : a.nin == 3 ? emu_exact_mm_m<EX_HEAVI, 3>(A) : emu_exact_mm_m<EX_HEAVI, 4>(A);
  }
  return 1;
}
extern "C" int emu_exact_mm(int op, int64_t np, int M, int mp, const double* in1, const double* in2,
                            const double* values, int n_values, double eps, int nb, double* out) {
  ExactArgs a;
  double cls_vmax = 0.0;
  std::vector<double> copy;
  if (op == EX_SQRT || op == EX_CLAMP01) {   // in place: the library passes a copy
    copy.assign(in1, in1 + np * nb * M);
    in1 = copy.data();
  }
  if (const int rc = emu_exact_setup(a, cls_vmax, op, np, M, mp, in1, in2, values, n_values, eps, nb, out)) return rc;
  exact_setup_sizes(a, np, M, mp);
  return emu_exact_mm_op(op, a);
}

// FFT_COMPUTE_ENTROPY_VISC_MOM: V = [V1 | V2 | V3] (3 x np*6*M), c (np,2,M),
// outputs (N, np); out2 may be null.  Both passes as the kernels run them.
extern "C" int emu_exact_emom(int64_t np, int M, int mp, int lg, const double* V, const double* c, const double* hloc,
                              double c2, double c4, double* out1, double* out2) {
  const int64_t n6 = np * 6 * M;
  ExactArgs a;
  exact_setup_emom(a, V, V + n6, V + 2 * n6, c, hloc, out1, out2, np, M, lg, c2, c4);
  exact_setup_sizes(a, np, M, mp);
  std::vector<double> tab;
  exact_host_tables(M, a.K, tab);
  a.ctab = tab.data();
  a.rtab = tab.data() + exact_ctab_size(M, a.K);
  const int N = 2 * a.K + 1;
  const int64_t me = np / lg, ne = me * N;
  std::vector<double> arr((size_t)3 * ne + 1, -1.0);
  a.nint = arr.data(); a.nint2 = a.nint + ne; a.nint3 = a.nint2 + ne; a.n_nint = ne;
  constexpr int NV = 2 * EXACT_EMOM_JC;
  const int nch = (a.K + 1 + EXACT_EMOM_JC - 1) / EXACT_EMOM_JC;
  double vmax = 0.0;
  std::vector<double> red((size_t)32 * lg * 3 * NV);
  for (int64_t eb = 0; eb < (me + 31) / 32; ++eb)
    for (int jc = 0; jc < nch; ++jc) {
      const int j0 = jc * EXACT_EMOM_JC;
      for (int t = 0; t < 32 * lg; ++t) {
        const int64_t p = eb * 32 * lg + t;
        double nv[NV] = {0}, nm[NV] = {0}, vr[NV] = {0};
        if (p < np) exact_emom_body(a, p, j0, nv, nm, vr);
        for (int v = 0; v < NV; ++v) {
          red[(size_t)t * 3 * NV + v] = nv[v];
          red[(size_t)t * 3 * NV + NV + v] = nm[v];
          red[(size_t)t * 3 * NV + 2 * NV + v] = vr[v];
          vmax = std::max(vmax, nv[v]);
        }
      }
      for (int le = 0; le < 32; ++le)
        for (int w = 0; w < 3 * NV; ++w) {
          const int64_t e = eb * 32 + le;
          const int k = w / NV, v = w % NV, j = j0 + v % EXACT_EMOM_JC;
          const bool mirror = v >= EXACT_EMOM_JC;
          if (e >= me || j > a.K || (mirror && j == 0)) continue;
          double x = red[(size_t)(le * lg) * 3 * NV + w];
          for (int l = 1; l < lg; ++l) x = std::max(x, red[(size_t)(le * lg + l) * 3 * NV + w]);
          double* dst = k == 0 ? a.nint : k == 1 ? a.nint2 : a.nint3;
          dst[e * N + (mirror ? N - j : j)] = x;
        }
    }
  for (int64_t i = 0; i < 3 * ne; ++i)
    if (arr[i] < 0) return 3;   // every (element, angle) written
  a.dmax = &vmax;
  for (int64_t p = 0; p < np; ++p)
    for (int j = 0; j < N; ++j) exact_emom_out_body(a, p, j);
  return 0;
}

// ---- inner product (dot_product_SF), Gauss values, column dot products
#include "../../sfemans_amd/csrc/sfx_inner_body.h"

static InnerArgs emu_inner_args(const int32_t* jj, const double* rr, int64_t me, int64_t np, const int32_t* lm,
                                int M, int nc, std::vector<double>& wgt, double* tab) {
  p2_reference_tables(tab);
  wgt.assign(7 * me + 1, 0.0);
  p2_assembly_weights(jj, rr, me, tab, wgt.data());
  InnerArgs a;
  std::memset(&a, 0, sizeof(a));
  a.jj = jj; a.tab = tab; a.wgt = wgt.data(); a.lmode = lm;
  a.nc = nc; a.ncols = nc * M; a.me = me; a.np = np; a.G = 7 * me;
  a.n_z = np * (int64_t)a.ncols;
  return a;
}

// dot_product_SF with the partial sums split over nblk work-groups (nblk >= 1).
extern "C" int emu_dotsf(const int32_t* jj, const double* rr, int64_t me, int64_t np, const int32_t* lm, int M,
                         int nc, const double* v, const double* w, int64_t nblk, double* out) {
  double tab[126];
  std::vector<double> wgt;
  InnerArgs a = emu_inner_args(jj, rr, me, np, lm, M, nc, wgt, tab);
  a.w0 = 1.0; a.wm = 0.5; a.v = v; a.w = w;
  const int64_t nitems = me > 0 && a.ncols > 0 ? elem_items(me, a.ncols) : 0;
  std::vector<double> part(nblk, 1e300);     // poisoned: a partial left unwritten shows up
  a.partial = part.data(); a.n_part = nblk;
  run_grid(nblk, INNER_THREADS, (INNER_THREADS + 1) / 2, [&](int t, int64_t b, double2* sm) {
    dotsf_block(a, b, nblk, nitems, t, reinterpret_cast<double*>(sm));
  });
  run_grid(1, INNER_THREADS, (INNER_THREADS + 1) / 2, [&](int t, int64_t, double2* sm) {
    sum_partials_block(part.data(), nblk, 2.0 * 3.14159265358979323846, out, t, reinterpret_cast<double*>(sm));
  });
  return 0;
}

// Gauss values of nodal columns z (np, nc*M) -> out (7*me, nc*M), scaled
// per column by w0 (mode 0) or wm, times rj*ray when weighted.
extern "C" int emu_gauss_values(const int32_t* jj, const double* rr, int64_t me, int64_t np, const int32_t* lm, int M,
                                int nc, int weighted, double w0, double wm, const double* z, double* out) {
  double tab[126];
  std::vector<double> wgt;
  InnerArgs a = emu_inner_args(jj, rr, me, np, lm, M, nc, wgt, tab);
  a.w0 = w0; a.wm = wm; a.weighted = weighted; a.z = z; a.out = out;
  a.n_out = a.G * (int64_t)a.ncols;
  const int64_t n = me > 0 && a.ncols > 0 ? elem_items(me, a.ncols) : 0;
  for (int64_t g = 0; g < n; ++g) gauss_values_body(a, g);
  return 0;
}

// out[c] = SUM_i A(i,c) B(i,c), one work-group per column.
extern "C" int emu_coldot(const double* A, const double* B, int64_t np, int ncols, double* out) {
  run_grid(ncols, INNER_THREADS, (INNER_THREADS + 1) / 2, [&](int t, int64_t c, double2* sm) {
    coldot_block(A, B, np, out, c, t, reinterpret_cast<double*>(sm));
  });
  return 0;
}

// Sanitizer self-check of the test harness (CPU only): which = 1 reads one
// element past a heap array, which = 2 overflows a signed int, 0 does
// neither.  Under the sanitizer build the first two must stop the process.
extern "C" int emu_sanitizer_probe(int which, int n) {
  std::vector<int> v(n > 0 ? n : 1, 1);
  volatile int s = v[0];
  if (which == 1) s = s + v.data()[v.size()];
  if (which == 2) {
    volatile int big = 2147483647 - 1;
    s = big + n;
  }
  return s;
}

// ---- fused nodal -> rhs_3x3 (gauss_body in its RHS form, then the gather):
// vb_145/vb_236 (np, 3, M) = scale * rhs_3x3((curl u + 2 Omega) x u)
template <int MP>
static void emu_nl_rhs_mp(const GaussArgs& a) {
  constexpr int NW = gauss_rhs_waves<MP, GV_CROSS_CURL>();
  constexpr int E = gauss_rhs_elems<MP>();
  const int64_t nblk = (a.me + E - 1) / E;
  run_grid(nblk, 64 * NW, GaussRhsCfg<MP, GV_CROSS_CURL>::LY::TOTAL,
           [&](int t, int64_t b, double2* s) { gauss_body<MP, GV_CROSS_CURL, NW, false, true, false, E>(a, t, b, s); });
}

extern "C" int emu_nl_rhs(const int32_t* jj, const double* rr, int64_t me, int64_t np, const double* U,
                          const int32_t* list_mode, int M, double* v145, double* v236, double scale, double om0,
                          double om1, double om2) {
  GaussArgs a;
  std::memset(&a, 0, sizeof(a));
  a.jj = jj; a.rr = rr; a.me = me; a.np = np; a.G = 7 * me;
  a.U = U; a.nU = np * 6 * (int64_t)M;
  a.list_mode = list_mode;
  double tab[126];
  p2_reference_tables(tab);
  a.tab = tab;
  std::vector<double> wgt(7 * me + 1);
  p2_assembly_weights(jj, rr, me, tab, wgt.data());
  std::vector<double> elo((size_t)36 * me * M + 1, 1e300);   // poisoned: every entry must be written
  a.wgt = wgt.data(); a.elo = elo.data(); a.nelo = 36 * me * (int64_t)M;
  a.M = M; a.MP = mp_for(M);
  a.om[0] = om0; a.om[1] = om1; a.om[2] = om2;
  std::vector<double2> wN, wMP;
  host_twiddles(a.MP, wN, wMP);
  a.wN = wN.data(); a.wMP = wMP.data();
  switch (a.MP) {
    case 4: emu_nl_rhs_mp<4>(a); break;
    case 8: emu_nl_rhs_mp<8>(a); break;
    case 16: emu_nl_rhs_mp<16>(a); break;
    case 32: emu_nl_rhs_mp<32>(a); break;
    case 64: emu_nl_rhs_mp<64>(a); break;
    case 128: emu_nl_rhs_mp<128>(a); break;
    case 256: emu_nl_rhs_mp<256>(a); break;
    default: return 1;
  }
  for (int64_t i = 0; i < a.nelo; ++i)
    if (elo[i] == 1e300) return 3;
  std::vector<int64_t> ptr;
  std::vector<int32_t> ent;
  build_adjacency(jj, me, np, ptr, ent);
  RhsArgs r;
  std::memset(&r, 0, sizeof(r));
  r.adj_ptr = ptr.data(); r.adj_ent = ent.data(); r.wgt = wgt.data(); r.tab = tab;
  r.jj = jj; r.me = me; r.np = np; r.G = 7 * me; r.M = M; r.scale = scale; r.n_adj = (int64_t)ent.size();
  r.v145 = v145; r.v236 = v236; r.elo = elo.data(); r.n_out = np * 3 * (int64_t)M; r.n_elo = a.nelo;
  run_grid((np + GATHER_NODES - 1) / GATHER_NODES, GATHER_THREADS, (gather_tile_doubles<6>() + 1) / 2,
           [&](int t, int64_t b, double2* sm) { rhs_gather_block(r, b, t, reinterpret_cast<double*>(sm)); });
  return 0;
}

// ---- fused u.grad c -> qs_00_gauss (gauss_body in its RHS form, then the gather):
// vect (np, 2, M) = scale * qs_00_gauss(hc, ff, (hc grad c).u + (div u)(hc c))
template <int MP>
static void emu_nl_qs00_mp(const GaussArgs& a) {
  constexpr int NW = gauss_rhs_waves<MP, GV_UGRADC>();
  constexpr int E = gauss_rhs_elems<MP>();
  const int64_t nblk = (a.me + E - 1) / E;
  run_grid(nblk, 64 * NW, GaussRhsCfg<MP, GV_UGRADC>::LY::TOTAL,
           [&](int t, int64_t b, double2* s) { gauss_body<MP, GV_UGRADC, NW, false, true, false, E>(a, t, b, s); });
}

extern "C" int emu_nl_qs00(const int32_t* jj, const double* rr, int64_t me, int64_t np, const double* U,
                           const double* c, const double* hc, const double* ff, const int32_t* list_mode, int M,
                           double* vect, double scale) {
  GaussArgs a;
  std::memset(&a, 0, sizeof(a));
  a.jj = jj; a.rr = rr; a.me = me; a.np = np; a.G = 7 * me;
  a.U = U; a.nU = np * 6 * (int64_t)M;
  a.U2 = c; a.nU2 = np * 2 * (int64_t)M;
  a.heat_capa = hc; a.ffn = ff; a.nffn = np * 2 * (int64_t)M;
  a.list_mode = list_mode;
  double tab[126];
  p2_reference_tables(tab);
  a.tab = tab;
  std::vector<double> wgt(7 * me + 1);
  p2_assembly_weights(jj, rr, me, tab, wgt.data());
  std::vector<double> elo((size_t)12 * me * M + 1, 1e300);   // poisoned: every entry must be written
  a.wgt = wgt.data(); a.elo = elo.data(); a.nelo = 12 * me * (int64_t)M;
  a.M = M; a.MP = mp_for(M);
  std::vector<double2> wN, wMP;
  host_twiddles(a.MP, wN, wMP);
  a.wN = wN.data(); a.wMP = wMP.data();
  switch (a.MP) {
    case 4: emu_nl_qs00_mp<4>(a); break;
    case 8: emu_nl_qs00_mp<8>(a); break;
    case 16: emu_nl_qs00_mp<16>(a); break;
    case 32: emu_nl_qs00_mp<32>(a); break;
    case 64: emu_nl_qs00_mp<64>(a); break;
    case 128: emu_nl_qs00_mp<128>(a); break;
    case 256: emu_nl_qs00_mp<256>(a); break;
    default: return 1;
  }
  for (int64_t i = 0; i < a.nelo; ++i)
    if (elo[i] == 1e300) return 3;
  std::vector<int64_t> ptr;
  std::vector<int32_t> ent;
  build_adjacency(jj, me, np, ptr, ent);
  RhsArgs r;
  std::memset(&r, 0, sizeof(r));
  r.adj_ptr = ptr.data(); r.adj_ent = ent.data(); r.wgt = wgt.data(); r.tab = tab;
  r.jj = jj; r.me = me; r.np = np; r.G = 7 * me; r.M = 2 * M; r.scale = scale; r.n_adj = (int64_t)ent.size();
  r.vect = vect; r.elo = elo.data(); r.n_out = np * 2 * (int64_t)M; r.n_elo = a.nelo;
  run_grid((np + GATHER_NODES - 1) / GATHER_NODES, GATHER_THREADS, (gather_tile_doubles<1>() + 1) / 2,
           [&](int t, int64_t b, double2* sm) { qs00_gather_block(r, b, t, reinterpret_cast<double*>(sm)); });
  return 0;
}
