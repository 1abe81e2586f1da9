// Kernels of the exact-grid products on the matrix cores (sfx_exact_mm_body.h).
#include "sfx_engine.h"
#include "sfx_exact_mm_body.h"
#include "sfx_kernels.h"

namespace sfx {

// Two waves per SIMD (256 registers, and no accumulation registers whose
// copies would cost more than the products), three where the accumulators of
// at most 16 modes leave room.
template <int OP, int NIN, int MB, int JB, bool ONE>
__global__ void __launch_bounds__(64 * exact_mm_waves(exact_mm_nin(OP, NIN), exact_mm_nout(OP)))
__attribute__((amdgpu_waves_per_eu(MB == 1 ? 3 : 2, MB == 1 ? 3 : 2))) exact_mm_kernel(ExactMmArgs A) {
  extern __shared__ double mm_smem[];
  // the groups of one tile are neighbours: they read the same real-space inputs
  constexpr int NG = exact_mm_groups(OP);
  const int64_t L = xcd_block(blockIdx.x, gridDim.x);
  exact_mm_body<OP, NIN, MB, JB, ONE>(A, threadIdx.x, L / NG, (int)(L % NG), blockIdx.y, mm_smem);
}

template <int OP, int NIN, int MB>
static hipError_t mm_launch(const ExactMmArgs& A, hipStream_t st) {
  constexpr int NI = exact_mm_nin(OP, NIN), NO = exact_mm_nout(OP);
  const int64_t tiles = (A.a.np + 15) / 16;
  const int64_t nblk = tiles * exact_mm_groups(OP);
  if (nblk > 0x7fffffffLL) return hipErrorInvalidValue;
  const dim3 grid((unsigned)nblk, NO > 0 ? (A.mbn + MB - 1) / MB : 1), wg(64 * exact_mm_waves(NI, NO));
  const size_t shmem = exact_mm_smem(NI) * sizeof(double);
  constexpr int JB = exact_mm_jb(MB);
  if (A.mbn == MB && A.jbn == JB)
    hipLaunchKernelGGL((exact_mm_kernel<OP, NIN, MB, JB, true>), grid, wg, shmem, st, A);
  else if (A.mbn == MB && A.jbn == JB - 1)
    hipLaunchKernelGGL((exact_mm_kernel<OP, NIN, MB, JB - 1, true>), grid, wg, shmem, st, A);
  else
    hipLaunchKernelGGL((exact_mm_kernel<OP, NIN, MB, JB, false>), grid, wg, shmem, st, A);
  return hipGetLastError();
}

template <int OP, int NIN>
static hipError_t mm_launch_m(const ExactMmArgs& A, hipStream_t st) {
  if (A.a.np <= 0) return hipSuccess;
  switch (exact_mm_mb(A.a.M)) {
    case 1: return mm_launch<OP, NIN, 1>(A, st);
    case 2: return mm_launch<OP, NIN, 2>(A, st);
    case 3: return mm_launch<OP, NIN, 3>(A, st);
    case 4: return mm_launch<OP, NIN, 4>(A, st);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_exact_mm(int op, const ExactArgs& a, hipStream_t st) {
  ExactMmArgs A;
  A.a = a;
  A.mbn = exact_mm_mbn(a.M);
  A.jbn = exact_mm_jbn(a.K);
  A.ct = a.mmtab;
  A.n_ct = (int64_t)exact_mm_ctab_size(a.M, a.K);
  A.rt = a.mmtab + A.n_ct;
  A.n_rt = (int64_t)exact_mm_rtab_size(a.M, a.K);
  switch (op) {
    case EX_DIV: return mm_launch_m<EX_DIV, 2>(A, st);
    case EX_SV2: return mm_launch_m<EX_SV2, 4>(A, st);
    case EX_SVCLAMP: return mm_launch_m<EX_SVCLAMP, 4>(A, st);
    case EX_SQRT: return mm_launch_m<EX_SQRT, 1>(A, st);
    case EX_CLAMP01: return mm_launch_m<EX_CLAMP01, 1>(A, st);
    case EX_TENSION: return mm_launch_m<MM_TENSROW, 4>(A, st);
    case EX_ENTRO: return mm_launch_m<EX_ENTRO, 4>(A, st);
    case EX_GRADMOM: return mm_launch_m<MM_SCALE3, 3>(A, st);
    case EX_COMPR: return mm_launch_m<EX_COMPR, 7>(A, st);
    case EX_CLS: return mm_launch_m<EX_CLS, 4>(A, st);
    case EX_ETA: return mm_launch_m<EX_ETA, 1>(A, st);
    case EX_ETA3: return mm_launch_m<EX_ETA3, 3>(A, st);
    case EX_FROMREAL: return mm_launch_m<EX_FROMREAL, 0>(A, st);
    case EX_EVISCV: return mm_launch_m<EX_EVISCV, 6>(A, st);
    case EX_HEAVI:
      switch (a.nin) {
        case 1: return mm_launch_m<EX_HEAVI, 1>(A, st);
        case 2: return mm_launch_m<EX_HEAVI, 2>(A, st);
        case 3: return mm_launch_m<EX_HEAVI, 3>(A, st);
        case 4: return mm_launch_m<EX_HEAVI, 4>(A, st);
      }
  }
  return hipErrorInvalidValue;
}

}  // namespace sfx
