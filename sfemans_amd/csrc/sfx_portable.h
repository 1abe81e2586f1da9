// Portability layer: the kernel bodies compile for gfx950 (hipcc) and, with
// SFX_EMULATE defined, for the host CPU, where tests run one work-group as
// std::threads with a barrier in place of __syncthreads and check every
// global and LDS index against its buffer.
#pragma once
#include <stdint.h>

#ifdef SFX_EMULATE
#include <cmath>
#include <cstdio>
#include <cstdlib>
struct double2 { double x, y; };
inline double2 make_double2(double x, double y) { return double2{x, y}; }
using std::fma;
#define SFX_DEV inline
#define SFX_DEV_NOINLINE inline
#define __restrict__
void sfx_emu_sync();
void sfx_emu_wave_sync();
[[noreturn]] void sfx_emu_oob(const char* what, long long idx, long long n, const char* file, int line);
#define SFX_SYNC() sfx_emu_sync()
struct sfx_d4 {
  double v[4];
  double& operator[](int i) { return v[i]; }
  const double& operator[](int i) const { return v[i]; }
};
sfx_d4 sfx_emu_mfma_f64(double a, double b, const sfx_d4& c);
#define SFX_MFMA_F64(a, b, c) sfx_emu_mfma_f64((a), (b), (c))
#define SFX_UNIFORM(x) (x)
void sfx_emu_lane_swap(double& a, double& b, int bit);
#define SFX_LANE_SWAP(a, b, bit) sfx_emu_lane_swap((a), (b), (bit))
#define SFX_WAVE_SYNC() sfx_emu_wave_sync()
#define SFX_OPAQUE(x) do { } while (0)
#define SFX_OPAQUE_S(x) do { } while (0)
#define SFX_KARG
#define SFX_SCHED_BARRIER() do { } while (0)
#define SFX_CHECK(what, idx, n) \
  do { if ((long long)(idx) < 0 || (long long)(idx) >= (long long)(n)) sfx_emu_oob(what, (long long)(idx), (long long)(n), __FILE__, __LINE__); } while (0)
#else
#include <hip/hip_runtime.h>
#define SFX_DEV __device__ __forceinline__
// a device function compiled on its own (own register allocation and stack frame)
#define SFX_DEV_NOINLINE __device__ __noinline__
#define SFX_SYNC() __syncthreads()
// Exchange inside one wave through its private LDS region: a wave's LDS
// instructions execute in order, so only compiler reordering must be stopped.
#define SFX_WAVE_SYNC()                                   \
  do {                                                    \
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); \
    __builtin_amdgcn_wave_barrier();                      \
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront"); \
  } while (0)
#define SFX_CHECK(what, idx, n) do { } while (0)
// c + a b on the matrix core: a 16x4 (lane l holds row l % 16, column l / 16),
// b 4x16 (row l / 16, column l % 16), c 16x16 (element v of lane l: row l / 16
// + 4 v, column l % 16).
typedef double sfx_d4 __attribute__((ext_vector_type(4)));
#define SFX_MFMA_F64(a, b, c) __builtin_amdgcn_mfma_f64_16x16x4f64((a), (b), (c), 0, 0, 0)
// An int that is the same in every lane of the wave, as a scalar.
#define SFX_UNIFORM(x) __builtin_amdgcn_readfirstlane(x)
// Transpose the pair (a, b) with a lane bit (32, 16, 8 or 4): lanes whose bit is
// 0 keep a and get the a of lane + BIT in b; lanes whose bit is 1 keep b and get
// the b of lane - BIT in a.
template <int BIT>
__device__ __forceinline__ void sfx_lane_swap(double& a, double& b) {
  union { double d; unsigned u[2]; } x, y;
  x.d = a;
  y.d = b;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if constexpr (BIT == 32) {
      const auto r = __builtin_amdgcn_permlane32_swap(x.u[i], y.u[i], false, false);
      x.u[i] = r[0];
      y.u[i] = r[1];
    } else if constexpr (BIT == 16) {
      const auto r = __builtin_amdgcn_permlane16_swap(x.u[i], y.u[i], false, false);
      x.u[i] = r[0];
      y.u[i] = r[1];
    } else {
      // DPP row_shr / row_shl by BIT, written to the banks of 4 lanes whose bit is 1 / 0
      constexpr int HI = BIT == 8 ? 0xc : 0xa, LO = BIT == 8 ? 0x3 : 0x5;
      const unsigned p = x.u[i], q = y.u[i];
      x.u[i] = __builtin_amdgcn_update_dpp(p, q, 0x110 + BIT, 0xf, HI, false);
      y.u[i] = __builtin_amdgcn_update_dpp(q, p, 0x100 + BIT, 0xf, LO, false);
    }
  }
  a = x.d;
  b = y.d;
}
#define SFX_LANE_SWAP(a, b, bit) sfx_lane_swap<bit>((a), (b))
// Hide a value's origin from the optimizer, so that what is computed from it
// is recomputed where it is used instead of being kept live (or spilled)
// across a long stretch of code.  Emits no instruction.
#define SFX_OPAQUE(x) __asm__ volatile("" : "+v"(x))
// The same for a wave-uniform value kept in scalar registers (a pointer
// read through redefined at this point: loads through it are not hoisted
// above it).
#define SFX_OPAQUE_S(x) __asm__ volatile("" : "+s"(x))
// Address space of the kernel arguments: uniform loads from it are scalar loads.
#define SFX_KARG __attribute__((address_space(4)))
// Keep the instruction scheduler from moving code across this point (for
// example loads hoisted above it, whose destinations would be live early).
#define SFX_SCHED_BARRIER() __builtin_amdgcn_sched_barrier(0)
#endif
