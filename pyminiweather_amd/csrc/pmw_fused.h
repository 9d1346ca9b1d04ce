// pmw_fused.h -- launch interface of the fused-direction kernels (internal).
#pragma once

#include "pmw_common.h"

namespace pmw {

// Arguments of one fused direction (three RK stages) of one grid.
struct DirArgs {
  const gdouble* in;   // start state of the direction (interior read; RK init)
  gdouble* st;         // receives the stage-1 halo refresh (reference `state`)
  gdouble* out;        // result interior; must not alias `in`
  gdouble* tmp;        // stage-2 interior + stage-3 halo refresh (`state_tmp`)
  const gdouble* hy_cell;   // hy_dens_cell (x flux rows, z wall halos)
  const gdouble* hyt_cell;  // hy_dens_theta_cell (x flux rows)
  const gdouble* hyr_int;   // hy_dens_int (z faces)
  const gdouble* hyt_int;   // hy_dens_theta_int (z faces)
  const gdouble* hyp_int;   // hy_pressure_int (z faces)
  const gdouble* src_w;     // (nz, nx) w source or nullptr
  double id, idl;          // 1/dx or 1/dz as a sum (set_spacing)
  double dt1, dt2, dt3;    // dt/3, dt/2, dt
  double hv;               // -hv_beta * d / (16 * dt_full)
  const PMW_GLOBAL int* inj_rows = nullptr;  // the inflow boundary's row mask: x
                                             // is not periodic (launch_dir_x)
  gdouble* s1 = nullptr;   // optional: receives the stage-1 interior
  bool tmp_interior = true;  // false: tmp gets only its halo refresh (its
                             // interior is dead when the next direction of
                             // the same step rewrites every interior cell)
  long long mstride = 0;   // batched launches: elements between members of
                           // in / st / out / tmp / s1 (member = blockIdx.y)
};

inline void set_spacing(DirArgs& a, double d) {
  a.id = 1.0 / d;
  a.idl = recip_lo(d, a.id);
}

// The inflow boundary's fused x direction needs rows of at least this many
// cells (its copy of the row's right end must not reach the left one).
constexpr int kMinInflowCells = 16;

bool fused_x_tile_ok(int nt);
bool fused_z_seg_ok(int seg);
// `members` identical grids (same hydrostatic profiles and source) laid out
// a.mstride elements apart are advanced by one launch.
int launch_dir_x(const DirArgs& a, Grid g, int nt, hipStream_t st, int members = 1);
int launch_dir_z(const DirArgs& a, Grid g, int seg, hipStream_t st, int members = 1);

// ---- device helpers shared by the register-tile kernels
constexpr int kNumXcd = 8;

__device__ __forceinline__ int xcd_logical(int b, int per_xcd) {
  return (b % kNumXcd) * per_xcd + b / kNumXcd;
}

// Periodic column of cell c; the division only for the few lanes outside
// the row (the tile halos at the row ends).
__device__ __forceinline__ int wrap_cell(int c, int nx) {
  if (c >= 0 && c < nx) return c;
  int w = c % nx;
  return w < 0 ? w + nx : w;
}

// Phase order between the waves of a block by flags in LDS instead of block
// barriers, for tiles whose every phase reads and writes only a wave's own
// cells and the 2 cells on either side of them along the tile's line (in
// the one-cell z tiles a wave holds 8 whole rows of 8 columns): a wave waits
// for its two neighbours alone, so one late wave no longer holds up the
// whole block. wf[1 + w] = the last phase wave w finished; wf[0] and
// wf[NW + 1] stay above every phase. Every wave passes every phase in order,
// so the wave with the lowest phase never waits and the block cannot stall.
// The flags are set before the block's first barrier, which publishes them.
__device__ __forceinline__ void wave_flags_init(int* wf, int nw, int t) {
  if (t < nw + 2)
    __hip_atomic_store(&wf[t], (t == 0 || t == nw + 1) ? 1 << 20 : 0, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Phase P (> 0, increasing) of the calling wave is done; returns once both
// neighbouring waves have done it too.
__device__ __forceinline__ void wave_phase_done(int* wf, int P, int t) {
  const int wv = t >> 6;
  __builtin_amdgcn_sched_barrier(0);
  // this wave's LDS writes of phase P are complete before its flag says so
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if ((t & 63) == 0)
    __hip_atomic_store(&wf[1 + wv], P, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  while (true) {
    const int lo = __hip_atomic_load(&wf[wv], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    const int hi = __hip_atomic_load(&wf[2 + wv], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (lo >= P && hi >= P) break;
    __builtin_amdgcn_s_sleep(1);
  }
  // the neighbours' LDS writes are read after their flags
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double x) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo =
      (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, CTRL, 0xf, 0xf, true);
  const unsigned hi =
      (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
// x of lane - 1 / lane + 1 (0 at the wave's end: a state at rest)
__device__ __forceinline__ double from_prev(double x) { return dpp_f64<0x138>(x); }
__device__ __forceinline__ double from_next(double x) { return dpp_f64<0x130>(x); }

// Two consecutive cells of a row: rows start at any multiple of 8 bytes (odd
// nx), which a 16-byte global access takes.
typedef double dpair __attribute__((ext_vector_type(2), aligned(8)));

}  // namespace pmw
