// pmw_fused.hip -- one launch per direction: the three RK stages of one
// dimensional-splitting direction fused into a single kernel (gfx950).
//
// For one direction the reference runs (solve/step.py:111-141)
//   S1 = S + dt/3 T(S),  S2 = S + dt/2 T(S1),  S3 = S + dt T(S2)
// with a halo refresh of each forcing state. Each stage widens the stencil
// by 2 cells, so an output tile needs S on the tile +- 6 cells: stage 1 is
// computed on tile +- 4, stage 2 on tile +- 2, stage 3 on the tile. Per
// interior cell and direction this reads S once and writes the result (and,
// in the last direction of a call, the stage-2 state, state_tmp): 64 or 96 B
// instead of the 256 B of three stage launches. Every stage value is computed
// with the same operations as the per-stage kernels, so results are bitwise
// identical to them.
//
// Buffers of a direction: `in` (its start state, read only), `out` (its
// result interior, never aliases `in`), `st` (the reference's `state`: it
// receives the halo refresh of stage 1, computed from `in`) and `tmp` (the
// reference's `state_tmp`: stage-2 interior plus the stage-3 halo refresh).
//
//  * x (k_dir_x<NS>): independent waves over the rows laid end to end, K cells
//    per lane in registers, neighbours by one-lane shifts; the periodic cells
//    are part of the extended rows.
//  * z: k_dir_zt1<NW,NR>, LDS tiles with three rows per thread in registers,
//    for large grids; k_dir_zw and k_dir_zs, columns as waves, for small ones;
//    k_dir_z1<NR>, LDS tiles with one cell per thread, between them, and
//    k_dir_z1d<NR>, the same over the column groups laid end to end. The wall
//    halo rows of every stage state are rebuilt from its edge row.
//  * k_ens_*: the same over the flattened tile list of an ensemble.
// Block ids are remapped so that each XCD runs a contiguous range of tiles.
#include <algorithm>
#include <mutex>
#include <new>
#include <unordered_map>

#include "pmw_common.h"
#include "pmw_fused.h"

using namespace pmw;

namespace {

// ------------------------------------------------------------------ x ------
// The extended rows of a grid (cells -6 .. nx+5, the periodic cells the three
// stages consume included) are laid end to end, E slots each (a multiple of K),
// and cut into waves of W = 64 K slots every W - 12: a lane holds K cells of
// one row in registers and runs the three stages on them. A row boundary
// inside a wave costs no more than the wave boundary does. A slot holds a
// correct stage-s value when it lies 2s slots inside its wave and inside its
// own extended row (-6+2s <= cell <= nx+5-2s); values computed across a row
// boundary are never written. The windows [6, W-6) partition the slots, so
// every interior cell is written by one wave; halo cells are written wherever
// they are correct (the same value). Of its neighbours a lane needs, per
// stage, two cells before its run, one after it and the flux behind its last
// cell: 16 doubles, shifted by one lane (DPP), no LDS traffic and no barrier.
// The RK init S waits in the lane's own LDS slots (written once, read in
// stages 2 and 3, no other lane looks at it), which frees 8 K registers: with
// K = 2, 96 VGPRs instead of 114 and 5 waves per SIMD instead of 4.
//
// Against LDS tiles of one cell per thread (48 KB and 6 barriers per 512
// cells; 108 doubles of LDS traffic per cell and direction, here 12) the waves
// are bound by FP64 issue in the steady state, with the start and the tail of
// the launch on top (2.5 of 5 waves per SIMD on average). Per launch between
// events, 512-thread LDS tiles / these waves / with the reciprocal pairs of
// recip() and tend_of() / with one table entry per power / tested once per wave:
// 2000 x 1000 52.3 / 42.5 / 38.7 / 37.8 / 37.0 us, 8192 x 4096 740 / 599 / 551 /
// 526 / 497 us (4.3 TB/s of reads and writes; a 4 GB copy reaches 4.6). The cheaper power alone took the tiles
// from 51 to 47 us, and they stayed at 42 with the power left out of a timing
// copy altogether.
constexpr int kXwWaves = 4;  // waves per block (they share nothing)

template <int K>
struct XWaveLds {
  double s[kXwWaves][K * kNv][64];
};

__host__ __device__ inline unsigned xw_row_slots(int nx, int K) { return (unsigned)(nx + 12 + K - 1) / K * K; }
inline long long xw_slots(int nx, int nz, int K) { return (long long)xw_row_slots(nx, K) * nz; }
inline int xw_blocks(int nx, int nz, int K, bool inflow = false) {
  const long long waves = (xw_slots(nx, nz, K) - 13) / (64 * K - (inflow ? 16 : 12)) + 1;
  return (int)((waves + kXwWaves - 1) / kXwWaves);
}

// With the injection inflow (INFLOW, ics/bcs.py:37-64) x is not periodic: the
// right halo is what the forcing buffer holds (state's in stage 1, state_tmp's
// in stages 2 and 3; nothing writes it), and the left halo is the right end's
// cells nx-2, nx-1 of each stage's state, with rho*u and (rho*theta)' set on
// the inflow rows. A row's E slots are then: its cells nx-6 .. nx-1 once more
// and the right halo (0-7: enough for nx-2, nx-1 to be right after two
// stages), the left halo (8, 9), cells 0 .. nx-1, the right halo. The halo
// slots are refreshed at the start of every stage, the left ones from 4 slots
// before. Cell 0 depends on 10 slots before it: windows [10, W-6). A step at
// 1003 x 517 took 36 us (33 now), 66 with one launch per RK stage and the copies
// of the right halo between them (60 launches and 20 copies per 10 steps became
// 20 launches).
//
// Wave `b` of rows rbase .. rbase+nrows-1; E = xw_row_slots(nx, K).
// ANY: the power of any argument; otherwise the table's alone, and the lanes that
// asked for another are returned.
template <int K, bool INFLOW, bool ANY>
__device__ __forceinline__ unsigned long long dir_x_run(const DirArgs& a, const Grid& g, int t,
                                                        unsigned b, unsigned E, int rbase,
                                                        int nrows, double (*init)[64]) {
  constexpr int W = 64 * K, LM = INFLOW ? 10 : 6, C = W - LM - 6;  // windows [LM, W-6)
  const int nx = g.nx, lane = t & 63;
  const unsigned slot0 = b * (unsigned)C;
  const unsigned row0 = __builtin_amdgcn_readfirstlane(slot0 / E);
  if ((int)row0 >= nrows) return 0;  // the last block's spare waves
  unsigned long long rare = 0;
  const unsigned rem = slot0 - row0 * E + (unsigned)(K * lane);
  const unsigned dr0 = rem / E;
  const int cell0 = (int)(rem - dr0 * E) - LM;
  const bool row_ok = (int)(row0 + dr0) < nrows;  // else: past the last row, not written
  const unsigned dr = row_ok ? dr0 : (unsigned)nrows - 1 - row0;
  const int prow = rbase + (int)(row0 + dr) + kHs;
  const long long rowoff = (long long)(rbase + (int)row0 + kHs) * g.ld;  // wave-uniform
  const unsigned lrow = dr * (unsigned)g.ld + kHs;                       // the lane's row
  const unsigned lo = (lrow + (unsigned)cell0) * 8u;
  const bool inner = cell0 >= 0 && cell0 + K <= nx;  // no halo or padding cell
  // every load of the wave is issued before the first is waited for (one memory
  // latency instead of two or three: 0.4 us of a launch on a small grid)
  const double hyr = a.hy_cell[prow], hyt = a.hyt_cell[prow];
  double s[K][4];
  if (inner) {
#pragma unroll
    for (int v = 0; v < kNv; ++v) {
      const PMW_GLOBAL char* p =
          (const PMW_GLOBAL char*)sgpr64((unsigned long long)(a.in + v * g.plane + rowoff)) + lo;
      if constexpr (K == 2) {
        const dpair q = *(const PMW_GLOBAL dpair*)p;
        s[0][v] = q.x;
        s[K - 1][v] = q.y;
      } else {
        s[0][v] = *(const gdouble*)p;
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const int c = cell0 + i;
      // inflow: slots 0-5 hold cells nx-6 .. nx-1; halo slots are refreshed
      const int cs = !INFLOW ? wrap_cell(c, nx) : c < -4 ? nx + 4 + c : min(max(c, 0), nx - 1);
      const unsigned bw = (lrow + (unsigned)cs) * 8u;
#pragma unroll
      for (int v = 0; v < kNv; ++v) s[i][v] = ld_off(a.in + v * g.plane + rowoff, bw);
    }
  }
#pragma unroll
  for (int i = 0; i < K; ++i)
#pragma unroll
    for (int v = 0; v < kNv; ++v) init[i * kNv + v][lane] = s[i][v];
  asm volatile("" ::: "memory");  // read back from LDS, not kept in registers
  if (!INFLOW && !inner && row_ok) {  // set_bc_x of stage 1
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const int c = cell0 + i;
      if (c == -2 || c == -1 || c == nx || c == nx + 1) {
#pragma unroll
        for (int v = 0; v < kNv; ++v) st_off(a.st + v * g.plane + rowoff, lo + 8u * i, s[i][v]);
      }
    }
  }
  const bool whole = inner && row_ok && K * lane >= LM && K * lane + K <= W - 6;
  const bool row_start =
      INFLOW && __builtin_amdgcn_ballot_w64(cell0 <= -1 && cell0 + K > -2) != 0;
#pragma unroll
  for (int stage = 0; stage < 3; ++stage) {
    const double dts = stage == 0 ? a.dt1 : stage == 1 ? a.dt2 : a.dt3;
    if constexpr (INFLOW) {
      gdouble* const halo = stage == 0 ? a.st : a.tmp;
      if (row_start) {  // wave-uniform: the left halo from 4 slots before
#pragma unroll
        for (int i = 0; i < K; ++i) {
          const int c = cell0 + i, sl = K * lane + i;
          double q[4];
#pragma unroll
          for (int v = 0; v < kNv; ++v) {
            q[v] = from_prev(from_prev(s[i][v]));
            if (K == 1) q[v] = from_prev(from_prev(q[v]));
          }
          if (c == -2 || c == -1) {
            if (a.inj_rows[prow - kHs]) {
              const double r = q[0] + hyr;
              q[1] = r * 50.0;
              q[3] = r * 298.0 - hyt;
            }
            // stored where the row's slots 0 .. 9 lie in this wave
            const bool put = stage != 1 && row_ok && sl >= c + LM;
#pragma unroll
            for (int v = 0; v < kNv; ++v) {
              s[i][v] = q[v];
              if (put) st_off(halo + v * g.plane + rowoff, lo + 8u * i, q[v]);
            }
          }
        }
      }
      if (!inner) {
#pragma unroll
        for (int i = 0; i < K; ++i) {
          const int c = cell0 + i, h = c < 0 ? c + 4 : c - nx;  // right halo 0, 1
          if (h == 0 || h == 1) {
#pragma unroll
            for (int v = 0; v < kNv; ++v)
              s[i][v] = ld_off(halo + v * g.plane + rowoff, (lrow + (unsigned)(nx + h)) * 8u);
          }
        }
      }
    }
    double b2[4], b1[4], nx1[4];  // cells -2, -1 and K of the lane's run
#pragma unroll
    for (int v = 0; v < kNv; ++v) {
      b1[v] = from_prev(s[K - 1][v]);
      b2[v] = K == 1 ? from_prev(b1[v]) : from_prev(s[0][v]);
      nx1[v] = from_next(s[0][v]);
    }
    auto update = [&](int i, const double cell[4], const double flo[4], const double fhi[4]) {
      double td[4];
#pragma unroll
      for (int v = 0; v < kNv; ++v) td[v] = tend_of(flo[v], fhi[v], a.id, a.idl);
      if (a.src_w)
        td[2] = td[2] + a.src_w[(long long)(prow - kHs) * nx + wrap_cell(cell0 + i, nx)];
#pragma unroll
      for (int v = 0; v < kNv; ++v)
        s[i][v] = (stage == 0 ? cell[v] : init[i * kNv + v][lane]) + dts * td[v];
    };
    double F0[4], Fp[4];
#pragma unroll
    for (int j = 0; j < K; ++j) {  // face j, between cells j-1 and j; then cell j-1
      double v4[4], d3[4], F[4], cur[4];
#pragma unroll
      for (int v = 0; v < kNv; ++v) {
        cur[v] = s[j][v];
        recon4(b2[v], b1[v], cur[v], j + 1 < K ? s[K - 1][v] : nx1[v], v4[v], d3[v]);
      }
      if constexpr (ANY)
        flux_x_face<false>(v4, d3, hyr, hyt, a.hv, F, PowGamma{});
      else
        flux_x_face<false>(v4, d3, hyr, hyt, a.hv, F, PowGammaIn{rare});
      if (j == 0) {
#pragma unroll
        for (int v = 0; v < kNv; ++v) F0[v] = F[v];
      } else {
        update(j - 1, b1, Fp, F);
      }
#pragma unroll
      for (int v = 0; v < kNv; ++v) {
        b2[v] = b1[v];
        b1[v] = cur[v];
        Fp[v] = F[v];
      }
      __builtin_amdgcn_sched_barrier(0);  // one face's values live at a time
    }
    double Fn[4];
#pragma unroll
    for (int v = 0; v < kNv; ++v) Fn[v] = from_next(F0[v]);
    update(K - 1, b1, Fp, Fn);
    gdouble* dst = stage == 0 ? a.s1 : stage == 1 ? (a.tmp_interior ? a.tmp : nullptr) : a.out;
    if (dst) {
      if (whole) {
#pragma unroll
        for (int v = 0; v < kNv; ++v) {
          PMW_GLOBAL char* p =
              (PMW_GLOBAL char*)sgpr64((unsigned long long)(dst + v * g.plane + rowoff)) + lo;
          if constexpr (K == 2)
            *(PMW_GLOBAL dpair*)p = dpair{s[0][v], s[K - 1][v]};
          else
            *(gdouble*)p = s[0][v];
        }
      } else if (row_ok) {
#pragma unroll
        for (int i = 0; i < K; ++i) {
          const int c = cell0 + i, sl = K * lane + i;
          if (sl >= LM && sl < W - 6 && c >= 0 && c < nx) {
#pragma unroll
            for (int v = 0; v < kNv; ++v)
              st_off(dst + v * g.plane + rowoff, lo + 8u * i, s[i][v]);
          }
        }
      }
    }
    if (!INFLOW && stage == 1 && !inner && row_ok) {  // set_bc_x of stage 3 into tmp
#pragma unroll
      for (int i = 0; i < K; ++i) {
        const int c = cell0 + i, sl = K * lane + i;
        if (sl >= 4 && sl < W - 4 && (c == -2 || c == -1 || c == nx || c == nx + 1)) {
#pragma unroll
          for (int v = 0; v < kNv; ++v)
            st_off(a.tmp + v * g.plane + rowoff, lo + 8u * i, s[i][v]);
        }
      }
    }
  }
  return rare;
}

// If any argument of the wave lay outside the table: once more, with the power
// of any argument. Nothing that the wave reads has been written since (a
// launch's waves write each their own cells, and halo cells with the values they
// have).
template <int K, bool INFLOW>
__device__ __forceinline__ void dir_x_wave(const DirArgs& a, const Grid& g, unsigned b,
                                           unsigned E, int rbase, int nrows,
                                           double (*init)[64]) {
  int t = (int)threadIdx.x;
  if (__builtin_expect(dir_x_run<K, INFLOW, false>(a, g, t, b, E, rbase, nrows, init) != 0, 0)) {
    asm volatile("" : "+v"(t));  // nothing of the first run is kept for this one
    dir_x_run<K, INFLOW, true>(a, g, t, b, E, rbase, nrows, init);
  }
}

// Member blockIdx.y of a batched launch: offset every per-member buffer.
__device__ __forceinline__ void member_offset(DirArgs& a) {
  const long long off = (long long)blockIdx.y * a.mstride;
  a.in += off;
  a.st += off;
  a.out += off;
  a.tmp += off;
  if (a.s1) a.s1 += off;
}

// Registers: K = 1 fits 6 waves per SIMD (74 VGPRs), K = 2 five (94; 96 with the
// inflow, which spills one).
constexpr int xw_waves_per_simd(int K) { return K == 1 ? 6 : 5; }

__device__ __forceinline__ unsigned xw_wave(int block) {
  return __builtin_amdgcn_readfirstlane((unsigned)block * kXwWaves + (threadIdx.x >> 6));
}

// NS = slots per block: 256 (K = 1) or 512 (K = 2). A launch covers `rows`
// rows per blockIdx.z (all of them, unless the slots would not fit 32 bits).
template <int NS>
__global__ __launch_bounds__(64 * kXwWaves)
    __attribute__((amdgpu_waves_per_eu(xw_waves_per_simd(NS / 256)))) void k_dir_x(
        DirArgs a, Grid g, unsigned E, int rows, int nreal, int per_xcd) {
  constexpr int K = NS / 256;
  __shared__ XWaveLds<K> sm;
  const int logical = xcd_logical(blockIdx.x, per_xcd);
  if (logical >= nreal) return;
  member_offset(a);
  const int rbase = (int)blockIdx.z * rows;
  dir_x_wave<K, false>(a, g, xw_wave(logical), E, rbase, min(rows, g.nz - rbase),
                       sm.s[threadIdx.x >> 6]);
}

// the same with the injection inflow
template <int NS>
__global__ __launch_bounds__(64 * kXwWaves)
    __attribute__((amdgpu_waves_per_eu(xw_waves_per_simd(NS / 256)))) void k_dir_xi(
        DirArgs a, Grid g, unsigned E, int rows, int nreal, int per_xcd) {
  constexpr int K = NS / 256;
  __shared__ XWaveLds<K> sm;
  const int logical = xcd_logical(blockIdx.x, per_xcd);
  if (logical >= nreal) return;
  member_offset(a);
  const int rbase = (int)blockIdx.z * rows;
  dir_x_wave<K, true>(a, g, xw_wave(logical), E, rbase, min(rows, g.nz - rbase),
                      sm.s[threadIdx.x >> 6]);
}

// ------------------------------------------------------------------ z ------
// z tiles, three rows per thread (k_dir_zt1): a block of NW waves holds 16
// columns x NR rows (slot row r of column c in thread (r/3)*16 + c), the
// running stage state and S in registers; LDS only carries what threads of
// neighbouring rows need of each other: the first and the last two rows of
// each thread's three and the flux at its first face (14 doubles of LDS
// traffic per cell and stage instead of the 33 of one cell per thread), and
// the rows' face hydrostatics. A wave holds 12 whole rows, and every phase
// reads and writes only the wave's rows and those of its neighbours, so the
// phases are ordered by the waves' flags (wave_phase_done).
//
// Rows of the tiles: the first holds rows -2 .. NR-3 of the column, the last
// rows nz+2-NR .. nz+1 (nz >= NR - 2), so that a wall's halo rows share a thread with their
// edge row and set_bc_z between the stages stays in one thread's registers;
// the tiles between start 6 rows before the first row they own. Next to a wall nothing is lost to the
// stencil, so the first and last own NR - 8 rows, the others NR - 12. Tiles
// overlap where nz does not divide; each row has one owner. Tiles of one row
// of blocks are neighbours along x (their 128-byte rows straddle cache lines,
// which then meet in one XCD's L2).
//
// Measured (between events, one cell per thread with the RK init in registers
// / this / with the reciprocal pairs / with one table entry per power / its range
// tested once per stage): 2000 x 1000 63.2 / 55 / 50 / 49.2 / 47.6 us, 8192 x 4096
// 980 / 867 / 786 / 769 / 738 us. (Tested once per tile, with a block barrier and
// the whole tile run again: no faster than once per face.) Three rows per thread
// fit 128 VGPRs (4 waves per SIMD, two 66 KB blocks per CU). Same
// boxes, not kept, against 55 and 867 us: 8 columns x 96 rows in 256 threads 58
// and 1200 us (64-byte rows), 4 rows per thread (x 24 row groups) 73 and 1190
// us, 6 rows (2 waves per SIMD) 53 and 874 us, 2 columns per wave without LDS
// 127 and 2740 us; block barriers instead of the flags 50.4 and 801 us against
// 50.0 and 786; two rows per thread, 64 to 128 rows, 4 to 6 waves per SIMD 64 to
// 99 us against 48.9 (spills, and twice the LDS traffic per row).
template <int NW, int NR>
struct ZTileLds {
  static constexpr int NT = 64 * NW;
  double hz[3][NR];    // rho, rho*theta, p at the rows' lower faces
  int wf[NW + 2];      // wave phase flags
  // the large arrays last: every slot within the 64 KB of an offset field
  double lo[kNv][NT];  // each thread's first row,
  double h1[kNv][NT];  // its last row
  double h2[kNv][NT];  // and the one before
  double f0[kNv][NT];  // flux at its first face
};

constexpr int kZtCols = 16, kZtK = 3;

// Tiles of 12 nw rows (nw waves) a column of nz >= 12 nw - 2 rows takes; they
// own 12 nw - 12 rows each inside and 12 nw - 8 at a wall.
__host__ __device__ inline int zt_tiles(int nz, int nw) {
  const int c = 12 * nw - 12, ce = 12 * nw - 8;
  return nz <= 2 * ce ? 2 : 2 + (nz - 2 * ce + c - 1) / c;
}
inline long long zt_blocks(int nx, int nz, int nw) {
  return (long long)((nx + kZtCols - 1) / kZtCols) * zt_tiles(nz, nw);
}
constexpr int kZtMinRows = 12 * 4 - 2;

// Waves per tile, 4 or 8, for a launch that takes b4 or b8 tiles of them. Four
// waves give more and smaller blocks (four per CU instead of two) but share
// less: a tile of 48 rows owns 36. The GPU holds 4096 of these waves either
// way, so a launch costs about its rounds of 4096 waves, half of that for the
// part of the last round that is filled and half for the round; at equal
// rounds four waves are 10 % faster (blocks start and end earlier). z time per
// step in us, 8 / 4 waves: 800x400 17.7 / 17.1, 2100x260 21.7 / 21.4, 1600x400
// (500 blocks of 8, just one round) 22.0 / 24.4, 1003x517 21.4 / 20.7, 3000x200
// 28.7 / 25.8, 1500x750 34.3 / 33.3, 2000x1000 50.7 / 53.8, 8192x4096 791 /
// 908; a step of 64 of 200x100 127.8 / 110.6, of 16 of 400x200 103.7 / 101.0;
// four steps of 48 grids of 200x100 to 800x400 1605 / 1567. Five to seven waves
// spread unevenly over a CU's four SIMDs: slower throughout (2000x1000 64.5,
// 64, 58).
int zt_waves(int min_nz, long long b4, long long b8) {
  constexpr long long kResident = 4096;
  auto cost = [](long long w) { return w + (w + kResident - 1) / kResident * kResident; };
  return min_nz < 12 * 8 - 2 || 10 * cost(4 * b4) <= 11 * cost(8 * b8) ? 4 : 8;
}

template <int NW, int NR>
__device__ __forceinline__ void dir_zt1_tile(const DirArgs& a, const Grid& g, int tile, int ntile,
                                             int c0, ZTileLds<NW, NR>& sm, bool corners) {
  constexpr int NT = 64 * NW, CW = kZtCols, K = kZtK, NG = NT / CW;
  constexpr int C = NR - 12, CE = NR - 8;  // rows owned: inside, at a wall
  static_assert(NG * K == NR && NT >= NR, "three rows per thread");
  const int nx = g.nx, nz = g.nz, t = threadIdx.x;
  const int col = t % CW, rg = t / CW;
  const gdouble* hy = a.hy_cell;
  const int plo = kHs, phi = nz + kHs - 1;
  const bool first = tile == 0, last = tile == ntile - 1;
  const int base = first ? -2 : last ? nz + 2 - NR : CE + (tile - 1) * C - 6;
  const int own0 = first ? 0 : last ? nz - CE : base + 6;
  const int own1 = last ? nz : min(first ? CE : base + 6 + C, nz - CE);
  const int k0 = base + rg * K;  // the thread's first row
  const bool colok = c0 + col < nx;
  const int lcol = colok ? col : nx - 1 - c0;
  const long long ubase = (long long)(base + kHs) * g.ld + c0 + kHs;  // block-uniform
  const unsigned lo = ((unsigned)(rg * K) * (unsigned)g.ld + (unsigned)lcol) * 8u;
  double S[K][4], s[K][4];
#pragma unroll
  for (int j = 0; j < K; ++j)
#pragma unroll
    for (int v = 0; v < kNv; ++v)
      S[j][v] = ld_off(a.in + v * g.plane + ubase + (long long)j * g.ld, lo);
  // the state's loads are on their way before the first wait
  if (t < NR) {
    const int k = min(max(base + t, 0), nz);
    sm.hz[0][t] = a.hyr_int[k];
    sm.hz[1][t] = a.hyt_int[k];
    sm.hz[2][t] = a.hyp_int[k];
  }
  if (corners && t < 8) {
    // corner columns (padded 0, 1, nx+2, nx+3) of the halo rows of st, tmp
    gdouble* buf = t < 4 ? a.st : a.tmp;
    const int qq = t & 3;
    const int cc = qq < 2 ? qq : nx + qq;
#pragma unroll
    for (int v = 0; v < kNv; ++v) {
      const double e = buf[g.at(v, plo, cc)];
      buf[g.at(v, 0, cc)] = wall_halo(v, e, hy[plo], hy[0]);
      buf[g.at(v, 1, cc)] = wall_halo(v, e, hy[plo], hy[1]);
      const double f = buf[g.at(v, phi, cc)];
      buf[g.at(v, nz + 2, cc)] = wall_halo(v, f, hy[phi], hy[nz + 2]);
      buf[g.at(v, nz + 3, cc)] = wall_halo(v, f, hy[phi], hy[nz + 3]);
    }
  }
#pragma unroll
  for (int j = 0; j < K; ++j)
#pragma unroll
    for (int v = 0; v < kNv; ++v) s[j][v] = S[j][v];
  // the wall halo rows of the running state, also stored to dst (set_bc_z)
  auto walls = [&](gdouble* dst) {
    if (first && rg == 0) {  // rows -2, -1 of the thread holding row 0
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < kNv; ++v) {
          s[j][v] = wall_halo(v, s[2][v], hy[plo], hy[j]);
          if (dst && colok) st_off(dst + v * g.plane + ubase + (long long)j * g.ld, lo, s[j][v]);
        }
    }
    if (last && rg == NG - 1) {  // rows nz, nz+1 of the thread holding row nz-1
#pragma unroll
      for (int j = 1; j < 3; ++j)
#pragma unroll
        for (int v = 0; v < kNv; ++v) {
          s[j][v] = wall_halo(v, s[0][v], hy[phi], hy[nz + 1 + j]);
          if (dst && colok) st_off(dst + v * g.plane + ubase + (long long)j * g.ld, lo, s[j][v]);
        }
    }
  };
  auto publish = [&]() {
#pragma unroll
    for (int v = 0; v < kNv; ++v) {
      sm.lo[v][t] = s[0][v];
      sm.h2[v][t] = s[1][v];
      sm.h1[v][t] = s[2][v];
    }
  };
  walls(a.st);
  publish();
  wave_flags_init(sm.wf, NW, t);
  __syncthreads();  // also publishes the flags
#pragma unroll
  for (int stage = 0; stage < 3; ++stage) {
    const double dts = stage == 0 ? a.dt1 : stage == 1 ? a.dt2 : a.dt3;
    gdouble* const dst = stage == 0 ? a.s1 : stage == 1 ? (a.tmp_interior ? a.tmp : nullptr) : a.out;
    auto update = [&](int j, const double cell[4], const double flo[4], const double fhi[4]) {
      double td[4];
#pragma unroll
      for (int v = 0; v < kNv; ++v) td[v] = tend_of(flo[v], fhi[v], a.id, a.idl);
      td[2] = td[2] - cell[0] * kGrav;
      if (a.src_w)
        td[2] = td[2] + a.src_w[(long long)min(max(k0 + j, 0), nz - 1) * nx + c0 + lcol];
#pragma unroll
      for (int v = 0; v < kNv; ++v) s[j][v] = S[j][v] + dts * td[v];
      if (dst && colok && k0 + j >= own0 && k0 + j < own1) {
#pragma unroll
        for (int v = 0; v < kNv; ++v)
          st_off(dst + v * g.plane + ubase + (long long)j * g.ld, lo, s[j][v]);
      }
    };
    const int tp = t >= CW ? t - CW : t, tn = t + CW < NT ? t + CW : t;  // rows before, after
    double b1[4], Fp[4];  // the row before, the flux behind
    // the stage's faces, each followed by the row before it but the last
    auto faces = [&](auto power) {
      double b2[4];
#pragma unroll
      for (int v = 0; v < kNv; ++v) {
        b2[v] = sm.h2[v][tp];
        b1[v] = sm.h1[v][tp];
      }
#pragma unroll
      for (int j = 0; j < K; ++j) {  // face k0+j, then row k0+j-1
        double v4[4], d3[4], F[4], cur[4];
#pragma unroll
        for (int v = 0; v < kNv; ++v) {
          cur[v] = s[j][v];
          recon4(b2[v], b1[v], cur[v], j + 1 < K ? s[j + 1 < K ? j + 1 : j][v] : sm.lo[v][tn],
                 v4[v], d3[v]);
        }
        const int q = rg * K + j;
        flux_z_face<false>(v4, d3, sm.hz[0][q], sm.hz[1][q], sm.hz[2][q], a.hv,
                           k0 + j == 0 || k0 + j == nz, F, power);
        if (j == 0) {
#pragma unroll
          for (int v = 0; v < kNv; ++v) sm.f0[v][t] = F[v];
        } else {
          update(j - 1, b1, Fp, F);
        }
#pragma unroll
        for (int v = 0; v < kNv; ++v) {
          b2[v] = b1[v];
          b1[v] = cur[v];
          Fp[v] = F[v];
        }
        __builtin_amdgcn_sched_barrier(0);  // one face's values live at a time
      }
    };
    unsigned long long rare = 0;
    faces(PowGammaIn{rare});
    if (__builtin_expect(rare != 0, 0)) {
      // an argument outside the table: once more, from the published rows (a
      // neighbour publishes again only after this wave's flag)
#pragma unroll
      for (int v = 0; v < kNv; ++v) {
        s[0][v] = sm.lo[v][t];
        s[1][v] = sm.h2[v][t];
        s[2][v] = sm.h1[v][t];
      }
      faces(PowGamma{});
    }
    wave_phase_done(sm.wf, 2 * stage + 1, t);
    {
      double Fn[4];
#pragma unroll
      for (int v = 0; v < kNv; ++v) Fn[v] = sm.f0[v][tn];
      update(K - 1, b1, Fp, Fn);
    }
    if (stage < 2) {
      walls(stage == 1 ? a.tmp : nullptr);
      publish();
      wave_phase_done(sm.wf, 2 * stage + 2, t);
    }
  }
}

template <int NW, int NR>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4))) void k_dir_zt1(
    DirArgs a, Grid g, int ncol, int ntile, int per_xcd) {
  __shared__ ZTileLds<NW, NR> sm;
  const int logical = xcd_logical(blockIdx.x, per_xcd);
  if (logical >= ncol * ntile) return;  // whole block, before any barrier
  member_offset(a);
  dir_zt1_tile<NW, NR>(a, g, logical / ncol, ntile, (logical % ncol) * kZtCols, sm, logical == 0);
}

// ---- z, one column per wave, for small grids: lane = row, the x waves turned
// by 90 degrees. Neighbouring rows come by one-lane shifts, no flags, no LDS
// between the stages: such a launch waits for latency, not for bandwidth.
// Tiles of a column: the first holds rows -2 .. 61, the last rows nz-62 ..
// nz+1, those between start 6 rows before the first row they own. A column of
// up to 60 rows is one wave.
// k_dir_zw, up to 512 waves: blocks of two columns that share nothing; a lane's
// loads and stores touch a cache line each. k_dir_zs, up to 4096 (four per
// SIMD): blocks of four columns whose loads and stores pass through LDS, rows
// of 32 bytes. Step in us with one-cell tiles of 32 rows / k_dir_zw / k_dir_zs:
// 37x5 11.8 / 9.9 / -, 100x50 12.0 / 10.4 / 10.8, 200x100 (400 waves) 12.3 /
// 10.9 / 11.4, 333x61 (666) 12.3 / 11.3 / 11.1, 300x150 (900) 12.4 / 11.8 /
// 11.3, 1000x60 13.7 / 13.1 / 12.5, 400x200 (1600) 13.7 / 14.6 / 13.0, 500x250
// 15.9 / - / 15.0, 600x300 (3600) 17.9 / - / 17.5, 4000x70 (8000) 27.3 / - /
// 30.0. Columns per block, k_dir_zw at 200x100 with 1, 2, 4, 8, 16: 11.2, 11.2,
// 11.4, 12.0, 14.8; k_dir_zs at 400x200 with 4, 8, 16: 13.0, 13.7, 15.7.
constexpr int kZwWaves = 2, kZsWaves = 4;  // columns per block
constexpr long long kZwMaxWaves = 512, kZsMaxWaves = 4096;

__host__ __device__ inline int zw_tiles(int nz) {
  return nz <= 60 ? 1 : nz <= 112 ? 2 : 2 + (nz - 112 + 51) / 52;
}

template <int NC>
struct ZwLds {
  double b[2][kNv][64][NC + 1];
};

// STAGED: the block's NC columns pass through LDS, so that loads and stores
// are rows of 8 NC bytes.
template <int NC, bool STAGED>
__device__ __forceinline__ void dir_z_wave(const DirArgs& a, const Grid& g, int tile, int ntile,
                                           int c0, int w, ZwLds<NC>* sm, bool corners) {
  const int nx = g.nx, nz = g.nz, lane = threadIdx.x & 63;
  const bool colok = c0 + w < nx;  // wave-uniform
  if (!STAGED && !colok) return;
  const int c = colok ? c0 + w : nx - 1;
  const bool first = tile == 0, last = tile == ntile - 1;
  const int base = first ? -2 : last ? nz - 62 : 50 + (tile - 1) * 52;
  const int own0 = first ? 0 : last ? nz - 56 : base + 6;
  const int own1 = last ? nz : min(first ? 56 : base + 58, nz - 56);
  const int k = base + lane;
  const gdouble* hy = a.hy_cell;
  const int plo = kHs, phi = nz + kHs - 1;
  const bool own = k >= own0 && k < own1;
  const int kc = min(max(k, 0), nz - 1), kf = min(max(k, 0), nz);
  const long long at = (long long)(kc + kHs) * g.ld + c + kHs;  // clamped row
  // every load is issued before the first is waited for
  double S[4], s[4];
  // STAGED: this thread's row and column of the block's loads and stores
  const int ri = threadIdx.x / NC, ci = threadIdx.x % NC, kr = base + ri;
  const long long rat = (long long)(min(max(kr, 0), nz - 1) + kHs) * g.ld + min(c0 + ci, nx - 1) + kHs;
  const bool rown = kr >= own0 && kr < own1 && c0 + ci < nx;
  int buf = 0;
  if constexpr (STAGED) {
    double q[4];
#pragma unroll
    for (int v = 0; v < kNv; ++v) q[v] = a.in[v * g.plane + rat];
#pragma unroll
    for (int v = 0; v < kNv; ++v) sm->b[0][v][ri][ci] = q[v];
  } else {
#pragma unroll
    for (int v = 0; v < kNv; ++v) S[v] = a.in[v * g.plane + at];
  }
  const double hyr = a.hyr_int[kf], hyt = a.hyt_int[kf], hyp = a.hyp_int[kf];
  const bool low = k == -2 || k == -1, high = k == nz || k == nz + 1;
  const bool wall = low || high;
  const double hye = hy[low ? plo : phi], hyh = hy[wall ? k + kHs : phi];
  const double src = a.src_w ? a.src_w[(long long)kc * nx + c] : 0.0;
  if (corners && threadIdx.x < 8) {
    // corner columns (padded 0, 1, nx+2, nx+3) of the halo rows of st, tmp
    const int t = threadIdx.x;
    gdouble* buf = t < 4 ? a.st : a.tmp;
    const int qq = t & 3;
    const int cc = qq < 2 ? qq : nx + qq;
#pragma unroll
    for (int v = 0; v < kNv; ++v) {
      const double e = buf[g.at(v, plo, cc)];
      buf[g.at(v, 0, cc)] = wall_halo(v, e, hy[plo], hy[0]);
      buf[g.at(v, 1, cc)] = wall_halo(v, e, hy[plo], hy[1]);
      const double f = buf[g.at(v, phi, cc)];
      buf[g.at(v, nz + 2, cc)] = wall_halo(v, f, hy[phi], hy[nz + 2]);
      buf[g.at(v, nz + 3, cc)] = wall_halo(v, f, hy[phi], hy[nz + 3]);
    }
  }
  if constexpr (STAGED) {
    __syncthreads();
#pragma unroll
    for (int v = 0; v < kNv; ++v) S[v] = sm->b[0][v][lane][w];
  }
#pragma unroll
  for (int v = 0; v < kNv; ++v) s[v] = S[v];
#pragma unroll
  for (int stage = 0; stage < 3; ++stage) {
    const double dts = stage == 0 ? a.dt1 : stage == 1 ? a.dt2 : a.dt3;
    if (base < 0 || base + 63 >= nz) {  // wall halo rows, stored by set_bc_z of stages 1 and 3
      gdouble* const halo = stage == 0 ? a.st : a.tmp;
#pragma unroll
      for (int v = 0; v < kNv; ++v) {
        double e;
        if (stage == 0) {
          e = s[v];  // loaded from the edge row
        } else {
          const double n1 = from_next(s[v]), p1 = from_prev(s[v]);
          const double n2 = from_next(n1), p2 = from_prev(p1);
          e = low ? (k == -1 ? n1 : n2) : (k == nz ? p1 : p2);
        }
        if (wall) {
          s[v] = wall_halo(v, e, hye, hyh);
          if (stage != 1 && colok && (low ? first : last))
            halo[v * g.plane + (long long)(k + kHs) * g.ld + c + kHs] = s[v];
        }
      }
    }
    double v4[4], d3[4], F[4];
#pragma unroll
    for (int v = 0; v < kNv; ++v) {
      const double b1 = from_prev(s[v]);
      recon4(from_prev(b1), b1, s[v], from_next(s[v]), v4[v], d3[v]);
    }
    flux_z_face<false>(v4, d3, hyr, hyt, hyp, a.hv, k == 0 || k == nz, F, PowGamma{});
    double td[4];
#pragma unroll
    for (int v = 0; v < kNv; ++v) td[v] = tend_of(F[v], from_next(F[v]), a.id, a.idl);
    td[2] = td[2] - s[0] * kGrav;
    if (a.src_w) td[2] = td[2] + src;
#pragma unroll
    for (int v = 0; v < kNv; ++v) s[v] = S[v] + dts * td[v];
    gdouble* const dst = stage == 0 ? a.s1 : stage == 1 ? (a.tmp_interior ? a.tmp : nullptr) : a.out;
    if constexpr (STAGED) {
      if (dst) {  // the same for the whole block
        // Two buffers in turn: when a wave writes a buffer again it has passed
        // the barrier of the store between, and with it every wave its reads.
        auto& b = sm->b[buf];
        buf ^= 1;
#pragma unroll
        for (int v = 0; v < kNv; ++v) b[v][lane][w] = s[v];
        __syncthreads();
        if (rown) {
#pragma unroll
          for (int v = 0; v < kNv; ++v) dst[v * g.plane + rat] = b[v][ri][ci];
        }
      }
    } else if (dst && own) {
#pragma unroll
      for (int v = 0; v < kNv; ++v) dst[v * g.plane + at] = s[v];
    }
  }
}

__global__ __launch_bounds__(64 * kZwWaves) void k_dir_zw(DirArgs a, Grid g, int ncol, int ntile,
                                                          int per_xcd) {
  const int logical = xcd_logical(blockIdx.x, per_xcd);
  if (logical >= ncol * ntile) return;
  member_offset(a);
  dir_z_wave<kZwWaves, false>(a, g, logical / ncol, ntile, (logical % ncol) * kZwWaves,
                              __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nullptr,
                              logical == 0);
}

__global__ __launch_bounds__(64 * kZsWaves) void k_dir_zs(DirArgs a, Grid g, int ncol, int ntile,
                                                          int per_xcd) {
  __shared__ ZwLds<kZsWaves> sm;
  const int logical = xcd_logical(blockIdx.x, per_xcd);
  if (logical >= ncol * ntile) return;  // whole block, before any barrier
  member_offset(a);
  dir_z_wave<kZsWaves, true>(a, g, logical / ncol, ntile, (logical % ncol) * kZsWaves,
                             __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), &sm, logical == 0);
}

// ---- z, one cell per thread, for small grids and low columns.
// A block holds 8 columns x NR rows (slot t = row*8 + col, tile row j =
// logical row r0-6+j; NR-12 rows are written), the RK init in registers and
// the stage state updated in place; the wall halo rows of each stage state are
// written by the edge row's thread in the update phase (no thread reads them
// then). A wave holds 8 whole rows: phases by wave flags. NR = 32 for small
// grids: a launch that leaves most of the GPU idle takes as long as one block,
// and at 200 x 100 4-wave blocks (one wave per SIMD) take 10.6 us between
// events where 12-wave blocks (NR = 96) take 12.7; NR = 24 (three waves) is
// 0.6 us faster there and 0.7 us slower at 400 x 200.
constexpr int kZ1Cols = 8;

template <int NR>
struct Z1Lds {
  double s[kNv][kZ1Cols * NR];
  double fl[kNv][kZ1Cols * NR];
  double hz[3][NR];
  int wf[kZ1Cols * NR / 64 + 2];
};

template <int NR>
__device__ __forceinline__ void dir_z1_tile(const DirArgs& a, const Grid& g, int c0, int r0,
                                            Z1Lds<NR>& sm, bool corners) {
  constexpr int CW = kZ1Cols, NT = CW * NR, C = NR - 12;
  auto& s = sm.s;
  auto& fl = sm.fl;
  auto& hz = sm.hz;
  const int nx = g.nx, nz = g.nz, t = threadIdx.x;
  wave_flags_init(sm.wf, NT / 64, t);
  const int col = t % CW, u = t, j = t / CW;
  const gdouble* hy = a.hy_cell;
  const int plo = kHs, phi = nz + kHs - 1;
  const int k = r0 - 6 + j;
  const int i = c0 + col;
  const bool colok = i < nx;
  const int pc = (colok ? i : 0) + kHs;
  const bool wl = k == -2 || k == -1, wh = k == nz || k == nz + 1;
  const bool own = colok && j >= 6 && j < 6 + C && k >= 0 && k < nz;
  // every load is issued before the first is waited for; halo rows take their
  // edge row's
  const int kc = min(max(k, 0), nz - 1);
  double S[4];
#pragma unroll
  for (int v = 0; v < kNv; ++v) S[v] = a.in[g.at(v, kc + kHs, pc)];
  if (t < NR) {
    const int k = r0 - 6 + t;
    const bool f = k >= 0 && k <= nz;
    hz[0][t] = f ? a.hyr_int[k] : 0.0;
    hz[1][t] = f ? a.hyt_int[k] : 0.0;
    hz[2][t] = f ? a.hyp_int[k] : 0.0;
  }
  if (wl || wh) {
    const int pe = kc + kHs;
#pragma unroll
    for (int v = 0; v < kNv; ++v) S[v] = wall_halo(v, S[v], hy[pe], hy[k + kHs]);
    if (colok && j - (k - kc) >= 6 && j - (k - kc) < NR - 6) {  // set_bc_z of stage 1 into st
#pragma unroll
      for (int v = 0; v < kNv; ++v) a.st[g.at(v, k + kHs, pc)] = S[v];
    }
  }
#pragma unroll
  for (int v = 0; v < kNv; ++v) s[v][u] = S[v];
  const double src = (a.src_w && colok && k >= 0 && k < nz) ? a.src_w[(long long)k * nx + i] : 0.0;
  if (corners && t < 8) {
    // corner columns (padded 0, 1, nx+2, nx+3) of the halo rows of st, tmp
    gdouble* buf = t < 4 ? a.st : a.tmp;
    const int qq = t & 3;
    const int cc = qq < 2 ? qq : nx + qq;
#pragma unroll
    for (int v = 0; v < kNv; ++v) {
      const double e = buf[g.at(v, plo, cc)];
      buf[g.at(v, 0, cc)] = wall_halo(v, e, hy[plo], hy[0]);
      buf[g.at(v, 1, cc)] = wall_halo(v, e, hy[plo], hy[1]);
      const double f = buf[g.at(v, phi, cc)];
      buf[g.at(v, nz + 2, cc)] = wall_halo(v, f, hy[phi], hy[nz + 2]);
      buf[g.at(v, nz + 3, cc)] = wall_halo(v, f, hy[phi], hy[nz + 3]);
    }
  }
  gdouble* const tmp_own = a.tmp_interior ? a.tmp : nullptr;
  __syncthreads();  // also publishes the flags
#pragma unroll
  for (int stage = 0; stage < 3; ++stage) {
    const int e = 2 + 2 * stage;
    if (colok && j >= e && j <= NR - e && k >= 0 && k <= nz) {
      double v4[4], d3[4], G[4];
#pragma unroll
      for (int v = 0; v < kNv; ++v)
        recon4(s[v][u - 2 * CW], s[v][u - CW], s[v][u], s[v][u + CW], v4[v], d3[v]);
      flux_z_face<false>(v4, d3, hz[0][j], hz[1][j], hz[2][j], a.hv, k == 0 || k == nz, G,
                         PowGamma{});
#pragma unroll
      for (int v = 0; v < kNv; ++v) fl[v][u] = G[v];
    }
    wave_phase_done(sm.wf, 2 * stage + 1, t);
    const double dts = stage == 0 ? a.dt1 : stage == 1 ? a.dt2 : a.dt3;
    if (colok && j >= e && j <= NR - e - 1 && k >= 0 && k < nz) {
      double td[4];
#pragma unroll
      for (int v = 0; v < kNv; ++v) td[v] = tend_of(fl[v][u], fl[v][u + CW], a.id, a.idl);
      td[2] = td[2] - s[0][u] * kGrav;
      if (a.src_w) td[2] = td[2] + src;
      double q[4];
#pragma unroll
      for (int v = 0; v < kNv; ++v) q[v] = S[v] + dts * td[v];
      if (stage < 2) {
#pragma unroll
        for (int v = 0; v < kNv; ++v) s[v][u] = q[v];  // in place: faces are done
        // the wall halo rows of the new stage state (slots u -+ CW, 2 CW of
        // this column group; no thread reads them in this phase)
#pragma unroll
        for (int side = 0; side < 2; ++side) {
          if (k == (side == 0 ? 0 : nz - 1)) {
            const int pe = side == 0 ? plo : phi;
            const int step = side == 0 ? -CW : CW;
#pragma unroll
            for (int h = 1; h <= 2; ++h) {
              const int kh = side == 0 ? -h : nz - 1 + h;  // the halo row's k
              double w[4];
#pragma unroll
              for (int v = 0; v < kNv; ++v) w[v] = wall_halo(v, q[v], hy[pe], hy[kh + kHs]);
#pragma unroll
              for (int v = 0; v < kNv; ++v) s[v][u + h * step] = w[v];
              if (stage == 1 && own) {  // set_bc_z of stage 3
#pragma unroll
                for (int v = 0; v < kNv; ++v) a.tmp[g.at(v, kh + kHs, pc)] = w[v];
              }
            }
          }
        }
      }
      if (own) {
        gdouble* dst = stage == 0 ? a.s1 : stage == 1 ? tmp_own : a.out;
        if (dst) {
#pragma unroll
          for (int v = 0; v < kNv; ++v) dst[g.at(v, k + kHs, pc)] = q[v];
        }
      }
    }
    if (stage == 2) break;
    wave_phase_done(sm.wf, 2 * stage + 2, t);
  }
}

// The same, dense: the extended columns of the CW-column groups (rows
// -2 .. nz+1: the wall halo rows are rebuilt from the edge row at every
// stage, so a column needs no more) laid end to end, slot row g of block b
// being b*(NR-12) + j - 4, cut into tiles of NR rows; the offset puts row 0
// of the first group at the first window row. Windows [6, NR-6)
// partition the interior rows; the wall halo rows written to st and tmp
// belong to the block whose window holds their edge row. A halo row whose
// edge row lies outside the block is left unrebuilt: no correct cell of the
// block reaches it.
inline long long dense_z_rows(int nx, int nz, int cw) {
  return (long long)((nx + cw - 1) / cw) * (nz + 4);
}
inline int dense_z_blocks(int nx, int nz, int cw, int nr) {
  return (int)((dense_z_rows(nx, nz, cw) - 5) / (nr - 12)) + 1;
}

// The dense tiles with one cell per thread (CW x NR threads, a wave holding 8
// whole slot rows): the RK init in registers, the stage state updated in
// place, the wall halo rows of each stage state written by the edge row's
// thread in the update phase, and the waves ordered by neighbour flags. A
// face that reads a wall halo row lies 2 slots inside the next stage's face
// window, so its edge row was updated, and its halo rows written, in this
// block at the stage before; halo rows of edge rows outside that window are
// left unwritten, as no face of the block that is kept reads them.
template <int NR>
__device__ __forceinline__ void dir_z1d_tile(const DirArgs& a, const Grid& g, int b,
                                              Z1Lds<NR>& sm, bool corners) {
  constexpr int CW = kZ1Cols, NT = CW * NR, C = NR - 12;
  auto& s = sm.s;
  auto& fl = sm.fl;
  auto& hz = sm.hz;
  const int nx = g.nx, nz = g.nz, t = threadIdx.x;
  const int Ez = nz + 4;
  wave_flags_init(sm.wf, NT / 64, t);
  const int col = t % CW, u = t, j = t / CW;
  const gdouble* hy = a.hy_cell;
  const int plo = kHs, phi = nz + kHs - 1;
  const int gr = b * C + j - 4;
  const int grp = gr >= 0 ? gr / Ez : -1;
  const int k = gr >= 0 ? gr - grp * Ez - 2 : -3;  // -3: padding before the first group
  const int i = grp * CW + col;
  const bool colok = gr >= 0 && i < nx;
  const int pc = (colok ? i : 0) + kHs;
  const bool wl = k == -2 || k == -1, wh = k == nz || k == nz + 1;
  const bool own = colok && j >= 6 && j < NR - 6 && k >= 0 && k < nz;
  // every load is issued before the first is waited for; halo rows take their
  // edge row's
  const int kc = min(max(k, 0), nz - 1);
  double S[4];
#pragma unroll
  for (int v = 0; v < kNv; ++v) S[v] = a.in[g.at(v, kc + kHs, pc)];
  if (t < NR) {  // a tile row is one row k of one column group
    const int gr = b * C + t - 4;
    const int k = gr >= 0 ? gr % Ez - 2 : -3;
    const bool f = k >= 0 && k <= nz;
    hz[0][t] = f ? a.hyr_int[k] : 0.0;
    hz[1][t] = f ? a.hyt_int[k] : 0.0;
    hz[2][t] = f ? a.hyp_int[k] : 0.0;
  }
  if (wl || wh) {
    const int pe = kc + kHs;
#pragma unroll
    for (int v = 0; v < kNv; ++v) S[v] = wall_halo(v, S[v], hy[pe], hy[k + kHs]);
    if (colok && j - (k - kc) >= 6 && j - (k - kc) < NR - 6) {  // set_bc_z of stage 1 into st
#pragma unroll
      for (int v = 0; v < kNv; ++v) a.st[g.at(v, k + kHs, pc)] = S[v];
    }
  }
#pragma unroll
  for (int v = 0; v < kNv; ++v) s[v][u] = S[v];
  const double src = (a.src_w && colok && k >= 0 && k < nz) ? a.src_w[(long long)k * nx + i] : 0.0;
  if (corners && t < 8) {
    // corner columns (padded 0, 1, nx+2, nx+3) of the halo rows of st, tmp
    gdouble* buf = t < 4 ? a.st : a.tmp;
    const int qq = t & 3;
    const int cc = qq < 2 ? qq : nx + qq;
#pragma unroll
    for (int v = 0; v < kNv; ++v) {
      const double e = buf[g.at(v, plo, cc)];
      buf[g.at(v, 0, cc)] = wall_halo(v, e, hy[plo], hy[0]);
      buf[g.at(v, 1, cc)] = wall_halo(v, e, hy[plo], hy[1]);
      const double f = buf[g.at(v, phi, cc)];
      buf[g.at(v, nz + 2, cc)] = wall_halo(v, f, hy[phi], hy[nz + 2]);
      buf[g.at(v, nz + 3, cc)] = wall_halo(v, f, hy[phi], hy[nz + 3]);
    }
  }
  gdouble* const tmp_own = a.tmp_interior ? a.tmp : nullptr;
  __syncthreads();  // also publishes the flags
#pragma unroll
  for (int stage = 0; stage < 3; ++stage) {
    const int e = 2 + 2 * stage;
    if (colok && j >= e && j <= NR - e && k >= 0 && k <= nz) {
      double v4[4], d3[4], G[4];
#pragma unroll
      for (int v = 0; v < kNv; ++v)
        recon4(s[v][u - 2 * CW], s[v][u - CW], s[v][u], s[v][u + CW], v4[v], d3[v]);
      flux_z_face<false>(v4, d3, hz[0][j], hz[1][j], hz[2][j], a.hv, k == 0 || k == nz, G,
                         PowGamma{});
#pragma unroll
      for (int v = 0; v < kNv; ++v) fl[v][u] = G[v];
    }
    wave_phase_done(sm.wf, 2 * stage + 1, t);
    const double dts = stage == 0 ? a.dt1 : stage == 1 ? a.dt2 : a.dt3;
    if (colok && j >= e && j <= NR - e - 1 && k >= 0 && k < nz) {
      double td[4];
#pragma unroll
      for (int v = 0; v < kNv; ++v) td[v] = tend_of(fl[v][u], fl[v][u + CW], a.id, a.idl);
      td[2] = td[2] - s[0][u] * kGrav;
      if (a.src_w) td[2] = td[2] + src;
      double q[4];
#pragma unroll
      for (int v = 0; v < kNv; ++v) q[v] = S[v] + dts * td[v];
      if (stage < 2) {
#pragma unroll
        for (int v = 0; v < kNv; ++v) s[v][u] = q[v];  // in place: faces are done
        // the wall halo rows of the new stage state (slots u -+ CW, 2 CW of
        // this column group; no thread reads them in this phase)
#pragma unroll
        for (int side = 0; side < 2; ++side) {
          if (k == (side == 0 ? 0 : nz - 1)) {
            const int pe = side == 0 ? plo : phi;
            const int step = side == 0 ? -CW : CW;
#pragma unroll
            for (int h = 1; h <= 2; ++h) {
              const int kh = side == 0 ? -h : nz - 1 + h;  // the halo row's k
              double w[4];
#pragma unroll
              for (int v = 0; v < kNv; ++v) w[v] = wall_halo(v, q[v], hy[pe], hy[kh + kHs]);
#pragma unroll
              for (int v = 0; v < kNv; ++v) s[v][u + h * step] = w[v];
              if (stage == 1 && own) {  // set_bc_z of stage 3
#pragma unroll
                for (int v = 0; v < kNv; ++v) a.tmp[g.at(v, kh + kHs, pc)] = w[v];
              }
            }
          }
        }
      }
      if (own) {
        gdouble* dst = stage == 0 ? a.s1 : stage == 1 ? tmp_own : a.out;
        if (dst) {
#pragma unroll
          for (int v = 0; v < kNv; ++v) dst[g.at(v, k + kHs, pc)] = q[v];
        }
      }
    }
    if (stage == 2) break;
    wave_phase_done(sm.wf, 2 * stage + 2, t);
  }
}

template <int NR>
__global__ __launch_bounds__(kZ1Cols * NR) __attribute__((amdgpu_waves_per_eu(6))) void k_dir_z1(
    DirArgs a, Grid g, int ncolgrp, int nreal, int per_xcd) {
  __shared__ Z1Lds<NR> sm;
  const int logical = xcd_logical(blockIdx.x, per_xcd);
  if (logical >= nreal) return;  // whole block, before any barrier
  member_offset(a);
  dir_z1_tile<NR>(a, g, (logical % ncolgrp) * kZ1Cols, (logical / ncolgrp) * (NR - 12), sm,
                  logical == 0);
}

template <int NR>
__global__ __launch_bounds__(kZ1Cols * NR) __attribute__((amdgpu_waves_per_eu(6))) void k_dir_z1d(
    DirArgs a, Grid g, int nreal, int per_xcd) {
  __shared__ Z1Lds<NR> sm;
  const int logical = xcd_logical(blockIdx.x, per_xcd);
  if (logical >= nreal) return;  // whole block, before any barrier
  member_offset(a);
  dir_z1d_tile<NR>(a, g, logical, sm, logical == 0);
}

// ------------------------------------------------------------- ensemble --
// Device descriptor of one member of an ensemble (uneven grids).
struct MemberDev {
  double* state;
  double* tmp;
  double* work;
  const double* hyc;   // hy_dens_cell
  const double* hytc;  // hy_dens_theta_cell
  const double* hyri;  // hy_dens_int
  const double* hyti;  // hy_dens_theta_int
  const double* hypi;  // hy_pressure_int
  const double* src;   // w source or nullptr
  int nx, nz;
  double dt1, dt2, dt3, hvx, hvz;
  double idx, idz, idxl, idzl;  // 1/dx, 1/dz as sums
  int x_start, z_start;  // first work item of this member in the x / z lists
  int x_blocks, z_ncol;  // blocks of the member's x waves, z column groups
};

__device__ __forceinline__ DirArgs member_args(const MemberDev& m, int dir, int pass,
                                               bool tmp_interior) {
  DirArgs a;
  a.in = gptr(pass == 0 ? m.state : m.work);
  a.out = gptr(pass == 0 ? m.work : m.state);
  a.st = gptr(m.state);
  a.tmp = gptr(m.tmp);
  a.tmp_interior = tmp_interior;
  a.hy_cell = gptr(m.hyc);
  a.hyt_cell = gptr(m.hytc);
  a.hyr_int = gptr(m.hyri);
  a.hyt_int = gptr(m.hyti);
  a.hyp_int = gptr(m.hypi);
  a.src_w = m.src ? gptr(m.src) : nullptr;
  a.id = dir == 0 ? m.idx : m.idz;
  a.idl = dir == 0 ? m.idxl : m.idzl;
  a.dt1 = m.dt1;
  a.dt2 = m.dt2;
  a.dt3 = m.dt3;
  a.hv = dir == 0 ? m.hvx : m.hvz;
  return a;
}

// Member owning work item `item`: binary search over the ascending start
// offsets (block-uniform, scalar loads). The offsets are also kept as two
// packed int arrays after the descriptors (x starts, then z starts): a
// search then touches a few cache lines instead of one descriptor per probe
// (256 descriptors are 39 KB, more than the scalar cache holds).
template <int DIR>
__device__ __forceinline__ int member_of(const MemberDev* m, int n, int item) {
  const PMW_GLOBAL int* start = (const PMW_GLOBAL int*)(m + n) + DIR * n;
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (start[mid] <= item) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Ensemble kernels: one launch covers the flattened work list of every
// member (tiles of member q are items x_start[q] .. ); block b takes item
// xcd_logical(b), so neighbouring tiles of a member share an XCD's L2, and
// finds its member by a scalar binary search over the start offsets. (A
// persistent form, each block looping over a chunk of items, kept ~70 more
// VGPRs live and halved the occupancy.) `pass`: bit 0 = direction of the
// step (0: state -> work, 1: work -> state), bit 1 = store state_tmp's
// interior (the last direction of the call only).
template <int NS>
__global__ __launch_bounds__(64 * kXwWaves)
    __attribute__((amdgpu_waves_per_eu(xw_waves_per_simd(NS / 256)))) void k_ens_x(
        const MemberDev* __restrict__ m, int n, int pass, int total, int per_xcd) {
  constexpr int K = NS / 256;
  __shared__ XWaveLds<K> sm;
  const int item = xcd_logical(blockIdx.x, per_xcd);
  if (item >= total) return;
  const MemberDev& md = m[member_of<0>(m, n, item)];
  const DirArgs a = member_args(md, 0, pass & 1, pass >> 1);
  const int local = item - md.x_start;
  if (local >= md.x_blocks) return;  // a plan that is not the prepared one: stay in bounds
  dir_x_wave<K, false>(a, Grid(md.nx, md.nz), xw_wave(local), xw_row_slots(md.nx, K), 0, md.nz,
                       sm.s[threadIdx.x >> 6]);
}

template <int NW, int NR>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4))) void k_ens_zt1(
    const MemberDev* __restrict__ m, int n, int pass, int total, int per_xcd) {
  __shared__ ZTileLds<NW, NR> sm;
  const int item = xcd_logical(blockIdx.x, per_xcd);
  if (item >= total) return;  // whole block, before any barrier
  const MemberDev& md = m[member_of<1>(m, n, item)];
  const DirArgs a = member_args(md, 1, pass & 1, pass >> 1);
  const int local = item - md.z_start, ntile = zt_tiles(md.nz, NW);
  if (local >= md.z_ncol * ntile) return;  // as in k_ens_x
  dir_zt1_tile<NW, NR>(a, Grid(md.nx, md.nz), local / md.z_ncol, ntile,
                       (local % md.z_ncol) * kZtCols, sm, local == 0);
}

template <int NR>
__global__ __launch_bounds__(kZ1Cols * NR) __attribute__((amdgpu_waves_per_eu(6))) void k_ens_z1(
    const MemberDev* __restrict__ m, int n, int pass, int total, int per_xcd) {
  __shared__ Z1Lds<NR> sm;
  const int item = xcd_logical(blockIdx.x, per_xcd);
  if (item >= total) return;  // whole block, before any barrier
  const MemberDev& md = m[member_of<1>(m, n, item)];
  const DirArgs a = member_args(md, 1, pass & 1, pass >> 1);
  const int local = item - md.z_start;
  if ((long long)(local / md.z_ncol) * (NR - 12) >= md.nz) return;  // as in k_ens_x
  dir_z1_tile<NR>(a, Grid(md.nx, md.nz), (local % md.z_ncol) * kZ1Cols,
                  (local / md.z_ncol) * (NR - 12), sm, local == 0);
}

template <int NR>
__global__ __launch_bounds__(kZ1Cols * NR) __attribute__((amdgpu_waves_per_eu(6))) void k_ens_z1d(
    const MemberDev* __restrict__ m, int n, int pass, int total, int per_xcd) {
  __shared__ Z1Lds<NR> sm;
  const int item = xcd_logical(blockIdx.x, per_xcd);
  if (item >= total) return;  // whole block, before any barrier
  const MemberDev& md = m[member_of<1>(m, n, item)];
  const DirArgs a = member_args(md, 1, pass & 1, pass >> 1);
  const int local = item - md.z_start;
  if (local >= md.z_ncol) return;  // dense z: z_ncol holds the member's blocks
  dir_z1d_tile<NR>(a, Grid(md.nx, md.nz), local, sm, local == 0);
}

int launch_zs(const DirArgs& a, Grid g, hipStream_t st, int members) {
  const int ncol = (g.nx + kZsWaves - 1) / kZsWaves, ntile = zw_tiles(g.nz);
  const int per = (ncol * ntile + kNumXcd - 1) / kNumXcd;
  k_dir_zs<<<dim3(per * kNumXcd, members), 64 * kZsWaves, 0, st>>>(a, g, ncol, ntile, per);
  PMW_CHECK_LAUNCH();
  return PMW_OK;
}

template <int NW>
int launch_zt1(const DirArgs& a, Grid g, hipStream_t st, int members) {
  constexpr int NR = 12 * NW;
  const int ncol = (g.nx + kZtCols - 1) / kZtCols, ntile = zt_tiles(g.nz, NW);
  const int per = (ncol * ntile + kNumXcd - 1) / kNumXcd;
  k_dir_zt1<NW, NR><<<dim3(per * kNumXcd, members), 64 * NW, 0, st>>>(a, g, ncol, ntile, per);
  PMW_CHECK_LAUNCH();
  return PMW_OK;
}

int launch_zw(const DirArgs& a, Grid g, hipStream_t st, int members) {
  const int ncol = (g.nx + kZwWaves - 1) / kZwWaves, ntile = zw_tiles(g.nz);
  const int per = (ncol * ntile + kNumXcd - 1) / kNumXcd;
  k_dir_zw<<<dim3(per * kNumXcd, members), 64 * kZwWaves, 0, st>>>(a, g, ncol, ntile, per);
  PMW_CHECK_LAUNCH();
  return PMW_OK;
}

template <int NR>
int launch_z1(const DirArgs& a, Grid g, hipStream_t st, int members) {
  constexpr int C = NR - 12;
  const int ncolgrp = (g.nx + kZ1Cols - 1) / kZ1Cols;
  const long long nreal = (long long)ncolgrp * ((g.nz + C - 1) / C);
  if (nreal > (1LL << 31) - 64) return PMW_EINVAL;
  const int per = (int)((nreal + kNumXcd - 1) / kNumXcd);
  k_dir_z1<NR><<<dim3(per * kNumXcd, members), kZ1Cols * NR, 0, st>>>(a, g, ncolgrp, (int)nreal,
                                                                      per);
  PMW_CHECK_LAUNCH();
  return PMW_OK;
}

template <int NR>
int launch_z1d(const DirArgs& a, Grid g, hipStream_t st, int members) {
  const int nreal = dense_z_blocks(g.nx, g.nz, kZ1Cols, NR);
  const int per = (nreal + kNumXcd - 1) / kNumXcd;
  k_dir_z1d<NR><<<dim3(per * kNumXcd, members), kZ1Cols * NR, 0, st>>>(a, g, nreal, per);
  PMW_CHECK_LAUNCH();
  return PMW_OK;
}

template <int K>
int launch_x(const DirArgs& a, Grid g, hipStream_t st, int members) {
  const unsigned E = xw_row_slots(g.nx, K);
  // slots are 32-bit: rows beyond 2^31 of them go to further blockIdx.z
  const int rows = (int)std::min<long long>(g.nz, std::max(1LL, (1LL << 31) / E));
  const int chunks = (g.nz + rows - 1) / rows;
  if (chunks > 65535) return PMW_EINVAL;
  const int nreal = xw_blocks(g.nx, rows, K, a.inj_rows != nullptr);
  const int per = (nreal + kNumXcd - 1) / kNumXcd;
  const dim3 grid(per * kNumXcd, members, chunks);
  if (a.inj_rows)
    k_dir_xi<256 * K><<<grid, 64 * kXwWaves, 0, st>>>(a, g, E, rows, nreal, per);
  else
    k_dir_x<256 * K><<<grid, 64 * kXwWaves, 0, st>>>(a, g, E, rows, nreal, per);
  PMW_CHECK_LAUNCH();
  return PMW_OK;
}

}  // namespace

namespace pmw {

bool fused_x_tile_ok(int nt) {
  return nt == 256 || nt == 448 || nt == 512 || nt == 1256 || nt == 1512;
}

// Cells per lane of the x waves for a launch over `cells` cells: code 256
// forces one, 1512 two; the other codes go by size. Two cells waste 10 % of
// the slots on wave overlap instead of 23 % and halve the neighbour exchange
// per cell, but each wave takes twice as long: one cell per lane is faster
// while all its waves (one per 52 slots) fit the 6 x 1024 the GPU holds at
// once. Step time in us, one / two cells per lane: 200x100 10.7 / 11.9, 400x200
// 12.6 / 12.8, 700x350 21.0 / 21.6, 774x387 23.3 / 23.1, 800x400 (just over one
// round of waves) 23.9 / 22.9, 900x450 25.3 / 25.1, 1003x517 29.1 / 29.8, 1100x550
// 32.7 / 33.1, 1200x600 36.9 / 36.6, 1500x750 50.7 / 49.2, 2000x1000 78.4 / 74.9,
// 4096x2048 367 / 334; with the inflow 400x200 13.4 / 14.5, 800x400 24.7 / 24.5,
// 1003x517 31.4 / 31.8, 2000x1000 81.9 / 76.9. The cost goes by rounds of waves, so
// a line by cells is up to 2.5 % off between 500000 and 600000 cells, where one
// cell per lane fills its second round.
int fused_x_cells(int nt, long long cells) {
  if (nt == 256 || nt == 1512) return nt == 256 ? 1 : 2;
  return cells <= 300000 ? 1 : 2;
}

bool fused_z_seg_ok(int seg) {
  return seg == 8 || seg == 16 || seg == 24 || seg == 32 || seg == 48 || seg == 64 ||
         seg == 8064 || seg == 4128 || seg == 8128 || seg == 18128 || seg == 8096 || seg == 18096;
}

// The z kernel of a launch over `cells` cells of grids whose smallest nz and
// largest nx are given. Codes 18096 and 18128 force the dense one-cell tiles,
// 8 to 64 the small ones; the others go by size. The three-row tiles need
// edge tiles that reach past their own rows into the grid only (nz >= 46 for
// their smallest) and 32-bit offsets inside a tile; they win once their blocks
// fill the GPU. Step time in us, one-cell tiles of 32 rows / three-row tiles:
// 800x400 23.3 / 22.9, 900x450 27.8 / 25.1, 1003x517 32.3 / 29.8, 1500x750 57.9 /
// 49.2, 2000x1000 93.1 / 74.7; below the line, with earlier x kernels, 600x300 18.3 /
// 20.3, 700x350 22.2 / 21.2, 1000x300 24.8 / 25.9.
// Against one-cell tiles of 96 rows, which remain for columns and rows outside
// those bounds: 10000x50 40.1 / 40.1, x60 43.3 / 41.4, x80 45.4 / 42.3, x93
// 66.4 / 53.0.
enum ZKernel { Z_ROWS3, Z_ONE96, Z_ONE32, Z_DENSE };
ZKernel fused_z_kernel(int seg, long long cells, int min_nz, int max_nx) {
  if (seg == 18096 || seg == 18128) return Z_DENSE;
  if (seg <= 64 || cells <= 300000) return Z_ONE32;
  if (min_nz >= kZtMinRows && max_nx < (1 << 22)) return Z_ROWS3;
  return min_nz > 40 ? Z_ONE96 : Z_ONE32;
}

int launch_dir_x(const DirArgs& a, Grid g, int nt, hipStream_t st, int members) {
  if (members < 1 || members > 65535 || (members > 1 && a.mstride <= 0)) return PMW_EINVAL;
  if (!fused_x_tile_ok(nt) || (a.inj_rows && g.nx < kMinInflowCells)) return PMW_EINVAL;
  // the bound of these codes; the inflow, which has always run whatever the code,
  // has none (the kernels take rows beyond 2^31 slots as further blockIdx.z)
  if (nt > 1000 && !a.inj_rows && (long long)g.nz * (g.nx + 12) > (1LL << 30))
    return PMW_EINVAL;
  return fused_x_cells(nt, (long long)g.nx * g.nz * members) == 1
             ? launch_x<1>(a, g, st, members)
             : launch_x<2>(a, g, st, members);
}

int launch_dir_z(const DirArgs& a, Grid g, int seg, hipStream_t st, int members) {
  if (members < 1 || members > 65535 || (members > 1 && a.mstride <= 0)) return PMW_EINVAL;
  if (!fused_z_seg_ok(seg)) return PMW_EINVAL;
  switch (fused_z_kernel(seg, (long long)g.nx * g.nz * members, g.nz, g.nx)) {
    case Z_ROWS3:
      return zt_waves(g.nz, zt_blocks(g.nx, g.nz, 4) * members,
                      zt_blocks(g.nx, g.nz, 8) * members) == 4
                 ? launch_zt1<4>(a, g, st, members)
                 : launch_zt1<8>(a, g, st, members);
    case Z_ONE96: return launch_z1<96>(a, g, st, members);
    case Z_ONE32:
      if (seg > 64) {  // no code that forces a kernel: columns as waves if they fit
        const long long waves = (long long)g.nx * zw_tiles(g.nz) * members;
        if (waves <= kZwMaxWaves) return launch_zw(a, g, st, members);
        if (waves <= kZsMaxWaves) return launch_zs(a, g, st, members);
      }
      return launch_z1<32>(a, g, st, members);
    default:
      if (dense_z_rows(g.nx, g.nz, kZ1Cols) > (1LL << 30)) return PMW_EINVAL;
      return launch_z1d<96>(a, g, st, members);
  }
}

}  // namespace pmw

// ============================================================ ensemble ABI ==
namespace {

struct EnsPlan {
  int x_total, z_total;
  int x_k;       // cells per lane of the x waves
  int z_kernel;  // a pmw::ZKernel
  int z_waves;   // of Z_ROWS3
};

int plan_members(const pmw_member* mem, int n, int x_nt, int z_seg, MemberDev* dev,
                 EnsPlan& plan) {
  long long xs = 0, zs = 0, cells = 0, zb4 = 0, zb8 = 0;
  int min_nz = 1 << 30, max_nx = 0;
  for (int q = 0; q < n; ++q) {
    cells += (long long)mem[q].nx * mem[q].nz;
    zb4 += zt_blocks(mem[q].nx, mem[q].nz, 4);
    zb8 += zt_blocks(mem[q].nx, mem[q].nz, 8);
    min_nz = std::min(min_nz, mem[q].nz);
    max_nx = std::max(max_nx, mem[q].nx);
  }
  plan.x_k = pmw::fused_x_cells(x_nt, cells);
  plan.z_kernel = pmw::fused_z_kernel(z_seg, cells, min_nz, max_nx);
  plan.z_waves = zt_waves(min_nz, zb4, zb8);
  for (int q = 0; q < n; ++q) {
    const pmw_member& m = mem[q];
    if (m.nx < 2 || m.nz < 2 || !m.state || !m.state_tmp || !m.state_work ||
        !m.hy_dens_cell || !m.hy_dens_theta_cell || !m.hy_dens_int ||
        !m.hy_dens_theta_int || !m.hy_pressure_int)
      return PMW_EINVAL;
    if (m.state == m.state_tmp || m.state == m.state_work || m.state_tmp == m.state_work)
      return PMW_EALIAS;
    if ((x_nt > 1000 && (long long)m.nz * (m.nx + 12) > (1LL << 30)) ||
        xw_slots(m.nx, m.nz, plan.x_k) > (1LL << 32) - 1024)
      return PMW_EINVAL;
    const int xt = xw_blocks(m.nx, m.nz, plan.x_k);
    int zc, zsg;
    if (plan.z_kernel == pmw::Z_DENSE) {  // zc = the member's blocks, one row of tiles
      if (dense_z_rows(m.nx, m.nz, kZ1Cols) > (1LL << 30)) return PMW_EINVAL;
      zc = dense_z_blocks(m.nx, m.nz, kZ1Cols, 96);
      zsg = 1;
    } else if (plan.z_kernel == pmw::Z_ROWS3) {
      zc = (m.nx + kZtCols - 1) / kZtCols;
      zsg = zt_tiles(m.nz, plan.z_waves);
    } else {
      const int rows = plan.z_kernel == pmw::Z_ONE96 ? 96 - 12 : 32 - 12;
      zc = (m.nx + kZ1Cols - 1) / kZ1Cols;
      zsg = (m.nz + rows - 1) / rows;
    }
    if (dev) {
      MemberDev& d = dev[q];
      d.state = m.state;
      d.tmp = m.state_tmp;
      d.work = m.state_work;
      d.hyc = m.hy_dens_cell;
      d.hytc = m.hy_dens_theta_cell;
      d.hyri = m.hy_dens_int;
      d.hyti = m.hy_dens_theta_int;
      d.hypi = m.hy_pressure_int;
      d.src = m.src_w;
      d.nx = m.nx;
      d.nz = m.nz;
      d.idx = 1.0 / m.dx;
      d.idz = 1.0 / m.dz;
      d.idxl = recip_lo(m.dx, d.idx);
      d.idzl = recip_lo(m.dz, d.idz);
      d.dt1 = m.dt / 3;
      d.dt2 = m.dt / 2;
      d.dt3 = m.dt / 1;
      d.hvx = -kHvBeta * m.dx / (16 * m.dt_full);
      d.hvz = -kHvBeta * m.dz / (16 * m.dt_full);
      d.x_start = (int)xs;
      d.z_start = (int)zs;
      d.x_blocks = xt;
      d.z_ncol = zc;
    }
    xs += xt;
    zs += (long long)zc * zsg;
    if (xs > (1LL << 30) || zs > (1LL << 30)) return PMW_EINVAL;
  }
  plan.x_total = (int)xs;
  plan.z_total = (int)zs;
  return PMW_OK;
}

int ens_tuning(const int* t, int& x_nt, int& z_seg) {
  x_nt = t ? t[1] : 512;
  z_seg = t ? t[2] : 4128;
  if (t && t[0] != 0) return PMW_EINVAL;  // ensembles run the fused kernels only
  if (!pmw::fused_x_tile_ok(x_nt) || !pmw::fused_z_seg_ok(z_seg)) return PMW_EINVAL;
  return PMW_OK;
}

// What a workspace was prepared for: pmw_ensemble_evolve refuses members or
// a tuning other than those (the device descriptors and work-list offsets
// would not match the launches). Kept on the host, keyed by the workspace's
// address, so that checking it needs no device read (a call stays
// capturable in a HIP graph).
struct EnsPrepared {
  int nmembers, x_nt, z_seg, x_total, z_total;
  unsigned long long members_hash;
  bool operator==(const EnsPrepared& o) const {
    return nmembers == o.nmembers && x_nt == o.x_nt && z_seg == o.z_seg &&
           x_total == o.x_total && z_total == o.z_total &&
           members_hash == o.members_hash;
  }
};

std::mutex g_prepared_mu;
std::unordered_map<const void*, EnsPrepared> g_prepared;

// FNV-1a over the member descriptors (plain pointers, ints and doubles with
// no padding between them).
unsigned long long hash_members(const pmw_member* m, int n) {
  const unsigned char* b = reinterpret_cast<const unsigned char*>(m);
  const size_t len = sizeof(pmw_member) * (size_t)n;
  unsigned long long h = 1469598103934665603ULL;
  for (size_t i = 0; i < len; ++i) {
    h ^= b[i];
    h *= 1099511628211ULL;
  }
  return h;
}

EnsPrepared prepared_for(const pmw_member* m, int n, int x_nt, int z_seg,
                         const EnsPlan& plan) {
  return EnsPrepared{n, x_nt, z_seg, plan.x_total, plan.z_total, hash_members(m, n)};
}

inline int ens_per_xcd(int total) { return (total + kNumXcd - 1) / kNumXcd; }

template <int K>
int launch_ens_x(const MemberDev* d, int n, int pass, int total, hipStream_t st) {
  const int per = ens_per_xcd(total);
  k_ens_x<256 * K><<<per * kNumXcd, 64 * kXwWaves, 0, st>>>(d, n, pass, total, per);
  PMW_CHECK_LAUNCH();
  return PMW_OK;
}

int launch_ens_z(const MemberDev* d, int n, int pass, const EnsPlan& plan, hipStream_t st) {
  const int total = plan.z_total, per = ens_per_xcd(total), nb = per * kNumXcd;
  switch (plan.z_kernel) {
    case pmw::Z_ROWS3:
      if (plan.z_waves == 4)
        k_ens_zt1<4, 48><<<nb, 256, 0, st>>>(d, n, pass, total, per);
      else
        k_ens_zt1<8, 96><<<nb, 512, 0, st>>>(d, n, pass, total, per);
      break;
    case pmw::Z_ONE96:
      k_ens_z1<96><<<nb, kZ1Cols * 96, 0, st>>>(d, n, pass, total, per);
      break;
    case pmw::Z_ONE32:
      k_ens_z1<32><<<nb, kZ1Cols * 32, 0, st>>>(d, n, pass, total, per);
      break;
    default:
      k_ens_z1d<96><<<nb, kZ1Cols * 96, 0, st>>>(d, n, pass, total, per);
  }
  PMW_CHECK_LAUNCH();
  return PMW_OK;
}

int launch_ens(int dir, const MemberDev* d, int n, int pass, const EnsPlan& plan,
               hipStream_t st) {
  if (dir == 1) return launch_ens_z(d, n, pass, plan, st);
  return plan.x_k == 1 ? launch_ens_x<1>(d, n, pass, plan.x_total, st)
                       : launch_ens_x<2>(d, n, pass, plan.x_total, st);
}

}  // namespace

extern "C" {

long long pmw_ensemble_workspace_size(int nmembers) {
  if (nmembers < 1) return 0;
  return ((long long)sizeof(MemberDev) + 2 * sizeof(int)) * nmembers;
}

int pmw_ensemble_prepare(const pmw_member* members, int nmembers, const int* tuning,
                         void* workspace, long long workspace_bytes, void* stream) {
  if (!members || nmembers < 1 || !workspace) return PMW_EINVAL;
  if (workspace_bytes < pmw_ensemble_workspace_size(nmembers)) return PMW_ESPACE;
  int x_nt, z_seg;
  int rc = ens_tuning(tuning, x_nt, z_seg);
  if (rc) return rc;
  // descriptors, then the packed x and z start offsets (see member_of)
  const long long bytes = pmw_ensemble_workspace_size(nmembers);
  char* host = new char[bytes];
  MemberDev* dev = reinterpret_cast<MemberDev*>(host);
  for (int q = 0; q < nmembers; ++q) new (&dev[q]) MemberDev();
  EnsPlan plan;
  rc = plan_members(members, nmembers, x_nt, z_seg, dev, plan);
  if (rc == PMW_OK) {
    int* starts = reinterpret_cast<int*>(dev + nmembers);
    for (int q = 0; q < nmembers; ++q) {
      starts[q] = dev[q].x_start;
      starts[nmembers + q] = dev[q].z_start;
    }
    hipStream_t st = (hipStream_t)stream;
    {
      // until the copy has landed the workspace matches no tuning
      std::lock_guard<std::mutex> lock(g_prepared_mu);
      g_prepared.erase(workspace);
    }
    hipError_t e = hipMemcpyAsync(workspace, host, bytes, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) rc = (int)e;
    if (rc == PMW_OK) {
      std::lock_guard<std::mutex> lock(g_prepared_mu);
      g_prepared[workspace] = prepared_for(members, nmembers, x_nt, z_seg, plan);
    }
  }
  delete[] host;
  return rc;
}

int pmw_ensemble_evolve(const pmw_member* members, int nmembers, const int* tuning,
                        const void* workspace, int* reverse_direction, int nsteps,
                        void* stream, double* kernel_ms) {
  if (!members || nmembers < 1 || !workspace || !reverse_direction || nsteps < 0 ||
      nsteps > 100000)
    return PMW_EINVAL;
  int x_nt, z_seg;
  int rc = ens_tuning(tuning, x_nt, z_seg);
  if (rc) return rc;
  EnsPlan plan;
  rc = plan_members(members, nmembers, x_nt, z_seg, nullptr, plan);
  if (rc) return rc;
  {
    std::lock_guard<std::mutex> lock(g_prepared_mu);
    const auto it = g_prepared.find(workspace);
    if (it == g_prepared.end() ||
        !(it->second == prepared_for(members, nmembers, x_nt, z_seg, plan)))
      return PMW_EINVAL;  // not prepared, or prepared for other members / tuning
  }
  const MemberDev* d = (const MemberDev*)workspace;
  hipStream_t st = (hipStream_t)stream;
  hipEvent_t ev[2] = {nullptr, nullptr};
  if (kernel_ms) {
    kernel_ms[0] = kernel_ms[1] = 0.0;
    if (hipEventCreate(&ev[0]) != hipSuccess || hipEventCreate(&ev[1]) != hipSuccess) {
      if (ev[0]) (void)hipEventDestroy(ev[0]);
      return PMW_EINVAL;
    }
  }
  for (int step = 0; step < nsteps && rc == PMW_OK; ++step) {
    const int first = *reverse_direction ? 0 : 1;  // 0 = x, 1 = z
    for (int pass = 0; pass < 2 && rc == PMW_OK; ++pass) {
      const int dir = pass == 0 ? first : 1 - first;
      if (kernel_ms) {
        const hipError_t e = hipEventRecord(ev[0], st);
        if (e != hipSuccess) { rc = (int)e; break; }
      }
      // state_tmp's interior: only the call's last direction keeps its stores
      const int keep_tmp = pass == 1 && step == nsteps - 1;
      rc = launch_ens(dir, d, nmembers, pass | keep_tmp << 1, plan, st);
      if (kernel_ms && rc == PMW_OK) {
        hipError_t e = hipEventRecord(ev[1], st);
        float ms = 0.f;
        if (e == hipSuccess) e = hipEventSynchronize(ev[1]);
        if (e == hipSuccess) e = hipEventElapsedTime(&ms, ev[0], ev[1]);
        if (e != hipSuccess) { rc = (int)e; break; }
        kernel_ms[dir] += ms;
      }
    }
    if (rc == PMW_OK) *reverse_direction = !*reverse_direction;
  }
  if (kernel_ms) {  // measurement only: a failed destroy changes nothing
    (void)hipEventDestroy(ev[0]);
    (void)hipEventDestroy(ev[1]);
  }
  return rc;
}

}  // extern "C"
