// k_kspace.hip -- random-batch Ewald structure factor and k-space force.
//
// rho(k_l) = sum_i q_i (cos k_l.r_i, sin k_l.r_i)
//   ComputePnumberChargeStructureFactorWorklet + ReduceByKey (RunWorklet.cpp:2209-2291,
//   ExecutionMD.cpp:469-501).  The reference writes a P x N scratch and reduces it by
//   key; here each thread folds 4 atoms, the workgroup reduces with wavefront
//   shuffles (no atomics), and a second pass sums the per-workgroup partials in
//   a fixed order.
// F_i = (S/P) sum_l -(4 pi q_i / (V k_l^2)) (cos(k.r) Im rho - sin(k.r) Re rho) k_l, x qqr2e
//   ComputeNewRBEForceWorklet (RunWorklet.cpp:2086-2141), ComputeRBEForceSum_fix
//   (ExecForceFunction.h:748-762), ComputeKspaceVirial (:397-410), UnitRescale
//   (ExecutionNVT.cpp:718).  (The Ewald sum over a kmax grid: k_ewald.hip.)
#include "dev.hpp"
#include "pack.hpp"
#include "reduce.hpp"
#include "cells.hpp"
#include "sincos.hpp"
#include "kspace.hpp"

namespace rbmd {

// k-vector blocks on x (a converged Ewald grid has millions), atom blocks on y
template <bool F32, int KB>
__global__ __launch_bounds__(kBlock) void k_rho_partial(SysView s, KView kv) {
  rho_partial_body<F32, KB>(s, kv, (int)blockIdx.x, (int)blockIdx.y);
}

int rho_kblocks(const SysView& s, int P) { return (P + kWave * s.rho_kb - 1) / (kWave * s.rho_kb); }

int rho_atoms_per_block(int n, int kblocks) {
  int a = 1024;
  while (a > 64 && (long)kblocks * ((n + a - 1) / a) < 2048) a >>= 1;
  return a;
}

// instantiate F(F32, KB) for the tile choice kb (1, 2 or 4 k vectors per lane)
#define RHO_DISPATCH(kb, f32, F)                 \
  do {                                           \
    if ((kb) == 1) {                             \
      if (f32) F(true, 1); else F(false, 1);     \
    } else if ((kb) == 4) {                      \
      if (f32) F(true, 4); else F(false, 4);     \
    } else {                                     \
      if (f32) F(true, 2); else F(false, 2);     \
    }                                            \
  } while (0)

// rho[t] = sum over the partial rows b of rho_part[b][t].  One workgroup per
// kRedCols columns (64 bytes of a row); row group g of its kRedGroups sums
// rows g, g + kRedGroups, ... (independent loads, in flight together), and the
// groups' sums are added in a fixed order.  With 64 columns and 16 groups the
// 400 columns of 30,000 atoms were 7 workgroups of 30 loads a thread: 13.5 us,
// now 7 (99,000 atoms: 33 and 12).  Four wavefronts, not more: the kernel runs
// beside the list build, whose small workgroups leave no room for 1024 threads
// at once (a pack's launch then waited 98 us for it).
constexpr int kRedCols = 8;
constexpr int kRedWaves = 4;
constexpr int kRedGroups = kRedWaves * kWave / kRedCols;

__device__ __forceinline__ void rho_reduce_body(const SysView& s, const KView& kv, const int bid) {
#pragma clang fp contract(off)
  __shared__ double part[kRedGroups][kRedCols];
  const int col = threadIdx.x % kRedCols;
  const int g = threadIdx.x / kRedCols;
  const int n2 = 2 * kv.P;
  const int t = bid * kRedCols + col;
  double acc = 0.0;
  if (t < n2) {
#pragma unroll 8
    for (int b = g; b < kv.nblk_rho; b += kRedGroups) acc += kv.rho_part[(size_t)b * n2 + t];
  }
  part[g][col] = acc;
  __syncthreads();
  if (threadIdx.x < kWave) {  // eight threads a column, four groups each, and a fixed tree
    constexpr int per = kRedGroups * kRedCols / kWave;
    double r = 0.0;
    for (int v = 0; v < per; ++v) r += part[g * per + v][col];
#pragma unroll
    for (int off = kRedCols; off < kWave; off <<= 1) r += __shfl_xor(r, off);
    if (t < n2 && g == 0) kv.rho[t] = r;
    // Im rho from the odd neighbour lane (2P is even: both lanes of a pair
    // are in range or both out); the whole wavefront takes part
    const double r_im = __shfl_xor(r, 1);
    if (kv.krec && t < n2 && !(t & 1) && g == 0) {
      KRec& rec = kv.krec[t >> 1];
      const int l = t >> 1;
      const double kx = kv.kvec[3 * l], ky = kv.kvec[3 * l + 1], kz = kv.kvec[3 * l + 2];
      const double k2 = kx * kx + ky * ky + kz * kz;
      const double pre = 1.0 / (s.volume * k2);
      rec.kx = kx;
      rec.ky = ky;
      rec.kz = kz;
      rec.pre = pre;
      rec.mx = k_to_m(kx, s.box[0]);
      rec.my = k_to_m(ky, s.box[1]);
      rec.mz = k_to_m(kz, s.box[2]);
      rec.rr = kv.f32 ? pre * r : r;
      rec.ri = kv.f32 ? pre * r_im : r_im;
      rec.pad = 0.0;
    }
  }
}

__global__ __launch_bounds__(kRedWaves * kWave) void k_rho_reduce(SysView s, KView kv) {
  rho_reduce_body(s, kv, (int)blockIdx.x);
}

// the k vectors of the current step (device step counter) from the
// double-buffered ring [2][R][3P] into a fixed buffer (step graphs read it)
__device__ __forceinline__ void kvec_slot_body(double* dst, const double* ring, int R, int per, const int64_t* step,
                                               const int bid, const int nblk) {
  const int64_t st = *step;
  const size_t slot = (size_t)((st / R) % 2) * R + (size_t)(st % R);
  for (int t = bid * blockDim.x + threadIdx.x; t < per; t += nblk * blockDim.x) dst[t] = ring[slot * per + t];
}

__global__ __launch_bounds__(kBlock) void k_kvec_slot(double* dst, const double* ring, int R, int per,
                                                      const int64_t* step) {
  kvec_slot_body(dst, ring, R, per, step, (int)blockIdx.x, (int)gridDim.x);
}

void launch_kvec_slot(double* dst, const double* ring, int R, int per, const int64_t* step, hipStream_t st) {
  hipLaunchKernelGGL(k_kvec_slot, dim3((per + kBlock - 1) / kBlock), dim3(kBlock), 0, st, dst, ring, R, per, step);
}

void launch_rho_partial(const SysView& s, const KView& k, hipStream_t st) {
  dim3 grid(rho_kblocks(s, k.P), k.nblk_rho);
#define RHO_LAUNCH(F32_, KB_) hipLaunchKernelGGL((k_rho_partial<F32_, KB_>), grid, dim3(kBlock), 0, st, s, k)
  RHO_DISPATCH(s.rho_kb, k.f32, RHO_LAUNCH);
#undef RHO_LAUNCH
}

void launch_rho_reduce(const SysView& s, const KView& k, hipStream_t st) {
  hipLaunchKernelGGL(k_rho_reduce, dim3((2 * k.P + kRedCols - 1) / kRedCols), dim3(kRedWaves * kWave), 0, st, s, k);
}

template <bool THERMO, bool PERATOM, bool F32, int LG>
__global__ __launch_bounds__(kWave << LG) void k_kforce(SysView s, KView kv, double* rows) {
  kforce_body<THERMO, PERATOM, F32, LG>(s, kv, rows, (int)blockIdx.x);
}

int kforce_blocks(const SysView& s) { return (s.n + kWave - 1) / kWave; }

template <bool THERMO, bool PERATOM, bool F32>
void launch_kforce_lg(const SysView& s, const KView& k, hipStream_t st, double* rows, int grid) {
  if (s.k_lanes_lg == 4)
    hipLaunchKernelGGL((k_kforce<THERMO, PERATOM, F32, 4>), dim3(grid), dim3(kWave << 4), 0, st, s, k, rows);
  else if (s.k_lanes_lg == 1)
    hipLaunchKernelGGL((k_kforce<THERMO, PERATOM, F32, 1>), dim3(grid), dim3(kWave << 1), 0, st, s, k, rows);
  else if (s.k_lanes_lg == 3)
    hipLaunchKernelGGL((k_kforce<THERMO, PERATOM, F32, 3>), dim3(grid), dim3(kWave << 3), 0, st, s, k, rows);
  else
    hipLaunchKernelGGL((k_kforce<THERMO, PERATOM, F32, 2>), dim3(grid), dim3(kWave << 2), 0, st, s, k, rows);
}

void launch_kforce(const SysView& s, const KView& k, hipStream_t st, int thermo, int peratom, double* rows,
                   int* nblocks) {
  int grid = kforce_blocks(s);
  if (nblocks) *nblocks = grid;
  if (k.f32) {
    if (peratom)
      launch_kforce_lg<true, true, true>(s, k, st, rows, grid);
    else if (thermo)
      launch_kforce_lg<true, false, true>(s, k, st, rows, grid);
    else
      launch_kforce_lg<false, false, true>(s, k, st, rows, grid);
    return;
  }
  if (peratom)
    launch_kforce_lg<true, true, false>(s, k, st, rows, grid);
  else if (thermo)
    launch_kforce_lg<true, false, false>(s, k, st, rows, grid);
  else
    launch_kforce_lg<false, false, false>(s, k, st, rows, grid);
}

// ------------------------------------------------------------------ packs

__global__ __launch_bounds__(kBlock) void kp_kvec_slot(PACK_PARAMS) {
  PACK_ENTRY(e, bid)
  kvec_slot_body(const_cast<double*>(e.kv.kvec), e.kring, e.ring_R, 3 * e.kv.P, &e.nhc->step, bid, PACK_GRID());
}

template <bool F32, int KB>
__global__ __launch_bounds__(kBlock) void kp_rho_partial(PACK_PARAMS) {
  PACK_ENTRY(e, bid)
  const int kb = (e.kv.P + kWave * KB - 1) / (kWave * KB);  // k-vector blocks (rho_kblocks)
  rho_partial_body<F32, KB>(e.v, e.kv, bid % kb, bid / kb);
}

__global__ __launch_bounds__(kRedWaves * kWave) void kp_rho_reduce(PACK_PARAMS) {
  PACK_ENTRY(e, bid)
  rho_reduce_body(e.v, e.kv, bid);
}

template <bool F32, int LG, bool THERMO>
__global__ __launch_bounds__(kWave << LG) void kp_kforce(PACK_PARAMS) {
  PACK_ENTRY(e, bid)
  kforce_body<THERMO, false, F32, LG>(e.v, e.kv, e.rows_k, bid);
}

void launch_pack_kspace(int kernel, const PackLaunch& L, int nblocks, const PackSig& g, hipStream_t st) {
  if (nblocks <= 0) return;
  const dim3 grid(nblocks);
  switch (kernel) {
    case PK_KSLOT:
      hipLaunchKernelGGL(kp_kvec_slot, grid, dim3(kBlock), 0, st, PACK_ARGS(L));
      break;
    case PK_RHO:
#define KP_RHO_LAUNCH(F32_, KB_) hipLaunchKernelGGL((kp_rho_partial<F32_, KB_>), grid, dim3(kBlock), 0, st, PACK_ARGS(L))
      RHO_DISPATCH(g.rho_kb, g.f32, KP_RHO_LAUNCH);
#undef KP_RHO_LAUNCH
      break;
    case PK_RHO_RED:
      hipLaunchKernelGGL(kp_rho_reduce, grid, dim3(kRedWaves * kWave), 0, st, PACK_ARGS(L));
      break;
    case PK_KFORCE:
    case PK_KFORCE_C:
#define KP_KF_LAUNCH(F32_, LG_)                                                                    \
  do {                                                                                             \
    if (g.thermo)                                                                                  \
      hipLaunchKernelGGL((kp_kforce<F32_, LG_, true>), grid, dim3(kWave << LG_), 0, st, PACK_ARGS(L));  \
    else                                                                                           \
      hipLaunchKernelGGL((kp_kforce<F32_, LG_, false>), grid, dim3(kWave << LG_), 0, st, PACK_ARGS(L)); \
  } while (0)
      if (kernel == PK_KFORCE_C) {
        if (g.f32) KP_KF_LAUNCH(true, 4); else KP_KF_LAUNCH(false, 4);
      } else if (g.k_lanes_lg == 1) {
        if (g.f32) KP_KF_LAUNCH(true, 1); else KP_KF_LAUNCH(false, 1);
      } else if (g.k_lanes_lg == 3) {
        if (g.f32) KP_KF_LAUNCH(true, 3); else KP_KF_LAUNCH(false, 3);
      } else {
        if (g.f32) KP_KF_LAUNCH(true, 2); else KP_KF_LAUNCH(false, 2);
      }
#undef KP_KF_LAUNCH
      break;
    default:
      break;
  }
}

// The grid of each kernel of the step for one system, as its own launches
// size it (k_first_half .. k_rattle above and in the other kernel files).
int pack_blocks(const SysView& s, const IntView& iv, int P, int kernel) {
  const int atoms = (s.n + kBlock - 1) / kBlock;
  const int mols = (iv.nmol + kBlock - 1) / kBlock;
  switch (kernel) {
    case PK_NHC:
    case PK_SCAN:
    case PK_ONE:
      return 1;
    case PK_KSLOT:
      return (3 * P + kBlock - 1) / kBlock;
    case PK_FIRST_HALF:
    case PK_SCATTER:
    case PK_BONDED:
    case PK_SECOND:
    case PK_ATOMS:
      return atoms;
    case PK_CELL_SORT:
      return s.ncell;
    case PK_SHAKE:
    case PK_RATTLE:
      return mols;
    case PK_NBR:
      return list_blocks(s);
    case PK_PAIR:
      return pair_blocks(s);
    case PK_RHO:
      return rho_kblocks(s, P) * ((s.n + rho_atoms_per_block(s.n, rho_kblocks(s, P)) - 1) /
                                  rho_atoms_per_block(s.n, rho_kblocks(s, P)));
    case PK_RHO_RED:
      return (2 * P + kRedCols - 1) / kRedCols;
    case PK_KFORCE:
    case PK_KFORCE_C:
      return (kernel == PK_KFORCE_C) == (s.compact != 0) ? kforce_blocks(s) : 0;
    default:
      return 0;
  }
}

}  // namespace rbmd
