// k_rbl.hip -- random-batch lists (RBL): list build, corrected pair force, mean
// removal, energies.
//
//   lists   ComputeRBLNeighboursOnceWorklet, RunWorklet.cpp:906-980
//   force   ComputeNearForceRBLERF(SpecialBonds)Worklet, RunWorklet.cpp:982-1266
//   means   SumRBLCorrForce / SumRBLCorrVirial, ExecutionMD.cpp:663-667
//   energy  ExecutionMD::ComputeLJCoulEnergy, ExecutionMD.cpp:670-750
//
// The list build and the energies walk the (2 nc + 1)^3 stencil around an
// atom's current cell over the binned cells, x offset outermost, z innermost.
// A workgroup takes up to 32 consecutive atoms of a cell, an equal share (of
// at most eight) a wavefront.  The
// stencil's atoms are one stream, staged in LDS for the four wavefronts (a
// cell of an RBL grid, of width rc / nc, holds 8 to 17 atoms, so a lane finds
// its candidate's cell by a search in the stencil's prefix counts), and each
// wavefront tests 64 candidates at a time, one per lane, against each of its
// atoms.  An atom whose current cell is not its binned one (moved by SHAKE
// after the binning) takes a stream of its own over its own stencil.
//
// Bound by the chain behind each distance test (1000 to 2000 candidates an
// atom, of which one in four is kept): the ballots, counts and branches are
// scalar work in series, and the vector ALUs are busy 29 % of the time (28 % in
// the energies).  Sharing the staged candidates among up to 32 atoms, equal
// shares (a cell's 17 atoms as 5 + 4 + 4 + 4) and one ballot per test hold it
// down.  One wavefront over 64 atoms of a cell,
// a candidate at a time, took 276 us (4096 salt atoms) and 593 us (30,000
// water atoms) for the lists, 162 and 1202 us for the energies; this one takes
// 22 and 139 us, 28 and 275 us.  A stream per wavefront, without the shared
// stage, took 50 and 381 us for the lists.
#include "cells.hpp"
#include "dev.hpp"
#include "pair.hpp"
#include "reduce.hpp"
#include "stream.hpp"

namespace rbmd {

constexpr int kRblWaves = kBlock / kWave;
constexpr int kRblAtoms = 8;                                        // atoms per wavefront, at most
constexpr int kRblParts = kChunk / (kRblWaves * kRblAtoms);         // workgroups per 64-atom work item
constexpr int kRblCells = 128;                                      // stencil cells per table (two per lane)
using RblTable = StreamTable<kRblCells>;

// Candidates staged for a workgroup: positions less the image offset, entries
constexpr int kRblStage = 512;
struct RblStage {
  double x[kRblStage], y[kRblStage], z[kRblStage];
  int e[kRblStage];
};

// The candidates around the workgroup's cell in traversal order, staged once
// for its wavefronts: f(live, entry, x, y, z) for 64 of them at a time.  Every
// thread of the workgroup calls this; wavefronts with nothing to do pass busy
// = false and help to stage.
template <class F>
__device__ __forceinline__ void rbl_stream_shared(const SysView& s, int c, bool busy, RblTable& tab, RblStage& stage,
                                                  int* shared_int, F&& f) {
  const int lane = threadIdx.x & (kWave - 1);
  const int ca = c % s.dims[0], cb = (c / s.dims[0]) % s.dims[1], cc = c / (s.dims[0] * s.dims[1]);
  const int wd = 2 * s.nc + 1, cells = wd * wd * wd;
  for (int c0 = 0; c0 < cells; c0 += kRblCells) {
    __syncthreads();  // the last table's reads
    if (threadIdx.x < kWave) {
      bool shifts;
      const int total = stream_table(s, s.nc, ca, cb, cc, c0, tab, 4, shifts);
      if (lane == 0) {
        shared_int[0] = total;
        shared_int[1] = shifts ? 1 : 0;
      }
    }
    __syncthreads();
    const int total = shared_int[0];
    const bool shifts = shared_int[1] != 0;
    for (int base = 0; base < total; base += kRblStage) {
      const int m = min(kRblStage, total - base);
      if (base > 0) __syncthreads();  // the last stage's reads
      for (int t = threadIdx.x; t < m; t += kBlock) {
        const int e = stream_entry(tab, base + t);
        const double4 p = stream_position(s, e, shifts);
        stage.x[t] = p.x;
        stage.y[t] = p.y;
        stage.z[t] = p.z;
        stage.e[t] = e;
      }
      __syncthreads();
      if (busy)
        for (int t0 = 0; t0 < m; t0 += kWave) {
          const int t = t0 + lane;  // past m: an earlier window's candidate, dead
          f(t < m, stage.e[t], stage.x[t], stage.y[t], stage.z[t]);
        }
    }
  }
}

// a wavefront's atoms: the item's cell, its first atom and their number; false
// if the workgroup has none
__device__ __forceinline__ bool rbl_atoms(const SysView& s, int bid, int& c, int& first, int& nmine) {
  const int item_idx = bid / kRblParts;
  if (item_idx >= s.n_items_dev[0]) return false;
  const int item = __builtin_amdgcn_readfirstlane(s.items[item_idx]);
  c = item >> 8;
  const int start = s.cell_start[c] + (item & 255) * kChunk;
  const int m = min(kChunk, s.cell_start[c + 1] - start);  // the item's atoms
  const int parts = (m + kRblWaves * kRblAtoms - 1) / (kRblWaves * kRblAtoms);
  const int shares = parts * kRblWaves;
  const int w = __builtin_amdgcn_readfirstlane((bid % kRblParts) * kRblWaves + threadIdx.x / kWave);
  const int a0 = w * m / shares;
  first = start + a0;
  nmine = w < shares ? (w + 1) * m / shares - a0 : 0;
  return bid % kRblParts < parts;
}

// One atom's list: core slots [0, rs_num), kept shell slots from rs_num, every
// pice_num-th shell atom in traversal order.  The shell atoms of a batch are a
// ballot; among them, the kept ones are those whose prefix count is a set bit
// of the mask of the multiples of pice_num, shifted by the number of shell
// atoms still to pass.
struct RblList {
  int core, kept;
  int wait;  // shell atoms to pass before the next kept one
};
__device__ __forceinline__ unsigned long long rbl_multiples(int pice) {
  unsigned long long m = 0ull;
  for (int r = 0; r < kWave; r += pice) m |= 1ull << r;
  return m;
}
__device__ __forceinline__ void rbl_consider(const SysView& s, RblList& L, int i, int entry, double d2, int pice,
                                             unsigned long long multiples) {
#pragma clang fp contract(off)
  const double e = d2 - s.rs2;  // rs2 - d2 = -e exactly
  const unsigned long long far = __ballot(e > 0.0001);
  const unsigned long long bs = __ballot(d2 <= s.accept_d2) & far;  // cut2 - d2 > 1e-4
  int* const row = s.nbr + nbr_index(0, i, s.cap);
  if (~far != 0ull) {  // wave-uniform
    const unsigned long long bc = __ballot(-e > 0.0001) & __ballot(d2 > 0.0001);
    const int slot = L.core + lanes_below(bc);
    if (lane_in(bc) & (slot < s.rs_num)) row_store(row, slot, entry);
    L.core += __popcll(bc);
  }
  const int num = __popcll(bs);
  if (L.wait < num) {  // wave-uniform; wait < 64 here
    const unsigned long long pick = multiples << L.wait;
    const unsigned long long bk = bs & __ballot((pick >> lanes_below(bs)) & 1ull);
    const int slot = s.rs_num + L.kept + lanes_below(bk);
    if (lane_in(bk) & (slot < s.cap)) row_store(row, slot, entry);
    const int kept = __popcll(bk);
    L.kept += kept;
    L.wait += kept * pice;
  }
  L.wait -= num;
}
__device__ __forceinline__ void rbl_finish(const SysView& s, const RblList& L, int i) {
  if (L.core > s.rs_num || s.rs_num + L.kept > s.cap) atomicOr(s.status, 4);
  s.nbr_num[2 * i] = L.core < s.rs_num ? L.core : s.rs_num;
  s.nbr_num[2 * i + 1] = s.rs_num + L.kept > s.cap ? s.cap - s.rs_num : L.kept;
}

// The first workgroups take the misfit atoms, a wavefront each: a stream by one
// wavefront is the longest chain of the launch, so it starts first.
// As a tail of the workgroup that holds the atom it cost 206 us instead of 149
// at 30,000 water atoms, 5 % of them misfit.
constexpr int kRblMisfitBlocks = 256;
__global__ __launch_bounds__(kBlock) void k_nbr_build_rbl(SysView s) {
#pragma clang fp contract(off)
  __shared__ RblTable tabs[kRblWaves];
  __shared__ RblStage stage;
  __shared__ int shared_int[2];
  const int lane = threadIdx.x & (kWave - 1);
  const int pice = max(abs(s.pice_num), 1);
  const unsigned long long multiples = rbl_multiples(pice);
  if ((int)blockIdx.x < kRblMisfitBlocks) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int count = s.misfit_count[0];
    for (int m = (int)blockIdx.x * kRblWaves + w; m < count; m += kRblMisfitBlocks * kRblWaves) {
      const int i = __builtin_amdgcn_readfirstlane(s.misfit_list[m]);
      const double4 pi = s.spos[i];
      RblList L = {0, 0, 0};
      wave_stream(s, s.nc, cell_axis(pi.x, s.lo[0], s.dxdydz[0]), cell_axis(pi.y, s.lo[1], s.dxdydz[1]),
                 cell_axis(pi.z, s.lo[2], s.dxdydz[2]), tabs[w], 1,
                 [&](bool live, int entry, double x, double y, double z) {
                   if (!live) x = __builtin_nan("");
                   rbl_consider(s, L, i, entry, dist2(x - pi.x, y - pi.y, z - pi.z), pice, multiples);
                 });
      if (lane == 0) rbl_finish(s, L, i);
    }
    return;
  }
  int c, first, nmine;
  if (!rbl_atoms(s, (int)blockIdx.x - kRblMisfitBlocks, c, first, nmine)) return;  // workgroup-uniform
  double4 pi = make_double4(0, 0, 0, 0);
  int mf_l = 0;
  if (lane < nmine) {
    pi = s.spos[first + lane];
    mf_l = s.misfit[first + lane];
  }
  const unsigned fit = (unsigned)__ballot(lane < nmine && mf_l == 0);
  double ax[kRblAtoms], ay[kRblAtoms], az[kRblAtoms];
  RblList L[kRblAtoms];
#pragma unroll
  for (int a = 0; a < kRblAtoms; ++a) {
    // no atom, or a misfit one: no distance to it is accepted
    const double px = __shfl(pi.x, a, kWave);
    ax[a] = (fit >> a) & 1u ? px : __builtin_nan("");
    ay[a] = __shfl(pi.y, a, kWave);  // in vector registers, as the scalar ones are short
    az[a] = __shfl(pi.z, a, kWave);
    L[a] = {0, 0, 0};
  }
  rbl_stream_shared(s, c, fit != 0u, tabs[0], stage, shared_int, [&](bool live, int entry, double x, double y, double z) {
    if (!live) x = __builtin_nan("");
#pragma unroll
    for (int a = 0; a < kRblAtoms; ++a)
      if (a < nmine) rbl_consider(s, L[a], first + a, entry, dist2(x - ax[a], y - ay[a], z - az[a]), pice, multiples);
  });
#pragma unroll
  for (int a = 0; a < kRblAtoms; ++a)
    if (((fit >> a) & 1u) && lane == 0) rbl_finish(s, L[a], first + a);
}

static int rbl_item_blocks(const SysView& s) { return s.n_items * kRblParts; }

void launch_nbr_build_rbl(const SysView& s, hipStream_t st) {
  hipLaunchKernelGGL(k_nbr_build_rbl, dim3(kRblMisfitBlocks + rbl_item_blocks(s)), dim3(kBlock), 0, st, s);
}

// The corrected force of an atom before the mean removal: 16 lanes walk its
// list row, core then shell, and a fixed xor-shuffle tree combines their sums.
// LJ from the core within rs and the shell within rc (hazard Q4), Coulomb with
// the analytic erfc (the Coulomb radial table) or the step table.  The virial
// keeps the reference's assignment of the running-sum force of the last pair
// (hazard Q5): -1/2 r_last x F summed over the list, core and shell apart.
// Gathers bound it; 16 lanes an atom and the table instead of one thread an
// atom with erfc and divisions: 72 -> 8 us at 4096 salt atoms, 181 -> 43 us at
// 30,000 water atoms.
//
// ERFC: the analytic erfc by the Coulomb radial table or, where sqrt(alpha) rc
// is too large for its 32 intervals (SysView::erfc_direct), by the functions
// themselves; or the step table.
enum { kErfcPoly = 0, kErfcStep = 1, kErfcDirect = 2 };
template <bool WEIGHTED, int ERFC, bool VIR>
__global__ __launch_bounds__(kBlock) void k_pair_rbl(SysView s, double* rows) {
#pragma clang fp contract(off)  // the pair vector and d2 rounded as the list build and the oracle round them
  constexpr int L = kMaxLanes;
  __shared__ double teps[kMaxTypes * kMaxTypes], tsig[kMaxTypes * kMaxTypes];
  __shared__ double2 ctab[ERFC == kErfcPoly ? kCoulTab / 2 : 1];
  const int nt = s.ntypes;
  const bool ltab = nt <= kMaxTypes;
  if (ltab)
    for (int k = threadIdx.x; k < nt * nt; k += kBlock) {
      teps[k] = s.eps_ij[k];
      tsig[k] = s.sig6_ij[k];
    }
  if (ERFC == kErfcPoly)
    for (int k = threadIdx.x; k < kCoulTab / 2; k += kBlock) ctab[k] = s.ctab[k];
  __syncthreads();
  const int t = (int)(blockIdx.x * kBlock + threadIdx.x);
  const int i = t / L, sub = t & (L - 1);
  double f[2][3] = {{0, 0, 0}, {0, 0, 0}};
  double4 pi = make_double4(0, 0, 0, 0);
  int num[2] = {0, 0};
  if (i < s.n) {
    pi = s.spos[i];
    const int ti = s.stype[i];
    num[0] = s.nbr_num[2 * i];
    num[1] = s.nbr_num[2 * i + 1];
    int spj[kMaxSpecial];
    double spw[kMaxSpecial];
    if (WEIGHTED) {
      const int id = s.point_ids[i];
      const int b = s.sp_off[id];
      int spn = s.sp_off[id + 1] - b;
      if (spn > kMaxSpecial) {
        atomicOr(s.status, 4);
        spn = kMaxSpecial;
      }
#pragma unroll
      for (int k = 0; k < kMaxSpecial; ++k) {
        spj[k] = k < spn ? s.rank[s.sp_ids[b + k]] : -1;
        spw[k] = k < spn ? s.sp_w[b + k] : 1.0;
      }
    }
    const double pice = (double)s.pice_num;
#pragma unroll
    for (int part = 0; part < 2; ++part) {
      const int* const row = s.nbr + nbr_index(part == 0 ? 0 : s.rs_num, i, s.cap);
      const int m = num[part];
      // entries two ahead, positions one ahead
      int e = sub < m ? row[sub] : 0, en = sub + L < m ? row[sub + L] : 0;
      double4 p = s.spos[e >> kShiftBits];
      int tj = s.stype[e >> kShiftBits];
      for (int k = sub; k < m; k += L) {
        const int e2 = k + 2 * L < m ? row[k + 2 * L] : 0;
        const double4 pn = s.spos[en >> kShiftBits];
        const int tn = s.stype[en >> kShiftBits];
        int j;
        double ox, oy, oz;
        decode(s, e, j, ox, oy, oz);
        double rx = (p.x - ox) - pi.x;
        double ry = (p.y - oy) - pi.y;
        double rz = (p.z - oz) - pi.z;
        min_image(s, rx, ry, rz);
        const double d2 = dist2(rx, ry, rz);
        const bool in = d2 < s.cut2 && d2 > 0.0001;
        if (in) {  // outside, neither term counts
          const int tix = ti * nt + tj;
          const double eps = ltab ? teps[tix] : s.eps_ij[tix];
          const double sig6 = ltab ? tsig[tix] : s.sig6_ij[tix];
          const double qq = pi.w * p.w;
          double w = 1.0;
          if (WEIGHTED) {
#pragma unroll
            for (int u = 0; u < kMaxSpecial; ++u)
              if (spj[u] == j) w = spw[u];
          }
          const double rinv = rsqrt_pos(d2);
          const double rinv2 = rinv * rinv;
          const double sd6 = sig6 * (rinv2 * rinv2 * rinv2);
          const double ljs = w * (-24.0 * eps * (fma(2.0, sd6, -1.0) * sd6) * rinv2);
          double cs;
          if (ERFC == kErfcStep) {
            cs = -qq * gnear_table(sqrt(d2)) * rinv;
          } else if (ERFC == kErfcDirect) {
            cs = -qq * gnear(s.alpha, s.sqrt_alpha, sqrt(d2)) * rinv;
          } else {
            const double fk = (d2 * rinv) * s.ctab_inv_h;
            int kk = (int)fk;
            kk = kk < kCoulM - 1 ? kk : kCoulM - 1;
            cs = -qq * coul_poly<false>(ctab, kk, fk - (double)kk - 0.5) * (rinv2 * rinv);
          }
          const bool lj_on = part == 0 ? d2 < s.rs2 : d2 > s.rs2;
          const bool c_on = part == 0 || !WEIGHTED || d2 > s.rs2;
          double sc = fma(s.qqr2e, c_on ? cs : 0.0, lj_on ? ljs : 0.0);
          if (part == 1) sc *= pice;
          f[part][0] = fma(sc, rx, f[part][0]);
          f[part][1] = fma(sc, ry, f[part][1]);
          f[part][2] = fma(sc, rz, f[part][2]);
        }
        e = en;
        en = e2;
        p = pn;
        tj = tn;
      }
    }
  }
#pragma unroll
  for (int off = 1; off < L; off <<= 1)
#pragma unroll
    for (int part = 0; part < 2; ++part)
#pragma unroll
      for (int d = 0; d < 3; ++d) f[part][d] += __shfl_xor(f[part][d], off, kWave);
  double vals[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (i < s.n && sub == 0) {
    for (int d = 0; d < 3; ++d) vals[d] = f[0][d] + f[1][d];
    s.fnx[i] = vals[0];
    s.fny[i] = vals[1];
    s.fnz[i] = vals[2];
    if (VIR) {
#pragma unroll
      for (int part = 0; part < 2; ++part)
        if (num[part] > 0) {
          int j;
          double ox, oy, oz;
          decode(s, s.nbr[nbr_index((part == 0 ? 0 : s.rs_num) + num[part] - 1, i, s.cap)], j, ox, oy, oz);
          const double4 p = s.spos[j];
          double rx = (p.x - ox) - pi.x;
          double ry = (p.y - oy) - pi.y;
          double rz = (p.z - oz) - pi.z;
          min_image(s, rx, ry, rz);
          vir_add(vals + 3, rx, ry, rz, f[part][0], f[part][1], f[part][2], -0.5);
        }
      for (int k = 0; k < 6; ++k) s.vir_near[(size_t)6 * i + k] = vals[3 + k];
    }
  }
  block_write_row<9>(vals, rows + (size_t)blockIdx.x * 9);
}

// Mean removal of the corrected force (and virial): every workgroup reduces
// the pair kernel's rows (the same order in each) and takes the means off its
// own atoms (one workgroup for the whole system took 20 us at 4096 atoms, 93 us
// at 30,000; this one 4 and 9).
constexpr int kMeanThreads = 1024, kMeanGroups = kMeanThreads / 9;
template <bool VIR>
__global__ __launch_bounds__(kMeanThreads) void k_rbl_mean(SysView s, const double* rows, int nrows) {
#pragma clang fp contract(off)
  __shared__ double part[kMeanGroups][9];
  __shared__ double mean[9];
  const int k = threadIdx.x % 9, g = threadIdx.x / 9;
  if (g < kMeanGroups) {
    double acc = 0.0;
    for (int r = g; r < nrows; r += kMeanGroups) acc += rows[(size_t)r * 9 + k];
    part[g][k] = acc;
  }
  __syncthreads();
  if (threadIdx.x < 9) {
    double acc = 0.0;
    for (int u = 0; u < kMeanGroups; ++u) acc += part[u][threadIdx.x];
    mean[threadIdx.x] = acc / (double)s.n;
  }
  __syncthreads();
  const int i = (int)(blockIdx.x * kMeanThreads + threadIdx.x);
  if (i >= s.n) return;
  s.fnx[i] -= mean[0];
  s.fny[i] -= mean[1];
  s.fnz[i] -= mean[2];
  if (VIR)
    for (int u = 0; u < 6; ++u) s.vir_near[(size_t)6 * i + u] -= mean[3 + u];
}

int rbl_pair_blocks(const SysView& s) { return (int)(((size_t)s.n * kMaxLanes + kBlock - 1) / kBlock); }

void launch_pair_rbl(const SysView& s, hipStream_t st, int virial) {
  const int grid = rbl_pair_blocks(s);
#define RBL_PAIR(W_, E_, V_) hipLaunchKernelGGL((k_pair_rbl<W_, E_, V_>), dim3(grid), dim3(kBlock), 0, st, s, s.rbl_rows)
#define RBL_PAIR_V(W_, E_)                                \
  do {                                                    \
    if (virial) RBL_PAIR(W_, E_, true); else RBL_PAIR(W_, E_, false); \
  } while (0)
#define RBL_PAIR_E(W_)                        \
  do {                                        \
    if (s.erfc_table) RBL_PAIR_V(W_, kErfcStep); else if (s.erfc_direct) RBL_PAIR_V(W_, kErfcDirect); else RBL_PAIR_V(W_, kErfcPoly); \
  } while (0)
  if (s.weighted) RBL_PAIR_E(true); else RBL_PAIR_E(false);
#undef RBL_PAIR_E
#undef RBL_PAIR_V
#undef RBL_PAIR
  const dim3 blocks((s.n + kMeanThreads - 1) / kMeanThreads);
  if (virial)
    hipLaunchKernelGGL(k_rbl_mean<true>, blocks, dim3(kMeanThreads), 0, st, s, s.rbl_rows, grid);
  else
    hipLaunchKernelGGL(k_rbl_mean<false>, blocks, dim3(kMeanThreads), 0, st, s, s.rbl_rows, grid);
}

// Energies.  The reference forms them every RBL step over a full Verlet list
// to rc (ComputeNeighbours over the RBL locator, then
// LJCoulEnergyVerletVirialWorklet RunWorklet.cpp:3145-3221, or
// SpecialLJCoulEnergyVerletWeightVirialWorklet :3047-3143 with special bonds):
// per pair with rc^2 - d^2 > 1e-4, d^2 > 1e-4 on the cell-offset vector, the
// minimum-image vector gives
//   e_lj   += w * 4 eps (s6/d6 - 1) s6/d6 / 2            (ComputePotentialEn_fix)
//   e_coul += qqr2e (q q erfc(sqrt(alpha) r) / 2r - (1 - w) q q / 2r)
// with the analytic erfc at the configured alpha (the Coulomb radial table, or
// erfc itself as in the force pass), not the step table.  No list is stored.  Runs on the steps that form thermo
// sums; its rows also carry the mean-removed RBL virial of each atom.
//
// A wavefront queues the accepted (atom, candidate) pairs of its atoms in LDS
// and evaluates them 64 at a time (one candidate in four is within rc).  What
// a pair's lane needs of its atom is read from LDS as well: the terms run with
// lanes off, where no other lane's register may be read.  PERATOM evaluates
// each atom's pairs of a batch apart, for its sums.
constexpr int kRblQueue = 2 * kWave;
template <bool WEIGHTED, bool PERATOM, bool DIRECT>
__global__ __launch_bounds__(kBlock) void k_rbl_energy(SysView s, double* rows) {
#pragma clang fp contract(off)
  __shared__ RblTable tabs[kRblWaves];
  __shared__ RblStage stage;
  __shared__ int shared_int[2];
  __shared__ double2 qtab[DIRECT ? 1 : kCoulTab / 2];
  __shared__ int2 queue[kRblWaves][kRblQueue];  // atom, entry
  __shared__ double4 atom[kRblWaves][kRblAtoms];
  __shared__ int type[kRblWaves][kRblAtoms];
  __shared__ int spj[kRblWaves][kRblAtoms][kMaxSpecial];
  __shared__ double spw[kRblWaves][kRblAtoms][kMaxSpecial];
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  double vals[kRowPair] = {0, 0, 0, 0, 0, 0, 0, 0};
  int c, first, nmine;
  if (rbl_atoms(s, (int)blockIdx.x, c, first, nmine)) {  // workgroup-uniform
    if (!DIRECT)
      for (int k = threadIdx.x; k < kCoulTab / 2; k += kBlock) qtab[k] = s.ctab[kCoulTab / 2 + k];
    int mf_l = 0;
    if (lane < nmine) {
      atom[w][lane] = s.spos[first + lane];
      type[w][lane] = s.stype[first + lane];
      mf_l = s.misfit[first + lane];
      for (int k = 0; k < 6; ++k) vals[2 + k] = s.vir_near[(size_t)6 * (first + lane) + k];
      if (WEIGHTED) {
        const int id = s.point_ids[first + lane];
        const int b = s.sp_off[id];
        const int spn = min(s.sp_off[id + 1] - b, kMaxSpecial);  // longer lists raise the force pass's flag
        for (int k = 0; k < kMaxSpecial; ++k) {
          spj[w][lane][k] = k < spn ? s.rank[s.sp_ids[b + k]] : -1;
          spw[w][lane][k] = k < spn ? s.sp_w[b + k] : 1.0;
        }
      }
    }
    const int spmax = min(s.sp_max, kMaxSpecial);
    const unsigned fit = (unsigned)__ballot(lane < nmine && mf_l == 0);
    unsigned todo = (unsigned)__ballot(lane < nmine && mf_l != 0);
    double elj = 0.0, ec = 0.0;      // this lane's pairs
    double alj = 0.0, acoul = 0.0;   // PERATOM: lane a, atom a
    int cnt = 0;
    // evaluate the last min(cnt, 64) queued pairs
    auto drain = [&]() __attribute__((always_inline)) {
      wave_sync();
      const int n = min(cnt, kWave);
      cnt -= n;
      const int2 q = queue[w][cnt + (lane < n ? lane : 0)];
      const double4 p = stream_position(s, q.y, true), pa = atom[w][q.x];
      const int j = q.y >> kShiftBits;
      double rx = p.x - pa.x, ry = p.y - pa.y, rz = p.z - pa.z;
      min_image(s, rx, ry, rz);  // MinDistanceVec(p_j, p_i)
      const double d2 = dist2(rx, ry, rz);
      double el = 0.0, eco = 0.0;
      if (lane < n && d2 < s.cut2 && d2 > 0.0001) {
        const int tix = type[w][q.x] * s.ntypes + s.stype[j];
        const double eps = s.eps_ij[tix], s6 = s.sig6_ij[tix];
        const double rinv = rsqrt_pos(d2);
        const double rinv2 = rinv * rinv;
        const double sd6 = s6 * (rinv2 * rinv2 * rinv2);
        el = 0.5 * (4.0 * eps * (sd6 - 1.0) * sd6);
        const double half = 0.5 * (pa.w * p.w) * rinv;
        if (DIRECT) {
          eco = half * erfc(s.sqrt_alpha * sqrt(d2));
        } else {
          const double fk = (d2 * rinv) * s.ctab_inv_h;
          int kk = (int)fk;
          kk = kk < kCoulM - 1 ? kk : kCoulM - 1;
          eco = half * coul_poly<false>(qtab, kk, fk - (double)kk - 0.5);  // qtab: the table's Q half
        }
        if (WEIGHTED) {
          double wt = 1.0;
          for (int u = 0; u < spmax; ++u)
            if (spj[w][q.x][u] == j) wt = spw[w][q.x][u];
          el *= wt;
          eco -= (1.0 - wt) * half;
        }
        eco *= s.qqr2e;
      }
      elj += el;
      ec += eco;
      if (PERATOM) {
        const double u = wave_sum(el), v = wave_sum(eco);
        if (lane == __builtin_amdgcn_readfirstlane(q.x)) {
          alj += u;
          acoul += v;
        }
      }
      wave_sync();
    };
    auto push = [&](int a, double d2, int entry) __attribute__((always_inline)) {
      const unsigned long long b = __ballot(d2 <= s.accept_d2) & __ballot(d2 > 0.0001);
      if (lane_in(b)) queue[w][cnt + lanes_below(b)] = make_int2(a, entry);
      cnt += __popcll(b);
      if (PERATOM ? cnt > 0 : cnt >= kWave) drain();  // wave-uniform
    };
    wave_sync();  // the wavefront's own atoms
    rbl_stream_shared(s, c, fit != 0u, tabs[0], stage, shared_int,
                      [&](bool live, int entry, double x, double y, double z) {
                        if (!live) x = __builtin_nan("");
                        for (int a = 0; a < nmine; ++a) {
                          if (!((fit >> a) & 1u)) continue;  // wave-uniform
                          const double4 pa = atom[w][a];
                          push(a, dist2(x - pa.x, y - pa.y, z - pa.z), entry);
                        }
                      });
    while (todo != 0u) {
      const int a = __builtin_ctz(todo);
      todo &= todo - 1;
      const double4 pa = atom[w][a];
      wave_stream(s, s.nc, cell_axis(pa.x, s.lo[0], s.dxdydz[0]), cell_axis(pa.y, s.lo[1], s.dxdydz[1]),
                 cell_axis(pa.z, s.lo[2], s.dxdydz[2]), tabs[w], 1,
                 [&](bool live, int entry, double x, double y, double z) {
                   if (!live) x = __builtin_nan("");
                   push(a, dist2(x - pa.x, y - pa.y, z - pa.z), entry);
                 });
    }
    if (cnt > 0) drain();
    vals[0] = elj;
    vals[1] = ec;
    if (PERATOM && lane < nmine) {
      s.e_lj[first + lane] = alj;
      s.e_coul[first + lane] = acoul;
    }
  }
  block_write_row<kRowPair>(vals, rows + (size_t)blockIdx.x * kRowPair);
}

int rbl_energy_blocks(const SysView& s) { return rbl_item_blocks(s); }

void launch_rbl_energy(const SysView& s, hipStream_t st, int peratom, double* rows, int* nblocks) {
  const int grid = rbl_energy_blocks(s);
  if (nblocks) *nblocks = grid;
#define RBL_ENERGY(W_, P_, D_) hipLaunchKernelGGL((k_rbl_energy<W_, P_, D_>), dim3(grid), dim3(kBlock), 0, st, s, rows)
#define RBL_ENERGY_D(W_, P_)                                               \
  do {                                                                     \
    if (s.erfc_direct) RBL_ENERGY(W_, P_, true); else RBL_ENERGY(W_, P_, false); \
  } while (0)
  if (s.weighted) {
    if (peratom) RBL_ENERGY_D(true, true); else RBL_ENERGY_D(true, false);
  } else {
    if (peratom) RBL_ENERGY_D(false, true); else RBL_ENERGY_D(false, false);
  }
#undef RBL_ENERGY_D
#undef RBL_ENERGY
}

__global__ __launch_bounds__(kBlock) void k_static_table(const double* dis, double* g, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) g[i] = gnear_table(dis[i]);
}

void launch_static_table(const double* dis, double* g, int n, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_static_table, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, dis, g, n);
}

}  // namespace rbmd
