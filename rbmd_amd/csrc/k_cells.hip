// k_cells.hip -- cell list (integer counting sort).
//
// Reference: ContPointLocator::Build (framework/locator/ContPointLocator.cxx:70-92)
// bins with BinPointsWorklet (:38-66) and sorts atom ids by cell with a
// comparison SortByKey.  Here binning is a counting sort: per-cell histogram
// with atomics, one exclusive scan, an atomic scatter, then a per-cell rank
// sort that restores the canonical within-cell order (ascending atom id), so
// the result is bit-exact and independent of atomic ordering.
#include "dev.hpp"
#include "pack.hpp"
#include "reduce.hpp"
#include "cells.hpp"

namespace rbmd {

__global__ void k_fill_int(int* p, int v, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
__global__ void k_fill_double(double* p, double v, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

void launch_fill_int(int* p, int v, int n, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill_int, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, p, v, n);
}
void launch_fill_double(double* p, double v, int n, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill_double, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, p, v, n);
}

__global__ __launch_bounds__(kBlock) void k_bin(SysView s, const double* __restrict__ x, const double* __restrict__ y,
                                                const double* __restrict__ z) {
  extern __shared__ int lds_cells[];
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  int cell = -1;
  if (i < s.n) {
    double px = x[i], py = y[i], pz = z[i];
    if (!isfinite(px) || !isfinite(py) || !isfinite(pz)) atomicOr(s.status, 1);
    int a = bin_axis(px, s.lo[0], s.dxdydz[0], s.dims[0]);
    int b = bin_axis(py, s.lo[1], s.dxdydz[1], s.dims[1]);
    int c = bin_axis(pz, s.lo[2], s.dxdydz[2], s.dims[2]);
    cell = a + b * s.dims[0] + c * s.dims[0] * s.dims[1];
    s.cell_of[i] = cell;
  }
  count_cells(s, cell, lds_cells);
}

size_t bin_lds_bytes(const SysView& s) { return s.lds_bins ? (size_t)s.ncell * sizeof(int) : 0; }

// Displacement of a coordinate since the last build, as the minimum image:
// image flags cannot unwrap it (SHAKE re-applies the periodic wrap to
// positions the drift already wrapped, so a flag can count one crossing twice,
// as the reference's does), and between builds every displacement is below
// skin / 2 plus one step's motion, far under half a box edge.
__device__ __forceinline__ double skin_disp(double x, double x0, double box) {
  const double d = x - x0;
  return d - box * rint(d / box);
}

// Skin lists: after the step's positions are final (after SHAKE), flag a
// rebuild when any atom is more than skin / 2 from its position at the last
// build (a non-finite distance counts as moved), and bin every atom with the
// current positions, as the rebuild's scan needs.  On a step without a
// rebuild the scan kernel clears the counts again.  One atomic per wavefront
// that saw a moved atom.
__global__ __launch_bounds__(kBlock) void k_skin_check(SysView s) {
  extern __shared__ int lds_cells[];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  int cell = -1;
  bool moved = false;
  if (i < s.n) {
    const double px = s.x[i], py = s.y[i], pz = s.z[i];
    if (!isfinite(px) || !isfinite(py) || !isfinite(pz)) atomicOr(s.status, 1);
    const double ux = skin_disp(px, s.x0[i], s.box[0]);
    const double uy = skin_disp(py, s.y0[i], s.box[1]);
    const double uz = skin_disp(pz, s.z0[i], s.box[2]);
    moved = !(ux * ux + uy * uy + uz * uz <= s.half_skin2);
    const int a = bin_axis(px, s.lo[0], s.dxdydz[0], s.dims[0]);
    const int b = bin_axis(py, s.lo[1], s.dxdydz[1], s.dims[1]);
    const int c = bin_axis(pz, s.lo[2], s.dxdydz[2], s.dims[2]);
    cell = a + b * s.dims[0] + c * s.dims[0] * s.dims[1];
    s.cell_of[i] = cell;
  }
  if (__ballot(moved) != 0ull && (threadIdx.x & (kWave - 1)) == 0)
    atomicMax((unsigned long long*)s.rebuild_at, (unsigned long long)*s.cur_step);
  count_cells(s, cell, lds_cells);
}

void launch_skin_check(const SysView& s, hipStream_t st) {
  hipLaunchKernelGGL(k_skin_check, dim3((s.n + kBlock - 1) / kBlock), dim3(kBlock), bin_lds_bytes(s), st, s);
}

__global__ void k_skin_request(int64_t* rebuild_at, const int64_t* cur_step, int ahead) {
  if (threadIdx.x == 0) *rebuild_at = *cur_step + ahead;
}

void launch_skin_request(const SysView& s, int ahead, hipStream_t st) {
  hipLaunchKernelGGL(k_skin_request, dim3(1), dim3(kWave), 0, st, s.rebuild_at, s.cur_step, ahead);
}

// a step without a rebuild: the counts binned this step are dropped
__device__ __forceinline__ void clear_counts(const SysView& s) {
  for (int c = threadIdx.x; c < s.ncell; c += blockDim.x) s.cell_count[c] = 0;
}

void launch_bin(const SysView& s, hipStream_t st, const double* x, const double* y, const double* z) {
  hipLaunchKernelGGL(k_bin, dim3((s.n + kBlock - 1) / kBlock), dim3(kBlock), bin_lds_bytes(s), st, s, x, y, z);
}

// block-wide exclusive scan of one int per thread (1024 threads = 16 waves)
__device__ __forceinline__ int block_exclusive_scan(int v, int* lds_wave, int* total) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  int inc = v;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    int t = __shfl_up(inc, off, kWave);
    if (lane >= off) inc += t;
  }
  if (lane == kWave - 1) lds_wave[wave] = inc;
  __syncthreads();
  if (threadIdx.x == 0) {
    int acc = 0;
    int nw = blockDim.x / kWave;
    for (int w = 0; w < nw; ++w) {
      int t = lds_wave[w];
      lds_wave[w] = acc;
      acc += t;
    }
    lds_wave[16] = acc;
  }
  __syncthreads();
  int ex = inc - v + lds_wave[wave];
  *total = lds_wave[16];
  __syncthreads();
  return ex;
}

// Exclusive scan of the cell counts by one workgroup.  With OUT it writes
// cell_start, the work items (cell, 64-atom chunk), the misfit count and the
// item count; with KERNEL (the scan kernel) also cursor = cell_start and the
// counts reset to zero for the next binning.  start (LDS, or null) receives
// every cell's start.
template <bool KERNEL>
__device__ __forceinline__ void cell_scan(const SysView& s, int* start, const bool out) {
  __shared__ int lds[17];
  int carry = 0, icarry = 0;
  for (int base = 0; base < s.ncell; base += blockDim.x) {
    int c = base + threadIdx.x;
    int cnt = c < s.ncell ? s.cell_count[c] : 0;
    int tot;
    int ex = block_exclusive_scan(cnt, lds, &tot);
    if (start && c < s.ncell) start[c] = carry + ex;
    if (out) {  // workgroup-uniform
      int nch = (cnt + kChunk - 1) / kChunk;
      int itot;
      int iex = block_exclusive_scan(nch, lds, &itot);
      if (c < s.ncell) {
        s.cell_start[c] = carry + ex;
        if (KERNEL) {
          s.cursor[c] = carry + ex;
          s.cell_count[c] = 0;
        }
        for (int k = 0; k < nch; ++k) {
          int it = icarry + iex + k;
          if (it < s.n_items) s.items[it] = (c << 8) | (k & 255);
        }
        if (nch > 256) atomicOr(s.status, 4);
      }
      icarry += itot;
    }
    carry += tot;
  }
  if (out && threadIdx.x == 0) {
    s.misfit_count[0] = 0;
    s.cell_start[s.ncell] = carry;
    s.n_items_dev[0] = icarry < s.n_items ? icarry : s.n_items;
    if (icarry > s.n_items) atomicOr(s.status, 4);
  }
}

__device__ __forceinline__ void scan_body(const SysView& s, const int bid) {
  if (!list_rebuild(s)) {
    clear_counts(s);
    return;
  }
  cell_scan<true>(s, nullptr, true);
}

__global__ __launch_bounds__(1024) void k_scan(SysView s) {
  scan_body(s, (int)blockIdx.x);
}

void launch_scan(const SysView& s, hipStream_t st) {
  hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, st, s);
}

// Scatter atom ids into their cells.  With LDS aggregation each workgroup
// reserves one range per cell with a single global atomic and places its atoms
// by their LDS rank; the order inside a cell is fixed afterwards by k_cell_sort.
__device__ __forceinline__ void scatter_body(const SysView& s, const int bid) {
  extern __shared__ int lds[];
  if (!list_rebuild(s)) return;
  int i = bid * blockDim.x + threadIdx.x;
  int cell = i < s.n ? s.cell_of[i] : -1;
  if (!s.lds_bins) {
    if (cell >= 0) s.point_ids[atomicAdd(&s.cursor[cell], 1)] = i;
    return;
  }
  int* cnt = lds;
  int* base = lds + s.ncell;
  for (int c = threadIdx.x; c < s.ncell; c += blockDim.x) cnt[c] = 0;
  __syncthreads();
  int local = cell >= 0 ? atomicAdd(&cnt[cell], 1) : 0;
  __syncthreads();
  for (int c = threadIdx.x; c < s.ncell; c += blockDim.x) {
    int v = cnt[c];
    base[c] = v ? atomicAdd(&s.cursor[c], v) : 0;
  }
  __syncthreads();
  if (cell >= 0) s.point_ids[base[cell] + local] = i;
}

__global__ __launch_bounds__(kBlock) void k_scatter(SysView s) {
  scatter_body(s, (int)blockIdx.x);
}

void launch_scatter(const SysView& s, hipStream_t st) {
  size_t lds = s.lds_bins ? 2 * (size_t)s.ncell * sizeof(int) : 0;
  hipLaunchKernelGGL(k_scatter, dim3((s.n + kBlock - 1) / kBlock), dim3(kBlock), lds, st, s);
}

// Scan and scatter in one launch, for few cells (scan_in_scatter): every
// workgroup scans the cell counts itself (block 0 also writes the scan's
// outputs) and reserves its range in each cell with one atomic on cursor,
// which starts at zero here (the cell sort resets it and the counts).  The
// order inside a cell is fixed afterwards by k_cell_sort, as with k_scatter.
__global__ __launch_bounds__(kBlock) void k_scan_scatter(SysView s) {
  extern __shared__ int lds[];
  int* start = lds;
  int* cnt = lds + s.ncell;
  int* base = cnt + s.ncell;
  const int bid = (int)blockIdx.x;
  if (!list_rebuild(s)) {
    if (bid == 0) clear_counts(s);
    return;
  }
  cell_scan<false>(s, start, bid == 0);
  const int i = bid * blockDim.x + threadIdx.x;
  const int cell = i < s.n ? s.cell_of[i] : -1;
  for (int c = threadIdx.x; c < s.ncell; c += blockDim.x) cnt[c] = 0;
  __syncthreads();
  const int local = cell >= 0 ? atomicAdd(&cnt[cell], 1) : 0;
  __syncthreads();
  for (int c = threadIdx.x; c < s.ncell; c += blockDim.x) {
    const int v = cnt[c];
    base[c] = v ? start[c] + atomicAdd(&s.cursor[c], v) : 0;
  }
  __syncthreads();
  if (cell >= 0) s.point_ids[base[cell] + local] = i;
}

bool scan_in_scatter(const SysView& s) { return s.lds_bins && s.ncell <= kScanScatterCells; }

void launch_scan_scatter(const SysView& s, hipStream_t st) {
  hipLaunchKernelGGL(k_scan_scatter, dim3((s.n + kBlock - 1) / kBlock), dim3(kBlock),
                     3 * (size_t)s.ncell * sizeof(int), st, s);
}

constexpr int kSortCap = 4096;

// One workgroup per cell: rank each id by the number of smaller ids in the
// cell, then write the atom's sorted copies at its sorted position p: x, y, z,
// q, type, and the misfit flag (the current position lies in a different
// cell than the binned one: possible after SHAKE moves atoms, or at x == hi,
// where binning clamps and InWhichCell does not).  Runs after the step's
// positions are final.
__device__ __forceinline__ void cell_sort_body(const SysView& s, const int bid) {
  __shared__ int4 quads[kSortCap / 4];
  int* const ids = (int*)quads;
  if (!list_rebuild(s)) {
    // skin list between builds: the build's sorted order is kept; the sorted
    // copy of each position is its build position plus its displacement, so
    // a list entry's image offset still applies
    const int stride = s.ncell * blockDim.x;
    for (int p = bid * blockDim.x + threadIdx.x; p < s.n; p += stride) {
      const int me = s.point_ids[p];
      const double x0 = s.x0[me], y0 = s.y0[me], z0 = s.z0[me];
      s.spos[p] = make_double4(x0 + skin_disp(s.x[me], x0, s.box[0]), y0 + skin_disp(s.y[me], y0, s.box[1]),
                               z0 + skin_disp(s.z[me], z0, s.box[2]), s.q[me]);
    }
    return;
  }
  int c = bid;
  // the same in all lanes, which a packed kernel's table does not tell
  const int start = __builtin_amdgcn_readfirstlane(s.cell_start[c]);
  const int cnt = __builtin_amdgcn_readfirstlane(s.cell_start[c + 1]) - start;
  if (threadIdx.x == 0) {  // read by the binning and scatter kernels before this one
    s.cell_count[c] = 0;
    s.cursor[c] = 0;
    if (c == 0 && s.list_builds) atomicAdd(s.list_builds, 1);
  }
  // A cell of more is refused by the status flag, but its atoms keep valid
  // copies, in the scatter's order: later kernels index by rank and type.
  const bool sorts = cnt <= kSortCap;
  if (!sorts && threadIdx.x == 0) atomicOr(s.status, 4);
  const int nq = sorts ? (cnt + 3) / 4 : 0;
  for (int t = threadIdx.x; t < 4 * nq; t += blockDim.x) ids[t] = t < cnt ? s.point_ids[start + t] : 0x7fffffff;
  __syncthreads();
  const int a = c % s.dims[0];
  const int b = (c / s.dims[0]) % s.dims[1];
  const int e = c / (s.dims[0] * s.dims[1]);
  for (int t = threadIdx.x; t < cnt; t += blockDim.x) {
    const int me = sorts ? ids[t] : s.point_ids[start + t];
    int r = sorts ? 0 : t;  // four ids a read: one a read took 29 us for a cell of 600, this 17
#pragma unroll 8
    for (int k = 0; k < nq; ++k) {
      const int4 v = quads[k];
      r += (v.x < me) + (v.y < me) + (v.z < me) + (v.w < me);
    }
    const int p = start + r;
    s.point_ids[p] = me;
    s.rank[me] = p;
    const double px = s.x[me], py = s.y[me], pz = s.z[me];
    s.spos[p] = make_double4(px, py, pz, s.q[me]);
    const int type = s.type[me];
    s.stype[p] = type;
    if (s.spos32)
      s.spos32[p] = make_float4((float)(px - s.lo[0]), (float)(py - s.lo[1]), (float)(pz - s.lo[2]),
                                __int_as_float(type));
    if (s.skin_on) {  // the build's positions, for the skin check and the gathers until the next build
      s.x0[me] = px;
      s.y0[me] = py;
      s.z0[me] = pz;
    }
    const int ua = cell_axis(px, s.lo[0], s.dxdydz[0]);
    const int ub = cell_axis(py, s.lo[1], s.dxdydz[1]);
    const int uc = cell_axis(pz, s.lo[2], s.dxdydz[2]);
    const int mf = (ua != a || ub != b || uc != e) ? 1 : 0;
    s.misfit[p] = mf;
    if (mf) s.misfit_list[atomicAdd(s.misfit_count, 1)] = p;
  }
}

__global__ __launch_bounds__(kBlock) void k_cell_sort(SysView s) {
  cell_sort_body(s, (int)blockIdx.x);
}

void launch_cell_sort(const SysView& s, hipStream_t st) {
  hipLaunchKernelGGL(k_cell_sort, dim3(s.ncell), dim3(kBlock), 0, st, s);
}

// ------------------------------------------------------------------ packs

__global__ __launch_bounds__(1024) void kp_scan(PACK_PARAMS) {
  PACK_ENTRY(e, bid)
  scan_body(e.v, bid);
}

__global__ __launch_bounds__(kBlock) void kp_scatter(PACK_PARAMS) {
  PACK_ENTRY(e, bid)
  scatter_body(e.v, bid);
}

__global__ __launch_bounds__(kBlock) void kp_cell_sort(PACK_PARAMS) {
  PACK_ENTRY(e, bid)
  cell_sort_body(e.v, bid);
}

void launch_pack_cells(int kernel, const PackLaunch& L, int nblocks, size_t lds, hipStream_t st) {
  if (nblocks <= 0) return;
  const dim3 grid(nblocks);
  switch (kernel) {
    case PK_SCAN:
      hipLaunchKernelGGL(kp_scan, grid, dim3(1024), 0, st, PACK_ARGS(L));
      break;
    case PK_SCATTER:
      hipLaunchKernelGGL(kp_scatter, grid, dim3(kBlock), lds, st, PACK_ARGS(L));
      break;
    case PK_CELL_SORT:
      hipLaunchKernelGGL(kp_cell_sort, grid, dim3(kBlock), 0, st, PACK_ARGS(L));
      break;
    case PK_NBR:
      launch_pack_list(L, nblocks, st);
      break;
    default:
      break;
  }
}

}  // namespace rbmd
