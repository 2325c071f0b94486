// k_list.hip -- VERLET neighbour lists (ComputeNeighboursWorklet): for each
// atom the entries of the 27 stencil cells within the list cutoff, in
// traversal order (x offset outermost, then y, then z, then the cell's sorted
// order), as one row.
//
// A workgroup takes up to 32 atoms of a cell, an equal share of at most eight
// a wavefront.  The stencil's candidates are read once: those farther than the
// cutoff from the atoms' bounding box are dropped, the rest staged in LDS in
// stream order, in FP32 relative to the cell's centre.  Each wavefront then
// tests 64 staged candidates at a time, one per lane, against its atoms: the
// squared distances |a|^2 - 2 a.c + |c|^2 of four atoms and 64 candidates are
// four 4x4x1 matrix instructions of 16 blocks (block b, column j: candidate
// 4 b + j, so lane l holds candidate l; row v of the result: atom v), which
// leaves the vector unit the range test and the append.  Accepted lanes store
// their entries side by side at the row's count plus the ballot prefix.
//
// Bound by instruction issue at 300,000 atoms (vector ALUs 77 % busy, the matrix
// instructions beside them): 15 slots per atom and 64 candidates (four of the
// matrix instructions per group of four atoms, 3 for the range and band tests,
// 7 to append).  At 30,000 they are 38 % busy: the latency of the chain from
// the cell to the first test, with few wavefronts in flight.  A lane per atom over LDS-staged
// candidates, 9 stencil columns apart, took 48 us at 12,000 water atoms, 60 at
// 30,000, 355 at 300,000 and 79 at 99,000 ions; this one 40, 55, 268 and 64,
// and one row per atom instead of nine segments takes the pair kernel from 63
// to 54, from 440 to 355 and from 70 to 55 us.  Four atoms a wavefront instead
// of eight: 35, 56, 312 and 82 us.
//
// Everything the wavefront's control flow depends on is read as a scalar: in
// the packed kernel the compiler took the counts for lane values and ran the
// loops under lane masks (118 us a launch for 16 water systems, 78 without).
//
// FP32 decides where it is clear of the thresholds by more than its error;
// otherwise the batch is decided by the FP64 predicate on the build's own
// vector (rc^2 - d^2 > 1e-4 and d^2 > 1e-4).
#include "dev.hpp"
#include "pack.hpp"
#include "stream.hpp"

namespace rbmd {

constexpr int kListWaves = kBlock / kWave;
constexpr int kListGroups = 2;                                 // four-atom groups of a wavefront
constexpr int kListAtoms = 4 * kListGroups;                    // atoms per wavefront, at most
constexpr int kListWork = kListWaves * kListAtoms;             // atoms per workgroup, at most
constexpr int kListParts = kChunk / kListWork;                 // workgroups per 64-atom work item
constexpr int kListWindow = 1024;                              // candidates staged at a time
constexpr int kListRounds = kListWindow / kBlock;
constexpr int kListMisfitMax = 1024;
typedef float F4 __attribute__((ext_vector_type(4)));
using ListTable = StreamTable<32>;                             // 27 cells

// workgroups for the misfit atoms (moved out of their binned cell by SHAKE),
// one at a time: first in the grid, as their chains are long
__host__ __device__ __forceinline__ int list_misfit_blocks(const SysView& s) {
  const int b = (s.n + 63) / 64;
  return b < kListMisfitMax ? b : kListMisfitMax;
}

int list_blocks(const SysView& s) { return list_misfit_blocks(s) + kListParts * s.n_items; }

__device__ __forceinline__ void list_finish(const SysView& s, int i, int cnt) {
  if (cnt > s.cap) atomicOr(s.status, 4);
  s.nbr_num[i] = min(cnt, s.cap);
}

__device__ __forceinline__ void list_body(const SysView& s, const int bid) {
#pragma clang fp contract(off)
  // 64 slots past the window pad the last batch
  __shared__ float sx[kListWindow + kWave], sy[kListWindow + kWave], sz[kListWindow + kWave];
  __shared__ int se[kListWindow + kWave];
  __shared__ ListTable tabs[kListWaves];
  __shared__ int kept[kListWaves], candidates;
  __shared__ float box[6];
  if (!list_rebuild(s)) return;  // skin list between builds
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int misfit_blocks = list_misfit_blocks(s);
  const double cut2 = s.list_cut2;  // rc^2, or (rc + skin)^2 for a skin list
  if (bid < misfit_blocks) {
    // One misfit atom at a time: the stream in windows, a quarter of a window
    // per wavefront, accepted entries gathered in LDS and copied to the row in
    // wavefront order.  (Stores to the row between the loads would make each
    // load wait for them.)
    const int count = global_scalar(s.misfit_count);
    int* const got = w == 0 ? (int*)sx : w == 1 ? (int*)sy : w == 2 ? (int*)sz : se;
    for (int m = bid; m < count; m += misfit_blocks) {
      const int i = global_scalar(s.misfit_list + m);
      const double4 pi = global_double4(s.spos + i);
      int* const row = s.nbr + nbr_index(0, i, s.cap);
      bool shifts;
      const int total = stream_table(s, 1, cell_axis(pi.x, s.lo[0], s.dxdydz[0]),
                                     cell_axis(pi.y, s.lo[1], s.dxdydz[1]), cell_axis(pi.z, s.lo[2], s.dxdydz[2]), 0,
                                     tabs[w], 4, shifts);
      wave_sync();
      int done = 0;  // entries of the windows before this one
      for (int base = 0; base < total; base += kListWaves * kListWindow) {
        const int span = min(total - base, kListWaves * kListWindow);
        const int quarter = (span + kListWaves * kWave - 1) / (kListWaves * kWave) * kWave;  // at most kListWindow
        const int t1 = base + min(span, (w + 1) * quarter);
        int n = 0;
        for (int t0 = base + w * quarter; t0 < t1; t0 += kListRounds * kWave) {
          double4 p[kListRounds];
          int e[kListRounds];
#pragma unroll
          for (int r = 0; r < kListRounds; ++r) {
            e[r] = stream_entry(tabs[w], min(t0 + r * kWave + lane, total - 1));
            p[r] = stream_position(s, e[r], shifts);
          }
#pragma unroll
          for (int r = 0; r < kListRounds; ++r) {
            const double d2 = dist2(p[r].x - pi.x, p[r].y - pi.y, p[r].z - pi.z);
            const unsigned long long b = __ballot(t0 + r * kWave + lane < t1) & __ballot(cut2 - d2 > 0.0001) &
                                         __ballot(d2 > 0.0001);
            if (lane_in(b)) got[n + lanes_below(b)] = e[r];
            n += __popcll(b);
          }
        }
        if (lane == 0) kept[w] = n;
        __syncthreads();
        int at = done;
        for (int v = 0; v < kListWaves; ++v) {
          at += v < w ? kept[v] : 0;
          done += kept[v];
        }
        for (int k = lane; k < n; k += kWave)
          if (at + k < s.cap) row[at + k] = got[k];
        __syncthreads();  // before the counts and the table are written again
      }
      if (threadIdx.x == 0) list_finish(s, i, done);
    }
    return;
  }
  const int wid = bid - misfit_blocks;
  if (wid / kListParts >= global_scalar(s.n_items_dev)) return;
  const int item = global_scalar(s.items + wid / kListParts);
  const int c = item >> 8;
  const int start = global_scalar(s.cell_start + c);
  const int cnt_c = global_scalar(s.cell_start + c + 1) - start;
  // the cell's atoms over its workgroups, and a workgroup's over its wavefronts
  const int g = (item & 255) * kListParts + wid % kListParts;
  const int parts = (cnt_c + kListWork - 1) / kListWork;
  if (g >= parts) return;
  const int shares = parts * kListWaves;
  const int wg0 = (int)((long)g * kListWaves * cnt_c / shares);
  const int wgn = (int)((long)(g + 1) * kListWaves * cnt_c / shares) - wg0;
  const int a0 = (int)((long)(g * kListWaves + w) * cnt_c / shares);
  const int nmine = (int)((long)(g * kListWaves + w + 1) * cnt_c / shares) - a0;
  const int first = start + a0;
  const int ca = c % s.dims[0], cb = (c / s.dims[0]) % s.dims[1], cc = c / (s.dims[0] * s.dims[1]);
  const double gx = s.lo[0] + (ca + 0.5) * s.dxdydz[0];
  const double gy = s.lo[1] + (cb + 0.5) * s.dxdydz[1];
  const double gz = s.lo[2] + (cc + 0.5) * s.dxdydz[2];
  // the workgroup's atoms (at most 32), one per lane
  bool fit = false;
  float x = 0, y = 0, z = 0;
  if (lane < wgn) {
    const double4 p = global_double4(s.spos + start + wg0 + lane);
    fit = global_int(s.misfit + start + wg0 + lane) == 0;
    x = (float)(p.x - gx);
    y = (float)(p.y - gy);
    z = (float)(p.z - gz);
  }
  const unsigned long long fits = __ballot(fit);
  if (fits == 0ull) return;  // the same in all wavefronts
  if (w == 0) {  // the stencil
    bool sh;
    const int t = stream_table<32, true>(s, 1, ca, cb, cc, 0, tabs[0], 4, sh);
    if (lane == 0) candidates = t;
  } else if (w == 1) {  // the atoms' bounding box
    float bl[3] = {fit ? x : 3e38f, fit ? y : 3e38f, fit ? z : 3e38f};
    float bh[3] = {fit ? x : -3e38f, fit ? y : -3e38f, fit ? z : -3e38f};
#pragma unroll
    for (int off = 1; off < kListWork; off <<= 1)
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        bl[d] = fminf(bl[d], __shfl_xor(bl[d], off, kWave));
        bh[d] = fmaxf(bh[d], __shfl_xor(bh[d], off, kWave));
      }
    if (lane == 0)
      for (int d = 0; d < 3; ++d) {
        box[d] = bl[d];
        box[3 + d] = bh[d];
      }
  }
  __syncthreads();
  const int total = __builtin_amdgcn_readfirstlane(candidates);
  float bl[3], bh[3], ra2 = 0.0f;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    bl[d] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(box[d])));
    bh[d] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(box[3 + d])));
    const float m = fmaxf(fabsf(bl[d]), fabsf(bh[d]));
    ra2 += m * m;
  }
  // Error of the FP32 d^2 near the cutoff, u = 2^-24, S the largest |a| + |c|:
  // rounded coordinates move it by 2 u S^2, |c|^2 and |a|^2 by 3 u S^2, the
  // four sums by 4 u S^2 (8 if products are rounded apart); 32 u S^2 is more
  // than twice that.  A box so large that the band is not small, or an rc so
  // near 0.01 that nothing lies clear of both thresholds, takes the FP64
  // predicate throughout.
  const float cutf = (float)cut2;
  const float span = 2.0f * sqrtf(ra2) + sqrtf(cutf);
  const float band = 0x1p-19f * (span * span);
  const float cut_m = (float)(cut2 - 0.0001);
  const bool narrow = band < 0.05f * cutf && cut_m - band > 1e-4f + 2.0f * band;
  const unsigned in_lo = __float_as_uint(1e-4f + 2.0f * band);
  const unsigned in_w = __float_as_uint(cut_m - band) - in_lo;
  const float out_f = cut_m + band;
  const float keep_f = cutf + band;  // box cull: its own FP32 error is within the band too
  // this wavefront's atoms as rows of the matrix products: lane l holds atom
  // l % 4 of each group; |a|^2 of row v in register v, no reach for a row
  // without an atom or with a misfit one
  float mx[kListGroups], my[kListGroups], mz[kListGroups];
  F4 aa[kListGroups];
#pragma unroll
  for (int u = 0; u < kListGroups; ++u) {
    const int at = a0 - wg0 + 4 * u + (lane & 3);  // at most 3 past the workgroup's last
    const bool on = 4 * u + (lane & 3) < nmine && ((fits >> at) & 1ull);
    const float ax = __shfl(x, at, kWave), ay = __shfl(y, at, kWave), az = __shfl(z, at, kWave);
    mx[u] = on ? -2.0f * ax : 0.0f;
    my[u] = on ? -2.0f * ay : 0.0f;
    mz[u] = on ? -2.0f * az : 0.0f;
    const float h = on ? ax * ax + ay * ay + az * az : 1e30f;
#pragma unroll
    for (int v = 0; v < 4; ++v) aa[u][v] = __shfl(h, v, kWave);
  }
  const unsigned long long mine = fits >> (a0 - wg0);
  // the wavefront's rows as a buffer, and where each atom's next entry goes
  // (bytes)
  const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
      s.nbr + nbr_index(0, first, s.cap), (short)0, (int)(4u * (unsigned)s.cap * (unsigned)nmine), 0x00020000);
  unsigned at4[kListAtoms];
#pragma unroll
  for (int a = 0; a < kListAtoms; ++a) at4[a] = 4u * a * (unsigned)s.cap;

  for (int base = 0; base < total; base += kListWindow) {
    // this wavefront's quarter of the window: loads back to back
    const int t0 = base + w * (kListWindow / kListWaves) + lane;
    double4 p[kListRounds];
    int e[kListRounds];
#pragma unroll
    for (int r = 0; r < kListRounds; ++r) {
      e[r] = stream_entry(tabs[0], min(t0 + r * kWave, total - 1));
      p[r] = stream_next_position(s, e[r]);
    }
    unsigned long long keep[kListRounds];
    float px[kListRounds], py[kListRounds], pz[kListRounds];
    int mykept = 0;
#pragma unroll
    for (int r = 0; r < kListRounds; ++r) {
      px[r] = (float)(p[r].x - gx);
      py[r] = (float)(p[r].y - gy);
      pz[r] = (float)(p[r].z - gz);
      const float dx = fmaxf(0.0f, fmaxf(bl[0] - px[r], px[r] - bh[0]));
      const float dy = fmaxf(0.0f, fmaxf(bl[1] - py[r], py[r] - bh[1]));
      const float dz = fmaxf(0.0f, fmaxf(bl[2] - pz[r], pz[r] - bh[2]));
      keep[r] = __ballot(dx * dx + dy * dy + dz * dz < keep_f) & __ballot(t0 + r * kWave < total);
      mykept += __popcll(keep[r]);
    }
    if (lane == 0) kept[w] = mykept;
    __syncthreads();  // the counts; the last window's reads of the stage
    int at = 0, m = 0;
#pragma unroll
    for (int v = 0; v < kListWaves; ++v) {
      const int k = __builtin_amdgcn_readfirstlane(kept[v]);
      at += v < w ? k : 0;
      m += k;
    }
#pragma unroll
    for (int r = 0; r < kListRounds; ++r) {
      if (lane_in(keep[r])) {
        const int slot = at + lanes_below(keep[r]);
        sx[slot] = px[r];
        sy[slot] = py[r];
        sz[slot] = pz[r];
        se[slot] = e[r];
      }
      at += __popcll(keep[r]);
    }
    if (w == kListWaves - 1) {  // out of every atom's reach
      sx[m + lane] = 1e15f;
      sy[m + lane] = sz[m + lane] = 0.0f;
      se[m + lane] = 0;
    }
    __syncthreads();
    if (nmine == 0) continue;
    // the next batch's reads are in flight over this one's tests
    float nx = sx[lane], ny = sy[lane], nz = sz[lane];
    int ne = se[lane];
    for (int b = 0; b < m; b += kWave) {
      const float qx = nx, qy = ny, qz = nz;
      const int entry = ne;
      const int nb = min(b + kWave, m) + lane;  // the padding after the last batch
      nx = sx[nb];
      ny = sy[nb];
      nz = sz[nb];
      ne = se[nb];
      const float q2 = qx * qx + qy * qy + qz * qz;
      F4 d[kListGroups];
#pragma unroll
      for (int u = 0; u < kListGroups; ++u) d[u] = __builtin_amdgcn_mfma_f32_4x4x1f32(mx[u], qx, aa[u], 0, 0, 0);
#pragma unroll
      for (int u = 0; u < kListGroups; ++u) d[u] = __builtin_amdgcn_mfma_f32_4x4x1f32(my[u], qy, d[u], 0, 0, 0);
#pragma unroll
      for (int u = 0; u < kListGroups; ++u) d[u] = __builtin_amdgcn_mfma_f32_4x4x1f32(mz[u], qz, d[u], 0, 0, 0);
#pragma unroll
      for (int u = 0; u < kListGroups; ++u) d[u] = __builtin_amdgcn_mfma_f32_4x4x1f32(1.0f, q2, d[u], 0, 0, 0);
      unsigned long long bal[kListAtoms], near = narrow ? 0ull : ~0ull;
#pragma unroll
      for (int a = 0; a < kListAtoms; ++a) {
        const float v = d[a / 4][a % 4];
        bal[a] = __ballot(__float_as_uint(v) - in_lo < in_w);
        near |= bal[a] ^ __ballot(v < out_f);  // accepted implies not rejected
      }
      if (__builtin_expect(near != 0ull, 0)) {
        // some lane's decision is the FP64 predicate's, unless it is an atom itself
        near = narrow ? 0ull : ~0ull;
#pragma unroll
        for (int a = 0; a < kListAtoms; ++a)
          near |= (bal[a] ^ __ballot(d[a / 4][a % 4] < out_f)) & ~__ballot(entry == pack_entry(first + a, 0, 0, 0));
        if (near != 0ull) {
          const bool live = b + lane < m;
          const double4 pj = stream_next_position(s, live ? entry : pack_entry(0, 0, 0, 0));
#pragma unroll
          for (int a = 0; a < kListAtoms; ++a) {
            if (a >= nmine) break;  // wave-uniform
            const double4 pi = global_double4(s.spos + first + a);
            const double d2 = dist2(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z);
            bal[a] = (mine >> a) & 1ull ? __ballot(cut2 - d2 > 0.0001) & __ballot(d2 > 0.0001) & __ballot(live) : 0ull;
          }
          // no load of this path is in flight past it: the wait for one in the
          // common path would wait for every store of a list entry before it
          __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
        }
      }
      // lanes that did not accept store past the buffer's end, where nothing is
      // written.  A list longer than its row (flagged below and not used) runs
      // into the next rows of the wavefront, but no further.
#pragma unroll
      for (int a = 0; a < kListAtoms; ++a) {
        const unsigned off = 4u * (unsigned)lanes_below(bal[a]) + at4[a];
        __builtin_amdgcn_raw_buffer_store_b32((unsigned)entry, rows, lane_in(bal[a]) ? off : 0xfffffff0u, 0, 0);
        at4[a] += 4u * (unsigned)__popcll(bal[a]);
      }
    }
  }
#pragma unroll
  for (int a = 0; a < kListAtoms; ++a)
    if (a < nmine && ((mine >> a) & 1ull) && lane == 0) list_finish(s, first + a, (int)((at4[a] - 4u * a * (unsigned)s.cap) / 4u));
}

__global__ __launch_bounds__(kBlock) void k_nbr_build_verlet(SysView s) { list_body(s, (int)blockIdx.x); }

void launch_nbr_build(const SysView& s, hipStream_t st) {
  if (s.rbl)
    launch_nbr_build_rbl(s, st);
  else
    hipLaunchKernelGGL(k_nbr_build_verlet, dim3(list_blocks(s)), dim3(kBlock), 0, st, s);
}

__global__ __launch_bounds__(kBlock) void kp_nbr_build(PACK_PARAMS) {
  PACK_ENTRY(e, bid)
  list_body(e.v, bid);
}

void launch_pack_list(const PackLaunch& L, int nblocks, hipStream_t st) {
  if (nblocks > 0) hipLaunchKernelGGL(kp_nbr_build, dim3(nblocks), dim3(kBlock), 0, st, PACK_ARGS(L));
}

}  // namespace rbmd
