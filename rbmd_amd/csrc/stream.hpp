// stream.hpp -- the atoms of a cell's stencil as one candidate stream, in
// traversal order (x offset outermost, z innermost, then the cell's sorted
// order): a table of the stencil cells' prefix counts in LDS, in which a lane
// finds the cell of its candidate by a binary search.
#pragma once
#include "cells.hpp"

namespace rbmd {

// Loads from memory that is known to be global: in the packed kernels the
// pointers come out of a table, where the compiler would otherwise use flat
// loads (which wait for LDS accesses and theirs for them)
typedef double StreamD4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ int global_int(const int* p) { return *(const __attribute__((address_space(1))) int*)p; }
__device__ __forceinline__ int global_scalar(const int* p) {  // the same address in all lanes
  return __builtin_amdgcn_readfirstlane(global_int(p));
}
__device__ __forceinline__ double4 global_double4(const double4* p) {
  const StreamD4 v = *(const __attribute__((address_space(1))) StreamD4*)p;
  return make_double4(v.x, v.y, v.z, v.w);
}

// stencil_cell for a grid cell and a step of at most one cell: one wrap at
// most, no division
__device__ __forceinline__ StencilCell stencil_next(const SysView& s, int ca, int cb, int cc, int a, int b, int e) {
  StencilCell t;
  int na = ca + a, nb = cb + b, ne = cc + e;
  t.sa = na < 0 ? 1 : (na >= s.dims[0] ? -1 : 0);
  t.sb = nb < 0 ? 1 : (nb >= s.dims[1] ? -1 : 0);
  t.sc = ne < 0 ? 1 : (ne >= s.dims[2] ? -1 : 0);
  na += t.sa * s.dims[0];
  nb += t.sb * s.dims[1];
  ne += t.sc * s.dims[2];
  const int cell = na + nb * s.dims[0] + ne * s.dims[0] * s.dims[1];
  t.ok = true;
  t.js = global_int(s.cell_start + cell);
  t.je = global_int(s.cell_start + cell + 1);
  return t;
}

template <int N>  // stencil cells of a table (a power of two)
struct StreamTable {
  int pre[N], jb[N], code[N];
};

// The stencil cells c0 .. c0 + N - 1 of half width nc around cell (ca, cb, cc)
// into the table; returns the number of their candidates.  shifts: some image
// offset is not zero; bad: status bit of a stencil cell out of reach.  One
// wavefront.
template <int N, bool INSIDE = false>  // INSIDE: nc is 1 and the cell a cell of the grid
__device__ __forceinline__ int stream_table(const SysView& s, int nc, int ca, int cb, int cc, int c0,
                                            StreamTable<N>& tab, int bad, bool& shifts) {
  constexpr int U = (N + kWave - 1) / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int wd = 2 * nc + 1, cells = wd * wd * wd;
  int js[U], num[U], code[U], sum = 0;
  bool sh = false;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    js[u] = num[u] = 0;
    code[u] = pack_entry(0, 0, 0, 0);
    const int k = c0 + U * lane + u;
    if (U * lane + u < N && k < cells) {
      const StencilCell t = INSIDE ? stencil_next(s, ca, cb, cc, k / 9 - 1, k / 3 % 3 - 1, k % 3 - 1)
                                   : stencil_cell(s, ca, cb, cc, k / (wd * wd) - nc, (k / wd) % wd - nc, k % wd - nc);
      if (t.ok) {
        js[u] = t.js;
        num[u] = t.je - t.js;
        code[u] = pack_entry(0, t.sa, t.sb, t.sc);
      } else {
        atomicOr(s.status, bad);
      }
    }
    sum += num[u];
    sh |= code[u] != pack_entry(0, 0, 0, 0);
  }
  int inc = sum;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int t = __shfl_up(inc, off, kWave);
    if (lane >= off) inc += t;
  }
  int p = inc - sum;
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (U * lane + u < N) {
      tab.pre[U * lane + u] = p;
      tab.jb[U * lane + u] = js[u] - p;
      tab.code[U * lane + u] = code[u];
      p += num[u];
    }
  shifts = __ballot(sh) != 0ull;
  return __builtin_amdgcn_readlane(inc, kWave - 1);
}

// candidate t (0 <= t < total) of a table: its entry
template <int N>
__device__ __forceinline__ int stream_entry(const StreamTable<N>& tab, int t) {
  int k = 0;
#pragma unroll
  for (int step = N / 2; step > 0; step >>= 1) k += tab.pre[k + step] <= t ? step : 0;
  return ((t + tab.jb[k]) << kShiftBits) | tab.code[k];
}

// an entry's position less its image offset (w: charge)
__device__ __forceinline__ double4 stream_position(const SysView& s, int e, bool shifts) {
#pragma clang fp contract(off)
  double4 p = global_double4(s.spos + (e >> kShiftBits));
  if (shifts) {
    p.x -= s.dxdydz[0] * (double)(((e & 7) - 3) * s.dims[0]);
    p.y -= s.dxdydz[1] * (double)((((e >> 3) & 7) - 3) * s.dims[1]);
    p.z -= s.dxdydz[2] * (double)((((e >> 6) & 7) - 3) * s.dims[2]);
  }
  return p;
}

// the same for an entry whose offsets are at most one box: shift_len is the
// product above for an offset of one, and times 1, 0 or -1 exact
__device__ __forceinline__ double4 stream_next_position(const SysView& s, int e) {
#pragma clang fp contract(off)
  double4 p = global_double4(s.spos + (e >> kShiftBits));
  if (__ballot((e & ((1 << kShiftBits) - 1)) != pack_entry(0, 0, 0, 0)) != 0ull) {
    p.x -= (double)((e & 7) - 3) * s.shift_len[0];
    p.y -= (double)(((e >> 3) & 7) - 3) * s.shift_len[1];
    p.z -= (double)(((e >> 6) & 7) - 3) * s.shift_len[2];
  }
  return p;
}

// The stream around one cell for one wavefront: f(live, entry, x, y, z) for 64
// candidates at a time (misfit atoms).
template <int N, class F>
__device__ __forceinline__ void wave_stream(const SysView& s, int nc, int ca, int cb, int cc,
                                            StreamTable<N>& tab, int bad, F&& f) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wd = 2 * nc + 1, cells = wd * wd * wd;
  for (int c0 = 0; c0 < cells; c0 += N) {
    bool shifts;
    wave_sync();  // the last table's reads
    const int total = stream_table(s, nc, ca, cb, cc, c0, tab, bad, shifts);
    wave_sync();
    if (total == 0) continue;
    // the next batch's positions are in flight over this one's tests
    int e = stream_entry(tab, min(lane, total - 1));
    double4 p = stream_position(s, e, shifts);
    for (int base = 0; base < total; base += kWave) {
      const int en = stream_entry(tab, min(base + kWave + lane, total - 1));
      const double4 pn = stream_position(s, en, shifts);
      f(base + lane < total, e, p.x, p.y, p.z);
      e = en;
      p = pn;
    }
  }
}

// the lanes of a ballot below this one
__device__ __forceinline__ int lanes_below(unsigned long long m) {
  return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
}

// this lane's bit of a ballot, as the condition of a branch
__device__ __forceinline__ bool lane_in(unsigned long long m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// slot of a list row (far below 2^32 bytes)
__device__ __forceinline__ void row_store(int* row, int slot, int entry) {
  *(int*)((char*)row + 4u * (unsigned)slot) = entry;
}

}  // namespace rbmd
