// k_stencil.hip -- compact systems (few atoms, where a step's length is a chain
// of launches): the pair forces straight from the cell list, without a stored
// neighbour list, in one launch with the structure factor and the bonded
// forces, and the k-space force in one launch with the second half step.
//
// Steps without thermo sums only.  The forces are those of the list build and
// the pair kernel to the bit: the same entries in the same order, walked by the
// same 16 lanes per atom, so a system may change between the two (the last step
// of a call and packs take the lists).
//
// NS wavefronts (one, or the four of a workgroup) own A consecutive atoms of
// one cell.  The candidates, the atoms of the 27 stencil cells in the
// reference's order, form one stream.  A wavefront takes 64 at a time, one per
// lane: the candidate's FP32 position is loaded once and tested against each
// of the A atoms, whose positions sit in scalar registers; near the thresholds
// the reference's FP64 predicate decides.  Accepted entries go to atom a's
// list in LDS at their ballot prefix.  In rounds that the lists can hold, 16
// lanes per atom then walk them, gather the neighbours' positions and keep
// partial force sums in registers.  No atomics: deterministic sums.
//
// An atom whose current cell is not its binned one (moved by SHAKE after the
// binning) takes a pass of its own over its own stencil.
#include <type_traits>

#include "atoms.hpp"
#include "cells.hpp"
#include "dev.hpp"
#include "kspace.hpp"
#include "pair.hpp"
#include "reduce.hpp"

namespace rbmd {

constexpr int kStWaves = kBlock / kWave;
constexpr int kStLanes = kMaxLanes;  // lanes per atom of the evaluation: the pair kernel's of a compact system

// The choices of (atoms A, wavefronts NS): (1, 4), (2, 4), (4, 4), (4, 1)
__host__ __device__ constexpr int stencil_lga(int cfg) { return cfg < 3 ? cfg : 2; }
__host__ __device__ constexpr int stencil_split(int cfg) { return cfg < 3 ? kStWaves : 1; }
// LDS list slots per wavefront and atom, a whole number of 64-candidate
// batches: 134 neighbours of an ion, a quarter of a water atom's 419
__host__ __device__ constexpr int stencil_cap(int cfg) { return stencil_lga(cfg) == 2 ? 256 : 512; }

typedef __amdgpu_buffer_rsrc_t StRsrc;
typedef double StD2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ StRsrc st_rsrc(const void* p, unsigned bytes) {
  // word 3 of a gfx9 buffer resource: 32-bit data format, untyped loads
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ double4 st_double4(StRsrc r, unsigned off) {
  const StD2 a = __builtin_bit_cast(StD2, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  const StD2 b = __builtin_bit_cast(StD2, __builtin_amdgcn_raw_buffer_load_b128(r, off + 16, 0, 0));
  return make_double4(a.x, a.y, b.x, b.y);
}
__device__ __forceinline__ float4 st_float4(StRsrc r, unsigned off) {
  return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
__device__ __forceinline__ float lane_float(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ int lane_int(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ double lane_double(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}

// LDS list entry: sorted index (19 bits, n at most kStAtoms), type (4 bits),
// image shift + 4 per axis (3 bits each, 1..7 as stencil_cell gives -3..3, so
// an entry is never 0)
constexpr int kStType = 9, kStIdx = kStType + 4, kStZero = 4;
__host__ __device__ __forceinline__ int st_code(int sa, int sb, int sc) {
  return (sa + kStZero) | ((sb + kStZero) << 3) | ((sc + kStZero) << 6);
}
__device__ __forceinline__ int st_shift(int e, int axis) { return ((e >> (3 * axis)) & 7) - kStZero; }

// Stencil cells of every cell of the grid, x offset outermost, then y, then z
// (32 slots a cell, 27 used): the wrapped cell above its image shift code.
std::vector<int> stencil_table(const SysView& s) {
  std::vector<int> tab((size_t)s.ncell * 32, -1);
  for (int c = 0; c < s.ncell; ++c)
    for (int k = 0; k < 27; ++k) {
      int at[3] = {c % s.dims[0] + k / 9 - 1, (c / s.dims[0]) % s.dims[1] + (k / 3) % 3 - 1,
                   c / (s.dims[0] * s.dims[1]) + k % 3 - 1};
      int shift[3];
      for (int d = 0; d < 3; ++d) {
        const int w = (at[d] + s.dims[d]) % s.dims[d];
        shift[d] = (w - at[d]) / s.dims[d];
        at[d] = w;
      }
      tab[(size_t)c * 32 + k] =
          (at[0] + at[1] * s.dims[0] + at[2] * s.dims[0] * s.dims[1]) << kStType | st_code(shift[0], shift[1], shift[2]);
    }
  return tab;
}

template <int MODE, int SP, bool F32, int CFG>
__device__ __forceinline__ void stencil_body(const SysView& s, const int bid) {
#pragma clang fp contract(off)  // fused multiply-adds are written out (see pair_term)
  constexpr int LGA = stencil_lga(CFG), NS = stencil_split(CFG);
  constexpr int A = 1 << LGA, L = kStLanes, CAP = stencil_cap(CFG);
  constexpr int PARTS = kChunk * NS / (kStWaves * A);  // workgroups per 64-atom work item
  constexpr int SPD = SP > 0 ? SP : 1;
  using TT = typename std::conditional<F32, float, double>::type;
  using CT = typename std::conditional<F32, float2, double2>::type;
  constexpr int kTab = (F32 ? kCoulTab32 : kCoulTab) / 2;  // the force half (P) of the Coulomb table
  __shared__ TT teps[kMaxTypes * kMaxTypes], tsig[kMaxTypes * kMaxTypes];
  __shared__ CT ctab[MODE == 2 ? 1 : kTab];
  __shared__ int lists[kStWaves][A][CAP];
  __shared__ int counts[kStWaves][A];
  const int item_idx = bid / PARTS;
  const int part = bid % PARTS;
  if (item_idx >= s.n_items_dev[0]) return;  // workgroup-uniform
  const int item = __builtin_amdgcn_readfirstlane(s.items[item_idx]);
  const int c = item >> 8;
  const int start = s.cell_start[c];
  const int cnt_c = s.cell_start[c + 1] - start;
  const int wg0 = (item & 255) * kChunk + part * (kStWaves / NS) * A;  // the workgroup's first atom within the cell
  if (wg0 >= cnt_c) return;
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int ws = NS == 1 ? 0 : w;  // this wavefront's share of the stream
  const int nt = s.ntypes;
  for (int k = threadIdx.x; k < nt * nt; k += kBlock) {
    teps[k] = (TT)s.eps_ij[k];
    tsig[k] = (TT)s.sig6_ij[k];
  }
  if (MODE != 2) {
    const CT* src;
    if constexpr (F32)
      src = s.ctab32;
    else
      src = s.ctab;
    for (int k = threadIdx.x; k < kTab; k += kBlock) ctab[k] = src[k];
  }
  const int first = NS == 1 ? wg0 + w * A : wg0;
  const int nmine = min(cnt_c - first, A);  // <= 0: none (only with NS = 1)
  const int a_l = lane / L, sub = lane & (L - 1);
  const int i = start + first + a_l;  // this lane's atom
  const bool valid = a_l < nmine;
  double4 pi = make_double4(0, 0, 0, 0);
  float4 p32 = make_float4(0, 0, 0, 0);
  int ti = 0, mf_l = 0;
  int spj[SPD];
  double spw[SPD];
  if (valid) {
    pi = s.spos[i];
    p32 = s.spos32[i];
    ti = __float_as_int(p32.w);
    mf_l = s.misfit[i];
    if (MODE == 1) {
      const int id = s.point_ids[i];
      const int b = s.sp_off[id];
      int spn = s.sp_off[id + 1] - b;
      if (spn > SP) {
        atomicOr(s.status, 4);
        spn = SP;
      }
#pragma unroll
      for (int k = 0; k < SPD; ++k) {
        spj[k] = k < spn ? s.rank[s.sp_ids[b + k]] : -1;
        spw[k] = k < spn ? s.sp_w[b + k] : 1.0;
      }
    }
  }
  __syncthreads();
  const StRsrc rp32 = st_rsrc(s.spos32, 16u * (unsigned)s.n);
  const StRsrc rpos = st_rsrc(s.spos, 32u * (unsigned)s.n);
  // FP32 test of d^2 (the error bound is s.test_band): accepted in
  // (1e-4 + band, hi - band), rejected from hi + band on, else the FP64 predicate
  const float hi_f = (float)s.accept_d2;
  const unsigned in_lo = __float_as_uint(1e-4f + s.test_band);
  const unsigned in_w = __float_as_uint(hi_f - s.test_band) - in_lo;
  const float out_f = hi_f + s.test_band;
  double fx = 0, fy = 0, fz = 0;
  unsigned long long todo = __ballot(valid && mf_l != 0 && sub == 0);  // misfit atoms, a pass each
  bool main_pass = __ballot(valid && mf_l == 0) != 0ull;
  while (main_pass || todo != 0ull) {  // the same passes on every wavefront of NS = 4
    // this pass's atoms and their cell
    int ca, cb, cc, only = -1;
    bool out = false;  // the atom has left the box, by any number of lengths: the FP64 predicate throughout
    if (main_pass) {
      ca = c % s.dims[0];
      cb = (c / s.dims[0]) % s.dims[1];
      cc = c / (s.dims[0] * s.dims[1]);
    } else {
      const int l = __builtin_ctzll(todo);
      todo &= todo - 1;
      only = l / L;
      ca = cell_axis(lane_double(pi.x, l), s.lo[0], s.dxdydz[0]);
      cb = cell_axis(lane_double(pi.y, l), s.lo[1], s.dxdydz[1]);
      cc = cell_axis(lane_double(pi.z, l), s.lo[2], s.dxdydz[2]);
      out = min(ca, min(cb, cc)) < 0 || ca >= s.dims[0] || cb >= s.dims[1] || cc >= s.dims[2];
    }
    main_pass = false;
    // candidates and atoms in FP32 around the cell's centre, both from the
    // FP32 sorted copy: d^2 = (|c|^2 + |a|^2) - 2 c.a
    const float gx = (float)(((double)ca + 0.5) * s.dxdydz[0]);
    const float gy = (float)(((double)cb + 0.5) * s.dxdydz[1]);
    const float gz = (float)(((double)cc + 0.5) * s.dxdydz[2]);
    float mx[A], my[A], mz[A], aa[A];
    {
      const float x = p32.x - gx, y = p32.y - gy, z = p32.z - gz;
      const bool on = valid && (only < 0 ? mf_l == 0 : a_l == only);
      const float h = on ? x * x + y * y + z * z : 1e30f;  // out of every candidate's reach
#pragma unroll
      for (int a = 0; a < A; ++a) {
        mx[a] = lane_float(-2.0f * x, a * L);
        my[a] = lane_float(-2.0f * y, a * L);
        mz[a] = lane_float(-2.0f * z, a * L);
        aa[a] = lane_float(h, a * L);
      }
    }
    // stencil cell `lane` (of 27, x offset outermost, then y, then z):
    // its candidates' first sorted index, count and image shift
    int js = 0, num = 0, code = st_code(0, 0, 0);
    if (only < 0) {
      const int e = s.stencil_tab[c * 32 + (lane & 31)];
      if (lane < 27) {
        js = s.cell_start[e >> kStType];
        num = s.cell_start[(e >> kStType) + 1] - js;
        code = e & ((1 << kStType) - 1);
      }
    } else if (lane < 27) {
      const StencilCell t = stencil_cell(s, ca, cb, cc, lane / 9 - 1, (lane / 3) % 3 - 1, lane % 3 - 1);
      if (t.ok) {
        js = t.js;
        num = t.je - t.js;
        code = st_code(t.sa, t.sb, t.sc);
      } else {
        atomicOr(s.status, 4);
      }
    }
    int pre = num;  // inclusive prefix of the counts
#pragma unroll
    for (int off = 1; off < 32; off <<= 1) {
      const int t = __shfl_up(pre, off, kWave);
      if (lane >= off) pre += t;
    }
    const int total = lane_int(pre, 26);
    const int jb = js - (pre - num);  // sorted index of candidate t of the stream: t + jb
    const bool shifts = __ballot(code != st_code(0, 0, 0)) != 0ull;
    int done = 0;  // this lane's atom: entries evaluated so far
    // rounds of NS x span candidates, wavefront by wavefront in stream order:
    // the whole stream at once, unless that overflows a list, then rounds
    // that cannot
    int span = (total + NS * kWave - 1) / (NS * kWave) * kWave;
    for (int round = 0; round < total;) {
      int base = round + ws * span, kc = 0;
      const int stop = min(total, base + span);
      int cnt[A];
#pragma unroll
      for (int a = 0; a < A; ++a) cnt[a] = 0;
      // the batch at `base`: candidate index and shift of this lane, and its load
      int cj = 0, ccd = 0;
      auto locate = [&]() {
        const int t = base + lane;
        int j = t + lane_int(jb, kc);
        ccd = lane_int(code, kc);
        int end = lane_int(pre, kc);
        while (end < base + kWave && kc < 26) {  // lanes from the next cell's start on take its base and shift
          ++kc;
          const bool sel = t >= end;
          const int jk = lane_int(jb, kc), ck = lane_int(code, kc);
          j = sel ? t + jk : j;
          ccd = sel ? ck : ccd;
          end = lane_int(pre, kc);
        }
        cj = t < stop ? j : -1;
        return st_float4(rp32, 16u * (unsigned)cj);  // past the end: out of the buffer's bounds, zeros
      };
      float4 nxt = make_float4(0, 0, 0, 0);
      if (base < stop) nxt = locate();
      while (base < stop) {
        const float4 c4 = nxt;
        const int j = cj, cd = ccd;
        base += kWave;
        if (base < stop) nxt = locate();  // in flight over this batch's tests
        float cx = c4.x - gx, cy = c4.y - gy, cz = c4.z - gz;
        if (shifts) {
          cx -= (float)st_shift(cd, 0) * s.shift32[0];
          cy -= (float)st_shift(cd, 1) * s.shift32[1];
          cz -= (float)st_shift(cd, 2) * s.shift32[2];
        }
        float c2 = fmaf(cx, cx, fmaf(cy, cy, cz * cz));
        c2 = j < 0 ? 1e30f : c2;
        const int entry = (j << kStIdx) | (__float_as_int(c4.w) << kStType) | cd;
        unsigned long long bal[A], near = out ? ~0ull : 0ull;
#pragma unroll
        for (int a = 0; a < A; ++a) {
          const float d2 = fmaf(cx, mx[a], fmaf(cy, my[a], fmaf(cz, mz[a], c2 + aa[a])));
          bal[a] = __ballot(__float_as_uint(d2) - in_lo < in_w);
          near |= bal[a] ^ __ballot(d2 < out_f);  // accepted implies not rejected
        }
        if (near != 0ull) {  // some lane's decision is the FP64 predicate's (the atom itself among them)
          const double4 pj = st_double4(rpos, 32u * (unsigned)j);
          const double x = pj.x - (double)st_shift(cd, 0) * s.shift_len[0];
          const double y = pj.y - (double)st_shift(cd, 1) * s.shift_len[1];
          const double z = pj.z - (double)st_shift(cd, 2) * s.shift_len[2];
#pragma unroll
          for (int a = 0; a < A; ++a) {
            const double d2 = dist2(x - lane_double(pi.x, a * L), y - lane_double(pi.y, a * L),
                                    z - lane_double(pi.z, a * L));
            const unsigned long long on = __ballot(j >= 0 && aa[a] < 1e29f);
            bal[a] = __ballot(d2 <= s.accept_d2) & __ballot(d2 > 0.0001) & on;
          }
        }
#pragma unroll
        for (int a = 0; a < A; ++a) {
          if ((bal[a] >> lane) & 1ull) {
            const int pos = __builtin_amdgcn_mbcnt_hi((unsigned)(bal[a] >> 32),
                                                      __builtin_amdgcn_mbcnt_lo((unsigned)bal[a], 0));
            lists[w][a][min(cnt[a] + pos, CAP - 1)] = entry;
          }
          cnt[a] += __popcll(bal[a]);
        }
      }
      // this round's lists, walked by the lanes of the wavefront that keeps
      // the atoms' sums: lane `sub` takes the positions sub, sub + L, ... of
      // the atom's whole list
      bool over = false;
      if (NS > 1) {
        if (lane == 0) {
#pragma unroll
          for (int a = 0; a < A; ++a) counts[w][a] = cnt[a];
        }
        __syncthreads();
        for (int u = 0; u < NS; ++u)
#pragma unroll
          for (int a = 0; a < A; ++a) over |= counts[u][a] > CAP;
      } else {
#pragma unroll
        for (int a = 0; a < A; ++a) over |= cnt[a] > CAP;
        wave_sync();
      }
      if (!over && ws == 0 && valid) {
        int num_l[NS], mine = 0;
        if (NS == 1) {
          num_l[0] = cnt[0];
#pragma unroll
          for (int a = 1; a < A; ++a) num_l[0] = a_l == a ? cnt[a] : num_l[0];
          mine = num_l[0];
        } else {
#pragma unroll
          for (int u = 0; u < NS; ++u) {
            num_l[u] = counts[u][a_l];
            mine += num_l[u];
          }
        }
        // entry at position k of the round's lists (0 past the end)
        auto entry_at = [&](int k) -> unsigned {
          if (k >= mine) return 0u;
          int u = NS == 1 ? w : 0;
#pragma unroll
          for (int v = 0; v < NS - 1; ++v) {
            const bool past = u == v && k >= num_l[v];
            k -= past ? num_l[v] : 0;
            u += past ? 1 : 0;
          }
          return (unsigned)lists[u][a_l][k];
        };
        int k = (sub - done) & (L - 1);
        done += mine;
        unsigned ea = entry_at(k), eb = entry_at(k + L);
        double4 pa = st_double4(rpos, 32u * (ea >> kStIdx));
        double4 pb = st_double4(rpos, 32u * (eb >> kStIdx));
        while (ea != 0u) {  // two entries per iteration, positions one iteration ahead
          k += 2 * L;
          const unsigned na = entry_at(k), nb = entry_at(k + L);
          const double4 qa = st_double4(rpos, 32u * (na >> kStIdx));
          const double4 qb = st_double4(rpos, 32u * (nb >> kStIdx));
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const unsigned e = h == 0 ? ea : eb;
            if (e == 0u) continue;
            const double4 p = h == 0 ? pa : pb;
            const double ox = (double)st_shift((int)e, 0) * s.shift_len[0];
            const double oy = (double)st_shift((int)e, 1) * s.shift_len[1];
            const double oz = (double)st_shift((int)e, 2) * s.shift_len[2];
            double rx = (p.x - ox) - pi.x;
            double ry = (p.y - oy) - pi.y;
            double rz = (p.z - oz) - pi.z;
            if (s.use_min_image) min_image(s, rx, ry, rz);
            const double d2 = dist2(rx, ry, rz);
            if (s.use_min_image && !pair_in<1>(s, d2)) continue;  // the force's range, on the minimum image
            const int tix = ti * nt + (int)((e >> kStType) & (kMaxTypes - 1));
            const TT epsij = teps[tix];
            const TT sig6 = tsig[tix];
            double wt = 1.0;
            if (MODE == 1) {
              const int j = (int)(e >> kStIdx);
#pragma unroll
              for (int u = 0; u < SPD; ++u)
                if (spj[u] == j) wt = spw[u];
            }
            double sc;
            if constexpr (F32) {
              float el32, ec32;
              sc = pair_term32<MODE, false, 0>(s, ctab, d2, (float)(pi.w * p.w), epsij, sig6, (float)wt, el32, ec32);
            } else {
              double elj, ec;
              sc = pair_term<MODE, false, 0>(s, ctab, d2, pi.w * p.w, epsij, sig6, wt, elj, ec);
            }
            fx = fma(sc, rx, fx);
            fy = fma(sc, ry, fy);
            fz = fma(sc, rz, fz);
          }
          ea = na;
          eb = nb;
          pa = qa;
          pb = qb;
        }
      }
      if (NS > 1)
        __syncthreads();
      else
        wave_sync();
      if (!over) round += NS * span;
      else span = CAP;
    }
  }
  if (ws != 0) return;
#pragma unroll
  for (int off = 1; off < L; off <<= 1) {
    fx += __shfl_xor(fx, off, kWave);
    fy += __shfl_xor(fy, off, kWave);
    fz += __shfl_xor(fz, off, kWave);
  }
  if (valid && sub == 0) {
    s.fnx[i] = fx;
    s.fny[i] = fy;
    s.fnz[i] = fz;
  }
}

// The pair forces, the structure factor and the bonded forces read the same
// positions and write apart, so they share one launch (the blocks of each one
// after the other); a side stream costs a small system more in events than it
// hides.
template <int MODE, int SP, bool F32, int CFG>
__global__ __launch_bounds__(kBlock, 4) void k_compact_forces(SysView s, IntView iv, KView kv, int n_pair, int kblocks,
                                                           int n_rho) {
  const int bid = (int)blockIdx.x;
  if (bid < n_pair)
    stencil_body<MODE, SP, F32, CFG>(s, bid);
  else if (bid < n_pair + n_rho)
    rho_partial_body<F32, 1>(s, kv, (bid - n_pair) % kblocks, (bid - n_pair) / kblocks);
  else if constexpr (MODE != 2)  // bonds and angles: not for LJ/CUT
    bonded_body<false>(s, iv, nullptr, bid - n_pair - n_rho);
}

template <bool F32>
__global__ __launch_bounds__(kWave << 4) void k_compact_finish(SysView s, IntView iv, KView kv, int has_b,
                                                               double* rows_ke) {
  kforce_body<false, false, F32, 4>(s, kv, nullptr, (int)blockIdx.x);
  if (threadIdx.x < kWave) second_half_wave(s, iv, 1, 1, has_b, rows_ke, (int)blockIdx.x);  // its own lanes' forces
}

// More atoms share each candidate load and the set-up, fewer atoms and a
// split stream give a small system more wavefronts.
int stencil_choice(const SysView& s) {
  const double cand = 27.0 * s.n / s.ncell;  // stencil candidates per atom
  if (cand > 2000) return s.n <= 1000 ? 0 : 1;
  return s.n <= 3000 ? 2 : 3;
}

static int64_t stencil_blocks_of(const SysView& s, int cfg) {
  return s.n_items * (int64_t)(kChunk * stencil_split(cfg) / (kStWaves << stencil_lga(cfg)));
}

// The list build and the pair kernel are two dependent launches whose length
// on a small system is one wavefront's serial work; here that is one launch
// with the work spread over as many wavefronts as help.  The candidate test
// costs more instructions than the list build's, so the rule is on their
// number.  Kernel times (list build + pair kernel against this one, us): salt
// 600 ions 30.4 / 16.4, 2,000 36.7 / 17.9, 4,000 33.5 / 21.7, 8,000 33.0 /
// 29.9; water 600 atoms 118 / 46, 1,800 70 / 51, 3,000 57 / 54, 6,000 mixed
// 77 / 104.
//
// Three lines: on the number of candidates (or, where cells are crowded, of the
// atoms: 3,000 of water are a tie, 57 / 54); on the atoms, as the list build
// has the chip full from about 8,000 on whatever the candidates (steps with
// lists and with this kernel, us: 8,000 ions 70 / 61 at 1,000 candidates, 75 /
// 75 at 216; 14,000 81 / 88 at 519, 84 / 106 at 172; 20,000 89 / 124 at 246);
// and on the workgroups, a fixed number per cell and its atoms, most of them
// empty where a cell holds few: 600 ions in 125 cells 74 / 47, in 729 75 / 82;
// 2,000 in 216 75 / 61, in 512 78 / 82, in 2,197 83 / 183; 4,000 in 1,000 80 /
// 65, in 4,913 91 / 114.
constexpr int kStAtoms = 8000, kStAtomsCrowded = 2400, kStBlocks = 5000;
bool stencil_pays(const SysView& s) {
  const double cand = 27.0 * s.n / s.ncell;
  if (stencil_blocks_of(s, stencil_choice(s)) > kStBlocks) return false;
  return cand > 2000 ? s.n <= kStAtomsCrowded : s.n <= kStAtoms && (double)s.n * cand <= 8e6;
}

int stencil_blocks(const SysView& s) { return (int)stencil_blocks_of(s, s.st_cfg); }

template <int MODE, int SP, bool F32>
void launch_compact_cfg(const SysView& s, const IntView& iv, const KView& k, hipStream_t st, int n_pair, int n_rho,
                        int n_bond) {
  const int kb = (k.P + kWave - 1) / kWave;
#define ST_LAUNCH(CFG_)                                                                                         \
  case CFG_:                                                                                                    \
    hipLaunchKernelGGL((k_compact_forces<MODE, SP, F32, CFG_>), dim3(n_pair + n_rho + n_bond), dim3(kBlock), 0, \
                       st, s, iv, k, n_pair, kb, n_rho);                                                        \
    break;
  switch (s.st_cfg) {
    ST_LAUNCH(0) ST_LAUNCH(1) ST_LAUNCH(2) ST_LAUNCH(3)
  }
#undef ST_LAUNCH
}

template <int MODE, int SP>
void launch_compact_v(const SysView& s, const IntView& iv, const KView& k, hipStream_t st, int n_pair, int n_rho,
                      int n_bond) {
  if (s.mixed)
    launch_compact_cfg<MODE, SP, true>(s, iv, k, st, n_pair, n_rho, n_bond);
  else
    launch_compact_cfg<MODE, SP, false>(s, iv, k, st, n_pair, n_rho, n_bond);
}

void launch_compact_forces(const SysView& s, const IntView& iv, const KView& k, hipStream_t st, int has_k, int has_b) {
  const int np = stencil_blocks(s);
  const int nr = has_k ? (k.P + kWave - 1) / kWave * k.nblk_rho : 0;
  const int nb = has_b ? (s.n + kBlock - 1) / kBlock : 0;
  if (s.lj_only)
    launch_compact_v<2, 0>(s, iv, k, st, np, nr, nb);
  else if (!s.weighted)
    launch_compact_v<0, 0>(s, iv, k, st, np, nr, nb);
  else if (s.sp_max <= 2)
    launch_compact_v<1, 2>(s, iv, k, st, np, nr, nb);
  else if (s.sp_max <= 4)
    launch_compact_v<1, 4>(s, iv, k, st, np, nr, nb);
  else
    launch_compact_v<1, 16>(s, iv, k, st, np, nr, nb);
}

void launch_compact_finish(const SysView& s, const IntView& iv, const KView& k, hipStream_t st, int has_b,
                           double* rows_ke, int* n_ke) {
  const int grid = kforce_blocks(s);
  *n_ke = grid;  // one row per 64 atoms, as launch_second_half
  if (k.f32)
    hipLaunchKernelGGL((k_compact_finish<true>), dim3(grid), dim3(kWave << 4), 0, st, s, iv, k, has_b, rows_ke);
  else
    hipLaunchKernelGGL((k_compact_finish<false>), dim3(grid), dim3(kWave << 4), 0, st, s, iv, k, has_b, rows_ke);
}

}  // namespace rbmd
