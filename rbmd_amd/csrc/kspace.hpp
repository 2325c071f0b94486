// kspace.hpp -- the structure-factor and k-space force bodies shared by their
// own kernels, the packed kernels and the fused launches of compact systems.
#pragma once
#include "cells.hpp"
#include "dev.hpp"
#include "reduce.hpp"
#include "sincos.hpp"

namespace rbmd {

// e^{i k.r} with k = 2 pi m / L is e^{2 pi i t} with the phase t = m.(r/L) in
// turns (several hundred radians at |m| ~ 30): sincos_turns_table reduces it
// exactly to a 64th of a turn and a remainder before its polynomials, so no
// large-argument reduction is needed (its table is copied to LDS: the lanes'
// entries differ).  Against sincos_turns: structure factor and force 17.8 + 23.7
// -> 13.7 + 15.3 us at 30,000 atoms x 200 vectors, 112 + 121 -> 76 + 83 us at
// 100,000 x 667.  F32 (mixed
// precision): the phase reduced exactly in FP64 to at most 1/2 turn, rounded
// to FP32, and the hardware sin / cos (sincos_turns32_hw, |error| <= 1.2e-7);
// the phase, the reduction and every sum stay FP64.
template <bool F32>
__device__ __forceinline__ void phase_sincos(double mx, double my, double mz, double sx, double sy, double sz,
                                             const double* turn, double* sn, double* cs) {
#pragma clang fp contract(off)
  const double t = fma(mz, sz, fma(my, sy, mx * sx));
  if constexpr (F32) {
    float s32, c32;
    sincos_turns32_hw(t, &s32, &c32);
    *sn = s32;
    *cs = c32;
  } else {
    sincos_turns_table(t, turn, sn, cs);
  }
}

// the workgroup's copy of the table (a barrier follows before its use)
__device__ __forceinline__ void load_turns(double* turn) {
  for (int k = threadIdx.x; k < 2 * kTurns; k += blockDim.x) turn[k] = kTurnTable[k];
}

// m = k L / (2 pi), an integer held in k to ~1e-13: the product with the
// reciprocal rounds to the same integer as the quotient
__device__ __forceinline__ double k_to_m(double k, double box) { return rint(k * box * (0.5 / kPi)); }

// Structure factor partials.  One workgroup: kWave * KB k vectors (KB per
// lane, a tile choice, SysView::rho_kb) against kv.rho_atoms atoms (64 to
// 1024, by system size: rho_atoms_per_block), which its kBlock / kWave
// wavefronts split into contiguous ranges.
// The lanes of a wavefront take the same atom at the same time, so the atom
// is wave-uniform and comes through scalar loads; the wavefronts' partial
// sums are added in wavefront order and written as row ba of rho_part.
// bk: block of k vectors, ba: block of atoms.
template <bool F32, int KB>
__device__ __forceinline__ void rho_partial_body(const SysView& s, const KView& kv, const int bk, const int ba) {
#pragma clang fp contract(off)  // fused multiply-adds are written out: the same rounding in every kernel
  constexpr int NW = kBlock / kWave;
  __shared__ double part[NW][2 * KB][kWave];
  __shared__ __attribute__((aligned(16))) double turn[F32 ? 2 : 2 * kTurns];
  if constexpr (!F32) {
    load_turns(turn);
    __syncthreads();
  }
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int kb0 = bk * kWave * KB;
  double mx[KB], my[KB], mz[KB], re[KB], im[KB];
#pragma unroll
  for (int t = 0; t < KB; ++t) {
    const int l = kb0 + t * kWave + lane;
    const bool ok = l < kv.P;
    mx[t] = ok ? k_to_m(kv.kvec[3 * l], s.box[0]) : 0.0;
    my[t] = ok ? k_to_m(kv.kvec[3 * l + 1], s.box[1]) : 0.0;
    mz[t] = ok ? k_to_m(kv.kvec[3 * l + 2], s.box[2]) : 0.0;
    re[t] = im[t] = 0.0;
  }
  const double ibx = 1.0 / s.box[0], iby = 1.0 / s.box[1], ibz = 1.0 / s.box[2];
  if constexpr (F32) {
    // mixed precision: the phase as (m / L).r, so the atom's coordinates are
    // not scaled per atom (a change of ~1e-15 turns in the phase)
#pragma unroll
    for (int t = 0; t < KB; ++t) {
      mx[t] *= ibx;
      my[t] *= iby;
      mz[t] *= ibz;
    }
  }
  const int per = kv.rho_atoms / NW;
  const int a0 = ba * kv.rho_atoms + w * per;
  const int a1 = a0 + per < s.n ? a0 + per : s.n;
  // constant address space: wave-uniform scalar loads (positions and charges
  // are not written during this kernel)
  typedef const __attribute__((address_space(4))) double const_double;
  const const_double* X = (const const_double*)s.x;
  const const_double* Y = (const const_double*)s.y;
  const const_double* Z = (const const_double*)s.z;
  const const_double* Q = (const const_double*)s.q;
#pragma unroll 2
  for (int i = a0; i < a1; ++i) {
    const double sx = F32 ? X[i] : X[i] * ibx, sy = F32 ? Y[i] : Y[i] * iby, sz = F32 ? Z[i] : Z[i] * ibz;
    const double q = Q[i];
#pragma unroll
    for (int t = 0; t < KB; ++t) {
      double sn, cs;
      phase_sincos<F32>(mx[t], my[t], mz[t], sx, sy, sz, turn, &sn, &cs);
      re[t] = fma(q, cs, re[t]);
      im[t] = fma(q, sn, im[t]);
    }
  }
#pragma unroll
  for (int t = 0; t < KB; ++t) {
    part[w][2 * t][lane] = re[t];
    part[w][2 * t + 1][lane] = im[t];
  }
  __syncthreads();
  if (w == 0) {
#pragma unroll
    for (int t = 0; t < KB; ++t) {
      const int l = kb0 + t * kWave + lane;
      if (l < kv.P) {
        double a = part[0][2 * t][lane], b = part[0][2 * t + 1][lane];
        for (int u = 1; u < NW; ++u) {
          a += part[u][2 * t][lane];
          b += part[u][2 * t + 1][lane];
        }
        kv.rho_part[(size_t)ba * 2 * kv.P + 2 * l] = a;
        kv.rho_part[(size_t)ba * 2 * kv.P + 2 * l + 1] = b;
      }
    }
  }
}

// Force pass.  One workgroup: 64 atoms (one per lane) against all P k
// vectors, split into KS = 2^LG contiguous ranges, one per wavefront (a tile
// choice, SysView::k_lanes_lg).  The lanes of a wavefront take the same k
// vector at the same time, so its record (KRec) is wave-uniform and comes
// through scalar loads; nothing of k passes through LDS.  The wavefronts'
// partial sums are added in wavefront order.
template <bool THERMO, bool PERATOM, bool F32, int LG>
__device__ __forceinline__ void kforce_body(const SysView& s, const KView& kv, double* rows, const int bid) {
#pragma clang fp contract(off)  // fused multiply-adds are written out: the same forces with or without the virial sums
  constexpr int KS = 1 << LG;
  constexpr int NX = PERATOM ? 9 : 3;  // per-atom sums the wavefronts hand over
  __shared__ double part[KS][NX][kWave];
  __shared__ __attribute__((aligned(16))) double turn[F32 ? 2 : 2 * kTurns];
  if constexpr (!F32) {
    load_turns(turn);
    __syncthreads();
  }
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int i = bid * kWave + lane;
  const bool act = i < s.n;
  double x = 0, y = 0, z = 0, q = 0, sx = 0, sy = 0, sz = 0;
  if (act) {
    x = s.x[i];
    y = s.y[i];
    z = s.z[i];
    q = s.q[i];
    sx = x * (1.0 / s.box[0]);
    sy = y * (1.0 / s.box[1]);
    sz = z * (1.0 / s.box[2]);
  }
  const double q4 = -4.0 * kPi * q;
  double fx = 0, fy = 0, fz = 0;
  double v[6] = {0, 0, 0, 0, 0, 0};
  const int per = (kv.P + KS - 1) / KS;
  const int l0 = w * per;
  const int l1 = l0 + per < kv.P ? l0 + per : kv.P;
  // constant address space: wave-uniform scalar loads (the records are not
  // written during this kernel)
  typedef const __attribute__((address_space(4))) KRec const_krec;
  const const_krec* rec = (const const_krec*)kv.krec;
  if constexpr (F32) {
    // Mixed precision: the term's coefficient pre Im rho cos - pre Re rho sin
    // from the record's products (FP64, so that the forces still sum to zero
    // over the atoms: sum_i q_i (a cos_i - b sin_i) = a Re rho - b Im rho
    // cancels only for a / b = Im rho / Re rho), the sums in FP64 and the
    // atom's -4 pi q applied to them.  The virial terms
    // (x k_a + x k_a) fs summed over k are 2 x F_a (and x F_b + y F_a off the
    // diagonal), formed from the wavefront's sums.  Two records per
    // iteration: their scalar loads are in flight together.
#pragma unroll 2
    for (int l = l0; l < l1; ++l) {
      const double t = fma(rec[l].mz, sz, fma(rec[l].my, sy, rec[l].mx * sx));
      float sn, cs;
      sincos_turns32_hw(t, &sn, &cs);
      const double g = fma((double)cs, rec[l].ri, -((double)sn * rec[l].rr));
      fx = fma(g, rec[l].kx, fx);
      fy = fma(g, rec[l].ky, fy);
      fz = fma(g, rec[l].kz, fz);
    }
    fx = q4 * fx;
    fy = q4 * fy;
    fz = q4 * fz;
    if (THERMO || PERATOM) {
      v[0] = (x + x) * fx;
      v[1] = (y + y) * fy;
      v[2] = (z + z) * fz;
      v[3] = x * fy + y * fx;
      v[4] = x * fz + z * fx;
      v[5] = y * fz + z * fy;
    }
  } else {
#pragma unroll 2
    for (int l = l0; l < l1; ++l) {
      const double kx = rec[l].kx, ky = rec[l].ky, kz = rec[l].kz;
      double sn, cs;
      phase_sincos<F32>(rec[l].mx, rec[l].my, rec[l].mz, sx, sy, sz, turn, &sn, &cs);
      const double fs = (q4 * rec[l].pre) * fma(cs, rec[l].ri, -(sn * rec[l].rr));
      fx = fma(fs, kx, fx);
      fy = fma(fs, ky, fy);
      fz = fma(fs, kz, fz);
      if (THERMO || PERATOM) {
        v[0] += (x * kx + x * kx) * fs;
        v[1] += (y * ky + y * ky) * fs;
        v[2] += (z * kz + z * kz) * fs;
        v[3] += (x * ky + y * kx) * fs;
        v[4] += (x * kz + z * kx) * fs;
        v[5] += (y * kz + z * ky) * fs;
      }
    }
  }
  const double sc = kv.S_over_P;
  if (THERMO) {
    const double vals[kRowK] = {v[0] * sc, v[1] * sc, v[2] * sc, v[3] * sc, v[4] * sc, v[5] * sc};
    block_write_row<kRowK, KS>(vals, rows + (size_t)bid * kRowK);
  }
  // the atom's totals: wavefront partials added in order
  if (w > 0) {
    part[w][0][lane] = fx;
    part[w][1][lane] = fy;
    part[w][2][lane] = fz;
    if (PERATOM)
      for (int k = 0; k < 6; ++k) part[w][3 + k][lane] = v[k];
  }
  __syncthreads();
  if (w == 0 && act) {
    for (int u = 1; u < KS; ++u) {
      fx += part[u][0][lane];
      fy += part[u][1][lane];
      fz += part[u][2][lane];
      if (PERATOM)
        for (int k = 0; k < 6; ++k) v[k] += part[u][3 + k][lane];
    }
    s.fkx[i] = s.qqr2e * (fx * sc);
    s.fky[i] = s.qqr2e * (fy * sc);
    s.fkz[i] = s.qqr2e * (fz * sc);
    if (PERATOM)
      for (int k = 0; k < 6; ++k) s.vir_k[(size_t)6 * i + k] = v[k] * sc;
  }
}

}  // namespace rbmd
