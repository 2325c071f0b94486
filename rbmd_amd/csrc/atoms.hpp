// atoms.hpp -- per-atom bodies shared by their own kernels, the packed kernels
// and the fused launches of compact systems: vector helpers, bonded forces, the
// force assembly with the second half step.
#pragma once
#include "dev.hpp"
#include "reduce.hpp"

namespace rbmd {

struct D3 {
  double x, y, z;
};
// The vector helpers, SHAKE and RATTLE compile with FMA contraction off: a
// product and a sum written in separate helpers are then rounded separately
// in every kernel that inlines them, so the fused and the separate launches
// of these steps agree to the bit.
__device__ __forceinline__ D3 sub(D3 a, D3 b) {
#pragma clang fp contract(off)
  return {a.x - b.x, a.y - b.y, a.z - b.z};
}
__device__ __forceinline__ D3 add(D3 a, D3 b) {
#pragma clang fp contract(off)
  return {a.x + b.x, a.y + b.y, a.z + b.z};
}
__device__ __forceinline__ D3 mul(double k, D3 a) {
#pragma clang fp contract(off)
  return {k * a.x, k * a.y, k * a.z};
}
__device__ __forceinline__ D3 divs(D3 a, double k) {
#pragma clang fp contract(off)
  return {a.x / k, a.y / k, a.z / k};
}
__device__ __forceinline__ double dotp(D3 a, D3 b) {
#pragma clang fp contract(off)
  return a.x * b.x + a.y * b.y + a.z * b.z;
}
__device__ __forceinline__ D3 mimg(const SysView& s, D3 a, D3 b) {
#pragma clang fp contract(off)
  D3 v = sub(a, b);
  if (fabs(v.x) > s.box[0] * 0.5) v.x -= (v.x > 0 ? s.box[0] : -s.box[0]);
  if (fabs(v.y) > s.box[1] * 0.5) v.y -= (v.y > 0 ? s.box[1] : -s.box[1]);
  if (fabs(v.z) > s.box[2] * 0.5) v.z -= (v.z > 0 ? s.box[2] : -s.box[2]);
  return v;
}
__device__ __forceinline__ D3 ld(const double* x, const double* y, const double* z, int i) { return {x[i], y[i], z[i]}; }
__device__ __forceinline__ void st3(double* x, double* y, double* z, int i, D3 v) {
  x[i] = v.x;
  y[i] = v.y;
  z[i] = v.z;
}

// bond + angle forces gathered per atom over its incident terms; the energy
// and virial of a term are counted by its first atom.  With iv.spec_coul
// (CVFF + RBL + special bonds) also the intramolecular Coulomb correction of
// ComputeSpecialCoulGeneralWorklet (RunWorklet.cpp:2012-2084, added to the
// force by ExecutionNVT::ComputeAllForce, ExecutionNVT.cpp:212-214): for the
// other atoms j of i's molecule (molecules of 3 or more atoms),
//   F_i += (1 - w_ij) (-332.06371 q_i q_j / r^3) r,  r = MinDistanceVec(x_i, x_j),
// 332.06371 hard-coded as in the reference (hazard Q24), w_ij the last match of
// j in i's special list (else 1); its virial +1/2 r (x) F (ComputePairVirial_fix)
// goes into the bond virial slots (both enter the pressure once,
// ExecutionMD.cpp:1323-1358).  The random-batch real space has no exclusions,
// so this removes the intramolecular erfc Coulomb the pair term added.
template <bool THERMO>
__device__ __forceinline__ void bonded_body(const SysView& s, const IntView& iv, double* rows, const int bid) {
  int i = bid * blockDim.x + threadIdx.x;
  double f[3] = {0, 0, 0};
  double eb = 0, ea = 0;
  double vb[6] = {0, 0, 0, 0, 0, 0}, va[6] = {0, 0, 0, 0, 0, 0};
  if (i < s.n && iv.spec_coul && iv.grp_off[i + 1] - iv.grp_off[i] >= 3) {
    const D3 pi = ld(s.x, s.y, s.z, i);
    const double qi = s.q[i];
    for (int k = iv.grp_off[i]; k < iv.grp_off[i + 1]; ++k) {
      const int j = iv.grp_ids[k];
      if (j == i) continue;
      const D3 r = mimg(s, pi, ld(s.x, s.y, s.z, j));
      const double dis = sqrt(dotp(r, r));
      const double fcomp = -332.06371 * qi * s.q[j] / (dis * dis * dis);
      double w = 1.0;
      if (s.sp_off)
        for (int t = s.sp_off[i]; t < s.sp_off[i + 1]; ++t)
          if (s.sp_ids[t] == j) w = s.sp_w[t];
      const D3 cp = mul((1.0 - w) * fcomp, r);
      f[0] += cp.x;
      f[1] += cp.y;
      f[2] += cp.z;
      if (THERMO) {
        vb[0] += 0.5 * (r.x * cp.x);
        vb[1] += 0.5 * (r.y * cp.y);
        vb[2] += 0.5 * (r.z * cp.z);
        vb[3] += 0.5 * (r.x * cp.y);
        vb[4] += 0.5 * (r.x * cp.z);
        vb[5] += 0.5 * (r.y * cp.z);
      }
    }
  }
  if (i < s.n) {
    for (int k = iv.inc_b_off[i]; k < iv.inc_b_off[i + 1]; ++k) {
      int b = iv.inc_b[k];
      int a0 = iv.bond_atoms[2 * b], a1 = iv.bond_atoms[2 * b + 1];
      D3 r = mimg(s, ld(s.x, s.y, s.z, a0), ld(s.x, s.y, s.z, a1));
      double d = sqrt(dotp(r, r));
      double dr = d - iv.bond_r0[b];
      double rk = iv.bond_k[b] * dr;
      double fb = d > 0.01 ? -2.0 * rk / d : 0.0;
      D3 fi = mul(fb, r);
      double sg = (a0 == i) ? 1.0 : -1.0;
      f[0] += sg * fi.x;
      f[1] += sg * fi.y;
      f[2] += sg * fi.z;
      if (THERMO && a0 == i) {
        eb += rk * dr;
        vb[0] += r.x * fi.x;
        vb[1] += r.y * fi.y;
        vb[2] += r.z * fi.z;
        vb[3] += r.x * fi.y;
        vb[4] += r.x * fi.z;
        vb[5] += r.y * fi.z;
      }
    }
    for (int k = iv.inc_a_off[i]; k < iv.inc_a_off[i + 1]; ++k) {
      int a = iv.inc_a[k];
      int ai = iv.angle_all[3 * a], aj = iv.angle_all[3 * a + 1], ak = iv.angle_all[3 * a + 2];
      D3 pj = ld(s.x, s.y, s.z, aj);
      D3 rij = mimg(s, ld(s.x, s.y, s.z, ai), pj);
      D3 rkj = mimg(s, ld(s.x, s.y, s.z, ak), pj);
      double dij2 = dotp(rij, rij), dij = sqrt(dij2);
      double dkj2 = dotp(rkj, rkj), dkj = sqrt(dkj2);
      double c = dotp(rij, rkj);
      c /= dij * dkj;
      if (c > 1.0) c = 1.0;
      if (c < -1.0) c = -1.0;
      double sn = sqrt(1.0 - c * c);
      if (sn < 0.001) sn = 0.001;
      sn = 1.0 / sn;
      double dth = acos(c) - (iv.angle_t0[a] * kPi) / 180;
      double tk = iv.angle_k[a] * dth;
      double aa = -2.0 * tk * sn;
      double a11 = aa * c / dij2, a12 = -aa / (dij * dkj), a22 = aa * c / dkj2;
      D3 fi = add(mul(a11, rij), mul(a12, rkj));
      D3 fk = add(mul(a22, rkj), mul(a12, rij));
      D3 mine = (i == ai) ? fi : ((i == ak) ? fk : mul(-1.0, add(fi, fk)));
      f[0] += mine.x;
      f[1] += mine.y;
      f[2] += mine.z;
      if (THERMO && i == ai) {
        ea += tk * dth;
        va[0] += rij.x * fi.x + rkj.x * fk.x;
        va[1] += rij.y * fi.y + rkj.y * fk.y;
        va[2] += rij.z * fi.z + rkj.z * fk.z;
        va[3] += rij.x * fi.y + rkj.x * fk.y;
        va[4] += rij.x * fi.z + rkj.x * fk.z;
        va[5] += rij.y * fi.z + rkj.y * fk.z;
      }
    }
    s.fbx[i] = f[0];
    s.fby[i] = f[1];
    s.fbz[i] = f[2];
  }
  if (THERMO) {
    // slots S_VIR_BOND .. S_VIR_ANGLE + 5, S_EBOND, S_EANGLE
    const double vals[kRowBond] = {vb[0], vb[1], vb[2], vb[3], vb[4], vb[5], va[0],
                                   va[1], va[2], va[3], va[4], va[5], eb,    ea};
    block_write_row<kRowBond>(vals, rows + (size_t)bid * kRowBond);
  }
}

// F = F_real[rank] (slab partials in order) + F_k + F_bonded; optional second kick;
// kinetic energy, one row per wavefront of 64 atoms (wave: the 64 atoms from
// 64 * wave on; every lane of the wavefront calls this)
__device__ __forceinline__ void second_half_wave(const SysView& s, const IntView& iv, int kick, int has_k, int has_b,
                                                 double* rows, const int wave) {
  const int lane = threadIdx.x & (kWave - 1);
  const int i = wave * kWave + lane;
  double ke = 0.0;
  if (i < s.n) {
    int r = s.rank[i];
    double fx = s.fnx[r], fy = s.fny[r], fz = s.fnz[r];
    for (int k = 1; k < s.nslab; ++k) {
      const size_t o = (size_t)k * s.n + r;
      fx += s.fnx[o];
      fy += s.fny[o];
      fz += s.fnz[o];
    }
    if (has_k) {
      fx = s.fkx[i] + fx;
      fy = s.fky[i] + fy;
      fz = s.fkz[i] + fz;
    }
    if (has_b) {
      fx += s.fbx[i];
      fy += s.fby[i];
      fz += s.fbz[i];
    }
    s.fx[i] = fx;
    s.fy[i] = fy;
    s.fz[i] = fz;
    double vx = s.vx[i], vy = s.vy[i], vz = s.vz[i];
    double m = s.mass[i];
    if (kick) {
      s.ovx[i] = vx;
      s.ovy[i] = vy;
      s.ovz[i] = vz;
      vx += 0.5 * fx / m * iv.dt * iv.fmt2v;
      vy += 0.5 * fy / m * iv.dt * iv.fmt2v;
      vz += 0.5 * fz / m * iv.dt * iv.fmt2v;
      s.vx[i] = vx;
      s.vy[i] = vy;
      s.vz[i] = vz;
    }
    ke = m * (vx * vx + vy * vy + vz * vz) * iv.mvv2e;
    if (!isfinite(fx + fy + fz)) atomicOr(s.status, 1);
  }
  ke = wave_sum(ke);
  if (lane == 0 && wave * kWave < s.n) rows[wave] = ke;
}

}  // namespace rbmd
