// k_ewald.hip -- the Ewald sum over a whole kmax grid (structure factor,
// force, energy), FP64.
//
//   rho(k) = sum_i q_i e^{i k.r_i},  F_i = -(4 pi q_i / V) sum_k e^{-k^2/4 alpha} / k^2 Im(rho(k) e^{-i k.r_i}) k
//   ComputeNewFarElectrostaticsWorklet (RunWorklet.cpp:2492-2540),
//   ComputePnumberChargeStructureFactorWorklet (:2209-2291), ComputeEwaldEnergy (ExecutionMD.cpp:405-443)
//
// A grid needs neither a sine and cosine per (atom, k) nor its second half:
// e^{i k.r} = ex(kx) ey(ky) ez(kz) with one sine and cosine per (atom, axis,
// k), and rho(-k) is the conjugate of rho(k).  Per row (kx, ky) of the half
// grid the structure factor is then a contraction over the atoms, of
// q ex ey (rows) with the cosines and sines of the z phases (columns): real
// FP64 matrix products, whose four products of real and imaginary parts give
// +kz and -kz together.  The force is the contraction over kz with weights
// formed from rho, times conj(ex ey) and summed over the rows.  Both run on
// v_mfma_f64_16x16x4f64 (the FP64 matrix rate equals the vector rate, but a
// 16 x 16 tile takes two operand loads where the vector form takes 256), 2
// matrix operations a (atom, k) of the full grid and pass, where the direct
// form takes about 60 vector instructions.
//
// Measured (kernels of one structure factor + force, HIP events): 12,000 atoms,
// 132,650 vectors 18.5 ms -> 0.35 ms (the products alone take 0.13 ms at the
// matrix rate; the rest is the operands' latency at two to four wavefronts a
// SIMD); 30,000 atoms, 328,508 vectors 1.97 ms.  The error against the direct
// sum in 64 bits falls from 1.3e-14 to 6.5e-15: an axis phase is smaller than
// their sum.
//
// Every sum has a fixed order (atom splits, then row splits, added in order).
#include <algorithm>

#include "dev.hpp"
#include "ewald.hpp"
#include "pack.hpp"
#include "reduce.hpp"
#include "sincos.hpp"

namespace rbmd {

typedef double EwD4 __attribute__((ext_vector_type(4)));

namespace {
int up(int v, int m) { return (v + m - 1) / m * m; }
}  // namespace

bool ewald_plan(int n, const int kmax[3], int64_t tab_bytes, int64_t part_bytes, EwView* v) {
  *v = EwView{};
  for (int d = 0; d < 3; ++d) {
    if (kmax[d] < 0) return false;
    v->K[d] = kmax[d];
  }
  if (kmax[0] + kmax[1] + kmax[2] == 0) return false;
  v->R = kmax[0] * (2 * kmax[1] + 1) + kmax[1] + 1;
  v->Rpad = up(v->R, 16);
  v->ldx = 2 * (kmax[0] + 1);
  v->ldy = 2 * (kmax[1] + 1);
  const int ct = up(2 * (kmax[2] + 1), 16) / 16;
  v->nt = ct >= 3 ? 4 : ct;
  v->ldz = up(ct, v->nt) * 16;
  v->Kd = up(2 * (kmax[2] + 1), 4);
  const int64_t atom = (int64_t)(v->ldx + v->ldy + v->ldz) * 8;
  v->batch = (int)std::min<int64_t>(n, std::max<int64_t>(64, tab_bytes / atom / 64 * 64));
  v->n = v->batch;  // the first batch
  const int batches = (n + v->batch - 1) / v->batch;
  // splits: about 4,096 wavefronts in all (four a SIMD), at least 64 atoms
  // each, and as many as the partials' memory allows
  const int64_t waves = (int64_t)(v->Rpad / 16) * (v->ldz / (16 * v->nt));
  int64_t sp = std::min<int64_t>(64, std::max<int64_t>(1, 4096 / waves));
  sp = std::min<int64_t>(sp, std::max<int64_t>(1, part_bytes / ((int64_t)2 * v->Rpad * v->ldz * 8) / batches));
  v->per = std::max(64, up((int)((v->batch + sp - 1) / sp), 16));
  v->splits = (v->batch + v->per - 1) / v->per;
  v->total_splits = (batches - 1) * v->splits + (n - (batches - 1) * v->batch + v->per - 1) / v->per;
  for (v->wgroups = 1; v->wgroups < 16 && v->total_splits > 8 * v->wgroups;) v->wgroups *= 2;
  // force: 128 atoms a workgroup, the row tiles split until about 2,048 wavefronts run
  const int wg = (v->batch + 127) / 128;
  const int tiles = v->Rpad / 16;
  int rs = std::min(tiles, std::max(1, 512 / wg));
  rs = std::min(rs, 16);
  v->rper = (tiles + rs - 1) / rs;
  v->rsplits = (tiles + v->rper - 1) / v->rper;
  return true;
}

static int64_t ew_up(int64_t doubles) { return (doubles * 8 + 255) / 256 * 256; }

int ewald_energy_rows(const EwView& v) {
  const int points = kBlock / v.wgroups;
  return (v.Rpad * (v.Kd / 2) + points - 1) / points;
}

int64_t ewald_bytes(const EwView& v, bool force) {
  int64_t b = ew_up((int64_t)v.batch * v.ldx) + ew_up((int64_t)v.batch * v.ldy) + ew_up((int64_t)v.batch * v.ldz) +
              ew_up((int64_t)v.total_splits * 2 * v.Rpad * v.ldz) + ew_up(ewald_energy_rows(v));
  if (force) b += ew_up((int64_t)4 * v.Kd * v.Rpad) + ew_up((int64_t)v.rsplits * 3 * v.batch);
  return b;
}

void ewald_buffers(EwView* v, void* base, bool force) {
  char* p = static_cast<char*>(base);
  auto take = [&](int64_t doubles) {
    double* q = reinterpret_cast<double*>(p);
    p += ew_up(doubles);
    return q;
  };
  v->tx = take((int64_t)v->batch * v->ldx);
  v->ty = take((int64_t)v->batch * v->ldy);
  v->tz = take((int64_t)v->batch * v->ldz);
  v->part = take((int64_t)v->total_splits * 2 * v->Rpad * v->ldz);
  v->erow = take(ewald_energy_rows(*v));
  v->W = force ? take((int64_t)4 * v->Kd * v->Rpad) : nullptr;
  v->fpart = force ? take((int64_t)v->rsplits * 3 * v->batch) : nullptr;
}

// row r of the half grid: kx, ky
__device__ __forceinline__ void ew_row(const EwView& v, int r, int& kx, int& ky) {
  const int w = 2 * v.K[1] + 1;
  const int q = r - (v.K[1] + 1);
  kx = q < 0 ? 0 : 1 + q / w;
  ky = q < 0 ? r : q % w - v.K[1];
}

// Phase tables: one thread an entry.  The phase m x / L in turns is reduced
// exactly (sincos_turns).
__device__ __forceinline__ void ew_table_body(const SysView& s, const EwView& v, const int bid) {
  const int ex = v.ldx / 2, ey = v.ldy / 2, ez = v.ldz / 2, per = ex + ey + ez;
  const int64_t t = (int64_t)bid * kBlock + threadIdx.x;
  const int i = (int)(t / per);
  if (i >= v.n) return;
  int m = (int)(t - (int64_t)i * per);
  const int g = v.n0 + i;
  double sn = 0, cs = 0;
  if (m < ex) {
    sincos_turns((double)m * (s.x[g] / s.box[0]), &sn, &cs);
    const double q = s.q[g];
    reinterpret_cast<double2*>(v.tx)[(size_t)i * ex + m] = make_double2(q * cs, q * sn);
  } else if (m < ex + ey) {
    m -= ex;
    sincos_turns((double)m * (s.y[g] / s.box[1]), &sn, &cs);
    reinterpret_cast<double2*>(v.ty)[(size_t)i * ey + m] = make_double2(cs, sn);
  } else {
    m -= ex + ey;
    if (m <= v.K[2]) sincos_turns((double)m * (s.z[g] / s.box[2]), &sn, &cs);  // columns past the grid: zero
    reinterpret_cast<double2*>(v.tz)[(size_t)i * ez + m] = make_double2(cs, sn);
  }
}

static int ew_table_blocks(const EwView& v) {
  return (int)(((int64_t)v.n * ((v.ldx + v.ldy + v.ldz) / 2) + kBlock - 1) / kBlock);
}

// q ex ey of atom a (batch index) on a row: kx, |ky|, and the sign of ky
__device__ __forceinline__ void ew_exy(const EwView& v, int a, int kx, int aky, double sg, double& er, double& ei) {
  const double2 x = reinterpret_cast<const double2*>(v.tx)[(size_t)a * (v.ldx / 2) + kx];
  const double2 y = reinterpret_cast<const double2*>(v.ty)[(size_t)a * (v.ldy / 2) + aky];
  const double yi = sg * y.y;
  er = fma(x.x, y.x, -(x.y * yi));
  ei = fma(x.x, yi, x.y * y.x);
}

// Structure-factor partials: one wavefront a tile of 16 rows x 16 NT columns
// and one split of the atoms, 4 atoms a step; the four wavefronts of a
// workgroup take four row tiles of the same columns and atoms.
template <int NT>
__device__ __forceinline__ void ew_rho_body(const EwView& v, const int bid) {
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int tiles = v.Rpad / 16, groups = (tiles + 3) / 4, cols = v.ldz / (16 * NT);
  const int rt = (bid % groups) * 4 + w, cg = (bid / groups) % cols, sp = bid / (groups * cols);
  if (rt >= tiles) return;
  const int r = rt * 16 + (lane & 15);
  int kx, ky;
  ew_row(v, r < v.R ? r : 0, kx, ky);
  const double sg = ky < 0 ? -1.0 : 1.0;
  const int aky = ky < 0 ? -ky : ky;
  const int a0 = sp * v.per, a1 = min(a0 + v.per, v.n);
  const double* const tz = v.tz + (size_t)cg * 16 * NT + (lane & 15);
  EwD4 cr[NT], ci[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) cr[t] = ci[t] = EwD4{0, 0, 0, 0};
  // operands of the next step in flight over this step's products
  double er, ei, z[NT];
  auto load = [&](int a) {
    const int i = a + lane / 16;
    const bool in = i < a1 && r < v.R;
    const int j = i < a1 ? i : a0;
    ew_exy(v, j, kx, aky, sg, er, ei);
    er = in ? er : 0.0;
    ei = in ? ei : 0.0;
#pragma unroll
    for (int t = 0; t < NT; ++t) z[t] = tz[(size_t)j * v.ldz + 16 * t];
  };
  load(a0);
#pragma unroll 2
  for (int a = a0; a < a1; a += 4) {
    const double ar = er, ai = ei;
    double b[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) b[t] = z[t];
    load(a + 4);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      cr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, b[t], cr[t], 0, 0, 0);
      ci[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, b[t], ci[t], 0, 0, 0);
    }
  }
  double* const out = v.part + (size_t)(v.split0 + sp) * 2 * v.Rpad * v.ldz;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const size_t at = (size_t)(rt * 16 + lane / 16 + 4 * u) * v.ldz + (cg * NT + t) * 16 + (lane & 15);
      out[at] = cr[t][u];
      out[(size_t)v.Rpad * v.ldz + at] = ci[t][u];
    }
}

static int ew_rho_blocks(const EwView& v) {
  return (v.Rpad / 16 + 3) / 4 * (v.ldz / (16 * v.nt)) * ((v.n + v.per - 1) / v.per);
}

// Sum of the partials, the force weights and the energy of each grid point (row,
// kz).  With rho+ = rho(kx, ky, kz), rho- = rho(kx, ky, -kz), U = rho+ + rho-,
// V = rho+ - rho- and the prefactor 2 e^{-k^2/4 alpha} / (V k^2) of k and -k:
//   sum over +-kz of rho conj(ez)    = U cos - i V sin
//   sum over +-kz of rho conj(ez) kz = kz (V cos - i U sin)
// On the row kx = ky = 0 the conjugate of +kz is -kz itself: rho- = 0 there.
//
// wgroups threads add the partials of a grid point (a small grid has few
// points and up to hundreds of partials: one thread each took 32 us at 6000
// atoms, this one 7), their sums added in order.
__device__ __forceinline__ void ew_weight_body(const SysView& s, const EwView& v, const int bid) {
#pragma clang fp contract(off)
  __shared__ double4 sums[kBlock];
  const int nz = v.Kd / 2;
  const int points = kBlock / v.wgroups;
  const int g = threadIdx.x / points;
  const int t = bid * points + threadIdx.x % points;
  const int r = t / nz, z = t % nz;
  const bool in = r < v.R && z <= v.K[2] && (r > 0 || z > 0);
  double2 a = make_double2(0, 0), b = make_double2(0, 0);
  if (in) {
    const size_t plane = (size_t)v.Rpad * v.ldz, at = (size_t)r * v.ldz + 2 * z;
#pragma unroll 8
    for (int sp = g; sp < v.total_splits; sp += v.wgroups) {
      const double2 p = *reinterpret_cast<const double2*>(v.part + (size_t)sp * 2 * plane + at);
      const double2 q = *reinterpret_cast<const double2*>(v.part + ((size_t)sp * 2 + 1) * plane + at);
      a.x += p.x;
      a.y += p.y;
      b.x += q.x;
      b.y += q.y;
    }
  }
  if (v.wgroups > 1) {
    sums[threadIdx.x] = make_double4(a.x, a.y, b.x, b.y);
    __syncthreads();
    if (g == 0)
      for (int u = 1; u < v.wgroups; ++u) {
        const double4 o = sums[u * points + threadIdx.x];
        a.x += o.x;
        a.y += o.y;
        b.x += o.z;
        b.y += o.w;
      }
  }
  double e = 0.0;
  if (g == 0 && r < v.Rpad) {
    double w[4][2] = {{0, 0}, {0, 0}, {0, 0}, {0, 0}};
    if (in) {
      int mx, my;
      ew_row(v, r, mx, my);
      const double kx = 2 * kPi * mx / s.box[0], ky = 2 * kPi * my / s.box[1], kz = 2 * kPi * z / s.box[2];
      const double k2 = kx * kx + ky * ky + kz * kz;
      const double gk = exp(-k2 / (4 * s.alpha)) / k2;
      const double pr = a.x - b.y, pi = a.y + b.x;  // rho+
      const bool two = r > 0 && z > 0;
      const double nr = two ? a.x + b.y : 0.0, ni = two ? b.x - a.y : 0.0;  // rho-
      e = 2.0 * gk * ((pr * pr + pi * pi) + (nr * nr + ni * ni));
      const double c = 2.0 * gk / s.volume;
      const double ur = c * (pr + nr), ui = c * (pi + ni), vr = c * (pr - nr), vi = c * (pi - ni);
      w[0][0] = ur;
      w[0][1] = vi;
      w[1][0] = ui;
      w[1][1] = -vr;
      w[2][0] = kz * vr;
      w[2][1] = kz * ui;
      w[3][0] = kz * vi;
      w[3][1] = -(kz * ur);
    }
    if (v.W) {
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        v.W[((size_t)f * v.Kd + 2 * z) * v.Rpad + r] = w[f][0];
        v.W[((size_t)f * v.Kd + 2 * z + 1) * v.Rpad + r] = w[f][1];
      }
    }
  }
  const double vals[1] = {e};
  block_write_row<1>(vals, v.erow + bid);
}

// Force partials: one wavefront 32 atoms (two tiles) and a range of row tiles.
// T = sum over kz of weights x z phases for 16 atoms x 16 rows (real and
// imaginary part, and the same with kz), then Im(T conj(q ex ey)) times kx, ky
// (and 1) summed over the rows.
__device__ __forceinline__ void ew_force_body(const SysView& s, const EwView& v, const int bid) {
  constexpr int AT = 2;
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int groups = (v.n + 64 * AT - 1) / (64 * AT);
  const int ag = bid % groups, rs = bid / groups;
  const int i0 = (ag * 4 + w) * 16 * AT;
  if (i0 >= v.n) return;
  const int c = lane & 15, h = lane / 16;
  const double* za[AT];
#pragma unroll
  for (int t = 0; t < AT; ++t) za[t] = v.tz + (size_t)min(i0 + 16 * t + c, v.n - 1) * v.ldz + h;
  double fx[AT][4], fy[AT][4], fz[AT][4];
#pragma unroll
  for (int t = 0; t < AT; ++t)
#pragma unroll
    for (int u = 0; u < 4; ++u) fx[t][u] = fy[t][u] = fz[t][u] = 0.0;
  const int rt1 = min((rs + 1) * v.rper, v.Rpad / 16);
  const size_t plane = (size_t)v.Kd * v.Rpad;
  for (int rt = rs * v.rper; rt < rt1; ++rt) {
    const int r = rt * 16 + c;
    EwD4 acc[AT][4];
#pragma unroll
    for (int t = 0; t < AT; ++t)
#pragma unroll
      for (int f = 0; f < 4; ++f) acc[t][f] = EwD4{0, 0, 0, 0};
    const double* wp = v.W + (size_t)h * v.Rpad + r;
    double bn[4], an[AT];
    auto load = [&](int kd) {
#pragma unroll
      for (int f = 0; f < 4; ++f) bn[f] = wp[f * plane + (size_t)kd * v.Rpad];
#pragma unroll
      for (int t = 0; t < AT; ++t) an[t] = za[t][kd];
    };
    load(0);
#pragma unroll 2
    for (int kd = 0; kd < v.Kd; kd += 4) {
      double b[4], a[AT];
#pragma unroll
      for (int f = 0; f < 4; ++f) b[f] = bn[f];
#pragma unroll
      for (int t = 0; t < AT; ++t) a[t] = an[t];
      if (kd + 4 < v.Kd) load(kd + 4);  // in flight over this step's products
#pragma unroll
      for (int t = 0; t < AT; ++t)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[t][f] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], b[f], acc[t][f], 0, 0, 0);
    }
    int mx, my;
    ew_row(v, r < v.R ? r : 0, mx, my);
    const double kx = 2 * kPi * mx / s.box[0], ky = 2 * kPi * my / s.box[1];
    const double sg = my < 0 ? -1.0 : 1.0;
    const int aky = my < 0 ? -my : my;
#pragma unroll
    for (int t = 0; t < AT; ++t)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        double er, ei;
        ew_exy(v, min(i0 + 16 * t + h + 4 * u, v.n - 1), mx, aky, sg, er, ei);
        const double im = fma(acc[t][1][u], er, -(acc[t][0][u] * ei));
        fx[t][u] = fma(kx, im, fx[t][u]);
        fy[t][u] = fma(ky, im, fy[t][u]);
        fz[t][u] += fma(acc[t][3][u], er, -(acc[t][2][u] * ei));
      }
  }
  double* const out = v.fpart + (size_t)rs * 3 * v.batch;
#pragma unroll
  for (int t = 0; t < AT; ++t)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
      for (int off = 1; off < 16; off <<= 1) {
        fx[t][u] += __shfl_xor(fx[t][u], off, kWave);
        fy[t][u] += __shfl_xor(fy[t][u], off, kWave);
        fz[t][u] += __shfl_xor(fz[t][u], off, kWave);
      }
      const int i = i0 + 16 * t + h + 4 * u;
      if (c == 0 && i < v.n) {
        out[i] = fx[t][u];
        out[v.batch + i] = fy[t][u];
        out[2 * v.batch + i] = fz[t][u];
      }
    }
}

static int ew_force_blocks(const EwView& v) { return (v.n + 127) / 128 * v.rsplits; }

// The atoms' forces from the row splits, and their virial terms
// x_a F_b + x_b F_a (ComputeKspaceVirial summed over k).
template <bool THERMO, bool PERATOM>
__device__ __forceinline__ void ew_finish_body(const SysView& s, const EwView& v, double* rows, const int bid) {
#pragma clang fp contract(off)
  const int i = bid * kBlock + threadIdx.x;
  double vir[6] = {0, 0, 0, 0, 0, 0};
  if (i < v.n) {
    double f[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      double a = v.fpart[(size_t)d * v.batch + i];
      for (int u = 1; u < v.rsplits; ++u) a += v.fpart[((size_t)u * 3 + d) * v.batch + i];
      f[d] = -4.0 * kPi * a;
    }
    const int g = v.n0 + i;
    s.fkx[g] = s.qqr2e * f[0];
    s.fky[g] = s.qqr2e * f[1];
    s.fkz[g] = s.qqr2e * f[2];
    if (THERMO || PERATOM) {
      const double x = s.x[g], y = s.y[g], z = s.z[g];
      vir[0] = (x + x) * f[0];
      vir[1] = (y + y) * f[1];
      vir[2] = (z + z) * f[2];
      vir[3] = x * f[1] + y * f[0];
      vir[4] = x * f[2] + z * f[0];
      vir[5] = y * f[2] + z * f[1];
      if (PERATOM)
        for (int k = 0; k < 6; ++k) s.vir_k[(size_t)6 * g + k] = vir[k];
    }
  }
  if (THERMO) block_write_row<kRowK>(vir, rows + (size_t)bid * kRowK);
}

__global__ __launch_bounds__(kBlock) void k_ew_table(SysView s, EwView v) { ew_table_body(s, v, (int)blockIdx.x); }
template <int NT>
__global__ __launch_bounds__(kBlock) void k_ew_rho(EwView v) {
  ew_rho_body<NT>(v, (int)blockIdx.x);
}
__global__ __launch_bounds__(kBlock) void k_ew_weight(SysView s, EwView v) { ew_weight_body(s, v, (int)blockIdx.x); }
__global__ __launch_bounds__(kBlock, 2) void k_ew_force(SysView s, EwView v) { ew_force_body(s, v, (int)blockIdx.x); }
template <bool THERMO, bool PERATOM>
__global__ __launch_bounds__(kBlock) void k_ew_finish(SysView s, EwView v, double* rows) {
  ew_finish_body<THERMO, PERATOM>(s, v, rows, (int)blockIdx.x);
}

static void ew_batch(EwView* v, int n, int b) {
  v->n0 = b * v->batch;
  v->n = n - v->n0 < v->batch ? n - v->n0 : v->batch;
  v->split0 = b * v->splits;
}

// structure factor, weights and energy rows of a planned grid
void launch_ewald_rho(const SysView& s, EwView v, hipStream_t st) {
  const int batches = (s.n + v.batch - 1) / v.batch;
  for (int b = 0; b < batches; ++b) {
    ew_batch(&v, s.n, b);
    hipLaunchKernelGGL(k_ew_table, dim3(ew_table_blocks(v)), dim3(kBlock), 0, st, s, v);
    const dim3 grid(ew_rho_blocks(v));
    if (v.nt == 1)
      hipLaunchKernelGGL(k_ew_rho<1>, grid, dim3(kBlock), 0, st, v);
    else if (v.nt == 2)
      hipLaunchKernelGGL(k_ew_rho<2>, grid, dim3(kBlock), 0, st, v);
    else
      hipLaunchKernelGGL(k_ew_rho<4>, grid, dim3(kBlock), 0, st, v);
  }
  hipLaunchKernelGGL(k_ew_weight, dim3(ewald_energy_rows(v)), dim3(kBlock), 0, st, s, v);
}

// forces after launch_ewald_rho (with the force buffers); thermo rows as launch_kforce
void launch_ewald_force(const SysView& s, EwView v, hipStream_t st, int thermo, int peratom, double* rows,
                        int* nblocks) {
  const int batches = (s.n + v.batch - 1) / v.batch;
  int blocks = 0;
  for (int b = batches - 1; b >= 0; --b) {  // the tables hold the last batch
    ew_batch(&v, s.n, b);
    if (b != batches - 1) hipLaunchKernelGGL(k_ew_table, dim3(ew_table_blocks(v)), dim3(kBlock), 0, st, s, v);
    hipLaunchKernelGGL(k_ew_force, dim3(ew_force_blocks(v)), dim3(kBlock), 0, st, s, v);
    const dim3 grid((v.n + kBlock - 1) / kBlock);
    double* const out = rows ? rows + (size_t)blocks * kRowK : nullptr;
    if (peratom)
      hipLaunchKernelGGL((k_ew_finish<true, true>), grid, dim3(kBlock), 0, st, s, v, out);
    else if (thermo)
      hipLaunchKernelGGL((k_ew_finish<true, false>), grid, dim3(kBlock), 0, st, s, v, out);
    else
      hipLaunchKernelGGL((k_ew_finish<false, false>), grid, dim3(kBlock), 0, st, s, v, out);
    blocks += (int)grid.x;
  }
  if (nblocks) *nblocks = blocks;
}

// ------------------------------------------------------------------ packs
// one batch a system

__global__ __launch_bounds__(kBlock) void kp_ew_table(PACK_PARAMS) {
  PACK_ENTRY(e, bid)
  ew_table_body(e.v, e.ew, bid);
}
template <int NT>
__global__ __launch_bounds__(kBlock) void kp_ew_rho(PACK_PARAMS) {
  PACK_ENTRY(e, bid)
  ew_rho_body<NT>(e.ew, bid);
}
__global__ __launch_bounds__(kBlock) void kp_ew_weight(PACK_PARAMS) {
  PACK_ENTRY(e, bid)
  ew_weight_body(e.v, e.ew, bid);
}
__global__ __launch_bounds__(kBlock, 2) void kp_ew_force(PACK_PARAMS) {
  PACK_ENTRY(e, bid)
  ew_force_body(e.v, e.ew, bid);
}
template <bool THERMO>
__global__ __launch_bounds__(kBlock) void kp_ew_finish(PACK_PARAMS) {
  PACK_ENTRY(e, bid)
  ew_finish_body<THERMO, false>(e.v, e.ew, e.rows_k, bid);
}

int pack_ewald_blocks(const EwView& v, int kernel) {
  switch (kernel) {
    case PK_EW_TABLE:
      return ew_table_blocks(v);
    case PK_EW_RHO1:
      return v.nt == 1 ? ew_rho_blocks(v) : 0;
    case PK_EW_RHO2:
      return v.nt == 2 ? ew_rho_blocks(v) : 0;
    case PK_EW_RHO4:
      return v.nt == 4 ? ew_rho_blocks(v) : 0;
    case PK_EW_WEIGHT:
      return ewald_energy_rows(v);
    case PK_EW_FORCE:
      return ew_force_blocks(v);
    case PK_EW_FINISH:
      return (v.n + kBlock - 1) / kBlock;
    default:
      return 0;
  }
}

void launch_pack_ewald(int kernel, const PackLaunch& L, int nblocks, int thermo, hipStream_t st) {
  if (nblocks <= 0) return;
  const dim3 grid(nblocks);
  switch (kernel) {
    case PK_EW_TABLE:
      hipLaunchKernelGGL(kp_ew_table, grid, dim3(kBlock), 0, st, PACK_ARGS(L));
      break;
    case PK_EW_RHO1:
      hipLaunchKernelGGL(kp_ew_rho<1>, grid, dim3(kBlock), 0, st, PACK_ARGS(L));
      break;
    case PK_EW_RHO2:
      hipLaunchKernelGGL(kp_ew_rho<2>, grid, dim3(kBlock), 0, st, PACK_ARGS(L));
      break;
    case PK_EW_RHO4:
      hipLaunchKernelGGL(kp_ew_rho<4>, grid, dim3(kBlock), 0, st, PACK_ARGS(L));
      break;
    case PK_EW_WEIGHT:
      hipLaunchKernelGGL(kp_ew_weight, grid, dim3(kBlock), 0, st, PACK_ARGS(L));
      break;
    case PK_EW_FORCE:
      hipLaunchKernelGGL(kp_ew_force, grid, dim3(kBlock), 0, st, PACK_ARGS(L));
      break;
    case PK_EW_FINISH:
      if (thermo)
        hipLaunchKernelGGL(kp_ew_finish<true>, grid, dim3(kBlock), 0, st, PACK_ARGS(L));
      else
        hipLaunchKernelGGL(kp_ew_finish<false>, grid, dim3(kBlock), 0, st, PACK_ARGS(L));
      break;
    default:
      break;
  }
}

}  // namespace rbmd
