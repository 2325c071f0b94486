// ewald.hpp -- the grid Ewald sum: sizes and buffers of its separable form
// (kernels in k_ewald.hip).
#pragma once
#include <stdint.h>

namespace rbmd {

// One pass over the kmax grid.  The half grid is rows (kx, ky), kx > 0 or kx =
// 0 and ky >= 0, times kz = 0 .. Kz; columns 2 kz, 2 kz + 1 are cos and sin of
// the z phase.
struct EwView {
  int K[3];
  int R, Rpad;        // rows, and rounded up to 16
  int ldx, ldy, ldz;  // doubles per atom of the phase tables (ldz: columns rounded up to whole tiles)
  int Kd;             // columns rounded up to 4 (the force pass's contraction length)
  int nt;             // column tiles of 16 per structure-factor wavefront (1, 2, 4)
  int n0, n;          // atoms of this batch: n from n0 on
  int per, split0, splits;  // structure factor: atoms per split, this batch's first split and their number
  int total_splits;
  int rper, rsplits;  // force: row tiles per split, splits
  int wgroups;        // weight pass: threads that share the partials of a grid point
  double *tx, *ty, *tz;  // phase tables of the batch: (cos, sin) of m 2 pi x / L, x's times the charge
  double* part;       // [total_splits][2][Rpad][ldz] structure-factor partials
  double* W;          // [4][Kd][Rpad] force weights
  double* erow;       // energy sums of the weight pass's workgroups
  double* fpart;      // [rsplits][3][batch] partial forces
  int batch;          // atoms the tables and fpart hold
};

// Sizes of the view for n atoms (no buffers): the tables hold at most
// tab_bytes, the partials about part_bytes; returns false for an empty grid.
bool ewald_plan(int n, const int kmax[3], int64_t tab_bytes, int64_t part_bytes, EwView* v);
int64_t ewald_bytes(const EwView& v, bool force);       // workspace of the plan
void ewald_buffers(EwView* v, void* base, bool force);  // its buffers within `base` (256-byte aligned)
int ewald_energy_rows(const EwView& v);                 // workgroups of the weight pass

}  // namespace rbmd
