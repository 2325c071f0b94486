// k_transfer.hip -- the arrays of a call between the device's layout (one array
// per component, list order for the real-space results) and the caller's (one
// record per atom, the caller's order), through pinned host memory that the
// kernels read and write themselves.
//
// Separate copies of each component through pageable memory, with the records
// put together on the host, cost 15 to 20 us each: most of a call on a few
// thousand atoms.  Here a call's arrays, or a part of them that fits the
// staging buffer, are one launch: reference forces of 12,000 atoms 620 -> 344 us,
// a pack's 32 states 1423 copies -> 32 launches (17.4 -> 14.0 ms with its steps),
// the state of 300,000 atoms both ways 10.4 -> 6 ms.
#include "dev.hpp"

namespace rbmd {

__device__ __forceinline__ int transfer_field(const TransferDesc& d, int e) {
  int f = 0;
  while (f + 1 < d.nfield && e >= d.field[f + 1].first * d.atoms) ++f;
  return f;
}

// element e of a part: its field, atom and component
template <bool OUT>
__global__ __launch_bounds__(kBlock) void k_transfer(TransferDesc d) {
#pragma clang fp contract(off)
  const int total = d.width * d.atoms;
  for (int e = blockIdx.x * kBlock + threadIdx.x; e < total; e += gridDim.x * kBlock) {
    const int f = transfer_field(d, e);
    const TransferField& F = d.field[f];
    const int t = e - F.first * d.atoms;
    const int a = t / F.width, k = t - a * F.width;
    if (F.is_int) {  // whole numbers, one record per atom on both sides
      int* dev = (int*)F.p[0] + (size_t)F.width * (d.a0 + a) + k;
      int* host = (int*)(d.host + F.first * (size_t)d.atoms) + t;
      if (OUT)
        *host = *dev;
      else
        *dev = *host;
      continue;
    }
    const size_t i = F.rank ? F.rank[d.a0 + a] : d.a0 + a;
    double* const p = F.split ? F.p[k] : F.p[0];
    const size_t at = F.split ? i : i * F.width + k;
    const size_t slab = F.split ? (size_t)d.n : (size_t)d.n * F.width;
    if (OUT) {
      double v = p[at];
      for (int sl = 1; sl < F.slabs; ++sl) v += p[at + sl * slab];  // slab partials in slab order
      d.host[e] = v;
    } else {
      p[at] = d.host[e];
    }
  }
}

void launch_transfer(const TransferDesc& d, bool out, hipStream_t st) {
  const long total = (long)d.width * d.atoms;
  if (total <= 0) return;
  const int grid = (int)((total + kBlock - 1) / kBlock);
  if (out)
    hipLaunchKernelGGL(k_transfer<true>, dim3(grid), dim3(kBlock), 0, st, d);
  else
    hipLaunchKernelGGL(k_transfer<false>, dim3(grid), dim3(kBlock), 0, st, d);
}

// the small results a thermo call reads, in one record
__global__ void k_thermo_out(const NhcState* nhc, const int* misfit, const int* status, const int* iter,
                             const int* builds, ThermoOut* out) {
  const int t = threadIdx.x;
  constexpr int words = (int)(sizeof(NhcState) / 8);
  for (int k = t; k < words; k += kWave) ((double*)&out->nhc)[k] = ((const double*)nhc)[k];
  if (t == 0) out->misfit = misfit[0];
  if (t == 1) out->status = status[0];
  if (t == 2) out->iter = iter[0];
  if (t == 3) out->builds = builds[0];
}

void launch_thermo_out(const NhcState* nhc, const int* misfit, const int* status, const int* iter, const int* builds,
                       ThermoOut* out, hipStream_t st) {
  hipLaunchKernelGGL(k_thermo_out, dim3(1), dim3(kWave), 0, st, nhc, misfit, status, iter, builds, out);
}

}  // namespace rbmd
