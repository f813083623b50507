// Force gather and per-structure sums from the bond forces, shared by the
// sparse GP's prediction and the mapped potential.
#pragma once
#include <hip/hip_runtime.h>

#include "fm_device.hpp"

namespace fm {

// Forces: F_i = sum_{bonds b of i} f_b - sum_{bonds b with neighbour i} f_b
// (normalized_dot_product.cpp:197-199 after K^T alpha), a fixed order for each
// atom: 16 lanes per atom take its bonds 16 apart, then sum over the lanes. The
// lanes read neighbouring bonds, so the own ones arrive as whole lines; a
// thread per atom walked two lists of about 50 scattered 12- or 24-byte values
// one after the other (262,144 atoms of the BCC alloy took 608 us with the sums,
// 137 + 8 now; 108 atoms 21 us, now 5 + 4). `mean_off` places F in
// the structures' mean_efs blocks, null in one array; `Eatom` (may be null)
// takes the row energies in atom order.
constexpr int kGatherAtoms = 16;  // atoms per workgroup of 256
template <typename TF>
__global__ __launch_bounds__(256) void k_forces(int n, const int *atom_struct, const int *atom_off,
                                                const long long *mean_off, const int *bond_off,
                                                const int *in_off, const int *in_bond,
                                                const TF *fbond, const int *row_of_atom,
                                                const double *E_row, double *out, double *Eatom) {
  int i = blockIdx.x * kGatherAtoms + (threadIdx.x >> 4), lane = threadIdx.x & 15;
  if (i >= n) return;  // whole rows of 16 lanes
  double f[3] = {0, 0, 0};
  for (int b = bond_off[i] + lane; b < bond_off[i + 1]; b += 16)
#pragma unroll
    for (int q = 0; q < 3; q++) f[q] += (double)fbond[3 * (size_t)b + q];
  for (int a = in_off[i] + lane; a < in_off[i + 1]; a += 16) {
    int b = in_bond[a];
#pragma unroll
    for (int q = 0; q < 3; q++) f[q] -= (double)fbond[3 * (size_t)b + q];
  }
#pragma unroll
  for (int q = 0; q < 3; q++) f[q] = row16_sum(f[q]);
  if (lane == 0) {
    double *F = out + 3 * (size_t)i;
    if (mean_off) {
      int k = atom_struct[i];
      F = out + mean_off[k] + 1 + 3 * (size_t)(i - atom_off[k]);
    }
    for (int q = 0; q < 3; q++) F[q] = f[q];
    if (Eatom) Eatom[i] = E_row[row_of_atom[i]];
  }
}

// Sums of every chunk of <= 256 atoms of one structure: its atoms' energies
// (first, when NQ is 7) and six virial components.
template <int NQ>
__global__ __launch_bounds__(256) void k_chunk_sums(const int *chunk_begin, const int *chunk_end,
                                                    const int *row_of_atom, const double *E_row,
                                                    const double *vir, double *part) {
  __shared__ double sh[4][NQ];
  int c = blockIdx.x;
  int i = chunk_begin[c] + threadIdx.x;
  bool in = i < chunk_end[c];
  double v[NQ];
  if (NQ == 7) v[0] = in ? E_row[row_of_atom[i]] : 0.0;
#pragma unroll
  for (int q = 0; q < 6; q++) v[NQ - 6 + q] = in ? vir[6 * (size_t)i + q] : 0.0;
#pragma unroll
  for (int q = 0; q < NQ; q++) v[q] = wave_sum(v[q]);
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int q = 0; q < NQ; q++) sh[threadIdx.x >> 6][q] = v[q];
  __syncthreads();
  if (threadIdx.x < NQ) {
    int q = threadIdx.x;
    part[(size_t)c * NQ + q] = (sh[0][q] + sh[1][q]) + (sh[2][q] + sh[3][q]);
  }
}

// Sum of one structure's chunk values, by one wave: lanes take chunks 64
// apart, then sum over the lanes (one thread over all 1,024 chunks of a
// 262,144-atom structure took 164 us, now 8). With the chunks in a launch before
// at every size: one workgroup that went through a structure's chunks itself was
// slower for one structure (gather and sums of 108 atoms 15 us, in three launches
// 11; of 2,048 atoms 21 and 12) and more so for many (2,000 of 40 atoms 78 and
// 32).
template <int NQ>
__device__ __forceinline__ void structure_sums(const int *struct_chunk_off, const double *part,
                                               int k, double (&acc)[NQ]) {
#pragma unroll
  for (int q = 0; q < NQ; q++) acc[q] = 0;
  for (int c = struct_chunk_off[k] + (threadIdx.x & 63); c < struct_chunk_off[k + 1]; c += 64)
#pragma unroll
    for (int q = 0; q < NQ; q++) acc[q] += part[(size_t)c * NQ + q];
#pragma unroll
  for (int q = 0; q < NQ; q++) acc[q] = wave_sum(acc[q]);
}

}  // namespace fm
