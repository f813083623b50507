// Fused bond-basis kernels for the B2 descriptor (descriptors/b2.cpp:181-399)
// and its adjoint (the arithmetic of lammps_descriptor.cpp:250-315 and
// pair_flare.cpp:141-174, driven by dE/dB from the kernel contraction).
//
// Descriptor (k_b2): an atom's bonds are taken in chunks of 32 or 64; lanes
// write the radial values g_n and all harmonics Y_lm of the chunk into LDS tables
// grouped by neighbour species, and the density coefficients accumulate as
// c_t += G_t^T Y_t on the matrix cores (16x16x4, FP32 or FP64) over that
// species' rows only. The power spectrum B_l = C_l C_l^T is a second MFMA
// product, stored straight to the atom's species-sorted row with |B| and
// B.B; c goes to HBM for the adjoint. The mixed variant computes all of
// this in FP64 and writes the FP32 rows and c the adjoint reads plus the
// int8 slices of the FP64 row that the exact kernel contraction consumes.
// Adjoint: u = dE/dc per atom (w = dE/dB and c staged in LDS, u_l = W_l C_l
// on the matrix cores), then the bond forces with lanes over bonds, each
// lane sweeping all (l, m) of its bond by recursion. Dense dc/dr and dB/dr
// are never formed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "fm_device.hpp"
#include "fm_gemm.hpp"
#include "fm_internal.hpp"

namespace fm {

constexpr int kAtomsPerBlock = 4;

struct B2Args {
  int n, nos, N, lmax, H, nrad, nd, cutkind;
  double r1;
  const int *species, *bond_off, *bond_q, *nspec, *row_of_atom;
  const double *rel, *cutoffs;
};

__constant__ double c_knorm[kMaxH];

// 1 / k for the associated-Legendre recursions (k <= lmax + 1).
__constant__ double c_rcp[kMaxL + 2];

// Every real Y_lm (l <= L) of one unit vector u by an (m, l) sweep:
// Y_lm = K_lm Q_l^|m|(u_z) {Re, Im}(u_x + i u_y)^|m| (no Condon-Shortley
// phase; l = 1 gives y, z, x as y_grad.cpp:718-736) with Q_l^m = d^m P_l/dt^m
// from the upward recursion in l. Calls f(lm, Y, px, py, pz); with kGrad,
// (px, py, pz) is the gradient in u of the degree-0 extension
// (dQ_l^m/du_z = Q_l^(m+1)), so grad Y_lm(r) = (p - (u . p) u) / r.
// With LC >= 0 the degree is the compile-time LC (L is ignored) and the
// sweep is fully unrolled: every index and constant-table offset is known
// at compile time.
template <typename T, bool kGrad>
struct YlmState {
  T cm = 1, sm = 0, cm1 = 0, sm1 = 0;  // (u_x + i u_y)^mm and ^(mm - 1)
  T dfact = 1;                         // (2 mm - 1)!!
  T q1 = 0, q2 = 0, p1 = 0, p2 = 0;
};

template <typename T, bool kGrad>
__device__ __forceinline__ void ylm_m_begin(YlmState<T, kGrad> &y, int mm, T ux, T uy) {
  if (mm > 0) {
    y.cm1 = y.cm;
    y.sm1 = y.sm;
    y.cm = y.cm1 * ux - y.sm1 * uy;
    y.sm = y.sm1 * ux + y.cm1 * uy;
    y.dfact *= (T)(2 * mm - 1);
  }
  y.q1 = y.dfact;
  y.q2 = 0;
  y.p1 = 0;
  y.p2 = 0;
}

template <typename T, bool kGrad, typename F>
__device__ __forceinline__ void ylm_step(YlmState<T, kGrad> &y, int mm, int l, T uz, F &f,
                                         const double *knorm = c_knorm) {
  T ql, pl = 0;
  if (l == mm) {
    ql = y.dfact;
  } else {
    ql = ((T)(2 * l - 1) * uz * y.q1 - (T)(l + mm - 1) * y.q2) * (T)c_rcp[l - mm];
    y.q2 = y.q1;
    y.q1 = ql;
    if (kGrad) {
      if (l == mm + 1)
        pl = y.dfact * (T)(2 * mm + 1);
      else
        pl = ((T)(2 * l - 1) * uz * y.p1 - (T)(l + mm) * y.p2) * (T)c_rcp[l - mm - 1];
      y.p2 = y.p1;
      y.p1 = pl;
    }
  }
  int base = l * l + l;
#pragma unroll
  for (int sgn = 0; sgn < 2; sgn++) {
    if (sgn == 1 && mm == 0) break;
    int lm = sgn ? base - mm : base + mm;
    T K = (T)knorm[lm];
    T trig, dtx = 0, dty = 0;
    if (mm == 0) {
      trig = 1;
    } else if (sgn == 0) {
      trig = y.cm;
      dtx = (T)mm * y.cm1;
      dty = -(T)mm * y.sm1;
    } else {
      trig = y.sm;
      dtx = (T)mm * y.sm1;
      dty = (T)mm * y.cm1;
    }
    T Kq = K * ql;
    if (kGrad)
      f(lm, Kq * trig, Kq * dtx, Kq * dty, K * pl * trig);
    else
      f(lm, Kq * trig, T(0), T(0), T(0));
  }
}

// `mine(m)` (wave-uniform) tells which m this wave takes.
struct AllM {
  __device__ __forceinline__ bool operator()(int) const { return true; }
};
template <typename T, bool kGrad, int LC = -1, typename F, typename Mine = AllM>
__device__ __forceinline__ void ylm_sweep(int L, T ux, T uy, T uz, F &&f, Mine mine = Mine(),
                                          const double *knorm = c_knorm) {
  YlmState<T, kGrad> y;
  if constexpr (LC >= 0) {
#pragma unroll
    for (int mm = 0; mm <= LC; mm++) {
      ylm_m_begin<T, kGrad>(y, mm, ux, uy);
      if (!mine(mm)) continue;
#pragma unroll
      for (int l = mm; l <= LC; l++) ylm_step<T, kGrad>(y, mm, l, uz, f, knorm);
    }
  } else {
    for (int mm = 0; mm <= L; mm++) {
      ylm_m_begin<T, kGrad>(y, mm, ux, uy);
      if (!mine(mm)) continue;
      for (int l = mm; l <= L; l++) ylm_step<T, kGrad>(y, mm, l, uz, f, knorm);
    }
  }
}


// 16 x 16 x 4 MFMA in the descriptor precision (FP32 accumulators hold
// rows 4 (lane / 16) + q, FP64 ones rows lane / 16 + 4 q; both take
// A[lane % 16][lane / 16] and B[lane / 16][lane % 16]).
template <typename T>
struct MfmaAcc;
template <>
struct MfmaAcc<float> {
  typedef float type __attribute__((ext_vector_type(4)));
};
template <>
struct MfmaAcc<double> {
  typedef double type __attribute__((ext_vector_type(4)));
};
__device__ __forceinline__ MfmaAcc<float>::type mfma_4(float a, float b,
                                                       MfmaAcc<float>::type c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ MfmaAcc<double>::type mfma_4(double a, double b,
                                                        MfmaAcc<double>::type c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// Keeps an accumulator in its registers across a loop's iterations (the
// compiler otherwise moves it to vector registers and back in each, after
// waiting for the product).
template <typename A>
__device__ __forceinline__ void keep_acc(A &acc) {
  asm volatile("" : "+a"(acc));
}
template <typename T>
__device__ __forceinline__ int mfma_row(int lane, int q) {
  return sizeof(T) == 8 ? (lane >> 4) + 4 * q : 4 * (lane >> 4) + q;
}

// 16-byte vectors in global memory at the alignment of their elements.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

__host__ __device__ inline int pad2(int n) { return (n + 1) & ~1; }

// Workspace (elements of T) of one atom of the descriptor kernel: c, then the
// bond tables of one chunk of ch bonds (Y ch x H, g ch x N) and later the row
// of nd values (0 without B2) over them; even, so that every atom's row is
// 16-byte aligned.
__host__ __device__ inline size_t b2_work(int nc, int H, int N, int ch, int nd) {
  size_t tab = (size_t)ch * ((size_t)H + (size_t)N), row = (size_t)nd;
  return (size_t)pad2(nc) + ((tab > row ? tab : row) + 1) / 2 * 2;
}

// Products of sizes and indices below 2^24 (a full 32-bit product takes four
// times as long).
__device__ __forceinline__ int mul24(int a, int b) {
  return (int)__umul24((unsigned)a, (unsigned)b);
}

// Ordering of LDS accesses among the W waves of an atom.
template <int W>
__device__ __forceinline__ void atom_sync() {
  if constexpr (W > 1) {
    __syncthreads();
  } else {
    wave_lds_sync();
  }
}

// c[(t N + n) H + lm] of atom i for all neighbour species t into LDS
// (b2.cpp:367-395). For each chunk of up to ch bonds, lane k takes
// bond k and writes its radial basis g_n and its Y_lm to LDS tables, the
// rows grouped by neighbour species (list order kept within a species); then,
// per species t and 16 harmonics, c_t += G_t^T Y_t on the matrix cores over
// that species' rows only (A = g_n of the bonds, B = their Y_lm). Of W waves
// per atom, wave w takes the harmonics with m mod 2 W in {w, 2 W - 1 - w}
// (wave 0 the radial basis too) and every W-th tile of 16 harmonics; each value
// is the same whoever computes it.
template <typename T, int LC, int W>
__device__ void accumulate_c(const B2Args &a, int i, int lane, int w, int ch, T *c, T *tab) {
  int si = a.species[i];
  int b0 = a.bond_off[i], b1 = a.bond_off[i + 1];
  int nc = a.nrad * a.H, H = a.H, N = a.N;
  T *Yt = tab, *gt = tab + ch * (size_t)H;
  if (b0 == b1)
    for (int k = 64 * w + lane; k < nc; k += 64 * W) c[k] = 0;
  int r16 = lane & 15, k4 = lane >> 4;
  unsigned long long below = (1ull << lane) - 1ull;
  for (int bb = b0; bb < b1; bb += ch) {
    int nk = min(ch, b1 - bb);
    int q = 0, sj = -1;
    if (lane < nk) {
      q = a.bond_q[bb + lane];
      sj = a.nspec[q];
    }
    // Table row of this lane's bond: its rank among the chunk's bonds of
    // its species, after the rows of the lower species.
    int pos = 0, off = 0;
    for (int t = 0; t < a.nos; t++) {
      unsigned long long m = __ballot(sj == t);
      if (sj == t) pos = off + __popcll(m & below);
      off += __popcll(m);
    }
    atom_sync<W>();
    if (lane < nk) {
      const double *rp = a.rel + 4 * (size_t)q;
      if (w == 0) {
        T g[kMaxN], dg[kMaxN];
        radial_basis<T>((T)rp[0], (T)a.cutoffs[si * a.nos + sj], (T)a.r1, N, a.cutkind, g, dg);
#pragma unroll
        for (int nn = 0; nn < kMaxN; nn++)
          if (nn < N) gt[pos * N + nn] = g[nn];
      }
      T rinv = T(1) / (T)rp[0];
      T *yrow = Yt + (size_t)pos * H;
      // Read in here, not before the loop: all of them exceed the scalar
      // registers.
      const double *knorm = c_knorm;
      if (LC < 0 || LC > 4) asm volatile("" : "+s"(knorm));
      ylm_sweep<T, false, LC>(
          a.lmax, (T)rp[1] * rinv, (T)rp[2] * rinv, (T)rp[3] * rinv,
          [&](int lm, T Y, T, T, T) { yrow[lm] = Y; },
          [&](int m) { m &= 2 * W - 1; return W == 1 || m == w || m == 2 * W - 1 - w; },
          knorm);
    }
    atom_sync<W>();
    // Wave w takes the tiles of 16 harmonics w, w + W, ..: g_n is read once for
    // all of them.
    constexpr int HT = LC >= 0 ? ((LC + 1) * (LC + 1) + 15) / 16 : -LC;
    constexpr int NT = (HT + W - 1) / W, n_step = sizeof(T) == 8 ? 4 : 1;
    int n0 = mfma_row<T>(lane, 0), lm0 = 16 * w + r16;
    int rc = min(r16, N - 1), r0 = 0;
    for (int t = 0; t < a.nos; t++) {
      int r1 = r0 + __popcll(__ballot(sj == t));  // rows [r0, r1) are species t
      // The first chunk sets all of c; a wave past the last harmonic has no tile.
      if ((r1 > r0 || bb == b0) && (W == 1 || 16 * w < H)) {
        typename MfmaAcc<T>::type acc[NT];
        // c of this lane's first value; the others are n_step H apart.
        int at = mul24(t * N + n0, H) + lm0;
#pragma unroll
        for (int j = 0; j < NT; j++) {
          acc[j] = {};
          if (bb > b0 && lm0 + 16 * W * j < H) {
#pragma unroll
            for (int q = 0; q < 4; q++)
              if (n0 + q * n_step < N) acc[j][q] = c[at + 16 * W * j + q * n_step * H];
          }
          keep_acc(acc[j]);
        }
        // Loads are clamped in bounds, then zeroed outside the species' rows.
        int rn = r16 < N ? r1 : 0;
#pragma unroll 1
        for (int k0 = r0; k0 < r1; k0 += 8) {
          T av[2], bv[NT][2];
#pragma unroll
          for (int u = 0; u < 2; u++) {
            int b = k0 + 4 * u + k4, bc = min(b, ch - 1);
            T x = gt[mul24(bc, N) + rc];
            av[u] = b < rn ? x : T(0);
            int yb = mul24(bc, H);
#pragma unroll
            for (int j = 0; j < NT; j++) {
              T y = Yt[yb + min(lm0 + 16 * W * j, H - 1)];
              bv[j][u] = b < r1 ? y : T(0);
            }
          }
#pragma unroll
          for (int u = 0; u < 2; u++)
#pragma unroll
            for (int j = 0; j < NT; j++) acc[j] = mfma_4(av[u], bv[j][u], acc[j]);
#pragma unroll
          for (int j = 0; j < NT; j++) keep_acc(acc[j]);
        }
#pragma unroll
        for (int j = 0; j < NT; j++)
          if (lm0 + 16 * W * j < H) {
#pragma unroll
            for (int q = 0; q < 4; q++)
              if (n0 + q * n_step < N) c[at + 16 * W * j + q * n_step * H] = acc[j][q];
          }
      }
      r0 = r1;
    }
  }
  atom_sync<W>();
}

// The chosen form's outputs of the FP64 descriptor pass (k_b2 with MIXED): the
// B row and c in FP32 (for the adjoint) and the FP64 row as kI8Slices int8
// slices with a power-of-two scale (the kernel contraction's operand, see
// k_slice_rows in fm_gemm.hip for the slicing).
struct MixedOut {
  float *B, *C;
  int8_t *q;  // tiled slice layout, kI8TileA rows per tile
  double *scale;
  long long nk;        // k steps of kI8Pad (the padded reduction length / kI8Pad)
  const int *shift;    // per species: slice row = species-sorted row + shift
};

// The slices of four consecutive values r (|r| < 1), packed four to a word.
// Adding 1.5 2^(52 - s) rounds r to a multiple of 2^-s (to nearest, ties to
// even) and leaves that multiple in the low bits of the sum; every difference
// is exact.
__device__ __forceinline__ void slice4(double (&r)[4], unsigned (&packed)[kI8Slices]) {
#pragma unroll
  for (int p = 0; p < kI8Slices; p++) {
    const double magic = 6755399441055744.0 / (double)(1ll << (6 + 7 * p));
    unsigned d[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      double u = r[j] + magic;
      d[j] = (unsigned)__builtin_bit_cast(unsigned long long, u);
      r[j] -= u - magic;
    }
    unsigned lo = __builtin_amdgcn_perm(d[1], d[0], 0x0c0c0400u);
    unsigned hi = __builtin_amdgcn_perm(d[3], d[2], 0x0c0c0400u);
    packed[p] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
  }
}

// B2 (b2.cpp:209-231) per atom: B[k] = sum_m c[n1, lm] c[n2, lm], written at
// the atom's species-sorted row, with |B| and B.B; the coefficients c go to
// HBM (Cg) for the adjoint. T = float is the bond pass of B3: c alone.
//
// What bounds it: each wave's chain of vector instructions (they take half of
// the cycles, the products an eighth; slicing each value on its own where the
// MFMA tile leaves it was more than half of them). So the FP64 row is staged in
// LDS (over the bond tables, no longer needed) and sliced four consecutive
// values at a time, the three tiles of an l share two operands, and the tiles of
// a species share g. 262144 atoms of three species, l_max 6, 42 bonds: 6.5 ms
// (10.4 before, 2.4 at the rates of copies and FP64 products). The
// row is the largest part of an atom's LDS; where that leaves a CU few atoms,
// W = 2 or 4 waves share one and split every phase. B.B keeps its order of
// sums (the variances depend on its last bit): wave 0 takes it from the staged
// row where the waves split the tiles. A row too long for LDS (stage = 0, one
// wave, more than 32 radial functions) is written from the tiles.
template <typename T, int LC, bool MIXED, int W>
__global__ __launch_bounds__(256) void k_b2(B2Args a, T *B, double *norm, double *nn, T *Cg,
                                            int want_b2, int work, int ch, int stage,
                                            MixedOut mo) {
  extern __shared__ __align__(16) unsigned char smem[];
  int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int w = wave % W, slot = wave / W;
  int i = blockIdx.x * (blockDim.x / (64 * W)) + slot;  // W > 1: one atom per block
  if (i >= a.n) return;
  constexpr int NT = 64 * W;
  int tid = 64 * w + lane;  // thread of this atom
  int nc = a.nrad * a.H, H = a.H, nr = a.nrad;
  T *c = reinterpret_cast<T *>(smem) + (size_t)slot * work;  // work: elements per atom
  T *tab = c + pad2(nc);
  accumulate_c<T, LC, W>(a, i, lane, w, ch, c, tab);
  if constexpr (MIXED) {
    for (int k = tid; k < nc; k += NT) mo.C[(size_t)i * nc + k] = (float)c[k];
  } else {
    for (int k = tid; k < nc; k += NT) Cg[(size_t)i * nc + k] = c[k];
  }
  if constexpr (sizeof(T) == 8) {
    if (!want_b2) return;
    // B_l = C_l C_l^T on the matrix cores (C_l[n][m] = c[n, l^2 + m]); the
    // upper triangle n2 >= n1 belongs at p(n1, n2) (L + 1) + l of the row.
    int L1 = a.lmax + 1;
    int r16 = lane & 15, k4 = lane >> 4;
    int row = a.row_of_atom[i];
    T *bst = tab;
    T s2 = 0;
    // One 16 x 16 tile of B_l (operand elements past 2 l + 1, which are the
    // next c values or lie in the tables, replaced by zero).
    auto tile_of = [&](int l, int rt, int cc) {
      int nm = 2 * l + 1, lm0 = l * l;
      typename MfmaAcc<T>::type acc = {};
      const T *ca = c + min(rt + r16, nr - 1) * H + lm0 + k4;
      const T *cb = c + min(cc + r16, nr - 1) * H + lm0 + k4;
#pragma unroll 1
      for (int k0 = 0; k0 < nm; k0 += 4) {
        T x = ca[k0], y = cb[k0];
        bool in = k0 + k4 < nm;
        acc = mfma_4(in ? x : T(0), in ? y : T(0), acc);
        keep_acc(acc);
      }
      return acc;
    };
    // Place of this lane's value q of tile (rt, cc) for l = 0, or -1.
    auto place = [&](int rt, int cc, int q) {
      int n1 = rt + mfma_row<T>(lane, q), n2 = cc + r16;
      int at = mul24(mul24(n1, nr) - (mul24(n1, n1 - 1) >> 1) + (n2 - n1), L1);
      return n1 < nr && n2 < nr && n2 >= n1 ? at : -1;
    };
    // The row's power-of-two scale 2^E from its largest element, which is a
    // diagonal one (Cauchy-Schwarz within each l); every wave finds it.
    auto exponent = [&](auto diagonal) {
      double mx = 0;
      for (int n = lane; n < nr; n += 64)
        for (int l = 0; l < L1; l++) mx = fmax(mx, diagonal(n, l));
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
      int E = 0;
      if (mx > 0) frexp(mx, &E);  // mx = m 2^E, m in [0.5, 1)
      return E;
    };
    if (nr <= 32) {
      // Up to three tiles, (0, 0), (0, 16) and (16, 16), of two operands; their
      // places kept. Wave of an l: the long ones first, each paired with a short
      // one.
      int at[3][4];
#pragma unroll
      for (int u = 0; u < 3; u++)
#pragma unroll
        for (int q = 0; q < 4; q++) at[u][q] = place(u == 2 ? 16 : 0, u ? 16 : 0, q);
      int nt = nr > 16 ? 3 : 1;
      const T *c0 = c + mul24(min(r16, nr - 1), H) + k4;
      const T *c1 = c + mul24(min(16 + r16, nr - 1), H) + k4;
      for (int l = 0; l <= a.lmax; l++) {
        if (W > 1 && (2 * l > a.lmax ? a.lmax - l : l + 1) % W != w) continue;
        int nm = 2 * l + 1, lm0 = l * l;
        typename MfmaAcc<T>::type acc[3] = {};
#pragma unroll
        for (int u = 0; u < 3; u++) keep_acc(acc[u]);
        if (nt == 3) {
#pragma unroll 1
          for (int k0 = 0; k0 < nm; k0 += 4) {
            bool in = k0 + k4 < nm;
            T x = c0[lm0 + k0], y = c1[lm0 + k0];
            x = in ? x : T(0);
            y = in ? y : T(0);
            acc[0] = mfma_4(x, x, acc[0]);
            acc[1] = mfma_4(x, y, acc[1]);
            acc[2] = mfma_4(y, y, acc[2]);
#pragma unroll
            for (int u = 0; u < 3; u++) keep_acc(acc[u]);
          }
        } else {
#pragma unroll 1
          for (int k0 = 0; k0 < nm; k0 += 4) {
            T x = c0[lm0 + k0];
            x = k0 + k4 < nm ? x : T(0);
            acc[0] = mfma_4(x, x, acc[0]);
            keep_acc(acc[0]);
          }
        }
#pragma unroll
        for (int u = 0; u < 3; u++) {
          if (u >= nt) continue;
#pragma unroll
          for (int q = 0; q < 4; q++)
            if (at[u][q] >= 0) {
              T v = acc[u][q];
              bst[at[u][q] + l] = v;
              if (W == 1) s2 += v * v;
            }
        }
      }
      if constexpr (W > 1) {
        atom_sync<W>();
        if (w == 0)
          for (int l = 0; l <= a.lmax; l++)
#pragma unroll
            for (int u = 0; u < 3; u++) {
              if (u >= nt) continue;
#pragma unroll
              for (int q = 0; q < 4; q++)
                if (at[u][q] >= 0) {
                  T v = bst[at[u][q] + l];
                  s2 += v * v;
                }
            }
      }
    } else if (W == 1 && !stage) {
      double inv = 0;
      int8_t *qp = nullptr;
      if constexpr (MIXED) {
        int E = exponent([&](int n, int l) {
          const T *cn = c + n * H + l * l;
          double sq = 0;
          for (int m = 0; m < 2 * l + 1; m++) sq += (double)cn[m] * (double)cn[m];
          return sq;
        });
        inv = ldexp(1.0, -E);
        if (lane == 0) mo.scale[row] = ldexp(1.0, E);
        qp = mo.q + i8_tile_offset(kI8TileA, mo.nk, row + mo.shift[a.species[i]], 0, 0);
      }
      auto slices = [&](int k, double r) {
        double rr[4] = {r, 0, 0, 0};
        unsigned packed[kI8Slices];
        slice4(rr, packed);
        int8_t *dst = qp + (size_t)(k >> 6) * (kI8Slices * kI8TileA * kI8Pad) + (k & (kI8Pad - 1));
        for (int p = 0; p < kI8Slices; p++) dst[p * (kI8TileA * kI8Pad)] = (int8_t)packed[p];
      };
      for (int l = 0; l <= a.lmax; l++)
        for (int rt = 0; rt < nr; rt += 16)
          for (int cc = rt; cc < nr; cc += 16) {
            auto acc = tile_of(l, rt, cc);
#pragma unroll
            for (int q = 0; q < 4; q++) {
              int k = place(rt, cc, q) + l;
              if (k < l) continue;
              T v = acc[q];
              s2 += v * v;
              if constexpr (MIXED) {
                mo.B[(size_t)row * a.nd + k] = (float)v;
                slices(k, (double)v * inv);
              } else {
                B[(size_t)row * a.nd + k] = v;
              }
            }
          }
      if constexpr (MIXED)
        for (int k = a.nd + lane; k < (int)(mo.nk * kI8Pad); k += 64) slices(k, 0.0);
    } else {
      int tile = 0;
      for (int l = 0; l <= a.lmax; l++)
        for (int rt = 0; rt < nr; rt += 16)
          for (int cc = rt; cc < nr; cc += 16) {
            if (W > 1 && tile++ % W != w) continue;
            auto acc = tile_of(l, rt, cc);
#pragma unroll
            for (int q = 0; q < 4; q++) {
              int k = place(rt, cc, q);
              if (k >= 0) {
                T v = acc[q];
                bst[k + l] = v;
                if (W == 1) s2 += v * v;
              }
            }
          }
      if constexpr (W > 1) {
        atom_sync<W>();
        if (w == 0)
          for (int l = 0; l <= a.lmax; l++)
            for (int rt = 0; rt < nr; rt += 16)
              for (int cc = rt; cc < nr; cc += 16)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                  int k = place(rt, cc, q);
                  if (k >= 0) {
                    T v = bst[k + l];
                    s2 += v * v;
                  }
                }
      }
    }
    if constexpr (W == 1) atom_sync<W>();
    if (!stage) {
    } else if constexpr (MIXED) {
      int E = exponent([&](int n, int l) {
        return (double)bst[mul24(mul24(n, nr) - (mul24(n, n - 1) >> 1), L1) + l];
      });
      double inv = ldexp(1.0, -E);
      if (tid == 0) mo.scale[row] = ldexp(1.0, E);
      long long qrow = row + mo.shift[a.species[i]];
      int Kq = (int)(mo.nk * kI8Pad);
      float *B32 = mo.B + (size_t)row * a.nd;
      int8_t *qp = mo.q + i8_tile_offset(kI8TileA, mo.nk, qrow, 0, 0);
      for (int k0 = 4 * tid; k0 < Kq; k0 += 4 * NT) {
        double r[4];
        if (k0 + 4 <= a.nd) {
          double2 x = *reinterpret_cast<const double2 *>(&bst[k0]);
          double2 y = *reinterpret_cast<const double2 *>(&bst[k0 + 2]);
          r[0] = x.x, r[1] = x.y, r[2] = y.x, r[3] = y.y;
          f4u v = {(float)r[0], (float)r[1], (float)r[2], (float)r[3]};
          *reinterpret_cast<f4u *>(B32 + k0) = v;
        } else {
#pragma unroll
          for (int j = 0; j < 4; j++) {
            r[j] = k0 + j < a.nd ? bst[k0 + j] : 0.0;
            if (k0 + j < a.nd) B32[k0 + j] = (float)r[j];
          }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) r[j] *= inv;
        unsigned packed[kI8Slices];
        slice4(r, packed);
        // k0's step of the row tile (kI8Slices blocks of kI8TileA rows), then
        // its place in the row.
        unsigned at = mul24(k0 >> 6, kI8Slices * kI8TileA * kI8Pad) + (k0 & (kI8Pad - 1));
#pragma unroll
        for (int p = 0; p < kI8Slices; p++) {
          int8_t *dst = qp + p * (kI8TileA * kI8Pad);
          asm volatile("" : "+s"(dst));  // scalar base, one vector offset
          *reinterpret_cast<unsigned *>(dst + at) = packed[p];
        }
      }
    } else {
      T *Brow = B + (size_t)row * a.nd;
      for (int k = 2 * tid; k + 1 < a.nd; k += 2 * NT)
        *reinterpret_cast<d2u *>(Brow + k) = *reinterpret_cast<const d2u *>(&bst[k]);
      if ((a.nd & 1) && tid == 0) Brow[a.nd - 1] = bst[a.nd - 1];
    }
    if (w == 0) {
      s2 = wave_sum(s2);
      if (lane == 0) {
        norm[row] = (double)sqrt(s2);
        nn[row] = (double)s2;
      }
    }
  }
}

// Adjoint, first half, per atom (one wavefront): with `project` set,
// w = dE/dB = (G - (G.B_hat) B_hat)/|B| from G = dE/dB_hat |B| (for the
// sparse GP, G = sum_j sigma^2 alpha_j p S_j^(p-1) x_hat_j, the closed form of
// normalized_dot_product.cpp:191-195); without it w = G (unnormalised
// kernels). Then u = dE/dc (lammps_descriptor.cpp:286-314):
// u[n1, lm] = sum_n2 (1 + [n1 = n2]) w[(min, max)(n1, n2), l] c[n2, lm]. An
// atom with |B| < empty_norm or B.B < empty_nn contributes nothing (its u is
// not read).
struct AdjArgs {
  int project;
  double empty_norm, empty_nn;
  // With project: G . B per row from the local energies when given,
  // G . B = p |B| E (G = sum_j sigma^2 alpha_j p S_j^(p-1) x_hat_j and
  // E = sum_j sigma^2 alpha_j S_j^p), else a pass over the G and B rows.
  const double *energy;
  double power;
};

__device__ __forceinline__ int pair_index(int lo, int hi, int nr) {
  return lo * nr - (lo * (lo - 1)) / 2 + (hi - lo);
}

__host__ __device__ inline int pad4(int n) { return (n + 3) & ~3; }

// n elements from global memory to LDS: 16-byte vectors when the source is
// 16-byte aligned (the LDS destination always is), four in flight per lane.
template <typename T>
__device__ __forceinline__ void stage_row(const T *src, T *dst, int n, int lane, int nt = 64) {
  constexpr int E = 16 / sizeof(T);
  int done = 0;
  if ((reinterpret_cast<uintptr_t>(src) & 15) == 0) {
    using V = typename std::conditional<sizeof(T) == 4, float4, double2>::type;
    const V *sv = reinterpret_cast<const V *>(src);
    V *dv = reinterpret_cast<V *>(dst);
    int nv = n / E;
#pragma unroll 4
    for (int v = lane; v < nv; v += nt) dv[v] = sv[v];
    done = nv * E;
  }
  for (int k = done + lane; k < n; k += nt) dst[k] = src[k];
}

// G . B over the elements of one row that this lane's wave takes (nt lanes
// stride the row; nt = 64: the whole row), summed over the wave: 16-byte
// loads of both rows when both are 16-byte aligned (all of a lane's vectors
// in flight together), a fixed order per lane and a fixed wave reduction.
template <typename T>
__device__ __forceinline__ T row_dot(const T *G, const T *B, int n, int lane, int nt = 64) {
  // Lane l takes the E-element groups v = l, l + nt, ... and the tail
  // elements nv E + l, ...: the same elements in the same order whether a
  // group arrives as one 16-byte load or as E scalar ones, so the sum does
  // not depend on where the rows sit in memory (an atom's row is placed
  // differently alone and in a batch).
  constexpr int E = 16 / sizeof(T);
  using V = typename std::conditional<sizeof(T) == 4, float4, double2>::type;
  T acc = 0;
  int nv = n / E;
  if (((reinterpret_cast<uintptr_t>(G) | reinterpret_cast<uintptr_t>(B)) & 15) == 0) {
    const V *gv = reinterpret_cast<const V *>(G), *bv = reinterpret_cast<const V *>(B);
#pragma unroll 8
    for (int v = lane; v < nv; v += nt) {
      V x = gv[v], y = bv[v];
      const T *xs = reinterpret_cast<const T *>(&x), *ys = reinterpret_cast<const T *>(&y);
#pragma unroll
      for (int e = 0; e < E; e++) acc = fma(xs[e], ys[e], acc);
    }
  } else {
#pragma unroll 4
    for (int v = lane; v < nv; v += nt)
#pragma unroll
      for (int e = 0; e < E; e++) acc = fma(G[E * v + e], B[E * v + e], acc);
  }
  for (int k = nv * E + lane; k < n; k += nt) acc = fma(G[k], B[k], acc);
  return wave_sum(acc);
}

// w = sg G - sb B (the atom's dE/dB row) into LDS, n elements: 16-byte
// loads of G and B when both rows are 16-byte aligned, four vectors of each
// in flight per lane; B is not read when sb is zero. Every element is the
// same fma(sg, G, -sb B) on either path.
template <typename T>
__device__ __forceinline__ T w_elem(T sg, T g, T sb, T b) {
  return fma(sg, g, -(sb * b));
}

template <typename T>
__device__ __forceinline__ void stage_w(const T *G, const T *B, T sg, T sb, T *w, int n,
                                        int lane, int nt = 64) {
  constexpr int E = 16 / sizeof(T);
  int done = 0;
  bool withb = sb != T(0);
  if (((reinterpret_cast<uintptr_t>(G) | (withb ? reinterpret_cast<uintptr_t>(B) : 0)) & 15) ==
      0) {
    using V = typename std::conditional<sizeof(T) == 4, float4, double2>::type;
    const V *gv = reinterpret_cast<const V *>(G), *bv = reinterpret_cast<const V *>(B);
    V *wv = reinterpret_cast<V *>(w);
    int nv = n / E;
    if (withb) {
#pragma unroll 4
      for (int v = lane; v < nv; v += nt) {
        V x = gv[v], y = bv[v], r;
        const T *xs = reinterpret_cast<const T *>(&x), *ys = reinterpret_cast<const T *>(&y);
        T *rs = reinterpret_cast<T *>(&r);
#pragma unroll
        for (int e = 0; e < E; e++) rs[e] = w_elem(sg, xs[e], sb, ys[e]);
        wv[v] = r;
      }
    } else {
#pragma unroll 4
      for (int v = lane; v < nv; v += nt) {
        V x = gv[v], r;
        const T *xs = reinterpret_cast<const T *>(&x);
        T *rs = reinterpret_cast<T *>(&r);
#pragma unroll
        for (int e = 0; e < E; e++) rs[e] = sg * xs[e];
        wv[v] = r;
      }
    }
    done = nv * E;
  }
  for (int k = done + lane; k < n; k += nt)
    w[k] = withb ? w_elem(sg, G[k], sb, B[k]) : sg * G[k];
}

// FP32 rows: G . B and w = sg G - sb B in one pass over both rows. Each of the
// atom's 128 threads loads all of its V-vectors of G and B (at most R of each,
// rows of at most 128 R E elements) before it uses the first; waiting for each
// in turn kept 80 % of the wave cycles idle (262144 atoms of 3,255 elements: the
// call 44.1 ms, now 42.7; 512 structures of 1,500 in two passes 11.6, now 11.4,
// beside the variance on the other stream). The partition and the order of the dot
// are those of row_dot for vectors of four, and single elements 128 apart for V =
// float. sb_of(a, b) makes sb of the two wavefronts' dots; red holds them; the
// barrier inside is reached by every thread of the block (dead atoms load the
// first row).
template <typename V, int R, typename F>
__device__ __forceinline__ void stage_w_onepass(const float *G, const float *B, float sg,
                                                F &&sb_of, float *wl, int n, bool live, int t2,
                                                int lane, int w, int slot, float *red) {
  constexpr int E = sizeof(V) / sizeof(float);
  const V *gv = reinterpret_cast<const V *>(G), *bv = reinterpret_cast<const V *>(B);
  int nv = n / E;
  V g[R], b[R];
#pragma unroll
  for (int j = 0; j < R; j++) {
    int v = max(min(t2 + 128 * j, nv - 1), 0);
    g[j] = nv > 0 ? gv[v] : V{};
    b[j] = nv > 0 ? bv[v] : V{};
  }
  int kt = nv * E + t2;
  bool tail = kt < n;
  float gt = tail ? G[kt] : 0.f, bt = tail ? B[kt] : 0.f;
  float acc = 0;
#pragma unroll
  for (int j = 0; j < R; j++) {
    const float *xs = reinterpret_cast<const float *>(&g[j]);
    const float *ys = reinterpret_cast<const float *>(&b[j]);
    float sum = acc;
#pragma unroll
    for (int e = 0; e < E; e++) sum = fma(xs[e], ys[e], sum);
    acc = t2 + 128 * j < nv ? sum : acc;
  }
  acc = fma(gt, bt, acc);
  acc = wave_sum(acc);
  if (lane == 0) red[w] = acc;
  __syncthreads();
  if (!live) return;
  float sb = sb_of(red[2 * slot], red[2 * slot + 1]);
  V *wv = reinterpret_cast<V *>(wl);
#pragma unroll
  for (int j = 0; j < R; j++) {
    int v = t2 + 128 * j;
    if (v < nv) {
      V r;
      float *rs = reinterpret_cast<float *>(&r);
      const float *xs = reinterpret_cast<const float *>(&g[j]);
      const float *ys = reinterpret_cast<const float *>(&b[j]);
#pragma unroll
      for (int e = 0; e < E; e++) rs[e] = w_elem(sg, xs[e], sb, ys[e]);
      wv[v] = r;
    }
  }
  if (tail) wl[kt] = w_elem(sg, gt, sb, bt);
}

// Longest row whose G and B k_dEdc<float, LC, OP> holds in registers, OP = 4 up to
// half of it and 8 above.
constexpr int kOnePassRow = 128 * 32;

// LC >= 0: l_max known at compile time (one accumulator per l up to it, in
// place of kMaxL + 1); LC = -1 for any l_max. OP > 0 (FP32 only):
// projection from the rows with one pass over G and B, of at most 512 OP elements
// (`single`: by single elements where rows are not 16-byte aligned). Two
// wavefronts per atom share
// its LDS rows: both stage (twice the loads in flight per atom for the same
// LDS) and each takes half of the 16-row output tiles.
template <typename T, int LC, int OP = 0>
__global__ __launch_bounds__(128 * kAtomsPerBlock) void k_dEdc(B2Args a, const T *B,
                                                                 const double *norm,
                                                                 const double *nnv, const T *G,
                                                                 long long g_ld, AdjArgs aa,
                                                                 const T *Cg, T *Ug,
                                                                 int single) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ T red[2 * kAtomsPerBlock];
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6, slot = w >> 1, sub = w & 1;
  int t2 = threadIdx.x & 127;  // thread of the atom's two wavefronts
  int i = blockIdx.x * (blockDim.x >> 7) + slot;
  int nc = a.nrad * a.H, ncp = pad4(nc), ndp = pad4(a.nd);
  T *c = reinterpret_cast<T *>(smem) + (size_t)slot * ((size_t)ncp + (size_t)ndp);
  T *wl = c + ncp;  // the w = dE/dB row
  // Atoms past the end or empty skip the work but stay for the barriers.
  bool live = i < a.n;
  int row = live ? a.row_of_atom[i] : 0;
  double nrm = live ? norm[row] : 1.0;
  live = live && !(nrm < aa.empty_norm || nnv[row] < aa.empty_nn);
  const T *Brow = B + (size_t)row * a.nd;
  const T *Grow = G + (size_t)row * g_ld;
  // w = dE/dB = (G - (G . B_hat) B_hat) / |B| = sg G - sb B.
  T ninv = T(1) / (T)nrm;
  T sg = aa.project ? ninv : T(1), sb = 0;
  if constexpr (OP > 0 && sizeof(T) == 4) {
    // The launch guarantees project, no energies and nd <= 512 OP.
    if (live) stage_row(Cg + (size_t)i * nc, c, nc, t2, 128);
    // Every row 16-byte aligned: the same for all atoms of the grid, so the
    // whole block takes one branch and one barrier.
    bool al = ((reinterpret_cast<uintptr_t>(G) | reinterpret_cast<uintptr_t>(B)) & 15) == 0 &&
              (g_ld & 3) == 0 && (a.nd & 3) == 0;
    float s3 = ninv * ninv * ninv;
    if (!single)
      stage_w_onepass<f4u, OP>(
          Grow, Brow, sg, [&](float x, float y) { return (x + y) * ninv * ninv * ninv; }, wl,
          a.nd, live, t2, lane, w, slot, red);
    else if (al)
      stage_w_onepass<f4u, OP>(
          Grow, Brow, sg, [&](float x, float y) { return (x + y) * s3; }, wl, a.nd, live, t2,
          lane, w, slot, red);
    else
      stage_w_onepass<float, 4 * OP>(
          Grow, Brow, sg, [&](float x, float y) { return (x + y) * s3; }, wl, a.nd, live, t2,
          lane, w, slot, red);
  } else {
    if (aa.project) {
      if (aa.energy) {
        if (live) sb = (T)(aa.power * aa.energy[row] / (nrm * nrm));
      } else {
        T part = live ? row_dot(Grow, Brow, a.nd, t2, 128) : T(0);
        if (lane == 0) red[w] = part;
        __syncthreads();
        sb = (red[2 * slot] + red[2 * slot + 1]) * ninv * ninv * ninv;
      }
    }
    // One pass over HBM with 16-byte loads: c and w to LDS.
    if (live) {
      stage_row(Cg + (size_t)i * nc, c, nc, t2, 128);
      stage_w(Grow, Brow, sg, sb, wl, a.nd, t2, 128);
    }
  }
  __syncthreads();
  if (!live) return;
  // u_l = W_l C_l per l on the matrix cores: W_l[n1][n2] = (1 + [n1 = n2])
  // w[p(min, max), l] (nr x nr, symmetric), C_l[n2][m] = c[n2, l^2 + m]
  // (nr x (2l + 1)); 16 x 16 output tiles, 4 n2 per MFMA. Lane L supplies
  // A[L % 16][L / 16] and B[L / 16][L % 16]; it holds output rows
  // tile_row(L, i), column L % 16. The l loop is innermost (one accumulator
  // per l) so the pair index of (n1, n2) is formed once for all l.
  int L1 = a.lmax + 1, nr = a.nrad;
  T *urow = Ug + (size_t)i * nc;
  int r16 = lane & 15, k4 = lane >> 4;
  for (int ct = 0; ct < 2 * a.lmax + 1; ct += 16) {
    for (int rt = 16 * sub; rt < nr; rt += 32) {
      constexpr int KL = LC >= 0 ? LC : kMaxL;
      typename MfmaAcc<T>::type acc[KL + 1];
#pragma unroll
      for (int l = 0; l <= KL; l++) acc[l] = {};
      int n1 = rt + r16, m = ct + r16;
      for (int k0 = 0; k0 < nr; k0 += 4) {
        int n2 = k0 + k4;
        bool ok = n1 < nr && n2 < nr;
        int lo = n1 < n2 ? n1 : n2, hi = n1 < n2 ? n2 : n1;
        int p0 = ok ? pair_index(lo, hi, nr) * L1 : 0;
        T coef = n1 == n2 ? T(2) : T(1);
        const T *cr = c + (n2 < nr ? n2 : 0) * a.H;
        // Loads clamped in bounds and zeroed by selects (no divergent branches).
#pragma unroll
        for (int l = 0; l <= KL; l++) {
          int nm = 2 * l + 1;
          if (l <= a.lmax && ct < nm) {
            int mc = m < nm ? m : nm - 1;
            T g = wl[p0 + l], x = cr[l * l + mc];
            T av = ok ? coef * g : T(0);
            T bv = (n2 < nr && m < nm) ? x : T(0);
            acc[l] = mfma_4(av, bv, acc[l]);
          }
        }
      }
#pragma unroll
      for (int l = 0; l <= KL; l++) {
        int nm = 2 * l + 1;
        if (l <= a.lmax && ct < nm) {
#pragma unroll
          for (int q = 0; q < 4; q++) {
            int row = rt + mfma_row<T>(lane, q);
            if (row < nr && m < nm) urow[row * a.H + l * l + m] = acc[l][q];
          }
        }
      }
    }
  }
}

__device__ __forceinline__ void load4_lds(const float *p, float (&o)[4]) {
  float4 v = *reinterpret_cast<const float4 *>(p);
  o[0] = v.x, o[1] = v.y, o[2] = v.z, o[3] = v.w;
}
__device__ __forceinline__ void load4_lds(const double *p, double (&o)[4]) {
  double2 v0 = *reinterpret_cast<const double2 *>(p);
  double2 v1 = *reinterpret_cast<const double2 *>(p + 2);
  o[0] = v0.x, o[1] = v0.y, o[2] = v1.x, o[3] = v1.y;
}

// Adjoint, second half: per bond f = dE_i/dr_ij = sum_{n,lm} u[s_j n, lm]
// grad(g_n Y_lm) (pair_flare.cpp:141-150, the adjoint of b2.cpp:219-228).
// One wavefront per atom, lanes over its bonds; each lane sweeps every
// (l, m) of its bond (ylm_sweep with gradients) and contracts with u staged
// in LDS:
//   f = a u_hat + (P - (u_hat . P) u_hat) / r,
//   a = sum_lm (sum_n u dg_n) Y_lm,  P = sum_lm (sum_n u g_n) grad_u Y_lm,
// with grad_u the gradient of the degree-0 extension in u. Writes f for every
// bond and the atom's virial -sum_b f (x) r_b (xx, xy, xz, yy, yz, zz).
//
// What bounds it: vector arithmetic (half of the sweep's instructions are the
// contraction's FMAs). NG, the groups of 4 radial functions, is a template
// argument, so that all of a step's u is read at once and no branch is left per
// radial function. u comes with several loads in flight and is placed without
// a division. With a branch per function, and u value by value with two
// divisions each, the kernel took 2.3 ms, now 1.4 (FP32, 262,144 atoms, 10
// radial functions, l_max 6, 42 bonds), and 204 us, now 143 (FP64, 64
// structures, 8 functions, l_max 4). fma is written out where the product that
// the compiler chooses to fuse depends on NG.
template <typename T, int NG>
__global__ __launch_bounds__(64 * kAtomsPerBlock) void k_bond_forces(B2Args a,
                                                                       const double *norm,
                                                                       const double *nnv,
                                                                       AdjArgs aa, const T *Ug,
                                                                       T *fbond, double *vir,
                                                                       const int *atom_list,
                                                                       int n_list) {
  extern __shared__ __align__(16) unsigned char smem[];
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int k = blockIdx.x * (blockDim.x >> 6) + w;
  if (k >= n_list) return;
  int i = atom_list ? atom_list[k] : k;  // all atoms, or those of a row tile
  constexpr int Np = 4 * NG;
  int nc = a.nrad * a.H;
  // u in LDS as [species][lm][n] with n padded to 4, so a lane reads the
  // radial coefficients of one (species, lm) with 16-byte loads.
  T *u = reinterpret_cast<T *>(smem) + (size_t)w * a.nos * a.H * Np;
  int row = a.row_of_atom[i];
  int b0 = a.bond_off[i], b1 = a.bond_off[i + 1];
  double nrm = norm[row];
  if (nrm < aa.empty_norm || nnv[row] < aa.empty_nn) {
    // Empty environment: no force contribution (normalized_dot_product.cpp:171,
    // pair_flare.cpp:134-136).
    for (int b = b0 + lane; b < b1; b += 64) {
      fbond[3 * (size_t)b] = 0;
      fbond[3 * (size_t)b + 1] = 0;
      fbond[3 * (size_t)b + 2] = 0;
    }
    if (lane < 6) vir[6 * (size_t)i + lane] = 0;
    return;
  }
  int si = a.species[i];
  int L = a.lmax, H = a.H, N = a.N;
  // A lane's bond: species, r, x, y, z. The first one is on its way while u is.
  int sj = 0;
  double rel[4];
  auto bond = [&](int b) {
    if (b >= b1) return;
    int q = a.bond_q[b];
    sj = a.nspec[q];
#pragma unroll
    for (int c = 0; c < 4; c++) rel[c] = a.rel[4 * (size_t)q + c];
  };
  bond(b0 + lane);
  {
    // Value k of u is (s, n, lm) = (k / (N H), k / H % N, k % H); 64 values on,
    // the indices move by `ds`, `dn` and `dl`.
    int n1 = lane / H, lm = lane - n1 * H, s = n1 / N, n = n1 - s * N;
    int d = 64 / H, dl = 64 - d * H, ds = d / N, dn = d - ds * N;
    const T *up = Ug + (size_t)i * nc;
    constexpr int U = 32 / sizeof(T);
    for (int k0 = lane; k0 < nc; k0 += 64 * U) {
      T in[U];
#pragma unroll
      for (int j = 0; j < U; j++) in[j] = up[min(k0 + 64 * j, nc - 1)];
#pragma unroll
      for (int j = 0; j < U; j++) {
        if (k0 + 64 * j < nc) u[((size_t)s * H + lm) * Np + n] = in[j];
        lm += dl, n += dn, s += ds;
        if (lm >= H) lm -= H, n++;
        if (n >= N) n -= N, s++;
      }
    }
    if (N < Np)  // zeros in the padding
      for (int k = lane; k < a.nos * H; k += 64)
        for (int n = N; n < Np; n++) u[(size_t)k * Np + n] = 0;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  double v[6] = {0, 0, 0, 0, 0, 0};
  for (int bb = b0; bb < b1; bb += 64) {
    int b = bb + lane;
    if (b < b1) {
      T r = (T)rel[0], x = (T)rel[1], y = (T)rel[2], z = (T)rel[3];
      T rc = (T)a.cutoffs[si * a.nos + sj];
      T g[kMaxN], dg[kMaxN];
      radial_basis<T>(r, rc, (T)a.r1, N, a.cutkind, g, dg);
      T rinv = T(1) / r;
      T ux = x * rinv, uy = y * rinv, uz = z * rinv;
      const T *ub = u + (size_t)sj * H * Np;
      T acc_a = 0, Px = 0, Py = 0, Pz = 0;
      ylm_sweep<T, true>(L, ux, uy, uz, [&](int lm, T Y, T px, T py, T pz) {
        T s0 = 0, s1 = 0, uu[NG][4];
        const T *ul = ub + lm * Np;
#pragma unroll
        for (int n4 = 0; n4 < NG; n4++) load4_lds(ul + 4 * n4, uu[n4]);
#pragma unroll
        for (int n = 0; n < 4 * NG; n++) {
          s0 = fma(uu[n / 4][n % 4], g[n], s0);
          s1 = fma(uu[n / 4][n % 4], dg[n], s1);
        }
        acc_a += s1 * Y;
        Px += s0 * px;
        Py += s0 * py;
        Pz += s0 * pz;
      });
      T up = fma(uz, Pz, fma(ux, Px, uy * Py));
      T fx = acc_a * ux + (Px - up * ux) * rinv;
      T fy = acc_a * uy + (Py - up * uy) * rinv;
      T fz = acc_a * uz + (Pz - up * uz) * rinv;
      fbond[3 * (size_t)b] = fx;
      fbond[3 * (size_t)b + 1] = fy;
      fbond[3 * (size_t)b + 2] = fz;
      double f3[3] = {(double)fx, (double)fy, (double)fz};
      double r3[3] = {rel[1], rel[2], rel[3]};
      int sc = 0;
      for (int c1 = 0; c1 < 3; c1++)
        for (int c2 = c1; c2 < 3; c2++) v[sc++] -= f3[c1] * r3[c2];
      bond(b + 64);
    }
  }
#pragma unroll
  for (int k = 0; k < 6; k++) v[k] = wave_sum(v[k]);
  if (lane == 0)
    for (int k = 0; k < 6; k++) vir[6 * (size_t)i + k] = v[k];
}

// Atoms (wavefronts) per block: of 1, 2 and 4, the one that keeps the most
// atoms resident on a CU within its 160 KB of LDS (larger on ties).
static int atoms_per_block(size_t lds_per_atom) {
  const size_t cap = 160 * 1024;
  FM_CHECK(lds_per_atom <= cap, FM_ERR_CAPACITY, "per-atom descriptor workspace exceeds LDS");
  int best = 1;
  size_t best_res = 0;
  for (int apb = 1; apb <= kAtomsPerBlock; apb <<= 1) {
    size_t blocks = cap / (apb * lds_per_atom);
    size_t res = std::min<size_t>(blocks, 8) * apb;  // at most 8 blocks of ours per CU here
    if (blocks > 0 && res >= best_res) {
      best = apb;
      best_res = res;
    }
  }
  return best;
}

// Atoms resident per CU with lds_per_atom bytes each (the residency
// atoms_per_block maximises).
static size_t resident_atoms(size_t lds_per_atom) {
  const size_t cap = 160 * 1024;
  if (lds_per_atom > cap) return 0;
  int apb = atoms_per_block(lds_per_atom);
  return std::min<size_t>(cap / (apb * lds_per_atom), 8) * apb;
}

// Calls f(std::integral_constant<int, L>) for the l_max values with an
// unrolled harmonic sweep (those of the common B2 / B3 settings), else with
// L = -1 (the sweep loops over the run-time l_max).
template <typename F>
static void with_lmax(int lmax, F &&f) {
  switch (lmax) {
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    default: f(std::integral_constant<int, -1>{}); break;
  }
}

// The same for the descriptor kernel, whose instances for other l_max values are
// by their tiles of 16 harmonics, L = -tiles: every tile of an instance is
// multiplied, whatever l_max (l_max 8 and 9 have 6 and 7 of the 8). 4,000 atoms of
// two species, 8 functions, FP64: l_max 2 18 us and 5 57 us (37 and 67 with one
// instance of eight tiles, 22 and 66 with a loop over the tiles).
template <typename F>
static void with_tiles(int lmax, F &&f) {
  switch (lmax) {
    case 0:
    case 1:
    case 2: f(std::integral_constant<int, -1>{}); break;
    case 5: f(std::integral_constant<int, -3>{}); break;
    case 7: f(std::integral_constant<int, -4>{}); break;
    case 8:
    case 9:
    case 10: f(std::integral_constant<int, -8>{}); break;
    default: with_lmax(lmax, f); break;
  }
}
static_assert(kMaxL == 10, "tiles of harmonics of the descriptor kernel");

static B2Args make_args(fm_structure s) {
  B2Args a;
  a.n = s->n;
  a.nos = s->nos;
  a.N = s->N;
  a.lmax = s->lmax;
  a.H = (s->lmax + 1) * (s->lmax + 1);
  a.nrad = s->nos * s->N;
  a.nd = s->nd;
  a.cutkind = s->cutkind;
  a.r1 = s->r1;
  a.species = s->species.as<int>();
  a.bond_off = s->bond_off.as<int>();
  a.bond_q = s->bond_q.as<int>();
  a.nspec = s->nspecies.as<int>();
  a.row_of_atom = s->row_of_atom.as<int>();
  a.rel = s->rel.as<double>();
  a.cutoffs = s->d_cutoffs.as<double>();
  return a;
}

void knorm_values(int lmax, double *out) {
  for (int l = 0; l <= lmax; l++)
    for (int m = -l; m <= l; m++) {
      int mm = m < 0 ? -m : m;
      double ratio = 1;
      for (int k = l - mm + 1; k <= l + mm; k++) ratio /= k;
      double K = std::sqrt((2 * l + 1) / (4 * 3.14159265358979323846) * ratio);
      if (mm > 0) K *= std::sqrt(2.0);
      out[l * l + m + l] = K;
    }
}

// The constant tables of the current device, l <= kMaxL.
void descriptor_setup() {
  double kn[kMaxH], rcp[kMaxL + 2] = {0};
  knorm_values(kMaxL, kn);
  for (int k = 1; k < kMaxL + 2; k++) rcp[k] = 1.0 / k;
  FM_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_knorm), kn, sizeof(kn), 0, hipMemcpyHostToDevice));
  FM_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_rcp), rcp, sizeof(rcp), 0, hipMemcpyHostToDevice));
}

void check_b2_limits(fm_structure s) {
  FM_CHECK(s->N <= kMaxN, FM_ERR_INVALID, "n_max above 16 is not supported");
  FM_CHECK(s->lmax <= kMaxL, FM_ERR_INVALID, "l_max above 10 is not supported");
}

void launch_b2(fm_structure s, bool want_b2) {
  fm_context ctx = s->ctx;
  hipStream_t st = ctx->stream;
  B2Args a = make_args(s);
  // The chosen form's B2 rows are computed in FP64 (mixed: FP32 row and c
  // for the adjoint, int8 slices of the FP64 row for the kernel
  // contraction); c alone (the B3 bond pass) stays FP32.
  bool mixed = want_b2 && s->form != FM_FORM_FP64;
  size_t esz = s->form == FM_FORM_FP64 ? sizeof(double) : sizeof(float);
  size_t csz = s->form == FM_FORM_FP64 || mixed ? sizeof(double) : sizeof(float);
  // 64-bond chunks fill all lanes of the bond basis and take half the passes;
  // they cost LDS only where the row is shorter than their tables, and are
  // used where four atoms still fit a CU. The size of a chunk is part of the order
  // of the sums, so it must not depend on the number of atoms (a batch equals its
  // structures); waves per atom may. In FP64, one wave with chunks of 32 is faster
  // than this on many atoms of a short row and slower on few (8 functions of one
  // species, l_max 4: 32,000 atoms 140 us, here 161; 108 atoms 14.7, here 12.2).
  // Waves per atom: one where it leaves the CU eight atoms, two where six, else
  // four (a CU's registers hold 16 waves). One, two and four waves: 8.5, 7.7 and
  // 6.5 ms (262144 atoms, three species, l_max 6, four atoms per CU), 0.71, 0.70 and
  // 0.57 ms (32000 atoms, two species, four per CU), 2.31, 2.24 and 3.22 ms (512
  // structures, l_max 4, seven per CU). 32,000 atoms in FP64, one and two waves:
  // 138 and 156 us (two species of 8 functions, l_max 3, ten per CU), 178 and 182
  // (the same, l_max 4, eight), 194 and 192 (one of 12, l_max 4, seven), 340 and
  // 291 (one of 8, l_max 5, six); 1,372 atoms of the first 14.1 and 15.6, 256 10.8
  // and 11.0.
  int row = a.nd;
  auto work_of = [&](int ch) {
    return b2_work(a.nrad * a.H, a.H, a.N, ch, want_b2 ? row : 0);
  };
  bool stage = work_of(32) * csz <= (size_t)160 * 1024;
  if (!stage && a.nrad > 32) row = 0;
  size_t res = resident_atoms(work_of(64) * csz);
  int chunk = res >= 4 ? 64 : 32;
  if (chunk == 32) res = resident_atoms(work_of(32) * csz);
  size_t work = work_of(chunk);
  size_t per = work * csz;
  int W = csz == 4 || !stage ? 1 : res >= 8 ? 1 : res >= 6 ? 2 : 4;
  int apb = W > 1 ? 1 : atoms_per_block(per);
  FM_CHECK(per <= (size_t)160 * 1024, FM_ERR_CAPACITY,
           "per-atom descriptor workspace exceeds LDS");
  size_t lds = apb * per;
  int nblk = (s->n + apb - 1) / apb;
  s->C.alloc(&ctx->pool, std::max<size_t>(1, (size_t)s->n * a.nrad * a.H * esz));
  MixedOut mo{};
  if (mixed) {
    // Each species' rows start a row tile of the slices (q_shift, from the
    // row build); at most a tile less one of padding per species.
    s->ldq = i8_ld(a.nd);
    long long qrows = s->n + (long long)s->nos * (kI8TileA - 1);
    FM_CHECK(qrows < (1LL << 31), FM_ERR_CAPACITY, "too many descriptor rows for the slices");
    s->Bq.alloc(&ctx->pool, std::max<size_t>(1, i8_tiled_bytes(qrows, kI8TileA, s->ldq)));
    s->Bq_scale.alloc(&ctx->pool, std::max<size_t>(1, (size_t)s->n * sizeof(double)));
    mo = MixedOut{s->B.as<float>(), s->C.as<float>(), s->Bq.as<int8_t>(),
                  s->Bq_scale.as<double>(), s->ldq / kI8Pad, s->q_shift.as<int>()};
  } else {
    s->Bq.release();
    s->Bq_scale.release();
  }
  s->has_q = mixed;
  if (nblk == 0) return;
  // FP32: the bond pass of B3 only, l_max <= 4.
  FM_CHECK(csz == 8 || a.lmax <= 4, FM_ERR_INVALID, "l_max above 4 of the FP32 bond pass");
  auto bond_pass = [&](auto &&f) {
    if (a.lmax == 3) f(std::integral_constant<int, 3>{});
    else if (a.lmax == 4) f(std::integral_constant<int, 4>{});
    else f(std::integral_constant<int, -1>{});
  };
  auto go = [&](auto waves) {
    constexpr int NW = decltype(waves)::value;
    dim3 grid(nblk), block(64 * NW * apb);
    with_tiles(a.lmax, [&](auto lc) {
      constexpr int LC = decltype(lc)::value;
      if (mixed)
        hipLaunchKernelGGL((k_b2<double, LC, true, NW>), grid, block, lds, st, a,
                           (double *)nullptr, s->norm.as<double>(), s->nn.as<double>(),
                           (double *)nullptr, 1, (int)work, chunk, (int)stage, mo);
      else
        hipLaunchKernelGGL((k_b2<double, LC, false, NW>), grid, block, lds, st, a,
                           s->B.as<double>(), s->norm.as<double>(), s->nn.as<double>(),
                           s->C.as<double>(), (int)want_b2, (int)work, chunk, (int)stage, mo);
    });
  };
  {
    KScope timer(ctx, KT_DESC);
    if (csz == 4)
      bond_pass([&](auto lc) {
        hipLaunchKernelGGL((k_b2<float, decltype(lc)::value, false, 1>), dim3(nblk),
                           dim3(64 * apb), lds, st, a, (float *)nullptr, s->norm.as<double>(),
                           s->nn.as<double>(), s->C.as<float>(), 0, (int)work, chunk, 1, mo);
      });
    else if (W == 4) go(std::integral_constant<int, 4>{});
    else if (W == 2) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 1>{});
  }
  FM_HIP(hipGetLastError());
}

void launch_adjoint(fm_structure s, const void *G, int64_t g_ld, void *fbond,
                    double *virial_atom, int project, double empty_norm, double empty_nn,
                    const double *energy, double power, void *u_buf) {
  fm_context ctx = s->ctx;
  hipStream_t st = ctx->stream;
  B2Args a = make_args(s);
  FM_CHECK(a.lmax + 1 < kMaxL + 2, FM_ERR_INVALID, "l_max above 10 is not supported");
  bool f64 = s->form == FM_FORM_FP64;
  size_t esz = f64 ? sizeof(double) : sizeof(float);
  size_t nc = (size_t)a.nrad * a.H;
  DevBuf U;
  if (!u_buf) {
    U.alloc(&ctx->pool, adjoint_u_bytes(s));
    u_buf = U.as<void>();
  }
  AdjArgs aa{project, empty_norm, empty_nn, energy, power};
  // dE/dc (B2): c and w rows in LDS per atom (each padded to 4 values).
  size_t per1 = ((size_t)pad4((int)nc) + (size_t)pad4(a.nd)) * esz;
  int apb1 = s->desc_kind == 2 ? atoms_per_block(per1) : 1;
  int nblk1 = (s->n + apb1 - 1) / apb1;
  if (s->n == 0) return;
  if (s->desc_kind == 3)
    launch_dEdc_b3(s, G, g_ld, project, empty_norm, empty_nn, u_buf);
  // FP32 projection from the rows in one pass over G and B. Rows whose LDS holds
  // a CU to two workgroups take single elements where they are not aligned and
  // the cube of 1 / |B| in one factor; the others have the order of row_dot.
  bool one_pass = !f64 && project && !energy && a.nd <= kOnePassRow;
  int single = 3 * (size_t)apb1 * per1 > (size_t)160 * 1024;
  if (s->desc_kind == 2) {
    KScope timer(ctx, KT_DEDC);
    with_lmax(a.lmax, [&](auto lc) {
      constexpr int LC = decltype(lc)::value;
      if (f64)
        hipLaunchKernelGGL((k_dEdc<double, LC>), dim3(nblk1), dim3(128 * apb1), apb1 * per1, st,
                           a, s->B.as<double>(), s->norm.as<double>(), s->nn.as<double>(),
                           (const double *)G, (long long)g_ld, aa, s->C.as<double>(),
                           (double *)u_buf, 0);
      else if (one_pass)
        hipLaunchKernelGGL((a.nd <= kOnePassRow / 2 ? k_dEdc<float, LC, kOnePassRow / 1024>
                                                    : k_dEdc<float, LC, kOnePassRow / 512>),
                           dim3(nblk1), dim3(128 * apb1), apb1 * per1, st, a, s->B.as<float>(),
                           s->norm.as<double>(), s->nn.as<double>(), (const float *)G,
                           (long long)g_ld, aa, s->C.as<float>(), (float *)u_buf, single);
      else
        hipLaunchKernelGGL((k_dEdc<float, LC>), dim3(nblk1), dim3(128 * apb1), apb1 * per1, st,
                           a, s->B.as<float>(), s->norm.as<double>(), s->nn.as<double>(),
                           (const float *)G, (long long)g_ld, aa, s->C.as<float>(),
                           (float *)u_buf, 0);
    });
  }
  FM_HIP(hipGetLastError());
  launch_bond_forces(s, u_buf, fbond, virial_atom, nullptr, s->n, empty_norm, empty_nn);
}

size_t adjoint_u_bytes(fm_structure s) {
  B2Args a = make_args(s);
  size_t esz = s->form == FM_FORM_FP64 ? sizeof(double) : sizeof(float);
  return std::max<size_t>(1, (size_t)s->n * a.nrad * a.H * esz);
}

void launch_bond_forces(fm_structure s, const void *U, void *fbond, double *virial_atom,
                        const int *atom_list, int n_list, double empty_norm, double empty_nn) {
  if (n_list == 0) return;
  hipStream_t st = s->ctx->stream;
  B2Args a = make_args(s);
  bool f64 = s->form == FM_FORM_FP64;
  size_t esz = f64 ? sizeof(double) : sizeof(float);
  AdjArgs aa{1, empty_norm, empty_nn, nullptr, 0};
  // u in LDS per atom (radial index padded to 4).
  size_t per2 = (size_t)a.nos * a.H * pad4(a.N) * esz;
  int apb2 = atoms_per_block(per2);
  int nblk2 = (n_list + apb2 - 1) / apb2;
  KScope timer(s->ctx, KT_BOND);
  auto launch = [&](auto ng) {
    constexpr int NG = decltype(ng)::value;
    if (f64)
      hipLaunchKernelGGL((k_bond_forces<double, NG>), dim3(nblk2), dim3(64 * apb2),
                         apb2 * per2, st, a, s->norm.as<double>(), s->nn.as<double>(), aa,
                         (const double *)U, (double *)fbond, virial_atom, atom_list, n_list);
    else
      hipLaunchKernelGGL((k_bond_forces<float, NG>), dim3(nblk2), dim3(64 * apb2),
                         apb2 * per2, st, a, s->norm.as<double>(), s->nn.as<double>(), aa,
                         (const float *)U, (float *)fbond, virial_atom, atom_list, n_list);
  };
  switch (pad4(a.N) / 4) {
    case 1: launch(std::integral_constant<int, 1>{}); break;
    case 2: launch(std::integral_constant<int, 2>{}); break;
    case 3: launch(std::integral_constant<int, 3>{}); break;
    default: launch(std::integral_constant<int, 4>{}); break;
  }
  static_assert(kMaxN == 16, "radial groups of k_bond_forces");
  FM_HIP(hipGetLastError());
}

}  // namespace fm
