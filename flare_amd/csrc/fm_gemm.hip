// Contractions on the matrix cores. Every contraction of the path has the
// form C = A . B^T with both operands contiguous along the reduction index
// and a fused epilogue:
//
//   EP_KERNEL C = B_s . X_hat_s^T (atoms x sparse): S = C / |B_i|,
//             k = sigma^2 S^p, w = sigma^2 alpha_j p S^(p-1); writes w and
//             (optionally) k atom-major and per-tile partial energies
//             sum_j k alpha_j (normalized_dot_product.cpp:117-177 contracted
//             with alpha as sparse_gp.cpp:664).
//   EP_STORE  plain store: G = W . X_hat_s (the kernel-gradient contraction).
//   EP_SUMSQ  Q = L_s^-1 . K^T with per-tile column sums of Q^2, the local
//             variance term |L_inv k|^2 (sparse_gp.cpp:121-131); A is lower
//             triangular so each row tile stops at its last nonzero column.
//
// FP64 form: k_gemm_f64, k_gemm_f64_dma or k_gemm_f64_lds for all three. Chosen form: EP_KERNEL is exact on
// int8 MFMA (v_mfma_i32_16x16x64_i8) over five power-of-two-scaled slices of
// each operand row, int32 accumulation per slice-pair diagonal and an FP64
// epilogue (k_gemm_i8); EP_STORE is split-BF16 x3 on
// v_mfma_f32_16x16x32_bf16 (a = a_hi + a_lo, ab ~ a_hi b_hi + a_hi b_lo +
// a_lo b_hi, FP32 accumulation), on operands split once where they are
// produced, the three products of a k-step run over all accumulators of a
// wave before the next, so consecutive MFMAs are independent; EP_SUMSQ stays
// FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>

#include "fm_device.hpp"
#include "fm_gemm.hpp"
#include "fm_internal.hpp"

namespace fm {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

// Workgroups are dealt to the 8 XCDs round robin (id % 8); the id is remapped so
// that each XCD gets a contiguous run of logical ones, whose operands share its
// L2.
__device__ __forceinline__ int xcd_id() {
  constexpr int kXcd = 8;
  int ntx = gridDim.x, nty = gridDim.y, nblk = ntx * nty;
  int pid = blockIdx.y * ntx + blockIdx.x;
  int per = (nblk + kXcd - 1) / kXcd;
  int tall = nblk % kXcd == 0 ? kXcd : nblk % kXcd;  // XCDs that get `per` ids
  int xcd = pid % kXcd, local = pid / kXcd;
  return xcd < tall ? xcd * per + local : tall * per + (xcd - tall) * (per - 1) + local;
}

// Kept out of line: inlined into every element of an unrolled epilogue, pow
// makes the loops too large to unroll.
__device__ __noinline__ double pow_general(double x, double p) { return pow(x, p); }
__device__ __forceinline__ double fpow(double x, double p, int pi) {
  if (pi == 2) return x * x;
  if (pi == 1) return x;
  return pow_general(x, p);
}

// ---------------------------------------------------------------------------
// Shared by the two contractions of the chosen form, whose operands are laid
// out in pieces that a wave copies straight to LDS (1 KB: 16 rows of 64 bytes).
// ---------------------------------------------------------------------------
typedef int v4i __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) const void gvoid;
typedef __attribute__((address_space(3))) void lvoid;

// 16-byte chunk position of k chunk c (0..3) in row r of an LDS slice block
// (rows of 64 bytes, no padding): an XOR swizzle that keeps the fragment
// reads (16 rows at four chunks) free of bank conflicts (a third of the LDS
// cycles were conflicts with r / 2 xor r / 8 in its place).
__device__ __forceinline__ int i8_chunk(int r, int c) { return c ^ (-(r >> 2) & 3); }

// This lane's 16 bytes of a piece: they land at 16 lane, so it fetches the chunk
// that belongs there.
__device__ __forceinline__ unsigned piece_lane(int lane) {
  return (lane >> 2) * 64 + 16 * i8_chunk(lane >> 2, lane & 3);
}
// Wave-uniform base `src`, kept in scalar registers so that one vector register
// addresses every piece.
__device__ __forceinline__ void copy_piece(const void *src, unsigned vsrc, void *dst) {
  asm volatile("" : "+s"(src));
  __builtin_amdgcn_global_load_lds((gvoid *)((const char *)src + vsrc), (lvoid *)dst, 16, 0, 0);
}
// Waits for this wave's copies, then for the other waves.
__device__ __forceinline__ void copies_landed() {
  __builtin_amdgcn_s_waitcnt(0x0f70);
  __syncthreads();
}

// ---------------------------------------------------------------------------
// FP64 contraction C = A B^T (rows of both K-contiguous) on
// v_mfma_f64_16x16x4: k_gemm_f64 with fragments straight from global memory,
// k_gemm_f64_dma with 32 x 32 and 64 x 64 tiles copied straight to LDS and
// k_gemm_f64_lds with 128 x 128 tiles staged there; f64_tile chooses.
//
// What bounds them: an FP64 16x16x4 MFMA holds its SIMD's vector ALU for 64
// cycles, so a wave with 64 x 64 outputs needs 16 KB per 4096 cycles; smaller
// wave tiles need more and are bound by their loads (12 TB/s from L2). The
// kernel these two replace (64 x 64 to 128 x 128 tiles in LDS, two barriers
// and transposed 8-byte LDS stores per 16 k, all accumulators moved between
// register files in every iteration) ran the kernel contraction of 32,000 x
// 1,000 x 2,100 at 48 TFLOP/s.
//
// The variance sigma^2 - |Q|^2 amplifies rounding (near the sparse set one ulp
// of |Q|^2 is 1e-9 of it), so the kernel contraction and Q keep one order of
// sums whatever the tile: 4 consecutive k per MFMA, ascending from k = 0, and
// |Q|^2 over 32 rows of L at a time. The gradient contraction (EP_STORE) takes
// its 16 k per step in an order that loads better, the same for any tile. So
// the choice of tile changes no bit: batched, tiled and single evaluations
// agree.
// ---------------------------------------------------------------------------
// Element j of lane group g (lanes 16 g .. 16 g + 15) becomes element g of
// group j: a 4 x 4 transpose across the four lane groups.
__device__ __forceinline__ void transpose_groups(double (&x)[4]) {
  unsigned d[4][2];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    unsigned long long v = __builtin_bit_cast(unsigned long long, x[j]);
    d[j][0] = (unsigned)v, d[j][1] = (unsigned)(v >> 32);
  }
#pragma unroll
  for (int w = 0; w < 2; w++) {
#pragma unroll
    for (int j = 0; j < 2; j++) {  // groups 2, 3 of j against 0, 1 of j + 2
      auto r = __builtin_amdgcn_permlane32_swap(d[j][w], d[j + 2][w], false, false);
      d[j][w] = r[0], d[j + 2][w] = r[1];
    }
#pragma unroll
    for (int j = 0; j < 4; j += 2) {  // groups 1, 3 of j against 0, 2 of j + 1
      auto r = __builtin_amdgcn_permlane16_swap(d[j][w], d[j + 1][w], false, false);
      d[j][w] = r[0], d[j + 1][w] = r[1];
    }
  }
#pragma unroll
  for (int j = 0; j < 4; j++)
    x[j] = __builtin_bit_cast(double, (unsigned long long)d[j][1] << 32 | d[j][0]);
}

// 16 bytes at 8-byte alignment (rows of odd length).
typedef double v2d __attribute__((ext_vector_type(2), aligned(8)));
typedef double v2da __attribute__((ext_vector_type(2)));

constexpr int kF64Groups = 8;
struct F64Groups {
  F64Gemm g[kF64Groups];
  int first[kF64Groups + 1];  // first workgroup of each group
  int ntx[kF64Groups], nty[kF64Groups];
  int n;
};

// Workgroup -> group and tile. Triangular operands keep the hardware's round
// robin over XCDs and take the longest rows first, so the last workgroups to
// start are the shortest; else each XCD gets a contiguous run of tiles, four
// row tiles at a time (their columns share its L2; 1 to 16 measured the same).
__device__ __forceinline__ int f64_workgroup(const F64Groups &gs, int &tx, int &ty) {
  constexpr int kRows = 4;
  int id = blockIdx.x;
  if (!gs.g[0].lower_tri) {
    int per = gridDim.x / 8, rest = gridDim.x % 8, x = id % 8, l = id / 8;
    id = x * per + min(x, rest) + l;
  }
  int gi = 0;
  while (gi + 1 < gs.n && id >= gs.first[gi + 1]) gi++;
  int local = id - gs.first[gi], ntx = gs.ntx[gi], nty = gs.nty[gi];
  if (gs.g[gi].lower_tri) {
    tx = local % ntx;
    ty = nty - 1 - local / ntx;
  } else {
    int f = local / (kRows * ntx) * kRows, n_in = min(kRows, nty - f), r = local % (kRows * ntx);
    tx = r / n_in;
    ty = f + r % n_in;
  }
  return gi;
}

// EP_KERNEL for powers other than 1 and 2: two calls of pow per element, in
// kernels of their own so that the common ones stay free of calls.
constexpr int EP_KERNEL_POW = 3;

// The last K % 4 values of k (zeros after them) of 16 rows of an operand.
__device__ __forceinline__ double f64_tail(const double *row, int K, int q4) {
  int k = (K & ~3) + q4;
  return k < K ? row[k] : 0.0;
}

// One accumulator tile in VGPRs, here and not before (without the empty
// statement the compiler copies all of them at once and spills).
__device__ __forceinline__ v4d f64_tile_out(const v4d &acc) {
  v4d t = acc;
  asm volatile("" : "+v"(t));
  return t;
}

// Epilogue of a wave's 16T x 16T tile at (row0, col0): lane l holds column
// l % 16 of each 16 x 16 tile, rows l / 16 + 4 i. `red` (EP_SUMSQ at T = 1):
// LDS through which the upper 16 rows of a 32-row half pass their sums on to
// the lower ones (wave rows 0 and 1 of the workgroup).
template <int EP, int T>
__device__ __forceinline__ void f64_epilogue(const F64Gemm &g, const v4d (&acc)[T][T], int row0,
                                             int col0, int wid, double *red) {
  const EpArgs &e = g.e;
  const int M = g.M, N = g.N;
  int lane = threadIdx.x & 63, r16 = lane & 15, q4 = lane >> 4;
  if constexpr (EP == EP_STORE) {
#pragma unroll
    for (int a = 0; a < T; a++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        int r = row0 + 16 * a + q4 + 4 * i;
        if (r >= M) continue;
        double *w = e.W_as<double>() + (size_t)r * e.ldw;
#pragma unroll
        for (int b = 0; b < T; b++) {
          int c = col0 + 16 * b + r16;
          if (c < N) w[c] = acc[a][b][i];
        }
      }
  } else if constexpr (EP == EP_KERNEL || EP == EP_KERNEL_POW) {
    // Rows: atoms, columns: sparse environments. k = sigma^2 S^p and
    // w = sigma^2 alpha p S^(p-1) per element, the energy summed over each
    // 16 columns.
    int pi = EP == EP_KERNEL_POW ? 0 : (e.power == 2.0 ? 2 : 1);
    double alpha[T];
#pragma unroll
    for (int b = 0; b < T; b++) alpha[b] = e.alpha[min(col0 + 16 * b + r16, N - 1)];
#pragma unroll
    for (int a = 0; a < T; a++) {
      double nrm[4];
#pragma unroll
      for (int i = 0; i < 4; i++) nrm[i] = e.row_norm[min(row0 + 16 * a + q4 + 4 * i, M - 1)];
      v4d t[T];
#pragma unroll
      for (int b = 0; b < T; b++) t[b] = f64_tile_out(acc[a][b]);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        int r = row0 + 16 * a + q4 + 4 * i;
        bool empty = nrm[i] < kEmptyThresh;
        double ninv = empty ? 0.0 : 1.0 / nrm[i];
        double *wr = e.W_as<double>() + (size_t)min(r, M - 1) * e.ldw;
        double *kr = e.K_as<double>() + (size_t)min(r, M - 1) * e.ldk;
#pragma unroll
        for (int b = 0; b < T; b++) {
          int c = col0 + 16 * b + r16;
          bool in = r < M && c < N;
          double s = t[b][i] * ninv;
          double sp, pm1;
          if constexpr (EP == EP_KERNEL_POW) {
            sp = pow_general(s, e.power);
            pm1 = pow_general(s, e.power - 1);
          } else {
            sp = pi == 2 ? s * s : s;
            pm1 = pi == 2 ? s : 1.0;
          }
          double kv = empty ? 0.0 : e.sig2 * sp;
          double wv = empty ? 0.0 : e.sig2 * alpha[b] * e.power * pm1;
          if (in) wr[c] = wv;
          if (in && e.K) kr[c] = kv;
          double sum = row16_sum(c < N ? kv * alpha[b] : 0.0);
          if (r16 == 0 && in) e.part[(size_t)(col0 / 16 + b) * e.part_ld + r] = sum;
        }
      }
    }
  } else {
    // Rows: rows of L, columns: atoms. Sums of squares over each 32 rows, per
    // lane in row order (rows past M are copies of the last one: left out),
    // then over the four lane groups.
    static_assert(T != 3, "a wave's rows must not straddle a 32-row half");
#pragma unroll
    for (int b = 0; b < T; b++)
#pragma unroll
      for (int a0 = 0; a0 < T; a0 += 2) {
        double v = 0;
        if constexpr (T == 1) {
          if (wid >> 1) v = red[64 * (wid & 1) + lane];
        }
#pragma unroll
        for (int a = a0; a < a0 + 2 && a < T; a++) {
          v4d t = f64_tile_out(acc[a][b]);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            double x = row0 + 16 * a + q4 + 4 * i < M ? t[i] : 0.0;
            v += x * x;
          }
        }
        if constexpr (T == 1) {
          if (!(wid >> 1)) {
            red[64 * (wid & 1) + lane] = v;
            continue;
          }
        }
        v += __shfl_xor(v, 16, 64);
        v += __shfl_xor(v, 32, 64);
        int half = (row0 + 16 * a0) / 32, c = col0 + 16 * b + r16;
        if (q4 == 0 && c < N && half < (M + 63) / 64 * 2) e.part[(size_t)half * e.part_ld + c] = v;
      }
  }
}

// A wave owns 16T x 16T outputs and loads its own fragments: lane l takes row
// l % 16 of each 16-row group and 4 of each 16 k, as two 16-byte loads. For
// EP_STORE these are k0 + 2 (l / 16) + {0, 1} and the same 8 further on, so one
// load covers 64 contiguous bytes of 16 rows, and MFMA j contracts the k set
// of element j, whatever k that is. In plain order (ORD) they are 4
// consecutive k, and a transpose over the four lane groups gives MFMA j its
// k = 4 j + {0, 1, 2, 3} (8-byte loads in that order cost twice the load
// instructions and twice the time). No LDS, no barriers: on small problems the
// waves are independent and the chain of one is short. Fragments of the next
// 16 U k are loaded into registers while the current ones feed the MFMAs, all
// loads of a step together: the two halves of a 128-byte line then meet in L1.
// A barrier that kept a workgroup's waves in step cost 35 % (their loads queue
// at one moment). U is 2 at T = 1 only, where a step of 16 k is 256 cycles.
template <int EP, int T, int U>
__global__ __launch_bounds__(256) void k_gemm_f64(F64Groups gs) {
  constexpr bool ORD = EP != EP_STORE;
  constexpr int LK = ORD ? 4 : 2, HS = ORD ? 16 : 64;  // k per lane group, bytes between its loads
  __shared__ double red[EP == EP_SUMSQ && T == 1 ? 128 : 1];
  int tx, ty;
  const F64Gemm &g = gs.g[f64_workgroup(gs, tx, ty)];
  const int M = g.M, N = g.N;
  int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int r16 = lane & 15, q4 = lane >> 4;
  int row0 = ty * 32 * T + (wid >> 1) * 16 * T, col0 = tx * 32 * T + (wid & 1) * 16 * T;
  // EP_SUMSQ writes zeros for the rows up to the next 64, and at T = 1 its wave
  // rows meet in the epilogue.
  constexpr bool MEET = EP == EP_SUMSQ && T == 1;
  if (EP != EP_SUMSQ && (row0 >= M || col0 >= N)) return;
  // Wave-uniform bases that advance along k and fixed lane offsets: an FP64
  // MFMA keeps its SIMD's vector ALU, so every vector instruction of the loop
  // (address arithmetic, register copies) adds to it. Rows past the end read
  // the last row (their outputs are not stored).
  const char *pa = reinterpret_cast<const char *>(g.A), *pb = reinterpret_cast<const char *>(g.B);
  size_t oa[T], ob[T];
#pragma unroll
  for (int t = 0; t < T; t++) {
    oa[t] = (min(row0 + 16 * t + r16, M - 1) * (size_t)g.lda + LK * q4) * 8;
    ob[t] = (min(col0 + 16 * t + r16, N - 1) * (size_t)g.ldb + LK * q4) * 8;
  }
  // k steps of KS end at the operands' last k (in plain order: its last
  // multiple of 4, the rest follows the loop); the first steps are padded with
  // zeros in front, to an even number of steps. Past the diagonal of a lower
  // triangular A every term is zero.
  constexpr int KS = 16 * U;
  int Kall = g.lower_tri ? min(g.K, row0 + 16 * T) : g.K;
  int K = ORD ? Kall & ~3 : Kall;
  int pairs = max(1, (K + 2 * KS - 1) / (2 * KS));
  int k0 = K - 2 * KS * pairs;  // the next step's first k (negative: padding)
  double ta[T], tb[T];
  if constexpr (ORD) {
    if (Kall & 3) {
#pragma unroll
      for (int t = 0; t < T; t++) {
        ta[t] = f64_tail(reinterpret_cast<const double *>(pa + oa[t]) - LK * q4, Kall, q4);
        tb[t] = f64_tail(reinterpret_cast<const double *>(pb + ob[t]) - LK * q4, Kall, q4);
      }
    }
  }
  v4d acc[T][T];
#pragma unroll
  for (int a = 0; a < T; a++)
#pragma unroll
    for (int b = 0; b < T; b++) acc[a][b] = v4d{0, 0, 0, 0};
  // Fragments of one step: KS k of every row tile, MFMA j of the four per 16 k
  // taking element j.
  struct Frag {
    double a[U][T][4], b[U][T][4];
  };
  // A step inside the rows: [k0, k0 + KS).
  auto load = [&](Frag &f) {
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int t = 0; t < T; t++) {
        const char *xa = pa + oa[t] + 128 * u, *xb = pb + ob[t] + 128 * u;
#pragma unroll
        for (int h = 0; h < 2; h++) {
          v2d va = *reinterpret_cast<const v2d *>(xa + HS * h);
          v2d vb = *reinterpret_cast<const v2d *>(xb + HS * h);
          f.a[u][t][2 * h] = va.x, f.a[u][t][2 * h + 1] = va.y;
          f.b[u][t][2 * h] = vb.x, f.b[u][t][2 * h + 1] = vb.y;
        }
      }
    k0 += KS;
    pa += 8 * KS;
    pb += 8 * KS;
  };
  // One of the first two steps: zeros for k < 0.
  auto load_head = [&](Frag &f) {
    if (k0 >= 0) return load(f);
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int t = 0; t < T; t++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          int k = k0 + 16 * u + (ORD ? j : 8 * (j >> 1) + (j & 1));
          bool in = k + LK * q4 >= 0;
          f.a[u][t][j] = in ? *reinterpret_cast<const double *>(pa + (ptrdiff_t)oa[t] + 8 * k) : 0.0;
          f.b[u][t][j] = in ? *reinterpret_cast<const double *>(pb + (ptrdiff_t)ob[t] + 8 * k) : 0.0;
        }
    k0 += KS;
    int adv = k0 > 0 ? 8 * k0 : 0;
    pa += adv;
    pb += adv;
  };
  auto mma = [&](Frag &f) {
    if constexpr (ORD) {
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int t = 0; t < T; t++) {
          transpose_groups(f.a[u][t]);
          transpose_groups(f.b[u][t]);
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int a = 0; a < T; a++)
#pragma unroll
          for (int b = 0; b < T; b++)
            acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(f.a[u][a][j], f.b[u][b][j],
                                                             acc[a][b], 0, 0, 0);
  };
  // Empty statements that take the accumulators in AGPRs: an epilogue that
  // computes with them would otherwise make the compiler carry them in VGPRs
  // from one iteration to the next and copy all of them there and back.
  auto pin = [&] {
#pragma unroll
    for (int a = 0; a < T; a++)
#pragma unroll
      for (int b = 0; b < T; b++) asm volatile("" : "+a"(acc[a][b]));
  };
  Frag f0, f1;
  load_head(f0);
  load_head(f1);
  // All of the first two steps, here: the loop then needs to wait for the
  // older of its two loads only (vmcnt; 0x0f70 leaves the other counters).
  __builtin_amdgcn_s_waitcnt(0x0f70);
  pin();
#pragma unroll 1
  for (int p = 1; p < pairs; p++) {
    mma(f0);
    __builtin_amdgcn_sched_barrier(0);
    load(f0);
    __builtin_amdgcn_sched_barrier(0);
    mma(f1);
    __builtin_amdgcn_sched_barrier(0);
    load(f1);
    __builtin_amdgcn_sched_barrier(0);
    pin();
  }
  mma(f0);
  mma(f1);
  if constexpr (ORD) {
    if (Kall & 3) {
#pragma unroll
      for (int a = 0; a < T; a++)
#pragma unroll
        for (int b = 0; b < T; b++)
          acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(ta[a], tb[b], acc[a][b], 0, 0, 0);
    }
  }
  pin();
  if constexpr (MEET) {
    if (!(wid >> 1)) f64_epilogue<EP, T>(g, acc, row0, col0, wid, red);
    __syncthreads();
    if (wid >> 1) f64_epilogue<EP, T>(g, acc, row0, col0, wid, red);
  } else {
    f64_epilogue<EP, T>(g, acc, row0, col0, wid, red);
  }
}

// The same 16T x 16T outputs per wave, T = 1 and 2, from operands that the
// workgroup's four waves copy straight to LDS once: four stages of 16 k, three
// of them on their way. k_gemm_f64 is bound by what a CU gets from L2 (20 bytes
// a cycle), where its waves fetch every row twice. Needs 16-byte aligned rows.
// LDS rows are 128 bytes, their 16-byte chunks swizzled by row / 2, so that the
// 8-byte fragment reads (16 rows at two k) are free of bank conflicts.
template <int EP, int T>
__global__ __launch_bounds__(256, 2) void k_gemm_f64_dma(F64Groups gs) {
  constexpr int R = 32 * T, ST = 2 * R * 128;
  __shared__ double red[EP == EP_SUMSQ && T == 1 ? 128 : 1];
  __shared__ __align__(16) int8_t s0[ST], s1[ST], s2[ST], s3[ST];
  int tx, ty;
  const F64Gemm &g = gs.g[f64_workgroup(gs, tx, ty)];
  const int M = g.M, N = g.N;
  int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int r16 = lane & 15, q4 = lane >> 4;
  int rowb = ty * R, colb = tx * R, row0 = rowb + (wid >> 1) * 16 * T, col0 = colb + (wid & 1) * 16 * T;
  // Past the diagonal of a lower triangular A every term is zero.
  constexpr bool ORD = EP != EP_STORE;
  int K = g.lower_tri ? min(g.K, rowb + R) : g.K, steps = K / 16;
  int head = ORD ? 0 : K & 15;  // k before the first step (even); in plain order the rest follows
  // Wave w copies the pieces (8 rows of 128 bytes) w T .. of either operand; rows
  // past the end repeat the last one.
  int ra0 = min(rowb, M - 1), rb0 = min(colb, N - 1);
  const char *pa = reinterpret_cast<const char *>(g.A) + ((size_t)ra0 * g.lda + head) * 8;
  const char *pb = reinterpret_cast<const char *>(g.B) + ((size_t)rb0 * g.ldb + head) * 8;
  unsigned va[T], vb[T];
#pragma unroll
  for (int p = 0; p < T; p++) {
    int r = 8 * (wid * T + p) + (lane >> 3), chunk = 16 * ((lane & 7) ^ ((r >> 1) & 7));
    va[p] = (unsigned)((min(rowb + r, M - 1) - ra0) * g.lda * 8) + chunk;
    vb[p] = (unsigned)((min(colb + r, N - 1) - rb0) * g.ldb * 8) + chunk;
  }
  auto copy = [&](int8_t *dst, int s) {
#pragma unroll
    for (int p = 0; p < T; p++) {
      copy_piece(pa + (size_t)s * 128, va[p], dst + (wid * T + p) * 1024);
      copy_piece(pb + (size_t)s * 128, vb[p], dst + R * 128 + (wid * T + p) * 1024);
    }
  };
  v4d acc[T][T];
#pragma unroll
  for (int a = 0; a < T; a++)
#pragma unroll
    for (int b = 0; b < T; b++) acc[a][b] = v4d{0, 0, 0, 0};
  auto pin = [&] {
#pragma unroll
    for (int a = 0; a < T; a++)
#pragma unroll
      for (int b = 0; b < T; b++) asm volatile("" : "+a"(acc[a][b]));
  };
  // MFMA j of 16 k takes k = 4 j + l / 16, or the k of k_gemm_f64 for EP_STORE.
  auto k_of = [&](int j) { return ORD ? 4 * j + q4 : 8 * (j >> 1) + 2 * q4 + (j & 1); };
  int ra = ((wid >> 1) * 16 * T + r16) * 128, swz = (r16 >> 1) & 7;
  int rb = R * 128 + ((wid & 1) * 16 * T + r16) * 128;
  int at[4];
#pragma unroll
  for (int j = 0; j < 4; j++) at[j] = 16 * ((k_of(j) >> 1) ^ swz) + 8 * (k_of(j) & 1);
  auto step = [&](const int8_t *__restrict__ rd, int8_t *__restrict__ wr, int s) {
    pin();
    // This wave's copies but those of the newest two stages have landed, and with
    // the barrier the other waves'; a __syncthreads would wait for all of them.
    // The stage that `wr` held was multiplied in the step before.
    __builtin_amdgcn_s_waitcnt(0x0f70 | (4 * T));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    copy(wr, min(s + 3, steps - 1));
    double fa[T][4], fb[T][4];
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int t = 0; t < T; t++) {
        fa[t][j] = *reinterpret_cast<const double *>(rd + ra + t * 2048 + at[j]);
        fb[t][j] = *reinterpret_cast<const double *>(rd + rb + t * 2048 + at[j]);
      }
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int a = 0; a < T; a++)
#pragma unroll
        for (int b = 0; b < T; b++)
          acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[a][j], fb[b][j], acc[a][b], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // The K % 16 of k outside the steps, zeros around them.
  double ta[T][4], tb[T][4];
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int t = 0; t < T; t++) {
      int k = (ORD ? 16 * steps : head - 16) + k_of(j);
      bool in = k >= 0 && k < K;
      ta[t][j] = in ? g.A[min(row0 + 16 * t + r16, M - 1) * (size_t)g.lda + k] : 0.0;
      tb[t][j] = in ? g.B[min(col0 + 16 * t + r16, N - 1) * (size_t)g.ldb + k] : 0.0;
    }
  auto rest = [&] {
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (ORD ? 16 * steps + 4 * j < K : head > 0) {
#pragma unroll
        for (int a = 0; a < T; a++)
#pragma unroll
          for (int b = 0; b < T; b++)
            acc[a][b] =
                __builtin_amdgcn_mfma_f64_16x16x4f64(ta[a][j], tb[b][j], acc[a][b], 0, 0, 0);
      }
    pin();
  };
  if constexpr (!ORD) rest();
  pin();
  if (steps > 0) {
    copy(s0, 0);
    copy(s1, min(1, steps - 1));
    copy(s2, min(2, steps - 1));
    int s = 0;
#pragma unroll 1
    for (; s + 4 <= steps; s += 4) {
      step(s0, s3, s);
      step(s1, s0, s + 1);
      step(s2, s1, s + 2);
      step(s3, s2, s + 3);
    }
    if (s < steps) step(s0, s3, s);
    if (s + 1 < steps) step(s1, s0, s + 1);
    if (s + 2 < steps) step(s2, s1, s + 2);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // no copy outlives the workgroup
  }
  pin();
  if constexpr (ORD) rest();
  if constexpr (EP == EP_SUMSQ && T == 1) {
    if (!(wid >> 1)) f64_epilogue<EP, T>(g, acc, row0, col0, wid, red);
    __syncthreads();
    if (wid >> 1) f64_epilogue<EP, T>(g, acc, row0, col0, wid, red);
  } else if (EP == EP_SUMSQ || (row0 < M && col0 < N)) {
    f64_epilogue<EP, T>(g, acc, row0, col0, wid, red);
  }
}

// 128 x 128 tiles in plain k order, four waves of 64 x 64: the next 16 k of
// both operands are in flight to registers while the current ones, in LDS,
// feed the MFMAs; two LDS buffers, one barrier per 16 k (4096 MFMA cycles), two
// workgroups per CU. A row's 16 k are 8 chunks of 16 bytes, chunk c of row r at
// place c ^ (r % 8), so that the 16-byte stores and the 8-byte fragment reads
// (16 rows, 4 consecutive k) spread over all banks.
template <int EP>
__global__ __launch_bounds__(256, 2) void k_gemm_f64_lds(F64Groups gs) {
  constexpr int T = 4, KS = 16, TILE = 128 * KS;
  __shared__ __align__(16) double As[2 * TILE], Bs[2 * TILE];
  int tx, ty;
  const F64Gemm &g = gs.g[f64_workgroup(gs, tx, ty)];
  const int M = g.M, N = g.N;
  int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int r16 = lane & 15, q4 = lane >> 4;
  int brow = ty * 128, bcol = tx * 128;
  int row0 = brow + (wid >> 1) * 64, col0 = bcol + (wid & 1) * 64;
  // Steps of 16 end at the last multiple of 4, with zeros in front of the first
  // one; past the diagonal of a lower triangular A every term is zero.
  int Kall = g.lower_tri ? min(g.K, brow + 128) : g.K;
  int K = Kall & ~3;
  int steps = (K + KS - 1) / KS;
  int k0 = K - KS * steps;
  // Load i of thread t: chunk t % 8 of row 32 i + t / 8.
  const double *pa[4], *pb[4];
  int tid = threadIdx.x, chunk = tid & 7;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    int r = 32 * i + (tid >> 3);
    pa[i] = g.A + (size_t)min(brow + r, M - 1) * g.lda + 2 * chunk + k0;
    pb[i] = g.B + (size_t)min(bcol + r, N - 1) * g.ldb + 2 * chunk + k0;
  }
  int put = (tid >> 3) * KS + 2 * (chunk ^ ((tid >> 3) & 7));  // its place in a tile's 32 rows
  v2d ra[4], rb[4];
  auto load = [&] {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      ra[i] = *reinterpret_cast<const v2d *>(pa[i]);
      rb[i] = *reinterpret_cast<const v2d *>(pb[i]);
      pa[i] += KS;
      pb[i] += KS;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      *reinterpret_cast<v2da *>(&As[buf * TILE + 32 * i * KS + put]) = ra[i];
      *reinterpret_cast<v2da *>(&Bs[buf * TILE + 32 * i * KS + put]) = rb[i];
    }
  };
  // The first step when it starts before k = 0.
  auto load_head = [&] {
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
      for (int e = 0; e < 2; e++) {
        bool in = k0 + 2 * chunk + e >= 0;
        ra[i][e] = in ? pa[i][e] : 0.0;
        rb[i][e] = in ? pb[i][e] : 0.0;
      }
      pa[i] += KS;
      pb[i] += KS;
    }
  };
  v4d acc[T][T];
#pragma unroll
  for (int a = 0; a < T; a++)
#pragma unroll
    for (int b = 0; b < T; b++) acc[a][b] = v4d{0, 0, 0, 0};
  auto pin = [&] {  // see k_gemm_f64
#pragma unroll
    for (int a = 0; a < T; a++)
#pragma unroll
      for (int b = 0; b < T; b++) asm volatile("" : "+a"(acc[a][b]));
  };
  // Lane offsets of MFMA j's fragments: k = 4 j + q4 of rows r16 of each 16.
  int fo[4];
#pragma unroll
  for (int j = 0; j < 4; j++)
    fo[j] = r16 * KS + 2 * ((2 * j + (q4 >> 1)) ^ (r16 & 7)) + (q4 & 1);
  auto compute = [&](int buf) {
    const double *as = As + buf * TILE + (wid >> 1) * 64 * KS;
    const double *bs = Bs + buf * TILE + (wid & 1) * 64 * KS;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      double af[T], bf[T];
#pragma unroll
      for (int t = 0; t < T; t++) {
        af[t] = as[t * 16 * KS + fo[j]];
        bf[t] = bs[t * 16 * KS + fo[j]];
      }
#pragma unroll
      for (int a = 0; a < T; a++)
#pragma unroll
        for (int b = 0; b < T; b++)
          acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[a], bf[b], acc[a][b], 0, 0, 0);
    }
  };
  if (steps > 0) {
    if (k0 < 0) load_head();
    else load();
    store(0);
  }
  if (steps > 1) load();
  __syncthreads();
  pin();
#pragma unroll 1
  for (int s = 0; s < steps; s++) {
    compute(s & 1);
    pin();
    if (s + 1 < steps) store((s + 1) & 1);  // read by compute(s - 1) last
    if (s + 2 < steps) load();
    __syncthreads();
  }
  if (Kall & 3) {
    double ta[T], tb[T];
#pragma unroll
    for (int t = 0; t < T; t++) {
      ta[t] = f64_tail(g.A + (size_t)min(row0 + 16 * t + r16, M - 1) * g.lda, Kall, q4);
      tb[t] = f64_tail(g.B + (size_t)min(col0 + 16 * t + r16, N - 1) * g.ldb, Kall, q4);
    }
#pragma unroll
    for (int a = 0; a < T; a++)
#pragma unroll
      for (int b = 0; b < T; b++)
        acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(ta[a], tb[b], acc[a][b], 0, 0, 0);
  }
  pin();
  f64_epilogue<EP, T>(g, acc, row0, col0, wid, nullptr);
}

// This workgroup's tile of a launch over several contractions (first tiles
// `first`): every XCD takes a contiguous run of the tiles, kI8Group row tiles at
// a time, row index fastest: the workgroups that it holds at once cover
// kI8Group row tiles by a few column tiles, which share its L2.
template <typename Groups>
__device__ __forceinline__ int group_tile(const Groups &gs, int bm, int bn, int &tx, int &ty) {
  int id = xcd_id(), gi = 0;
  while (gi + 1 < gs.n && id >= gs.first[gi + 1]) gi++;
  id -= gs.first[gi];
  int ntx = (gs.g[gi].N + bn - 1) / bn, nty = (gs.g[gi].M + bm - 1) / bm;
  int f = id / (kI8Group * ntx) * kI8Group, n_in = min(kI8Group, nty - f);
  tx = id % (kI8Group * ntx) / n_in;
  ty = f + id % (kI8Group * ntx) % n_in;
  return gi;
}

// ---------------------------------------------------------------------------
// Split-BF16 x3 GEMM (chosen form) on operands stored as two BF16 pieces of FP32
// values (x = x_0 + x_1, split once where the operand is produced: the sparse
// set on first use, w in the kernel contraction's epilogue), in the tiled split
// layout. The products x_1 y_0, x_0 y_1 and x_0 y_0 of 32 k are summed in that
// order (smallest first), then those of the next 32.
// ---------------------------------------------------------------------------

// X (n rows of K FP64 values) as BF16 pieces of their FP32 values, zeros in the
// padding. One thread per 8 k of a row.
__global__ __launch_bounds__(256) void k_split_rows(const double *X, long long ldx, int n, int K,
                                                    long long nk, uint16_t *hi, uint16_t *lo) {
  long long i = blockIdx.x * 256ll + threadIdx.x;  // chunk of the layout
  long long blocks = (n + kSplitRows - 1) / kSplitRows * nk;
  if (i >= blocks * 64) return;
  long long row = i / 64 / nk * kSplitRows + (i & 63) / 4, k0 = i / 64 % nk * kSplitPad + (i & 3) * 8;
  v8bf h, l;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    float x = row < n && k0 + j < K ? (float)X[row * ldx + k0 + j] : 0.0f;
    h[j] = (__bf16)x;
    l[j] = (__bf16)(x - (float)h[j]);
  }
  *reinterpret_cast<v8bf *>(hi + 8 * i) = h;
  *reinterpret_cast<v8bf *>(lo + 8 * i) = l;
}

constexpr int kSplitGroups = 8;
struct SplitGroups {
  SplitGemm g[kSplitGroups];
  int first[kSplitGroups], n;
};

// Tiles of 16 RA WR x 16 RB WC, WR x WC waves of RA x RB blocks of
// v_mfma_f32_16x16x32_bf16. One step of 32 k of either operand is copied to one of
// two LDS buffers a step ahead; between the products the fragments of the next
// row block, and in a step's last one those of the next step, are read.
//
// Bound by power like the integer contraction, so by the bytes moved per
// product. Three groups of 87,381 x 3,255 x 1,365: 5.4 ms, 1.29 PFLOP/s of
// products (8.0 ms before, from row-major operands through registers with all
// waves reading LDS or multiplying at the same time, on tiles of which the first
// call of a shape timed seven).
template <int RA, int RB, int WR, int WC>
__global__ __launch_bounds__(64 * WR * WC, 2) void k_gemm_split(SplitGroups gs) {
  constexpr int NW = WR * WC, BM = 16 * RA * WR, BN = 16 * RB * WC;
  constexpr int A_PC = BM * 64, B_PC = BN * 64;  // bytes of one piece of a step
  constexpr int A_ST = 2 * A_PC, B_ST = 2 * B_PC;
  constexpr int NA = A_ST / 1024 / NW, NB = B_ST / 1024 / NW;  // copies per wave
  static_assert(NA % 2 == 0 && NB % 2 == 0 && NA + NB <= 3 * RB && 2 * RB + 2 <= 3 * RB, "split");
  __shared__ __align__(16) int8_t buf0[A_ST + B_ST], buf1[A_ST + B_ST];
  int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  int wr = wid / WC, wc = wid % WC, tx, ty;
  const SplitGemm &g = gs.g[group_tile(gs, BM, BN, tx, ty)];
  const int M = g.M, N = g.N, nk = g.nk;
  int row0 = ty * BM, col0 = tx * BN;
  v4f acc[RA][RB];
#pragma unroll
  for (int a = 0; a < RA; a++)
#pragma unroll
    for (int b = 0; b < RB; b++) acc[a][b] = v4f{0, 0, 0, 0};
  // Wave w copies both pieces of the blocks w NA / 2 .. of A and w NB / 2 .. of
  // B (past the last block of an operand that one again).
  unsigned vsrc = piece_lane(lane);
  const char *src0[NA + NB];
#pragma unroll
  for (int i = 0; i < NA + NB; i++) {
    int j = i < NA ? i : i - NA, blk = wid * ((i < NA ? NA : NB) / 2) + (j >> 1);
    int at = min((i < NA ? row0 : col0) / 16 + blk, ((i < NA ? M : N) + 15) / 16 - 1);
    src0[i] = reinterpret_cast<const char *>((i < NA ? g.A : g.B)[j & 1]) + (size_t)at * nk * 1024;
  }
  auto copy = [&](int8_t *dst, int ks, int i) {
    if (i >= NA + NB) return;
    int j = i < NA ? i : i - NA, blk = wid * ((i < NA ? NA : NB) / 2) + (j >> 1);
    copy_piece(src0[i] + (size_t)ks * 1024, vsrc,
               dst + (i < NA ? 0 : A_ST) + (j & 1) * (i < NA ? A_PC : B_PC) + blk * 1024);
  };
  v8bf fa[2][2], fb[2][RB][2];  // A of two blocks in turn, B of two steps in turn
  int r16 = lane & 15, frag = r16 * 64 + 16 * i8_chunk(r16, lane >> 4);
  int oa = wr * RA * 1024 + frag, ob = A_ST + wc * RB * 1024 + frag;
  auto read_a = [&](const int8_t *src, int r, int pc) {
    fa[r & 1][pc] = *reinterpret_cast<const v8bf *>(&src[pc * A_PC + r * 1024 + oa]);
  };
  auto read_b = [&](const int8_t *src, int set, int i) {
    fb[set][i >> 1][i & 1] =
        *reinterpret_cast<const v8bf *>(&src[(i & 1) * B_PC + (i >> 1) * 1024 + ob]);
  };
  // The products of row block r; other(i) issues reads and copies between them.
  auto products = [&](int r, int set, auto other) {
#pragma unroll
    for (int p = 0; p < 3; p++)
#pragma unroll
      for (int h = 0; h < RB; h++) {
        acc[r][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            fa[r & 1][p == 0 ? 1 : 0], fb[set][h][p == 1 ? 1 : 0], acc[r][h], 0, 0, 0);
        other(p * RB + h);
        __builtin_amdgcn_sched_barrier(0);
      }
  };
  auto body = [&](const int8_t *__restrict__ src, int set) {
#pragma unroll
    for (int a = 0; a < RA; a++)
#pragma unroll
      for (int b = 0; b < RB; b++) asm volatile("" : "+v"(acc[a][b]));
#pragma unroll
    for (int r = 0; r < RA - 1; r++)
      products(r, set, [&](int i) {
        if (i < 2) read_a(src, r + 1, 1 - i);
      });
  };
  // The step's last row block: after the barrier, so the next step is in
  // `next` and this one's buffer takes step ks.
  auto tail = [&](const int8_t *__restrict__ next, int8_t *__restrict__ dst, int ks, int set) {
    products(RA - 1, set, [&](int i) {
      if (i == 0) read_a(next, 0, 1);
      else if (i == 1) read_a(next, 0, 0);
      else if (i < 2 + 2 * RB) read_b(next, set ^ 1, i - 2);
      copy(dst, ks, i);
    });
  };
#pragma unroll
  for (int i = 0; i < NA + NB; i++) copy(buf0, 0, i);
#pragma unroll
  for (int i = 0; i < NA + NB; i++) copy(buf1, min(1, nk - 1), i);
  copies_landed();
#pragma unroll
  for (int pc = 0; pc < 2; pc++) read_a(buf0, 0, pc);
#pragma unroll
  for (int i = 0; i < 2 * RB; i++) read_b(buf0, 0, i);
  int ks = 0;
#pragma unroll 1
  for (; ks + 2 <= nk; ks += 2) {
    body(buf0, 0);
    copies_landed();
    tail(buf1, buf0, min(ks + 2, nk - 1), 0);
    body(buf1, 1);
    copies_landed();
    tail(buf0, buf1, min(ks + 3, nk - 1), 1);
  }
  if (ks < nk) {
    body(buf0, 0);
    products(RA - 1, 0, [](int) {});
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // no copy outlives the workgroup
  float *W = g.e.W_as<float>();
#pragma unroll
  for (int a = 0; a < RA; a++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      int r = row0 + (wr * RA + a) * 16 + 4 * (lane >> 4) + i;
      if (r >= M) continue;
      float *out = W + (size_t)r * g.e.ldw;
#pragma unroll
      for (int b = 0; b < RB; b++) {
        int c = col0 + (wc * RB + b) * 16 + r16;
        if (c < N) out[c] = acc[a][b][i];
      }
    }
}

// ---------------------------------------------------------------------------
// Exact-integer kernel contraction (chosen form). Every row x of either
// operand is scaled by a power of two s = 2^E with max|x| < s, and r = x / s
// is cut into kI8Slices signed 8-bit slices, r = sum_p a_p 2^-(6 + 7p) + tail
// (|a_p| <= 64, |tail| <= 2^-(7 kI8Slices)): the first slice takes 6 bits and
// every further one 7 (rounding to nearest, so each residual is at most half
// a unit of the previous slice). The product x . y is then
//   s_x s_y sum_{p + q < kI8Slices} 2^-(12 + 7(p + q)) (A_p . B_q),
// each A_p . B_q exact on the int8 matrix cores (int32 accumulation; the
// terms of equal p + q share one accumulator). Dropping the products with
// p + q >= kI8Slices leaves about 34 significant bits, so the kernel values
// k = sigma^2 S^p that the local variance amplifies by L_inv carry FP64-like
// accuracy, where FP32 accumulation of BF16 pieces carries about 16 bits.
// ---------------------------------------------------------------------------
// One wave per row: the row maximum, its power-of-two scale and the slices
// of 4 consecutive values per lane (zeros past nd up to Kq), stored in the
// tiled slice layout (tr rows per tile).
template <typename T>
__global__ __launch_bounds__(256) void k_slice_rows(const T *X, long long ldx, int n, int nd,
                                                    int8_t *Q, long long nk, int tr,
                                                    double *scale) {
  int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= n) return;
  const T *x = X + (size_t)row * ldx;
  double mx = 0;
  for (int k = lane; k < nd; k += 64) mx = fmax(mx, fabs((double)x[k]));
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
  int E = 0;
  if (mx > 0) frexp(mx, &E);  // mx = m 2^E, m in [0.5, 1)
  double inv = ldexp(1.0, -E);
  if (lane == 0) scale[row] = ldexp(1.0, E);
  long long Kq = nk * kI8Pad;
  for (int k0 = 4 * lane; k0 < Kq; k0 += 256) {
    int packed[kI8Slices];
#pragma unroll
    for (int p = 0; p < kI8Slices; p++) packed[p] = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      int k = k0 + j;
      double r = k < nd ? (double)x[k] * inv : 0.0;
#pragma unroll
      for (int p = 0; p < kI8Slices; p++) {
        double a = rint(ldexp(r, 6 + 7 * p));
        r -= ldexp(a, -(6 + 7 * p));
        packed[p] |= ((int)a & 0xff) << (8 * j);
      }
    }
#pragma unroll
    for (int p = 0; p < kI8Slices; p++)
      *reinterpret_cast<int *>(Q + i8_tile_offset(tr, nk, row, k0, p)) = packed[p];
  }
}

// An int32 accumulator sums at most kI8Slices products per k of |a b| <=
// 64^2 = 4096: 65536 k keep it below 2^31 (5 x 4096 x 65536 = 1.3e9).
constexpr int kI8Flush = 65536;

// 128 x 32 RA tiles, 8 waves, each 16 RA x 32 of v_mfma_i32_16x16x64_i8 (lane
// l: operand row l % 16, bytes k = 16 (l / 16) .. + 15; result column l % 16,
// rows 4 (l / 16) + i).
//
// What bounds it: power. With operands in registers the card reaches 4.3
// POP/s on such data with this instruction (3.4 with 32 x 32 x 32, 4.9 on
// zeros), at a lower clock; every byte moved takes from that. So the tiles are as
// large as the registers allow and are copied to LDS directly. 87,381 x 1,365 x
// 3,264: 2.5 POP/s (70 % of the cycles have an MFMA in flight at 1.8 GHz; 1.8
// before, with 32 x 32 x 32 on 128 x 64 tiles that passed through registers,
// and all waves reading LDS or multiplying at the same time).
//
// One k step (64) of a row tile and of a column tile is one contiguous run of
// either operand (the tiled slice layout), copied straight to one of two LDS
// buffers a step ahead. The 15 slice products of a pair of 16-row blocks run
// in rounds (round r: slice r of A against each slice of B it pairs with), so
// consecutive MFMAs accumulate into different diagonals; between them the
// fragments that the next pair of blocks needs are read (the pairs are walked
// in a serpentine, so that is one block of 5 fragments at a time).
// Epilogue as EpKernel, in FP64 from the exact sums: S, k (FP64), w as BF16
// pairs, energy partials per kI8TileN columns; k, then w, are staged in LDS and
// stored as whole rows of the tile.
constexpr int kI8Groups = 8;
struct I8Groups {
  I8Gemm g[kI8Groups];
  int first[kI8Groups], n;
};

template <bool LONG, int RA>
__global__ __launch_bounds__(512) void k_gemm_i8(I8Groups gs) {
  constexpr int S = kI8Slices, BM = kI8TileA, BN = 32 * RA, NT = 512, WC = RA;  // wave columns
  constexpr int A_SL = BM * kI8Pad, B_SL = BN * kI8Pad;  // bytes of one slice block in LDS
  constexpr int A_ST = S * A_SL, B_ST = S * B_SL;        // bytes of one k step
  constexpr int G_SL = kI8TileN * kI8Pad, G_ST = S * G_SL;  // of B in memory
  constexpr int NB = (B_ST / 1024 + 7) / 8;  // 1 KB pieces of B per wave (A: S)
  static_assert(BM == 128 && kI8TileN == 64 && kI8Pad == 64 && (RA == 2 || RA == 4), "tiling");
  static_assert(BM * BN * 4 + 8 * BM * WC <= A_ST + B_ST && BM * (BN + 8) * 2 <= A_ST + B_ST,
                "epilogue staging fits");
  __shared__ __align__(16) int8_t buf0[A_ST + B_ST], buf1[A_ST + B_ST];
  int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  int wr = wid / WC, wc = wid % WC;
  int tx, ty;
  const I8Gemm &g = gs.g[group_tile(gs, BM, BN, tx, ty)];
  const int M = g.M, N = g.N, nk = g.nk;
  const EpArgs &e = g.e;
  int row0 = ty * BM, col0 = tx * BN;
  v4i acc[S][RA][2];
  // With LONG (Kq > kI8Flush) the int32 sums of the slice products
  // (p + q = d) are folded into one FP64 sum every kI8Flush k, before they
  // could overflow; otherwise once, after the loop.
  constexpr int NV = 8 * RA, SJ = LONG ? NV : 1;  // values per lane
  double sacc[SJ];
  auto clear = [&]() {
#pragma unroll
    for (int d = 0; d < S; d++)
#pragma unroll
      for (int q = 0; q < 2 * RA; q++) acc[d][q >> 1][q & 1] = v4i{};
  };
  auto diag_sum = [&](int j) {
    double sum = 0;
#pragma unroll
    for (int d = S - 1; d >= 0; d--)
      sum += ldexp((double)acc[d][j >> 3][(j >> 2) & 1][j & 3], -(12 + 7 * d));
    return sum;
  };
  auto flush = [&](int ks) {
    if constexpr (LONG) {
      if (ks > 0 && (ks % (kI8Flush / kI8Pad) == 0 || ks == nk)) {
#pragma unroll
        for (int j = 0; j < NV; j++) sacc[j] += diag_sum(j);
        clear();
      }
    }
  };
#pragma unroll
  for (int j = 0; j < SJ; j++) sacc[j] = 0;
  clear();
  // Copies of a step's 1 KB pieces (16 rows of a slice): wave w takes piece w
  // of each slice of A and of B (with 64 columns, which have 4 pieces a slice,
  // piece w % 4 of slices w / 4, w / 4 + 2 and the last one). A column tile
  // past the last 64 columns repeats them.
  unsigned vsrc = piece_lane(lane);
  int wb = wid % (B_SL / 1024), pb = wid / (B_SL / 1024);
  int tb = min(tx * (BN / kI8TileN) + (wb >> 2), (N - 1) / kI8TileN);
  const int8_t *Aw = g.A + (size_t)ty * nk * A_ST + wid * 1024;
  const int8_t *Bw = g.B + (size_t)tb * nk * G_ST + (wb & 3) * 1024;
  auto copy = [&](int8_t *dst, int ks, int i) {
    if (i >= S + NB) return;
    int p = i < S ? i : RA == 4 ? i - S : min(2 * (i - S) + pb, S - 1);
    const int8_t *src = i < S ? Aw + ((size_t)ks * A_ST + p * A_SL)
                              : Bw + ((size_t)ks * G_ST + p * G_SL);
    dst += i < S ? p * A_SL + wid * 1024 : A_ST + p * B_SL + wb * 1024;
    copy_piece(src, vsrc, dst);
  };
  // Fragments: all slices of 16 rows of A and of 32 of B for a whole step.
  v4i fa[S], fb[2][S];
  int r16 = lane & 15, k16 = lane >> 4;
  int frag = r16 * 64 + 16 * i8_chunk(r16, k16);
  int oa = wr * 16 * RA * 64 + frag, ob = A_ST + wc * 32 * 64 + frag;
  auto read_a = [&](const int8_t *src, int r, int p) {
    fa[p] = *reinterpret_cast<const v4i *>(&src[p * A_SL + r * 1024 + oa]);
  };
  auto read_b = [&](const int8_t *src, int h, int p) {
    fb[h][p] = *reinterpret_cast<const v4i *>(&src[p * B_SL + h * 1024 + ob]);
  };
  // The 15 slice products of blocks (r, h); other(i) issues copies and reads
  // between them, after(rd) follows the last use of slice rd of A.
  auto products = [&](int r, int h, auto other, auto after) {
    int i = 0;
#pragma unroll
    for (int rd = 0; rd < S; rd++) {
#pragma unroll
      for (int d = S - 1; d >= rd; d--) {
        acc[d][r][h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[rd], fb[h][d - rd],
                                                             acc[d][r][h], 0, 0, 0);
        other(i++);
        if (d == rd) after(rd);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // Step ks, its column block h first: all pairs of blocks but the last, during
  // which the next step's first fragments are read. dst receives step `next`.
  auto body = [&](const int8_t *__restrict__ src, int8_t *__restrict__ dst, int next, int h) {
#pragma unroll
    for (int d = 0; d < S; d++)
#pragma unroll
      for (int q = 0; q < 2 * RA; q++) asm volatile("" : "+v"(acc[d][q >> 1][q & 1]));
#pragma unroll
    for (int r = 0; r < RA; r++) {
      products(
          r, (r & 1) ? h ^ 1 : h,
          [&](int i) {
            if (r == 0 && i % 3 == 0) read_b(src, h ^ 1, i / 3);
            if (r == 0 && i % 3 == 1) copy(dst, next, i / 3);
          },
          [](int) {});
      if (r < RA - 1)
        products(
            r, (r & 1) ? h : h ^ 1,
            [&](int i) {
              if (r == 0 && i % 3 == 1) copy(dst, next, 5 + i / 3);
            },
            [&](int rd) { read_a(src, r + 1, rd); });
    }
  };
  auto tail = [&](const int8_t *src, int h) {
    products(
        RA - 1, h, [&](int i) { if (i % 3 == 1) read_b(src, h ^ 1, i / 3); },
        [&](int rd) { read_a(src, 0, rd); });
  };
#pragma unroll
  for (int i = 0; i < S + NB; i++) copy(buf0, 0, i);
  copies_landed();
#pragma unroll
  for (int p = 0; p < S; p++) {
    read_a(buf0, 0, p);
    read_b(buf0, 0, p);
  }
  int ks = 0;
#pragma unroll 1
  for (; ks + 2 <= nk; ks += 2) {
    flush(ks);
    body(buf0, buf1, ks + 1, 0);
    copies_landed();
    tail(buf1, 0);
    flush(ks + 1);
    body(buf1, buf0, min(ks + 2, nk - 1), 1);
    copies_landed();
    tail(buf0, 1);
  }
  if (ks < nk) {
    flush(ks);
    body(buf0, buf1, ks, 0);
    tail(buf0, 0);
  }
  flush(nk);
  copies_landed();
  // Epilogue: values in FP64 per element. k is staged in LDS over the operand
  // buffers, w after it.
  constexpr int HN = BN / 2, WLD = BN + 8;  // k: columns in each buffer; w: padded rows
  double *Kst = reinterpret_cast<double *>(wc < WC / 2 ? buf0 : buf1);
  double *red = reinterpret_cast<double *>(buf0 + BM * HN * 8);  // [WC][BM]
  uint16_t *Hst = reinterpret_cast<uint16_t *>(buf0), *Lst = reinterpret_cast<uint16_t *>(buf1);
  int pi = e.power == 2.0 ? 2 : (e.power == 1.0 ? 1 : 0);
  // Value j of a lane: row block j / 8, column block (j / 4) % 2, row j % 4.
  bool cin[2];
  double a_c[2], s_c[2], rsum[NV / 2];
  float wf[NV];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    int c = col0 + wc * 32 + 16 * h + r16;
    cin[h] = c < N;
    a_c[h] = cin[h] ? e.alpha[c] : 0.0;
    s_c[h] = cin[h] ? g.sb[c] : 0.0;
  }
#pragma unroll
  for (int j = 0; j < NV; j++) {
    int h = (j >> 2) & 1, cc = wc * 32 + 16 * h + r16;
    int rr = wr * 16 * RA + 16 * (j >> 3) + 4 * k16 + (j & 3);
    int r = row0 + rr;
    double kv = 0.0;
    wf[j] = 0.0f;
    if (r < M && cin[h]) {
      double sum;
      if constexpr (LONG) sum = sacc[j];
      else sum = 0.0 + diag_sum(j);
      double nrm = e.row_norm[r];
      bool empty = nrm < kEmptyThresh;
      double s = empty ? 0.0 : sum * g.sa[r] * s_c[h] / nrm;
      kv = empty ? 0.0 : e.sig2 * fpow(s, e.power, pi);
      double pm1 = pi == 2 ? s : (pi == 1 ? 1.0 : fpow(s, e.power - 1, 0));
      wf[j] = (float)(empty ? 0.0 : e.sig2 * a_c[h] * e.power * pm1);
    }
    Kst[rr * HN + cc % HN] = kv;
    int i = 4 * (j >> 3) + (j & 3);
    if (h == 0) rsum[i] = kv * a_c[0];
    else rsum[i] += kv * a_c[1];
  }
  // Row sums over the wave's 32 columns, then over each two wave columns
  // through LDS: one energy partial per (kI8TileN columns, row).
#pragma unroll
  for (int i = 0; i < NV / 2; i++) {
    double v = rsum[i];
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    if (r16 == 0) red[wc * BM + wr * 16 * RA + 16 * (i >> 2) + 4 * k16 + (i & 3)] = v;
  }
  __syncthreads();
  // k: rows of the tile as 16-byte pairs of columns (ldk even, 16-byte base).
  if (e.K) {
    double *K = e.K_as<double>();
    for (int q = tid; q < BM * (BN / 2); q += NT) {
      int rr = q / (BN / 2), c2 = 2 * (q % (BN / 2)), r = row0 + rr, cg = col0 + c2;
      if (r >= M || cg >= N) continue;
      double *dst = K + (size_t)r * e.ldk + cg;
      const double *src =
          reinterpret_cast<const double *>(c2 < HN ? buf0 : buf1) + rr * HN + c2 % HN;
      if (cg + 1 < N)
        *reinterpret_cast<double2 *>(dst) = *reinterpret_cast<const double2 *>(src);
      else
        dst[0] = src[0];
    }
  }
  for (int q = tid; q < BM * (BN / kI8TileN); q += NT) {
    int r = row0 + q % BM, t = q / BM, ct = col0 / kI8TileN + t;
    if (r < M && ct * kI8TileN < N)
      e.part[(size_t)ct * e.part_ld + r] =
          red[2 * t * BM + q % BM] + red[(2 * t + 1) * BM + q % BM];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NV; j++) {
    int rr = wr * 16 * RA + 16 * (j >> 3) + 4 * k16 + (j & 3);
    int cc = wc * 32 + 16 * ((j >> 2) & 1) + r16;
    __bf16 hi = (__bf16)wf[j], lo = (__bf16)(wf[j] - (float)hi);
    Hst[rr * WLD + cc] = __builtin_bit_cast(uint16_t, hi);
    Lst[rr * WLD + cc] = __builtin_bit_cast(uint16_t, lo);
  }
  __syncthreads();
  // w pieces in the tiled split layout, 8 columns per 16-byte store; the padding
  // columns [N, ldw) are zero (the reduction tail of the gradient contraction),
  // none past ldw (a multiple of 32) is written.
  for (int q = tid; q < BM * (BN / 8); q += NT) {
    int blk = q >> 6, rr = blk / (BN / 32) * 16 + ((q >> 2) & 15);
    int c8 = blk % (BN / 32) * 32 + 8 * (q & 3), r = row0 + rr, cg = col0 + c8;
    if (r >= M || cg >= e.ldw) continue;
    size_t o = split_offset(r, cg, e.ldw / kSplitPad);
    *reinterpret_cast<v4i *>(reinterpret_cast<uint16_t *>(e.Wh) + o) =
        *reinterpret_cast<const v4i *>(&Hst[rr * WLD + c8]);
    *reinterpret_cast<v4i *>(reinterpret_cast<uint16_t *>(e.Wl) + o) =
        *reinterpret_cast<const v4i *>(&Lst[rr * WLD + c8]);
  }
}

int gemm_col_tiles(int form, int N) {
  int bn = form == FM_FORM_FP64 ? 16 : kI8TileN;
  return (N + bn - 1) / bn;
}

int gemm_row_tiles(int M) { return (M + 63) / 64 * 2; }

namespace {

// FLARE_MI_TILE_SHAPE=i pins shape i of every contraction that has as many (tests
// check that every shape gives the same results); -1 without it or past the last.
// Largest first: wave tiles of 64, 48, 32 and 16 (FP64; 48 for EP_STORE only),
// tiles of 128 and 64 columns (int8), of 256 and 128 (split BF16).
int pinned_shape(int n_shapes) {
  const char *f = std::getenv("FLARE_MI_TILE_SHAPE");
  int i = f ? std::atoi(f) : -1;
  return i < n_shapes ? i : -1;
}

template <int EP>
void f64_launch(hipStream_t st, int T, bool dma, int blocks, const F64Groups &gs) {
  dim3 grid(blocks), block(256);
  if (T <= 2 && dma) {
    if (T == 1) hipLaunchKernelGGL((k_gemm_f64_dma<EP, 1>), grid, block, 0, st, gs);
    else hipLaunchKernelGGL((k_gemm_f64_dma<EP, 2>), grid, block, 0, st, gs);
  } else if (T == 1) {
    hipLaunchKernelGGL((k_gemm_f64<EP, 1, 2>), grid, block, 0, st, gs);
  } else if (T == 2) {
    hipLaunchKernelGGL((k_gemm_f64<EP, 2, 1>), grid, block, 0, st, gs);
  } else if constexpr (EP == EP_STORE) {
    if (T == 3) hipLaunchKernelGGL((k_gemm_f64<EP, 3, 1>), grid, block, 0, st, gs);
    else hipLaunchKernelGGL((k_gemm_f64<EP, 4, 1>), grid, block, 0, st, gs);
  } else {
    hipLaunchKernelGGL((k_gemm_f64_lds<EP>), grid, block, 0, st, gs);
  }
}

}  // namespace

void slice_rows(hipStream_t st, const float *X, long long ldx, int n, int nd, int8_t *Q,
                long long Kq, int tr, double *scale) {
  if (n <= 0) return;
  FM_CHECK(Kq % kI8Pad == 0 && Kq >= nd && tr > 0, FM_ERR_INVALID, "bad slice layout");
  hipLaunchKernelGGL(k_slice_rows<float>, dim3((n + 3) / 4), dim3(256), 0, st, X, ldx, n, nd, Q,
                     Kq / kI8Pad, tr, scale);
  FM_HIP(hipGetLastError());
}

void slice_rows(hipStream_t st, const double *X, long long ldx, int n, int nd, int8_t *Q,
                long long Kq, int tr, double *scale) {
  if (n <= 0) return;
  FM_CHECK(Kq % kI8Pad == 0 && Kq >= nd && tr > 0, FM_ERR_INVALID, "bad slice layout");
  hipLaunchKernelGGL(k_slice_rows<double>, dim3((n + 3) / 4), dim3(256), 0, st, X, ldx, n, nd,
                     Q, Kq / kI8Pad, tr, scale);
  FM_HIP(hipGetLastError());
}

// Columns of the integer contraction's tiles, 32 RA: 128 (RA = 4) moves less
// data per product and is the faster one where the tiles fill the GPU (one
// workgroup per CU: two LDS buffers of a step take 160 KB), 64 (RA = 2) where they
// are few. A round of tiles over the 256 CUs takes 1.75 times as long at 128
// columns (us per launch with 64 and with 128: 46 and 78 for 3,000 x 130 x 2,112,
// one round each; 489 and 421 for 16,000 x 1,000 x 2,112, eight and four).
// Reductions long enough for the LONG form have it at 64 columns.
void gemm_i8_groups(hipStream_t st, const std::vector<I8Gemm> &all) {
  for (size_t g0 = 0; g0 < all.size(); g0 += kI8Groups) {
    I8Groups gs{};
    gs.n = (int)std::min<size_t>(kI8Groups, all.size() - g0);
    long long b2 = 0, b4 = 0, nk = 0;
    for (int k = 0; k < gs.n; k++) {
      const I8Gemm &g = gs.g[k] = all[g0 + k];
      const EpArgs &e = g.e;
      FM_CHECK(g.M > 0 && g.N > 0 && g.nk > 0, FM_ERR_INVALID, "empty integer contraction");
      FM_CHECK(g.A && g.B && g.sa && g.sb && ((uintptr_t)g.A | (uintptr_t)g.B) % 16 == 0,
               FM_ERR_INVALID, "sliced operands must be 16-byte aligned");
      FM_CHECK(e.Wh && e.Wl && e.alpha && e.row_norm && e.part, FM_ERR_INVALID,
               "integer contraction: missing epilogue outputs");
      FM_CHECK(e.ldw % 32 == 0 && e.ldw >= g.N && ((uintptr_t)e.Wh | (uintptr_t)e.Wl) % 16 == 0 &&
                   (!e.K || (e.ldk % 2 == 0 && e.ldk >= g.N && (uintptr_t)e.K % 16 == 0)),
               FM_ERR_INVALID, "integer contraction: k and w must be 16-byte aligned rows");
      long long rows = (g.M + kI8TileA - 1) / kI8TileA;
      b2 += rows * ((g.N + 63) / 64);
      b4 += rows * ((g.N + 127) / 128);
      nk = std::max<long long>(nk, g.nk);
      FM_CHECK(b2 < (1LL << 31), FM_ERR_CAPACITY, "contraction too large for one launch");
    }
    bool is_long = nk * kI8Pad > kI8Flush;
    int pin = pinned_shape(2);
    bool wide = pin < 0 ? 7 * ((b4 + 255) / 256) <= 4 * ((b2 + 255) / 256) : pin == 0;
    int RA = wide && !is_long ? 4 : 2;
    for (int k = 0, first = 0; k < gs.n; k++) {
      gs.first[k] = first;
      first += (gs.g[k].M + kI8TileA - 1) / kI8TileA * ((gs.g[k].N + 32 * RA - 1) / (32 * RA));
    }
    dim3 grid(RA == 4 ? b4 : b2), block(512);
    if (is_long) hipLaunchKernelGGL((k_gemm_i8<true, 2>), grid, block, 0, st, gs);
    else if (RA == 2) hipLaunchKernelGGL((k_gemm_i8<false, 2>), grid, block, 0, st, gs);
    else hipLaunchKernelGGL((k_gemm_i8<false, 4>), grid, block, 0, st, gs);
    FM_HIP(hipGetLastError());
  }
}

// Wave tile of a launch, 16T x 16T: the least estimated time per 16 k, rounds
// of waves over the SIMDs times the measured time of one wave's 16 k. That
// time is nearly the same whether a wave has its SIMD to itself (three groups
// of 170 x 167 x 1,500) or the chip is full (32,000 x 1,000 x 2,100):
//   T = 4  2.1 us (full chip: 68 TFLOP/s for EP_STORE, 60 for EP_KERNEL
//                  through LDS; the matrix cores' limit, where the kernel
//                  before had 48)
//   T = 3  1.25   (63, EP_STORE only)
//   T = 2  0.58   (63, 61; k_gemm_f64 without aligned rows 0.72: 50, 47)
//   T = 1  0.18   (54, 53; without 0.35: 27)
// EP_KERNEL in us at T = 4, 2, 1 (and 2, 1 without aligned rows): 2 x 2,000 x
// 500 x 2,100 takes 309, 159, 174 (207, 359); 3 x 8,000 x 200 x 1,500 402, 312, 344
// (421, 615); 2 x 512 x 200 x 4,080 572, 158, 51 (228, 120); 3 x 170 x 167 x
// 1,500 219, 62, 21 (73, 34); 108 x 32 x 144 31, 11, 5 (13, 9). EP_SUMSQ, 3 x 200 x
// 8,000, triangular: 64, 42, 43 (50, 66).
static int f64_tile(int ep, const std::vector<F64Gemm> &gs, bool dma) {
  const double kTime[5] = {0, dma ? 0.18 : 0.35, dma ? 0.58 : 0.72, 1.25, 2.1};
  int pin = pinned_shape(4);
  if (pin >= 0 && !(pin == 1 && ep != EP_STORE)) return 4 - pin;
  constexpr int kSimds = 1024;  // 256 CUs
  int best = 0;
  double best_cost = 0;
  for (int T = 4; T >= 1; T--) {
    if (T == 3 && ep != EP_STORE) continue;
    int b = 16 * T;
    double waves = 0;
    for (const F64Gemm &g : gs)
      waves += (double)((g.M + b - 1) / b) * ((g.N + b - 1) / b);
    double rounds = std::ceil(waves / kSimds);
    // Triangular rows take half the steps on average, the last ones all.
    if (gs[0].lower_tri) rounds = 0.5 * rounds + 0.5;
    if (best == 0 || rounds * kTime[T] < best_cost) {
      best = T;
      best_cost = rounds * kTime[T];
    }
  }
  return best;
}

void gemm_f64_groups(hipStream_t st, int ep, const std::vector<F64Gemm> &all) {
  std::vector<F64Gemm> live;
  for (const F64Gemm &g : all)
    if (g.M > 0 && g.N > 0) live.push_back(g);
  if (live.empty()) return;
  // Operands whose rows start at 16 bytes (and 64 rows within 2 GB); for EP_STORE
  // the steps end at the last k, so K is even, too.
  bool dma = true;
  for (const F64Gemm &g : live)
    dma = dma && ((uintptr_t)g.A | (uintptr_t)g.B) % 16 == 0 && g.lda % 2 == 0 &&
          g.ldb % 2 == 0 && std::max(g.lda, g.ldb) < (1ll << 22) && (ep != EP_STORE || g.K % 2 == 0);
  int T = f64_tile(ep, live, dma);
  for (size_t g0 = 0; g0 < live.size(); g0 += kF64Groups) {
    F64Groups gs{};
    gs.n = (int)std::min<size_t>(kF64Groups, live.size() - g0);
    long long blocks = 0;
    for (int k = 0; k < gs.n; k++) {
      const F64Gemm &g = gs.g[k] = live[g0 + k];
      FM_CHECK(g.lower_tri == live[g0].lower_tri, FM_ERR_INVALID,
               "one launch takes triangular operands only or none");
      gs.first[k] = (int)blocks;
      gs.ntx[k] = (g.N + 32 * T - 1) / (32 * T);
      int rows = ep == EP_SUMSQ ? (g.M + 63) / 64 * 64 : g.M;
      gs.nty[k] = (rows + 32 * T - 1) / (32 * T);
      blocks += (long long)gs.ntx[k] * gs.nty[k];
      FM_CHECK(blocks < (1LL << 31), FM_ERR_CAPACITY, "contraction too large for one launch");
    }
    gs.first[gs.n] = (int)blocks;
    bool p12 = live[g0].e.power == 2.0 || live[g0].e.power == 1.0;  // one model, one power
    if (ep == EP_KERNEL && p12) f64_launch<EP_KERNEL>(st, T, dma, (int)blocks, gs);
    else if (ep == EP_KERNEL) f64_launch<EP_KERNEL_POW>(st, T, dma, (int)blocks, gs);
    else if (ep == EP_STORE) f64_launch<EP_STORE>(st, T, dma, (int)blocks, gs);
    else f64_launch<EP_SUMSQ>(st, T, dma, (int)blocks, gs);
    FM_HIP(hipGetLastError());
  }
}

void gemm_f64(hipStream_t st, int ep, int M, int N, int K, const double *A, long long lda,
              const double *B, long long ldb, int lower_tri, const EpArgs &e) {
  gemm_f64_groups(st, ep, {F64Gemm{A, B, lda, ldb, M, N, K, lower_tri, e}});
}

void split_rows(hipStream_t st, const double *X, long long ldx, int n, int K, uint16_t *hi,
                uint16_t *lo) {
  if (n <= 0 || K <= 0) return;
  long long nk = split_ld(K) / kSplitPad, chunks = (long long)(n + 15) / 16 * nk * 64;
  hipLaunchKernelGGL(k_split_rows, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, st, X,
                     ldx, n, K, nk, hi, lo);
  FM_HIP(hipGetLastError());
}

// Tiles of 256 x 256 (one workgroup per CU) move half the data of 128 x 128 ones
// (two per CU), but leave more of the last round and of ragged edges empty. A
// round of large ones takes 1.92 times as long as one of small ones (us with
// small and with large: 330 in 9 rounds and 359 in 5 for two groups of 16,000 x
// 2,100 x 1,000; 1039 in 24 and 999 in 12 for three of 43,000 x 1,500 x 500; 5670
// in 105 and 5405 in 53 for three of 87,381 x 3,255 x 1,365).
void gemm_split_groups(hipStream_t st, const std::vector<SplitGemm> &all) {
  for (size_t g0 = 0; g0 < all.size(); g0 += kSplitGroups) {
    SplitGroups gs{};
    gs.n = (int)std::min<size_t>(kSplitGroups, all.size() - g0);
    auto tiles = [&](int k, int bm, int bn) {
      return (long long)((gs.g[k].M + bm - 1) / bm) * ((gs.g[k].N + bn - 1) / bn);
    };
    long long small = 0, large = 0;
    for (int k = 0; k < gs.n; k++) {
      const SplitGemm &g = gs.g[k] = all[g0 + k];
      FM_CHECK(g.M > 0 && g.N > 0 && g.nk > 0 && g.e.W, FM_ERR_INVALID, "empty split contraction");
      for (int pc = 0; pc < 2; pc++)
        FM_CHECK(g.A[pc] && g.B[pc] && ((uintptr_t)g.A[pc] | (uintptr_t)g.B[pc]) % 16 == 0,
                 FM_ERR_INVALID, "split operands must be 16-byte aligned");
      small += tiles(k, 128, 128);
      large += tiles(k, 256, 256);
      FM_CHECK(small < (1LL << 31), FM_ERR_CAPACITY, "contraction too large for one launch");
    }
    int pin = pinned_shape(2);
    bool big = pin < 0 ? 25 * ((large + 255) / 256) <= 13 * ((small + 511) / 512) : pin == 0;
    int t = big ? 256 : 128;
    for (int k = 0, first = 0; k < gs.n; k++) {
      gs.first[k] = first;
      first += (int)tiles(k, t, t);
    }
    if (big)
      hipLaunchKernelGGL((k_gemm_split<8, 4, 2, 4>), dim3(large), dim3(512), 0, st, gs);
    else
      hipLaunchKernelGGL((k_gemm_split<4, 4, 2, 2>), dim3(small), dim3(256), 0, st, gs);
    FM_HIP(hipGetLastError());
  }
}

}  // namespace fm
