// Full kernel matrices for the DTC and SOR variances of small structures
// (sparse_gp.cpp:667-729): dense descriptor derivatives dB/dr
// (b2.cpp:181-242), the kernel matrix K = envs_struc(sparse, structure)
// (normalized_dot_product.cpp:117-214), the self kernel
// (normalized_dot_product.cpp:450-586), and diag(K^T Kuu^-1 K) and
// diag(K^T Sigma K) as |L_inv K|^2 and |R_inv^T K|^2 on the matrix cores.
//
// These follow the reference's dense formulation on purpose (the DTC
// variance needs the force-force products); memory grows as nb_s^2 per
// species, so they are meant for structures of up to a few thousand atoms,
// as in the reference.
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "fm_device.hpp"
#include "fm_gemm.hpp"
#include "fm_internal.hpp"

namespace fm {

constexpr int kMaxHCd = 2;

__constant__ double c_knorm_d[kMaxH];

// Species-sorted bonds: rows in species order, the bonds of a row contiguous
// (b2.cpp:150-154). One wavefront per row.
__global__ __launch_bounds__(256) void k_row_bonds(int n, const int *atom_of_row,
                                                   const int *bond_off, int *cnt) {
  int r = blockIdx.x * 256 + threadIdx.x;
  if (r < n) cnt[r] = bond_off[atom_of_row[r] + 1] - bond_off[atom_of_row[r]];
}
__global__ __launch_bounds__(256) void k_sorted_bonds(int n, const int *atom_of_row,
                                                      const int *bond_off, const int *sb_off,
                                                      int *sb_pos, int *sb_row, int *sb_bond) {
  int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (r >= n) return;
  int i = atom_of_row[r], b0 = bond_off[i], b1 = bond_off[i + 1], f0 = sb_off[r];
  for (int b = b0 + lane; b < b1; b += 64) {
    int f = f0 + b - b0;
    sb_pos[b] = f;
    sb_row[f] = r;
    sb_bond[f] = b;
  }
}

// ---------------------------------------------------------------------------
// Dense dB/dr per bond and component (b2.cpp:219-228), written at the
// bond's species-sorted position f (rows 3 f + m: the layout of
// DescriptorValues::descriptor_force_dervs), and the force dots dB . B
// (b2.cpp:236-240). A wavefront per bond at a time: the blocks of atom
// blockIdx.x (gridDim.y of them) deal its bonds to their waves. c comes from the
// descriptor pass. What bounds it: the LDS reads of the pair loop; 14,000 bonds
// of d = 544 take 80 us (640 with one wave per atom, which summed c first, at
// 256 waves on the whole GPU).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_b2_dervs(
    int nos, int N, int H, int nrad, int nd, int L1, int cutkind, double r1, const int *species,
    const int *bond_off, const int *bond_q, const int *nspec, const double *rel,
    const double *cutoffs, const int *row_of_atom, const int *sb_off, const double *C,
    const double *B, double *DB, double *fdots) {
  extern __shared__ __align__(16) unsigned char smem[];
  int i = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6, W = blockDim.x >> 6;
  double *c = reinterpret_cast<double *>(smem);                          // nrad x H
  double *dc = c + (size_t)nrad * H + (size_t)w * N * H * 3;  // N x H x 3 (this wave's bond)
  int si = species[i], b0 = bond_off[i], b1 = bond_off[i + 1], row = row_of_atom[i];
  for (int q = threadIdx.x; q < nrad * H; q += blockDim.x) c[q] = C[(size_t)i * nrad * H + q];
  __syncthreads();
  int ls[kMaxHCd], ms[kMaxHCd];
  double kn[kMaxHCd];
  for (int ch = 0; ch < kMaxHCd; ch++) {
    int lm = lane + 64 * ch;
    int lmc = lm < H ? lm : 0;
    int l = 0;
    while ((l + 1) * (l + 1) <= lmc) l++;
    ls[ch] = l;
    ms[ch] = lmc - l * l - l;
    kn[ch] = c_knorm_d[lmc];
  }
  const double *Brow = B + (size_t)row * nd;
  for (int b = b0 + blockIdx.y * W + w; b < b1; b += gridDim.y * W) {
    int qn = bond_q[b];
    int sj = nspec[qn];
    const double *rp = rel + 4 * (size_t)qn;
    double rc = cutoffs[si * nos + sj];
    double g[kMaxN], dg[kMaxN];
    radial_basis<double>(rp[0], rc, r1, N, cutkind, g, dg);
    double r = rp[0], rinv = 1.0 / r;
    double ux = rp[1] * rinv, uy = rp[2] * rinv, uz = rp[3] * rinv;
    wave_lds_sync();  // the last bond's dc has been read
    for (int ch = 0; ch < kMaxHCd; ch++) {
      int lm = lane + 64 * ch;
      if (lm >= H) continue;
      double Y, Yx, Yy, Yz;
      sph_harm_lane<double, true>(ls[ch], ms[ch], kn[ch], ux, uy, uz, rinv, Y, Yx, Yy, Yz);
      for (int nn = 0; nn < N; nn++) {
        double *o = dc + ((size_t)nn * H + lm) * 3;
        o[0] = dg[nn] * ux * Y + g[nn] * Yx;
        o[1] = dg[nn] * uy * Y + g[nn] * Yy;
        o[2] = dg[nn] * uz * Y + g[nn] * Yz;
      }
    }
    wave_lds_sync();
    int f = sb_off[row] + (b - b0);
    double fd[3] = {0, 0, 0};
    for (int k = lane; k < nd; k += 64) {
      int p = k / L1, l = k - p * L1;
      // Pair p is (n1, n2 >= n1), those of n1 from first(n1) on.
      auto first = [&](int a) { return a * nrad - a * (a - 1) / 2; };
      float t = 2 * nrad + 1;
      int n1 = (int)((t - sqrtf(t * t - 8 * p)) * 0.5f);
      n1 += first(n1 + 1) <= p;
      n1 -= first(n1) > p;
      int n2 = n1 + p - first(n1);
      double acc[3] = {0, 0, 0};
      // dB = c1 dc2 + dc1 c2; dc is zero but for the neighbour's species.
      if (n2 / N == sj || n1 / N == sj) {
        bool in1 = n1 / N == sj, in2 = n2 / N == sj;
        const double *d1 = dc + ((size_t)(in1 ? n1 - sj * N : 0) * H + l * l) * 3;
        const double *d2 = dc + ((size_t)(in2 ? n2 - sj * N : 0) * H + l * l) * 3;
        const double *c1 = c + n1 * H + l * l, *c2 = c + n2 * H + l * l;
        for (int mm = 0; mm < 2 * l + 1; mm++) {
          double c1v = in2 ? c1[mm] : 0.0, c2v = in1 ? c2[mm] : 0.0;
          for (int comp = 0; comp < 3; comp++)
            acc[comp] += c1v * d2[3 * mm + comp] + d1[3 * mm + comp] * c2v;
        }
      }
      for (int comp = 0; comp < 3; comp++) {
        DB[((size_t)3 * f + comp) * nd + k] = acc[comp];
        fd[comp] += acc[comp] * Brow[k];
      }
    }
    for (int comp = 0; comp < 3; comp++) {
      double v = wave_sum(fd[comp]);
      if (lane == 0) fdots[3 * (size_t)f + comp] = v;
    }
  }
}

__device__ __forceinline__ double dpow(double x, double p) {
  if (p == 2.0) return x * x;
  if (p == 1.0) return x;
  return pow(x, p);
}

// ---------------------------------------------------------------------------
// K = envs_struc for the sparse environments of one species t, written
// transposed (Kt: n_out x M, column cs + j).
// ---------------------------------------------------------------------------
struct EnvsArgs {
  int n, M, cs, Ms, t, ro, nt, sbo, nbt;
  double sig2, power, vol_inv;
  const int *species, *row_of_atom, *bond_off, *in_off, *in_bond, *sb_pos, *sb_row, *bond_q;
  const double *norm, *xnorm, *rel;
  const double *S;   // nt x Ms: x_hat_j . B_r (raw B)
  const double *FD;  // 3 nbt x Ms: x_hat_j . dB_f,m
  const double *fdots;
  double *P;   // nt x 7 x Ms: energy and sums of fk(m) coord(n), n >= m, per row
  double *Kt;
};

// Forces on atom blockIdx.x: + its own bonds, - bonds pointing at it
// (normalized_dot_product.cpp:197-199), owners of species t only, and the row's
// part of the energy and stress, with fk(j, f, m) = sigma^2 p S^(p-1)
// (x_hat . dB / |B| - S fdot / |B|^2), the force kernel of
// normalized_dot_product.cpp:187-195 with S = x.B/(|x||B|). Lanes are sparse
// environments (S, FD and Kt are read and written in whole lines), the block's
// four waves split the bonds. 256 atoms, 150 environments: 25 us (165 with
// threads on atoms, whose loads and stores of one environment were a row apart).
__global__ __launch_bounds__(256) void k_envs_rows(EnvsArgs e) {
  __shared__ double sh[4][10][64];
  int a = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int j = blockIdx.y * 64 + lane, jc = min(j, e.Ms - 1);
  double acc[10] = {};  // force, energy, stress
  auto fk = [&](int r, int f, double *out) {
    double inv = 1.0 / e.norm[r], s = e.S[(size_t)(r - e.ro) * e.Ms + jc] * inv;
    double dval = e.sig2 * e.power * dpow(s, e.power - 1) * inv;
    const double *FD = e.FD + (size_t)3 * (f - e.sbo) * e.Ms + jc;
#pragma unroll
    for (int m = 0; m < 3; m++)
      out[m] = dval * (FD[(size_t)m * e.Ms] - s * e.fdots[3 * (size_t)f + m] * inv);
  };
  int row = e.row_of_atom[a];
  bool own = e.species[a] == e.t;
  if (own && e.norm[row] >= kEmptyThresh) {
    if (w == 0)
      acc[3] = e.sig2 * dpow(e.S[(size_t)(row - e.ro) * e.Ms + jc] / e.norm[row], e.power);
    for (int b = e.bond_off[a] + w; b < e.bond_off[a + 1]; b += 4) {
      double v[3];
      fk(row, e.sb_pos[b], v);
      const double *co = e.rel + 4 * (size_t)e.bond_q[b] + 1;
      int sc = 4;
#pragma unroll
      for (int m = 0; m < 3; m++) {
        acc[m] += v[m];
#pragma unroll
        for (int nn = m; nn < 3; nn++) acc[sc++] += v[m] * co[nn];
      }
    }
  }
  for (int q = e.in_off[a] + w; q < e.in_off[a + 1]; q += 4) {
    int f = e.sb_pos[e.in_bond[q]];
    if (f < e.sbo || f >= e.sbo + e.nbt) continue;  // owner of another species
    int r = e.sb_row[f];
    if (e.norm[r] < kEmptyThresh) continue;
    double v[3];
    fk(r, f, v);
#pragma unroll
    for (int m = 0; m < 3; m++) acc[m] -= v[m];
  }
#pragma unroll
  for (int q = 0; q < 10; q++) sh[w][q][lane] = acc[q];
  __syncthreads();
  if (j >= e.Ms) return;
  bool empty = e.xnorm[j] < kEmptyThresh;
  for (int q = w; q < (own ? 10 : 3); q += 4) {
    double v = (sh[0][q][lane] + sh[1][q][lane]) + (sh[2][q][lane] + sh[3][q][lane]);
    if (empty) v = 0;
    if (q < 3) e.Kt[(size_t)(1 + 3 * a + q) * e.M + e.cs + j] = v;
    else e.P[((size_t)(row - e.ro) * 7 + (q - 3)) * e.Ms + j] = v;
  }
}

// Energy and stress of the sparse environments: E = sum_r sigma^2 S^p;
// S_mn = -1/V sum_f fk(m) coord_f(n), n >= m (normalized_dot_product.cpp:175-177,
// 201-206) from the rows' parts, quantity blockIdx.y. 16 waves take 16 rows each
// at a time, one per running sum, and the 256 sums are added pairwise: one sum per
// wave made the energies' rounding 10 to 40 % larger.
__global__ __launch_bounds__(1024) void k_envs_sums(EnvsArgs e) {
  constexpr int U = 16;
  __shared__ double sh[16][64];
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = blockIdx.y;
  int j = blockIdx.x * 64 + lane, jc = min(j, e.Ms - 1);
  double v[U] = {};
  auto pairwise = [&] {
#pragma unroll
    for (int d = U / 2; d > 0; d /= 2)
#pragma unroll
      for (int u = 0; u < d; u++) v[u] += v[u + d];
  };
  for (int r0 = w; r0 < e.nt; r0 += 16 * U)
#pragma unroll
    for (int u = 0; u < U; u++) {
      int r = r0 + 16 * u;
      if (r < e.nt) v[u] += e.P[((size_t)r * 7 + q) * e.Ms + jc];
    }
  pairwise();
  sh[w][lane] = v[0];
  __syncthreads();
  if (w > 0 || j >= e.Ms) return;
#pragma unroll
  for (int u = 0; u < U; u++) v[u] = sh[u][lane];
  pairwise();
  int c = q == 0 ? 0 : 1 + 3 * e.n + (q - 1);
  e.Kt[(size_t)c * e.M + e.cs + j] = q == 0 ? v[0] : -v[0] * e.vol_inv;
}

// out (cols x rows) = in (rows x cols)^T.
__global__ __launch_bounds__(256) void k_transpose(int rows, int cols, const double *in,
                                                   double *out) {
  __shared__ double t[32][33];
  int c0 = blockIdx.y * 32, r0 = blockIdx.x * 32, x = threadIdx.x & 31, y = threadIdx.x >> 5;
  for (int k = y; k < 32; k += 8)
    if (r0 + k < rows && c0 + x < cols) t[k][x] = in[(size_t)(r0 + k) * cols + c0 + x];
  __syncthreads();
  for (int k = y; k < 32; k += 8)
    if (c0 + k < cols && r0 + x < rows) out[(size_t)(c0 + k) * rows + r0 + x] = t[x][k];
}

// ---------------------------------------------------------------------------
// Self kernel of one species (normalized_dot_product.cpp:450-586), literally:
// pairs j >= i with factor 2 off the diagonal, bond pairs (f1 of i, f2 of j)
// and components m, scattered by the atom-index coincidences of the
// reference. One wavefront per row i; lanes take bonds f1 of i.
// ---------------------------------------------------------------------------
struct SelfArgs {
  int ro, nt, sbo, nbt, n;
  double sig2, power, vol_inv_sq;
  const int *atom_of_row, *sb_off, *nbr_of_f, *sb_bond, *bond_q;
  const double *norm, *rel;
  const double *BB;   // nt x nt raw dots
  const double *FD2;  // 3 nbt x nt: dB_f,m . B_r
  const double *FF;   // 3 x nbt x nbt: dB_f1,m . dB_f2,m
  const double *fdots;
  double *Pn;  // 3 nb: per bond (species-sorted position)
  double *Pc;  // 3 n rows
  double *Ps;  // 6 n rows
  double *Pe;  // n rows
  int *bad;
};

__global__ __launch_bounds__(64) void k_self_pairs(SelfArgs a) {
  int il = blockIdx.x, lane = threadIdx.x;
  if (il >= a.nt) return;
  int ri = a.ro + il;
  double norm_i = a.norm[ri];
  double ec = 0, cc[3] = {0, 0, 0}, sc6[6] = {0, 0, 0, 0, 0, 0};
  int fb0 = a.sb_off[ri], fb1 = a.sb_off[ri + 1];
  if (norm_i >= kEmptyThresh) {
    double norm_i2 = norm_i * norm_i, norm_i3 = norm_i2 * norm_i;
    int ci1 = a.atom_of_row[ri];
    for (int fc = fb0; fc < fb1 || fc == fb0; fc += 64) {
      int f1 = fc + lane;
      bool own = f1 < fb1;
      int ni1 = own ? a.nbr_of_f[f1] : -1;
      const double *co1 = own ? a.rel + 4 * (size_t)a.bond_q[a.sb_bond[f1]] + 1 : nullptr;
      double nacc[3] = {0, 0, 0};
      for (int jl = il; jl < a.nt; jl++) {
        int rj = a.ro + jl;
        double norm_j = a.norm[rj];
        if (norm_j < kEmptyThresh) continue;
        double mult = (jl == il) ? 1 : 2;
        double norm_j2 = norm_j * norm_j, norm_j3 = norm_j2 * norm_j;
        double norm_ij = norm_i * norm_j;
        double norm_dot = a.BB[(size_t)il * a.nt + jl] / norm_ij;
        double c1 = (a.power - 1) * a.power * dpow(norm_dot, a.power - 2);
        if (fabs(norm_dot) < kEmptyThresh && a.power < 2) a.bad[0] = 1;
        double c2 = a.power * dpow(norm_dot, a.power - 1);
        if (fc == fb0 && lane == 0) ec += a.sig2 * mult * dpow(norm_dot, a.power);
        if (!own) continue;
        int ci2 = a.atom_of_row[rj];
        int fj0 = a.sb_off[rj], fj1 = a.sb_off[rj + 1];
        int fl1 = f1 - a.sbo;
        for (int f2 = fj0; f2 < fj1; f2++) {
          int ni2 = a.nbr_of_f[f2];
          int fl2 = f2 - a.sbo;
          const double *co2 = a.rel + 4 * (size_t)a.bond_q[a.sb_bond[f2]] + 1;
          int s_c = 0;
          for (int m = 0; m < 3; m++) {
            double fd1 = a.fdots[3 * (size_t)f1 + m], fd2 = a.fdots[3 * (size_t)f2 + m];
            double fdj = a.FD2[(3 * (size_t)fl1 + m) * a.nt + jl];
            double fdi = a.FD2[(3 * (size_t)fl2 + m) * a.nt + il];
            double v1 = fdj / norm_ij - norm_dot * fd1 / norm_i2;
            double v2 = fdi / norm_ij - norm_dot * fd2 / norm_j2;
            double v3 = a.FF[((size_t)m * a.nbt + fl1) * a.nbt + fl2] / norm_ij;
            double v4 = fd1 * fdi / (norm_i3 * norm_j);
            double v5 = fd2 * fdj / (norm_i * norm_j3);
            double v6 = fd1 * fd2 * norm_dot / (norm_i2 * norm_j2);
            double kv = a.sig2 * mult * (c1 * v1 * v2 + c2 * (v3 - v4 - v5 + v6));
            if (ci1 == ci2) cc[m] += kv;
            if (ci1 == ni2) cc[m] -= kv;
            if (ni1 == ci2) nacc[m] -= kv;
            if (ni1 == ni2) nacc[m] += kv;
            for (int nn = m; nn < 3; nn++) {
              sc6[s_c] += kv * co1[nn] * co2[nn] * a.vol_inv_sq;
              s_c++;
            }
          }
        }
      }
      if (own)
        for (int m = 0; m < 3; m++) a.Pn[3 * (size_t)f1 + m] = nacc[m];
      if (fb1 == fb0) break;
    }
  } else {
    for (int f1 = fb0 + lane; f1 < fb1; f1 += 64)
      for (int m = 0; m < 3; m++) a.Pn[3 * (size_t)f1 + m] = 0;
  }
  for (int m = 0; m < 3; m++) cc[m] = wave_sum(cc[m]);
  for (int q = 0; q < 6; q++) sc6[q] = wave_sum(sc6[q]);
  ec = wave_sum(ec);
  if (lane == 0) {
    for (int m = 0; m < 3; m++) a.Pc[3 * (size_t)ri + m] = cc[m];
    for (int q = 0; q < 6; q++) a.Ps[6 * (size_t)ri + q] = sc6[q];
    a.Pe[ri] = ec;
  }
}

// K_self columns: energy and stress as sums over rows, forces as the own
// row's partial plus the partials of bonds pointing at the atom.
__global__ void k_self_forces(int n, const int *row_of_atom, const int *in_off,
                              const int *in_bond, const int *sb_pos, const double *Pc,
                              const double *Pn, double *kself) {
  int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= n) return;
  int r = row_of_atom[a];
  double acc[3] = {Pc[3 * (size_t)r], Pc[3 * (size_t)r + 1], Pc[3 * (size_t)r + 2]};
  for (int q = in_off[a]; q < in_off[a + 1]; q++) {
    int f = sb_pos[in_bond[q]];
    for (int m = 0; m < 3; m++) acc[m] += Pn[3 * (size_t)f + m];
  }
  for (int m = 0; m < 3; m++) kself[1 + 3 * a + m] = acc[m];
}

__global__ __launch_bounds__(256) void k_self_sums(int n, const double *Pe, const double *Ps,
                                                   double *kself) {
  __shared__ double sh[7][256];
  double acc[7] = {0, 0, 0, 0, 0, 0, 0};
  for (int r = threadIdx.x; r < n; r += blockDim.x) {
    acc[0] += Pe[r];
    for (int q = 0; q < 6; q++) acc[1 + q] += Ps[6 * (size_t)r + q];
  }
  for (int q = 0; q < 7; q++) sh[q][threadIdx.x] = acc[q];
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (threadIdx.x < st)
      for (int q = 0; q < 7; q++) sh[q][threadIdx.x] += sh[q][threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) kself[0] = sh[0][0];
  if (threadIdx.x >= 1 && threadIdx.x < 7) kself[1 + 3 * n + threadIdx.x - 1] = sh[threadIdx.x][0];
}

// var = kself - sum Q partials + sum V partials (DTC) or the V partials (SOR).
__global__ void k_var_efs(int n_out, int dtc, const double *kself, const double *Qp, int nq,
                          const double *Vp, int nv, double *var) {
  int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n_out) return;
  double q = 0, v = 0;
  for (int t = 0; t < nq; t += 2)
    q += Qp[(size_t)t * n_out + c] + Qp[(size_t)(t + 1) * n_out + c];
  for (int t = 0; t < nv; t += 2)
    v += Vp[(size_t)t * n_out + c] + Vp[(size_t)(t + 1) * n_out + c];
  var[c] = dtc ? kself[c] - q + v : v;
}

// ---------------------------------------------------------------------------
// Host orchestration
// ---------------------------------------------------------------------------
void dense_setup() {
  double kn[kMaxH];
  knorm_values(kMaxL, kn);
  FM_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_knorm_d), kn, sizeof(kn), 0, hipMemcpyHostToDevice));
}

void compute_dervs(fm_structure s) {
  if (s->has_dervs) return;
  FM_CHECK(s->has_b2 && s->form == FM_FORM_FP64, FM_ERR_STATE,
           "dense descriptor derivatives need FP64 descriptors");
  FM_CHECK(s->desc_kind == 2, FM_ERR_INVALID,
           "dense descriptor derivatives are built for the B2 descriptor");
  fm_context ctx = s->ctx;
  hipStream_t st = ctx->stream;
  Pool *pool = &ctx->pool;
  int n = s->n, nd = s->nd, H = (s->lmax + 1) * (s->lmax + 1), nrad = s->nos * s->N;
  size_t nb = (size_t)s->n_bonds;
  FM_CHECK((double)nb * 3 * nd * 8 < 64e9, FM_ERR_CAPACITY,
           "dense descriptor derivatives exceed 64 GB; the adjoint path needs none");
  s->nbt_off.assign(s->nos + 1, 0);
  for (int t = 0; t < s->nos; t++) s->nbt_off[t + 1] = s->nbt_off[t] + s->nb_by_type[t];
  for (DevBuf *b : {&s->sb_pos, &s->sb_row, &s->sb_bond})
    b->alloc(pool, std::max<size_t>(1, nb * sizeof(int)));
  s->sb_off.alloc(pool, (size_t)(n + 1) * sizeof(int));
  s->DB.alloc(pool, std::max<size_t>(1, nb * 3 * nd * sizeof(double)));
  s->fdots.alloc(pool, std::max<size_t>(1, nb * 3 * sizeof(double)));
  DevBuf cnt(pool, std::max<size_t>(1, (size_t)n * sizeof(int)));
  if (n > 0) {
    hipLaunchKernelGGL(k_row_bonds, dim3((n + 255) / 256), dim3(256), 0, st, n,
                       s->atom_of_row.as<int>(), s->bond_off.as<int>(), cnt.as<int>());
    scan_exclusive(ctx, cnt.as<int>(), s->sb_off.as<int>(), n);
    hipLaunchKernelGGL(k_sorted_bonds, dim3((n + 3) / 4), dim3(256), 0, st, n,
                       s->atom_of_row.as<int>(), s->bond_off.as<int>(), s->sb_off.as<int>(),
                       s->sb_pos.as<int>(), s->sb_row.as<int>(), s->sb_bond.as<int>());
  }
  // Four waves per block where their workspaces keep two blocks on a CU, and
  // blocks per atom for some 8192 waves in all, no more than the bonds need.
  auto lds_of = [&](int W) {
    return ((size_t)nrad * H + (size_t)W * s->N * H * 3) * sizeof(double);
  };
  int W = lds_of(4) <= 80 * 1024 ? 4 : 1;
  size_t lds = lds_of(W);
  FM_CHECK(lds <= 160 * 1024, FM_ERR_CAPACITY, "derivative workspace exceeds LDS");
  if (n > 0) {
    int need = (int)std::min<size_t>((nb / n + W) / W, 1024);
    int y = std::max(1, std::min(need, 8192 / (n * W)));
    hipLaunchKernelGGL(k_b2_dervs, dim3(n, y), dim3(64 * W), lds, st, s->nos, s->N, H, nrad, nd,
                       s->lmax + 1, s->cutkind, s->r1, s->species.as<int>(),
                       s->bond_off.as<int>(), s->bond_q.as<int>(), s->nspecies.as<int>(),
                       s->rel.as<double>(), s->d_cutoffs.as<double>(), s->row_of_atom.as<int>(),
                       s->sb_off.as<int>(), s->C.as<double>(),
                       s->B.as<double>(), s->DB.as<double>(), s->fdots.as<double>());
  }
  FM_HIP(hipGetLastError());
  s->has_dervs = true;
}

// Kt (n_out x M) = envs_struc(sparse, structure)^T. The products of all species
// in one launch, up to 4 GB of them at a time.
static void envs_struc_t(fm_model m, fm_structure s, DevBuf &Kt) {
  fm_context ctx = s->ctx;
  hipStream_t st = ctx->stream;
  Pool *pool = &ctx->pool;
  int n = s->n, nd = s->nd, M = m->M;
  size_t n_out = 1 + 3 * (size_t)n + 6;
  Kt.alloc(pool, std::max<size_t>(1, n_out * M * sizeof(double)));
  auto doubles = [&](int t) {  // S, FD and P of species t
    return (size_t)m->M_by_type[t] * (8 * (size_t)s->n_by_type[t] + 3 * (size_t)s->nb_by_type[t]);
  };
  for (int t0 = 0, t1; t0 < s->nos; t0 = t1) {
    size_t total = doubles(t0);
    for (t1 = t0 + 1; t1 < s->nos && total + doubles(t1) <= (4ull << 30) / 8; t1++)
      total += doubles(t1);
    DevBuf work(pool, std::max<size_t>(1, total * sizeof(double)));
    double *at = work.as<double>();
    std::vector<F64Gemm> products;
    std::vector<EnvsArgs> envs;
    for (int t = t0; t < t1; t++) {
      int Ms = m->M_by_type[t], nt = s->n_by_type[t], ro = s->type_off[t];
      int sbo = s->nbt_off[t], nbt = s->nbt_off[t + 1] - s->nbt_off[t];
      if (Ms == 0) continue;
      FM_CHECK(Ms < 65536, FM_ERR_CAPACITY,
               "more than 65535 sparse environments of one species");
      EnvsArgs e;
      e.S = at;
      e.FD = at + (size_t)nt * Ms;
      e.P = at + ((size_t)nt + 3 * (size_t)nbt) * Ms;
      at += doubles(t);
      auto product = [&](const double *rows, int count, const double *out) {
        EpArgs ep;
        ep.W = const_cast<double *>(out);
        ep.ldw = Ms;
        products.push_back(
            {rows, m->X[t].as<double>(), nd, nd, count, Ms, nd, 0, ep});
      };
      product(s->B.as<double>() + (size_t)ro * nd, nt, e.S);
      product(s->DB.as<double>() + (size_t)3 * sbo * nd, 3 * nbt, e.FD);
      e.n = n;
      e.M = M;
      e.cs = m->off[t];
      e.Ms = Ms;
      e.t = t;
      e.ro = ro;
      e.nt = nt;
      e.sbo = sbo;
      e.nbt = nbt;
      e.sig2 = m->sigma * m->sigma;
      e.power = m->power;
      e.vol_inv = 1.0 / s->volume;
      e.species = s->species.as<int>();
      e.row_of_atom = s->row_of_atom.as<int>();
      e.bond_off = s->bond_off.as<int>();
      e.in_off = s->in_off.as<int>();
      e.in_bond = s->in_bond.as<int>();
      e.sb_pos = s->sb_pos.as<int>();
      e.sb_row = s->sb_row.as<int>();
      e.bond_q = s->bond_q.as<int>();
      e.norm = s->norm.as<double>();
      e.xnorm = m->xnorm.as<double>() + m->off[t];
      e.rel = s->rel.as<double>();
      e.fdots = s->fdots.as<double>();
      e.Kt = Kt.as<double>();
      envs.push_back(e);
    }
    gemm_f64_groups(st, EP_STORE, products);
    for (const EnvsArgs &e : envs) {
      unsigned by = (e.Ms + 63) / 64;
      if (n > 0) hipLaunchKernelGGL(k_envs_rows, dim3(n, by), dim3(256), 0, st, e);
      hipLaunchKernelGGL(k_envs_sums, dim3(by, 7), dim3(1024), 0, st, e);
    }
    FM_HIP(hipGetLastError());
    FM_HIP(hipStreamSynchronize(st));
  }
}

// One 32 x 32 tile per block, both results in whole lines.
__global__ __launch_bounds__(256) void k_normalize_rows(int rows, int cols, const double *norm,
                                                        double *X, double *XT) {
  __shared__ double t[32][33];
  int r0 = blockIdx.x * 32, c0 = blockIdx.y * 32, x = threadIdx.x & 31, y = threadIdx.x >> 5;
  for (; c0 < cols; c0 += 32 * gridDim.y) {
    for (int k = y; k < 32; k += 8) {
      int r = r0 + k, c = c0 + x;
      if (r >= rows || c >= cols) continue;
      double v = norm[r] < kEmptyThresh ? 0.0 : X[(size_t)r * cols + c] / norm[r];
      X[(size_t)r * cols + c] = t[k][x] = v;
    }
    __syncthreads();
    for (int k = y; k < 32; k += 8)
      if (c0 + k < cols && r0 + x < rows) XT[(size_t)(c0 + k) * rows + r0 + x] = t[x][k];
    __syncthreads();
  }
}

void normalize_rows(hipStream_t st, int rows, int cols, const double *norm, double *X,
                    double *XT) {
  if (rows == 0) return;
  int ty = std::min((cols + 31) / 32, 65535);
  hipLaunchKernelGGL(k_normalize_rows, dim3((rows + 31) / 32, ty), dim3(256), 0, st, rows, cols,
                     norm, X, XT);
  FM_HIP(hipGetLastError());
}

static void self_kernel(fm_model m, fm_structure s, DevBuf &kself) {
  fm_context ctx = s->ctx;
  hipStream_t st = ctx->stream;
  Pool *pool = &ctx->pool;
  int n = s->n, nd = s->nd;
  size_t n_out = 1 + 3 * (size_t)n + 6;
  kself.alloc(pool, n_out * sizeof(double));
  FM_HIP(hipMemsetAsync(kself.as<double>(), 0, n_out * sizeof(double), st));
  if (n == 0) return;
  DevBuf Pn(pool, std::max<size_t>(1, (size_t)3 * s->n_bonds * sizeof(double)));
  DevBuf Pc(pool, (size_t)3 * n * sizeof(double)), Ps(pool, (size_t)6 * n * sizeof(double)),
      Pe(pool, (size_t)n * sizeof(double)), bad(pool, sizeof(int));
  FM_HIP(hipMemsetAsync(bad.as<int>(), 0, sizeof(int), st));
  // Neighbour (structure index) of every species-sorted bond.
  std::vector<int> sbb(s->n_bonds), bq(s->n_bonds), sidx(s->n_nb);
  if (s->n_bonds) {
    FM_HIP(hipMemcpyAsync(sbb.data(), s->sb_bond.as<int>(), sbb.size() * sizeof(int),
                          hipMemcpyDeviceToHost, st));
    FM_HIP(hipMemcpyAsync(bq.data(), s->bond_q.as<int>(), bq.size() * sizeof(int),
                          hipMemcpyDeviceToHost, st));
  }
  if (s->n_nb)
    FM_HIP(hipMemcpyAsync(sidx.data(), s->sidx.as<int>(), sidx.size() * sizeof(int),
                          hipMemcpyDeviceToHost, st));
  FM_HIP(hipStreamSynchronize(st));
  std::vector<int> nbr(s->n_bonds);
  for (size_t f = 0; f < nbr.size(); f++) nbr[f] = sidx[bq[sbb[f]]];
  DevBuf d_nbr(pool, std::max<size_t>(1, nbr.size() * sizeof(int)));
  if (!nbr.empty())
    FM_HIP(hipMemcpyAsync(d_nbr.as<int>(), nbr.data(), nbr.size() * sizeof(int),
                          hipMemcpyHostToDevice, st));
  for (int t = 0; t < s->nos; t++) {
    int nt = s->n_by_type[t], ro = s->type_off[t];
    int sbo = s->nbt_off[t], nbt = s->nbt_off[t + 1] - s->nbt_off[t];
    if (nt == 0) continue;
    FM_CHECK((double)nbt * nbt * 3 * 8 < 64e9, FM_ERR_CAPACITY,
             "the self kernel's force-force products exceed 64 GB");
    DevBuf BB(pool, (size_t)nt * nt * sizeof(double));
    DevBuf FD2(pool, std::max<size_t>(1, (size_t)3 * nbt * nt * sizeof(double)));
    DevBuf FF(pool, std::max<size_t>(1, (size_t)3 * nbt * nbt * sizeof(double)));
    const double *Bs = s->B.as<double>() + (size_t)ro * nd;
    const double *DBs = s->DB.as<double>() + (size_t)3 * sbo * nd;
    EpArgs e;
    e.W = BB.as<void>();
    e.ldw = nt;
    gemm_f64(st, EP_STORE, nt, nt, nd, Bs, nd, Bs, nd, 0, e);
    if (nbt > 0) {
      e.W = FD2.as<void>();
      e.ldw = nt;
      gemm_f64(st, EP_STORE, 3 * nbt, nt, nd, DBs, nd, Bs, nd, 0, e);
      for (int mm = 0; mm < 3; mm++) {
        e.W = FF.as<double>() + (size_t)mm * nbt * nbt;
        e.ldw = nbt;
        gemm_f64(st, EP_STORE, nbt, nbt, nd, DBs + (size_t)mm * nd, 3 * (long long)nd,
                 DBs + (size_t)mm * nd, 3 * (long long)nd, 0, e);
      }
    }
    SelfArgs a;
    a.ro = ro;
    a.nt = nt;
    a.sbo = sbo;
    a.nbt = nbt;
    a.n = n;
    a.sig2 = m->sigma * m->sigma;
    a.power = m->power;
    a.vol_inv_sq = 1.0 / (s->volume * s->volume);
    a.atom_of_row = s->atom_of_row.as<int>();
    a.sb_off = s->sb_off.as<int>();
    a.nbr_of_f = d_nbr.as<int>();
    a.sb_bond = s->sb_bond.as<int>();
    a.bond_q = s->bond_q.as<int>();
    a.norm = s->norm.as<double>();
    a.rel = s->rel.as<double>();
    a.BB = BB.as<double>();
    a.FD2 = FD2.as<double>();
    a.FF = FF.as<double>();
    a.fdots = s->fdots.as<double>();
    a.Pn = Pn.as<double>();
    a.Pc = Pc.as<double>();
    a.Ps = Ps.as<double>();
    a.Pe = Pe.as<double>();
    a.bad = bad.as<int>();
    hipLaunchKernelGGL(k_self_pairs, dim3(nt), dim3(64), 0, st, a);
    FM_HIP(hipGetLastError());
    FM_HIP(hipStreamSynchronize(st));
  }
  int hb = 0;
  FM_HIP(hipMemcpyAsync(&hb, bad.as<int>(), sizeof(int), hipMemcpyDeviceToHost, st));
  FM_HIP(hipStreamSynchronize(st));
  FM_CHECK(!hb, FM_ERR_INVALID,
           "Dot product of descriptors is 0, and the negative power function in force-force "
           "kernel diverges.");
  hipLaunchKernelGGL(k_self_forces, dim3((n + 255) / 256), dim3(256), 0, st, n,
                     s->row_of_atom.as<int>(), s->in_off.as<int>(), s->in_bond.as<int>(),
                     s->sb_pos.as<int>(), Pc.as<double>(), Pn.as<double>(), kself.as<double>());
  hipLaunchKernelGGL(k_self_sums, dim3(1), dim3(256), 0, st, n, Pe.as<double>(), Ps.as<double>(),
                     kself.as<double>());
  FM_HIP(hipGetLastError());
  FM_HIP(hipStreamSynchronize(st));
}

void envs_struc(fm_model m, fm_structure s, double *K_out) {
  FM_CHECK(s->n_struct == 1, FM_ERR_INVALID, "kernel matrices are per single structure");
  compute_dervs(s);
  DevBuf Kt;
  envs_struc_t(m, s, Kt);
  hipStream_t st = s->ctx->stream;
  int n_out = 1 + 3 * s->n + 6, M = m->M;
  if (M == 0) return;
  size_t bytes = (size_t)n_out * M * sizeof(double);
  DevBuf K(&s->ctx->pool, bytes);
  hipLaunchKernelGGL(k_transpose, dim3((n_out + 31) / 32, (M + 31) / 32), dim3(256), 0, st, n_out,
                     M, Kt.as<double>(), K.as<double>());
  FM_HIP(hipGetLastError());
  FM_HIP(hipMemcpyAsync(K_out, K.as<double>(), bytes, hipMemcpyDeviceToHost, st));
  FM_HIP(hipStreamSynchronize(st));
}

void self_kernel_struc(fm_model m, fm_structure s, double *kself_out) {
  FM_CHECK(s->n_struct == 1, FM_ERR_INVALID, "kernel matrices are per single structure");
  compute_dervs(s);
  DevBuf ks;
  self_kernel(m, s, ks);
  size_t n_out = 1 + 3 * (size_t)s->n + 6;
  FM_HIP(hipMemcpyAsync(kself_out, ks.as<double>(), n_out * sizeof(double), hipMemcpyDeviceToHost,
                        s->ctx->stream));
  FM_HIP(hipStreamSynchronize(s->ctx->stream));
}

void predict_dense(fm_model m, fm_structure s, int kind, double *mean_efs, double *var_efs) {
  FM_CHECK(s->n_struct == 1, FM_ERR_INVALID, "DTC/SOR variances are per single structure");
  FM_CHECK(m->has_R, FM_ERR_STATE, "R_inv is needed for the DTC and SOR variances");
  FM_CHECK(kind != 1 || m->has_L, FM_ERR_STATE,
           "L_inv must be up to date to make predictions. Please call update_matrices_QR and try "
           "again.");
  fm_context ctx = s->ctx;
  hipStream_t st = ctx->stream;
  Pool *pool = &ctx->pool;
  compute_dervs(s);
  int M = m->M;
  size_t n_out = 1 + 3 * (size_t)s->n + 6;
  DevBuf Kt, ks;
  envs_struc_t(m, s, Kt);
  // mean = K^T alpha
  DevBuf mean(pool, n_out * sizeof(double));
  {
    EpArgs e;
    e.W = mean.as<void>();
    e.ldw = 1;
    gemm_f64(st, EP_STORE, (int)n_out, 1, M, Kt.as<double>(), M, m->alpha_full.as<double>(), M, 0,
             e);
  }
  int dtc = kind == 1;
  if (dtc) self_kernel(m, s, ks);
  // |L_inv K_c|^2 per species block and |R_inv^T K_c|^2.
  int nq = 0;
  for (int t = 0; t < m->nos; t++) nq += dtc ? gemm_row_tiles(m->L_rows[t]) : 0;
  int nv = gemm_row_tiles(M);
  DevBuf Qp(pool, std::max<size_t>(1, (size_t)nq * n_out * sizeof(double)));
  DevBuf Vp(pool, std::max<size_t>(1, (size_t)nv * n_out * sizeof(double)));
  int qo = 0;
  if (dtc)
    for (int t = 0; t < m->nos; t++) {
      if (m->M_by_type[t] == 0 || m->L_rows[t] == 0) continue;
      EpArgs eq;
      eq.part = Qp.as<double>() + (size_t)qo * n_out;
      eq.part_ld = n_out;
      gemm_f64(st, EP_SUMSQ, m->L_rows[t], (int)n_out, m->M_by_type[t], m->L[t].as<double>(),
               m->M_by_type[t], Kt.as<double>() + m->off[t], M, m->L_lower[t], eq);
      qo += gemm_row_tiles(m->L_rows[t]);
    }
  {
    EpArgs ev;
    ev.part = Vp.as<double>();
    ev.part_ld = n_out;
    gemm_f64(st, EP_SUMSQ, M, (int)n_out, M, m->RinvT.as<double>(), M, Kt.as<double>(), M,
             m->R_lower, ev);
  }
  DevBuf var(pool, n_out * sizeof(double));
  hipLaunchKernelGGL(k_var_efs, dim3((unsigned)((n_out + 255) / 256)), dim3(256), 0, st,
                     (int)n_out, dtc, dtc ? ks.as<double>() : nullptr, Qp.as<double>(), qo,
                     Vp.as<double>(), nv, var.as<double>());
  FM_HIP(hipGetLastError());
  if (mean_efs)
    FM_HIP(hipMemcpyAsync(mean_efs, mean.as<double>(), n_out * sizeof(double),
                          hipMemcpyDeviceToHost, st));
  if (var_efs)
    FM_HIP(hipMemcpyAsync(var_efs, var.as<double>(), n_out * sizeof(double), hipMemcpyDeviceToHost,
                          st));
  FM_HIP(hipStreamSynchronize(st));
}

}  // namespace fm
