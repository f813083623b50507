// Prediction pipeline on the device: per species, the kernel contraction
// (S = B_s X_hat^T with its fused epilogue), the gradient contraction
// G = W X_hat, the optional variance contraction Q = L_s^-1 K^T, then the
// adjoint bond forces and a deterministic gather of forces, energy and
// stress (sparse_gp.cpp:643-665 and 731-757; output layout of
// normalized_dot_product.cpp:117-214).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "fm_device.hpp"
#include "fm_gather.hpp"
#include "fm_gemm.hpp"
#include "fm_internal.hpp"

namespace fm {

// Per row (species-sorted atom): E = sum of the energy partials over column
// tiles; var = sigma^2 (B.B / |B|^2)^p - sum of the |Q|^2 partials over row
// tiles (the diagonal of envs_envs(cluster, cluster) minus diag(Q1^T Q1),
// sparse_gp.cpp:116-136). Partials are summed in tile order.
// Rows [ro, ro + n_rows); partial t of row r at t * part_ld + r.
__device__ __forceinline__ double row_variance(int r, const double *Qpart, int n_qtiles,
                                               long long part_ld, double nrm, double nnr,
                                               double sig2, double power) {
  double v = 0;
  if (nrm >= kEmptyThresh) {
    double nd = nnr / (nrm * nrm);
    double ks = sig2 * (power == 2.0 ? nd * nd : pow(nd, power));
    double q = 0;
#pragma unroll 8
    for (int t = 0; t < n_qtiles; t += 2)
      q += Qpart[(size_t)t * part_ld + r] + Qpart[(size_t)(t + 1) * part_ld + r];
    v = ks - q;
  }
  return v;
}

__global__ void k_species_final(int n_rows, int ro, const double *Epart, int n_etiles,
                                const double *Qpart, int n_qtiles, long long part_ld,
                                const double *norm, const double *nn, double sig2, double power,
                                double *E_row, double *var_row) {
  int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n_rows) return;
  double e = 0;
#pragma unroll 8
  for (int t = 0; t < n_etiles; t++) e += Epart[(size_t)t * part_ld + r];
  E_row[ro + r] = e;
  if (var_row)
    var_row[ro + r] =
        row_variance(r, Qpart, n_qtiles, part_ld, norm[ro + r], nn[ro + r], sig2, power);
}

// Row sums of the untiled path for up to kFinalTypes species in one launch:
// species u's rows are [ro[u], ro[u + 1]), its nt[u] partials of ld ro[u + 1] -
// ro[u] at part[u].
constexpr int kFinalTypes = 8;
struct FinalArgs {
  int types, ro[kFinalTypes + 1], nt[kFinalTypes];
  const double *part[kFinalTypes];
};

// Local energies.
__global__ void k_energy_final(FinalArgs a, double *E_row) {
  int r = a.ro[0] + blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= a.ro[a.types]) return;
  int u = 0;
  while (r >= a.ro[u + 1]) u++;
  long long ld = a.ro[u + 1] - a.ro[u];
  const double *p = a.part[u] + (r - a.ro[u]);
  double e = 0;
#pragma unroll 8
  for (int t = 0; t < a.nt[u]; t++) e += p[t * ld];
  E_row[r] = e;
}

// Local variances.
__global__ void k_var_final(FinalArgs a, const double *norm, const double *nn, double sig2,
                            double power, double *var_row) {
  int r = a.ro[0] + blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= a.ro[a.types]) return;
  int u = 0;
  while (r >= a.ro[u + 1]) u++;
  var_row[r] = row_variance(r - a.ro[u], a.part[u], a.nt[u], a.ro[u + 1] - a.ro[u], norm[r],
                            nn[r], sig2, power);
}

// Calls launch(args, rows) for the species of a structure, kFinalTypes at a
// time; part(t) gives species t's partials and their count.
template <typename Part, typename Launch>
static void for_final_types(fm_structure s, Part &&part, Launch &&launch) {
  for (int t0 = 0; t0 < s->nos; t0 += kFinalTypes) {
    FinalArgs a{};
    a.types = std::min(kFinalTypes, s->nos - t0);
    for (int u = 0; u < a.types; u++) {
      a.ro[u] = s->type_off[t0 + u];
      part(t0 + u, a.part[u], a.nt[u]);
    }
    a.ro[a.types] = s->type_off[t0 + a.types];
    if (a.ro[a.types] > a.ro[0]) launch(a, a.ro[a.types] - a.ro[0]);
  }
  FM_HIP(hipGetLastError());
}

// Per structure (one wave each): energy and stress -1/V sum_b f (x) r
// (normalized_dot_product.cpp:201-206).
__global__ __launch_bounds__(64) void k_final_sum(const int *struct_chunk_off, const double *part,
                                                  const double *vol_inv, const long long *mean_off,
                                                  const int *atom_off, double *out) {
  int k = blockIdx.x;
  double acc[7];
  structure_sums<7>(struct_chunk_off, part, k, acc);
  if (threadIdx.x != 0) return;
  double *o = out + mean_off[k];
  int nk = atom_off[k + 1] - atom_off[k];
  o[0] = acc[0];
  for (int q = 0; q < 6; q++) o[1 + 3 * nk + q] = acc[1 + q] * vol_inv[k];
}

__global__ void k_fill(double *p, long long n, double v) {
  long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Per-atom forces (own bonds minus incoming bonds), energies and virials
// into `o` (one mean_efs block per structure).
static void gather_forces(fm_structure s, bool f64, DevBuf &fbond, DevBuf &vir, DevBuf &E_row,
                          double *o) {
  hipStream_t st = s->ctx->stream;
  Pool *pool = &s->ctx->pool;
  KScope timer(s->ctx, KT_GATHER);
  auto forces = [&](auto *f) {
    using TF = std::remove_const_t<std::remove_pointer_t<decltype(f)>>;
    hipLaunchKernelGGL(k_forces<TF>, dim3((s->n + kGatherAtoms - 1) / kGatherAtoms), dim3(256), 0,
                       st, s->n, s->atom_struct.as<int>(), s->d_atom_off.as<int>(),
                       s->d_mean_off.as<long long>(), s->bond_off.as<int>(), s->in_off.as<int>(),
                       s->in_bond.as<int>(), (const TF *)f, s->row_of_atom.as<int>(),
                       E_row.as<double>(), o, (double *)nullptr);
  };
  if (f64) forces(fbond.as<double>());
  else forces(fbond.as<float>());
  DevBuf blk(pool, (size_t)s->n_chunks * 7 * sizeof(double));
  hipLaunchKernelGGL(k_chunk_sums<7>, dim3(s->n_chunks), dim3(256), 0, st,
                     s->d_chunk_begin.as<int>(), s->d_chunk_end.as<int>(),
                     s->row_of_atom.as<int>(), E_row.as<double>(), vir.as<double>(),
                     blk.as<double>());
  hipLaunchKernelGGL(k_final_sum, dim3(s->n_struct), dim3(64), 0, st,
                     s->d_struct_chunk_off.as<int>(), blk.as<double>(), s->d_vol_inv.as<double>(),
                     s->d_mean_off.as<long long>(), s->d_atom_off.as<int>(), o);
}

// out[pos[r]] = in[r]: species-sorted rows to another order on the device.
__global__ void k_scatter_rows(int n, const int *pos, const double *in, double *out) {
  int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r < n) out[pos[r]] = in[r];
}

// Atoms of each (species, structure) of a batch, species-major. A wavefront
// whose atoms all lie in one structure (atoms of a structure are
// consecutive) adds one count per species from lane 0.
__global__ void k_struct_species_count(int n, const int *species, const int *atom_struct,
                                       int n_struct, int nos, int *cnt) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  bool ok = i < n;
  int k = ok ? atom_struct[i] : -1, t = ok ? species[i] : -1;
  int k0 = __shfl(k, 0, 64);
  if (nos <= 8 && __all(!ok || k == k0)) {
    for (int u = 0; u < nos; u++) {
      unsigned long long m = __ballot(ok && t == u);
      if (m != 0 && (threadIdx.x & 63) == 0)
        atomicAdd(&cnt[(size_t)u * n_struct + k0], (int)__popcll(m));
    }
  } else if (ok) {
    atomicAdd(&cnt[(size_t)t * n_struct + k], 1);
  }
}

// Position of species-sorted row r in its structure's species-sorted order.
// Rows of one species keep atom order, so structure k's atoms of species t
// are the rows [ex[t][k], ex[t][k] + cnt[t][k]), ex the exclusive scan of
// the species-major counts.
__global__ void k_var_pos(int n, const int *atom_of_row, const int *species,
                          const int *atom_struct, const int *atom_off, const int *cnt,
                          const int *ex, int n_struct, int *var_pos) {
  int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  int i = atom_of_row[r], t = species[i], k = atom_struct[i];
  int before = 0;
  for (int u = 0; u < t; u++) before += cnt[(size_t)u * n_struct + k];
  var_pos[r] = atom_off[k] + before + (r - ex[(size_t)t * n_struct + k]);
}

void build_var_pos(fm_structure s) {
  fm_context ctx = s->ctx;
  hipStream_t st = ctx->stream;
  int n = s->n, ns = s->n_struct;
  if (ns <= 1 || n == 0) {
    s->var_pos.release();
    return;
  }
  int m = s->nos * ns;
  DevBuf cnt(&ctx->pool, (size_t)m * sizeof(int)), ex(&ctx->pool, (size_t)(m + 1) * sizeof(int));
  FM_HIP(hipMemsetAsync(cnt.as<int>(), 0, (size_t)m * sizeof(int), st));
  hipLaunchKernelGGL(k_struct_species_count, dim3((n + 255) / 256), dim3(256), 0, st, n,
                     s->species.as<int>(), s->atom_struct.as<int>(), ns, s->nos, cnt.as<int>());
  scan_exclusive(ctx, cnt.as<int>(), ex.as<int>(), m);
  s->var_pos.alloc(&ctx->pool, (size_t)n * sizeof(int));
  hipLaunchKernelGGL(k_var_pos, dim3((n + 255) / 256), dim3(256), 0, st, n,
                     s->atom_of_row.as<int>(), s->species.as<int>(), s->atom_struct.as<int>(),
                     s->d_atom_off.as<int>(), cnt.as<int>(), ex.as<int>(), ns,
                     s->var_pos.as<int>());
  FM_HIP(hipGetLastError());
}

struct StageOut {
  const double *src[3];
  size_t count[3];
};
// Up to three arrays to pinned host memory, one after the other: one launch (4 us
// for 108 atoms) where a copy each took 4 us and 9 of the caller's time.
__global__ __launch_bounds__(256) void k_stage_out(StageOut a, double *dst) {
  size_t i = blockIdx.x * (size_t)256 + threadIdx.x, at = i;
  for (int k = 0; k < 3; k++) {
    if (at < a.count[k]) {
      dst[i] = a.src[k][at];
      return;
    }
    at -= a.count[k];
  }
}

// Memory that the runtime does not know: pageable host memory.
static bool pageable_host(const void *p) {
  hipPointerAttribute_t a{};
  hipError_t rc = hipPointerGetAttributes(&a, p);
  if (rc != hipSuccess) (void)hipGetLastError();
  return rc != hipSuccess || a.type == hipMemoryTypeUnregistered;
}

// Up to kStageOut bytes in all go through the context's pinned memory if every
// destination is pageable (a copy to pageable memory waits for itself, 15 us
// each). The limit bounds the pinned memory: a call of 108, 8,192, 24,000 and
// 65,536 atoms takes 231, 374, 634 and 1,316 us with staging, 255, 390, 654 and
// 1,328 with copies.
constexpr size_t kStageOut = 256 << 10;

void read_back(fm_context ctx, const Output (&parts)[3], bool may_stage) {
  hipStream_t st = ctx->stream;
  size_t total = 0;
  StageOut so{};
  for (int k = 0; k < 3; k++)
    if (parts[k].dst) {
      so.src[k] = parts[k].src;
      so.count[k] = parts[k].count;
      total += parts[k].count;
    }
  bool staged = may_stage && total > 0 && total * sizeof(double) <= kStageOut;
  for (const Output &p : parts) staged = staged && (!p.dst || pageable_host(p.dst));
  if (!staged) {
    for (const Output &p : parts)
      if (p.dst && p.count)
        FM_HIP(hipMemcpyAsync(p.dst, p.src, p.count * sizeof(double), hipMemcpyDefault, st));
    FM_HIP(hipStreamSynchronize(st));
    return;
  }
  char *stage = ctx->stage(total * sizeof(double));
  void *dev = nullptr;
  FM_HIP(hipHostGetDevicePointer(&dev, stage, 0));
  hipLaunchKernelGGL(k_stage_out, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, so,
                     (double *)dev);
  FM_HIP(hipGetLastError());
  FM_HIP(hipStreamSynchronize(st));
  for (const Output &p : parts) {
    if (!p.dst) continue;
    std::memcpy(p.dst, stage, p.count * sizeof(double));
    stage += p.count * sizeof(double);
  }
}

// Results to the caller's buffers (any may be null).
static void read_outputs(fm_structure s, const double *o, size_t n_out, const double *var_row,
                         const double *E_row, double *mean_efs, double *local_var,
                         double *local_energy) {
  hipStream_t st = s->ctx->stream;
  Pool *pool = &s->ctx->pool;
  size_t n = s->n;
  DevBuf vperm, eperm;
  Output parts[3] = {{mean_efs, o, n_out}, {}, {}};
  if (local_var && var_row && n > 0) {
    // Species-sorted rows of the batch to each structure's species-sorted
    // order (compute_cluster_uncertainties order).
    const double *src = var_row;
    if (s->n_struct > 1) {
      vperm.alloc(pool, n * sizeof(double));
      hipLaunchKernelGGL(k_scatter_rows, dim3((n + 255) / 256), dim3(256), 0, st, (int)n,
                         s->var_pos.as<int>(), var_row, vperm.as<double>());
      src = vperm.as<double>();
    }
    parts[1] = {local_var, src, n};
  }
  if (local_energy && n > 0) {
    // E_row is in species-sorted order; local energies are in atom order.
    eperm.alloc(pool, n * sizeof(double));
    hipLaunchKernelGGL(k_scatter_rows, dim3((n + 255) / 256), dim3(256), 0, st, (int)n,
                       s->atom_of_row.as<int>(), E_row, eperm.as<double>());
    parts[2] = {local_energy, eperm.as<double>(), n};
  }
  FM_HIP(hipGetLastError());
  read_back(s->ctx, parts);
}

// Rows per tile of one species in the chosen form: at most T and, when T
// allows, a whole number of rounds of the kernel contraction's 128 x 128
// tiles over the GPU's CUs (one workgroup per CU), so the last round of each
// launch is not left nearly empty. Rows of a tile do not change any result.
static int species_tile_rows(fm_context ctx, int T, int Ms, int form) {
  if (form != FM_FORM_CHOSEN || Ms == 0) return T;
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) !=
          hipSuccess ||
      cus <= 0)
    return T;
  int per_round = cus / ((Ms + 2 * kI8TileN - 1) / (2 * kI8TileN));
  int rounds = per_round > 0 ? (T / kI8TileA) / per_round : 0;
  return rounds > 0 ? rounds * per_round * kI8TileA : T;
}

// The model's sparse rows as int8 slices for the chosen form's kernel
// contraction and their transpose as BF16 pieces for its gradient contraction,
// made on the context stream from the FP64 rows on first use.
static void model_slices(fm_model m, hipStream_t st) {
  if (m->xq_ready) return;
  int nd = m->nd;
  long long ldq = i8_ld(nd);
  Pool *pool = &m->ctx->pool;
  m->Xq.resize(m->nos);
  m->Xq_scale.resize(m->nos);
  m->XTs0.resize(m->nos);
  m->XTs1.resize(m->nos);
  for (int t = 0; t < m->nos; t++) {
    int Ms = m->M_by_type[t];
    if (Ms == 0) continue;
    m->Xq[t].alloc(pool, i8_tiled_bytes(Ms, kI8TileN, ldq));
    m->Xq_scale[t].alloc(pool, (size_t)Ms * sizeof(double));
    slice_rows(st, m->X[t].as<double>(), nd, Ms, nd, m->Xq[t].as<int8_t>(), ldq, kI8TileN,
               m->Xq_scale[t].as<double>());
    for (DevBuf *b : {&m->XTs0[t], &m->XTs1[t]})
      b->alloc(pool, split_elems(nd, Ms) * sizeof(uint16_t));
    split_rows(st, m->XT[t].as<double>(), Ms, nd, Ms, m->XTs0[t].as<uint16_t>(),
               m->XTs1[t].as<uint16_t>());
  }
  m->xq_ready = true;
}

// Chosen form: kernel contraction of `cnt` sliced descriptor rows against
// species t's sparse set.
static I8Gemm kernel_contraction_i8(fm_model m, int t, const int8_t *A, const double *scale,
                                    int cnt, int nd, const EpArgs &ek) {
  return {A, m->Xq[t].as<int8_t>(), scale, m->Xq_scale[t].as<double>(), cnt, m->M_by_type[t],
          (int)(i8_ld(nd) / kI8Pad), ek};
}

// Chosen form: gradient contraction of `cnt` rows of w (pieces Wh, Wl) with
// species t's sparse set.
static SplitGemm gradient_contraction(fm_model m, int t, const uint16_t *Wh, const uint16_t *Wl,
                                      int cnt, int nd, const EpArgs &eg) {
  return {{Wh, Wl},
          {m->XTs0[t].as<uint16_t>(), m->XTs1[t].as<uint16_t>()},
          cnt,
          nd,
          (int)(split_ld(m->M_by_type[t]) / kSplitPad),
          eg};
}

// The kernel contraction of `cnt` FP32 descriptor rows (leading dimension nd) without slices
// of their FP64 values, sliced into Aq / Aq_scale first (Aq holds at least
// i8_tiled_bytes(cnt, kI8TileA, i8_ld(nd)) bytes).
static void contract_fp32_rows(fm_model m, hipStream_t st, int t, const float *rows, int cnt,
                               int nd, DevBuf &Aq, DevBuf &Aq_scale, const EpArgs &ek) {
  {
    KScope timer(m->ctx, KT_SLICE, st);
    slice_rows(st, rows, nd, cnt, nd, Aq.as<int8_t>(), i8_ld(nd), kI8TileA,
               Aq_scale.as<double>());
  }
  KScope timer(m->ctx, KT_SGEMM, st);
  gemm_i8_groups(
      st, {kernel_contraction_i8(m, t, Aq.as<int8_t>(), Aq_scale.as<double>(), cnt, nd, ek)});
}

// B3 structures too large to keep their descriptors (s->row_tile > 0): each
// species' rows are processed in tiles of row_tile rows. Per tile: B3 rows
// (from the coefficients c kept for every atom), the kernel contraction with
// its energy partials, the variance contraction, the gradient contraction
// and the adjoint of the tile's atoms (their u and bond forces); the force
// gather runs once at the end. Every output element sums its terms in the
// order of the untiled path, so the results are the same bit for bit.
static void predict_tiled(fm_model m, fm_structure s, int flags, int form, double *mean_efs,
                          double *local_var, double *local_energy) {
  fm_context ctx = s->ctx;
  hipStream_t st = ctx->stream;
  Pool *pool = &ctx->pool;
  bool want_var = (flags & FM_PREDICT_LOCAL) != 0;
  bool f64 = form == FM_FORM_FP64;
  size_t esz = f64 ? sizeof(double) : sizeof(float);
  int n = s->n, nd = s->nd, nos = s->nos;
  size_t n_out = (size_t)s->mean_off[s->n_struct];
  int T = (int)std::min<int64_t>(s->row_tile, std::max(1, n));
  std::vector<size_t> eo(nos + 1, 0), qo(nos + 1, 0);
  int Mmax = 0;
  for (int t = 0; t < nos; t++) {
    size_t ns = s->n_by_type[t];
    int Ms = m->M_by_type[t];
    Mmax = std::max(Mmax, Ms);
    eo[t + 1] = eo[t] + ns * (size_t)std::max(1, gemm_col_tiles(form, Ms));
    int Lr = want_var ? m->L_rows[t] : 0;
    qo[t + 1] = qo[t] + ns * (size_t)gemm_row_tiles(Lr);
  }
  // Whole-structure buffers.
  DevBuf Epart(pool, std::max<size_t>(1, eo[nos] * sizeof(double)));
  DevBuf Qpart(pool, std::max<size_t>(1, qo[nos] * sizeof(double)));
  DevBuf E_row(pool, std::max<size_t>(1, (size_t)n * sizeof(double)));
  DevBuf var_row(pool, std::max<size_t>(1, (size_t)n * sizeof(double)));
  DevBuf out(pool, (size_t)n_out * sizeof(double));
  size_t nc = (size_t)s->nos * s->N * (s->lmax + 1) * (s->lmax + 1);
  DevBuf U(pool, std::max<size_t>(1, (size_t)n * nc * esz));
  DevBuf fbond(pool, std::max<size_t>(1, (size_t)3 * s->n_bonds * esz));
  DevBuf vir(pool, std::max<size_t>(1, (size_t)6 * n * sizeof(double)));
  // Tile buffers. k is FP64 in both forms (rows padded to 128 bytes).
  size_t kld = ((size_t)Mmax + 15) / 16 * 16;  // rows of whole 128-byte lines
  DevBuf Bt(pool, std::max<size_t>(1, (size_t)T * nd * esz));
  DevBuf Gt(pool, std::max<size_t>(1, (size_t)T * nd * esz));
  DevBuf Tq, Tq_scale, Wt, Wh, Wl, Kt;
  if (f64) {
    Wt.alloc(pool, std::max<size_t>(1, (size_t)T * Mmax * sizeof(double)));
  } else {
    model_slices(m, st);
    Tq.alloc(pool, std::max<size_t>(1, i8_tiled_bytes(T, kI8TileA, i8_ld(nd))));
    Tq_scale.alloc(pool, std::max<size_t>(1, (size_t)T * sizeof(double)));
    size_t w = split_elems(T, std::max(Mmax, 1)) * sizeof(uint16_t);
    Wh.alloc(pool, w);
    Wl.alloc(pool, w);
  }
  if (want_var) Kt.alloc(pool, std::max<size_t>(1, (size_t)T * kld * sizeof(double)));
  double sig2 = m->sigma * m->sigma;
  ctx->mark_begin(ST_SGEMM);
  for (int t = 0; t < nos; t++) {
    int ns = s->n_by_type[t], Ms = m->M_by_type[t], ro = s->type_off[t];
    int n_et = Ms == 0 ? 1 : gemm_col_tiles(form, Ms);
    int n_qt = (want_var && Ms > 0) ? gemm_row_tiles(m->L_rows[t]) : 0;
    int Ts = species_tile_rows(ctx, T, Ms, form);
    for (int c0 = 0; c0 < ns; c0 += Ts) {
      int cnt = std::min(Ts, ns - c0), r0 = ro + c0;
      launch_b3_rows(s, r0, cnt, true, Bt.as<void>());
      double *ep = Epart.as<double>() + eo[t] + c0;
      if (Ms == 0) {
        hipLaunchKernelGGL(k_fill, dim3((cnt + 255) / 256), dim3(256), 0, st, ep,
                           (long long)cnt, 0.0);
        FM_HIP(hipMemsetAsync(Gt.as<void>(), 0, (size_t)cnt * nd * esz, st));
      } else {
        // Kernel contraction of the tile.
        EpArgs ek;
        ek.sig2 = sig2;
        ek.power = m->power;
        ek.row_norm = s->norm.as<double>() + r0;
        ek.alpha = m->alpha[t].as<double>();
        if (f64) {
          ek.W = Wt.as<double>();
          ek.ldw = Ms;
        } else {
          ek.Wh = Wh.as<uint16_t>();
          ek.Wl = Wl.as<uint16_t>();
          ek.ldw = split_ld(Ms);
        }
        size_t kl = ((size_t)Ms + 1) / 2 * 2;
        if (want_var) {
          ek.K = Kt.as<void>();
          ek.ldk = (long long)kl;
        }
        ek.part = ep;
        ek.part_ld = ns;
        if (f64)
          gemm_f64(st, EP_KERNEL, cnt, Ms, nd, Bt.as<double>(), nd, m->X[t].as<double>(), nd, 0,
                   ek);
        else
          contract_fp32_rows(m, st, t, Bt.as<float>(), cnt, nd, Tq, Tq_scale, ek);
        // Variance contraction of the tile.
        if (want_var && m->L_rows[t] > 0) {
          EpArgs eq;
          eq.part = Qpart.as<double>() + qo[t] + c0;
          eq.part_ld = ns;
          gemm_f64(st, EP_SUMSQ, m->L_rows[t], cnt, Ms, m->L[t].as<double>(), Ms,
                   Kt.as<double>(), (long long)kl, m->L_lower[t], eq);
        }
        // Gradient contraction of the tile.
        EpArgs eg;
        eg.W = Gt.as<void>();
        eg.ldw = nd;
        if (f64) {
          gemm_f64(st, EP_STORE, cnt, nd, Ms, Wt.as<double>(), Ms, m->XT[t].as<double>(), Ms, 0,
                   eg);
        } else {
          gemm_split_groups(st, {gradient_contraction(m, t, Wh.as<uint16_t>(),
                                                      Wl.as<uint16_t>(), cnt, nd, eg)});
        }
      }
      hipLaunchKernelGGL(k_species_final, dim3((cnt + 255) / 256), dim3(256), 0, st, cnt, r0, ep,
                         n_et, Qpart.as<double>() + qo[t] + c0, n_qt, (long long)ns,
                         s->norm.as<double>(), s->nn.as<double>(), sig2, m->power,
                         E_row.as<double>(), want_var ? var_row.as<double>() : nullptr);
      // Adjoint of the tile's atoms: u, then their bonds' forces.
      launch_dEdc_b3_rows(s, r0, cnt, true, Bt.as<void>(), Gt.as<void>(), nd, 1, kEmptyThresh,
                          -1.0, U.as<void>());
      launch_bond_forces(s, U.as<void>(), fbond.as<void>(), vir.as<double>(),
                         s->atom_of_row.as<int>() + r0, cnt, kEmptyThresh, -1.0);
      FM_HIP(hipGetLastError());
    }
  }
  ctx->mark_end(ST_SGEMM);
  ctx->mark_begin(ST_ADJ);
  double *o = out.as<double>();
  if (n == 0) FM_HIP(hipMemsetAsync(o, 0, (size_t)n_out * sizeof(double), st));
  if (n > 0) gather_forces(s, f64, fbond, vir, E_row, o);
  FM_HIP(hipGetLastError());
  ctx->mark_end(ST_ADJ);
  read_outputs(s, o, n_out, want_var ? var_row.as<double>() : nullptr, E_row.as<double>(),
               mean_efs, local_var, local_energy);
}

void predict(fm_model m, fm_structure s, int flags, int form, double *mean_efs,
             double *local_var, double *local_energy) {
  fm_context ctx = s->ctx;
  hipStream_t st = ctx->stream;
  Pool *pool = &ctx->pool;
  FM_CHECK(s->has_b2, FM_ERR_STATE, "descriptors have not been computed for this structure");
  FM_CHECK(s->form == form, FM_ERR_STATE, "structure descriptors were computed in another form");
  FM_CHECK(m->nos == s->nos && m->nd == s->nd, FM_ERR_INVALID,
           "model and descriptor settings disagree (species or descriptor size)");
  if (s->desc_kind == 3)
    b3_order_model(m, s);  // the sparse set in the rows' (l-set major) order
  else
    FM_CHECK(m->b3_ntri == 0, FM_ERR_INVALID,
             "the model's sparse set is in B3 order (it was used with a B3 descriptor)");
  bool want_var = (flags & FM_PREDICT_LOCAL) != 0;
  FM_CHECK(!want_var || m->has_L, FM_ERR_STATE,
           "L_inv must be up to date to evaluate uncertainties");
  ctx->kt_clear(KT_SLICE, KT_GATHER);
  if (s->desc_kind == 3 && s->row_tile > 0)
    return predict_tiled(m, s, flags, form, mean_efs, local_var, local_energy);
  bool f64 = form == FM_FORM_FP64;
  size_t esz = f64 ? sizeof(double) : sizeof(float);
  int n = s->n, nd = s->nd, nos = s->nos;
  // mean_efs of every structure of the batch, concatenated.
  size_t n_out = (size_t)s->mean_off[s->n_struct];
  // Per-species slices of the atom-major w and k matrices (n_s x M_s each)
  // and of the energy / variance partials.
  // The chosen form keeps w as BF16 pairs in the tiled split layout.
  // k is FP64 in both forms, rows padded to 16 values (whole 128-byte lines).
  std::vector<size_t> wo(nos + 1, 0), eo(nos + 1, 0), qo(nos + 1, 0), so(nos + 1, 0),
      ko(nos + 1, 0), kld(nos, 0);
  for (int t = 0; t < nos; t++) {
    size_t ns = s->n_by_type[t], Ms = m->M_by_type[t];
    kld[t] = (Ms + 15) / 16 * 16;  // rows of whole 128-byte lines (w and k)
    wo[t + 1] = wo[t] + ns * kld[t];
    ko[t + 1] = ko[t] + ns * kld[t];
    so[t + 1] = so[t] + split_elems((long long)ns, (long long)Ms);
    eo[t + 1] = eo[t] + ns * (size_t)std::max(1, gemm_col_tiles(form, (int)Ms));
    int Lr = want_var ? m->L_rows[t] : 0;
    qo[t + 1] = qo[t] + ns * (size_t)gemm_row_tiles(Lr);
  }
  DevBuf W, Wh, Wl;
  if (f64) {
    W.alloc(pool, std::max<size_t>(1, wo[nos] * esz));
  } else {
    Wh.alloc(pool, std::max<size_t>(1, so[nos] * sizeof(uint16_t)));
    Wl.alloc(pool, std::max<size_t>(1, so[nos] * sizeof(uint16_t)));
  }
  DevBuf Kb;
  size_t ksz = sizeof(double);
  if (want_var) Kb.alloc(pool, std::max<size_t>(1, ko[nos] * ksz));
  // Chosen form: the descriptor rows' int8 slices, made by the descriptor
  // pass from the FP64 rows (B2), or here from the FP32 rows one species at
  // a time (B3).
  DevBuf Aq, Aq_scale;
  if (!f64) {
    model_slices(m, st);
    if (!s->has_q) {
      int nmax = 0;
      for (int t = 0; t < nos; t++) nmax = std::max(nmax, s->n_by_type[t]);
      Aq.alloc(pool, std::max<size_t>(1, i8_tiled_bytes(nmax, kI8TileA, i8_ld(nd))));
      Aq_scale.alloc(pool, std::max<size_t>(1, (size_t)nmax * sizeof(double)));
    }
  }
  DevBuf G(pool, std::max<size_t>(1, (size_t)n * nd * esz));
  DevBuf Epart(pool, std::max<size_t>(1, eo[nos] * sizeof(double)));
  DevBuf Qpart(pool, std::max<size_t>(1, qo[nos] * sizeof(double)));
  DevBuf E_row(pool, std::max<size_t>(1, (size_t)n * sizeof(double)));
  DevBuf var_row(pool, std::max<size_t>(1, (size_t)n * sizeof(double)));
  DevBuf out(pool, (size_t)n_out * sizeof(double));
  double sig2 = m->sigma * m->sigma;

  // Kernel contraction S = B_s X_hat_s^T with the fused epilogue, all species
  // in one launch.
  ctx->mark_begin(ST_SGEMM);
  std::vector<F64Gemm> f64_k, f64_g, f64_q;
  std::vector<I8Gemm> i8_k;
  std::vector<SplitGemm> split_g;
  for (int t = 0; t < nos; t++) {
    int ns = s->n_by_type[t], Ms = m->M_by_type[t], ro = s->type_off[t];
    if (ns == 0) continue;
    if (Ms == 0) continue;
    EpArgs ek;
    ek.sig2 = sig2;
    ek.power = m->power;
    ek.row_norm = s->norm.as<double>() + ro;
    ek.alpha = m->alpha[t].as<double>();
    if (f64) {
      ek.W = W.as<double>() + wo[t];
      ek.ldw = (long long)kld[t];
    } else {
      ek.Wh = Wh.as<uint16_t>() + so[t];
      ek.Wl = Wl.as<uint16_t>() + so[t];
      ek.ldw = split_ld(Ms);
    }
    if (want_var) {
      ek.K = Kb.as<char>() + ko[t] * ksz;
      ek.ldk = (long long)kld[t];
    }
    ek.part = Epart.as<double>() + eo[t];
    ek.part_ld = ns;
    if (f64) {
      f64_k.push_back({s->B.as<double>() + (size_t)ro * nd, m->X[t].as<double>(), nd, nd, ns, Ms,
                       nd, 0, ek});
    } else if (s->has_q) {
      // Species t's rows start a tile of the structure's slices.
      i8_k.push_back(kernel_contraction_i8(
          m, t, s->Bq.as<int8_t>() + i8_tiled_bytes(s->q_tile_row[t], kI8TileA, s->ldq),
          s->Bq_scale.as<double>() + ro, ns, nd, ek));
    } else {
      contract_fp32_rows(m, st, t, s->B.as<float>() + (size_t)ro * nd, ns, nd, Aq, Aq_scale, ek);
    }
    ctx->launches[ST_SGEMM]++;
  }
  if (!f64_k.empty() || !i8_k.empty()) {
    KScope timer(ctx, KT_SGEMM);
    gemm_f64_groups(st, EP_KERNEL, f64_k);
    gemm_i8_groups(st, i8_k);
  }
  ctx->mark_end(ST_SGEMM);

  // Gradient contraction G = W X_hat_s.
  ctx->mark_begin(ST_GGEMM);
  for (int t = 0; t < nos; t++) {
    int ns = s->n_by_type[t], Ms = m->M_by_type[t], ro = s->type_off[t];
    if (ns == 0) continue;
    void *Grow = (char *)G.as<char>() + (size_t)ro * nd * esz;
    if (Ms == 0) {
      FM_HIP(hipMemsetAsync(Grow, 0, (size_t)ns * nd * esz, st));
      continue;
    }
    EpArgs eg;
    eg.W = Grow;
    eg.ldw = nd;
    if (f64) {
      f64_g.push_back({W.as<double>() + wo[t], m->XT[t].as<double>(), (long long)kld[t], Ms, ns,
                       nd, Ms, 0, eg});
    } else {
      split_g.push_back(gradient_contraction(m, t, Wh.as<uint16_t>() + so[t],
                                             Wl.as<uint16_t>() + so[t], ns, nd, eg));
    }
    ctx->launches[ST_GGEMM]++;
  }
  if (!f64_g.empty() || !split_g.empty()) {
    KScope timer(ctx, KT_GGEMM);
    gemm_f64_groups(st, EP_STORE, f64_g);
    gemm_split_groups(st, split_g);
  }
  ctx->mark_end(ST_GGEMM);

  // Local energies from the energy partials (main stream).
  for_final_types(
      s,
      [&](int t, const double *&p, int &nt) {
        p = Epart.as<double>() + eo[t];
        nt = m->M_by_type[t] == 0 ? 0 : gemm_col_tiles(form, m->M_by_type[t]);
      },
      [&](const FinalArgs &a, int rows) {
        hipLaunchKernelGGL(k_energy_final, dim3((rows + 255) / 256), dim3(256), 0, st, a,
                           E_row.as<double>());
      });

  // Variance contraction Q = L_s^-1 K^T (FP64 in both forms) on the side
  // stream, after the kernel contraction that wrote k; it overlaps the
  // gradient contraction and the adjoint, and is joined before the results
  // are read back.
  // Against one stream: 108 atoms 259 and 275 us, 64 structures in FP64
  // 1,971 and 2,018, 32,000 atoms in the chosen form 3,321 and 3,369; on the larger
  // ones, whose stages fill the GPU by themselves, neither is faster (512
  // structures 10.9 ms, 262,144 atoms 41.8 to 41.9).
  // Joins the side stream into the main one when predict leaves this scope
  // by any path (declared after the buffers the side stream uses, so it runs
  // before they return to the pool).
  struct SideJoin {
    fm_context c;
    bool active = false;
    ~SideJoin() {
      if (active) (void)hipStreamWaitEvent(c->stream, c->ev_join, 0);
    }
  } join{ctx};
  if (want_var) {
    hipStream_t sd = ctx->side;
    FM_HIP(hipEventRecord(ctx->ev_fork, st));
    FM_HIP(hipStreamWaitEvent(sd, ctx->ev_fork, 0));
    ctx->mark_begin(ST_VAR, sd);
    std::vector<F64Gemm> full_q;  // species whose L block is not triangular
    for (int t = 0; t < nos; t++) {
      int ns = s->n_by_type[t], Ms = m->M_by_type[t];
      if (ns == 0 || Ms == 0 || m->L_rows[t] == 0) continue;
      EpArgs eq;
      eq.part = Qpart.as<double>() + qo[t];
      eq.part_ld = ns;
      std::vector<F64Gemm> &q = m->L_lower[t] ? f64_q : full_q;
      q.push_back({m->L[t].as<double>(), Kb.as<double>() + ko[t], Ms, (long long)kld[t],
                   m->L_rows[t], ns, Ms, m->L_lower[t], eq});
      ctx->launches[ST_VAR]++;
    }
    {
      KScope timer(ctx, KT_VAR, sd);
      gemm_f64_groups(sd, EP_SUMSQ, f64_q);
      gemm_f64_groups(sd, EP_SUMSQ, full_q);
    }
    for_final_types(
        s,
        [&](int t, const double *&p, int &nt) {
          p = Qpart.as<double>() + qo[t];
          nt = m->M_by_type[t] > 0 ? gemm_row_tiles(m->L_rows[t]) : 0;
        },
        [&](const FinalArgs &a, int rows) {
          hipLaunchKernelGGL(k_var_final, dim3((rows + 255) / 256), dim3(256), 0, sd, a,
                             s->norm.as<double>(), s->nn.as<double>(), sig2, m->power,
                             var_row.as<double>());
        });
    ctx->mark_end(ST_VAR, sd);
    FM_HIP(hipEventRecord(ctx->ev_join, sd));
    join.active = true;
  }

  // Adjoint bond forces and the deterministic gather.
  ctx->mark_begin(ST_ADJ);
  DevBuf fbond(pool, std::max<size_t>(1, (size_t)3 * s->n_bonds * esz));
  DevBuf vir(pool, std::max<size_t>(1, (size_t)6 * n * sizeof(double)));
  double *o = out.as<double>();
  if (n == 0) FM_HIP(hipMemsetAsync(o, 0, (size_t)n_out * sizeof(double), st));
  if (n > 0) {
    // FP64: G . B from the local energies (G . B = p |B| E, exact to
    // rounding). Split form: from the G and B rows, since G carries the
    // BF16-pair rounding of w that E does not, and the projection
    // G - (G . B_hat) B_hat must see the G it is applied to.
    launch_adjoint(s, G.as<void>(), nd, fbond.as<void>(), vir.as<double>(), 1, kEmptyThresh,
                   -1.0, f64 ? E_row.as<double>() : nullptr, m->power);
    gather_forces(s, f64, fbond, vir, E_row, o);
    ctx->launches[ST_ADJ] += 3;
  }
  FM_HIP(hipGetLastError());
  ctx->mark_end(ST_ADJ);
  if (join.active) {
    FM_HIP(hipStreamWaitEvent(st, ctx->ev_join, 0));
    join.active = false;
  }

  read_outputs(s, o, n_out, want_var ? var_row.as<double>() : nullptr, E_row.as<double>(),
               mean_efs, local_var, local_energy);
}

}  // namespace fm
