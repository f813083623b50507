// Periodic neighbour list on the device, bit-identical to the reference
// Structure::compute_neighbors (src/flare_pp/structure.cpp:52-118): same
// image vector ((d + s1 a) + s2 b) + s3 c, same test dist < cutoff && dist != 0,
// same order (j, s1, s2, s3). Built through a cell list: atoms are binned
// along the fractional axes (bin width >= cutoff perpendicular to each face),
// every candidate in the stencil is tested with the exact expression, images
// outside [-sweep, sweep]^3 are dropped (the reference loop never visits them)
// and each atom's list is sorted by its (j, s) key in LDS.
//
// This file is compiled with -ffp-contract=off so the FP64 expressions round
// exactly as written.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "fm_device.hpp"
#include "fm_gemm.hpp"
#include "fm_internal.hpp"

namespace fm {

// ---------------------------------------------------------------------------
// Scans
// ---------------------------------------------------------------------------
constexpr int kScanBlock = 1024;

template <typename V>
__device__ __forceinline__ V block_excl_scan(V v, V *sh, V &total) {
  // 1024 threads = 16 waves.
  int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  V x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    V y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  if (lane == 63) sh[wid] = x;
  __syncthreads();
  if (wid == 0) {
    V w = lane < 16 ? sh[lane] : 0;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
      V y = __shfl_up(w, off, 64);
      if (lane >= off) w += y;
    }
    if (lane < 16) sh[lane] = w;
  }
  __syncthreads();
  V base = wid ? sh[wid - 1] : 0;
  total = sh[15];
  __syncthreads();
  return base + x - v;
}

// One block: each thread scans kScanItems consecutive values.
constexpr int kScanItems = 8;
__global__ __launch_bounds__(kScanBlock) void k_scan_one(const int *in, int n, int *out,
                                                         int *host, const int *extra) {
  __shared__ int sh[16];
  int i0 = threadIdx.x * kScanItems, v[kScanItems], sum = 0, tot;
#pragma unroll
  for (int e = 0; e < kScanItems; e++) {
    v[e] = i0 + e < n ? in[i0 + e] : 0;
    sum += v[e];
  }
  int x = block_excl_scan(sum, sh, tot);
#pragma unroll
  for (int e = 0; e < kScanItems; e++) {
    if (i0 + e < n) out[i0 + e] = x;
    x += v[e];
  }
  if (threadIdx.x == 0) {
    out[n] = tot;
    if (host) host[0] = tot;
    if (host && extra) host[1] = *extra;
  }
}

__global__ __launch_bounds__(kScanBlock) void k_scan_block_sums(const int *in, int n, int *bsum) {
  __shared__ int sh[16];
  int i = blockIdx.x * kScanBlock + threadIdx.x, tot;
  block_excl_scan(i < n ? in[i] : 0, sh, tot);
  if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// Every block takes the sum of the blocks before it (bsum holds these sums if
// `scanned`, else the blocks' totals, which it sums), then scans its own values.
__global__ __launch_bounds__(kScanBlock) void k_scan_apply(const int *in, int n, const int *bsum,
                                                           int scanned, int *out, int *host,
                                                           const int *extra) {
  __shared__ int sh[16];
  int before = 0, base, tot;
  if (scanned) {
    base = bsum[blockIdx.x];
  } else {
    for (int b = threadIdx.x; b < blockIdx.x; b += kScanBlock) before += bsum[b];
    block_excl_scan(before, sh, base);  // base: the sum over all threads
  }
  int i = blockIdx.x * kScanBlock + threadIdx.x;
  int v = i < n ? in[i] : 0;
  int e = block_excl_scan(v, sh, tot);
  if (i < n) out[i] = base + e;
  if (i == n - 1) {
    out[n] = base + e + v;
    if (host) host[0] = base + e + v;
    if (host && extra) host[1] = *extra;
  }
}

// One launch up to 8,192 values (a block of 1,024 threads, 4 us). Then two, in
// which every block of the second sums the totals before it, a load per thread
// and 1,024 blocks. That grows with the square of the blocks, so from kScanSums
// blocks on the totals are scanned first, for two more launches. A structure of
// 3,000 atoms in an ever larger cell, without and with them: 65 and 67 us (a
// million bins), 88 and 89 (4), 193 and 156 (16), 925 and 472 (64), 28 and 3.6 ms
// (512).
constexpr int kScanSums = 4096;
void scan_exclusive(fm_context ctx, const int *in, int *out, int n, int *host,
                    const int *extra) {
  hipStream_t st = ctx->stream;
  if (n <= kScanBlock * kScanItems) {
    hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(kScanBlock), 0, st, in, n, out, host,
                       extra);
  } else {
    int nb = (n - 1) / kScanBlock + 1;
    DevBuf bsum(&ctx->pool, nb * sizeof(int)), boff;
    hipLaunchKernelGGL(k_scan_block_sums, dim3(nb), dim3(kScanBlock), 0, st, in, n,
                       bsum.as<int>());
    bool scanned = nb >= kScanSums;
    if (scanned) {
      boff.alloc(&ctx->pool, ((size_t)nb + 1) * sizeof(int));
      scan_exclusive(ctx, bsum.as<int>(), boff.as<int>(), nb);
    }
    hipLaunchKernelGGL(k_scan_apply, dim3(nb), dim3(kScanBlock), 0, st, in, n,
                       scanned ? boff.as<int>() : bsum.as<int>(), (int)scanned, out, host, extra);
  }
  FM_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Per-structure geometry (CellArgs, built on the host by fm_capi.hip). A
// structure object may hold a batch of structures: atoms of structure k are
// the contiguous range [atom_off[k], atom_off[k+1]) and only see each other.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void row3(const double *a, const double *B, double *o) {
  for (int k = 0; k < 3; k++) o[k] = (a[0] * B[k] + a[1] * B[3 + k]) + a[2] * B[6 + k];
}

// Zeros at the start of a build: the neighbour flags and maximum, the bin
// counts.
struct SetupWords {
  int flags, max_species, max_count;
};

struct SetupArgs {
  int n, n_struct, n_bins;
  const double *src_pos;
  const int *src_species;
  double *pos;
  int *species;
  const CellArgs *cas;
  const int *atom_off, *bin_off;
  int *atom_struct;
  double *wrapped;
  int *bin, *bstart, *order;
  SetupWords *words;
};

// Atom i: the structure it belongs to, its own copy of the caller's species
// and position (where those are in device memory), their checks (bad: bit 1
// non-finite position, bit 2 negative species), the wrapped position
// (structure.cpp:120-133) and its bin, which is returned.
__device__ __forceinline__ int setup_atom(const SetupArgs &a, int i, int &sp, int &bad) {
  sp = a.src_species[i];
  int k = 0;  // the structure with atom_off[k] <= i < atom_off[k + 1]
  if (a.n_struct > 1) {
    int lo = 0, hi = a.n_struct;
    while (hi - lo > 1) {
      int mid = (lo + hi) >> 1;
      if (a.atom_off[mid] <= i) lo = mid;
      else hi = mid;
    }
    k = lo;
  }
  a.atom_struct[i] = k;
  const CellArgs &ca = a.cas[k];
  double p[3] = {a.src_pos[3 * i], a.src_pos[3 * i + 1], a.src_pos[3 * i + 2]};
  if (a.pos != a.src_pos) {
    for (int q = 0; q < 3; q++) a.pos[3 * i + q] = p[q];
    a.species[i] = sp;
  }
  for (int q = 0; q < 3; q++)
    if (!isfinite(p[q])) bad |= 1;
  if (sp < 0) bad |= 2;
  double r1[3], fr[3], w1[3], w[3];
  row3(p, ca.ct, r1);
  row3(r1, ca.cdi, fr);
  for (int q = 0; q < 3; q++) fr[q] = fr[q] - floor(fr[q]);
  row3(fr, ca.cd, w1);
  row3(w1, ca.cti, w);
  for (int q = 0; q < 3; q++) a.wrapped[3 * i + q] = w[q];
  // Bin from the fractional coordinates of the wrapped position.
  row3(w, ca.ct, r1);
  row3(r1, ca.cdi, fr);
  int q3[3];
  for (int q = 0; q < 3; q++) {
    int b = (int)floor(fr[q] * ca.nb[q]);
    q3[q] = min(max(b, 0), ca.nb[q] - 1);
  }
  return a.bin_off[k] + (q3[0] * ca.nb[1] + q3[1]) * ca.nb[2] + q3[2];
}

// One atom per thread; bcount is zero on entry.
__global__ __launch_bounds__(256) void k_setup(SetupArgs a, int *bcount) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  int sp = -1, bad = 0;
  if (i < a.n) {
    int b = setup_atom(a, i, sp, bad);
    a.bin[i] = b;
    atomicAdd(&bcount[b], 1);
  }
  // One atomic per wave for the largest species.
  int mx = sp;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) mx = max(mx, __shfl_xor(mx, off, 64));
  if ((threadIdx.x & 63) == 0 && mx > 0) atomicMax(&a.words->max_species, mx);
  if (bad) atomicOr(&a.words->flags, bad);
}

// The whole of it (zeros, k_setup, the scan of the bins and k_bin_fill) in one
// workgroup, for up to kSmallAtoms atoms and as many bins as one scan takes:
// 5 us for 108 atoms and 13 us for 1,024 of them, where the four launches took
// 12 and 15 and the gaps between them. Creating a structure of 108, 2,048, 3,000
// and 4,096 atoms takes 52, 67, 77 and 86 us with it, 61, 72, 78 and 81 without.
constexpr int kSmallAtoms = 2048;
__global__ __launch_bounds__(kScanBlock) void k_setup_small(SetupArgs a, int *host_words) {
  __shared__ int cnt[kScanBlock * kScanItems], sh[16], flags, mx;
  for (int k = threadIdx.x; k < a.n_bins; k += kScanBlock) cnt[k] = 0;
  if (threadIdx.x == 0) flags = mx = 0;
  __syncthreads();
  int bin[kSmallAtoms / kScanBlock];
#pragma unroll
  for (int e = 0; e < kSmallAtoms / kScanBlock; e++) {
    int i = threadIdx.x + e * kScanBlock, sp = -1, bad = 0;
    if (i >= a.n) continue;
    bin[e] = a.bin[i] = setup_atom(a, i, sp, bad);
    atomicAdd(&cnt[bin[e]], 1);
    if (sp > 0) atomicMax(&mx, sp);
    if (bad) atomicOr(&flags, bad);
  }
  __syncthreads();
  int i0 = threadIdx.x * kScanItems, v[kScanItems], sum = 0, tot;
#pragma unroll
  for (int e = 0; e < kScanItems; e++) {
    v[e] = i0 + e < a.n_bins ? cnt[i0 + e] : 0;
    sum += v[e];
  }
  int x = block_excl_scan(sum, sh, tot);
#pragma unroll
  for (int e = 0; e < kScanItems; e++) {
    if (i0 + e < a.n_bins) a.bstart[i0 + e] = cnt[i0 + e] = x;
    x += v[e];
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < kSmallAtoms / kScanBlock; e++) {
    int i = threadIdx.x + e * kScanBlock;
    if (i < a.n) a.order[atomicAdd(&cnt[bin[e]], 1)] = i;
  }
  if (threadIdx.x == 0) {
    a.bstart[a.n_bins] = tot;
    a.words->max_count = 0;
    host_words[0] = flags;
    host_words[1] = mx;
  }
}

// Places each atom in its bin (any order within a bin: neighbours are sorted
// later), counting bcount down. Thread 0 passes the checks on to the host.
__global__ __launch_bounds__(256) void k_bin_fill(int n, const int *bin, const int *bstart,
                                                  int *bcount, int *order,
                                                  const SetupWords *words, int *host_words) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) {
    host_words[0] = words->flags;
    host_words[1] = words->max_species;
  }
  if (i < n) {
    int b = bin[i];
    order[bstart[b] + atomicAdd(&bcount[b], -1) - 1] = i;
  }
}

__device__ __forceinline__ int floor_div(int a, int b) {
  int q = a / b;
  if ((a % b != 0) && ((a < 0) != (b < 0))) q--;
  return q;
}

// structure.cpp:72-75.
__device__ __forceinline__ double image_dist(const double *wi, const double *wj,
                                             const CellArgs &ca, int s1, int s2, int s3,
                                             double *im) {
  for (int k = 0; k < 3; k++) {
    double d = wj[k] - wi[k];
    im[k] = ((d + (double)s1 * ca.cell[k]) + (double)s2 * ca.cell[3 + k]) +
            (double)s3 * ca.cell[6 + k];
  }
  return sqrt(im[0] * im[0] + im[1] * im[1] + im[2] * im[2]);
}

__device__ __forceinline__ long long nbr_key(int j, int s1, int s2, int s3, int sw) {
  int span = 2 * sw + 1;
  long long key = ((long long)j * span + (s1 + sw)) * span;
  return (key + (s2 + sw)) * span + (s3 + sw);
}

__device__ __forceinline__ void nbr_unkey(long long key, int sw, int &j, int &s1, int &s2,
                                          int &s3) {
  int span = 2 * sw + 1;
  s3 = (int)(key % span) - sw;
  key /= span;
  s2 = (int)(key % span) - sw;
  key /= span;
  s1 = (int)(key % span) - sw;
  j = (int)(key / span);
}

// One wavefront per atom. kFill = false counts the neighbours; kFill = true
// collects the keys in LDS, sorts them and writes the list. The stencil's
// bins (up to kStencilCap per pass) are laid out in LDS with a prefix sum of
// their sizes, so the wave's 64 lanes take consecutive candidates across
// bins instead of one bin at a time.
// Keys per atom held in LDS: lists of up to kNbrCapSmall (every common
// setting) use the small-LDS instance (seven workgroups per CU instead of
// two), up to kNbrCap the large one, longer lists the fallback below.
constexpr int kNbrCapSmall = 512;
constexpr int kNbrCap = 2048;
constexpr int kNbrWaves = 4;
constexpr int kStencilCap = 128;

// With kFill and `slots` set (one pass instead of count + fill): each atom's
// count goes to count[i] and, when it fits CAP, its sorted keys to
// slots[i CAP, ...), for k_neighbors_emit to write at the scanned offsets.
template <bool kFill, int CAP = kNbrCap>
__global__ __launch_bounds__(64 * kNbrWaves) void k_neighbors(
    int n, const double *wrapped, const int *bin_of, const int *bstart, const int *order,
    const int *species, const CellArgs *cas, const int *atom_struct, const int *bin_off,
    int *count, const int *cum, int *sidx, int *nspec, double *rel, int *max_count,
    long long *slots = nullptr) {
  __shared__ long long keys[kNbrWaves][kFill ? CAP : 1];
  __shared__ int s_off[kNbrWaves][kStencilCap + 1];
  __shared__ int s_p0[kNbrWaves][kStencilCap];
  __shared__ int s_img[kNbrWaves][kStencilCap];
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int i = blockIdx.x * kNbrWaves + w;
  if (i >= n) return;
  int st = atom_struct[i];
  const CellArgs &ca = cas[st];
  int boff = bin_off[st];
  double wi[3] = {wrapped[3 * i], wrapped[3 * i + 1], wrapped[3 * i + 2]};
  int b = bin_of[i] - boff;
  int bx = b / (ca.nb[1] * ca.nb[2]), by = (b / ca.nb[2]) % ca.nb[1], bz = b % ca.nb[2];
  int sw = ca.sweep, span = 2 * sw + 1;
  int e0 = 2 * ca.K[0] + 1, e1 = 2 * ca.K[1] + 1, e2 = 2 * ca.K[2] + 1;
  int nst = e0 * e1 * e2;
  int found = 0;
  for (int sbase = 0; sbase < nst; sbase += kStencilCap) {
    int scount = min(kStencilCap, nst - sbase);
    if (sbase > 0) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    for (int e = lane; e < scount; e += 64) {
      int sidx_ = sbase + e;
      int o2 = sidx_ % e2 - ca.K[2], o1 = (sidx_ / e2) % e1 - ca.K[1],
          o0 = sidx_ / (e1 * e2) - ca.K[0];
      int t0 = bx + o0, s1 = floor_div(t0, ca.nb[0]), b0 = t0 - s1 * ca.nb[0];
      int t1 = by + o1, s2 = floor_div(t1, ca.nb[1]), b1 = t1 - s2 * ca.nb[1];
      int t2 = bz + o2, s3 = floor_div(t2, ca.nb[2]), b2 = t2 - s3 * ca.nb[2];
      bool valid = s1 >= -sw && s1 <= sw && s2 >= -sw && s2 <= sw && s3 >= -sw && s3 <= sw;
      int size = 0, p0 = 0, img = 0;
      if (valid) {
        int q = boff + (b0 * ca.nb[1] + b1) * ca.nb[2] + b2;
        p0 = bstart[q];
        size = bstart[q + 1] - p0;
        img = ((s1 + sw) * span + (s2 + sw)) * span + (s3 + sw);
      }
      s_p0[w][e] = p0;
      s_img[w][e] = img;
      s_off[w][e + 1] = size;
    }
    if (lane == 0) s_off[w][0] = 0;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // Inclusive prefix sum of the sizes, 64 entries at a time.
    int carry = 0;
    for (int cb = 0; cb < scount; cb += 64) {
      int e = cb + lane;
      int v = e < scount ? s_off[w][e + 1] : 0;
      for (int d = 1; d < 64; d <<= 1) {
        int u = __shfl_up(v, d, 64);
        if (lane >= d) v += u;
      }
      if (e < scount) s_off[w][e + 1] = v + carry;
      carry += __shfl(v, 63, 64);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    int total = s_off[w][scount];
    for (int c0 = 0; c0 < total; c0 += 64) {
      int t = c0 + lane;
      bool ok = false;
      int j = 0, s1 = 0, s2 = 0, s3 = 0;
      if (t < total) {
        // The bin holding candidate t: s_off[lo] <= t < s_off[lo + 1].
        int lo = 0, hi = scount;
        while (hi - lo > 1) {
          int mid = (lo + hi) >> 1;
          if (s_off[w][mid] <= t) lo = mid;
          else hi = mid;
        }
        j = order[s_p0[w][lo] + (t - s_off[w][lo])];
        int img = s_img[w][lo];
        s3 = img % span - sw;
        s2 = (img / span) % span - sw;
        s1 = img / (span * span) - sw;
        double wj[3] = {wrapped[3 * j], wrapped[3 * j + 1], wrapped[3 * j + 2]};
        double im[3];
        double dist = image_dist(wi, wj, ca, s1, s2, s3, im);
        ok = (dist < ca.cutoff) && (dist != 0);
      }
      unsigned long long mask = __ballot(ok);
      if (kFill && ok) {
        int pre = __popcll(mask & ((1ull << lane) - 1ull));
        int slot = found + pre;
        if (slot < CAP) keys[w][slot] = nbr_key(j, s1, s2, s3, sw);
      }
      found += __popcll(mask);
    }
  }
  if (!kFill || slots) {
    if (lane == 0) {
      count[i] = found;
      // Only lists longer than the small LDS capacity need another instance.
      if (found > kNbrCapSmall) atomicMax(max_count, found);
    }
    if (!kFill || found > CAP) return;
  }
  // Bitonic sort of the keys (padded to a power of two with the largest key).
  int np2 = 1;
  while (np2 < found) np2 <<= 1;
  for (int t = found + lane; t < np2; t += 64) keys[w][t] = 0x7fffffffffffffffLL;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  for (int k = 2; k <= np2; k <<= 1) {
    for (int jj = k >> 1; jj > 0; jj >>= 1) {
      for (int t = lane; t < np2; t += 64) {
        int partner = t ^ jj;
        if (partner > t) {
          long long a = keys[w][t], c = keys[w][partner];
          bool up = (t & k) == 0;
          if ((a > c) == up) {
            keys[w][t] = c;
            keys[w][partner] = a;
          }
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
  if (slots) {
    for (int t = lane; t < found; t += 64) slots[(size_t)i * CAP + t] = keys[w][t];
    return;
  }
  int base = cum[i];
  for (int t = lane; t < found; t += 64) {
    int j, s1, s2, s3;
    nbr_unkey(keys[w][t], sw, j, s1, s2, s3);
    double wj[3] = {wrapped[3 * j], wrapped[3 * j + 1], wrapped[3 * j + 2]};
    double im[3];
    double dist = image_dist(wi, wj, ca, s1, s2, s3, im);
    int o = base + t;
    sidx[o] = j;
    nspec[o] = species[j];
    rel[4 * (size_t)o] = dist;
    rel[4 * (size_t)o + 1] = im[0];
    rel[4 * (size_t)o + 2] = im[1];
    rel[4 * (size_t)o + 3] = im[2];
  }
}

// The lists parked by the one-pass k_neighbors: one wavefront per atom writes
// its sorted keys at cum[i] with the same image expression as the fill.
__global__ __launch_bounds__(64 * kNbrWaves) void k_neighbors_emit(
    int n, const double *wrapped, const int *species, const CellArgs *cas,
    const int *atom_struct, const int *count, const int *cum, const long long *slots, int cap,
    int *sidx, int *nspec, double *rel) {
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int i = blockIdx.x * kNbrWaves + w;
  if (i >= n) return;
  const CellArgs &ca = cas[atom_struct[i]];
  int sw = ca.sweep, cnt = count[i], base = cum[i];
  double wi[3] = {wrapped[3 * i], wrapped[3 * i + 1], wrapped[3 * i + 2]};
  for (int t = lane; t < cnt; t += 64) {
    int j, s1, s2, s3;
    nbr_unkey(slots[(size_t)i * cap + t], sw, j, s1, s2, s3);
    double wj[3] = {wrapped[3 * j], wrapped[3 * j + 1], wrapped[3 * j + 2]};
    double im[3];
    double dist = image_dist(wi, wj, ca, s1, s2, s3, im);
    int o = base + t;
    sidx[o] = j;
    nspec[o] = species[j];
    rel[4 * (size_t)o] = dist;
    rel[4 * (size_t)o + 1] = im[0];
    rel[4 * (size_t)o + 2] = im[1];
    rel[4 * (size_t)o + 3] = im[2];
  }
}

// Fallback for atoms with more than kNbrCap neighbours (tiny cells with a
// large sweep): one thread per atom, keys sorted in place in global memory.
__global__ void k_neighbors_big(int n, const double *wrapped, const int *bin_of,
                                const int *bstart, const int *order, const int *species,
                                const CellArgs *cas, const int *atom_struct, const int *bin_off,
                                const int *cum, long long *scratch, int *sidx, int *nspec,
                                double *rel) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int st = atom_struct[i];
  const CellArgs &ca = cas[st];
  int boff = bin_off[st];
  double wi[3] = {wrapped[3 * i], wrapped[3 * i + 1], wrapped[3 * i + 2]};
  int b = bin_of[i] - boff;
  int bx = b / (ca.nb[1] * ca.nb[2]), by = (b / ca.nb[2]) % ca.nb[1], bz = b % ca.nb[2];
  int sw = ca.sweep;
  long long *keys = scratch + cum[i];
  int cnt = cum[i + 1] - cum[i];
  int found = 0;
  for (int o0 = -ca.K[0]; o0 <= ca.K[0]; o0++) {
    int t0 = bx + o0, s1 = floor_div(t0, ca.nb[0]), b0 = t0 - s1 * ca.nb[0];
    if (s1 < -sw || s1 > sw) continue;
    for (int o1 = -ca.K[1]; o1 <= ca.K[1]; o1++) {
      int t1 = by + o1, s2 = floor_div(t1, ca.nb[1]), b1 = t1 - s2 * ca.nb[1];
      if (s2 < -sw || s2 > sw) continue;
      for (int o2 = -ca.K[2]; o2 <= ca.K[2]; o2++) {
        int t2 = bz + o2, s3 = floor_div(t2, ca.nb[2]), b2 = t2 - s3 * ca.nb[2];
        if (s3 < -sw || s3 > sw) continue;
        int q = boff + (b0 * ca.nb[1] + b1) * ca.nb[2] + b2;
        for (int p = bstart[q]; p < bstart[q + 1]; p++) {
          int j = order[p];
          double wj[3] = {wrapped[3 * j], wrapped[3 * j + 1], wrapped[3 * j + 2]};
          double im[3];
          double dist = image_dist(wi, wj, ca, s1, s2, s3, im);
          if ((dist < ca.cutoff) && (dist != 0) && found < cnt)
            keys[found++] = nbr_key(j, s1, s2, s3, sw);
        }
      }
    }
  }
  for (int a = 1; a < found; a++) {  // insertion sort
    long long v = keys[a];
    int c = a - 1;
    while (c >= 0 && keys[c] > v) {
      keys[c + 1] = keys[c];
      c--;
    }
    keys[c + 1] = v;
  }
  for (int t = 0; t < found; t++) {
    int j, s1, s2, s3;
    nbr_unkey(keys[t], sw, j, s1, s2, s3);
    double wj[3] = {wrapped[3 * j], wrapped[3 * j + 1], wrapped[3 * j + 2]};
    double im[3];
    double dist = image_dist(wi, wj, ca, s1, s2, s3, im);
    int o = cum[i] + t;
    sidx[o] = j;
    nspec[o] = species[j];
    rel[4 * (size_t)o] = dist;
    rel[4 * (size_t)o + 1] = im[0];
    rel[4 * (size_t)o + 2] = im[1];
    rel[4 * (size_t)o + 3] = im[2];
  }
}

void build_neighbors(fm_structure s, const int *species_dev, const double *positions_dev) {
  fm_context ctx = s->ctx;
  hipStream_t st = ctx->stream;
  int n = s->n;
  Pool *pool = &ctx->pool;
  int ncell = s->n_bins;
  const CellArgs *cas = s->d_cellargs.as<CellArgs>();
  const int *ast = s->atom_struct.as<int>();
  const int *boffp = s->d_bin_off.as<int>();
  s->wrapped.alloc(pool, 3 * (size_t)n * sizeof(double));
  s->count.alloc(pool, (size_t)n * sizeof(int));
  s->cumulative.alloc(pool, ((size_t)n + 1) * sizeof(int));
  DevBuf bin(pool, (size_t)n * sizeof(int));
  DevBuf zeros(pool, sizeof(SetupWords) + (size_t)ncell * sizeof(int));
  DevBuf bstart(pool, ((size_t)ncell + 1) * sizeof(int));
  DevBuf order(pool, (size_t)n * sizeof(int));
  SetupWords *words = zeros.as<SetupWords>();
  int *bcount = reinterpret_cast<int *>(words + 1), *maxc = &words->max_count;
  int *hw = ctx->pinned_dev;
  int tpb = 256, nblk = (n + tpb - 1) / tpb;
  SetupArgs sa{n,
               s->n_struct,
               ncell,
               positions_dev ? positions_dev : s->positions.as<double>(),
               species_dev ? species_dev : s->species.as<int>(),
               s->positions.as<double>(),
               s->species.as<int>(),
               cas,
               s->d_atom_off.as<int>(),
               boffp,
               s->atom_struct.as<int>(),
               s->wrapped.as<double>(),
               bin.as<int>(),
               bstart.as<int>(),
               order.as<int>(),
               words};
  if (n <= kSmallAtoms && ncell <= kScanBlock * kScanItems) {
    hipLaunchKernelGGL(k_setup_small, dim3(1), dim3(kScanBlock), 0, st, sa, hw);
  } else {
    FM_HIP(hipMemsetAsync(zeros.as<void>(), 0, sizeof(SetupWords) + (size_t)ncell * sizeof(int),
                          st));
    hipLaunchKernelGGL(k_setup, dim3(nblk), dim3(tpb), 0, st, sa, bcount);
    scan_exclusive(ctx, bcount, bstart.as<int>(), ncell);
    hipLaunchKernelGGL(k_bin_fill, dim3(nblk), dim3(tpb), 0, st, n, bin.as<int>(),
                       bstart.as<int>(), bcount, order.as<int>(), words, hw);
  }
  int wblk = (n + kNbrWaves - 1) / kNbrWaves;
  // One pass over the candidates that also parks each atom's sorted keys
  // (kNbrCapSmall per atom, while that area stays within 16 GB); else a
  // counting pass first.
  bool one_pass = (size_t)n * kNbrCapSmall * sizeof(long long) <= (16ull << 30);
  DevBuf slots;
  if (one_pass) {
    slots.alloc(pool, std::max<size_t>(1, (size_t)n * kNbrCapSmall * sizeof(long long)));
    hipLaunchKernelGGL((k_neighbors<true, kNbrCapSmall>), dim3(wblk), dim3(64 * kNbrWaves), 0, st,
                       n, s->wrapped.as<double>(), bin.as<int>(), bstart.as<int>(),
                       order.as<int>(), s->species.as<int>(), cas, ast, boffp,
                       s->count.as<int>(), nullptr, nullptr, nullptr, nullptr, maxc,
                       slots.as<long long>());
  } else {
    hipLaunchKernelGGL(k_neighbors<false>, dim3(wblk), dim3(64 * kNbrWaves), 0, st, n,
                       s->wrapped.as<double>(), bin.as<int>(), bstart.as<int>(), order.as<int>(),
                       s->species.as<int>(), cas, ast, boffp, s->count.as<int>(), nullptr,
                       nullptr, nullptr, nullptr, maxc);
  }
  FM_HIP(hipGetLastError());
  // Total and largest count to pinned words 2 and 3, then one synchronisation.
  scan_exclusive(ctx, s->count.as<int>(), s->cumulative.as<int>(), n, hw + 2, maxc);
  FM_HIP(hipStreamSynchronize(st));
  int total = ctx->pinned[2], max_count = ctx->pinned[3];
  s->n_nb = total;
  s->sidx.alloc(pool, std::max<size_t>(1, (size_t)total * sizeof(int)));
  s->nspecies.alloc(pool, std::max<size_t>(1, (size_t)total * sizeof(int)));
  s->rel.alloc(pool, std::max<size_t>(1, 4 * (size_t)total * sizeof(double)));
  if (max_count <= kNbrCapSmall && one_pass) {
    hipLaunchKernelGGL(k_neighbors_emit, dim3(wblk), dim3(64 * kNbrWaves), 0, st, n,
                       s->wrapped.as<double>(), s->species.as<int>(), cas, ast,
                       s->count.as<int>(), s->cumulative.as<int>(), slots.as<long long>(),
                       kNbrCapSmall, s->sidx.as<int>(), s->nspecies.as<int>(),
                       s->rel.as<double>());
  } else if (max_count <= kNbrCapSmall) {
    hipLaunchKernelGGL((k_neighbors<true, kNbrCapSmall>), dim3(wblk), dim3(64 * kNbrWaves), 0, st,
                       n, s->wrapped.as<double>(), bin.as<int>(), bstart.as<int>(),
                       order.as<int>(), s->species.as<int>(), cas, ast, boffp, nullptr,
                       s->cumulative.as<int>(), s->sidx.as<int>(), s->nspecies.as<int>(),
                       s->rel.as<double>(), nullptr);
  } else if (max_count <= kNbrCap) {
    hipLaunchKernelGGL((k_neighbors<true, kNbrCap>), dim3(wblk), dim3(64 * kNbrWaves), 0, st, n,
                       s->wrapped.as<double>(), bin.as<int>(), bstart.as<int>(), order.as<int>(),
                       s->species.as<int>(), cas, ast, boffp, nullptr, s->cumulative.as<int>(),
                       s->sidx.as<int>(), s->nspecies.as<int>(), s->rel.as<double>(), nullptr);
  } else {
    DevBuf scratch(pool, (size_t)total * sizeof(long long));
    hipLaunchKernelGGL(k_neighbors_big, dim3(nblk), dim3(tpb), 0, st, n, s->wrapped.as<double>(),
                       bin.as<int>(), bstart.as<int>(), order.as<int>(), s->species.as<int>(), cas,
                       ast, boffp, s->cumulative.as<int>(), scratch.as<long long>(),
                       s->sidx.as<int>(), s->nspecies.as<int>(), s->rel.as<double>());
    FM_HIP(hipStreamSynchronize(st));
  }
  FM_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Descriptor bond list (b2.cpp:262-304: r <= rc(s_i, s_j), list order kept),
// its transpose by neighbour atom (for the deterministic force gather), and
// the species-sorted row of each atom (b2.cpp:148-176).
// ---------------------------------------------------------------------------
// Bonds are the neighbours within the species-pair cutoff, kept in neighbour
// order. One wave per atom walks its neighbour list 64 entries at a time; a
// ballot gives each kept entry its place.
// Cutoffs passed by value for up to four species, written to memory by the
// first kernel that has them.
struct CutoffArgs {
  double c[16];
  int n;  // 0: in memory already
};

__global__ __launch_bounds__(256) void k_bond_count(int n, const int *species, const int *cum,
                                                    const int *nspec, const double *rel,
                                                    CutoffArgs cut, double *cutoffs, int nos,
                                                    int *bcount, int *in_count) {
  int lane = threadIdx.x & 63;
  int i = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (blockIdx.x == 0 && threadIdx.x < cut.n) cutoffs[threadIdx.x] = cut.c[threadIdx.x];
  const double *rc = cut.n ? cut.c : cutoffs;
  if (i >= n) return;
  int si = species[i], c = 0;
  for (int q0 = cum[i]; q0 < cum[i + 1]; q0 += 64) {
    int q = q0 + lane;
    bool keep = q < cum[i + 1] && rel[4 * (size_t)q] <= rc[si * nos + nspec[q]];
    c += __popcll(__ballot(keep));
  }
  if (lane == 0) {
    bcount[i] = c;
    in_count[i] = 0;
  }
}

__global__ __launch_bounds__(256) void k_bond_fill(int n, const int *species, const int *cum,
                                                   const int *nspec, const double *rel,
                                                   const double *cutoffs, int nos,
                                                   const int *boff, const int *sidx, int *bond_q,
                                                   int *in_count, int *in_slot,
                                                   const int *bonds_by_type, int *host_by_type) {
  int lane = threadIdx.x & 63;
  int i = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (bonds_by_type && blockIdx.x == 0 && threadIdx.x < nos)
    host_by_type[threadIdx.x] = bonds_by_type[threadIdx.x];
  if (i >= n) return;
  int si = species[i], o = boff[i];
  unsigned long long below = (1ull << lane) - 1ull;
  for (int q0 = cum[i]; q0 < cum[i + 1]; q0 += 64) {
    int q = q0 + lane;
    bool keep = q < cum[i + 1] && rel[4 * (size_t)q] <= cutoffs[si * nos + nspec[q]];
    unsigned long long m = __ballot(keep);
    if (keep) {
      int b = o + __popcll(m & below);
      bond_q[b] = q;
      in_slot[b] = atomicAdd(&in_count[sidx[q]], 1);
    }
    o += __popcll(m);
  }
}

// Incoming bonds of each atom in the order in which the fill counted them (the
// launch covers all neighbours; the bonds are the first bond_off[n] of them).
// With in_count (up to one scan of atoms) every workgroup scans the counts itself
// and the first one writes in_off, for a launch less.
__global__ __launch_bounds__(kScanBlock) void k_in_fill(int n, const int *bond_off,
                                                        const int *bond_q, const int *sidx,
                                                        const int *in_count, int *in_off,
                                                        const int *in_slot, int *in_bond) {
  __shared__ int off[kScanBlock * kScanItems], sh[16];
  if (in_count) {
    int i0 = threadIdx.x * kScanItems, v[kScanItems], sum = 0, tot;
#pragma unroll
    for (int e = 0; e < kScanItems; e++) {
      v[e] = i0 + e < n ? in_count[i0 + e] : 0;
      sum += v[e];
    }
    int x = block_excl_scan(sum, sh, tot);
#pragma unroll
    for (int e = 0; e < kScanItems; e++) {
      off[i0 + e] = x;
      if (blockIdx.x == 0 && i0 + e < n) in_off[i0 + e] = x;
      x += v[e];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) in_off[n] = tot;
    __syncthreads();
  }
  int b = blockIdx.x * kScanBlock + threadIdx.x;
  if (b >= bond_off[n]) return;
  int j = sidx[bond_q[b]];
  in_bond[(in_count ? off[j] : in_off[j]) + in_slot[b]] = b;
}

// Incoming bonds of atom j in ascending bond order (so the force gather sums
// them in a fixed order): one wave per atom; each lane takes elements of the
// unordered list and writes each to its rank, the number of smaller bond ids
// in the list (ids are distinct). The list is read with wave-uniform loads.
__global__ __launch_bounds__(256) void k_in_rank(int n, const int *in_off, const int *unordered,
                                                 int *in_bond) {
  int lane = threadIdx.x & 63;
  int j = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (j >= n) return;
  int a0 = in_off[j], cnt = in_off[j + 1] - a0;
  const int *u = unordered + a0;
  for (int e = lane; e < cnt; e += 64) {
    int v = u[e], r = 0;
    for (int k = 0; k < cnt; k++) r += u[k] < v;
    in_bond[a0 + r] = v;
  }
}

// Species-sorted rows (b2.cpp:148-176; atom order kept within a species).
constexpr int kRowBlock = 1024;

// Atoms of each species per block of 1,024, species-major.
__global__ __launch_bounds__(kRowBlock) void k_species_count(int n, const int *species, int nos,
                                                             int *hist) {
  extern __shared__ int cnt[];
  for (int t = threadIdx.x; t < nos; t += kRowBlock) cnt[t] = 0;
  __syncthreads();
  int i = blockIdx.x * kRowBlock + threadIdx.x;
  int sp = i < n ? species[i] : -1;
  for (int t = 0; t < nos; t++) {
    unsigned long long m = __ballot(sp == t);
    if ((threadIdx.x & 63) == 0 && m) atomicAdd(&cnt[t], (int)__popcll(m));
  }
  __syncthreads();
  for (int t = threadIdx.x; t < nos; t += kRowBlock) hist[(size_t)t * gridDim.x + blockIdx.x] = cnt[t];
}

// Row of each atom: the rows of the lower species and of the blocks before
// (`off`, the scan of the counts above), then the atom's rank in its block. Block 0
// also writes the species' atom counts to the host, the slice-row shift of each
// species (its rows start a tile of `tile` slice rows) and zeros for the bond
// counts by species.
__global__ __launch_bounds__(kRowBlock) void k_species_rows(int n, const int *species, int nos,
                                                            const int *off, int *row_of_atom,
                                                            int *atom_of_row, int *host_by_type,
                                                            int tile, int *shift,
                                                            int *bonds_by_type) {
  extern __shared__ int wc[];  // [16 waves][nos]
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nb = gridDim.x;
  int i = blockIdx.x * kRowBlock + threadIdx.x;
  int sp = i < n ? species[i] : -1;
  int rank = 0;
  for (int t = 0; t < nos; t++) {
    unsigned long long m = __ballot(sp == t);
    if (sp == t) rank = __popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) wc[w * nos + t] = __popcll(m);
  }
  __syncthreads();
  if (sp >= 0) {
    int r = off[(size_t)sp * nb + blockIdx.x] + rank;
    for (int v = 0; v < w; v++) r += wc[v * nos + sp];
    row_of_atom[i] = r;
    atom_of_row[r] = i;
  }
  if (blockIdx.x == 0) {
    auto first = [&](int t) { return off[(size_t)t * nb]; };  // first(nos) = n
    for (int t = threadIdx.x; t < nos; t += kRowBlock) {
      host_by_type[t] = first(t + 1) - first(t);
      bonds_by_type[t] = 0;
    }
    if (threadIdx.x == 0) {
      int rows = 0;
      for (int t = 0; t < nos; t++) {
        shift[t] = rows - first(t);
        rows += (first(t + 1) - first(t) + tile - 1) / tile * tile;
      }
    }
  }
}

// Bonds by the species of their centre (b2.cpp:106-112), summed per block.
__global__ __launch_bounds__(256) void k_bonds_by_type(int n, const int *species,
                                                       const int *bcount, int nos,
                                                       int *bonds_by_type) {
  extern __shared__ int cnt[];
  for (int t = threadIdx.x; t < nos; t += blockDim.x) cnt[t] = 0;
  __syncthreads();
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    atomicAdd(&cnt[species[i]], bcount[i]);
  __syncthreads();
  for (int t = threadIdx.x; t < nos; t += blockDim.x)
    if (cnt[t]) atomicAdd(&bonds_by_type[t], cnt[t]);
}

// Species rows, bonds by species and bond offsets in one workgroup, for as many
// atoms as one scan takes (eight consecutive ones per thread): a scan of (atoms,
// bonds) per species, then one of the bonds. 5 us for 108 atoms, 7 us for 1,024
// and 20 us for 8,190, where three to five launches took 10 to 20 and the gaps
// between them. A structure and its descriptors, 108, 2,048 and 8,192 atoms: 105,
// 130 and 190 us with it, 112, 136 and 194 without; more atoms do not fit a scan.
__global__ __launch_bounds__(kScanBlock) void k_rows_bonds(int n, const int *species, int nos,
                                                           const int *bcount, int *row_of_atom,
                                                           int *atom_of_row, int *bond_off,
                                                           int tile, int *shift,
                                                           int *host_by_type, int *host_bonds,
                                                           int *host_total) {
  __shared__ long long sh[16];
  __shared__ int sh1[16];
  int i0 = threadIdx.x * kScanItems, sp[kScanItems], bc[kScanItems], sum = 0, tot;
#pragma unroll
  for (int e = 0; e < kScanItems; e++) {
    bool in = i0 + e < n;
    sp[e] = in ? species[i0 + e] : -1;
    bc[e] = in ? bcount[i0 + e] : 0;
    sum += bc[e];
  }
  int first = 0, slice_rows = 0;
  for (int t = 0; t < nos; t++) {
    long long v = 0, all;
#pragma unroll
    for (int e = 0; e < kScanItems; e++)
      if (sp[e] == t) v += (1ll << 32) + bc[e];
    int r = first + (int)(block_excl_scan(v, sh, all) >> 32);
#pragma unroll
    for (int e = 0; e < kScanItems; e++)
      if (sp[e] == t) {
        row_of_atom[i0 + e] = r;
        atom_of_row[r++] = i0 + e;
      }
    int atoms = (int)(all >> 32);
    if (threadIdx.x == 0) {
      host_by_type[t] = atoms;
      host_bonds[t] = (int)all;
      shift[t] = slice_rows - first;
    }
    first += atoms;
    slice_rows += (atoms + tile - 1) / tile * tile;
  }
  int x = block_excl_scan(sum, sh1, tot);
#pragma unroll
  for (int e = 0; e < kScanItems; e++) {
    if (i0 + e < n) bond_off[i0 + e] = x;
    x += bc[e];
  }
  if (threadIdx.x == 0) {
    bond_off[n] = tot;
    host_total[0] = tot;
  }
}

// Pinned words of a bond build: the bond total, then atoms and bonds by species.
constexpr int kWordBonds = 4, kWordTypes = 8;
constexpr int kMaxSpecies = 255;
static_assert(kWordTypes + 2 * kMaxSpecies <= fm_context_s::kPinnedWords, "pinned words");

void build_bonds(fm_structure s) {
  fm_context ctx = s->ctx;
  hipStream_t st = ctx->stream;
  Pool *pool = &ctx->pool;
  int n = s->n, nos = s->nos, tpb = 256;
  FM_CHECK(nos <= kMaxSpecies, FM_ERR_INVALID, "too many species");
  int *hw = ctx->pinned_dev;
  int *host_types = hw + kWordTypes, *host_bonds = hw + kWordTypes + nos;
  int nc = nos * nos;
  s->d_cutoffs.alloc(pool, nc * sizeof(double));
  CutoffArgs cut{};
  if (nc <= 16) {
    std::copy(s->cutoffs.begin(), s->cutoffs.end(), cut.c);
    cut.n = nc;
  } else {
    FM_HIP(hipMemcpyAsync(s->d_cutoffs.as<double>(), s->cutoffs.data(), nc * sizeof(double),
                          hipMemcpyHostToDevice, st));
  }
  s->row_of_atom.alloc(pool, (size_t)n * sizeof(int));
  s->atom_of_row.alloc(pool, (size_t)n * sizeof(int));
  s->q_shift.alloc(pool, nos * sizeof(int));
  s->bond_off.alloc(pool, ((size_t)n + 1) * sizeof(int));
  DevBuf by_type(pool, nos * sizeof(int));
  DevBuf bcount(pool, (size_t)n * sizeof(int)), in_count(pool, (size_t)n * sizeof(int));
  hipLaunchKernelGGL(k_bond_count, dim3((n + 3) / 4), dim3(256), 0, st, n, s->species.as<int>(),
                     s->cumulative.as<int>(), s->nspecies.as<int>(), s->rel.as<double>(), cut,
                     s->d_cutoffs.as<double>(), nos, bcount.as<int>(), in_count.as<int>());
  bool one_block = n <= kScanBlock * kScanItems;
  DevBuf hist, off;
  if (one_block) {
    hipLaunchKernelGGL(k_rows_bonds, dim3(1), dim3(kScanBlock), 0, st, n, s->species.as<int>(),
                       nos, bcount.as<int>(), s->row_of_atom.as<int>(),
                       s->atom_of_row.as<int>(), s->bond_off.as<int>(), kI8TileA,
                       s->q_shift.as<int>(), host_types, host_bonds, hw + kWordBonds);
  } else {
    int nb = (n + kRowBlock - 1) / kRowBlock;
    hist.alloc(pool, (size_t)nos * nb * sizeof(int));
    off.alloc(pool, ((size_t)nos * nb + 1) * sizeof(int));
    hipLaunchKernelGGL(k_species_count, dim3(nb), dim3(kRowBlock), nos * sizeof(int), st, n,
                       s->species.as<int>(), nos, hist.as<int>());
    scan_exclusive(ctx, hist.as<int>(), off.as<int>(), nos * nb);
    hipLaunchKernelGGL(k_species_rows, dim3(nb), dim3(kRowBlock), 16 * nos * sizeof(int),
                       st, n, s->species.as<int>(), nos, off.as<int>(), s->row_of_atom.as<int>(),
                       s->atom_of_row.as<int>(), host_types, kI8TileA, s->q_shift.as<int>(),
                       by_type.as<int>());
    hipLaunchKernelGGL(k_bonds_by_type, dim3(std::min(64, (n + 255) / 256)), dim3(256),
                       nos * sizeof(int), st, n, s->species.as<int>(), bcount.as<int>(), nos,
                       by_type.as<int>());
    scan_exclusive(ctx, bcount.as<int>(), s->bond_off.as<int>(), n, hw + kWordBonds);
  }
  // Bond arrays hold every neighbour, so nothing waits for the bond total.
  size_t cap = std::max<size_t>(1, (size_t)s->n_nb);
  s->bond_q.alloc(pool, cap * sizeof(int));
  DevBuf in_slot(pool, cap * sizeof(int));
  if (one_block) FM_HIP(hipEventRecord(ctx->ev_sizes, st));
  hipLaunchKernelGGL(k_bond_fill, dim3((n + 3) / 4), dim3(256), 0, st, n, s->species.as<int>(),
                     s->cumulative.as<int>(), s->nspecies.as<int>(), s->rel.as<double>(),
                     s->d_cutoffs.as<double>(), nos, s->bond_off.as<int>(), s->sidx.as<int>(),
                     s->bond_q.as<int>(), in_count.as<int>(), in_slot.as<int>(),
                     one_block ? nullptr : by_type.as<int>(), host_bonds);
  if (!one_block) FM_HIP(hipEventRecord(ctx->ev_sizes, st));
  s->in_off.alloc(pool, ((size_t)n + 1) * sizeof(int));
  bool own_scan = one_block && s->n_nb > 0;
  if (!own_scan) scan_exclusive(ctx, in_count.as<int>(), s->in_off.as<int>(), n);
  s->in_bond.alloc(pool, cap * sizeof(int));
  DevBuf unordered(pool, cap * sizeof(int));
  if (s->n_nb > 0) {
    hipLaunchKernelGGL(k_in_fill, dim3((unsigned)((s->n_nb + kScanBlock - 1) / kScanBlock)),
                       dim3(kScanBlock), 0, st, n, s->bond_off.as<int>(), s->bond_q.as<int>(),
                       s->sidx.as<int>(), own_scan ? in_count.as<int>() : nullptr,
                       s->in_off.as<int>(), in_slot.as<int>(), unordered.as<int>());
    hipLaunchKernelGGL(k_in_rank, dim3((n + 3) / 4), dim3(256), 0, st, n, s->in_off.as<int>(),
                       unordered.as<int>(), s->in_bond.as<int>());
  }
  FM_HIP(hipGetLastError());
}

void bonds_ready(fm_structure s) {
  fm_context ctx = s->ctx;
  FM_HIP(hipEventSynchronize(ctx->ev_sizes));
  const int *hw = ctx->pinned;
  int nos = s->nos;
  s->n_bonds = hw[kWordBonds];
  s->n_by_type.assign(hw + kWordTypes, hw + kWordTypes + nos);
  s->nb_by_type.assign(hw + kWordTypes + nos, hw + kWordTypes + 2 * nos);
  s->type_off.assign(nos + 1, 0);
  s->q_tile_row.assign(nos, 0);
  long long rows = 0;
  for (int t = 0; t < nos; t++) {
    s->type_off[t + 1] = s->type_off[t] + s->n_by_type[t];
    s->q_tile_row[t] = rows;
    rows += (s->n_by_type[t] + kI8TileA - 1) / kI8TileA * kI8TileA;
  }
}

}  // namespace fm
