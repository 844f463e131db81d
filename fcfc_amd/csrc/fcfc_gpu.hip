/*
 * fcfc_gpu.hip -- gfx950 pair-count engine for FCFC: grid build, tiling,
 * the persistent counting kernels (FP64, FP32 + FP64 edge recheck, weight
 * backward) and the C ABI declared in include/fcfc_gpu.h.
 *
 * Build (see fcfc_amd/build.py):
 *   hipcc --offload-arch=gfx950 -O3 -ffp-contract=off -fPIC -shared ...
 * -ffp-contract=off matters: the FP64 pair arithmetic must round exactly as
 * the reference's (every fma below is explicit).
 */
#include <hip/hip_runtime.h>
#include <algorithm>
#include <chrono>
#include <climits>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <type_traits>
#include <vector>

#include "fcfc_gpu.h"
#include "fcfc_kernels.h"

#define MODE_C64  0   /* FP64 counts                                    */
#define MODE_C32  1   /* FP32 distances + FP64 recheck near bin edges   */
#define MODE_GRAD 2   /* weight gradient (FP64 bins)                    */
#define MODE_C32C 3   /* MODE_C32 with the rounding census of the rechecked pairs */
#define MODE_P64  4   /* FP64, the reference's per-pair arithmetic as written */
#define MODE_GRADL 5  /* MODE_GRAD of a masked form whose range starts above zero */

/* ======================================================================== */
/*                          grid build kernels                              */
/* ======================================================================== */

__device__ __forceinline__ int fk_cell1(double v, double o, double w, int nc) {
  int q = (int) floor((v - o) / w);
  return q < 0 ? 0 : (q >= nc ? nc - 1 : q);
}

__global__ void k_zero_u64(unsigned long long *p, size_t n) {
  for (size_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0ull;
}
/* the counters and histograms of a call and the cell counts of its sort */
__global__ void k_zero_call(unsigned long long *p, size_t n, int *q, size_t m) {
  const size_t t = blockIdx.x * blockDim.x + threadIdx.x, st = gridDim.x * blockDim.x;
  for (size_t i = t; i < n; i += st) p[i] = 0ull;
  for (size_t i = t; i < m; i += st) q[i] = 0;
}

/* Exclusive scan of n ints into out[0..n] (out[n] = total).  Workgroups of
 * 1024 threads scan FK_SCAN consecutive ints each; with more than one, k_scan_sum
 * has written the workgroups' totals before, and each adds up those of the
 * workgroups ahead of it (a chain between the workgroups would serialize
 * them).  One workgroup walking all cells took 190 us for 1.1e5 and 1.1 ms for
 * 5.8e5 cells, these two launches 4.8 + 4.9 us for 2.9e5. */
#define FK_SCAN 4096
__device__ __forceinline__ int fk_scan_load(const int *in, int n, int i, int v[4]) {
  int s = 0;
#pragma unroll
  for (int q = 0; q < 4; q++) { v[q] = i + q < n ? in[i + q] : 0; s += v[q]; }
  return s;
}
/* sum of v over the workgroup's threads before this one (and of all) */
__device__ __forceinline__ int fk_scan_block(int v, int *all) {
  __shared__ int part[16];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  int inc = v;
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(inc, o, 64);
    if (lane >= o) inc += u;
  }
  if (lane == 63) part[w] = inc;
  __syncthreads();
  int base = 0, tot = 0;
  for (int q = 0; q < 16; q++) { if (q < w) base += part[q]; tot += part[q]; }
  __syncthreads();
  *all = tot;
  return base + inc - v;
}
__global__ void __launch_bounds__(1024) k_scan_sum(const int *__restrict__ in, int n,
    int *__restrict__ sums) {
  int v[4], all;
  const int s = fk_scan_load(in, n, blockIdx.x * FK_SCAN + threadIdx.x * 4, v);
  (void) fk_scan_block(s, &all);
  if (threadIdx.x == 0) sums[blockIdx.x] = all;
}
__global__ void __launch_bounds__(1024) k_scan_out(const int *__restrict__ in,
    int *__restrict__ out, int n, const int *__restrict__ sums) {
  int v[4], all, ahead = 0, base = 0;
  if (gridDim.x > 1) {
    for (int q = threadIdx.x; q < (int) blockIdx.x; q += 1024) ahead += sums[q];
    (void) fk_scan_block(ahead, &base);
  }
  const int i = blockIdx.x * FK_SCAN + threadIdx.x * 4;
  const int s = fk_scan_load(in, n, i, v);
  int run = base + fk_scan_block(s, &all);
#pragma unroll
  for (int q = 0; q < 4; q++) if (i + q < n) { out[i + q] = run; run += v[q]; }
  if (threadIdx.x == 0 && blockIdx.x + 1 == gridDim.x) out[n] = base + all;
}

/* ---- grid build: every catalogue of a call sorted into its job's grid
 * in one pass per stage (cell counting sort), so that a batch of hundreds
 * of small catalogues costs a handful of launches ---- */
struct FkStage {
  int n, obj0, cell0;         /* objects; offsets in the concatenated object
                                 and cell spaces */
  int need_s;                 /* survey |r|^2 wanted (computed when s is null) */
  FkGrid g;
  const double *x, *y, *z, *s, *w;      /* inputs; s, w may be null */
  FkRec *rec;                 /* sorted copies, from the catalogue's first object */
  double *ow;                 /* sorted weights beside |r|^2 (else null) */
  int wt;                     /* weights wanted */
  int *oidx;                  /* original index (null when unused) */
};

/* request owning index v of the concatenated space whose starts are off */
__device__ __forceinline__ int fk_stage_find(const FkStage *__restrict__ st, int nst, int v,
    int FkStage::*off) {
  int lo = 0, hi = nst - 1;                   /* last request with start <= v */
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (st[mid].*off <= v) lo = mid; else hi = mid - 1;
  }
  return lo;
}

__device__ __forceinline__ int fk_cell(const FkGrid &g, double x, double y, double z) {
  const int ix = fk_cell1(x, g.ox, g.wx, g.ncx);
  const int iy = fk_cell1(y, g.oy, g.wy, g.ncy);
  const int iz = fk_cell1(z, g.oz, g.wz, g.ncz);
  return (ix * g.ncy + iy) * g.ncz + iz;
}

__global__ void k_stage_assign(int nobj, int nst, const FkStage *__restrict__ st,
    int *__restrict__ count, int *__restrict__ rank, unsigned long long *bad) {
  for (int o = blockIdx.x * blockDim.x + threadIdx.x; o < nobj; o += gridDim.x * blockDim.x) {
    const FkStage &q = st[fk_stage_find(st, nst, o, &FkStage::obj0)];
    const int i = o - q.obj0;
    const double x = q.x[i], y = q.y[i], z = q.z[i];
    /* a non-finite coordinate has no cell and no bin: the call fails */
    if (!(__builtin_isfinite(x) && __builtin_isfinite(y) && __builtin_isfinite(z))) atomicOr(bad, 1ull);
    rank[o] = atomicAdd(count + q.cell0 + fk_cell(q.g, x, y, z), 1);
  }
}

/* sorted copies; |r|^2 with FCFC's data_preprocess lane rule
 * (2pt/build_tree.c:59-92: FMA for the first floor(n/8)*8 objects, unfused
 * for the tail), unit weights where a weighted count has none
 * (build_tree.c:143-156).  The cell is found again, which costs less than
 * storing it; its place in the cell comes from k_stage_assign (a second atomic
 * per object here took 85 us for 5e5 clustered objects, the rank 12). */
__global__ void k_stage_scatter(int nobj, int nst, const FkStage *__restrict__ st,
    const int *__restrict__ gstart, const int *__restrict__ rank) {
  for (int o = blockIdx.x * blockDim.x + threadIdx.x; o < nobj; o += gridDim.x * blockDim.x) {
    const FkStage &q = st[fk_stage_find(st, nst, o, &FkStage::obj0)];
    const int i = o - q.obj0;
    const double a = q.x[i], b = q.y[i], c = q.z[i];
    const int d = gstart[q.cell0 + fk_cell(q.g, a, b, c)] + rank[o] - q.obj0;
    const double w = q.wt ? (q.w ? q.w[i] : 1.0) : 0.0;
    double v = w;
    if (q.need_s) {
      if (q.s) v = q.s[i];
      else if (i < (q.n / 8) * 8) v = __builtin_fma(c, c, __builtin_fma(b, b, a * a));
      else { double t = a * a; t = t + b * b; v = t + c * c; }
      if (q.ow) q.ow[d] = w;
    }
    q.rec[d] = FkRec{a, b, c, v};
    if (q.oidx) q.oidx[d] = i;
  }
}

/* Work items of a job's runs: run ti becomes S items for ti < tt and St > S
 * finer items from tt on, so that the items the wavefronts take last are short
 * and the launch ends evenly.  An item is a share of the strip list and, of
 * each segment there, every SQ-th (StQ-th) chunk of 64 B objects: S / SQ
 * shares, SQ items each.  ncap runs in all: of each group of G consecutive
 * runs of the list, its first `run` runs.  A full count has one group (G = run
 * = the number of runs); the autotuner's samples take stretches spread over
 * the whole catalogue, each keeping the neighbourhood, and so the cache reuse,
 * of a full count. */
struct FkSplit { int S, SQ, tt, St, StQ, ncap, G, run, nitems, run0; };   /* run0: first run */

/* The split of nrun runs of smax strips at most and of about `chunks` chunks
 * of candidate B objects each, for nw wavefronts: ipw items per wavefront, but
 * none of fewer than 4 chunks (an item loads its A objects and searches its
 * strips first, about the work of a chunk); where that leaves wavefronts
 * without an item, one each, of 2 chunks at least.  More items than strips
 * share the chunks of a strip: sparse catalogues have few strips (weight
 * gradient of DD of 4e4 objects, 5 strips: 1.29 -> 0.40 ms).  ipw = 16 for a
 * single job (8: DR of 2e5 x 2e6 16.7 against 15.2 ms, survey (s, mu) RR 16.8
 * against 16.1); 2 for the jobs of a batch, whose workgroups move on to other
 * jobs (16: 16 mocks 5.1 against 4.2 ms, DD + DR of a fit 1.52 against 1.23).
 * At least 8 chunks: small-scale cross count 1.12 against 1.00 ms. */
__host__ __device__ inline FkSplit fk_split(int nrun, int nw, int ipw, int chunks, int smax, int frac) {
  FkSplit sp = {1, 1, 0, 1, 1, 0, nrun > 1 ? nrun : 1, nrun > 1 ? nrun : 1, 0, 0};
  if (nrun <= 0) return sp;
  if (frac > 1) {
    sp.G = (nrun + 15) / 16;
    sp.run = sp.G / frac > 1 ? sp.G / frac : 1;
  }
  const int last = (nrun - 1) / sp.G, rest = nrun - last * sp.G;
  sp.ncap = last * sp.run + (sp.run < rest ? sp.run : rest);
  auto lim = [](long long v, int most) -> int { return (int) (v < most ? v : most); };
  auto one = [](int v) -> int { return v > 1 ? v : 1; };
  /* n items of at most smax shares: q per share */
  auto parts = [&](int n, int *q) -> int { *q = (n + smax - 1) / smax; return (n + *q - 1) / *q * *q; };
  const int s16 = lim(((long long) ipw * nw + sp.ncap - 1) / sp.ncap, one(chunks / 4));
  const int s1 = lim(((long long) nw + sp.ncap - 1) / sp.ncap, one(chunks / 2));
  const int S = one(lim(s16 > s1 ? s16 : s1, 1024));
  sp.S = parts(S, &sp.SQ);
  /* the runs of about two items per wavefront at the end of the list are
   * split up to four times finer, into items of 2 chunks at least */
  const int St = lim(4LL * S, chunks / 2 > S ? chunks / 2 : S);
  sp.St = parts(lim(St, 1024), &sp.StQ);
  const long long tail = (2LL * nw + sp.S - 1) / sp.S;
  sp.tt = tail < sp.ncap ? sp.ncap - (int) tail : 0;
  if (sp.St <= sp.S) { sp.St = sp.S; sp.StQ = sp.SQ; sp.tt = sp.ncap; }
  if ((long long) sp.St * sp.ncap > (1LL << 30)) { sp.S = sp.St = sp.SQ = sp.StQ = 1; sp.tt = sp.ncap; }
  sp.nitems = sp.S * sp.tt + sp.St * (sp.ncap - sp.tt);
  return sp;
}

/* Runs of all jobs of a launch: job k owns nunit units from unit0 (ascending);
 * a unit is one block of zm z-cells of one row, cut into runs of T consecutive
 * objects.  nw, ipw, chunks, smax, frac: its split (fk_split). */
struct FkTileJob { int unit0, nunit, nblk, zm, ncz, T, nw, ipw, chunks, smax, frac; const int *cs; };

__device__ __forceinline__ int fk_tile_job(const FkTileJob *__restrict__ tj, int njob, int u) {
  int lo = 0, hi = njob - 1;                  /* last job with unit0 <= u */
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (tj[mid].unit0 <= u) lo = mid; else hi = mid - 1;
  }
  return lo;
}

/* objects [p0, p1) and row of a unit */
__device__ __forceinline__ int fk_unit(const FkTileJob &t, int u, int &p0, int &p1) {
  const int v = u - t.unit0, row = v / t.nblk, c0 = (v - row * t.nblk) * t.zm;
  const int *cs = t.cs + (size_t) row * t.ncz;
  p0 = cs[c0]; p1 = cs[min(c0 + t.zm, t.ncz)];
  return row;
}

__global__ void k_run_count(int nunit, int njob, const FkTileJob *__restrict__ tj,
    int *__restrict__ nrun) {
  for (int u = blockIdx.x * blockDim.x + threadIdx.x; u < nunit; u += gridDim.x * blockDim.x) {
    const FkTileJob t = tj[fk_tile_job(tj, njob, u)];
    int p0, p1;
    fk_unit(t, u, p0, p1);
    nrun[u] = (p1 - p0 + t.T - 1) / t.T;
  }
}
/* the runs of unit u are numbered from roff[u]; the split of every job (no
 * work item when the sort has met a non-finite coordinate) */
__global__ void k_run_emit(int nunit, int njob, const FkTileJob *__restrict__ tj,
    const int *__restrict__ roff, FkRun *__restrict__ runs, FkSplit *__restrict__ splits,
    const unsigned long long *__restrict__ bad) {
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < njob; k += gridDim.x * blockDim.x) {
    const FkTileJob t = tj[k];
    FkSplit sp = fk_split(roff[t.unit0 + t.nunit] - roff[t.unit0], max(t.nw, FK_NW), t.ipw, t.chunks, t.smax,
                          t.frac);
    sp.run0 = roff[t.unit0];
    if (*bad) sp.nitems = 0;                  /* a non-finite coordinate: nothing is counted */
    splits[k] = sp;
  }
  for (int u = blockIdx.x * blockDim.x + threadIdx.x; u < nunit; u += gridDim.x * blockDim.x) {
    const FkTileJob t = tj[fk_tile_job(tj, njob, u)];
    int p0, p1;
    const int row = fk_unit(t, u, p0, p1);
    FkRun *o = runs + roff[u];
    for (int p = p0; p < p1; p += t.T) *o++ = FkRun{row, p, min(p + t.T, p1), 0};
  }
}

/* ======================================================================== */
/*                             count kernel                                 */
/* ======================================================================== */

/* Loads through explicit address spaces: pointers that come out of the job
 * descriptors are generic to the compiler, which would use flat loads. */
template <class T>
__device__ __forceinline__ T fk_gld(const T *p, int i) {
  return ((const __attribute__((address_space(1))) T *) p)[i];
}
__device__ __forceinline__ FkRec fk_gld(const FkRec *p, int i) {
  typedef double d2 __attribute__((ext_vector_type(2)));
  const __attribute__((address_space(1))) d2 *q = (const __attribute__((address_space(1))) d2 *) (p + i);
  const d2 a = q[0], b = q[1];
  return FkRec{a.x, a.y, b.x, b.y};
}
/* a descriptor at a uniform address, read with scalar loads (only the fields
 * in use are kept) */
template <class T>
__device__ __forceinline__ T fk_cld(const T *p) {
  struct Raw { int v[sizeof(T) / 4]; } r;
  const __attribute__((address_space(4))) int *q = (const __attribute__((address_space(4))) int *) p;
#pragma unroll
  for (int i = 0; i < (int) (sizeof(T) / 4); i++) r.v[i] = q[i];
  return __builtin_bit_cast(T, r);
}
/* element i of p at an address that the compiler cannot take for one it has
 * read before: descriptors read through it are read again where they are used
 * instead of being held in (and spilled from) scalar registers */
template <class T>
__device__ __forceinline__ const T *fk_again(const T *p, int i) {
  i = __builtin_amdgcn_readfirstlane(i);
  asm volatile("" : "+s"(i));
  return p + i;
}
/* order LDS writes and reads of one wavefront (its LDS operations execute in
 * order: only the compiler has to be held) */
__device__ __forceinline__ void fk_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ int fk_lane_of(int v, int lane) {
  return __builtin_amdgcn_readlane(v, lane);
}

/* v of lane (lane with the DPP pattern CTRL applied), both halves moved */
template <int CTRL>
__device__ __forceinline__ double fk_dpp(double v) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int) (unsigned) u, CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int) (unsigned) (u >> 32), CTRL, 0xF, 0xF, true);
  return __builtin_bit_cast(double, ((unsigned long long) (unsigned) hi << 32) | (unsigned) lo);
}

/* Sum of v over each row of 16 lanes, in every lane of the row: quad
 * butterflies (lane ^ 1, lane ^ 2), then the row's half mirror (lane i of
 * 8 with 7 - i) and mirror (lane i of 16 with 15 - i).  Every lane of the
 * wavefront must be active. */
__device__ __forceinline__ double fk_row_sum(double v) {
  v += fk_dpp<0xB1>(v);       /* quad_perm [1, 0, 3, 2] */
  v += fk_dpp<0x4E>(v);       /* quad_perm [2, 3, 0, 1] */
  v += fk_dpp<0x141>(v);      /* row_half_mirror */
  v += fk_dpp<0x140>(v);      /* row_mirror */
  return v;
}

/* smallest v of the wavefront, in a scalar register; every lane active */
__device__ __forceinline__ double fk_wave_min(double v) {
  v = __builtin_fmin(v, fk_dpp<0xB1>(v));
  v = __builtin_fmin(v, fk_dpp<0x4E>(v));
  v = __builtin_fmin(v, fk_dpp<0x141>(v));
  v = __builtin_fmin(v, fk_dpp<0x140>(v));
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  double m = 0.0;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const unsigned lo = (unsigned) __builtin_amdgcn_readlane((int) (unsigned) u, 16 * r);
    const unsigned hi = (unsigned) __builtin_amdgcn_readlane((int) (unsigned) (u >> 32), 16 * r);
    const double w = __builtin_bit_cast(double, ((unsigned long long) hi << 32) | lo);
    m = r ? __builtin_fmin(m, w) : w;
  }
  const unsigned long long um = __builtin_bit_cast(unsigned long long, m);
  const unsigned lo = (unsigned) __builtin_amdgcn_readfirstlane((int) (unsigned) um);
  const unsigned hi = (unsigned) __builtin_amdgcn_readfirstlane((int) (unsigned) (um >> 32));
  return __builtin_bit_cast(double, ((unsigned long long) hi << 32) | lo);
}

/* FP32 exactness windows (see fp32_windows on the host). */
struct FkWin {
  float e_s2, e_s2x2;         /* absolute window on s^2 (or s_perp^2), 2 e_s2 */
  float e_pi, e_pix2;         /* absolute window on pi, 2 e_pi                */
  float idle_x, idle_z;       /* FP32 coordinates of idle lanes             */
  float mu_sh;                /* error bound of the FP32 mu value t         */
  float mu_c;                 /* 129 - sh: the fixed-point t (fk_mu32)      */
  unsigned mu_t16;            /* mu bin certain if t's fraction is below it */
  float s2_floor;             /* pairs below this s^2 are re-evaluated      */
  float nmu_f;
  float m2_floor;             /* survey: pairs with |a + b|^2 below this    */
};                            /* are re-evaluated                          */

/* Flags of the integer cells of the FP32 tables, set while they are staged
 * (the LDS cells then carry a float threshold in place of the flags). */
#define FK_F_EDGE 0x10000u    /* a bin edge at the lower end of the integer cell */
#define FK_F_ALW  0x20000u    /* always re-evaluate (with FK_F_EDGE set too)     */
#define FK_F_ALWAYS 0x4000u   /* FP32 threshold (high half) of FK_F_ALW cells: 2 */
#define FK_F_NEVER  0xBF80u   /* ... of cells without flags: -1                  */

/* Atomics on one address take 11.4 ns each, wherever they come from (8192
 * wavefronts: 93 us); spread over 64 lines 0.25 to 0.4 ns.  So the statistics
 * of a call are summed in FK_STATS lines, and a job's work items are dealt to
 * up to FK_GROUPS groups of workgroups with a counter each. */
#define FK_LINE 64
#define FK_STATS 64
#define FK_GROUPS 64

/* One counting job: a catalogue pair and its histogram.  A launch counts the
 * runs of one or many jobs (batched mocks); runs carry their job index. */
struct FkJob {
  FkCat A, B;
  FkGrid g;
  const int *strips;          /* (dx, dy, diag) triples */
  int nstrips;
  int autoc;                  /* COUNT: A == B, half shell + the run;
                                 GRAD: A == B, exclude j == i          */
  int wt;                     /* weighted histogram (double)          */
  int wg0, wg1;               /* workgroups that start with it        */
  int q0, G;                  /* its counters: line q0 of the queue, G of them */
  long long hist_off;         /* histogram of this job: gcnt + hist_off */
  double *gA;                 /* GRAD: output for A objects, indexed as the records (or null) */
  double *gB;                 /* GRAD: output for B objects (or null; auto counts: gA) */
  FkWin win;                  /* FP32 error model (MODE_C32)          */
};

struct FkArgs {
  const FkJob *jobs;
  int njobs;
  FkBins bins;
  const FkRun *runs;
  const FkSplit *splits;      /* work items of each job              */
  unsigned int *queue;        /* work items taken: counters of FK_LINE bytes */
  unsigned long long *gcnt_u;
  double *gcnt_d;
  unsigned long long *stats;  /* FK_STATS lines of evals, rechecked, census  */
  int nh;                     /* LDS histogram copies */
  /* LDS byte offsets */
  int off_hist, off_stab, off_ptab, off_edges, off_chunk, off_queue;
  int stab_c0, ptab_c0;       /* table entries before cell 0 */
  int census;
  const double *G;            /* GRAD: dL/dcnt */
};

/* The (up to three) B segments of one strip for a run of row t.row whose
 * objects span [zlo, zhi]: the objects of the strip's row within the z window
 * of that span, unwrapped (main), and its images at -Lz and +Lz. */
__device__ __forceinline__ void fk_strip_segments(const FkGrid &g, const int *cell_start,
    const FkRun &t, double zlo, double zhi, int dx, int dy, int diag, int *b0, int *len,
    int *code) {
  b0[0] = b0[1] = b0[2] = 0;
  len[0] = len[1] = len[2] = 0;
  code[0] = code[1] = code[2] = 13;
  const int ix = t.row / g.ncy, iy = t.row - ix * g.ncy;
  int bx = ix + dx, by = iy + dy, cx = 0, cy = 0;
  if (g.periodic) {
    if (bx < 0) { bx += g.ncx; cx = -1; } else if (bx >= g.ncx) { bx -= g.ncx; cx = 1; }
    if (by < 0) { by += g.ncy; cy = -1; } else if (by >= g.ncy) { by -= g.ncy; cy = 1; }
  }
  else if (bx < 0 || bx >= g.ncx || by < 0 || by >= g.ncy) return;
  const double gx = (double) max(abs(dx) - 1, 0) * g.wx;
  const double gy = (double) max(abs(dy) - 1, 0) * g.wy;
  const double d2 = gx * gx + gy * gy;
  if (d2 >= g.Rxy2) return;
  const double hz = (g.hz_const >= 0) ? g.hz_const : sqrt(fmax(g.R2 - d2, 0.0));
  const int izlo = (int) floor((zlo - hz - g.oz) / g.wz - 1e-6);
  const int izhi = (int) floor((zhi + hz - g.oz) / g.wz + 1e-6);
  const int base = (bx * g.ncy + by) * g.ncz;
  const int cxy = (cx + 1) + 3 * (cy + 1);
  const int c0 = max(izlo, 0), c1 = min(izhi, g.ncz - 1);
  code[1] = cxy + 9 * 1;
  if (c1 >= c0) {
    const int e = fk_gld(cell_start, base + c1 + 1);
    /* auto counts, same row: only objects after the run (j > i) */
    b0[1] = diag ? t.p1 : fk_gld(cell_start, base + c0);
    len[1] = max(e - b0[1], 0);
  }
  if (g.periodic) {
    if (izlo < 0) {                    /* image below z = 0: B shifted by -Lz */
      const int l0 = max(izlo + g.ncz, 0);
      b0[0] = fk_gld(cell_start, base + l0);
      len[0] = fk_gld(cell_start, base + g.ncz) - b0[0];
      code[0] = cxy + 9 * 0;
    }
    if (izhi >= g.ncz && !diag) {      /* image above: B shifted by +Lz */
      const int l1 = min(izhi - g.ncz, g.ncz - 1);
      b0[2] = fk_gld(cell_start, base);
      len[2] = fk_gld(cell_start, base + l1 + 1) - b0[2];
      code[2] = cxy + 9 * 2;
    }
  }
}

/* ---------------- FP64 pair evaluation (the arithmetic contract) -------- */

/* Pair functions return an LDS histogram index sb + nsh * mb; every value
 * >= ntoh = nsh * rows means "not counted".  The row stride nsh is an odd
 * number above ns: lanes of one histogram atomic that share an s bin but
 * differ in mu (or pi) then fall on different LDS banks (an even stride such
 * as 40 folds them onto a few).  Table sentinels are FK_OUT = 0xFFFF >= ntoh
 * (the histogram lives in LDS, so ntoh < 40960), hence sb + nsh * mb needs no
 * range test of its own: an out-of-range s (or pi) gives sb >= ntoh, a dropped
 * mu gives mb = nmu and sb + nsh * nmu >= ntoh.
 *
 * The forms that mask the lanes out of range before the binning (`masked` in
 * k_count) have neither sentinel nor test: their tables give values below the
 * range the unused column ns (or, for pi, the dummy row after the last one),
 * whose counts are never read.  fk_hslot maps an LDS slot to the reference
 * layout sb + ns * mb, -1 for unused ones. */
__device__ __forceinline__ int fk_hslot(int i, int ns, int nsh) {
  const int row = i / nsh, col = i - row * nsh;
  return col < ns ? col + ns * row : -1;
}
#define FK_NONE 0xFFFFFFFFu
#define FK_NMU32 126          /* most mu bins of the FP32 (s, mu) form      */
#define FK_DBL_EPS 2.220446049250313e-16
#define FK_FAR 1.0e30          /* coordinates of idle lanes: every pair out */

/* s^2 (or s_perp^2) bin from the LDS table, FK_OUT outside [s2min, s2max).
 * Integer tables (setup_cf.c:385-410): cell (int) s2 - (int) s2min, exactly
 * the reference's cvtt lookup (metric_common.c:500-510).  The LDS copy is
 * zero-based: entry k belongs to (int) s2 = k, the entries below (int) s2min
 * and the one at (int) s2min + len are FK_OUT, so with s2 >= 0 the range
 * check is one min.  Hybrid tables (pointer at cell 0) refine downwards
 * against the edges (FCFC_LOOKUP_HYBRID, metric_common.c:56-64): the result
 * is the last edge at or below s2 (bin 0 below the first edge).  Tables too
 * long for LDS are replaced by a binary search for that same edge.  MK: the
 * table is an FP32 one, whose cells hold the bin in their low half. */
__device__ __forceinline__ unsigned fk_edge_search(const double *e, int n, double v) {
  int lo = 0, hi = n - 1;                 /* last i in [0, n) with e[i] <= v, else 0 */
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (e[mid] <= v) lo = mid; else hi = mid - 1;
  }
  return (unsigned) lo;
}

template <bool HYB, bool MK = false>
__device__ __forceinline__ unsigned fk_sbin(double s2, const FkBins &bn,
    const unsigned *stab, const double *s2e) {
  if (HYB) {
    if (!(s2 < bn.s2max) || (bn.s2min != 0 && s2 < bn.s2min)) return FK_OUT;
    if (bn.ssearch) return fk_edge_search(s2e, bn.ns, s2);
    int k = (int) s2 - bn.soff;
    k = k < 0 ? 0 : (k >= bn.stab_len ? bn.stab_len - 1 : k);
    unsigned sb = MK ? (stab[k] & 0xFFFFu) : stab[k];
    if (sb >= (unsigned) bn.ns) {
      sb -= bn.ns;
      while (sb != 0 && s2 < s2e[sb]) sb--;
    }
    return sb;
  }
  /* unsigned: a value below -1 (a survey s_perp^2 from an infinite pi^2)
   * reads the "out" sentinel, as for values above the range */
  const unsigned k = min((unsigned) (int) s2, (unsigned) (bn.soff + bn.stab_len));
  return MK ? (stab[k] & 0xFFFFu) : stab[k];
}

template <bool HYB, bool MK = false>
__device__ __forceinline__ unsigned fk_pbin(double p, const FkBins &bn,
    const unsigned *ptab, const double *pe) {
  if (HYB) {
    if (!(p < bn.pmax) || p < bn.pmin) return FK_OUT;
    if (bn.psearch) return fk_edge_search(pe, bn.np, p);
    int k = (int) p - bn.poff;
    k = k < 0 ? 0 : (k >= bn.ptab_len ? bn.ptab_len - 1 : k);
    unsigned pb = MK ? (ptab[k] & 0xFFFFu) : ptab[k];
    if (pb >= (unsigned) bn.np) {
      pb -= bn.np;
      while (pb != 0 && p < pe[pb]) pb--;
    }
    return pb;
  }
  const unsigned k = min((unsigned) (int) p, (unsigned) (bn.poff + bn.ptab_len));
  return MK ? (ptab[k] & 0xFFFFu) : ptab[k];
}

/* mu bin of (s, mu) counts.  The reference takes m = floor of the exact
 * quotient a / s2 with a = fl(num * nmu^2) (trunc of the RZ division,
 * metric_common.c:484-486), sets m = 0 when s2 < DBL_EPSILON, drops the pair
 * when m >= nmu^2 and bins it in mutab[m] = isqrt(m) (setup_cf.c:513-531).
 * Since isqrt(floor(q)) = floor(sqrt(q)) for q >= 0, the bin is floor(t),
 * t = sqrt(a / s2), and the drop rule is floor(t) >= nmu.
 *
 * Fast path: x = nmu |dz| rsq(s2) (hardware reciprocal square root; |x - t|
 * < D = nmu 2^-20 including the products) goes into one fma with the addend
 * mu_c = 2^36 + 1 - sh, sh a multiple of 2^-16 with sh >= D + 2^-16.  The
 * sum lies in [2^36, 2^37), where doubles are spaced 2^-16, so the fma
 * rounds it once onto that grid and the low word of the result is the
 * fixed-point v = round((x - sh + 1) 2^16): its high half is K =
 * floor(x - sh) + 1 and its low half f the fraction.  When f < mu_t16 =
 * floor(2^16 (1 - 2 sh)), x lies in [K - 1 + sh - 2^-17, K - 1 + 1 - sh) and
 * the exact t strictly inside (K - 1, K): the bin is K - 1, and the
 * histogram index plus nsh is K nsh + sb, one 16-bit multiply-add of the
 * high half (fk_mad_hi16).  A t within sh of an integer (K = 0 included)
 * fails the fraction test.  Those pairs, and all with s2 below s2_exact =
 * s2max 2^-12 (which covers s2 < DBL_EPSILON and bounds t by nmu (1 +
 * 2^-21) on the fast path), are settled exactly: t_sh = v 2^-16 - 1 (exact:
 * the fma result minus 2^36 + 1) is within 1/2 of t, so k = rint(t_sh) is
 * the bin if a - k^2 s2 >= 0 (one fma, exact sign; k^2 is exact), else
 * k - 1. */
#define FK_MU_C0 68719476737.0          /* 2^36 + 1 */

/* hi16(v) * m + c (m < 2^16) in one instruction: the 16-bit multiply-add
 * reading the high half of its first operand */
__device__ __forceinline__ unsigned fk_mad_hi16(unsigned v, unsigned m, unsigned c) {
  unsigned r;
  asm("v_mad_u32_u16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(r) : "v"(v), "s"(m), "v"(c));
  return r;
}

/* hi16(v) * 4 + c, c uniform: the LDS byte address of entry hi16(v) of a
 * table of 32-bit entries at byte address c */
__device__ __forceinline__ unsigned fk_mad4_hi16(unsigned v, unsigned c) {
  unsigned r;
  asm("v_mad_u32_u16 %0, %1, 4, %2 op_sel:[1,0,0,0]" : "=v"(r) : "v"(v), "s"(c));
  return r;
}

/* lo16(a) * m + c in one instruction (the high half of a is ignored) */
__device__ __forceinline__ unsigned fk_mad_lo16(unsigned a, unsigned m, unsigned c) {
  unsigned r;
  asm("v_mad_u32_u16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(m), "v"(c));
  return r;
}

/* min / max of x and a uniform bound, one v_min_f64 / v_max_f64 (fmin and
 * fmax would also canonicalise the bound on every call); a NaN x gives the
 * bound */
__device__ __forceinline__ double fk_min64(double x, double c) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(x), "s"(c));
  return r;
}
__device__ __forceinline__ double fk_max64(double x, double c) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(x), "s"(c));
  return r;
}

/* x truncated to an unsigned integer; 0 for every negative x */
__device__ __forceinline__ unsigned fk_trunc_u32(double x) {
  unsigned r;
  asm("v_cvt_u32_f64 %0, %1" : "=v"(r) : "v"(x));
  return r;
}

/* LDS byte address of a pointer into the workgroup's LDS, and a 32-bit
 * LDS read at such an address (an ordinary load: no asm) */
__device__ __forceinline__ unsigned fk_lds_addr(const void *p) {
  return (unsigned) (uintptr_t) (const __attribute__((address_space(3))) char *) p;
}
__device__ __forceinline__ unsigned fk_lds_u32(unsigned addr) {
  return *(const __attribute__((address_space(3))) unsigned *) (uintptr_t) addr;
}

__device__ __forceinline__ unsigned fk_mu_exact(double a, double s2, double t_sh,
    const FkBins &bn) {
  if (!(s2 >= FK_DBL_EPS)) return 0u;
  double k = __builtin_rint(t_sh);
  if (__builtin_fma(-(k * k), s2, a) < 0.0) k -= 1.0;
  return (unsigned) (int) __builtin_fmin(k, bn.nmu_d);
}

/* The same mu bin transcribed directly from the reference's arithmetic:
 * the correctly rounded quotient q = fl(a / s2), floored, with the one
 * correction that turns round-to-nearest into truncation of the exact
 * quotient (q can only round up onto an integer k, and then a - k s2 < 0),
 * and the isqrt table mapping m to the bin. */
__device__ __forceinline__ unsigned fk_mu_plain(double num, double s2, const FkBins &bn) {
  if (!(s2 >= FK_DBL_EPS)) return 0u;
  const double a = num * bn.nmu2;
  const double q = a / s2;
  double m = __builtin_floor(q);
  if (m == q && __builtin_fma(-m, s2, a) < 0.0) m -= 1.0;
  if (m >= bn.nmu2) return (unsigned) bn.nmu;
  return (unsigned) fk_isqrt((int) m);
}

/* The (s, mu) index plus nsh from x = anmu r = nmu |dz| rsq(s2) >= 0; fa()
 * gives a = dz^2 nmu^2 for the exact path (evaluated there only).  Every
 * index that leaves the fast path is at least nsh (K >= 1).  CAP: survey
 * pairs, whose x has no bound near a = -b (|a + b|^2 cancels) and may be
 * NaN there, have the value capped at K = nmu + 1 (not counted, as the
 * reference drops mu >= 1).  MUT: sb is the raw cell of an integer table
 * whose high half holds the fraction threshold, mu_t16, or 0 in the cells
 * below s2_exact (whose pairs all take the exact path), so one compare of
 * the two low halves replaces the threshold and s2_exact compares; the
 * threshold then rides in the index too, which grows by mu_t16 << 16.  With
 * both, an s2 below s2low (whose cell, the first, takes the exact path) is
 * not counted. */
template <bool CAP, bool MUT, class FA>
__device__ __forceinline__ unsigned fk_smu_index(double anmu, double r, FA fa, double s2,
    unsigned sb, const FkBins &bn, bool *slow = nullptr) {
  double tm = __builtin_fma(anmu, r, bn.mu_c);
  if (CAP) tm = fk_min64(tm, bn.mu_cmax);
  const unsigned v = (unsigned) __builtin_bit_cast(unsigned long long, tm);
  unsigned idx = fk_mad_hi16(v, (unsigned) bn.nsh, sb);
  const bool exact = MUT ? !((v & 0xFFFFu) < (sb >> 16))
                         : (!((v & 0xFFFFu) < bn.mu_t16) || s2 < bn.s2_exact);
  if (slow) *slow = exact;
  if (__builtin_expect(exact, 0)) {
    unsigned k = fk_mu_exact(fa(), s2, tm - FK_MU_C0, bn);
    if (CAP && MUT && !(s2 >= bn.s2low)) k = (unsigned) bn.nmu;
    idx = (sb & 0xFFFFu) + __umul24((unsigned) bn.nsh, k + 1u) + (MUT ? bn.mu_t16 << 16 : 0u);
  }
  return idx;
}

/* Box pair, B already at its periodic image (b' = fl(b + D)).  Returns the
 * histogram index, plus nsh for (s, mu) bins outside the plain form
 * (fk_smu_index); >= ntot (+ that): not counted. */
template <int BIN, bool HYB, bool MK = false, bool PLAIN = false>
__device__ __forceinline__ unsigned fk_box64(double dx, double dy, double dz,
    const FkBins &bn, const unsigned *stab, const unsigned *ptab,
    const double *s2e, const double *pe) {
  if (BIN == FCFC_BIN_SPI) {
    const double pi = __builtin_fabs(dz);
    const double s2 = __builtin_fma(dy, dy, dx * dx);          /* :416-420 */
    const unsigned sb = fk_sbin<HYB, MK>(s2, bn, stab, s2e);
    const unsigned pb = fk_pbin<HYB, MK>(pi, bn, ptab, pe);
    if (MK && (sb == (unsigned) bn.ns || pb == (unsigned) bn.np)) return FK_NONE;
    return sb + __umul24((unsigned) bn.nsh, pb);
  }
  const double dz2 = dz * dz;
  const double s2 = __builtin_fma(dy, dy, __builtin_fma(dx, dx, dz2));  /* :426-430 */
  const unsigned sb = fk_sbin<HYB, MK>(s2, bn, stab, s2e);
  if (MK && sb == (unsigned) bn.ns) return FK_NONE;
  if (BIN == FCFC_BIN_ISO) return sb;
  if (PLAIN) return sb + __umul24((unsigned) bn.nsh, fk_mu_plain(dz2, s2, bn));
  return fk_smu_index<false, false>(__builtin_fabs(dz) * bn.nmu_d, __builtin_amdgcn_rsq(s2),
                      [&] { return dz2 * bn.nmu2; }, s2, sb, bn);
}

/* Survey pair (src/fcfc/2pt/metric_common.c:283-460, FMA vector formulas):
 * t = 2 a.b, s = |a|^2 + |b|^2, d = |a|^2 - |b|^2, pi^2 = d^2 / (t + s),
 * s^2 = s - t, s_perp^2 = (s - t) - pi^2.  (s, mu) bins need pi^2 only in
 * the exact branch of the mu bin: sqrt(pi^2) = |d| / sqrt(t + s).  QT:
 * (s_perp, pi) integer tables read in fixed point, below; os (op) is the s
 * (pi) table's LDS byte address for those lookups. */
template <int BIN, bool HYB, bool PLAIN = false, bool MK = false, bool QT = false>
__device__ __forceinline__ unsigned fk_sv64(double ax, double ay, double az,
    double as, double bx, double by, double bz, double bs, const FkBins &bn,
    const unsigned *stab, const unsigned *ptab, const double *s2e, const double *pe,
    unsigned os = 0u, unsigned op = 0u) {
  if (BIN == FCFC_BIN_ISO) {
    const double dx = ax - bx, dy = ay - by, dz = az - bz;
    const double s2 = __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
    const unsigned sb = fk_sbin<HYB, MK>(s2, bn, stab, s2e);
    return MK && sb == (unsigned) bn.ns ? FK_NONE : sb;
  }
  const double t = __builtin_fma(az, bz, __builtin_fma(ay, by, ax * bx)) * 2.0;
  const double s = as + bs;
  const double d = as - bs;
  if (BIN == FCFC_BIN_SMU) {
    const double s2 = s - t;
    const unsigned sb = fk_sbin<HYB, MK>(s2, bn, stab, s2e);
    if (MK && sb == (unsigned) bn.ns) return FK_NONE;
    if (PLAIN) return sb + __umul24((unsigned) bn.nsh, fk_mu_plain((d * d) / (t + s), s2, bn));
    return fk_smu_index<true, false>(__builtin_fabs(d) * bn.nmu_d,
                        __builtin_amdgcn_rsq((t + s) * s2),
                        [&] { return ((d * d) / (t + s)) * bn.nmu2; }, s2, sb, bn);
  }
  /* (s_perp, pi): pbin holds pi^2 edges; with s2min == 0 the reference has
   * no lower bound on s_perp^2 (a rounding-negative value lands in bin 0) */
  if (QT) {
    /* Integer tables in the FP64 forms: no division on the fast path.
     * With y = rcp(B) refined once (B = t + s, |y - 1/B| <= 2^-45.9 / B for
     * the documented 2^-23 of v_rcp_f64 and B >= q_bmin), q = n y is within
     * 2^-29.8 of the reference's correctly rounded n / B below 2^16, and
     * s_perp^2 = (s - t) - q within 2^-29.7 of the reference's.  Each is
     * read in fixed point as the mu bin is (fk_smu_index): x + q_c, q_c =
     * 2^36 + 2 - h (h = 2^-15), lies in [2^36, 2^37) (clamped to it) and is
     * rounded once onto the grid 2^-16, so the low word holds K = floor(x -
     * h) + 2 in its high half and the fraction f in its low half.  The
     * tables (staged by k_count, qt_entry) are indexed by K: entry K holds
     * the bin of (int) x for x in (K - 2, K - 1) (entry 0: out, entry 1:
     * the cell of (-1, 0)) and in its high half the largest f for which x
     * is certainly in that interval (q_t16) when the bin changes at K - 1,
     * 0xFFFF when it does not.  Anything else -- f above it, B below q_bmin (zero,
     * negative, NaN) -- is binned with the reference's division. */
    const double n = d * d, bb = t + s;
    const double y0 = __builtin_amdgcn_rcp(bb);
    const double q = n * __builtin_fma(y0, __builtin_fma(-bb, y0, 1.0), y0);
    const double sp = (s - t) - q;
    const unsigned vq = (unsigned) __builtin_bit_cast(unsigned long long,
        fk_min64(q + bn.q_c, bn.q_capp));
    const unsigned vs = (unsigned) __builtin_bit_cast(unsigned long long,
        fk_min64(fk_max64(sp + bn.q_c, 68719476736.0), bn.q_caps));
    const unsigned eq = fk_lds_u32(fk_mad4_hi16(vq, op));
    const unsigned es = fk_lds_u32(fk_mad4_hi16(vs, os));
    unsigned idx = fk_mad_lo16(eq, (unsigned) bn.nsh, es & 0xFFFFu);
    const bool clear = (bb >= bn.q_bmin) & ((vq & 0xFFFFu) <= (eq >> 16)) &
                       ((vs & 0xFFFFu) <= (es >> 16));
    if (__builtin_expect(!clear, 0)) {
      const double p2 = n / bb;
      const double sp2 = (s - t) - p2;
      const unsigned ks = min((unsigned) (int) sp2, (unsigned) (bn.soff + bn.stab_len)) + 2u;
      const unsigned kp = min((unsigned) (int) p2, (unsigned) (bn.poff + bn.ptab_len)) + 2u;
      idx = (stab[ks] & 0xFFFFu) + __umul24((unsigned) bn.nsh, ptab[kp] & 0xFFFFu);
    }
    return idx;
  }
  const double p2 = (d * d) / (t + s);
  const double sp2 = (s - t) - p2;
  const unsigned sb = fk_sbin<HYB, MK>(sp2, bn, stab, s2e);
  const unsigned pb = fk_pbin<HYB, MK>(p2, bn, ptab, pe);
  return sb + __umul24((unsigned) bn.nsh, pb);
}

/* The other arithmetic paths of the reference, for the rounding census
 * (box only): vectorised a-side ((a+S)-b, var 0), per-pair periodic wrap
 * (var 2) and the unfused scalar remainder path (var 3). */
template <int BIN, bool HYB>
__device__ unsigned fk_box_variant(int var, const double a[3], const double bo[3],
    const int dcode[3], const FkGrid &g, const FkBins &bn, const unsigned *stab,
    const unsigned *ptab, const double *s2e, const double *pe) {
  const double L[3] = {g.Lx, g.Ly, g.Lz};
  double d[3];
  for (int k = 0; k < 3; k++) {
    const double D = dcode[k] * L[k];        /* b image = b + D, S = -D */
    if (var == 0 || var == 3) d[k] = (a[k] - D) - bo[k];
    else {
      double v = a[k] - bo[k];
      const double h = L[k] * 0.5;
      if (v > h) v = v - L[k]; else if (v < -h) v = v + L[k];
      d[k] = v;
    }
  }
  const int scalar = (var == 3);
  if (BIN == FCFC_BIN_SPI) {
    const double pi = fabs(d[2]);
    const double s2 = scalar ? (d[0] * d[0] + d[1] * d[1]) : __builtin_fma(d[1], d[1], d[0] * d[0]);
    const unsigned sb = fk_sbin<HYB, true>(s2, bn, stab, s2e);
    const unsigned pb = fk_pbin<HYB, true>(pi, bn, ptab, pe);
    if (sb == (unsigned) bn.ns || pb == (unsigned) bn.np) return FK_NONE;
    return sb + __umul24((unsigned) bn.nsh, pb);
  }
  const double dz2 = d[2] * d[2];
  double s2;
  if (scalar) { double t = d[0] * d[0]; t = t + d[1] * d[1]; s2 = t + dz2; }
  else s2 = __builtin_fma(d[1], d[1], __builtin_fma(d[0], d[0], dz2));
  const unsigned sb = fk_sbin<HYB, true>(s2, bn, stab, s2e);
  if (sb == (unsigned) bn.ns) return FK_NONE;
  if (BIN == FCFC_BIN_ISO || sb == FK_OUT) return sb;
  int m = 0;
  if (s2 >= FK_DBL_EPS) {
    if (scalar) {
      const double q = (dz2 / s2) * bn.nmu2;           /* :184 */
      if (q >= bn.nmu2) return FK_NONE;
      m = (int) q;
    }
    else {
      const double mq = fk_floor_div(dz2 * bn.nmu2, s2);
      if (mq >= bn.nmu2) return FK_NONE;
      m = (int) mq;
    }
  }
  return sb + __umul24((unsigned) bn.nsh, (unsigned) fk_isqrt(m));
}

/* ---------------- FP32 pair evaluation with exactness windows ----------- */
/* Coordinates relative to the centre of the A run in FP32.  A pair within the
 * rounding bound of a bin edge that matters is re-evaluated in FP64 and its
 * index ignored.  Window test of s^2 (and pi): with
 * u = s2 + e, s2 is within e of an integer k exactly when fract(u) < 2e,
 * and then k = (int) u; otherwise (int) u = (int) s2.  So the table entry
 * at (int) u is the cell of s2 when s2 is clear of the integers, and the
 * cell above the nearby integer otherwise, whose FK_F_EDGE flag says
 * whether that integer is a bin edge (if not, both cells give the same
 * bin).  A cell of the FP32 tables holds the bin in its low 16 bits and in
 * its high 16 bits those of a float threshold: -1 without flags, the window
 * 2e rounded up (the largest of the launch's jobs) with FK_F_EDGE, 2 with
 * FK_F_ALW.  Read as a float, the cell lies within 2^-7 relative of its
 * threshold, on the side away from zero (thresholds are normal numbers:
 * comparisons with subnormals are slow), so the test is one compare of the
 * cell itself: fract(u) < cell.  The zero-based FP32 tables run to (int)
 * s2min + len + 1: the entry after the last cell flags the edge at s2max, the
 * last one is a plain FK_OUT for pairs certainly out of range (survey
 * (s_perp, pi), whose pairs are not masked). */


/* FP32 mu bin floor(t) from x = anmu r (|x - t| < D above s2_floor, the
 * cells below s2_floor carry FK_F_ALW: every pair there is re-evaluated;
 * t <= nmu (1 + 2^-20) <= 126), in fixed point as in fk_mu_exact: the fma
 * with mu_c = 129 - sh (sh a multiple of 2^-16, sh >= D + 2^-16) rounds
 * once onto the grid 2^-16 of [128, 256), so the float's bits are
 * 0x43000000 + round((x - sh + 1) 2^16): the high half is 0x4300 + K, K =
 * floor(x - sh) + 1, the low half the fraction f.  f < mu_t16 = floor(2^16
 * (1 - 2 sh)) puts the exact t strictly inside (K - 1, K); otherwise
 * ambig_mu.  Returns the index plus 0x4301 nsh: (0x4300 + K) nsh + sb. */
__device__ __forceinline__ unsigned fk_mu32(float anmu, float r, unsigned sb,
    const FkBins &bn, const FkWin &wn, bool &ambig_mu) {
  const unsigned v = __float_as_uint(__builtin_fmaf(anmu, r, wn.mu_c));
  ambig_mu = !((v & 0xFFFFu) < wn.mu_t16);
  return fk_mad_hi16(v, (unsigned) bn.nsh, sb);
}

/* FP32 survey pairs.  d = b - a from coordinates relative to the run's
 * centre (as for box pairs) and m = a + b = 2 a + d (m* = 2 a in FP32), so
 * that s^2 = |d|^2, pi = d.m / |m| and mu = pi / s carry the FP32 error of
 * differences, not the cancellation of |a|^2 + |b|^2 - 2 a.b that the
 * reference's FP64 formulas have (metric_common.c:338-364): its values
 * differ from the exact ones by its own rounding, which the windows include
 * (fp32_windows).  Pairs with |m|^2 below m2_floor (both objects near the
 * observer, on opposite sides) are always re-evaluated, as are pairs of
 * cells flagged for it.  (s_perp, pi): the tables hold pi^2 and s_perp^2 =
 * s^2 - pi^2, whose FP32 value may come out slightly negative (index 0, as
 * the reference's truncation gives); lanes whose indices come out below -1
 * (pairs below m2_floor) read the "out" sentinel (the three conditions come
 * back apart, so that each ballot is its compare's own mask). */
__device__ __forceinline__ unsigned fk_sv32_spi(float dx, float dy, float dz, float mx, float my,
    float mz, const FkBins &bn, const FkWin &wn, const unsigned *stab, const unsigned *ptab,
    bool &ambig, bool &ambig_pi, bool &ambig_m) {
  const float s2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
  const float p = __builtin_fmaf(dz, mz, __builtin_fmaf(dy, my, dx * mx));
  const float m2 = __builtin_fmaf(mz, mz, __builtin_fmaf(my, my, mx * mx));
  ambig_m = m2 < wn.m2_floor;          /* near the observer: re-evaluate */
  const float p2 = (p * p) * __builtin_amdgcn_rcpf(m2);
  const float sp2 = s2 - p2;
  const float u = sp2 + wn.e_s2;
  const unsigned e = stab[min((unsigned) (int) u, (unsigned) bn.scap32)];
  ambig = __builtin_amdgcn_fractf(u) < __uint_as_float(e);
  const float up = p2 + wn.e_pi;
  const unsigned ep = ptab[min((unsigned) (int) up, (unsigned) bn.pcap32)];
  ambig_pi = __builtin_amdgcn_fractf(up) < __uint_as_float(ep);
  return (e & 0xFFFFu) + __umul24((unsigned) bn.nsh, ep & 0xFFFFu);
}

/* Exact FP64 re-evaluation of a pair flagged by the FP32 windows (rare: the
 * pairs are queued and re-evaluated together after each chunk).  The tables
 * are the flagged FP32 ones, read through their bin bits.  With census
 * enabled the other rounding paths of the reference are evaluated as well
 * and pairs whose bin depends on the path are counted. */
template <int BIN, bool HYB>
__device__ __forceinline__ bool fk_census(const FkBins &bn, const FkJob &J, double ax,
    double ay, double az, const double bo[3], const int c3[3], unsigned idx,
    const unsigned *stab, const unsigned *ptab, const double *s2e, const double *pe) {
  const unsigned nt = (unsigned) bn.ntoh;
  const double av3[3] = {ax, ay, az};
  bool differ = false;
  for (int v = 0; v < 4; v++) {
    if (v == 1) continue;
    unsigned iv = fk_box_variant<BIN, HYB>(v, av3, bo, c3, J.g, bn, stab, ptab, s2e, pe);
    if (iv >= nt) iv = FK_NONE;
    differ = differ || (iv != idx);
  }
  return differ;
}

template <int BIN, bool HYB, bool CEN>
__device__ __forceinline__ unsigned fk_recheck(const FkBins &bn, const FkJob &J,
    double ax, double ay, double az, int jg, int code, const unsigned *stab,
    const unsigned *ptab, const double *s2e, const double *pe, unsigned int *ncensus) {
  const int c3[3] = {code % 3 - 1, (code / 3) % 3 - 1, code / 9 - 1};
  const FkRec b = fk_gld(J.B.rec, jg);
  const double bo[3] = {b.x, b.y, b.z};
  const double ex = bo[0] + c3[0] * J.g.Lx;
  const double ey = bo[1] + c3[1] * J.g.Ly;
  const double ez = bo[2] + c3[2] * J.g.Lz;
  unsigned idx = fk_box64<BIN, HYB, true>(ex - ax, ey - ay, ez - az, bn, stab, ptab, s2e, pe);
  if (BIN == FCFC_BIN_SMU) idx -= (unsigned) bn.nsh;
  if (idx >= (unsigned) bn.ntoh) idx = FK_NONE;
  if (CEN && fk_census<BIN, HYB>(bn, J, ax, ay, az, bo, c3, idx, stab, ptab, s2e, pe))
    (*ncensus)++;
  return idx;
}

/* The same for a survey pair: A object p, B object jg, with the reference's
 * FP64 formulas (fk_sv64). */
template <int BIN, bool HYB>
__device__ __forceinline__ unsigned fk_recheck_sv(const FkBins &bn, const FkJob &J, int p,
    int jg, const unsigned *stab, const unsigned *ptab, const double *s2e, const double *pe) {
  const FkRec a = fk_gld(J.A.rec, p), b = fk_gld(J.B.rec, jg);
  unsigned idx = fk_sv64<BIN, HYB, false, true>(a.x, a.y, a.z, a.q, b.x, b.y, b.z, b.q, bn, stab,
                                                ptab, s2e, pe);
  if (BIN == FCFC_BIN_SMU) idx -= (unsigned) bn.nsh;
  return idx >= (unsigned) bn.ntoh ? FK_NONE : idx;
}

/* ---------------------------- the kernel --------------------------------- */

/* LDS bytes of one staged B object: FP32 coordinates relative to the run's
 * centre, weight and sorted index; the gradient form keeps the gradient share
 * and the sorted index of each B object, the FP64 counts nothing */
/* (wsep: the weights are not in the records; G > 1: groups of lanes, k_count) */
__host__ __device__ constexpr int fk_chunk_bytes(bool f32, bool wt, bool grad, bool wsep, int G) {
  return f32 ? 12 + (wt ? 8 : 0) + 4
             : (grad ? 8 : 0) + (G > 1 ? 36 + (wsep && (wt || grad) ? 8 : 0) : 0);
}

/* One persistent kernel for counts (FP64 or FP32 + recheck) and for the
 * weight gradient.  Template parameters: binning, geometry, weighted
 * histogram support, mode, hybrid tables, A objects per lane, groups of lanes.
 * Unweighted
 * kernels are held to 64 VGPRs (8 waves per SIMD, 4 workgroups per CU):
 * occupancy pays more than the FP32 form's spills, which sit in its rare
 * re-evaluation paths.  Weighted ones get 80 (6 waves per SIMD), as their
 * FP64 LDS histograms limit them to 3 workgroups per CU anyway.
 *
 * The kernel is bound by the VALU instructions of the evaluated pairs, so the
 * split is chosen to evaluate few: a wavefront takes 64 R objects on its own
 * (a compact box, no lanes idle because a tile of 8 wavefronts is not full,
 * no barrier in the loop), and a B object that is beyond the separation from
 * that box costs one lane's share of a test instead of 64 R distances.
 * Against tiles of 512 R objects that shared their B chunks (same data, ms of
 * the whole call): (s, mu) RR of 4e6 objects 331 -> 232, weighted DD of 5e5
 * 16.9 -> 9.1, w_p of 1e6 to 40 Mpc/h (128 objects in tiles of 1024) 11.8 ->
 * 4.6, survey (s, mu) RR of 1.2e6 27.1 -> 16.1.
 *
 * The weighted FP64 counts are bound by the LDS next: a table entry and an
 * FP64 atomic per lane and pair, and with the B objects in LDS four more
 * 8-byte reads per object, about half of the LDS's cycles (LDS 81 % busy,
 * VALU 65 %, and room for 2 workgroups per CU).  The FP64 forms therefore
 * read each kept B object from its sorted record into scalar registers (one
 * 32-byte line per object, mostly hits of the scalar cache, as the wavefront
 * has just loaded the line to test the object): weighted DD of 5e5 9.1 -> 7.5
 * ms, DR of 2e5 x 2e6 20.9 -> 16.6, the hybrid w_p count 3.5 -> 3.0; the
 * unweighted RR, bound by the VALU, is unchanged (232).  The FP32 forms keep
 * the chunk: their coordinates are converted once for 64 R pairs there, and
 * its 4-byte reads cost the LDS half as much.
 *
 * NG > 1: NG groups of 64 / NG lanes hold the same run of 64 / NG A objects
 * and take every NG-th kept B object each, from the chunk.  In a sparse
 * catalogue 64 objects spread over more than the separations counted, and most
 * pairs of a run are out of range: 16 objects have a quarter of the volume
 * (iso cross count of 3e5 x 1e6: 1.10 -> 0.56 ms, w_p of 1e6 2.5 -> 1.8). */
template <int BIN, int GEOM, bool WT, int MODE, bool HYB, int R, int NG = 1>
__global__ void __launch_bounds__(FK_NT, WT ? 6 : 8)
k_count(const FkArgs a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr bool F32 = (MODE == MODE_C32 || MODE == MODE_C32C);
  constexpr bool CENS = (MODE == MODE_C32C);
  constexpr bool PLAIN = (MODE == MODE_P64);
  constexpr bool GRAD = (MODE == MODE_GRAD || MODE == MODE_GRADL);
  constexpr bool SV32 = (GEOM == FCFC_GEOM_SURVEY && (MODE == MODE_C32 || MODE == MODE_C32C));
  /* |r|^2 of the objects: survey (s, mu) and (s_perp, pi) in FP64 (the FP32
   * form reads them from the catalogue when it re-evaluates a pair) */
  constexpr bool NEED_S = (GEOM == FCFC_GEOM_SURVEY && BIN != FCFC_BIN_ISO && !SV32);
  /* weights beside the records (which then hold |r|^2) */
  constexpr bool WSEP = (GEOM == FCFC_GEOM_SURVEY && BIN != FCFC_BIN_ISO);
  const int tid = threadIdx.x;
  /* the wavefront index, in a scalar register (with everything derived
   * from it: the wavefront's histogram copy and queue) */
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const FkBins &bn = a.bins;
  const unsigned ntot = (unsigned) bn.ntoh;   /* LDS histogram slots */
  /* the pair functions' (s, mu) indices carry an offset (fk_mu_exact,
   * fk_mu32); indices below it are never counted.  MUT: the FP64 integer
   * table cells carry the mu fraction threshold (fk_smu_index) */
  constexpr bool MUT = (BIN == FCFC_BIN_SMU && !F32 && !PLAIN && !HYB);
  /* QT: survey (s_perp, pi) in the FP64 forms with integer tables, pi^2
   * and s_perp^2 read in fixed point (fk_sv64); the tables start at floor
   * cell -2 and carry fraction thresholds (qt_entry below) */
  constexpr bool QT = (GEOM == FCFC_GEOM_SURVEY && BIN == FCFC_BIN_SPI && !F32 && !PLAIN && !HYB);
  /* MASKED: the lanes out of range are masked off before the binning, so that
   * neither the table index nor the histogram index needs a test of its own
   * (the pair loop is bound by its VALU instructions: two of seventeen less.
   * (s, mu) RR of 4e6 213 -> 208 ms, FP32 survey RR of 1.2e6 16.2 -> 15.5,
   * weighted DD of 5e5 7.0 -> 6.7).  FP64 with integer tables and FP32, except
   * survey (s_perp, pi), whose s_perp^2 and pi^2 are found together. */
  constexpr bool MASKED = !(GEOM == FCFC_GEOM_SURVEY && BIN == FCFC_BIN_SPI) &&
                          (F32 || (!HYB && !PLAIN));
  const unsigned ioff = (BIN != FCFC_BIN_SMU || PLAIN) ? 0u
                        : F32 ? 0x4301u * (unsigned) bn.nsh
                        : (unsigned) bn.nsh + (MUT ? bn.mu_t16 << 16 : 0u);
  const unsigned ntot_o = ntot + ioff;

  /* ---- LDS carve-up (lds_plan on the host computes the same offsets) ---- */
  unsigned int *hist_u = (unsigned int *) (lds + a.off_hist);
  double *hist_d = (double *) (lds + a.off_hist);
  /* tables: raw[c0 + c] is integer cell c, c0 = a.stab_c0 (a.ptab_c0)
   * entries precede cell 0 and two follow the last one.  Integer tables and
   * all FP32 ones are zero-based (c0 = (int) s2min: entry k is the one of
   * (int) s2 = k); hybrid ones for the FP64 forms may have c0 = 1.  Hybrid
   * lookups index cells from raw + c0 */
  unsigned *stab_raw = (unsigned *) (lds + a.off_stab);
  unsigned *ptab_raw = (unsigned *) (lds + a.off_ptab);
  const unsigned *stab = HYB ? stab_raw + a.stab_c0 : stab_raw;
  const unsigned *ptab = HYB ? ptab_raw + a.ptab_c0 : ptab_raw;
  const unsigned os_lds = fk_lds_addr(stab_raw), op_lds = fk_lds_addr(ptab_raw);
  double *s2e = (double *) (lds + a.off_edges);
  double *pe = s2e + (bn.ns + 1);
  /* the wavefront's chunk of B objects */
  char *cp = lds + a.off_chunk + wave * (FK_CH * fk_chunk_bytes(F32, WT, GRAD, WSEP, NG));
  FkRec *cr = (FkRec *) cp;                    /* FP64, NG > 1: records at the image of B */
  if (!F32 && NG > 1) cp += sizeof(FkRec) * FK_CH;
  double *cb = (double *) cp;                  /* GRAD: gradient share of each B object */
  if (GRAD) cp += 8 * FK_CH;
  double *cw = (double *) cp;                  /* weights: FP32, and FP64 with NG > 1 */
  if (F32 ? WT : NG > 1 && WSEP && (WT || GRAD)) cp += 8 * FK_CH;
  float *fx = (float *) cp, *fy = fx + FK_CH, *fz = fy + FK_CH;
  int *cj = F32 ? (int *) (fz + FK_CH) : (int *) cp;   /* sorted index */
  /* FP32 re-evaluation queue of this wavefront: sorted index of the B
   * object, A slot in the run << 5 | periodic image code */
  unsigned *wqj = (unsigned *) (lds + a.off_queue + wave * (FK_QCAP * 6));
  uint16_t *wqs = (uint16_t *) (wqj + FK_QCAP);
  __shared__ int s_job;
  __shared__ double s_box[FK_NW][6];           /* bounding boxes of the runs */
  double *box = s_box[wave];

  /* ---- stage tables ---- */
  const int hist_elems = a.nh * bn.nslot;
  if (GRAD) {
    for (int i = tid; i < bn.nslot; i += FK_NT) {
      const int g = i < bn.ntoh ? fk_hslot(i, bn.ns, bn.nsh) : -1;
      hist_d[i] = g >= 0 ? a.G[g] : 0.0;
    }
  }
  else if (WT) { for (int i = tid; i < hist_elems; i += FK_NT) hist_d[i] = 0.0; }   /* covers the u32 view */
  else { for (int i = tid; i < hist_elems; i += FK_NT) hist_u[i] = 0u; }
  {
    /* cell c of a table of len cells; FP32 entries carry the edge flags */
    auto cell = [](const uint16_t *t, int len, int c) -> unsigned {
      return (c >= 0 && c < len) ? (unsigned) t[c] : FK_OUT;
    };
    /* alw_below > 0: cells whose lower end lies below alw_below + 1 are
     * always re-evaluated (the extra cell covers pairs just below the first
     * other cell, which the window test reads through that cell).  Hybrid
     * tables (lut_hybrid, setup_cf.c) give the cell holding a non-integer
     * lower range edge the first bin and leave values below the edge to the
     * lookup's explicit range check, so that cell is always re-evaluated as
     * well (refinement cells, v >= nb, always are). */
    auto entry = [&](const uint16_t *t, int len, int nb, int c, double off, double alw_below,
                     double lo_edge) -> unsigned {
      unsigned v = cell(t, len, c);
      if (!F32) return MASKED && c < 0 ? (unsigned) nb : v;
      unsigned f = 0;
      if (cell(t, len, c - 1) != v) f |= FK_F_EDGE;
      /* the cell after one holding a non-integer lower edge: a value just
       * below that edge may land at its lower end (same bin, no edge of the
       * table there) */
      if (HYB && c == 1 && off != lo_edge) f |= FK_F_EDGE;
      const bool low = alw_below > 0 && off + c < alw_below + 1.0;
      if (v != FK_OUT && (v >= (unsigned) nb || low || (HYB && c == 0 && off != lo_edge)))
        f |= FK_F_ALW | FK_F_EDGE;
      /* masked lanes reach the first sentinel only within the window of the
       * upper range edge, and the cells below the range with any s^2 down to
       * 0.  There the mu estimate is no bin: 0 * inf at zero distance, whose
       * NaN passes the fraction test of fk_mu32, so those below s2_floor are
       * re-evaluated like the others (and dropped) */
      if (MASKED && (c == len || (c < 0 && low))) f |= FK_F_ALW | FK_F_EDGE;
      if (MASKED && c < 0) v = (unsigned) nb;
      return v | f;
    };
    /* FP32 tables: bin and the high half of the threshold of fract(u),
     * the window rounded up */
    auto put = [&](unsigned *raw, int i, unsigned v, float win2) {
      if (!F32) { raw[i] = v; return; }
      const unsigned th = (v & FK_F_ALW) ? FK_F_ALWAYS
                          : ((v & FK_F_EDGE) ? (__float_as_uint(win2) + 0xFFFFu) >> 16 : FK_F_NEVER);
      raw[i] = (th << 16) | (v & 0xFFFFu);
    };
    /* QT tables: entry K holds the bin of (int) x for x in (K - 2, K - 1)
     * (entry 0: out; entry 1, x in (-1, 0): cell 0) and in its high half
     * the fraction threshold of fk_sv64's fixed-point lookup: q_t16 where
     * the bin changes at x = K - 1, 0xFFFF where it does not; off + len + 4
     * entries (the last one out, also for the ceilings q_caps / q_capp) */
    auto qt_entry = [&](const uint16_t *t, int len, int off, int k) -> unsigned {
      auto low = [&](int e) -> unsigned { return e == 0 ? FK_OUT : cell(t, len, max(e - 2, 0) - off); };
      const unsigned v = low(k);
      return ((v != low(k + 1) ? bn.q_t16 : 0xFFFFu) << 16) | v;
    };
    if (QT) {
      for (int i = tid; i < bn.soff + bn.stab_len + 4; i += FK_NT)
        stab_raw[i] = qt_entry(bn.stab, bn.stab_len, bn.soff, i);
      for (int i = tid; i < bn.poff + bn.ptab_len + 4; i += FK_NT)
        ptab_raw[i] = qt_entry(bn.ptab, bn.ptab_len, bn.poff, i);
    }
    const double s2f = (F32 && BIN == FCFC_BIN_SMU) ? (double) a.jobs[0].win.s2_floor : 0.0;
    if (!QT)
    for (int i = tid; i < a.stab_c0 + bn.stab_len + 2; i += FK_NT) {
      unsigned v = entry(bn.stab, bn.stab_len, bn.ns, i - a.stab_c0, bn.soff, s2f, bn.s2min);
      /* MUT (zero-based: entry i holds (int) s2 = i): the mu fraction
       * threshold, 0 where the cell reaches below s2_exact */
      if (MUT && !((double) i < bn.s2_exact)) v |= bn.mu_t16 << 16;
      put(stab_raw, i, v, bn.win2s);
    }
    if (BIN == FCFC_BIN_SPI && !QT)
      for (int i = tid; i < a.ptab_c0 + bn.ptab_len + 2; i += FK_NT)
        put(ptab_raw, i, entry(bn.ptab, bn.ptab_len, bn.np, i - a.ptab_c0, bn.poff, 0.0, bn.pmin),
            bn.win2p);
  }
  if (HYB) {
    for (int i = tid; i <= bn.ns; i += FK_NT) s2e[i] = bn.s2bin[i];
    if (BIN == FCFC_BIN_SPI) for (int i = tid; i <= bn.np; i += FK_NT) pe[i] = bn.pbin[i];
  }

  unsigned long long evals = 0;               /* uniform: distances evaluated */
  unsigned int nrecheck = 0, ncensus = 0;
  /* pairs this wavefront may have added to 32-bit counters since the
   * workgroup's last flush (FK_NW such budgets stay below 2^32) */
  unsigned since = 0;
  unsigned int *myhist_u = hist_u + (wave % a.nh) * bn.nslot;
  double *myhist_d = hist_d + (wave % a.nh) * bn.nslot;
  /* byte offsets in lds of these histograms, minus the pair functions'
   * index offset times the slot size: lds + (o + idx * size) is slot
   * idx - ioff (unsigned arithmetic, modulo 2^32; in range for every
   * counted index) */
  const unsigned ohist_u = (unsigned) a.off_hist + 4u * ((unsigned) (wave % a.nh) * (unsigned) bn.nslot - ioff);
  const unsigned ohist_d = (unsigned) a.off_hist + 8u * ((unsigned) (wave % a.nh) * (unsigned) bn.nslot - ioff);
  const unsigned ohist_g = (unsigned) a.off_hist - 8u * ioff;
  const int lane = tid & 63;
  /* NG groups of NA lanes hold the same A objects, each for its own B objects */
  constexpr int NA = 64 / NG;
  const int slot = lane & (NA - 1), sub = NG > 1 ? lane / NA : 0;

  /* 32-bit counters: a wavefront that may have added FK_BUDGET pairs since
   * it last did so adds the workgroup's counters to the job's global histogram
   * (the others go on counting meanwhile), so that FK_NW budgets bound every
   * counter below 2^32 */
#define FK_BUDGET 500000000u
  int cur = -1;
  auto spill_counts = [&]() {
    unsigned long long *g0 = a.gcnt_u + fk_cld(&fk_again(a.jobs, cur)->hist_off);
    for (int i = lane; i < hist_elems; i += 64) {
      const int k = i % bn.nslot, g = k < bn.ntoh ? fk_hslot(k, bn.ns, bn.nsh) : -1;
      const unsigned v = atomicExch(hist_u + i, 0u);
      if (g >= 0 && v) atomicAdd(g0 + g, (unsigned long long) v);
    }
    since = 0;
  };

  /* wavefronts of the workgroups of group g (of G) of a job that nwg
   * workgroups start with, and the counter of line q of the queue */
  auto group_waves = [](int nwg, int G, int g) -> int { return FK_NW * ((nwg - g + G - 1) / G); };
  auto queue_load = [&](int q) -> unsigned {
    return __hip_atomic_load(a.queue + (size_t) q * (FK_LINE / 4), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };

  /* Each workgroup counts one job at a time; its wavefronts take the job's
   * items on their own and meet when it has none left.  Then the LDS
   * histograms are added to the job's global one and the workgroup goes on to
   * a job that has some: in a batch the workgroups start dealt out to the jobs
   * in proportion to their expected work, so that most count one job and
   * flush once (with one queue for all jobs every workgroup visited every job:
   * 16 mocks, 48 jobs, 8.7 -> 5.9 ms). */
  for (;;) {
    __syncthreads();
    if (!GRAD && cur >= 0) {
      const FkJob *pj = fk_again(a.jobs, cur);
      const bool w = WT && fk_cld(&pj->wt);
      const long long ho = fk_cld(&pj->hist_off);
      for (int i = tid; i < bn.ntoh; i += FK_NT) {
        const int g = fk_hslot(i, bn.ns, bn.nsh);    /* unused slots are left */
        if (g < 0) continue;
        if (w) {
          double v = 0;
          for (int c = 0; c < a.nh; c++) { v += hist_d[c * bn.nslot + i]; hist_d[c * bn.nslot + i] = 0.0; }
          if (v != 0) unsafeAtomicAdd(a.gcnt_d + ho + g, v);
        }
        else {
          unsigned long long v = 0;
          for (int c = 0; c < a.nh; c++) { v += hist_u[c * bn.nslot + i]; hist_u[c * bn.nslot + i] = 0u; }
          if (v) atomicAdd(a.gcnt_u + ho + g, v);
        }
      }
    }
    since = 0;
    bool first = cur < 0;
    if (wave == 0) {
      int nx = -1;
      if (first) {
        int hi = a.njobs - 1;                 /* last job with wg0 <= this workgroup */
        nx = 0;
        while (nx < hi) {
          const int mid = (nx + hi + 1) >> 1;
          if (a.jobs[mid].wg0 <= (int) blockIdx.x) nx = mid; else hi = mid - 1;
        }
      }
      /* the next job (in turn from this one) with items for every wavefront */
      else for (int k0 = 1; k0 < a.njobs && nx < 0; k0 += 64) {
        bool has = false;
        if (k0 + lane < a.njobs) {
          int q = cur + k0 + lane;
          if (q >= a.njobs) q -= a.njobs;
          const FkJob *pj = a.jobs + q;
          const int n = a.splits[q].nitems, nwg = pj->wg1 - pj->wg0;
          long long left = 0;
          for (int g = 0; g < pj->G; g++) {
            const int taken = group_waves(nwg, pj->G, g) + (int) queue_load(pj->q0 + g);
            left += max((n - g + pj->G - 1) / pj->G - taken, 0);
          }
          has = left >= (nwg ? FK_NW : 1);
        }
        const unsigned long long m = __builtin_amdgcn_ballot_w64(has);
        if (m) { nx = cur + k0 + (int) __builtin_ctzll(m); if (nx >= a.njobs) nx -= a.njobs; }
      }
      if (lane == 0) s_job = nx;
    }
    __syncthreads();
    cur = __builtin_amdgcn_readfirstlane(s_job);
    if (cur < 0) break;

    /* The job's items: item i belongs to group i % G.  The first one of each
     * wavefront that starts with the job follows from its place among the
     * group's wavefronts, the others from the group's counter; when the group
     * has none left, another one's (every wavefront ends when no group has any). */
    int grp = first ? ((int) blockIdx.x - fk_cld(&fk_again(a.jobs, cur)->wg0)) % fk_cld(&fk_again(a.jobs, cur)->G)
                    : (int) blockIdx.x % fk_cld(&fk_again(a.jobs, cur)->G);
    for (;;) {
      const FkSplit sp = fk_cld(a.splits + cur);
      const FkJob *pq = fk_again(a.jobs, cur);
      const int wg0 = fk_cld(&pq->wg0), nwg = fk_cld(&pq->wg1) - wg0, G = fk_cld(&pq->G), q0 = fk_cld(&pq->q0);
      int it = ((int) blockIdx.x - wg0) / G * FK_NW + wave;
      if (!first) {
        if (lane == 0)
          it = group_waves(nwg, G, grp) + (int) atomicAdd(a.queue + (size_t) (q0 + grp) * (FK_LINE / 4), 1u);
        it = __builtin_amdgcn_readfirstlane(it);
      }
      first = false;
      it = grp + G * it;
      if (it >= sp.nitems) {
        bool has = false;
        if (lane < G) has = lane + (long long) G * (group_waves(nwg, G, lane) + (int) queue_load(q0 + lane)) < sp.nitems;
        const unsigned long long m = __builtin_amdgcn_ballot_w64(has), mn = m >> grp >> 1;
        if (m == 0) break;
        grp = mn ? grp + 1 + (int) __builtin_ctzll(mn) : (int) __builtin_ctzll(m);
        continue;
      }
      /* work item -> run, share of its strips, chunks of their segments */
      int part, S, SQ, ri;
      const int h = sp.S * sp.tt;
      if (it < h) { S = sp.S; SQ = sp.SQ; ri = it / S; part = it - ri * S; }
      else { S = sp.St; SQ = sp.StQ; ri = (it - h) / S; part = it - h - ri * S; ri += sp.tt; }
      const int sq = part % SQ;
      S /= SQ;
      part /= SQ;
      const int smp = ri / sp.run;
      const FkRun t = fk_cld(a.runs + __builtin_amdgcn_readfirstlane(
          sp.run0 + smp * sp.G + (ri - smp * sp.run)));

      const FkJob J = fk_cld(a.jobs + cur);
      const int s0 = (int) ((long long) J.nstrips * part / S);
      const int s1 = (int) ((long long) J.nstrips * (part + 1) / S);
      /* weights exist for this job (a weighted-capable kernel may run
       * unweighted jobs of a batch, whose catalogues carry no weights) */
      const bool jw = GRAD || (WT && J.wt);
      const bool jwt = WT && J.wt;
      const bool hasB = GRAD && J.gB != nullptr;

      /* A objects of this lane (a wavefront holds one run) and the bounding box
       * of the run; idle lanes sit far away, so that every pair they form is
       * out of range */
      double ax[R], ay[R], az[R], as[R], aw[R], gacc[R];
      float fax[R], fay[R], faz[R];
      int ai[R];
      double lox = 1e300, loy = 1e300, loz = 1e300, hix = -1e300, hiy = -1e300, hiz = -1e300;
      unsigned long long actm[R];
#pragma unroll
      for (int r = 0; r < R; r++) {
        const int p = t.p0 + r * 64 + slot;
        const bool v = p < t.p1;
        const int pc = v ? p : t.p0;
        const FkRec ra = fk_gld(J.A.rec, pc);
        const double x = ra.x, y = ra.y, z = ra.z;
        lox = __builtin_fmin(lox, x); hix = __builtin_fmax(hix, x);
        loy = __builtin_fmin(loy, y); hiy = __builtin_fmax(hiy, y);
        loz = __builtin_fmin(loz, z); hiz = __builtin_fmax(hiz, z);
        ai[r] = v ? p : 0x7fffffff;
        ax[r] = v ? x : FK_FAR;
        ay[r] = v ? y : FK_FAR;
        az[r] = v ? z : FK_FAR;
        as[r] = NEED_S ? (v ? ra.q : 3.0 * FK_FAR * FK_FAR) : 0.0;
        aw[r] = (jw && v) ? (WSEP ? fk_gld(J.A.w, pc) : ra.q) : 1.0;
        gacc[r] = 0.0;
        actm[r] = __builtin_amdgcn_ballot_w64(v);
      }
      lox = fk_wave_min(lox); hix = -fk_wave_min(-hix);
      loy = fk_wave_min(loy); hiy = -fk_wave_min(-hiy);
      loz = fk_wave_min(loz); hiz = -fk_wave_min(-hiz);
      fk_wave_sync();
      if (lane == 0) { box[0] = lox; box[1] = hix; box[2] = loy; box[3] = hiy; box[4] = loz; box[5] = hiz; }
      fk_wave_sync();
      /* FP32 coordinates are relative to the centre of the box */
      const double tcx = 0.5 * (lox + hix), tcy = 0.5 * (loy + hiy), tcz = 0.5 * (loz + hiz);
      /* idle lanes: |a| = 1e18 and |dz| / s = 1 / (2 nmu), so that the mu
       * estimate of their pairs is 1/2, clear of the windows */
      const FkWin wn = J.win;
#pragma unroll
      for (int r = 0; r < R; r++) {
        const bool v = ai[r] != 0x7fffffff;
        fax[r] = v ? (float) (ax[r] - tcx) : wn.idle_x;
        fay[r] = v ? (float) (ay[r] - tcy) : 0.0f;
        faz[r] = v ? (float) (az[r] - tcz) : wn.idle_z;
      }
      /* survey FP32: m = a + b = 2 a' + d + 2 c (a' = a - c, c = the centre).
       * Idle lanes (a' = (10^6, 0, 0): s^2 and pi^2 far out of range) may
       * look ambiguous in mu: their queue bits are masked off */
      const float c2x = (float) (2.0 * tcx), c2y = (float) (2.0 * tcy), c2z = (float) (2.0 * tcz);
      const int nva = t.p1 - t.p0;

      /* FP32: FP64 re-evaluation of the n queued pairs of this wavefront */
      int qn = 0;
      unsigned kept = 0;          /* B objects evaluated (at most all of the call, in two images) */
      auto drain = [&]() __attribute__((always_inline)) {
        fk_wave_sync();
        const FkJob J = fk_cld(fk_again(a.jobs, cur));
        for (int e0 = 0; e0 < qn; e0 += 64) {
          if (e0 + lane < qn) {
            const int jg = (int) wqj[e0 + lane];
            const unsigned v = wqs[e0 + lane];
            const int p = t.p0 + (int) (v >> 5);
            unsigned idx;
            if (GEOM == FCFC_GEOM_SURVEY)
              idx = fk_recheck_sv<BIN, HYB>(bn, J, p, jg, stab, ptab, s2e, pe);
            else {
              const FkRec ra = fk_gld(J.A.rec, p);
              idx = fk_recheck<BIN, HYB, CENS>(bn, J, ra.x, ra.y, ra.z, jg, (int) (v & 31u), stab,
                                               ptab, s2e, pe, &ncensus);
            }
            nrecheck++;
            if (idx < ntot) {
              if (WT && jwt)
                atomicAdd(myhist_d + idx, WSEP ? fk_gld(J.A.w, p) * fk_gld(J.B.w, jg)
                                               : fk_gld(J.A.rec, p).q * fk_gld(J.B.rec, jg).q);
              else atomicAdd(myhist_u + idx, 1u);
            }
          }
        }
        qn = 0;
        fk_wave_sync();
      };

      /* one B object against the lane's A objects: FP64 coordinates, |r|^2 and
       * weight, or FP32 coordinates relative to the run's centre; jj its sorted
       * index, j its place in the chunk, code its periodic image */
      auto step = [&](auto selfc, double bx, double by, double bz, double bs, double wj, float gx,
                      float gy, float gz, int jj, int j, int code) __attribute__((always_inline)) {
        constexpr bool SELF = decltype(selfc)::value;
        if (MASKED) {
          double bsum = 0.0;        /* GRAD: sum of G[bin] w_a over this lane's pairs */
          auto add = [&](unsigned idx, int r) __attribute__((always_inline)) {
            if (GRAD) {
              const double gk = *(const double *) (lds + (ohist_g + 8u * idx));
              gacc[r] = __builtin_fma(gk, wj, gacc[r]);
              bsum = __builtin_fma(gk, aw[r], bsum);
            }
            else if (WT && jwt) atomicAdd((double *) (lds + (ohist_d + 8u * idx)), aw[r] * wj);
            else atomicAdd((unsigned int *) (lds + (ohist_u + 4u * idx)), 1u);
          };
          if (F32) {
            float ex[R], ey[R], ez[R], s2[R];
            bool in[R], any = false;
#pragma unroll
            for (int r = 0; r < R; r++) {
              ex[r] = gx - fax[r]; ey[r] = gy - fay[r]; ez[r] = gz - faz[r];
              if (BIN == FCFC_BIN_SPI) s2[r] = __builtin_fmaf(ey[r], ey[r], ex[r] * ex[r]);
              else if (SV32) s2[r] = __builtin_fmaf(ez[r], ez[r], __builtin_fmaf(ey[r], ey[r], ex[r] * ex[r]));
              else s2[r] = __builtin_fmaf(ey[r], ey[r], __builtin_fmaf(ex[r], ex[r], ez[r] * ez[r]));
              in[r] = s2[r] + wn.e_s2 < bn.m32s;
              if (BIN == FCFC_BIN_SPI) in[r] = in[r] & (__builtin_fabsf(ez[r]) + wn.e_pi < bn.m32p);
              if (SELF) in[r] = in[r] & (jj > ai[r]);
              any |= in[r];
            }
            if (__builtin_amdgcn_ballot_w64(any) == 0) return;
#pragma unroll
            for (int r = 0; r < R; r++) {
              bool amb = false;
              if (in[r]) {
                const float u = s2[r] + wn.e_s2;
                const unsigned e = stab_raw[(int) u];
                amb = __builtin_amdgcn_fractf(u) < __uint_as_float(e);
                unsigned idx = e & 0xFFFFu;
                if (BIN == FCFC_BIN_SPI) {
                  const float up = __builtin_fabsf(ez[r]) + wn.e_pi;
                  const unsigned ep = ptab_raw[(int) up];
                  amb |= __builtin_amdgcn_fractf(up) < __uint_as_float(ep);
                  idx += __umul24((unsigned) bn.nsh, ep & 0xFFFFu);
                }
                if (BIN == FCFC_BIN_SMU) {
                  bool ambm;
                  if (SV32) {
                    const float mx = __builtin_fmaf(2.0f, fax[r], ex[r]) + c2x;
                    const float my = __builtin_fmaf(2.0f, fay[r], ey[r]) + c2y;
                    const float mz = __builtin_fmaf(2.0f, faz[r], ez[r]) + c2z;
                    const float p = __builtin_fmaf(ez[r], mz, __builtin_fmaf(ey[r], my, ex[r] * mx));
                    const float m2 = __builtin_fmaf(mz, mz, __builtin_fmaf(my, my, mx * mx));
                    idx = fk_mu32(wn.nmu_f * __builtin_fabsf(p), __builtin_amdgcn_rsqf(m2 * s2[r]), idx,
                                  bn, wn, ambm);
                    amb |= m2 < wn.m2_floor;         /* near the observer */
                  }
                  else
                    idx = fk_mu32(wn.nmu_f * __builtin_fabsf(ez[r]), __builtin_amdgcn_rsqf(s2[r]), idx,
                                  bn, wn, ambm);
                  amb |= ambm;
                }
                if (!amb) add(idx, r);
              }
              /* pairs near an edge: queue (B object, A slot, image) for FP64 */
              const unsigned long long m = __builtin_amdgcn_ballot_w64(amb);
              if (__builtin_expect(m != 0, 0)) {
                if (amb) {
                  const int pos = qn + (int) __builtin_amdgcn_mbcnt_hi((unsigned) (m >> 32),
                                             __builtin_amdgcn_mbcnt_lo((unsigned) m, 0u));
                  wqj[pos] = (unsigned) (SELF ? jj : cj[j]);
                  wqs[pos] = (uint16_t) (((unsigned) (r * 64 + slot) << 5) | (unsigned) code);
                }
                qn += __popcll(m);
              }
            }
          }
          else {
            double s2[R], ez[R], dz2[R];
            bool in[R], any = false;
#pragma unroll
            for (int r = 0; r < R; r++) {
              if (GEOM == FCFC_GEOM_BOX) {
                const double ex = bx - ax[r], ey = by - ay[r];
                ez[r] = bz - az[r];
                dz2[r] = ez[r] * ez[r];
                if (BIN == FCFC_BIN_SPI) s2[r] = __builtin_fma(ey, ey, ex * ex);             /* :416-420 */
                else s2[r] = __builtin_fma(ey, ey, __builtin_fma(ex, ex, dz2[r]));           /* :426-430 */
              }
              else if (BIN == FCFC_BIN_ISO) {
                const double ex = ax[r] - bx, ey = ay[r] - by, e3 = az[r] - bz;
                s2[r] = __builtin_fma(e3, e3, __builtin_fma(ey, ey, ex * ex));
              }
              else {
                /* t (in dz2) and s^2 = s - t of the survey formulas (fk_sv64) */
                dz2[r] = __builtin_fma(az[r], bz, __builtin_fma(ay[r], by, ax[r] * bx)) * 2.0;
                s2[r] = (as[r] + bs) - dz2[r];
              }
              in[r] = s2[r] < bn.s2max;
              if (BIN == FCFC_BIN_SPI) in[r] = in[r] & (__builtin_fabs(ez[r]) < bn.pmax);
              /* the gradient reads no slot for a pair below the range: its zero
               * would make NaN of an infinite weight */
              if (MODE == MODE_GRADL) {
                in[r] = in[r] & (s2[r] >= bn.s2min);
                if (BIN == FCFC_BIN_SPI) in[r] = in[r] & (__builtin_fabs(ez[r]) >= bn.pmin);
              }
              if (SELF) in[r] = in[r] & (jj > ai[r]);
              any |= in[r];
            }
            if (__builtin_amdgcn_ballot_w64(any) == 0) return;
#pragma unroll
            for (int r = 0; r < R; r++) {
              if (!in[r]) continue;
              /* a survey s^2 may come out negative: slightly by rounding (bin 0,
               * as the reference's truncation gives), or far below -1 where
               * |r|^2 is huge or not that of the coordinates.  Either reads cell
               * 0, whose pairs all take the exact path, which drops the latter
               * (s2low; in the mask it cost the count of 1.2e6 objects 4 %) */
              const unsigned cell = stab[GEOM == FCFC_GEOM_SURVEY && BIN == FCFC_BIN_SMU
                                         ? fk_trunc_u32(s2[r]) : (unsigned) (int) s2[r]];
              if (BIN == FCFC_BIN_ISO) add(cell, r);
              else if (BIN == FCFC_BIN_SPI)
                add(cell + __umul24((unsigned) bn.nsh, ptab[(int) __builtin_fabs(ez[r])]), r);
              else {
                bool slow;
                unsigned idx;
                if (GEOM == FCFC_GEOM_BOX)
                  idx = fk_smu_index<false, MUT>(__builtin_fabs(ez[r]) * bn.nmu_d, __builtin_amdgcn_rsq(s2[r]),
                                                 [&] { return dz2[r] * bn.nmu2; }, s2[r], cell, bn, &slow);
                else {
                  const double d = as[r] - bs, m2 = dz2[r] + (as[r] + bs);
                  idx = fk_smu_index<true, MUT>(__builtin_fabs(d) * bn.nmu_d, __builtin_amdgcn_rsq(m2 * s2[r]),
                                                [&] { return ((d * d) / m2) * bn.nmu2; }, s2[r], cell, bn, &slow);
                }
                /* a mu that the exact path drops; the fast path has none (a
                 * survey value at its cap falls on the dummy row) */
                if (!slow || idx < ntot_o) add(idx, r);
              }
            }
          }
          if (GRAD && hasB) {
            /* the B object's share over the wavefront's pairs: one sum per
             * row of 16 lanes, added into the chunk's LDS accumulator */
            const double v = fk_row_sum(bsum);
            if ((lane & 15) == 0 && v != 0.0) atomicAdd(cb + j, v);
          }
          return;
        }
        if (GEOM == FCFC_GEOM_BOX) {
          /* when this B object is out of range of every A object of the run,
           * skip the binning (same expressions as the pair functions, so the
           * compiler shares them) */
          bool any = false;
#pragma unroll
          for (int r = 0; r < R; r++) {
            const double ex = bx - ax[r], ey = by - ay[r], ez = bz - az[r];
            if (BIN == FCFC_BIN_SPI)
              any |= (__builtin_fma(ey, ey, ex * ex) < bn.s2skip) &
                     (__builtin_fabs(ez) < bn.pskip);
            else any |= __builtin_fma(ey, ey, __builtin_fma(ex, ex, ez * ez)) < bn.s2skip;
          }
          if (__builtin_amdgcn_ballot_w64(any) == 0) return;
        }
        if (GEOM == FCFC_GEOM_SURVEY) {
          /* the same skip for survey pairs: |a - b|^2 (iso) or s - t
           * (= s^2 = s_perp^2 + pi^2) beyond the largest counted value */
          bool any = false;
#pragma unroll
          for (int r = 0; r < R; r++) {
            if (SV32) {
              const float ex = gx - fax[r], ey = gy - fay[r], ez = gz - faz[r];
              any |= __builtin_fmaf(ez, ez, __builtin_fmaf(ey, ey, ex * ex)) < bn.s2skip32;
            }
            else if (BIN == FCFC_BIN_ISO) {
              const double ex = ax[r] - bx, ey = ay[r] - by, ez = az[r] - bz;
              any |= __builtin_fma(ez, ez, __builtin_fma(ey, ey, ex * ex)) < bn.s2skip;
            }
            else {
              const double tt = __builtin_fma(az[r], bz, __builtin_fma(ay[r], by, ax[r] * bx)) * 2.0;
              any |= (as[r] + bs) - tt < bn.s2skip;
            }
          }
          if (__builtin_amdgcn_ballot_w64(any) == 0) return;
        }
        double bsum = 0.0;          /* GRAD: sum of G[bin] w_a over this lane's pairs */
#pragma unroll
        for (int r = 0; r < R; r++) {
          unsigned idx;
          bool queued = false;      /* FP32: left to the FP64 re-evaluation */
          if (F32) {
            bool amb, ambm, ambx;
            const float ex = gx - fax[r], ey = gy - fay[r], ez = gz - faz[r];
            idx = fk_sv32_spi(ex, ey, ez, __builtin_fmaf(2.0f, fax[r], ex) + c2x,
                              __builtin_fmaf(2.0f, fay[r], ey) + c2y,
                              __builtin_fmaf(2.0f, faz[r], ez) + c2z, bn, wn, stab_raw,
                              ptab_raw, amb, ambm, ambx);
            if (SELF) {
              const bool keep = jj > ai[r];
              amb = amb & keep; ambm = ambm & keep; idx = keep ? idx : FK_NONE;
            }
            /* pairs near an edge: queue (B object, A slot, image) for FP64.
             * The conditions are balloted apart (each ballot is its compare's
             * own mask) and the lane's bit is read back from the mask inside
             * the rare branch, so no lane value is kept across it */
            if (SELF) ambx = ambx & (jj > ai[r]);
            unsigned long long m = __builtin_amdgcn_ballot_w64(amb) |
                __builtin_amdgcn_ballot_w64(ambm) | __builtin_amdgcn_ballot_w64(ambx);
            m &= actm[r];
            if (__builtin_expect(m != 0, 0)) {
              if ((m >> lane) & 1ull) {
                const int pos = qn + (int) __builtin_amdgcn_mbcnt_hi((unsigned) (m >> 32),
                                           __builtin_amdgcn_mbcnt_lo((unsigned) m, 0u));
                wqj[pos] = (unsigned) (SELF ? jj : cj[j]);
                wqs[pos] = (uint16_t) (((unsigned) (r * 64 + slot) << 5) | (unsigned) code);
              }
              qn += __popcll(m);
            }
            queued = amb | ambm | ambx;
          }
          else if (GEOM == FCFC_GEOM_BOX)
            idx = fk_box64<BIN, HYB, false, PLAIN>(bx - ax[r], by - ay[r], bz - az[r], bn, stab,
                                                   ptab, s2e, pe);
          else
            idx = fk_sv64<BIN, HYB, PLAIN, false, QT>(ax[r], ay[r], az[r], as[r], bx, by, bz, bs,
                                                     bn, stab, ptab, s2e, pe, os_lds, op_lds);
          if (!F32 && SELF && !(jj > ai[r])) idx = FK_NONE;
          if (idx < ntot_o && !queued) {
            if (GRAD) {
              const double gk = *(const double *) (lds + (ohist_g + 8u * idx));
              gacc[r] = __builtin_fma(gk, wj, gacc[r]);
              bsum = __builtin_fma(gk, aw[r], bsum);
            }
            else if (WT && jwt) atomicAdd((double *) (lds + (ohist_d + 8u * idx)), aw[r] * wj);
            else atomicAdd((unsigned int *) (lds + (ohist_u + 4u * idx)), 1u);
          }
        }
        if (GRAD && hasB) {
          /* the B object's share over the wavefront's pairs: one sum per
           * row of 16 lanes, added into the chunk's LDS accumulator */
          const double v = fk_row_sum(bsum);
          if ((lane & 15) == 0 && v != 0.0) atomicAdd(cb + j, v);
        }
      };


      /* B objects [b0, b0 + n) of the other catalogue (SELF: of the run itself),
       * at the periodic image of code (IMG: not the object's own place) */
      auto segment = [&](auto selfc, auto imgc, int b0, int n, int code) __attribute__((always_inline)) {
        constexpr bool SELF = decltype(selfc)::value;
        constexpr bool IMG = decltype(imgc)::value;
        for (int c0 = SELF ? 0 : sq * FK_CH; c0 < n; c0 += SELF ? FK_CH : SQ * FK_CH) {
          const FkJob *pj = fk_again(a.jobs, cur);
          const FkCat B = fk_cld(SELF ? &pj->A : &pj->B);
          const FkGrid g = fk_cld(&pj->g);
          const double Dx = IMG ? (double) (code % 3 - 1) * g.Lx : 0.0;
          const double Dy = IMG ? (double) ((code / 3) % 3 - 1) * g.Ly : 0.0;
          const double Dz = IMG ? (double) (code / 9 - 1) * g.Lz : 0.0;
          const bool in = c0 + lane < n;
          const int jg = b0 + (in ? c0 + lane : 0);
          const FkRec rb = fk_gld(B.rec, jg);
          double x = rb.x, y = rb.y, z = rb.z;
          if (IMG) { x = x + Dx; y = y + Dy; z = z + Dz; }
          /* drop the objects beyond the maximum separation from the run's
           * bounding box (the grid's padded ranges) */
          bool keep = in;
          const double lx = box[0], hx = box[1], ly = box[2], hy = box[3], lz = box[4], hz = box[5];
          if (!SELF) {
            const double ex = __builtin_fmax(__builtin_fmax(lx - x, x - hx), 0.0);
            const double ey = __builtin_fmax(__builtin_fmax(ly - y, y - hy), 0.0);
            const double ez = __builtin_fmax(__builtin_fmax(lz - z, z - hz), 0.0);
            const double exy = __builtin_fma(ey, ey, ex * ex);
            if (g.hz_const >= 0) keep &= (exy < g.Rxy2) & (ez < g.hz_const);
            else keep &= __builtin_fma(ez, ez, exy) < g.R2;
          }
          unsigned long long m = __builtin_amdgcn_ballot_w64(keep);
          if (m == 0) continue;
          const int cnt = __popcll(m);
          kept += (unsigned) cnt;
          if (!GRAD && !jwt) {
            if (__builtin_expect(since + (unsigned) cnt * (unsigned) nva > FK_BUDGET, 0)) spill_counts();
            since += (unsigned) cnt * (unsigned) nva;
          }
          /* place in the chunk of a kept object */
          const int q = (int) __builtin_amdgcn_mbcnt_hi((unsigned) (m >> 32),
                                    __builtin_amdgcn_mbcnt_lo((unsigned) m, 0u));
          if (F32) {
            /* pack the kept objects into the wavefront's chunk */
            fk_wave_sync();
            if (keep) {
              fx[q] = (float) (x - 0.5 * (lx + hx));
              fy[q] = (float) (y - 0.5 * (ly + hy));
              fz[q] = (float) (z - 0.5 * (lz + hz));
              if (WT) cw[q] = jw ? (WSEP ? fk_gld(B.w, jg) : rb.q) : 1.0;
              cj[q] = jg;
            }
            /* NG > 1: up to a multiple of NG objects, out of range of all others */
            if (NG > 1 && lane < (-cnt & (NG - 1))) {
              fx[cnt + lane] = -1e18f;
              fy[cnt + lane] = fz[cnt + lane] = 0.0f;
              if (WT) cw[cnt + lane] = 0.0;
              cj[cnt + lane] = 0;
            }
            fk_wave_sync();
            for (int j = 0; j < cnt;) {
              /* while the queue has room for the pairs of one more object */
#pragma unroll 2
              for (; j < cnt; j += NG) {
                if (qn > FK_QCAP - 64 * R) break;
                const int q = j + sub;
                step(selfc, 0.0, 0.0, 0.0, 0.0, WT ? cw[q] : 1.0, fx[q], fy[q], fz[q],
                     SELF ? cj[q] : 0, q, code);
              }
              if (qn > FK_QCAP - 64 * R) drain();
            }
          }
          else {
            if (GRAD && hasB) { fk_wave_sync(); cb[lane] = 0.0; fk_wave_sync(); }
            if (NG > 1) {
              fk_wave_sync();
              if (keep) {
                cr[q] = FkRec{x, y, z, rb.q};
                if (WSEP && (WT || GRAD)) cw[q] = jw ? fk_gld(B.w, jg) : 1.0;
                cj[q] = jg;
              }
              if (lane < (-cnt & (NG - 1))) {
                cr[cnt + lane] = FkRec{-FK_FAR, -FK_FAR, -FK_FAR, NEED_S ? 3.0 * FK_FAR * FK_FAR : 0.0};
                if (WSEP && (WT || GRAD)) cw[cnt + lane] = 0.0;
                cj[cnt + lane] = 0;
              }
              fk_wave_sync();
#pragma unroll 2
              for (int j = sub; j < cnt + sub; j += NG) {
                const double px = cr[j].x, py = cr[j].y, pz = cr[j].z;
                const double pq = NEED_S || ((WT || GRAD) && !WSEP) ? cr[j].q : 0.0;
                double wj = 1.0;
                if (WT || GRAD) wj = WSEP ? cw[j] : (jw ? pq : 1.0);
                step(selfc, px, py, pz, pq, wj, 0.0f, 0.0f, 0.0f, SELF ? cj[j] : 0, j, code);
              }
            }
            else {
              /* the kept objects, one at a time, into scalar registers */
              typedef const __attribute__((address_space(4))) double cdouble;
              cdouble *rp = (cdouble *) (B.rec + b0 + c0);
              cdouble *wp = (cdouble *) (B.w + b0 + c0);
              unsigned long long k = m;
              while (k) {
                const int j = __builtin_ctzll(k);
                k &= k - 1;
                const double px = rp[4 * j], py = rp[4 * j + 1], pz = rp[4 * j + 2], pq = rp[4 * j + 3];
                double wj = 1.0;
                if (WSEP && (WT || GRAD)) { if (jw) wj = wp[j]; }
                else if (WT || GRAD) wj = jw ? pq : 1.0;
                step(selfc, IMG ? px + Dx : px, IMG ? py + Dy : py, IMG ? pz + Dz : pz,
                     NEED_S ? pq : 0.0, wj, 0.0f, 0.0f, 0.0f, SELF ? b0 + c0 + j : 0, j, code);
              }
            }
            /* GRAD: the B objects' shares go to the output */
            if (GRAD && hasB) {
              fk_wave_sync();
              if (keep) {
                const double v = cb[NG > 1 ? q : lane];
                if (v != 0.0) unsafeAtomicAdd(fk_cld(&fk_again(a.jobs, cur)->gB) + jg, v);
              }
            }
          }
        }
      };

      /* ---- auto counts: pairs inside the run (j > i), first item only ---- */
      if (J.autoc && part == 0 && sq == 0) {
        evals -= (unsigned long long) nva * (unsigned) nva / 2;
        segment(std::true_type(), std::false_type(), t.p0, nva, 13);
      }

      /* ---- strips, one per lane at a time ---- */
      for (int sb0 = s0; sb0 < s1; sb0 += 64) {
        int b0[FK_MAXSEG], len[FK_MAXSEG], code[FK_MAXSEG];
        {
          const int l = min(sb0 + lane, s1 - 1);
          const FkJob *pj = fk_again(a.jobs, cur);
          const int *sp = fk_cld(&pj->strips);
          fk_strip_segments(fk_cld(&pj->g), fk_cld(&pj->B.cell_start), t, box[4], box[5],
                            fk_gld(sp, 3 * l), fk_gld(sp, 3 * l + 1), fk_gld(sp, 3 * l + 2), b0, len, code);
          if (sb0 + lane >= s1) len[0] = len[1] = len[2] = 0;
        }
        unsigned long long m0 = __builtin_amdgcn_ballot_w64(len[0] > 0),
                           m1 = __builtin_amdgcn_ballot_w64(len[1] > 0),
                           m2 = __builtin_amdgcn_ballot_w64(len[2] > 0);
        while (m0 | m1 | m2) {
          int b, n, cd, q;
          if (m1) {
            q = __builtin_ctzll(m1); m1 &= m1 - 1;
            b = fk_lane_of(b0[1], q); n = fk_lane_of(len[1], q); cd = fk_lane_of(code[1], q);
          }
          else if (m0) {
            q = __builtin_ctzll(m0); m0 &= m0 - 1;
            b = fk_lane_of(b0[0], q); n = fk_lane_of(len[0], q); cd = fk_lane_of(code[0], q);
          }
          else {
            q = __builtin_ctzll(m2); m2 &= m2 - 1;
            b = fk_lane_of(b0[2], q); n = fk_lane_of(len[2], q); cd = fk_lane_of(code[2], q);
          }
          if (GEOM == FCFC_GEOM_SURVEY || (!F32 && cd == 13))
            segment(std::false_type(), std::false_type(), b, n, cd);
          else segment(std::false_type(), std::true_type(), b, n, cd);
        }
      }
      if (F32 && qn) drain();
      evals += (unsigned long long) kept * (unsigned) nva;

      if (GRAD) {
        double *gA = fk_cld(&fk_again(a.jobs, cur)->gA);
        if (gA)
#pragma unroll
          for (int r = 0; r < R; r++) {
            double v = gacc[r];
#pragma unroll
            for (int k = 32; k >= NA; k >>= 1) v += __shfl_xor(v, k);
            if (sub == 0 && ai[r] != 0x7fffffff && v != 0.0) unsafeAtomicAdd(gA + ai[r], v);
          }
      }
    }
  }

  /* statistics: summed over the workgroup, then in one of FK_STATS lines */
  __shared__ unsigned long long s_stat[3];
  if (tid < 3) s_stat[tid] = 0ull;
  __syncthreads();
  if (lane == 0) atomicAdd(&s_stat[0], evals);
  if (F32) {
    if (nrecheck) atomicAdd(&s_stat[1], (unsigned long long) nrecheck);
    if (ncensus) atomicAdd(&s_stat[2], (unsigned long long) ncensus);
  }
  __syncthreads();
  if (tid < 3 && s_stat[tid]) atomicAdd(a.stats + blockIdx.x % FK_STATS * (FK_LINE / 8) + tid, s_stat[tid]);
}

/* add a device histogram into the caller's device array */
__global__ void k_add_u64(long long *dst, const unsigned long long *src, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    dst[i] += (long long) src[i];
}
__global__ void k_add_f64(double *dst, const double *src, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    dst[i] += src[i];
}

/* ======================================================================== */
/*                                host side                                 */
/* ======================================================================== */

/* Device scratch of the no-allocation count (fcfc_gpu_count_noalloc): every
 * device buffer of such a call -- uploads of host catalogues, sorted copies,
 * cell and tiling arrays, histograms, queue and counters -- is carved from
 * this array.  Each GPU the library runs on holds its own copy until the
 * process ends.  In host code the name is only a stand-in: fcfc_gpu_init
 * resolves the address of the current GPU's copy with hipGetSymbolAddress
 * (once per device) and every host use goes through that address. */
#define FK_SCRATCH_BYTES ((size_t) 128 << 20)
#define FK_MAXDEV 64
#define FK_PIN_BYTES ((size_t) 1 << 20)     /* pinned at the start; grown to twice   */
#define FK_PIN_MOST ((size_t) 64 << 20)     /* what a call needs, up to this much    */
static __device__ __align__(256) unsigned char scratch[FK_SCRATCH_BYTES];
static void *g_scratch_ptr[FK_MAXDEV];
static std::mutex g_scratch_mu;

struct DevBuf { void *p = nullptr; size_t cap = 0; };

struct fcfc_gpu_ctx {
  int device = 0;
  int ncu = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  char err[512] = {0};
  fcfc_gpu_stats stats{};
  int t_cell_div = 0, t_tile = 0, t_zdiv = 0, t_nblock = 0;
  int t_nh = 0;                /* LDS histogram copies (0: by occupancy) */
  int census = 0;
  int tile_frac = 0;           /* autotuner: count about 1/tile_frac of the
                                  runs (16 stretches of the list) */
  int last_T = 0;              /* tile size of the last launch built */
  const int *last_nrun = nullptr;  /* device: runs of the last launch built */
  struct Tuned { int geom, bintype, mode, autoc, wt, bucket, cd, zd, T; };
  std::vector<Tuned> tuned;    /* autotuner results per density bucket */
  std::vector<DevBuf> bufs;
  char *pin = nullptr;         /* pinned host memory: a call's upload, then its results */
  size_t pin_cap = 0;
  /* histogram copies and workgroups per CU of a kernel at an LDS size */
  struct Occ { const void *fn; int lds1, nh, lds, occ; };
  std::vector<Occ> occs;
  void *scratch = nullptr;     /* device address of this GPU's scratch array */
  char scratch_err[128] = {0};
};

static void set_err(fcfc_gpu_ctx *c, const char *fmt, ...) {
  if (!c) return;
  va_list ap; va_start(ap, fmt);
  vsnprintf(c->err, sizeof c->err, fmt, ap);
  va_end(ap);
}

#define HIPCHK(ctx, call) do { hipError_t _e = (call); if (_e != hipSuccess) { \
    set_err(ctx, "%s failed: %s (%s:%d)", #call, hipGetErrorString(_e), __FILE__, __LINE__); \
    return FCFC_ERR_GPU; } } while (0)

/* Words of a call's results, zeroed before its launches: FK_STATS lines of
 * statistics (pairs evaluated, re-evaluated, of the census; the first line
 * also holds the flag of non-finite coordinates), the histograms, and after
 * them the queue. */
enum { RES_EVALS, RES_RECHECKED, RES_CENSUS, RES_BAD, RES_HIST = FK_STATS * (FK_LINE / 8) };
/* counters per job of a call */
static int queue_lines(int njob) { return njob <= 64 ? FK_GROUPS : 16; }
static size_t queue_words(int njob) { return (size_t) njob * queue_lines(njob) * (FK_LINE / 8); }

/* workspace slots */
enum {
  WS_IN_X, WS_IN_Y, WS_IN_Z, WS_IN_S, WS_IN_W,          /* uploads, catalogue A */
  WS_IN2_X, WS_IN2_Y, WS_IN2_Z, WS_IN2_S, WS_IN2_W,     /* uploads, catalogue B */
  WS_A_REC, WS_A_W, WS_A_IDX, WS_B_REC, WS_B_W, WS_B_IDX, WS_COUNT, WS_RANK, WS_SUMS, WS_GSTART, WS_ROWN, WS_ROWOFF, WS_TILES, WS_SPLITS,
  WS_RES, WS_UP, WS_BOX, WS_GA, WS_GB,
  WS_NSLOT
};

static void *ws(fcfc_gpu_ctx *c, int slot, size_t bytes, int *err) {
  if ((int) c->bufs.size() < WS_NSLOT) c->bufs.resize(WS_NSLOT);
  DevBuf &b = c->bufs[slot];
  if (bytes == 0) bytes = 8;
  if (b.cap < bytes) {
    if (b.p) { (void) hipStreamSynchronize(c->stream); (void) hipFree(b.p); b.p = nullptr; b.cap = 0; }
    size_t nb = bytes + bytes / 8 + 256;
    if (hipMalloc(&b.p, nb) != hipSuccess) {
      set_err(c, "hipMalloc of %zu bytes failed", nb);
      *err = FCFC_ERR_MEMORY;
      return nullptr;
    }
    b.cap = nb;
  }
  return b.p;
}

extern "C" int fcfc_gpu_init(fcfc_gpu_ctx **out, int device) {
  if (!out) return FCFC_ERR_ARG;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return FCFC_ERR_GPU;
  if (device < 0 || device >= ndev) return FCFC_ERR_ARG;
  fcfc_gpu_ctx *c = new (std::nothrow) fcfc_gpu_ctx();
  if (!c) return FCFC_ERR_MEMORY;
  c->device = device;
  if (hipSetDevice(device) != hipSuccess) { delete c; return FCFC_ERR_GPU; }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) != hipSuccess) { delete c; return FCFC_ERR_GPU; }
  c->ncu = prop.multiProcessorCount;
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess) {
    delete c; return FCFC_ERR_GPU;
  }
  /* address of this GPU's scratch array (no-allocation counts), resolved
   * once per device with the device current; a failure leaves the context
   * usable and makes fcfc_gpu_count_noalloc report it */
  if (device < FK_MAXDEV) {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
      void *p = nullptr;
      const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e == hipSuccess && p) g_scratch_ptr[device] = p;
      else snprintf(c->scratch_err, sizeof c->scratch_err, "hipGetSymbolAddress: %s",
                    hipGetErrorString(e));
    }
    c->scratch = g_scratch_ptr[device];
  }
  else snprintf(c->scratch_err, sizeof c->scratch_err, "device index beyond %d", FK_MAXDEV - 1);
  if (hipHostMalloc((void **) &c->pin, FK_PIN_BYTES, hipHostMallocDefault) == hipSuccess) c->pin_cap = FK_PIN_BYTES;
  else { c->pin = nullptr; (void) hipGetLastError(); }
  *out = c;
  return 0;
}

extern "C" int fcfc_gpu_destroy(fcfc_gpu_ctx *c) {
  if (!c) return 0;
  (void) hipSetDevice(c->device);
  if (c->stream) (void) hipStreamSynchronize(c->stream);
  for (auto &b : c->bufs) if (b.p) (void) hipFree(b.p);
  if (c->pin) (void) hipHostFree(c->pin);
  if (c->ev0) (void) hipEventDestroy(c->ev0);
  if (c->ev1) (void) hipEventDestroy(c->ev1);
  if (c->stream) (void) hipStreamDestroy(c->stream);
  delete c;
  return 0;
}

extern "C" const char *fcfc_gpu_last_error(const fcfc_gpu_ctx *c) {
  return c ? c->err : "no context";
}

extern "C" int fcfc_gpu_last_stats(const fcfc_gpu_ctx *c, fcfc_gpu_stats *st) {
  if (!c || !st) return FCFC_ERR_ARG;
  *st = c->stats;
  return 0;
}

extern "C" int fcfc_gpu_set_tuning(fcfc_gpu_ctx *c, int cell_div, int tile,
    int zdiv, int nblock) {
  if (!c) return FCFC_ERR_ARG;
  if (cell_div < 0 || cell_div > 32 || tile < 0 || tile > 4 * FK_NT || zdiv < 0 || zdiv > 64 || nblock < 0)
    return FCFC_ERR_ARG;
  c->t_cell_div = cell_div; c->t_tile = tile; c->t_zdiv = zdiv; c->t_nblock = nblock;
  return 0;
}

/* ---- per-job plan ------------------------------------------------------ */

/* groups of lanes of the kernels for sparse catalogues (NG of k_count) */
#define FK_NG 4
struct JobPlan {
  int bucket;       /* density bucket for the autotuner cache */
  FkGrid g;
  int T;            /* objects per tile (the FK_NW runs of a workgroup) */
  int zmaxc;        /* z-cells per block of a row: no run crosses blocks */
  int nblk;         /* blocks per row */
  double cand;      /* candidate B objects of one run in a uniform catalogue */
  int R;            /* objects per lane */
  int G;            /* lanes per A object (k_count) */
  int run;          /* objects of a run */
  int T_auto;       /* T chosen by the plan (not by the caller's tuning) */
  std::vector<int> strips;
  int nstrips;
};

static bool groups_keep_tables(const fcfc_bins *b, int mode, int wt);

static double max_sep2(const fcfc_bins *b, double *rxy2, double *hzc) {
  double s2max = b->s2bin[b->ns];
  *hzc = -1;
  if (b->bintype == FCFC_BIN_SPI) {
    double pm = b->pbin[b->np];
    if (b->geometry == FCFC_GEOM_BOX) {
      *rxy2 = s2max;
      *hzc = pm;
      return s2max + pm * pm;
    }
    /* survey: s^2 = s_perp^2 + pi^2 with pbin holding pi^2 */
    *rxy2 = s2max + pm;
    return s2max + pm;
  }
  *rxy2 = s2max;
  return s2max;
}

/* Side of the box that holds m objects of a catalogue of density nden with
 * extents ext: of a cube, where the extents have room for one, else of a slab
 * as thick as the catalogue, or a piece of a line.  (The cube of a plane
 * catalogue, its thickness 1e-6, is far too small: 1e6 objects in a plane to
 * 50 Mpc/h took 14.7 ms on cells of a twelfth of that, 0.67 on cells of 50.) */
static double box_side(double m, double nden, const double ext[3]) {
  double e[3] = {ext[0], ext[1], ext[2]};
  std::sort(e, e + 3);
  const double v = m / std::max(nden, 1e-300);
  double side = cbrt(v);
  if (side > e[0]) side = sqrt(v / e[0]);
  if (side > e[1]) side = v / (e[0] * e[1]);
  return side;
}

/* Build the grid geometry and strip list.  lo/hi: bounding box (survey);
 * groups: runs of 16 objects held by groups of lanes may be planned. */
static int make_plan(fcfc_gpu_ctx *c, const fcfc_bins *b, const double *bsize,
    const double lo[3], const double hi[3], int autoc, int wt, int mode, int64_t nA,
    int64_t nB, bool groups, JobPlan *P) {
  double rxy2, hzc;
  double r2 = max_sep2(b, &rxy2, &hzc);
  /* pad: the survey formula carries ~1e-10 absolute rounding in s^2 */
  const double pad = (b->geometry == FCFC_GEOM_SURVEY) ? 1e-6 : 1e-9;
  r2 = r2 * (1 + pad) + pad;
  rxy2 = rxy2 * (1 + pad) + pad;
  if (hzc >= 0) hzc = hzc * (1 + pad) + pad;
  const double R = sqrt(r2), Rxy = sqrt(rxy2);
  FkGrid &g = P->g;
  memset(&g, 0, sizeof g);
  g.R2 = r2; g.Rxy2 = rxy2; g.hz_const = hzc;
  /* objects per unit volume decides the default cell division */
  int cd = c->t_cell_div;
  int zd = c->t_zdiv;
  double vol;
  double ext[3];
  if (b->geometry == FCFC_GEOM_BOX) {
    for (int k = 0; k < 3; k++) ext[k] = bsize[k];
  }
  else {
    for (int k = 0; k < 3; k++) { ext[k] = hi[k] - lo[k]; if (!(ext[k] > 0)) ext[k] = 1e-6 * (1 + fabs(hi[k])); }
  }
  vol = ext[0] * ext[1] * ext[2];
  const double nden = (double) std::max<int64_t>(nB, 1) / vol;
  /* shapes picked by fcfc_gpu_autotune for this kind of job */
  /* density buckets (half octaves of objects per separation volume) of
   * B and of A: a tuned shape serves counts of the same kind only */
  const double ndenA = (double) std::max<int64_t>(nA, 1) / vol;
  const double rv = sqrt(rxy2) * sqrt(rxy2) * sqrt(r2);
  const int bucket = 4096 * (int) floor(2 * log2(nden * rv + 1e-300)) +
                     (int) floor(2 * log2(ndenA * rv + 1e-300));
  int tT = c->t_tile;
  if (cd <= 0 || zd <= 0 || tT <= 0) {
    for (const auto &t : c->tuned)
      if (t.geom == b->geometry && t.bintype == b->bintype && t.mode == mode &&
          t.autoc == autoc && t.wt == wt && t.bucket == bucket) {
        if (cd <= 0) cd = t.cd;
        if (zd <= 0) zd = t.zd;
        if (tT <= 0) tT = t.T;
        break;
      }
  }
  P->bucket = bucket;
  /* Objects per tile: two per lane, which halves the B objects read per pair,
   * unless a run of 128 objects is about as wide as the separations it is
   * counted to (sparse catalogues): then one (iso DD of 1e5 to 200 Mpc/h,
   * whose cube is half the separation: 0.39 against 0.36 ms). */
  P->T_auto = (tT <= 0);
  const double cube = box_side(128, ndenA, ext);
  if (tT > 0) P->T = std::min(tT, 4 * FK_NT);
  else P->T = cube > 0.75 * R ? FK_NT : 2 * FK_NT;
  P->R = (P->T + FK_NT - 1) / FK_NT;
  /* Sparser catalogues than that: runs of 16 objects, four groups of lanes
   * (k_count), unless B is far sparser than A (its strips then hold too few
   * objects for four groups).  Kernel ms, without and with: iso cross count
   * of 3e5 x 1e6 to 30 Mpc/h 1.10, 0.56; w_p of 1e6 to 40 Mpc/h 2.5, 1.8; iso
   * DD of 2e3 0.040, 0.026; box (s, mu) DD to 200 of the unit box of 1000:
   * n = 3e4 (cube / R = 0.81) 0.136, 0.103; 6e4 (0.64) 0.207, 0.185; 1.2e5
   * (0.51) weighted 0.55, 0.63; survey (s, mu) to 150 of 6e4 (0.86) 0.20,
   * 0.16; iso DD of 1e5 (0.54) 0.31, 0.42; DR of 6e3 x 6e4 (0.64) 0.087,
   * 0.12. */
  const bool can = groups && mode != MODE_P64 && !c->census &&
      !(b->geometry == FCFC_GEOM_SURVEY && b->bintype == FCFC_BIN_SPI);
  P->G = can && (P->T <= 64 / FK_NG || (P->T == FK_NT && cube > 0.75 * R && 8 * nden >= ndenA)) &&
      groups_keep_tables(b, mode, wt) ? FK_NG : 1;
  P->run = P->G > 1 ? 64 / P->G : 64 * P->R;
  /* Runs as compact as their object number allows: the objects of B within
   * the maximum separation of a run's bounding box are evaluated, and a cube
   * has the least of them.  The side of the cube that holds 128 objects of A
   * (32 for runs of 16) is the cell width in x and y (rounded to cells per
   * separation, one at least: thinner columns of a sparse catalogue would
   * only lengthen its runs), four z-cells per width.  Measured (kernel ms at
   * cd = 2, 3, 4, 6, 8): (s, mu) RR of 4e6 objects in the unit box 296, 245,
   * 232, 231, 230 (rule: 6); weighted DD of 5e5 9.1, 8.7, 8.9, 10.1, 12 (3);
   * iso DD of 1e5 0.36, 0.36, 0.55, 0.82, 1.2 (2); survey (s, mu) RR of 1.2e6
   * 16.6, 15.5, 16.4, 19.9, 25 (3). */
  const double width = P->G > 1 ? box_side(32, ndenA, ext) : cube;
  if (cd <= 0) cd = (int) std::min(std::max(floor(Rxy / width + 0.6), 1.0), 12.0);
  if (zd <= 0) zd = 4;
  /* cells of Rxy / cd, but never more cells than about 4 per object
   * (between 2^18 and 2^25): a sparse catalogue in a large volume gets
   * larger cells instead of a grid of mostly empty ones */
  const double cap = std::min(std::max(4.0 * (double) (nA + nB), 262144.0), 33554432.0);
  const double w_cap = cbrt(ext[0] * ext[1] * ext[2] * zd / cap);
  double w = std::max(Rxy / cd, w_cap);
  if (b->geometry == FCFC_GEOM_BOX) {
    g.periodic = 1;
    g.Lx = bsize[0]; g.Ly = bsize[1]; g.Lz = bsize[2];
    int n[2];
    for (int k = 0; k < 2; k++) {
      int nc = (int) floor(ext[k] / w);
      if (nc < 1) nc = 1;
      for (;;) {
        double wk = ext[k] / nc;
        int reach = (int) ceil(Rxy / wk);
        if (2 * reach + 1 <= nc) break;
        nc++;
        if (nc > 4096) { set_err(c, "separation range too close to half the box"); return FCFC_ERR_CFG; }
      }
      n[k] = nc;
    }
    g.ncx = n[0]; g.ncy = n[1];
    g.wx = ext[0] / g.ncx; g.wy = ext[1] / g.ncy;
    double wzt = std::min(g.wx, g.wy) / zd;
    /* z windows must stay shorter than the box: Lz - 2 R >= 4 wz */
    double zroom = ext[2] - 2 * (hzc >= 0 ? hzc : R);
    if (zroom <= 0) { set_err(c, "separation range not below half the box"); return FCFC_ERR_CFG; }
    if (wzt > zroom / 6) wzt = zroom / 6;
    g.ncz = std::max(1, (int) floor(ext[2] / wzt));
    g.wz = ext[2] / g.ncz;
    g.ox = g.oy = g.oz = 0;
  }
  else {
    g.periodic = 0;
    g.ncx = std::max(1, (int) ceil(ext[0] / w));
    g.ncy = std::max(1, (int) ceil(ext[1] / w));
    g.wx = w * (1 + 1e-12); g.wy = w * (1 + 1e-12);
    g.wz = w / zd;
    g.ncz = std::max(1, (int) ceil(ext[2] / g.wz) + 1);
    g.ox = lo[0]; g.oy = lo[1]; g.oz = lo[2];
    if ((double) g.ncx * g.ncy * g.ncz > 2.0e8) {
      set_err(c, "grid too large (%d x %d x %d cells)", g.ncx, g.ncy, g.ncz);
      return FCFC_ERR_CFG;
    }
  }
  /* blocks of about sixteen runs (the last run of a block is half empty on
   * average: four runs, (s, mu) DR 15.9 -> 15.1 ms), at least two cells wide:
   * the z extent of a run, and with it the FP32 windows, stays bounded in
   * sparse rows.  Four for the survey FP32 form, whose windows grow most
   * (more pairs re-evaluated: (s, mu) RR 15.6 against 16.5 ms). */
  const double nrb = (mode == MODE_C32 && b->geometry == FCFC_GEOM_SURVEY) ? 4.0 : 16.0;
  {
    const double per_cell = (double) nA / ((double) g.ncx * g.ncy * g.ncz);
    const double zc = std::max(2.0 * zd, ceil(nrb * P->run / std::max(per_cell, 1e-9)));
    P->zmaxc = (int) std::min((double) g.ncz, zc);
    P->nblk = (g.ncz + P->zmaxc - 1) / P->zmaxc;
  }
  /* strips */
  P->strips.clear();
  int kx = (int) ceil(Rxy / g.wx), ky = (int) ceil(Rxy / g.wy);
  if (!g.periodic) { kx = std::min(kx, g.ncx - 1); ky = std::min(ky, g.ncy - 1); }   /* rows there are */
  for (int dx = -kx; dx <= kx; dx++) {
    for (int dy = -ky; dy <= ky; dy++) {
      double gx = std::max(abs(dx) - 1, 0) * g.wx, gy = std::max(abs(dy) - 1, 0) * g.wy;
      if (gx * gx + gy * gy >= rxy2) continue;
      int diag = 0;
      if (autoc) {
        /* auto counts and their gradient: half plane, and on the own row
         * only the objects after the run */
        if (dx < 0 || (dx == 0 && dy < 0)) continue;
        if (dx == 0 && dy == 0) diag = 1;
      }
      P->strips.push_back(dx); P->strips.push_back(dy); P->strips.push_back(diag);
    }
  }
  P->nstrips = (int) P->strips.size() / 3;
  P->cand = 0;
  const double rlen = std::min(P->run / std::max(ndenA * g.wx * g.wy, 1e-300), ext[2]);
  for (int q = 0; q < P->nstrips; q++) {
    const double gx = std::max(abs(P->strips[3 * q]) - 1, 0) * g.wx;
    const double gy = std::max(abs(P->strips[3 * q + 1]) - 1, 0) * g.wy;
    const double hz = (hzc >= 0) ? hzc : sqrt(std::max(r2 - gx * gx - gy * gy, 0.0));
    P->cand += nden * g.wx * g.wy * std::min(2 * hz + rlen, ext[2]);
  }
  return 0;
}

/* sorted catalogue on the device: records, weights beside them (survey bins
 * with |r|^2) and original indices from its first object; obj0, cell0: its
 * place in the objects and cells of the call, cs: its cell starts, which
 * count objects of the call (set once the call's sort is queued) */
struct DevCat {
  int n = 0, obj0 = 0, cell0 = 0;
  FkRec *rec = nullptr;
  double *w = nullptr;
  int *idx = nullptr;
  const int *cs = nullptr;
  FkCat dev() const { return FkCat{n, 0, rec - obj0, w ? w - obj0 : nullptr,
                                   idx ? idx - obj0 : nullptr, cs}; }
};

/* A job ready to count: plan, sorted catalogues, output. */
struct PJob {
  JobPlan P;
  DevCat A, B;
  int autoc = 0, wt = 0;
  double *gA = nullptr, *gB = nullptr;
  long long hist_off = 0;
  int qi = 0;                   /* its place in the call's queue */
};

static inline int nblk(int64_t n, int bs) {
  int64_t b = (n + bs - 1) / bs;
  if (b < 1) b = 1;
  if (b > 65536) b = 65536;
  return (int) b;
}

/* Device memory of one call: the context's reusable workspace slots for a
 * single job, or allocations owned by the call (freed at its end) when many
 * jobs need their own sorted catalogues. */
struct Alloc {
  fcfc_gpu_ctx *c;
  bool own;
  std::vector<void *> blocks;
  char *cur = nullptr;         /* own: buffers are carved from 64 MiB chunks */
  size_t left = 0;             /* (a batch of hundreds of small catalogues   */
  int err = 0;                 /* would otherwise pay a hipMalloc per array) */
  char *arena = nullptr;       /* no-allocation calls: every buffer, the     */
  size_t arena_cap = 0;        /* temporaries included, is carved from the   */
  size_t arena_used = 0;       /* device scratch array; nothing is allocated */
  Alloc(fcfc_gpu_ctx *c_, bool own_) : c(c_), own(own_) {}
  ~Alloc() { for (void *p : blocks) (void) hipFree(p); }
  void use_arena(void *p, size_t cap) { arena = (char *) p; arena_cap = cap; arena_used = 0; own = false; }
  void *carve(size_t bytes) {
    bytes = (bytes + 255) & ~(size_t) 255;
    if (bytes > arena_cap - arena_used) {
      if (!err) set_err(c, "no-allocation count: its %zu-byte device scratch is exhausted "
                        "(%zu bytes in use, %zu more requested); count these catalogues "
                        "with fcfc_gpu_count", arena_cap, arena_used, bytes);
      err = FCFC_ERR_MEMORY;
      return nullptr;
    }
    void *r = arena + arena_used;
    arena_used += bytes;
    return r;
  }
  /* temporaries of one call (sort, tiling, histograms): the context's
   * reusable slots, or the arena */
  void *tmp(int slot, size_t bytes) {
    if (bytes == 0) bytes = 8;
    if (arena) return carve(bytes);
    return ws(c, slot, bytes, &err);
  }
  void *get(int slot, size_t bytes) {
    if (bytes == 0) bytes = 8;
    if (arena) return carve(bytes);
    if (!own) return ws(c, slot, bytes, &err);
    bytes = (bytes + 255) & ~(size_t) 255;
    if (bytes > left) {
      const size_t chunk = std::max(bytes, (size_t) 64 << 20);
      void *p = nullptr;
      if (hipMalloc(&p, chunk) != hipSuccess) {
        set_err(c, "hipMalloc of %zu bytes failed", chunk);
        err = FCFC_ERR_MEMORY;
        return nullptr;
      }
      blocks.push_back(p);
      cur = (char *) p;
      left = chunk;
    }
    void *r = cur;
    cur += bytes;
    left -= bytes;
    return r;
  }
};

__global__ void k_gather(int n, const int *__restrict__ idx, const double *__restrict__ src,
    double *__restrict__ dst, int stride) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    dst[(size_t) stride * i] = src[idx[i]];
}

/* sorted values into the original order.  The gradient kernel adds each B
 * object's share once per chunk and run, 64 neighbours of the sorted order at
 * a time: 8 lines where the original order has up to 64 (weight gradient of
 * DR, 4e4 x 2e5: 1.66 -> 1.54 ms). */
__global__ void k_unsort(int n, const int *__restrict__ idx, const double *__restrict__ src,
    double *__restrict__ dst) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    dst[idx[i]] = src[i];
}

__global__ void k_fill_f64(double *p, int64_t n, double v) {
  for (int64_t i = blockIdx.x * (int64_t) blockDim.x + threadIdx.x; i < n; i += (int64_t) gridDim.x * blockDim.x) p[i] = v;
}

__global__ void k_minmax(int n, const double *__restrict__ x, const double *__restrict__ y,
    const double *__restrict__ z, double *out) {
  __shared__ double sm[6][256];
  double v[6] = {1e300, 1e300, 1e300, -1e300, -1e300, -1e300};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    v[0] = fmin(v[0], x[i]); v[1] = fmin(v[1], y[i]); v[2] = fmin(v[2], z[i]);
    v[3] = fmax(v[3], x[i]); v[4] = fmax(v[4], y[i]); v[5] = fmax(v[5], z[i]);
  }
  for (int k = 0; k < 6; k++) sm[k][threadIdx.x] = v[k];
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int) threadIdx.x < s)
      for (int k = 0; k < 6; k++)
        sm[k][threadIdx.x] = (k < 3) ? fmin(sm[k][threadIdx.x], sm[k][threadIdx.x + s])
                                     : fmax(sm[k][threadIdx.x], sm[k][threadIdx.x + s]);
    __syncthreads();
  }
  /* out[8 + 6 b + q]: block b's minima (q < 3) and maxima (q >= 3); the
   * first 8 slots are not written */
  if (threadIdx.x < 6) out[8 + blockIdx.x * 6 + threadIdx.x] = sm[threadIdx.x][0];
}



/* Bounding box of one or two catalogues. */
static int bbox(fcfc_gpu_ctx *c, Alloc &al, const fcfc_cat *const *ks, int nk, double lo[3], double hi[3]) {
  const int nbk = 64, nd = 8 + 6 * nbk;
  double *d = nullptr;
  for (int q = 0; q < nk; q++) {
    const fcfc_cat *k = ks[q];
    if (k->n <= 0) continue;
    if (!k->on_device) {
      for (int64_t i = 0; i < k->n; i++) {
        const double v[3] = {k->x[i], k->y[i], k->z[i]};
        for (int m = 0; m < 3; m++) { lo[m] = fmin(lo[m], v[m]); hi[m] = fmax(hi[m], v[m]); }
      }
      continue;
    }
    if (!d) d = (double *) al.tmp(WS_BOX, sizeof(double) * 2 * nd);
    if (al.err) return al.err;
    hipLaunchKernelGGL(k_minmax, dim3(nbk), dim3(256), 0, c->stream, (int) k->n, k->x, k->y, k->z, d + q * nd);
  }
  if (!d) return 0;
  std::vector<double> hv;
  double *h = (double *) c->pin;
  if (c->pin_cap < sizeof(double) * 2 * nd) { hv.resize(2 * nd); h = hv.data(); }
  HIPCHK(c, hipMemcpyAsync(h, d, sizeof(double) * 2 * nd, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  for (int q = 0; q < nk; q++) {
    if (ks[q]->n <= 0 || !ks[q]->on_device) continue;
    for (int bk = 0; bk < nbk; bk++)
      for (int m = 0; m < 3; m++) {
        lo[m] = fmin(lo[m], h[q * nd + 8 + bk * 6 + m]);
        hi[m] = fmax(hi[m], h[q * nd + 8 + bk * 6 + 3 + m]);
      }
  }
  return 0;
}

/* What a call uploads besides catalogues -- sort requests, tables, strips,
 * job descriptors -- gathered in (pinned) host memory and copied at once.  The
 * device addresses are known as soon as something is put. */
struct Upload {
  fcfc_gpu_ctx *c;
  char *h = nullptr, *d = nullptr;
  size_t cap = 0, used = 0;
  std::vector<char> own;
  explicit Upload(fcfc_gpu_ctx *c_) : c(c_) {}
  int reserve(Alloc &al, size_t bytes, bool plan) {
    cap = (bytes + 255) & ~(size_t) 255;
    d = (char *) al.get(WS_UP, cap);
    if (al.err) return al.err;
    if (!plan && pin_fit(c, cap, al.arena != nullptr)) h = c->pin;
    else { own.resize(cap); h = own.data(); }
    return 0;
  }
  /* room for bytes of pinned memory in the context (grown when allowed) */
  static bool pin_fit(fcfc_gpu_ctx *c, size_t bytes, bool fixed) {
    if (bytes <= c->pin_cap) return true;
    if (fixed || bytes > FK_PIN_MOST) return false;
    char *p = nullptr;
    if (hipStreamSynchronize(c->stream) != hipSuccess ||
        hipHostMalloc((void **) &p, 2 * bytes, hipHostMallocDefault) != hipSuccess) {
      (void) hipGetLastError();
      return false;
    }
    if (c->pin) (void) hipHostFree(c->pin);
    c->pin = p;
    c->pin_cap = 2 * bytes;
    return true;
  }
  template <class T> T *put(const T *src, size_t n) {
    const size_t bytes = (sizeof(T) * n + 15) & ~(size_t) 15;
    if (used + bytes > cap) return nullptr;
    memcpy(h + used, src, sizeof(T) * n);
    T *r = (T *) (d + used);
    used += bytes;
    return r;
  }
  int flush() {
    if (used) HIPCHK(c, hipMemcpyAsync(d, h, used, hipMemcpyHostToDevice, c->stream));
    return 0;
  }
};

/* Prepare the sort of one catalogue into the grid of a job: upload host
 * inputs, allocate the sorted copies (so the job's descriptors can point
 * at them at once) and queue the work for stage_run.  slot: first of 3
 * consecutive workspace slots (single-job calls). */
static int stage_prep(fcfc_gpu_ctx *c, Alloc &al, const fcfc_cat *k, int need_s,
    int wt, int need_idx, const FkGrid &g, int slot, int upslot, DevCat *out, std::vector<FkStage> &st) {
  const int n = (int) k->n;
  const size_t nb = sizeof(double) * (size_t) (n > 0 ? n : 1);
  /* inputs on the device */
  const double *x = k->x, *y = k->y, *z = k->z, *s = need_s ? k->s : nullptr, *w = wt ? k->w : nullptr;
  if (!k->on_device && n > 0) {
    double *dx = (double *) al.get(upslot + 0, nb), *dy = (double *) al.get(upslot + 1, nb),
           *dz = (double *) al.get(upslot + 2, nb);
    if (al.err) return al.err;
    HIPCHK(c, hipMemcpyAsync(dx, k->x, nb, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(dy, k->y, nb, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(dz, k->z, nb, hipMemcpyHostToDevice, c->stream));
    x = dx; y = dy; z = dz;
    if (s) {
      double *ds = (double *) al.get(upslot + 3, nb);
      if (al.err) return al.err;
      HIPCHK(c, hipMemcpyAsync(ds, k->s, nb, hipMemcpyHostToDevice, c->stream));
      s = ds;
    }
    if (w) {
      double *dw = (double *) al.get(upslot + 4, nb);
      if (al.err) return al.err;
      HIPCHK(c, hipMemcpyAsync(dw, k->w, nb, hipMemcpyHostToDevice, c->stream));
      w = dw;
    }
  }
  const size_t no = (size_t) (n > 0 ? n : 1);
  out->n = n;
  out->rec = (FkRec *) al.get(slot + 0, sizeof(FkRec) * no);
  out->w = (need_s && wt) ? (double *) al.get(slot + 1, nb) : nullptr;
  out->idx = need_idx ? (int *) al.get(slot + 2, sizeof(int) * no) : nullptr;
  if (al.err) return al.err;
  FkStage q;
  memset(&q, 0, sizeof q);
  q.n = n; q.need_s = need_s; q.wt = wt; q.g = g;
  q.x = x; q.y = y; q.z = z; q.s = s; q.w = w;
  q.rec = out->rec; q.ow = out->w; q.oidx = out->idx;
  if (!st.empty()) {
    const FkStage &p = st.back();
    const long long nc = p.cell0 + (long long) p.g.ncx * p.g.ncy * p.g.ncz;
    const long long nobj = (long long) p.obj0 + p.n;
    if (nobj + n > INT_MAX / 2 || nc + (long long) g.ncx * g.ncy * g.ncz > INT_MAX / 2) {
      set_err(c, "catalogues of one call too large");
      return FCFC_ERR_CFG;
    }
    q.obj0 = (int) nobj;
    q.cell0 = (int) nc;
  }
  out->obj0 = q.obj0;
  out->cell0 = q.cell0;
  st.push_back(q);
  return 0;
}

/* exclusive scan of in[0..n-1] into out[0..n] */
static int scan(fcfc_gpu_ctx *c, Alloc &al, const int *in, int *out, int n) {
  const int nb = std::max(1, (n + FK_SCAN - 1) / FK_SCAN);
  int *sums = nb > 1 ? (int *) al.tmp(WS_SUMS, sizeof(int) * (size_t) nb) : nullptr;
  if (al.err) return al.err;
  if (nb > 1) hipLaunchKernelGGL(k_scan_sum, dim3(nb), dim3(1024), 0, c->stream, in, n, sums);
  hipLaunchKernelGGL(k_scan_out, dim3(nb), dim3(1024), 0, c->stream, in, out, n, sums);
  return 0;
}

/* The queued sorts of a call: one launch per stage for all of them.  The
 * cell starts of all catalogues come from one scan and stay where it leaves
 * them (cs of every job). */
struct Sort {
  int nobj = 0, ncell = 0, nst = 0;
  FkStage *st = nullptr;             /* uploaded requests */
  int *count = nullptr, *gstart = nullptr, *rank = nullptr;
};

static int sort_alloc(fcfc_gpu_ctx *c, Alloc &al, const std::vector<FkStage> &st,
    std::vector<PJob> &jobs, Sort *so) {
  if (st.empty()) return 0;
  const FkStage &last = st.back();
  const long long ncl = last.cell0 + (long long) last.g.ncx * last.g.ncy * last.g.ncz;
  if ((long long) last.obj0 + last.n > INT_MAX / 2 || ncl > INT_MAX / 2) {
    set_err(c, "catalogues of one call too large");
    return FCFC_ERR_CFG;
  }
  so->nobj = last.obj0 + last.n;
  so->ncell = (int) ncl;
  so->nst = (int) st.size();
  so->count = (int *) al.tmp(WS_COUNT, sizeof(int) * (size_t) so->ncell);
  so->gstart = (int *) al.get(WS_GSTART, sizeof(int) * ((size_t) so->ncell + 1));
  so->rank = (int *) al.tmp(WS_RANK, sizeof(int) * (size_t) std::max(so->nobj, 1));
  if (al.err) return al.err;
  for (PJob &J : jobs) { J.A.cs = so->gstart + J.A.cell0; J.B.cs = so->gstart + J.B.cell0; }
  return 0;
}

/* zero the call's result words and sort its catalogues */
static int sort_run(fcfc_gpu_ctx *c, Alloc &al, const Sort &so, unsigned long long *res, size_t nres) {
  hipLaunchKernelGGL(k_zero_call, dim3(nblk(std::max<int64_t>(nres, so.ncell), 256)), dim3(256), 0,
                     c->stream, res, nres, so.count, (size_t) so.ncell);
  if (so.nobj > 0)
    hipLaunchKernelGGL(k_stage_assign, dim3(nblk(so.nobj, 256)), dim3(256), 0, c->stream, so.nobj,
                       so.nst, so.st, so.count, so.rank, res + RES_BAD);
  if (int e = scan(c, al, so.count, so.gstart, so.ncell)) return e;
  if (so.nobj > 0)
    hipLaunchKernelGGL(k_stage_scatter, dim3(nblk(so.nobj, 256)), dim3(256), 0, c->stream, so.nobj,
                       so.nst, so.st, so.gstart, so.rank);
  HIPCHK(c, hipGetLastError());
  return 0;
}

/* the kernels with a masked pair loop (see k_count) */
static bool masked_form(const fcfc_bins *b, int mode, int hyb) {
  if (b->geometry == FCFC_GEOM_SURVEY && b->bintype == FCFC_BIN_SPI) return false;
  return mode == MODE_C32 || (!hyb && mode != MODE_P64);
}

/* LDS histogram geometry: an odd row stride (rows of mu or pi bins), see
 * fk_hslot.  Masked forms whose tables have entries below the s range need a
 * column beyond ns for them, and a dummy row for pi below the range and for
 * survey mu values at their ceiling. */
struct HistDim { int nsh, ntoh, nslot; };
static HistDim hist_dim(const fcfc_bins *b, int mode, int hyb) {
  HistDim h;
  const bool msk = masked_form(b, mode, hyb);
  if (msk && b->soff > 0) h.nsh = (b->ns + 1) | 1;
  else h.nsh = b->bintype == FCFC_BIN_ISO ? b->ns : (b->ns | 1);
  h.ntoh = h.nsh * (b->ntot / b->ns);
  const bool dummy = (b->bintype == FCFC_BIN_SPI && b->poff > 0) ||
      (b->bintype == FCFC_BIN_SMU && b->geometry == FCFC_GEOM_SURVEY);
  h.nslot = h.ntoh + (msk && dummy ? h.nsh : 0);
  return h;
}

struct LdsPlan { int off_hist, off_stab, off_ptab, off_edges, off_chunk, off_queue, total, nh, stab_c0, ptab_c0; };

static int align16(int v) { return (v + 15) & ~15; }

/* Table entries staged before cell 0: the integer tables and every FP32
 * table are zero-based (entry k is the one of (int) s2 = k, so the lookup
 * needs no lower range check), the hybrid tables of the FP64 forms keep one
 * sentinel.  A zero-based table costs 4 bytes per entry below s2min; tables
 * that start beyond FK_ZB_MAXOFF entries run through the hybrid lookups
 * instead, which check the range against the edges and give the same bins
 * for integer edges. */
#define FK_ZB_MAXOFF 4096
static bool zb_fits(const fcfc_bins *b) {
  return b->soff <= FK_ZB_MAXOFF && (b->bintype != FCFC_BIN_SPI || b->poff <= FK_ZB_MAXOFF);
}

static LdsPlan lds_plan(const fcfc_bins *b, int mode, int wt, int need_s, int nh, int hyb,
    int ssearch = 0, int psearch = 0, int G = 1) {
  LdsPlan L;
  int o = 0;
  L.nh = nh;
  L.off_hist = o;
  const int nslot = hist_dim(b, mode, hyb).nslot;
  if (mode == MODE_GRAD) o += nslot * 8;
  else o += nh * nslot * (wt ? 8 : 4);
  o = align16(o);
  L.off_edges = o;
  if (hyb) o = align16(o + 8 * (b->ns + 1 + (b->bintype == FCFC_BIN_SPI ? b->np + 1 : 0)));
  L.off_chunk = o;
  const bool f32 = (mode == MODE_C32), grad = (mode == MODE_GRAD);
  o = align16(o + FK_NW * FK_CH * fk_chunk_bytes(f32, wt, grad, need_s, G));
  L.off_queue = o;
  if (f32) o += FK_NW * FK_QCAP * 6;
  o = align16(o);
  const int zero_based = (!hyb || mode == MODE_C32);
  L.stab_c0 = zero_based ? b->soff : 1;
  L.ptab_c0 = zero_based ? b->poff : 1;
  /* two entries after the last cell (four for the survey (s_perp, pi)
   * tables of the FP64 forms, which start at floor cell -2) */
  L.off_stab = o; o = align16(o + (L.stab_c0 + (ssearch ? 0 : b->stab_len) + 4) * 4);
  L.off_ptab = o;
  if (b->bintype == FCFC_BIN_SPI)
    o = align16(o + (L.ptab_c0 + (psearch ? 0 : b->ptab_len) + 4) * 4);
  L.total = o;
  return L;
}

/* dynamic LDS of a workgroup: all but the 412 bytes of k_count's own arrays */
#define FK_LDS_MOST (160 * 1024 - 512)

/* does a plan fit?  (The unused slots of the masked forms come out of the
 * margin.) */
static bool lds_fits(const fcfc_bins *b, const LdsPlan &P, int mode, int hyb) {
  return P.total <= (masked_form(b, mode, hyb) ? FK_LDS_MOST : 160 * 1024 - 2048);
}

/* Form and tables of a count of this mode, with G groups of lanes.  FP32
 * tables are zero-based, and the fixed-point mu value of that form holds
 * t <= nmu (1 + 2^-20) below 127: other binnings run in FP64.  Tables too long
 * for LDS (hybrid binnings rescaled to large integers) are replaced by hybrid
 * lookups that binary-search the edges, in the FP64 forms. */
struct TabForm {
  int m, hyb, ssearch, psearch;
  bool fits;
  bool operator==(const TabForm &o) const {
    return m == o.m && hyb == o.hyb && ssearch == o.ssearch && psearch == o.psearch && fits == o.fits;
  }
};
static TabForm table_form(const fcfc_bins *b, int mode, int wt, int G) {
  const int need_s = (b->geometry == FCFC_GEOM_SURVEY && b->bintype != FCFC_BIN_ISO);
  const bool zb = zb_fits(b);
  TabForm f = {mode, (b->tabtype || !zb) ? 1 : 0, 0, 0, true};
  if (f.m == MODE_C32 && (!zb || (b->bintype == FCFC_BIN_SMU && b->nmu > FK_NMU32))) f.m = MODE_C64;
  auto fit = [&]() {
    return lds_fits(b, lds_plan(b, f.m, wt, need_s, 1, f.hyb, f.ssearch, f.psearch, G), f.m, f.hyb);
  };
  if (!fit()) {
    if (f.m == MODE_C32) f.m = MODE_C64;
    f.hyb = 1;
    f.ssearch = 1;
    if (!fit()) f.psearch = 1;
    f.fits = fit();
  }
  return f;
}

/* The chunks of the groups of lanes take 18 KB or more of LDS: they must not
 * cost a binning its tables (tables that do not fit without them either are
 * searched in any case, and the search needs next to no LDS: a w_p count of
 * 1e6 objects 1.8 ms in groups and 2.5 without). */
static bool groups_keep_tables(const fcfc_bins *b, int mode, int wt) {
  return table_form(b, mode, wt, FK_NG) == table_form(b, mode, wt, 1);
}

typedef void (*kfn_t)(const FkArgs);

/* Kernel variants: binning x geometry x weights x mode x table type x A
 * objects per lane (R = 1: tiles of FK_NT objects, R = 2: 2 FK_NT, R = 4:
 * 4 FK_NT).  The gradient with hybrid tables uses R = 1; R = 4 exists for
 * the weighted FP64 box counts with integer tables only and for callers that
 * set such tiles (fk_lanes_max gives the largest R of a kernel family).  The
 * survey kernels hold four more FP64 values per object and spill at R = 4
 * (weighted (s_perp, pi) DR: 950 ms against 830 at R = 2). */
static int fk_lanes_max(int geom, int mode, int wt, int hyb) {
  if (hyb && mode == MODE_GRAD) return 1;
  if (hyb) return 2;
  return (wt && mode == MODE_C64 && geom == FCFC_GEOM_BOX) ? 4 : 2;
}

template <int BIN, int GEOM, bool WT, int MODE>
static kfn_t pick5(int hyb, int R, int G) {
  if constexpr ((MODE == MODE_C64 || MODE == MODE_C32 || MODE == MODE_GRAD) &&
                !(GEOM == FCFC_GEOM_SURVEY && BIN == FCFC_BIN_SPI))
    if (G > 1)
      return hyb ? k_count<BIN, GEOM, WT, MODE, true, 1, FK_NG> : k_count<BIN, GEOM, WT, MODE, false, 1, FK_NG>;
  if constexpr (MODE == MODE_GRAD) {
    if (hyb) return k_count<BIN, GEOM, WT, MODE, true, 1>;
    return R == 1 ? k_count<BIN, GEOM, WT, MODE, false, 1> : k_count<BIN, GEOM, WT, MODE, false, 2>;
  }
  else {
    if (hyb) return R == 1 ? k_count<BIN, GEOM, WT, MODE, true, 1> : k_count<BIN, GEOM, WT, MODE, true, 2>;
    if constexpr (WT && MODE == MODE_C64 && GEOM == FCFC_GEOM_BOX)
      if (R == 4) return k_count<BIN, GEOM, WT, MODE, false, 4>;
    return R == 1 ? k_count<BIN, GEOM, WT, MODE, false, 1> : k_count<BIN, GEOM, WT, MODE, false, 2>;
  }
}

template <int BIN, int GEOM>
static kfn_t pick3(int wt, int mode, int hyb, int R, int G) {
  if constexpr (!(GEOM == FCFC_GEOM_SURVEY && BIN == FCFC_BIN_SPI))
    if (mode == MODE_GRADL) {
      if (G > 1) return k_count<BIN, GEOM, true, MODE_GRADL, false, 1, FK_NG>;
      return R == 1 ? k_count<BIN, GEOM, true, MODE_GRADL, false, 1> : k_count<BIN, GEOM, true, MODE_GRADL, false, 2>;
    }
  if (mode == MODE_GRAD) return pick5<BIN, GEOM, true, MODE_GRAD>(hyb, R, G);
  if (mode == MODE_C32)
    return wt ? pick5<BIN, GEOM, true, MODE_C32>(hyb, R, G) : pick5<BIN, GEOM, false, MODE_C32>(hyb, R, G);
  if constexpr (GEOM == FCFC_GEOM_BOX) {
    if (mode == MODE_C32C)
      return wt ? pick5<BIN, GEOM, true, MODE_C32C>(hyb, R, G) : pick5<BIN, GEOM, false, MODE_C32C>(hyb, R, G);
  }
  if (mode == MODE_P64)
    return wt ? pick5<BIN, GEOM, true, MODE_P64>(hyb, R, G) : pick5<BIN, GEOM, false, MODE_P64>(hyb, R, G);
  return wt ? pick5<BIN, GEOM, true, MODE_C64>(hyb, R, G) : pick5<BIN, GEOM, false, MODE_C64>(hyb, R, G);
}

static kfn_t pick_kernel(int bintype, int geom, int wt, int mode, int hyb, int R, int G) {
  if (geom == FCFC_GEOM_BOX) {
    if (bintype == FCFC_BIN_ISO) return pick3<FCFC_BIN_ISO, FCFC_GEOM_BOX>(wt, mode, hyb, R, G);
    if (bintype == FCFC_BIN_SMU) return pick3<FCFC_BIN_SMU, FCFC_GEOM_BOX>(wt, mode, hyb, R, G);
    return pick3<FCFC_BIN_SPI, FCFC_GEOM_BOX>(wt, mode, hyb, R, G);
  }
  if (bintype == FCFC_BIN_ISO) return pick3<FCFC_BIN_ISO, FCFC_GEOM_SURVEY>(wt, mode, hyb, R, G);
  if (bintype == FCFC_BIN_SMU) return pick3<FCFC_BIN_SMU, FCFC_GEOM_SURVEY>(wt, mode, hyb, R, G);
  return pick3<FCFC_BIN_SPI, FCFC_GEOM_SURVEY>(wt, mode, hyb, R, G);
}

/* FP32 exactness windows.  With coordinates relative to the A run's centre
 * c, each FP32 difference satisfies |d32 - d| <= u (2|d| + E) + tiny
 * (u = 2^-24, E = run extent), so
 *   |s2_32 - s2| <= 7 u s2 + 2 sqrt(3) u E s + 3 (u (2 s + E))^2,
 * evaluated at the largest in-range s^2 (plus the first integer above it:
 * beyond that the table answers "outside" without a window).  The mu bin
 * floor(t), t = nmu |dz| / s, has |t32 - t| <= t 10u + (sqrt(3) u E t +
 * nmu u E) / s; with s^2 >= s2_floor (fp32_s2_floor) and t <= nmu this is
 * a constant D, and the bin is certain when |fract(t32) - 1/2| <= 1/2 - D.
 * All bounds are inflated by 25%; pairs below s2_floor are always
 * re-evaluated.
 *
 * Survey pairs (fk_sv32_spi) add two things.  The reference's own values carry
 * the rounding of its FP64 formulas: s^2 = (|a|^2 + |b|^2) - 2 a.b is off
 * the exact value by at most about 8 eps R^2 (R = largest |r| of the grid,
 * eps = 2^-53, |r|^2 given with 2 eps), and its pi = (|a|^2 - |b|^2) / |m|
 * by 5 eps R^2 / |m| (m = a + b).  And the FP32 m = (2 a' + d) + 2 c (c the
 * run's centre, a' = a - c) has error |dm| <= 2u|c| + 2 sqrt(3) ek + 2u|m| +
 * 2uE (ek = u (2 s + E) + tiny, 2|c| <= |m| + s + E), so p = d.m is off by
 * at most |m| (sqrt(3) ek + 6 u s) + s (u (s + 3E) + 2 sqrt(3) ek) and pi
 * by e_pi = sqrt(3) ek + 6 u s + s (u (s + 3E) + 2 sqrt(3) ek) / |m|.  With |m|^2 >= m2_floor (smaller |m| is re-evaluated) these are
 * constants: the pi^2 window is 2 pi e_pi + e_pi^2 + pi^2 (relative error of
 * |m|^2, 4u of the reciprocal, 2u of the products) plus the reference's
 * terms, the s_perp^2 window the sum of the s^2 and pi^2 windows plus the
 * rounding of the difference, and the mu window (t = nmu |p| / (|m| s))
 * gets e_pi / s plus half the relative errors of s^2 and |m|^2 and 8u for
 * the reciprocal square root of |m|^2 s^2 and that product. */
static double fp32_extent(const FkGrid &g, int zmaxc) {
  return std::max(g.wx, std::max(g.wy, (zmaxc + 1) * g.wz));
}

static void fp32_windows(const fcfc_bins *b, const FkGrid &g, int zmaxc, double s2f,
    FkWin *win);

/* s^2 below which a job's pairs are always re-evaluated (the LDS table flags
 * those cells once per launch, so a launch uses the largest over its jobs).
 * For (s, mu) bins the floor trades the pairs below it -- about
 * ((floor + 1) / s2max)^(3/2) of a uniform catalogue's in-range pairs,
 * counting the flagged cell above it -- against the mu windows, 2 D of the
 * pairs above it with D growing as 1 / sqrt(floor): the candidate with the
 * fewest expected re-evaluations is taken. */
static double fp32_s2_floor(const fcfc_bins *b, const FkGrid &g, int zmaxc) {
  const double u = ldexp(1.0, -24);
  const double s2max = b->s2bin[b->ns];
  const double lo = pow(1e4 * u * fp32_extent(g, zmaxc), 2);
  if (b->bintype != FCFC_BIN_SMU) return std::max(s2max / 64.0, lo);
  double best = std::max(s2max / 64.0, lo), bcost = 1e300;
  for (double x = 1.0 / 64; x >= 1.0 / 16384; x *= 0.5) {
    const double s2f = std::max(x * s2max, lo);
    FkWin w;
    fp32_windows(b, g, zmaxc, s2f, &w);
    const double cost = pow(std::min((s2f + 1) / s2max, 1.0), 1.5) + 2.0 * w.mu_sh;
    if (cost < bcost) { bcost = cost; best = s2f; }
  }
  return best;
}

/* largest |r| of a survey grid (its corners) */
static double grid_rmax(const FkGrid &g) {
  double r2 = 0;
  for (int k = 0; k < 8; k++) {
    const double x = (k & 1) ? g.ox + g.ncx * g.wx : g.ox;
    const double y = (k & 2) ? g.oy + g.ncy * g.wy : g.oy;
    const double z = (k & 4) ? g.oz + g.ncz * g.wz : g.oz;
    r2 = std::max(r2, x * x + y * y + z * z);
  }
  return sqrt(r2);
}

static void fp32_windows(const fcfc_bins *b, const FkGrid &g, int zmaxc, double s2f,
    FkWin *win) {
  const double u = ldexp(1.0, -24), eps = ldexp(1.0, -53);
  const bool sv = (b->geometry == FCFC_GEOM_SURVEY);
  const double s2max = b->s2bin[b->ns];
  /* box (s_perp, pi): pbin holds pi edges; survey: pi^2 edges */
  const double pmx = (b->bintype == FCFC_BIN_SPI) ? b->pbin[b->np] : 0;
  const double S2 = s2max + (sv ? pmx : pmx * pmx) + 2.0;
  const double s = sqrt(S2);
  const double E = fp32_extent(g, zmaxc);
  const double R = sv ? grid_rmax(g) : 0.0;
  const double tiny = ldexp(1.0, -44) * std::max(std::max(g.Lx, std::max(g.Ly, g.Lz)), R) * 4;
  const double ek = u * (2 * s + E) + tiny;
  double es2 = 7 * u * S2 + 2 * sqrt(3.0) * u * E * s + 3 * ek * ek + 6 * ek * tiny;
  double epi = u * (2 * pmx + E) + tiny;          /* box: window on pi */
  const double m2f = sv ? S2 : 0.0;
  const double mf = sqrt(m2f);
  double dmu = 0;                                 /* survey mu window terms */
  if (sv) {
    es2 += 8 * eps * R * R + 4 * eps * S2;        /* the reference's s^2 */
    const double epa = sqrt(3.0) * ek + 6 * u * s + s * (u * (s + 3 * E) + 2 * sqrt(3.0) * ek) / mf;
    const double m2rel = u * (9 + 2 * (s + 3 * E) / mf) + 4 * sqrt(3.0) * ek / mf;
    if (b->bintype == FCFC_BIN_SPI) {
      const double pi = sqrt(pmx);
      const double ep2 = 2 * pi * epa + epa * epa + pmx * (m2rel + 6 * u)
                         + 2 * pi * 5 * eps * R * R / mf + pmx * 6 * eps * R * R / m2f + 4 * eps * pmx;
      epi = ep2;                                  /* window on pi^2 */
      es2 = es2 + ep2 + u * S2;                   /* window on s_perp^2 */
    }
    else {
      const double sf = sqrt(std::max(s2f, 1e-300));
      const double es2rel = 7 * u + 2 * sqrt(3.0) * u * E / sf + 3 * pow(u * (2 + E / sf), 2);
      dmu = (sqrt(3.0) * u * (2 + E / sf) + sqrt(3.0) * tiny / sf + 5 * u + u * s / mf
             + sqrt(3.0) * ek / mf) + 0.5 * es2rel + 0.5 * m2rel + 8 * u + 3 * u
            + 5 * eps * R * R / (mf * sf) + 4 * eps * R * R / (sf * sf);
    }
  }
  FkWin &w = *win;
  w.e_s2 = (float) (es2 * 1.25 + 1e-7);
  w.e_pi = (float) (epi * 1.25 + 1e-7);
  w.e_s2x2 = 2.0f * w.e_s2;
  w.e_pix2 = 2.0f * w.e_pi;
  const double cz = 0.5 / std::max(b->nmu, 1);
  if (sv) { w.idle_x = 1.0e6f; w.idle_z = 0.0f; }
  else {
    w.idle_z = (float) (1e18 * cz);
    w.idle_x = (float) (1e18 * sqrt(1.0 - cz * cz));
  }
  const double nmu = b->nmu;
  double D = 1.25 * (nmu * 10 * u + (sqrt(3.0) * u * E * nmu + nmu * (u * E + tiny)) / sqrt(s2f))
             + 4 * nmu * u;
  if (sv) D = 1.25 * nmu * dmu + 4 * nmu * u;
  /* fixed-point mu (fk_mu32): sh >= D + 2^-16 on the grid 2^-16; the
   * fraction threshold is 0 (every pair re-evaluated) when the windows
   * cover everything */
  const double sh = ceil((std::min(D, 0.5) + ldexp(1.0, -16)) * 65536.0) / 65536.0;
  w.mu_sh = (float) sh;
  w.mu_c = (float) (129.0 - sh);
  w.mu_t16 = (unsigned) std::max(0.0, floor(65536.0 * (1.0 - 2.0 * sh)));
  w.s2_floor = (float) s2f;
  w.nmu_f = (float) b->nmu;
  w.m2_floor = (float) m2f;
}

/* The FP32 window test reads one table cell and the edge at its lower end:
 * windows must stay well inside a cell (wide only for a few objects in a huge
 * volume, whose grid cells, and so runs, are large). */
static bool fp32_ok(const fcfc_bins *b, const JobPlan &P) {
  FkWin w;
  fp32_windows(b, P.g, P.zmaxc, fp32_s2_floor(b, P.g, P.zmaxc), &w);
  return w.e_s2x2 < 0.5f && w.e_pix2 < 0.5f;
}

static int cat_ok(const fcfc_cat *k) {
  return k && k->n >= 0 && k->n < 0x7fffffff && (k->n == 0 || (k->x && k->y && k->z));
}

static int bins_ok(const fcfc_bins *b) {
  return b && b->ns > 0 && b->s2bin && b->stab && b->ntot > 0 &&
      (b->bintype != FCFC_BIN_SPI || (b->pbin && b->ptab));
}

/* Plan a job and stage its catalogues.  Sorted copies are shared between
 * jobs of one call when every array a copy is built from (coordinates,
 * |r|^2, weights of weighted jobs) and the grid coincide: two catalogues on
 * the same positions with different weights (jackknife or bootstrap
 * weights) get copies of their own. */
struct CopyKey {
  const double *x, *y, *z, *s, *w; int64_t n; int wt; FkGrid g; DevCat d;
  bool same(const fcfc_cat *k, int wt_, int need_s, const FkGrid &g_) const;
};

static bool same_grid(const FkGrid &a, const FkGrid &b) {
  return a.ncx == b.ncx && a.ncy == b.ncy && a.ncz == b.ncz && a.ox == b.ox && a.oy == b.oy &&
      a.oz == b.oz && a.wx == b.wx && a.wy == b.wy && a.wz == b.wz;
}

bool CopyKey::same(const fcfc_cat *k, int wt_, int need_s, const FkGrid &g_) const {
  return x == k->x && y == k->y && z == k->z && n == k->n && wt == wt_ &&
      (!need_s || s == k->s) && (!wt_ || w == k->w) && same_grid(g, g_);
}

/* weights of a sorted catalogue re-read from the caller's device array */
struct Gather { const double *src; const int *idx; double *dst; int n, stride; };

static int setup_job(fcfc_gpu_ctx *c, Alloc &al, std::vector<CopyKey> &copies,
    const fcfc_cat *a, const fcfc_cat *b, const fcfc_bins *bins, const double *bsize,
    int autoc, int wt, int mode, PJob *J, std::vector<FkStage> &stages,
    std::vector<Gather> *gathers = nullptr) {
  const int need_s = (bins->geometry == FCFC_GEOM_SURVEY && bins->bintype != FCFC_BIN_ISO);
  /* cross counts are symmetric in the two catalogues: the larger one goes to
   * the lanes (fuller tiles, tighter windows and fewer lanes sharing one
   * histogram bin when the other is clustered); the gradient keeps the
   * caller's orientation */
  if (!autoc && mode != MODE_GRAD && b->n > a->n) std::swap(a, b);
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  int e;
  if (bins->geometry == FCFC_GEOM_SURVEY) {
    const fcfc_cat *ks[2] = {a, b};
    if ((e = bbox(c, al, ks, autoc ? 1 : 2, lo, hi))) return e;
    if (!(lo[0] <= hi[0])) { for (int k = 0; k < 3; k++) { lo[k] = 0; hi[k] = 1; } }
  }
  const int64_t nb = autoc ? a->n : b->n;
  if ((e = make_plan(c, bins, bsize, lo, hi, autoc, wt, mode, a->n, nb, true, &J->P))) return e;
  /* a grid for longer runs where windows take a count to FP64 whose tables
   * leave no room for groups of lanes */
  if (J->P.G > 1 && mode == MODE_C32 && !fp32_ok(bins, J->P) && !groups_keep_tables(bins, MODE_C64, wt) &&
      (e = make_plan(c, bins, bsize, lo, hi, autoc, wt, mode, a->n, nb, false, &J->P))) return e;
  J->autoc = autoc;
  J->wt = wt;
  const fcfc_cat *cs[2] = {a, autoc ? a : b};
  DevCat *dst[2] = {&J->A, &J->B};
  for (int q = 0; q < (autoc ? 1 : 2); q++) {
    const fcfc_cat *k = cs[q];
    bool found = false;
    for (auto &cp : copies)
      if (cp.same(k, wt, need_s, J->P.g)) { *dst[q] = cp.d; found = true; break; }
    if (found) continue;
    const int slot = (q == 0) ? WS_A_REC : WS_B_REC;
    const int upslot = (q == 0) ? WS_IN_X : WS_IN2_X;
    if ((e = stage_prep(c, al, k, need_s, wt, gathers || mode == MODE_GRAD, J->P.g, slot, upslot, dst[q], stages))) return e;
    if (al.own) copies.push_back(CopyKey{k->x, k->y, k->z, k->s, k->w, k->n, wt, J->P.g, *dst[q]});
    if (gathers && wt && k->w && k->on_device && k->n > 0)
      gathers->push_back(need_s ? Gather{k->w, dst[q]->idx, dst[q]->w, (int) k->n, 1}
                                : Gather{k->w, dst[q]->idx, &dst[q]->rec->q, (int) k->n, 4});
  }
  if (autoc) J->B = J->A;
  return 0;
}

/* A recorded count launch: kernel, grid, LDS bytes and arguments, and the
 * arrays of its run list. */
struct Launch {
  kfn_t fn = nullptr;
  int nblock = 0, lds = 0;
  FkArgs a;
  int nunit = 0, njob = 0;
  const FkTileJob *tj = nullptr;
  int *unitn = nullptr, *unitoff = nullptr;
  FkRun *runs = nullptr;
  FkSplit *splits = nullptr;
};

/* binning tables of a call on the device */
struct DevTabs { const uint16_t *stab = nullptr, *ptab = nullptr; const double *s2e = nullptr, *pe = nullptr, *G = nullptr; };

/* bytes to reserve for the uploads of a call */
static size_t upload_bytes(const fcfc_bins *b, const std::vector<PJob> &jobs, size_t nst, bool grad) {
  size_t n = 64 * 16 + sizeof(FkStage) * nst + 2 * (b->stab_len + 1) + 8 * (b->ns + 1);
  if (b->bintype == FCFC_BIN_SPI) n += 2 * (b->ptab_len + 1) + 8 * (b->np + 1);
  if (grad) n += 8 * (size_t) b->ntot;
  for (const PJob &J : jobs) n += sizeof(FkJob) + sizeof(FkTileJob) + 4 * J.P.strips.size() + 64;
  return n;
}

static void put_tables(Upload &up, const fcfc_bins *b, DevTabs *t) {
  t->stab = up.put(b->stab, b->stab_len);
  t->s2e = up.put(b->s2bin, b->ns + 1);
  if (b->bintype == FCFC_BIN_SPI) {
    t->ptab = up.put(b->ptab, b->ptab_len);
    t->pe = up.put(b->pbin, b->np + 1);
  }
}

/* Prepare the run list and the persistent launch that counts (or
 * differentiates) the jobs; every buffer comes from al, descriptors go to up,
 * res are the result words of the call and ncall its jobs. */
static int build_launch(fcfc_gpu_ctx *c, Alloc &al, Upload &up, const DevTabs &tabs, const fcfc_bins *b,
    std::vector<PJob> &jobs, int mode, unsigned long long *res, int ncall, Launch *out) {
  const int geom = b->geometry;
  int m = mode;
  const int need_s = (geom == FCFC_GEOM_SURVEY && b->bintype != FCFC_BIN_ISO);
  int anywt = 0;
  for (auto &j : jobs) anywt |= j.wt;
  if (m == MODE_GRAD) anywt = 1;
  /* a launch has runs of one kind (launch_groups) */
  int G = jobs.empty() ? 1 : jobs[0].P.G;
  for (const PJob &J : jobs) if (m == MODE_C32 && !fp32_ok(b, J.P)) m = MODE_C64;
  /* (only a job whose own plan did not see this launch's form: another job of
   * the batch has taken it to FP64) */
  if (G > 1 && !groups_keep_tables(b, m, anywt)) G = 1;
  const TabForm tf = table_form(b, m, anywt, G);
  m = tf.m;
  const int hyb = tf.hyb, ssearch = tf.ssearch, psearch = tf.psearch;
  /* one kernel serves every job of the launch: runs of the longest kind.
   * A lane holds R objects (1, 2 or 4), so no run may exceed 64 R objects
   * (a tile is the FK_NW runs of a workgroup): R is cut to what the kernel family provides (fk_lanes_max),
   * and a tile size set by the caller or the autotuner is clamped to what
   * the kernel covers */
  {
    int R = 1;
    for (auto &j : jobs) R = std::max(R, (j.P.T + FK_NT - 1) / FK_NT);
    if (R > 2) R = 4;
    R = std::min(R, fk_lanes_max(geom, m, anywt, hyb));
    for (auto &j : jobs) {
      j.P.R = R;
      if (j.P.T_auto || j.P.T > R * FK_NT) j.P.T = R * FK_NT;
    }
  }
  /* ---- kernel and LDS plan ---- */
  const int R = jobs.empty() ? 1 : jobs[0].P.R;
  /* (the limit belongs to the kernel, whose launches of other sizes -- other
   * contexts', replayed plans' -- share it: always the same, the most there is) */
  auto occ_of = [&](kfn_t f, const LdsPlan &P, int *occ) -> int {
    HIPCHK(c, hipFuncSetAttribute((const void *) f, hipFuncAttributeMaxDynamicSharedMemorySize, FK_LDS_MOST));
    HIPCHK(c, hipOccupancyMaxActiveBlocksPerMultiprocessor(occ, (const void *) f, FK_NT, P.total));
    return 0;
  };
  /* the rounding census compares the box arithmetic paths */
  const bool above0 = b->soff > 0 || (b->bintype == FCFC_BIN_SPI && b->poff > 0);
  const int km = (m == MODE_C32 && c->census && geom == FCFC_GEOM_BOX) ? MODE_C32C
                 : (m == MODE_GRAD && above0 && masked_form(b, m, hyb)) ? MODE_GRADL : m;
  kfn_t fn = pick_kernel(b->bintype, geom, anywt, km, hyb, R, G);
  /* histogram copies: as many as keep the occupancy of a single copy */
  LdsPlan L = lds_plan(b, m, anywt, need_s, 1, hyb, ssearch, psearch, G);
  if (!tf.fits) {
    set_err(c, "binning tables need %d bytes of LDS (limit %d)", L.total, FK_LDS_MOST);
    return FCFC_ERR_CFG;
  }
  /* (the choice depends on the kernel and the LDS size of one copy alone, and
   * is kept: it takes several queries) */
  int occ = 0;
  const int lds1 = L.total;
  for (const auto &o : c->occs)
    if (o.fn == (const void *) fn && o.lds1 == lds1 && c->t_nh <= 0) {
      L = lds_plan(b, m, anywt, need_s, o.nh, hyb, ssearch, psearch, G);
      if (L.total == o.lds) occ = o.occ;
      else L = lds_plan(b, m, anywt, need_s, 1, hyb, ssearch, psearch, G);
      break;
    }
  if (!occ) {
    int occ1 = 0;
    if (int e = occ_of(fn, L, &occ1)) return e;
    if (m != MODE_GRAD) {
      const int nhmax = c->t_nh > 0 ? c->t_nh : 8;
      for (int nh = 2; nh <= nhmax; nh *= 2) {
        LdsPlan L2 = lds_plan(b, m, anywt, need_s, nh, hyb, ssearch, psearch, G);
        int o2 = 0;
        if (!lds_fits(b, L2, m, hyb)) break;
        if (int e = occ_of(fn, L2, &o2)) return e;
        if (o2 < occ1 && c->t_nh <= 0) break;
        L = L2;
      }
    }
    if (int e = occ_of(fn, L, &occ)) return e;
    if (occ < 1) occ = 1;
    if (c->t_nh <= 0) {
      if (c->occs.size() >= 256) c->occs.clear();
      c->occs.push_back({(const void *) fn, lds1, L.nh, L.total, occ});
    }
  }
  /* ---- runs of all jobs ---- */
  /* persistent workgroups, dealt out to the jobs in proportion to the
   * candidate pairs of their runs (each run at least one chunk) */
  int nwg = c->t_nblock > 0 ? c->t_nblock : occ * c->ncu;
  const int njob = (int) jobs.size();
  std::vector<FkTileJob> htj(jobs.size());
  std::vector<int> wg0(jobs.size() + 1, 0);
  long long nunit_l = 0, maxrun = 0, maxitem = 0;
  double work = 0, done = 0;
  for (int k = 0; k < njob; k++) {
    const PJob &J = jobs[k];
    FkTileJob &t = htj[k];
    memset(&t, 0, sizeof t);
    const long long nu = (long long) J.P.g.ncx * J.P.g.ncy * J.P.nblk;
    t.unit0 = (int) nunit_l;
    t.nunit = (int) nu;
    t.nblk = J.P.nblk; t.zm = J.P.zmaxc; t.ncz = J.P.g.ncz;
    t.T = std::min(J.P.T, G > 1 ? 64 / G : 64 * J.P.R);
    t.chunks = (int) std::min(J.P.cand / (64 * G), 1e9);   /* in steps of 64 pairs per lane */
    t.smax = std::min(std::max(J.P.nstrips, 1), 64);
    t.ipw = njob > 1 ? 2 : 16;
    t.frac = c->tile_frac;
    t.cs = J.A.cs;
    nunit_l += nu;
    if (nunit_l > INT_MAX / 2) { set_err(c, "catalogues of one call too large"); return FCFC_ERR_CFG; }
    /* at most as many runs as full ones and one remainder per non-empty unit */
    const long long nr = J.A.n / t.T + std::min<long long>(nu, J.A.n);
    maxrun += nr;
    maxitem += nr * std::min<long long>(std::max(1, t.chunks / 2), 1024);
    work += (double) J.A.n * std::max(J.P.cand, 64.0);
  }
  nwg = (int) std::max<long long>(1, std::min<long long>(nwg, (maxitem + FK_NW - 1) / FK_NW));
  for (int k = 0; k < njob; k++) {
    done += (double) jobs[k].A.n * std::max(jobs[k].P.cand, 64.0);
    wg0[k + 1] = k + 1 == njob ? nwg : (int) (work > 0 ? nwg * std::min(done / work, 1.0) : 0.0);
    htj[k].nw = (wg0[k + 1] - wg0[k]) * FK_NW;
  }
  const int nunit = (int) nunit_l;
  int *unitn = (int *) al.get(WS_ROWN, sizeof(int) * (size_t) nunit);
  int *unitoff = (int *) al.get(WS_ROWOFF, sizeof(int) * ((size_t) nunit + 1));
  const FkTileJob *dtj = up.put(htj.data(), htj.size());
  FkRun *runs = (FkRun *) al.get(WS_TILES, sizeof(FkRun) * (size_t) (maxrun > 0 ? maxrun : 1));
  FkSplit *splits = (FkSplit *) al.get(WS_SPLITS, sizeof(FkSplit) * jobs.size());
  if (al.err) return al.err;
  /* ---- strips, job descriptors ---- */
  std::vector<int> hstr;
  for (auto &j : jobs) hstr.insert(hstr.end(), j.P.strips.begin(), j.P.strips.end());
  const int *dstrips = up.put(hstr.data(), hstr.size());
  std::vector<FkJob> hj(jobs.size(), FkJob{});
  size_t str0 = 0;
  double s2f = 0;
  float win2s = 0.0f, win2p = 0.0f;
  if (m == MODE_C32)
    for (const PJob &J : jobs) s2f = std::max(s2f, fp32_s2_floor(b, J.P.g, J.P.zmaxc));
  for (size_t k = 0; k < jobs.size(); k++) {
    const PJob &J = jobs[k];
    FkJob &f = hj[k];
    memset(&f, 0, sizeof f);
    f.A = J.A.dev();
    f.B = J.B.dev();
    f.g = J.P.g;
    f.strips = dstrips + str0;
    str0 += J.P.strips.size();
    f.nstrips = J.P.nstrips;
    f.autoc = J.autoc;
    f.wt = J.wt;
    f.hist_off = J.hist_off;
    f.wg0 = wg0[k];
    f.wg1 = wg0[k + 1];
    f.q0 = J.qi * queue_lines(ncall);
    f.G = std::min(std::max((wg0[k + 1] - wg0[k]) / 8, 1), queue_lines(ncall));
    f.gA = J.gA ? J.gA - J.A.obj0 : nullptr;
    f.gB = J.gB ? J.gB - J.B.obj0 : nullptr;
    if (m == MODE_C32) {
      fp32_windows(b, J.P.g, J.P.zmaxc, s2f, &f.win);
      win2s = std::max(win2s, f.win.e_s2x2);
      win2p = std::max(win2p, f.win.e_pix2);
    }
  }
  const FkJob *djobs = up.put(hj.data(), hj.size());
  if (!dtj || !dstrips || !djobs) { set_err(c, "upload buffer too small"); return FCFC_ERR_UNKNOWN; }

  FkArgs a;
  memset(&a, 0, sizeof a);
  a.jobs = djobs;
  a.njobs = (int) jobs.size();
  FkBins &fb = a.bins;
  fb.bintype = b->bintype; fb.geometry = geom;
  fb.ns = b->ns; fb.nmu = b->nmu; fb.np = b->np; fb.ntot = b->ntot;
  const HistDim hd = hist_dim(b, m, hyb);
  fb.nsh = hd.nsh; fb.ntoh = hd.ntoh; fb.nslot = hd.nslot;
  fb.scap32 = b->soff + b->stab_len + 1; fb.pcap32 = b->poff + b->ptab_len + 1;
  fb.tabtype = b->tabtype; fb.soff = b->soff; fb.poff = b->poff;
  /* searched tables are not staged to LDS (length 0: sentinels only) */
  fb.stab_len = ssearch ? 0 : b->stab_len; fb.ptab_len = psearch ? 0 : b->ptab_len;
  fb.ssearch = ssearch; fb.psearch = psearch;
  fb.s2min = b->s2bin[0]; fb.s2max = b->s2bin[b->ns];
  fb.pmin = (b->bintype == FCFC_BIN_SPI) ? b->pbin[0] : 0;
  fb.pmax = (b->bintype == FCFC_BIN_SPI) ? b->pbin[b->np] : 0;
  fb.nmu2 = (double) b->nmu * b->nmu;
  fb.nmu_d = (double) b->nmu;
  fb.s2_exact = std::max(b->s2bin[b->ns] * ldexp(1.0, -12), 4 * FK_DBL_EPS);
  /* no pair at or beyond these is counted (margins cover the other rounding
   * orientation of the gradient and the FP32 windows) */
  /* survey (s_perp, pi): s^2 = s_perp^2 + pi^2 (pbin holds pi^2 edges) */
  fb.s2skip = (geom == FCFC_GEOM_SURVEY && b->bintype == FCFC_BIN_SPI)
      ? (fb.s2max + fb.pmax) * (1 + ldexp(1.0, -30)) + 1e-6 * (fb.s2max + fb.pmax + 1)
      : fb.s2max * (1 + ldexp(1.0, -30));
  fb.s2low = fb.s2min > 0 ? fb.s2min : nextafter(-1.0, 0.0);
  fb.pskip = (b->bintype == FCFC_BIN_SPI) ? fb.pmax * (1 + ldexp(1.0, -30)) : 1e300;
  fb.s2skip32 = (float) (fb.s2max + fb.pmax + 2.0);
  /* the upper end of the window of s2max (pmax): FP32 values at or beyond it
   * are out of range */
  fb.m32s = nextafterf((float) (fb.s2max + win2s), INFINITY);
  fb.m32p = nextafterf((float) (fb.pmax + win2p), INFINITY);
  fb.win2s = win2s;
  fb.win2p = win2p;
  {
    /* fixed-point mu (fk_mu_exact): sh >= nmu 2^-20 + 2^-16 on the grid
     * 2^-16, the addend 2^36 + 1 - sh exact */
    const double sh = ceil((ldexp((double) b->nmu, -20) + ldexp(1.0, -16)) * 65536.0) / 65536.0;
    fb.mu_c = ldexp(1.0, 36) + 1.0 - sh;
    fb.mu_cmax = ldexp(1.0, 36) + b->nmu + 1.5;
    fb.mu_t16 = (unsigned) std::max(0.0, floor(65536.0 * (1.0 - 2.0 * sh)));
    /* the FP64 integer-table kernels add mu_t16 << 16 to their (s, mu)
     * indices (fk_smu_index): keep the largest, (nmu + 1) nsh + 0xFFFF +
     * (mu_t16 << 16), below 2^32 (a lower threshold only sends more pairs
     * to the exact path) */
    const unsigned long long room = (0xFFFF0000ull - (unsigned long long) (b->nmu + 2) * fb.nsh) >> 16;
    fb.mu_t16 = (unsigned) std::min<unsigned long long>(fb.mu_t16, room);
    fb.mu_pad = 0;
  }
  {
    /* survey (s_perp, pi) with integer tables (fk_sv64): x + q_c rounds
     * onto the grid 2^-16 of [2^36, 2^37) with K = floor(x - h) + 2, h =
     * 2^-15 >= 2^-16 plus the 2^-29.7 error bound of the fast pi^2 and
     * s_perp^2; a fraction f <= q_t16 = 65532 puts x strictly inside
     * (K - 2, K - 1) (f/2^16 + h + 2^-17 + 2^-29.7 < 1).  The ceilings are
     * the last table entries, off + len + 3 (< 2^16: the tables fit in LDS) */
    fb.q_c = ldexp(1.0, 36) + 2.0 - ldexp(1.0, -15);
    fb.q_caps = ldexp(1.0, 36) + (double) (b->soff + b->stab_len + 3);
    fb.q_capp = ldexp(1.0, 36) + (double) (b->poff + b->ptab_len + 3);
    fb.q_bmin = ldexp(1.0, -1000);
    fb.q_t16 = 65532u;
    fb.q_pad = 0;
  }
  fb.stab = tabs.stab; fb.ptab = tabs.ptab; fb.s2bin = tabs.s2e; fb.pbin = tabs.pe;
  a.runs = runs; a.splits = splits;
  a.queue = (unsigned int *) (res + RES_HIST + (size_t) b->ntot * (m == MODE_GRAD ? 0 : ncall));
  a.gcnt_u = res + RES_HIST; a.gcnt_d = (double *) (res + RES_HIST);
  a.stats = res;
  a.nh = L.nh;
  a.off_hist = L.off_hist; a.off_stab = L.off_stab; a.off_ptab = L.off_ptab;
  a.stab_c0 = L.stab_c0; a.ptab_c0 = L.ptab_c0;
  a.off_edges = L.off_edges;
  a.off_chunk = L.off_chunk; a.off_queue = L.off_queue;
  a.census = c->census;
  a.G = tabs.G;
  c->last_nrun = unitoff + nunit;
  c->last_T = jobs.empty() ? 0 : jobs[0].P.T;
  c->stats.tile = G > 1 ? std::min(c->last_T, FK_NW * 64 / G) : c->last_T;
  c->stats.cell_div = jobs.empty() ? 0 : (int) lround(sqrt(jobs[0].P.g.Rxy2) / jobs[0].P.g.wx);
  out->fn = fn; out->nblock = nwg; out->lds = L.total; out->a = a;
  out->nunit = nunit; out->njob = njob; out->tj = dtj;
  out->unitn = unitn; out->unitoff = unitoff; out->runs = runs; out->splits = splits;
  return 0;
}

/* Waits for the stream when it goes out of scope: declared after the
 * launches of a call (destroyed before them), it keeps their host copies
 * alive until the stream has drained, on the error returns as well. */
struct StreamDrain {
  fcfc_gpu_ctx *c;
  ~StreamDrain() { (void) hipStreamSynchronize(c->stream); }
};

/* the run list of a launch, on its sorted catalogues */
static int list_runs(fcfc_gpu_ctx *c, Alloc &al, const Launch &L, const unsigned long long *res) {
  hipLaunchKernelGGL(k_run_count, dim3(nblk(L.nunit, 64)), dim3(64), 0, c->stream, L.nunit, L.njob, L.tj, L.unitn);
  if (int e = scan(c, al, L.unitn, L.unitoff, L.nunit)) return e;
  hipLaunchKernelGGL(k_run_emit, dim3(nblk(L.nunit, 64)), dim3(64), 0, c->stream, L.nunit, L.njob, L.tj,
                     L.unitoff, L.runs, L.splits, res + RES_BAD);
  HIPCHK(c, hipGetLastError());
  return 0;
}

static int launch(fcfc_gpu_ctx *c, const Launch &Lc) {
  hipLaunchKernelGGL(Lc.fn, dim3(Lc.nblock), dim3(FK_NT), Lc.lds, c->stream, Lc.a);
  HIPCHK(c, hipGetLastError());
  return 0;
}

/* Jobs of a batch grouped for their launches: one kernel variant per
 * launch, so weighted and unweighted jobs, and jobs whose runs want one or
 * two objects per lane or four groups of lanes, go to separate persistent launches. */
static std::vector<std::vector<PJob>> launch_groups(const std::vector<PJob> &jobs) {
  std::vector<std::vector<PJob>> g;
  std::vector<int> key;
  for (const PJob &j : jobs) {
    const int k = 2 * (j.wt ? 1 : 0) + ((j.P.T > FK_NT) ? 1 : 0) + (j.P.G > 1 ? 4 : 0);
    size_t q = 0;
    while (q < key.size() && key[q] != k) q++;
    if (q == key.size()) { key.push_back(k); g.emplace_back(); }
    g[q].push_back(j);
  }
  return g;
}

/* Wait for a call and take its results: statistics, the check for
 * non-finite coordinates, and (nhist words from the histograms on) the
 * histograms of its jobs added into the caller's cnt, 8 bytes per bin (int64
 * or double), in device or host memory. */
static int deliver(fcfc_gpu_ctx *c, const std::vector<PJob> &jobs, int ntot,
    const unsigned long long *res, int nhist, uint32_t flags, void *cnt, bool fixed) {
  const int njob = (int) jobs.size(), off = RES_HIST;
  const bool dev = (flags & FCFC_GPU_CNT_DEVICE) != 0;
  const size_t n = (size_t) off + (dev ? 0 : nhist);
  std::vector<unsigned long long> hv;
  unsigned long long *h;
  /* (pinned memory that the call's upload used is free: the device has read
   * it before anything this copy waits for) */
  if (Upload::pin_fit(c, 8 * n, fixed)) h = (unsigned long long *) c->pin;
  else { hv.resize(n); h = hv.data(); }
  HIPCHK(c, hipMemcpyAsync(h, res, 8 * n, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  unsigned long long st[3] = {0, 0, 0};
  for (int q = 0; q < FK_STATS; q++)
    for (int k = 0; k < 3; k++) st[k] += h[q * (FK_LINE / 8) + k];
  c->stats.evals = (double) st[RES_EVALS];
  c->stats.rechecked = (double) st[RES_RECHECKED];
  c->stats.census = (double) st[RES_CENSUS];
  if (h[RES_BAD]) { set_err(c, "a catalogue has a non-finite coordinate"); return FCFC_ERR_DATA; }
  if (!nhist) return 0;
  for (int k = 0; k < njob; k++) {
    const size_t o = (size_t) k * ntot;
    if (dev) {
      const unsigned long long *src = res + off + o;
      if (jobs[k].wt) hipLaunchKernelGGL(k_add_f64, dim3(nblk(ntot, 256)), dim3(256), 0, c->stream, (double *) cnt + o, (const double *) src, ntot);
      else hipLaunchKernelGGL(k_add_u64, dim3(nblk(ntot, 256)), dim3(256), 0, c->stream, (long long *) cnt + o, src, ntot);
    }
    else if (jobs[k].wt) { double *dst = (double *) cnt + o; const double *hd = (const double *) (h + off) + o; for (int i = 0; i < ntot; i++) dst[i] += hd[i]; }
    else { int64_t *dst = (int64_t *) cnt + o; for (int i = 0; i < ntot; i++) dst[i] += (int64_t) h[off + o + i]; }
  }
  if (dev) {
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipStreamSynchronize(c->stream));
  }
  return 0;
}

/* counts of njob jobs; job k's histogram lands in cnt + k * ntot */
static int count_jobs(fcfc_gpu_ctx *c, int njob, const fcfc_cat *const *as,
    const fcfc_cat *const *bs, const double *const *bsz, const uint32_t *fl,
    const fcfc_bins *bins, uint32_t flags, void *cnt, void *arena = nullptr,
    size_t arena_cap = 0) {
  auto t0 = std::chrono::steady_clock::now();
  HIPCHK(c, hipSetDevice(c->device));
  memset(&c->stats, 0, sizeof c->stats);
  c->census = (flags & FCFC_GPU_CENSUS) ? 1 : 0;
  const int mode = (flags & FCFC_GPU_PREC_FP32) ? MODE_C32 :
                   ((flags & FCFC_GPU_PREC_PLAIN) ? MODE_P64 : MODE_C64);
  Alloc al(c, njob > 1);
  if (arena) al.use_arena(arena, arena_cap);
  std::vector<CopyKey> copies;
  std::vector<FkStage> stages;
  std::vector<PJob> jobs(njob);
  for (int k = 0; k < njob; k++) {
    const int autoc = (fl[k] & FCFC_GPU_AUTO) ? 1 : 0;
    const int wt = (fl[k] & FCFC_GPU_WEIGHTED) ? 1 : 0;
    if (!cat_ok(as[k]) || (!autoc && !cat_ok(bs[k]))) { set_err(c, "invalid catalogue in job %d", k); return FCFC_ERR_ARG; }
    if (bins->geometry == FCFC_GEOM_BOX && !bsz[k]) { set_err(c, "box size required"); return FCFC_ERR_ARG; }
    int e = setup_job(c, al, copies, as[k], bs[k], bins, bsz[k], autoc, wt, mode, &jobs[k], stages);
    if (e) return e;
    jobs[k].hist_off = (long long) k * bins->ntot;
    jobs[k].qi = k;
  }
  Sort so;
  if (int e = sort_alloc(c, al, stages, jobs, &so)) return e;
  const int nhist = bins->ntot * njob;
  const size_t nres = RES_HIST + nhist + queue_words(njob);
  unsigned long long *res = (unsigned long long *) al.tmp(WS_RES, 8 * nres);
  if (al.err) return al.err;
  /* one persistent launch per group */
  std::vector<std::vector<PJob>> groups = launch_groups(jobs);
  std::vector<Launch> L(groups.size());
  Upload up(c);
  StreamDrain drain{c};
  if (int e = up.reserve(al, upload_bytes(bins, jobs, stages.size(), false), false)) return e;
  DevTabs tabs;
  put_tables(up, bins, &tabs);
  so.st = up.put(stages.data(), stages.size());
  for (size_t q = 0; q < groups.size(); q++)
    if (int e = build_launch(c, al, up, tabs, bins, groups[q], mode, res, njob, &L[q]))
      return e;
  if (int e = up.flush()) return e;
  if (int e = sort_run(c, al, so, res, nres)) return e;
  for (const Launch &Lq : L) if (int e = list_runs(c, al, Lq, res)) return e;
  HIPCHK(c, hipEventRecord(c->ev0, c->stream));
  for (const Launch &Lq : L) if (int e = launch(c, Lq)) return e;
  HIPCHK(c, hipEventRecord(c->ev1, c->stream));
  if (int e = deliver(c, jobs, bins->ntot, res, nhist, flags, cnt, arena != nullptr)) return e;
  float ms = 0;
  HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
  c->stats.kernel_ms = ms;
  c->stats.total_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return 0;
}

extern "C" int fcfc_gpu_count(fcfc_gpu_ctx *c, const fcfc_cat *a,
    const fcfc_cat *b, const fcfc_bins *bins, const double *bsize,
    uint32_t flags, void *cnt) {
  if (!c) return FCFC_ERR_ARG;
  if (!bins_ok(bins) || !cnt) { set_err(c, "invalid argument"); return FCFC_ERR_ARG; }
  const fcfc_cat *as[1] = {a}, *bs[1] = {b};
  const double *bz[1] = {bsize};
  uint32_t fl[1] = {flags & (FCFC_GPU_AUTO | FCFC_GPU_WEIGHTED)};
  return count_jobs(c, 1, as, bs, bz, fl, bins, flags, cnt);
}

/* Device bytes a no-allocation count needs at least (uploads, sorted copies);
 * cells, runs and histograms come on top. */
static size_t noalloc_floor(const fcfc_cat *k, const fcfc_bins *bins, int wt) {
  if (!k || k->n <= 0) return 0;
  const int need_s = (bins->geometry == FCFC_GEOM_SURVEY && bins->bintype != FCFC_BIN_ISO);
  size_t per = sizeof(FkRec) + 4 + (wt && need_s ? 8 : 0);       /* sorted copy, rank */
  if (!k->on_device) per += 24 + (wt && k->w ? 8 : 0) + (need_s && k->s ? 8 : 0);
  return per * (size_t) k->n;
}

extern "C" int fcfc_gpu_count_noalloc(fcfc_gpu_ctx *c, const fcfc_cat *a,
    const fcfc_cat *b, const fcfc_bins *bins, const double *bsize,
    uint32_t flags, void *cnt) {
  if (!c) return FCFC_ERR_ARG;
  if (!bins_ok(bins) || !cnt) { set_err(c, "invalid argument"); return FCFC_ERR_ARG; }
  if (!c->scratch) {
    set_err(c, "no-allocation count: the device scratch of GPU %d is unavailable (%s)",
            c->device, c->scratch_err);
    return FCFC_ERR_GPU;
  }
  const int autoc = (flags & FCFC_GPU_AUTO) ? 1 : 0;
  const int wt = (flags & FCFC_GPU_WEIGHTED) ? 1 : 0;
  if (!cat_ok(a) || (!autoc && !cat_ok(b))) { set_err(c, "invalid catalogue"); return FCFC_ERR_ARG; }
  const size_t need = noalloc_floor(a, bins, wt) + (autoc ? 0 : noalloc_floor(b, bins, wt));
  if (need > FK_SCRATCH_BYTES) {
    set_err(c, "no-allocation count: at most %zu bytes of device scratch, these catalogues "
            "need more than %zu; count them with fcfc_gpu_count", FK_SCRATCH_BYTES, need);
    return FCFC_ERR_MEMORY;
  }
  const fcfc_cat *as[1] = {a}, *bs[1] = {b};
  const double *bz[1] = {bsize};
  uint32_t fl[1] = {flags & (FCFC_GPU_AUTO | FCFC_GPU_WEIGHTED)};
  return count_jobs(c, 1, as, bs, bz, fl, bins, flags, cnt, c->scratch, FK_SCRATCH_BYTES);
}

extern "C" int fcfc_gpu_count_batch(fcfc_gpu_ctx *c, int njob,
    const fcfc_batch_job *jobs, const fcfc_bins *bins, uint32_t flags,
    void *cnt) {
  if (!c || njob < 0 || (njob && !jobs) || !cnt) return FCFC_ERR_ARG;
  if (!bins_ok(bins)) { set_err(c, "invalid bins"); return FCFC_ERR_ARG; }
  if (njob == 0) return 0;
  std::vector<const fcfc_cat *> as(njob), bs(njob);
  std::vector<const double *> bz(njob);
  std::vector<uint32_t> fl(njob);
  for (int k = 0; k < njob; k++) {
    as[k] = &jobs[k].a; bs[k] = &jobs[k].b; bz[k] = jobs[k].bsize;
    fl[k] = jobs[k].flags & (FCFC_GPU_AUTO | FCFC_GPU_WEIGHTED);
  }
  return count_jobs(c, njob, as.data(), bs.data(), bz.data(), fl.data(), bins,
      flags & ~(FCFC_GPU_AUTO | FCFC_GPU_WEIGHTED), cnt);
}

extern "C" int fcfc_gpu_count_backward(fcfc_gpu_ctx *c, const fcfc_cat *a,
    const fcfc_cat *b, const fcfc_bins *bins, const double *bsize,
    uint32_t flags, const double *grad_cnt, double *ga, double *gb) {
  if (!c) return FCFC_ERR_ARG;
  auto t0 = std::chrono::steady_clock::now();
  const int autoc = (flags & FCFC_GPU_AUTO) ? 1 : 0;
  if (!cat_ok(a) || (!autoc && !cat_ok(b)) || !bins_ok(bins) || !grad_cnt || !ga) {
    set_err(c, "invalid argument"); return FCFC_ERR_ARG;
  }
  if (bins->geometry == FCFC_GEOM_BOX && !bsize) { set_err(c, "box size required"); return FCFC_ERR_ARG; }
  HIPCHK(c, hipSetDevice(c->device));
  memset(&c->stats, 0, sizeof c->stats);
  c->census = 0;
  const int dev = (flags & FCFC_GPU_CNT_DEVICE) ? 1 : 0;
  /* one pass over the pairs exactly as the count enumerates them (auto: each
   * unordered pair once; cross: the larger catalogue in the lanes), so every
   * pair is binned as in the count; each pair adds G[bin] w_b to its A object
   * and G[bin] w_a to its B object */
  const int sw = (!autoc && b->n > a->n) ? 1 : 0;
  const fcfc_cat *pa = sw ? b : a, *pb = autoc ? a : (sw ? a : b);
  Alloc al(c, false);
  std::vector<CopyKey> copies;
  std::vector<FkStage> stages;
  std::vector<PJob> jobs(1);
  StreamDrain drain{c};
  if (int e = setup_job(c, al, copies, pa, pb, bins, bsize, autoc, 1, MODE_GRAD, &jobs[0], stages))
    return e;
  /* gradients of the sorted objects, then in the original order */
  const int64_t na = std::max<int64_t>(a->n, 1), nb = autoc || !gb ? 0 : std::max<int64_t>(b->n, 1);
  double *dga = (double *) al.get(WS_GA, sizeof(double) * 2 * (size_t) na);
  double *dgb = nb ? (double *) al.get(WS_GB, sizeof(double) * 2 * (size_t) nb) : nullptr;
  if (al.err) return al.err;
  hipLaunchKernelGGL(k_fill_f64, dim3(nblk(na, 256)), dim3(256), 0, c->stream, dga, na, 0.0);
  if (dgb) hipLaunchKernelGGL(k_fill_f64, dim3(nblk(nb, 256)), dim3(256), 0, c->stream, dgb, nb, 0.0);
  jobs[0].gA = sw ? dgb : dga;
  jobs[0].gB = autoc ? dga : (sw ? dga : dgb);
  Sort so;
  if (int e = sort_alloc(c, al, stages, jobs, &so)) return e;
  const size_t nres = RES_HIST + queue_words(1);
  unsigned long long *res = (unsigned long long *) al.tmp(WS_RES, 8 * nres);
  if (al.err) return al.err;
  Launch L;
  Upload up(c);
  StreamDrain drain2{c};
  if (int e = up.reserve(al, upload_bytes(bins, jobs, stages.size(), true), false)) return e;
  DevTabs tabs;
  put_tables(up, bins, &tabs);
  if (dev) tabs.G = grad_cnt;
  else tabs.G = up.put(grad_cnt, bins->ntot);
  so.st = up.put(stages.data(), stages.size());
  if (int e = build_launch(c, al, up, tabs, bins, jobs, MODE_GRAD, res, 1, &L)) return e;
  if (int e = up.flush()) return e;
  if (int e = sort_run(c, al, so, res, nres)) return e;
  if (int e = list_runs(c, al, L, res)) return e;
  HIPCHK(c, hipEventRecord(c->ev0, c->stream));
  if (int e = launch(c, L)) return e;
  HIPCHK(c, hipEventRecord(c->ev1, c->stream));
  if (int e = deliver(c, jobs, 0, res, 0, 0, nullptr, false)) return e;
  float ms = 0;
  HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
  for (int p = 0; p < 2; p++) {
    const fcfc_cat *k = p ? b : a;
    double *gout = p ? gb : ga, *gsrt = p ? dgb : dga;
    if (!gsrt) continue;
    double *gdev = gsrt + (p ? nb : na);
    const DevCat &dc = p == sw ? jobs[0].A : jobs[0].B;
    hipLaunchKernelGGL(k_unsort, dim3(nblk(k->n, 256)), dim3(256), 0, c->stream, (int) k->n, dc.idx, gsrt, gdev);
    if (dev) {
      hipLaunchKernelGGL(k_add_f64, dim3(nblk(k->n, 256)), dim3(256), 0, c->stream, gout, gdev, (int) k->n);
      HIPCHK(c, hipGetLastError());
    }
    else if (k->n > 0) {
      std::vector<double> hv;
      const size_t bytes = sizeof(double) * (size_t) k->n;
      double *h;
      if (Upload::pin_fit(c, bytes, false)) h = (double *) c->pin;
      else { hv.resize((size_t) k->n); h = hv.data(); }
      HIPCHK(c, hipMemcpyAsync(h, gdev, bytes, hipMemcpyDeviceToHost, c->stream));
      HIPCHK(c, hipStreamSynchronize(c->stream));
      for (int64_t i = 0; i < k->n; i++) gout[i] += h[i];
    }
  }
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->stats.kernel_ms = ms;
  c->stats.total_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return 0;
}

/* ---- prepared batches replayed as a HIP graph -------------------------- */

struct fcfc_gpu_plan {
  fcfc_gpu_ctx *c;
  Alloc al;                          /* every device buffer of the plan */
  std::vector<PJob> jobs;
  std::vector<Gather> gathers;
  int ntot = 0;
  uint32_t flags = 0;
  std::vector<Launch> L;             /* one per launch group */
  unsigned long long *res = nullptr; /* result words: counters, njob x ntot histograms */
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  explicit fcfc_gpu_plan(fcfc_gpu_ctx *c_) : c(c_), al(c_, true) {}
  ~fcfc_gpu_plan() {
    if (c && c->stream) (void) hipStreamSynchronize(c->stream);
    if (exec) (void) hipGraphExecDestroy(exec);
    if (graph) (void) hipGraphDestroy(graph);
  }
};

/* Sort and tile the catalogues of njob jobs once; record the launch
 * sequence of one count -- weight gathers from the callers' device arrays,
 * histogram and queue clears (fill kernels), the persistent count kernel --
 * as a HIP graph. */
extern "C" int fcfc_gpu_plan_create(fcfc_gpu_ctx *c, int njob, const fcfc_batch_job *jobs,
    const fcfc_bins *bins, uint32_t flags, fcfc_gpu_plan **out) {
  if (!c || !out || njob < 1 || !jobs || !bins_ok(bins)) return FCFC_ERR_ARG;
  *out = nullptr;
  HIPCHK(c, hipSetDevice(c->device));
  memset(&c->stats, 0, sizeof c->stats);
  c->census = 0;
  const int mode = (flags & FCFC_GPU_PREC_FP32) ? MODE_C32 :
                   ((flags & FCFC_GPU_PREC_PLAIN) ? MODE_P64 : MODE_C64);
  std::unique_ptr<fcfc_gpu_plan> P(new fcfc_gpu_plan(c));
  P->ntot = bins->ntot;
  P->flags = flags;
  P->jobs.resize(njob);
  std::vector<CopyKey> copies;
  std::vector<FkStage> stages;
  StreamDrain drain{c};
  for (int k = 0; k < njob; k++) {
    const fcfc_batch_job &j = jobs[k];
    const int autoc = (j.flags & FCFC_GPU_AUTO) ? 1 : 0;
    const int wt = (j.flags & FCFC_GPU_WEIGHTED) ? 1 : 0;
    if (!cat_ok(&j.a) || (!autoc && !cat_ok(&j.b))) { set_err(c, "invalid catalogue in job %d", k); return FCFC_ERR_ARG; }
    int e = setup_job(c, P->al, copies, &j.a, &j.b, bins, j.bsize, autoc, wt, mode, &P->jobs[k], stages,
                      &P->gathers);
    if (e) return e;
    P->jobs[k].hist_off = (long long) k * bins->ntot;
    P->jobs[k].qi = k;
  }
  Sort so;
  if (int e = sort_alloc(c, P->al, stages, P->jobs, &so)) return e;
  const size_t nres = RES_HIST + (size_t) bins->ntot * njob + queue_words(njob);
  P->res = (unsigned long long *) P->al.get(WS_RES, 8 * nres);
  if (P->al.err) return P->al.err;
  std::vector<std::vector<PJob>> groups = launch_groups(P->jobs);
  P->L.resize(groups.size());
  Upload up(c);
  StreamDrain drain2{c};
  int e = up.reserve(P->al, upload_bytes(bins, P->jobs, stages.size(), false), true);
  if (e) return e;
  DevTabs tabs;
  put_tables(up, bins, &tabs);
  so.st = up.put(stages.data(), stages.size());
  for (size_t q = 0; q < groups.size(); q++)
    if ((e = build_launch(c, P->al, up, tabs, bins, groups[q], mode, P->res, njob, &P->L[q]))) return e;
  if ((e = up.flush())) return e;
  if ((e = sort_run(c, P->al, so, P->res, nres))) return e;
  for (const Launch &Lq : P->L) if ((e = list_runs(c, P->al, Lq, P->res))) return e;
  unsigned long long bad = 0;
  HIPCHK(c, hipMemcpyAsync(&bad, P->res + RES_BAD, 8, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  if (bad) { set_err(c, "a catalogue has a non-finite coordinate"); return FCFC_ERR_DATA; }
  HIPCHK(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
  for (const Gather &g : P->gathers)
    hipLaunchKernelGGL(k_gather, dim3(nblk(g.n, 256)), dim3(256), 0, c->stream, g.n, g.idx, g.src, g.dst, g.stride);
  hipLaunchKernelGGL(k_zero_u64, dim3(nblk(nres, 256)), dim3(256), 0, c->stream, P->res, nres);
  for (const Launch &Lq : P->L) if ((e = launch(c, Lq))) break;
  hipGraph_t graph = nullptr;
  const hipError_t ce = hipStreamEndCapture(c->stream, &graph);
  if (e) { if (graph) (void) hipGraphDestroy(graph); return e; }
  if (ce != hipSuccess) { set_err(c, "graph capture failed: %s", hipGetErrorString(ce)); return FCFC_ERR_GPU; }
  P->graph = graph;
  HIPCHK(c, hipGraphInstantiate(&P->exec, P->graph, nullptr, nullptr, 0));
  *out = P.release();
  return 0;
}

/* One count of every job of the plan, histograms added into cnt (njob x
 * ntot; FCFC_GPU_CNT_DEVICE in the plan's flags: a device pointer). */
extern "C" int fcfc_gpu_plan_run(fcfc_gpu_plan *P, void *cnt) {
  if (!P || !cnt) return FCFC_ERR_ARG;
  fcfc_gpu_ctx *c = P->c;
  auto t0 = std::chrono::steady_clock::now();
  HIPCHK(c, hipSetDevice(c->device));
  HIPCHK(c, hipEventRecord(c->ev0, c->stream));
  HIPCHK(c, hipGraphLaunch(P->exec, c->stream));
  HIPCHK(c, hipEventRecord(c->ev1, c->stream));
  if (int e = deliver(c, P->jobs, P->ntot, P->res, P->ntot * (int) P->jobs.size(), P->flags, cnt, false)) return e;
  float ms = 0;
  HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
  c->stats.kernel_ms = ms;
  c->stats.total_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return 0;
}

extern "C" int fcfc_gpu_plan_destroy(fcfc_gpu_plan *P) {
  delete P;
  return 0;
}

/* Project-written autotuner: for jobs like (a, b, bins, flags) try grid and
 * run shapes (cells per maximum separation, z-cells per cell, A objects
 * per tile of FK_NW runs), timing each on a part of the list of runs (16
 * stretches spread over it: an eighth, a sixteenth beyond 16384 tiles) and
 * extrapolating to all runs (counts of at most 4096 tiles are timed
 * whole).  Every pair of cell_div and zdiv is timed (the best zdiv depends
 * on cell_div: a descent over one, then the other, missed the best pair of
 * a cross count), then the tile size.  The winner is cached in the
 * context for this geometry / binning / precision and density bucket and
 * used by later counts whose shape is left automatic. */
extern "C" int fcfc_gpu_autotune(fcfc_gpu_ctx *c, const fcfc_cat *a,
    const fcfc_cat *b, const fcfc_bins *bins, const double *bsize,
    uint32_t flags, int *best) {
  if (!c || !bins_ok(bins)) return FCFC_ERR_ARG;
  const int autoc = (flags & FCFC_GPU_AUTO) ? 1 : 0;
  if (!cat_ok(a) || (!autoc && !cat_ok(b))) { set_err(c, "invalid argument"); return FCFC_ERR_ARG; }
  const int grad = (flags & FCFC_GPU_GRADIENT) ? 1 : 0;
  const int mode = grad ? MODE_GRAD : (flags & FCFC_GPU_PREC_FP32) ? MODE_C32 :
                   ((flags & FCFC_GPU_PREC_PLAIN) ? MODE_P64 : MODE_C64);
  const int save_cd = c->t_cell_div, save_zd = c->t_zdiv, save_t = c->t_tile;
  std::vector<unsigned char> hcnt(8 * (size_t) bins->ntot);
  /* gradient timing: dL/dcnt = 1 in every bin (every pair contributes),
   * gradient of a only, as weight fitting asks for it */
  std::vector<double> gone(grad ? (size_t) bins->ntot : 0, 1.0);
  std::vector<double> gout(grad ? (size_t) std::max<int64_t>(a->n, 1) : 0);
  const uint32_t cflags = flags & ~(FCFC_GPU_CNT_DEVICE | FCFC_GPU_GRADIENT);
  auto run = [&]() -> int {
    if (grad)
      return fcfc_gpu_count_backward(c, a, b, bins, bsize, flags & FCFC_GPU_AUTO, gone.data(),
                                     gout.data(), nullptr);
    memset(hcnt.data(), 0, hcnt.size());
    return fcfc_gpu_count(c, a, b, bins, bsize, cflags, hcnt.data());
  };
  double bestms = 1e300;
  int bcd = 3, bzd = 8, bT = 0;
  int last_T = 0;
  /* FCFC_GPU_TUNE_LOG set and not "0": every candidate's timing on stderr */
  const char *tl = getenv("FCFC_GPU_TUNE_LOG");
  const bool tune_log = tl && strcmp(tl, "0") != 0;
  auto measure = [&](int cd, int zd, int T, double *est) -> int {
    c->t_cell_div = cd; c->t_zdiv = zd; c->t_tile = T;
    /* first pass: learn the number of tiles of this shape, counting 16 */
    c->tile_frac = 1 << 30;
    int e = run();
    if (e) return e;
    int nt = 0;
    HIPCHK(c, hipMemcpyAsync(&nt, c->last_nrun, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    /* small counts (a few thousand tiles, milliseconds) are timed whole: an
     * eighth of them is too few tiles to rank shapes */
    c->tile_frac = (nt <= 4096 * FK_NW) ? 1 : (nt > 16384 * FK_NW ? 16 : 8);
    e = run();
    if (e) return e;
    const int ns = fk_split(nt, 1, 1, 1, 1, c->tile_frac).ncap;     /* runs counted */
    *est = c->stats.kernel_ms * (double) nt / (double) std::max(1, ns);
    last_T = c->last_T;
    if (tune_log)
      fprintf(stderr, "fcfc_gpu_autotune: cell_div %d zcell_div %d tile %d: %d of %d runs "
              "in %.3f ms, estimate %.3f ms\n", cd, zd, last_T, ns, nt,
              c->stats.kernel_ms, *est);
    return 0;
  };
  int e = 0;
  const int cds[] = {2, 3, 4, 6};
  const int zds[] = {1, 2, 4, 8, 16};
  struct Cand { double est; int cd, zd, T; };
  std::vector<Cand> grid;
  for (int cd : cds) {
    for (int zd : zds) {
      double est;
      if ((e = measure(cd, zd, 0, &est))) break;
      grid.push_back({est, cd, zd, last_T});
      if (est < bestms) { bestms = est; bcd = cd; bzd = zd; bT = last_T; }
    }
    if (e) break;
  }
  /* the grid runs each shape at its automatic tile size; the best three
   * shapes are also timed at the other size the kernel family holds (FK_NT
   * for the hybrid gradient kernel).  4 FK_NT is left to the caller: since B
   * objects are read by scalar loads it loses (weighted DR of 2e5 x 2e6 15.6
   * against 15.1 ms, DD of 5e5 7.6 against 6.9) */
  std::sort(grid.begin(), grid.end(), [](const Cand &x, const Cand &y) { return x.est < y.est; });
  const int lmax = fk_lanes_max(bins->geometry, mode, grad || (flags & FCFC_GPU_WEIGHTED) ? 1 : 0,
                                (bins->tabtype || !zb_fits(bins)) ? 1 : 0);
  const int Ts[] = {FK_NT, 2 * FK_NT};
  for (size_t k = 0; k < grid.size() && k < 3 && !e; k++) {
    for (int T : Ts) {
      double est;
      if (T == grid[k].T || T > lmax * FK_NT) continue;
      if ((e = measure(grid[k].cd, grid[k].zd, T, &est))) break;
      if (est < bestms) { bestms = est; bcd = grid[k].cd; bzd = grid[k].zd; bT = last_T; }
    }
  }
  c->tile_frac = 0;
  c->t_cell_div = save_cd; c->t_zdiv = save_zd; c->t_tile = save_t;
  if (e) return e;
  /* cache for the density bucket of this job, keyed as the count (or the
   * gradient) plans it: the larger catalogue of a cross count is A */
  {
    JobPlan P;
    double lo[3] = {0, 0, 0}, hi[3] = {1, 1, 1};
    const fcfc_cat *ka = a, *kb = autoc ? a : b;
    if (!autoc && kb->n > ka->n) std::swap(ka, kb);
    if (bins->geometry == FCFC_GEOM_SURVEY) {
      for (int k = 0; k < 3; k++) { lo[k] = 1e300; hi[k] = -1e300; }
      Alloc tal(c, false);
      const fcfc_cat *ks[2] = {ka, kb};
      if ((e = bbox(c, tal, ks, autoc ? 1 : 2, lo, hi))) return e;
    }
    const int wt = (grad || (flags & FCFC_GPU_WEIGHTED)) ? 1 : 0;
    make_plan(c, bins, bsize, lo, hi, autoc, wt, mode, ka->n, kb->n, true, &P);
    bool found = false;
    for (auto &t : c->tuned)
      if (t.geom == bins->geometry && t.bintype == bins->bintype && t.mode == mode &&
          t.autoc == autoc && t.wt == wt && t.bucket == P.bucket) {
        t.cd = bcd; t.zd = bzd; t.T = bT; found = true;
      }
    if (!found) c->tuned.push_back({bins->geometry, bins->bintype, mode, autoc, wt,
                                    P.bucket, bcd, bzd, bT});
  }
  if (best) { best[0] = bcd; best[1] = bzd; best[2] = bT; best[3] = (int) lround(bestms * 1000); }
  return 0;
}
