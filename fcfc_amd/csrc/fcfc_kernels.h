/*
 * fcfc_kernels.h -- device-side data layout and pair arithmetic shared by the
 * gfx950 kernels of the pair-count engine.
 *
 * Layout in HBM (one catalogue, after the grid build):
 *   objects sorted by cell id  cid = (ix * ncy + iy) * ncz + iz,
 *   records of four FP64 values (x, y, z and |r|^2 for survey (s,mu) and
 *   (s_perp,pi), else the weight), w[] the weights where |r|^2 is in the
 *   record, idx[] = original object index, cell_start[ncell + 1].
 * A "row" is the set of cells sharing (ix, iy): its objects are contiguous and
 * ordered by z-cell, so every z-window of a row is one contiguous range.
 *
 * Work unit: a run = up to 64 R consecutive A objects of one row (R per lane
 * of one wavefront) inside a bounded z range, against a share of the strips.
 * For each xy offset (a "strip") the B objects that can be within the maximum
 * separation form at most three contiguous segments (three periodic images in
 * z).  Every wavefront of the persistent workgroups takes its own runs from a
 * global queue: its lanes load 64 B objects, drop those farther than the
 * maximum separation from the bounding box of the run, and every lane
 * evaluates its A objects against each of the others, which the FP64 forms
 * read into scalar registers and the FP32 ones pack, relative to the run's
 * centre, into the wavefront's LDS chunk.  The histograms are shared by the
 * workgroup.
 *
 * Arithmetic contract (FP64 path), after FCFC's AVX-512 leaf kernels
 * (src/fcfc/2pt_box/metric_common.c:377-534):  B objects are staged as
 *   b' = fl(b + D)  with D the periodic image offset in {-L, 0, +L},
 * and every pair computes  dx = fl(b'.x - a.x), dz2 = fl(dz*dz),
 *   s2 = fma(dy, dy, fma(dx, dx, dz2)),
 * which is the reference's "vectorise node b" block (x1 = b - shift,
 * metric_common.c:1154-1163).  The mu index is floor of the EXACT quotient
 * fl(dz2*nmu^2)/s2, i.e. trunc(RZ(.)) as in metric_common.c:484-486.
 */
#ifndef FCFC_KERNELS_H
#define FCFC_KERNELS_H

#include <stdint.h>

#define FK_NT        512       /* threads per workgroup (8 wave64)          */
#define FK_NW        8         /* wavefronts per workgroup                  */
#define FK_MAXSEG    3         /* z images per strip                        */
#define FK_CH        64        /* B objects per wavefront's LDS chunk       */
#define FK_OUT       0xFFFFu   /* table sentinel: outside [s2min, s2max)    */
#define FK_QCAP      160       /* FP32 re-evaluation queue per wavefront    */

/* Binning constants passed by value to the kernels. */
struct FkBins {
  int bintype, geometry;
  int ns, nmu, np, ntot;
  int nsh, ntoh;             /* LDS histogram row stride (odd, > ns), slots */
  int nslot, slot_pad;       /* slots of one copy, with the dummy row       */
  int tabtype;               /* 0 integer table, 1 hybrid table             */
  int soff, poff;            /* (int) s2min, (int) pmin (or pi^2 min)       */
  int stab_len, ptab_len;    /* table lengths without sentinels             */
  int ssearch, psearch;      /* hybrid lookups: tables too long for LDS, bin
                                by binary search over the edges instead    */
  int scap32, pcap32;        /* last entry of the zero-based FP32 tables    */
  double s2min, s2max;       /* squared s (or s_perp) range                 */
  double pmin, pmax;         /* pi range (box) or pi^2 range (survey)       */
  double nmu2;               /* nmu * nmu as double                          */
  double nmu_d;              /* nmu as double                                */
  double mu_c;               /* 2^36 + 1 - mu_sh: the fixed-point mu value  */
  double mu_cmax;            /* 2^36 + nmu + 1.5: its ceiling (survey)       */
  unsigned mu_t16, mu_pad;   /* mu bin settled exactly when the fraction     */
                             /* (low 16 bits) of that value is >= mu_t16     */
  double s2_exact;           /* ... or s^2 is below this value               */
  double q_c;                /* survey (s_perp, pi), FP64 integer tables,   */
  double q_caps, q_capp;     /* pi^2 and s_perp^2 in fixed point (fk_sv64): */
  double q_bmin;             /* addend, ceilings, least |a+b|^2 of the fast */
  unsigned q_t16, q_pad;     /* path, fraction threshold of edge cells      */
  double s2low;              /* masked survey (s,mu): least s^2 of a counted   */
                             /* pair (just above -1 for ranges from 0)         */
  double s2skip, pskip;      /* forms without a mask: a pair at s^2 >= s2skip */
  float s2skip32, skip_pad;  /* or pi >= pskip is out of range (FP64 / FP32) */
  float m32s, m32p;          /* FP32: values at or beyond are out of range   */
  float win2s, win2p;        /* FP32 tables: window 2 e of the edge cells,   */
                             /* the largest over the jobs of a launch        */
  const uint16_t *stab;      /* device tables (global), staged to LDS       */
  const uint16_t *ptab;
  const double *s2bin;       /* edges for the hybrid refinement              */
  const double *pbin;
};

/* Grid geometry (shared by A and B of one job). */
struct FkGrid {
  int ncx, ncy, ncz;
  int periodic;
  double ox, oy, oz;         /* origin                                       */
  double wx, wy, wz;         /* cell widths                                  */
  double Lx, Ly, Lz;         /* box sizes (periodic)                         */
  double R2;                 /* squared maximum 3-D separation (padded)     */
  double Rxy2;               /* squared maximum xy separation (padded)      */
  double hz_const;           /* >= 0: fixed z half-window (box s_perp,pi)   */
};

/* One sorted object, read as a whole by scalar and vector loads.  q: |r|^2
 * for survey (s,mu) and (s_perp,pi) bins, else the weight (weighted jobs). */
struct alignas(32) FkRec { double x, y, z, q; };

/* rec, w and idx are indexed as cell_start counts: from the first object of
 * the call's first catalogue */
struct FkCat {
  int n, pad;
  const FkRec *rec;
  const double *w;           /* weights that are not in the records          */
  const int *idx;
  const int *cell_start;
};

/* A run: the A objects [p0, p1) of one row, counted against the strips of
 * its job.  A work item is a run with a share of the strip list, so that the
 * queue stays long (items of one run add into the same histograms; only the
 * item of the first share counts the pairs inside the run). */
struct FkRun { int row, p0, p1, pad; };

/* Floor of the exact quotient a / b for a >= 0, b > 0 (b not tiny):
 * approximate quotient from the hardware reciprocal, then one-step
 * corrections with exact-sign fma residuals. */
__device__ __forceinline__ double fk_floor_div(double a, double b) {
  double q = a * __builtin_amdgcn_rcp(b);
  double m = __builtin_floor(q);
  if (__builtin_fma(-m, b, a) < 0.0) m -= 1.0;
  else if (__builtin_fma(-(m + 1.0), b, a) >= 0.0) m += 1.0;
  return m;
}

/* integer square root of 0 <= m < 2^22 (mu table, setup_cf.c:513-531):
 * sqrt(m + 1/2) is at least 1/(4(n+1)) away from any integer. */
__device__ __forceinline__ int fk_isqrt(int m) {
  return (int) __builtin_sqrtf((float) m + 0.5f);
}

#endif
