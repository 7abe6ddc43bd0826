// Batched CG-Lanczos Fiedler solver: every segment of a bisection level runs
// the reference's restarted CG-Lanczos (fiedler.c:434-621) at once.
//
// Rows of the level are grouped in tiles of RSB_TILE rows that never cross a
// segment, one workgroup per tile.  Each workgroup writes the partial sums of
// its tile (fixed reduction tree), so results do not depend on block
// scheduling.  The segment totals and scalar updates are formed by the launch
// that needs them (segments of at most LZ_FUSE_TILES tiles, "Fused
// iterations" below) or by a small k_lz_fin launch after each reduction (one
// workgroup per segment), so no workgroup ever waits on another inside a
// launch.  One CG-Lanczos iteration is two launches over all rows of the
// level:
//   k_lz_apply    p = beta (p_old - mean) + r formed on the fly for each row
//                 and its neighbours (staged in LDS per tile), w = L p from the
//                 tile's 12- or 16-bit entries (the SELL-64 global form where a
//                 tile's halo does not fit), pap = w . (p - mean(p))
//   k_lz_rupdate  r = r - alpha w, rtr = r . r, tridiagonal entries, stop test
// (FP32 passes on few tiles fold the update into the next apply, below).
// The Lanczos basis vector of iteration it is r_it / |r_it|: the residuals
// themselves are kept, r_it in basis slot it, and the Ritz step scales them.
// The mean of p is removed lazily (fiedler.c:20-30 `ortho`): w = L p is
// evaluated in the difference form sum_j w_ij (p_i - p_j), which the mean
// does not change, and the stored p keeps its mean, subtracted when used.
// Segments that converged or are between passes skip every launch at the
// first instruction.
//
// Precision: vectors are T (double, or float); every scalar and the
// tridiagonal eigen-solve are FP64.  With T = float, the dot products of a
// thread's rows are summed in FP32 with a running correction, to within
// 2^-24 of the sum of the products' magnitudes (acc_t), and block partials
// are combined in FP64.
#include <algorithm>
#include <vector>

#include <cfloat>

#include "state.hpp"

struct lz_args {
  const int *seg;        // 5*nseg: cstart, n, p, r0, pstart
  const int *tile;       // 3*ntiles: seg, row0, row1
  const int *seg_tiles;  // 2*nseg: first tile, tile count
  const int *row_elem;
  int nseg;
  int *status, *iter, *k, *npass, *niter, *miter;
  double *sc, *T, *y, *partial;
  double *rn;  // (miter_max + 1) per segment: 1 / |r_j|
  int mpass;
  int mode;  // start vector: 0 reference, 1 caller per element, 2 learned per row
  int max_n; // mode 2: segments with more rows take the reference start
  double tol;
  double stall;  // > 0: a pass whose Ritz value moved by at most this (relative) ends the solve
  int stall_min; // ... from this pass on
  double plateau; // > 0: a pass whose Ritz residual is at most plateau_max and not below
                  // this times the one two passes back ends the solve (from the fourth pass)
  double plateau_max;
  int miter_max;
  const int *act_tiles;  // if set: blockIdx.x -> tile (compacted active list)
  const int *act_segs;   // if set: blockIdx.x -> segment, for k_lz_fin
  int pstride;           // partial is slot-major: slot k of tile t at k * pstride + t
  struct lz_it *st0;     // if set: FIN_SETUP1 fills the state the fused iterations start from
};

// What a tile's workgroup needs to know, in one record of 64 bytes: one
// load instead of a chain of them (list entry -> tile -> segment table,
// halo table).  The running list of the fused iterations holds copies.
struct __attribute__((aligned(16))) lz_desc {
  int s, row0, row1, pstart;
  int n, first, count, nhalo;
  int64_t halo_off;
  int ti, pad0;
  int pad[4];
};

// Scalar state of a segment between two launches of the fused iterations.
struct lz_it {
  double rtz1, rtz2, beta, pap, pap_old, meanp, alpha, rtol;
  int it, mi;  // iteration whose apply ran last; the pass's length
};
// field by field: a struct copy went through LDS
__device__ inline void it_load(lz_it &x, const lz_it *__restrict__ p) {
  x.rtz1 = p->rtz1, x.rtz2 = p->rtz2, x.beta = p->beta, x.pap = p->pap, x.pap_old = p->pap_old;
  x.meanp = p->meanp, x.alpha = p->alpha, x.rtol = p->rtol, x.it = p->it, x.mi = p->mi;
}
__device__ inline void it_store(lz_it *__restrict__ p, const lz_it &x) {
  p->rtz1 = x.rtz1, p->rtz2 = x.rtz2, p->beta = x.beta, p->pap = x.pap, p->pap_old = x.pap_old;
  p->meanp = x.meanp, p->alpha = x.alpha, p->rtol = x.rtol, p->it = x.it, p->mi = x.mi;
}

#define SC(s, j) a.sc[(size_t)(s) * LZ_NSC + (j)]

// Every product that meets a sum on the iterations' path is an explicit
// fused multiply-add, and the sums themselves contract nothing: left to the
// compiler, which products were fused depended on the code around them, and
// two kernels doing the same sum differed in the last bit.
__device__ inline float fmat(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ inline double fmat(double a, double b, double c) { return __builtin_fma(a, b, c); }

template <typename T>
struct acc_t;
template <>
struct acc_t<double> {
  double v = 0.0;
  __device__ inline void dot(double x, double y) { v = fmat(x, y, v); }
  // the product rounded before it is added
  __device__ inline void dot2(double x, double y) {
#pragma clang fp contract(off)
    v = v + x * y;
  }
  __device__ inline void add(double x) {
#pragma clang fp contract(off)
    v = v + x;
  }
  __device__ inline double value() const { return v; }
};
template <>
struct acc_t<float> {
  float s = 0.f, c = 0.f;
  // s + xy rounded once (et: that rounding's error).  ep, the rounding error
  // of the product alone, belongs to the sum of rounded products (dot2); here
  // it is counted although the product was never rounded, so a sum is off by
  // up to 2^-24 sum |x y| (at most 5e-8, 1.3e-8 and 4e-9 of it in 20,000 sums
  // of 4, 64 and 1,024 terms of one sign; 1e-14, 1e-13 and 2e-12 without ep).
  // It stays because it decides bits: this is what the two-sum of x * y has
  // always compiled to under contraction, and c + et moves 2.3% of the
  // elements of 250k holed quads in 256 parts and 0.2% of a 2M-hex pipe's to
  // other parts, at the same cut (-0.002% on the pipe) and 0.4% and 0.2% fewer
  // iterations, as many as without the folded update; the parts of four other
  // meshes stay the same.
  __device__ inline void dot(float x, float y) {
#pragma clang fp contract(off)
    const float ep = fmat(x, y, -(x * y));
    const float t = fmat(x, y, s), bb = t - s;
    const float et = (s - (t - bb)) + fmat(x, y, -bb);
    s = t;
    c = c + (ep + et);
  }
  // the product rounded before it is added
  __device__ inline void dot2(float x, float y) {
#pragma clang fp contract(off)
    const float p = x * y, ep = fmat(x, y, -p);
    const float t = s + p, bb = t - s;
    const float et = (s - (t - bb)) + (p - bb);
    s = t;
    c = c + (ep + et);
  }
  __device__ inline void add(float x) {
#pragma clang fp contract(off)
    const float t = s + x, bb = t - s;
    const float et = (s - (t - bb)) + (x - bb);
    s = t;
    c = c + et;
  }
  __device__ inline double value() const { return (double)s + (double)c; }
};

// Tile prologue: returns false if the block has nothing to do.
struct tile_t {
  int ti, s, row0, row1, pstart, n, first, count;
};
// Workgroups are handed to the XCDs round robin (workgroup b to XCD b % 8),
// so consecutive tiles, which are neighbours in space, would land in eight
// different L2 caches.  With nlist > 0 the list of nlist tiles is split in
// eight contiguous parts, one per XCD, so a tile's halo rows are mostly rows
// its XCD has just read (grid: nlist rounded up to a multiple of 8).
#define LZ_XCDS 8
// running tiles up to which an FP32 pass folds its r-update into the apply.
// Whole calls at 0 / 1,024 / 2,048 / 4,096, fused launches: 250k holed quads
// 311 / 256 / 254 / 254 ms, 2M-hex pipe 693 / 690 / 670 / 671, 1M hexes with the
// learned start 63.3 / 61.9 / 61.1 / 61.4; 256^3 hexes in 65,536 parts at 2,048
// / 4,096 / 8,192: 4,796 / 4,792 / 4,798
#define LZ_FOLD_TILES 4096
// segments of more tiles than this take 512-thread finishing workgroups
#define LZ_FIN_WIDE 1024
// profiling samples one SpMV launch in this many (coprime with the 8
// iterations between list compactions and the 50 of a pass)
#define LZ_PROF_EVERY 11
__device__ inline int list_index(int nlist) {
  if (nlist <= 0) return blockIdx.x;
  const int per = (int)(gridDim.x / LZ_XCDS);
  const int i = (int)(blockIdx.x % LZ_XCDS) * per + (int)(blockIdx.x / LZ_XCDS);
  return i < nlist ? i : -1;
}
__device__ inline bool tile_of(const lz_args &a, int want_status, tile_t &t, int nlist = 0) {
  const int li = list_index(nlist);
  if (li < 0) return false;
  const int ti = a.act_tiles ? a.act_tiles[li] : li;
  t.ti = ti;
  t.s = a.tile[3 * ti];
  if (a.status[t.s] != want_status) return false;
  t.row0 = a.tile[3 * ti + 1];
  t.row1 = a.tile[3 * ti + 2];
  t.n = a.seg[a.nseg + t.s];
  t.pstart = a.seg[4 * a.nseg + t.s];
  t.first = a.seg_tiles[2 * t.s];
  t.count = a.seg_tiles[2 * t.s + 1];
  return true;
}

// Write the block's partial sums (a fixed reduction tree) for the tile.
// The segment totals are formed by k_lz_fin in the next launch: no
// cross-workgroup handshake inside a kernel, so no device-scope fences.
template <int NV>
__device__ inline void publish(const lz_args &a, const tile_t &t, double (&v)[NV]) {
  __shared__ double red[(RSB_BLOCK / RSB_WAVE) * (NV > 4 ? NV : 4)];
  block_sum<NV, RSB_BLOCK / RSB_WAVE>(v, red);
  if (threadIdx.x == 0)
    for (int k = 0; k < NV; k++) a.partial[(size_t)k * a.pstride + t.ti] = v[k];
}

// ---------------------------------------------------------------------------
// Start vector (fiedler.c:570-585): x_i = i + 1, plus 1000 n on the first half
// of the pre-partition order; then mean removed and normalised (FP64).
// mode 0: reference start; mode 1: caller-supplied per-element start;
// mode 2: per-row start (the learned warm start's prediction).
__device__ inline double start_value(int mode, int i, int n, const float *start, int e,
                                     int row) {
  if (mode == 1) return (double)start[e];
  if (mode == 2) return (double)start[row];
  double v = i + 1.0;
  if (i < n / 2) v += (double)(1000 * (long long)n);
  return v;
}

template <typename T>
__global__ void __launch_bounds__(RSB_BLOCK) k_lz_start(lz_args a, int phase, int mode,
                                                        const float *start, T *f) {
  tile_t t;
  if (!tile_of(a, LZ_SETUP, t)) return;
  double m = phase > 0 ? SC(t.s, SC_M0) : 0.0;
  double sc = phase > 1 ? SC(t.s, SC_N0) : 0.0;
  double v[1] = {0.0};
  for (int row = t.row0 + threadIdx.x; row < t.row1; row += blockDim.x) {
    int i = row - t.pstart;
    double x = 0.0;
    if (i < t.n) {
      x = start_value(mode, i, t.n, start, a.row_elem[row], row);
      if (phase == 0) v[0] += x;
      else if (phase == 1) v[0] += (x - m) * (x - m);
    }
    if (phase == 2) f[row] = i < t.n ? (T)((x - m) * sc) : (T)0;
  }
  if (phase == 2) return;
  publish<1>(a, t, v);
}

// Pass setup (fiedler.c:441-456): r = f - mean_f; then r -= mean(r);
// rtr, |r|, target tol |r|.
template <typename T>
__global__ void __launch_bounds__(RSB_BLOCK) k_lz_setup(lz_args a, int phase, const T *f, T *r,
                                                        T *p) {
  tile_t t;
  if (!tile_of(a, LZ_SETUP, t)) return;
  acc_t<T> acc;
  if (phase == 0) {
    T mf = (T)SC(t.s, SC_MEANF);
    for (int row = t.row0 + threadIdx.x; row < t.row1; row += blockDim.x) {
      int i = row - t.pstart;
      T x = i < t.n ? (T)(f[row] - mf) : (T)0;
      r[row] = x;
      p[row] = (T)0;
      acc.add(x);
    }
  } else {
    T mr = (T)SC(t.s, SC_TMP);
    for (int row = t.row0 + threadIdx.x; row < t.row1; row += blockDim.x) {
      int i = row - t.pstart;
      if (i < t.n) {
        T x = r[row] - mr;
        r[row] = x;
        acc.dot(x, x);
      }
    }
  }
  double v[1] = {acc.value()};
  publish<1>(a, t, v);
}

// ---------------------------------------------------------------------------
// One row of L q in the difference form sum_j w_ij (q_i - q_j), where q is
// formed on the fly from the previous search direction and the residual:
// q = beta (p - m) + r (q = r on the first iteration of a pass).  The packed
// entries of a SELL-64 slice are read 8 at a time so that each thread keeps 8
// gathers in flight.
// The residual of iteration it: r itself, or with FOLD (the FP32 path)
// r_prev - alpha w_prev, the update of the previous iteration, formed where
// it is read (fiedler.c:486-488).
// r - alpha w with one rounding (the r-update of both forms)
__device__ inline float rsub(float r, float alpha, float w) { return __builtin_fmaf(-alpha, w, r); }
__device__ inline double rsub(double r, double alpha, double w) { return __builtin_fma(-alpha, w, r); }
template <typename T, bool FOLD>
__device__ inline T rval(const T *__restrict__ r, const T *__restrict__ wp, uint32_t c, T alpha) {
  return FOLD ? rsub(r[c], alpha, wp[c]) : r[c];
}
template <typename T, bool FIRST, bool FOLD>
__device__ inline T qval(const T *__restrict__ p, const T *__restrict__ r,
                         const T *__restrict__ wp, uint32_t c, T beta, T m, T alpha) {
  return FIRST ? r[c] : fmat(beta, p[c] - m, rval<T, FOLD>(r, wp, c, alpha));
}

template <typename T, bool FIRST, bool FOLD>
__device__ inline T lap_row_q(const uint32_t *__restrict__ e, int wd, T qi,
                              const T *__restrict__ p, const T *__restrict__ r,
                              const T *__restrict__ wp, T beta, T m, T alpha) {
  T sum = (T)0;
  int j = 0;
  for (; j + 8 <= wd; j += 8) {
    uint32_t q[8];
    T v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) q[u] = __builtin_nontemporal_load(e + (size_t)(j + u) * RSB_WAVE);
#pragma unroll
    for (int u = 0; u < 8; u++)
      v[u] = qval<T, FIRST, FOLD>(p, r, wp, q[u] & 0x0fffffffu, beta, m, alpha);
#pragma unroll
    for (int u = 0; u < 8; u++) sum = fmat((T)(q[u] >> 28), qi - v[u], sum);
  }
  for (; j < wd; j++) {
    uint32_t q = __builtin_nontemporal_load(e + (size_t)j * RSB_WAVE);
    sum = fmat((T)(q >> 28), qi - qval<T, FIRST, FOLD>(p, r, wp, q & 0x0fffffffu, beta, m, alpha),
               sum);
  }
  return sum;
}

// What the folded apply adds: the residual of iteration it written for the
// tile's rows, and the sums r.r, r.w and w.w from which the finishing step
// forms |r - alpha w|^2, the next residual's norm.
template <typename T>
struct fold_t {
  const T *wp;  // w of the previous iteration
  T *rn;        // r of this iteration (written)
  T alpha;      // alpha of the previous iteration
  acc_t<T> rr, rw, ww;
};

// Fused search-direction update and Laplacian apply (fiedler.c:460-475):
//   q = beta (p_old - mean_p) + r,  w = L q  (r: basis slot it)
// and the segment sums of q, w.q and w, from which the last block forms
// mean_p and pap = w.(q - mean_p), then alpha = rtz1 / pap.
template <typename T, bool FIRST, bool FOLD>
__device__ inline void lz_apply_rows(const lz_args &a, const tile_t &t, const T *__restrict__ r,
                                     const T *__restrict__ pold, T *__restrict__ pnew,
                                     T *__restrict__ w, T beta, T m,
                                     const int64_t *__restrict__ slice_off,
                                     const int *__restrict__ slice_w,
                                     const uint32_t *__restrict__ ell, acc_t<T> &sq,
                                     acc_t<T> &swq, acc_t<T> &sw, fold_t<T> &fd) {
  constexpr bool UPD = FOLD && !FIRST;
  for (int row = t.row0 + threadIdx.x; row < t.row1; row += blockDim.x) {
    const bool real = row - t.pstart < t.n;
    const T ri = rval<T, UPD>(r, fd.wp, (uint32_t)row, fd.alpha);
    T qi = (T)0, wi = (T)0;
    if (real) {
      qi = FIRST ? ri : fmat(beta, pold[row] - m, ri);
      const int sl = row >> 6;
      wi = lap_row_q<T, FIRST, UPD>(ell + slice_off[sl] + (row & 63), slice_w[sl], qi, pold, r,
                                    fd.wp, beta, m, fd.alpha);
      sq.add(qi);
      swq.dot(wi, qi);
      sw.add(wi);
      if (FOLD) fd.rr.dot(ri, ri), fd.rw.dot(ri, wi), fd.ww.dot(wi, wi);
    }
    pnew[row] = qi;
    w[row] = wi;
    if (UPD) fd.rn[row] = ri;
  }
}

// LDS-tiled rows (tiles.hip): q for the tile's rows and its halo is staged
// in LDS once; every neighbour is then read from LDS through a 16-bit local
// index, 8 entries per 16-byte load.
// Where a slice's entries lie in the form the solve reads: its offset, width
// and (12-bit form) class slots, one 16-byte record instead of three arrays.
struct __attribute__((aligned(16))) slice_rec {
  int64_t off;
  int w, c;
};
struct tiled_args {
  const slice_rec *slice;
  const int64_t *slice_off;
  const int *slice_w;
  const uint32_t *ell;
  const int *nhalo;
  const int64_t *halo_off;
  const int *halo;
  const int64_t *off16;
  const int *w16;
  const uint16_t *e16;
  const uint32_t *e12;  // the 12-bit form (tiles.hip), or nullptr
};

#define TB_LOCAL 4096
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

template <typename T>
__device__ inline void acc_entry(uint32_t e, T qi, const T *ql, T &sum) {
  sum = fmat((T)(e >> 12), qi - ql[e & 0xfffu], sum);
}

// The sums a row of the 16-bit form adds.  ODD: the thread's second and
// fourth row; there the last product of the row (w.q, or w.w with the folded
// update) is rounded before it is added.  (That is how the rows of this form
// have been summed since it exists; results stay what they were to the bit.)
template <bool ODD, typename T, bool FOLD>
__device__ inline void row_sums16(T qi, T wi, T ri, acc_t<T> &sq, acc_t<T> &swq, acc_t<T> &sw,
                                  fold_t<T> &fd) {
  sq.add(qi);
  if (ODD && !FOLD) swq.dot2(wi, qi);
  else swq.dot(wi, qi);
  sw.add(wi);
  if (FOLD) {
    fd.rr.dot(ri, ri), fd.rw.dot(ri, wi);
    if (ODD) fd.ww.dot2(wi, wi);
    else fd.ww.dot(wi, wi);
  }
}

// One row of the tiled apply: its 16-bit entries (groups of 8, then groups
// of 4 and 2) against the LDS window; writes p', w and the basis entry.
template <bool ODD, typename T, bool FOLD>
__device__ inline void apply_row_tiled(int row, const tile_t &t, const tiled_args &ta,
                                       const T *ql, const T *rl, T *__restrict__ pnew,
                                       T *__restrict__ w, int nreal, acc_t<T> &sq,
                                       acc_t<T> &swq, acc_t<T> &sw, fold_t<T> &fd) {
  const int li = row - t.row0, sl = row >> 6;
  const uint16_t *sbase = ta.e16 + ta.off16[sl];
  const u32x4 *ep = (const u32x4 *)(sbase + (row & 63) * 8);
  const int w16 = ta.w16[sl], nb = w16 >> 3;
  const T qi = ql[li];
  T sum = (T)0;
  for (int jb = 0; jb < nb; jb++) {
    const u32x4 v = __builtin_nontemporal_load(ep + (size_t)jb * RSB_WAVE);
    acc_entry(v.x & 0xffffu, qi, ql, sum);
    acc_entry(v.x >> 16, qi, ql, sum);
    acc_entry(v.y & 0xffffu, qi, ql, sum);
    acc_entry(v.y >> 16, qi, ql, sum);
    acc_entry(v.z & 0xffffu, qi, ql, sum);
    acc_entry(v.z >> 16, qi, ql, sum);
    acc_entry(v.w & 0xffffu, qi, ql, sum);
    acc_entry(v.w >> 16, qi, ql, sum);
  }
  if (w16 & 4) {  // a group of 4 entries
    const u32x2 v =
        __builtin_nontemporal_load((const u32x2 *)(sbase + nb * 512 + (row & 63) * 4));
    acc_entry(v.x & 0xffffu, qi, ql, sum);
    acc_entry(v.x >> 16, qi, ql, sum);
    acc_entry(v.y & 0xffffu, qi, ql, sum);
    acc_entry(v.y >> 16, qi, ql, sum);
  }
  if (w16 & 2) {  // a group of 2 entries
    const unsigned v = __builtin_nontemporal_load(
        (const unsigned *)(sbase + nb * 512 + (w16 & 4) * 64 + (row & 63) * 2));
    acc_entry(v & 0xffffu, qi, ql, sum);
    acc_entry(v >> 16, qi, ql, sum);
  }
  pnew[row] = qi;
  w[row] = sum;
  const T ri = FOLD ? rl[li] : (T)0;  // the tile's r is kept in LDS only to fold
  if (li < nreal) row_sums16<ODD, T, FOLD>(qi, sum, ri, sq, swq, sw, fd);
}

// Where the entries of a thread's (up to four) rows lie: row t.row0 +
// threadIdx.x + 256 k is in slice (t.row0 >> 6) + wave + 4 k, the same for
// the whole wave, so these are scalar loads; they are issued before the
// window is staged (the kernel has stored nothing yet) and are back when the
// rows want them.
#define LZ_RPT (RSB_TILE / RSB_BLOCK)
struct slice_meta {
  int64_t off[LZ_RPT];
  int w[LZ_RPT], c[LZ_RPT];  // widths (0: no such rows); class slots (12-bit form)
};
__device__ inline slice_meta load_meta(const tile_t &t, const tiled_args &ta) {
  slice_meta m;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / RSB_WAVE);
#pragma unroll
  for (int k = 0; k < LZ_RPT; k++) {
    const int r = t.row0 + wave * RSB_WAVE + k * RSB_BLOCK;
    const slice_rec q = ta.slice[min(r, t.row1 - 1) >> 6];
    m.off[k] = q.off, m.w[k] = r < t.row1 ? q.w : 0, m.c[k] = q.c;
  }
  return m;
}

// R rows per thread and step: the entries of all R rows are loaded before
// any is summed, so each lane keeps up to 4R 16-byte loads in flight.  Rows
// whose slice is wider than 32 entries take apply_row_tiled.  Missing groups
// are zero words (weight 0), which add exact zeros.
template <typename T, int R, bool FOLD>
__device__ inline void apply_rows_batched(const tile_t &t, const tiled_args &ta,
                                          const slice_meta &sm, const T *ql, const T *rl,
                                          T *__restrict__ pnew, T *__restrict__ w, int nreal,
                                          acc_t<T> &sq, acc_t<T> &swq, acc_t<T> &sw,
                                          fold_t<T> &fd) {
#pragma unroll
  for (int k0 = 0; k0 < LZ_RPT; k0 += R) {
    const int row0 = t.row0 + threadIdx.x + k0 * RSB_BLOCK;
    if (row0 >= t.row1) break;
    int rows[R], wd[R];
    const uint16_t *base[R];
    bool wide = false;
#pragma unroll
    for (int k = 0; k < R; k++) {
      rows[k] = row0 + k * RSB_BLOCK;
      base[k] = ta.e16 + sm.off[k0 + k];
      wd[k] = sm.w[k0 + k];
      wide |= wd[k] > 32;
    }
    if (wide) {
#pragma unroll
      for (int k = 0; k < R; k++)
        if (rows[k] < t.row1) {
          if (k & 1)
            apply_row_tiled<true, T, FOLD>(rows[k], t, ta, ql, rl, pnew, w, nreal, sq, swq, sw, fd);
          else
            apply_row_tiled<false, T, FOLD>(rows[k], t, ta, ql, rl, pnew, w, nreal, sq, swq, sw,
                                            fd);
        }
      continue;
    }
    u32x4 v[R][4];
    u32x2 tl[R];
    unsigned t2[R];
#pragma unroll
    for (int k = 0; k < R; k++) {
#pragma unroll
      for (int g = 0; g < 4; g++)
        v[k][g] = g < (wd[k] >> 3)
                      ? __builtin_nontemporal_load((const u32x4 *)(base[k] + (rows[k] & 63) * 8) +
                                                   g * RSB_WAVE)
                      : (u32x4){0u, 0u, 0u, 0u};
      const uint16_t *tail = base[k] + (wd[k] >> 3) * 512;
      tl[k] = (wd[k] & 4) ? __builtin_nontemporal_load((const u32x2 *)(tail + (rows[k] & 63) * 4))
                          : (u32x2){0u, 0u};
      t2[k] = (wd[k] & 2) ? __builtin_nontemporal_load(
                                (const unsigned *)(tail + (wd[k] & 4) * 64 + (rows[k] & 63) * 2))
                          : 0u;
    }
#pragma unroll
    for (int k = 0; k < R; k++) {
      if (rows[k] >= t.row1) continue;
      const int li = rows[k] - t.row0;
      const T qi = ql[li];
      T sum = (T)0;
#pragma unroll
      for (int g = 0; g < 4; g++) {
        acc_entry(v[k][g].x & 0xffffu, qi, ql, sum);
        acc_entry(v[k][g].x >> 16, qi, ql, sum);
        acc_entry(v[k][g].y & 0xffffu, qi, ql, sum);
        acc_entry(v[k][g].y >> 16, qi, ql, sum);
        acc_entry(v[k][g].z & 0xffffu, qi, ql, sum);
        acc_entry(v[k][g].z >> 16, qi, ql, sum);
        acc_entry(v[k][g].w & 0xffffu, qi, ql, sum);
        acc_entry(v[k][g].w >> 16, qi, ql, sum);
      }
      acc_entry(tl[k].x & 0xffffu, qi, ql, sum);
      acc_entry(tl[k].x >> 16, qi, ql, sum);
      acc_entry(tl[k].y & 0xffffu, qi, ql, sum);
      acc_entry(tl[k].y >> 16, qi, ql, sum);
      acc_entry(t2[k] & 0xffffu, qi, ql, sum);
      acc_entry(t2[k] >> 16, qi, ql, sum);
      pnew[rows[k]] = qi;
      w[rows[k]] = sum;
      const T ri = FOLD ? rl[li] : (T)0;
      if (li < nreal) {
        if (k & 1) row_sums16<true, T, FOLD>(qi, sum, ri, sq, swq, sw, fd);
        else row_sums16<false, T, FOLD>(qi, sum, ri, sq, swq, sw, fd);
      }
    }
  }
}

// 12-bit index k (0..20) of a 32-byte block held in eight words
template <int K>
__device__ inline unsigned e12_at(const unsigned (&wd)[8]) {
  constexpr int bit = 12 * K, i = bit / 32, sh = bit % 32;
  if constexpr (sh <= 20) return (wd[i] >> sh) & 0xfffu;
  else return __builtin_amdgcn_alignbit(wd[i + 1], wd[i], sh) & 0xfffu;
}

// One slot of the 12-bit form: its weight 2^e from the slice's class
// bounds (slots ordered 4s, 2s, 1s; n42 = n4 + n2; both uniform in the
// wave, so e is scalar work).  Scaling by 2^e is exact: the sum rounds as
// sum + w (qi - q) would.
__device__ inline float ldexp_t(float x, int e) { return __builtin_ldexpf(x, e); }
__device__ inline double ldexp_t(double x, int e) { return __builtin_ldexp(x, e); }
// m4 and m42 hold bit s for the slots s < n4 and s < n42 (shifts and masks
// of wave-uniform words: scalar work).
template <typename T>
__device__ inline void acc12(unsigned idx, int s, uint64_t m4, uint64_t m42, T qi, const T *ql,
                             T &sum) {
  const int e = (int)((m4 >> s) & 1u) + (int)((m42 >> s) & 1u);
  sum += ldexp_t(qi - ql[idx], e);
}

template <typename T, int K0, int N>
__device__ inline void acc12_words(const unsigned (&wd)[8], int s0, uint64_t m4, uint64_t m42,
                                   T qi, const T *ql, T &sum) {
  if constexpr (N > 0) {
    acc12(e12_at<K0>(wd), s0 + K0, m4, m42, qi, ql, sum);
    acc12_words<T, K0 + 1, N - 1>(wd, s0, m4, m42, qi, ql, sum);
  }
}

// The tiled rows on the 12-bit form: R rows per thread and step, every
// word of their blocks and tails loaded before any is summed.  The 64 rows
// of a wave are one slice, so block and tail counts are uniform in a wave.
template <typename T, int R, bool FOLD>
__device__ inline void apply_rows_e12(const tile_t &t, const tiled_args &ta, const slice_meta &sm,
                                      const T *ql, const T *rl, T *__restrict__ pnew,
                                      T *__restrict__ w, int nreal, acc_t<T> &sq, acc_t<T> &swq,
                                      acc_t<T> &sw, fold_t<T> &fd) {
#pragma unroll
  for (int k0 = 0; k0 < LZ_RPT; k0 += R) {
    const int row0 = t.row0 + threadIdx.x + k0 * RSB_BLOCK;
    if (row0 >= t.row1) break;
    int rows[R], nb[R], tw[R], cc[R];
    u32x4 bw[R][2][2], tl[R];
#pragma unroll
    for (int k = 0; k < R; k++) {
      rows[k] = row0 + k * RSB_BLOCK;
      const int lane = rows[k] & 63, info = sm.w[k0 + k];
      nb[k] = info & 0xff, tw[k] = info >> 8;
      const uint32_t *base = ta.e12 + sm.off[k0 + k];
      cc[k] = sm.c[k0 + k];
#pragma unroll
      for (int b = 0; b < 2; b++)
#pragma unroll
        for (int h = 0; h < 2; h++)
          bw[k][b][h] = b < nb[k] ? __builtin_nontemporal_load(
                                        (const u32x4 *)(base + (size_t)(2 * b + h) * 256 + lane * 4))
                                  : (u32x4){0u, 0u, 0u, 0u};
      const uint32_t *tail = base + (size_t)nb[k] * 512;
      if (tw[k] == 4)
        tl[k] = __builtin_nontemporal_load((const u32x4 *)(tail + lane * 4));
      else if (tw[k] == 2) {
        const u32x2 v = __builtin_nontemporal_load((const u32x2 *)(tail + lane * 2));
        tl[k] = (u32x4){v.x, v.y, 0u, 0u};
      } else {
        tl[k] = (u32x4){0u, 0u, 0u, 0u};
      }
    }
#pragma unroll
    for (int k = 0; k < R; k++) {
      if (rows[k] >= t.row1) continue;
      const int li = rows[k] - t.row0;
      const T qi = ql[li];
      // the slice's class bounds: every active lane holds the same value
      const int c = __builtin_amdgcn_readfirstlane(cc[k]);
      const int n4 = c & 0xff, n42 = n4 + ((c >> 8) & 0xff);  // at most 42 each
      const uint64_t m4 = (1ull << n4) - 1u, m42 = (1ull << n42) - 1u;
      T sum = (T)0;
#pragma unroll
      for (int b = 0; b < 2; b++)
        if (b < nb[k]) {
          const unsigned wd[8] = {bw[k][b][0].x, bw[k][b][0].y, bw[k][b][0].z, bw[k][b][0].w,
                                  bw[k][b][1].x, bw[k][b][1].y, bw[k][b][1].z, bw[k][b][1].w};
          acc12_words<T, 0, 21>(wd, 21 * b, m4, m42, qi, ql, sum);
        }
      if (tw[k]) {
        const unsigned wd[8] = {tl[k].x, tl[k].y, tl[k].z, tl[k].w, 0u, 0u, 0u, 0u};
        if (tw[k] == 4) acc12_words<T, 0, 10>(wd, 21 * nb[k], m4, m42, qi, ql, sum);
        else acc12_words<T, 0, 5>(wd, 21 * nb[k], m4, m42, qi, ql, sum);
      }
      pnew[rows[k]] = qi;
      w[rows[k]] = sum;
      const T ri = FOLD ? rl[li] : (T)0;
      if (li < nreal) {
        sq.add(qi);
        swq.dot(sum, qi);
        sw.add(sum);
        if (FOLD) fd.rr.dot(ri, ri), fd.rw.dot(ri, sum), fd.ww.dot(sum, sum);
      }
    }
  }
}

// Stages q = beta (p_old - m) + r (q = r on the first iteration of a pass)
// for the tile's rows and its nh halo rows into LDS (tile rows first), and r
// of the tile's rows; rows past the segment's end get q = 0.  FP32 without
// the folded update: four consecutive tile rows per thread in 16-byte
// accesses (tiles are whole 64-row slices), then the halo rows.  SU indices
// per thread and step, all their loads issued before any value is used (the
// halo rows are gathers).  Ends with a barrier.
template <typename T, bool FIRST, bool KEEP_R = true, bool FOLD = false>
__device__ inline void stage_window(const tile_t &t, const int *__restrict__ halo, int nh, T *ql,
                                    T *rl, const T *__restrict__ r, const T *__restrict__ pold,
                                    T beta, T m, const T *__restrict__ wp = nullptr,
                                    T alpha = (T)0, T *__restrict__ rn = nullptr) {
  constexpr bool UPD = FOLD && !FIRST;
  const int nrows = t.row1 - t.row0;
  const int nreal = min(nrows, t.pstart + t.n - t.row0);
  const int tot = nrows + nh;
  constexpr int SU = 4;
  int ibeg = threadIdx.x;
  if constexpr (sizeof(T) == 4) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    for (int i = 4 * (int)threadIdx.x; i < nrows; i += 4 * RSB_BLOCK) {
      f32x4 rv = *(const f32x4 *)(r + t.row0 + i);
      if (UPD) {
        const f32x4 wv = *(const f32x4 *)(wp + t.row0 + i);
        rv.x = rsub(rv.x, alpha, wv.x), rv.y = rsub(rv.y, alpha, wv.y);
        rv.z = rsub(rv.z, alpha, wv.z), rv.w = rsub(rv.w, alpha, wv.w);
        if (rn) *(f32x4 *)(rn + t.row0 + i) = rv;  // r_it to its basis slot
      }
      f32x4 q = rv;
      if (!FIRST) {
        const f32x4 pv = *(const f32x4 *)(pold + t.row0 + i);
        q.x = fmat(beta, pv.x - m, rv.x), q.y = fmat(beta, pv.y - m, rv.y);
        q.z = fmat(beta, pv.z - m, rv.z), q.w = fmat(beta, pv.w - m, rv.w);
      }
      if (i + 0 >= nreal) q.x = 0.f;
      if (i + 1 >= nreal) q.y = 0.f;
      if (i + 2 >= nreal) q.z = 0.f;
      if (i + 3 >= nreal) q.w = 0.f;
      *(f32x4 *)(ql + i) = q;
      if (KEEP_R) *(f32x4 *)(rl + i) = rv;
    }
    ibeg = nrows + threadIdx.x;
  }
  for (int i0 = ibeg; i0 < tot; i0 += SU * RSB_BLOCK) {
    int gr[SU];
    T rg[SU], po[SU], wg[SU];
#pragma unroll
    for (int k = 0; k < SU; k++) {
      const int idx = i0 + k * RSB_BLOCK;
      gr[k] = idx < nrows ? t.row0 + idx : (idx < tot ? halo[idx - nrows] : t.row0);
    }
#pragma unroll
    for (int k = 0; k < SU; k++) {
      rg[k] = r[gr[k]];
      po[k] = FIRST ? (T)0 : pold[gr[k]];
      wg[k] = UPD ? wp[gr[k]] : (T)0;
    }
    if (UPD)
#pragma unroll
      for (int k = 0; k < SU; k++) rg[k] = rsub(rg[k], alpha, wg[k]);
#pragma unroll
    for (int k = 0; k < SU; k++) {
      const int idx = i0 + k * RSB_BLOCK;
      if (idx >= tot) break;
      T q = FIRST ? rg[k] : fmat(beta, po[k] - m, rg[k]);
      if (idx < nrows) {
        if (KEEP_R) rl[idx] = rg[k];
        if (UPD && rn) rn[gr[k]] = rg[k];  // r_it to its basis slot
        if (idx >= nreal) q = (T)0;
      }
      ql[idx] = q;
    }
  }
  __syncthreads();
}

template <typename T, bool FIRST, bool FOLD = false>
__device__ inline void lz_apply_tiled(const lz_args &a, const tile_t &t, const tiled_args &ta,
                                      int nh, T *ql, T *rl, const T *__restrict__ r,
                                      const T *__restrict__ pold, T *__restrict__ pnew,
                                      T *__restrict__ w, T beta, T m, acc_t<T> &sq,
                                      acc_t<T> &swq, acc_t<T> &sw, fold_t<T> &fd) {
  const int nrows = t.row1 - t.row0;
  const int nreal = min(nrows, t.pstart + t.n - t.row0);
  // the tile's r in LDS: the folded update's row phase reads it; the FP32
  // kernel writes it anyway, its 4 KB holding the kernel at seven
  // workgroups per CU (at eight, with rl dropped, the level-0 apply of the
  // 256^3 box took 279 us against 269); the FP64 kernel drops it and runs
  // four workgroups per CU instead of three (0.217 -> 0.209 ms per launch)
  constexpr bool KEEP_R = FOLD || sizeof(T) == 4;
  const slice_meta sm = load_meta(t, ta);
  stage_window<T, FIRST, KEEP_R, FOLD>(t, ta.halo + ta.halo_off[t.ti], nh, ql, rl, r, pold, beta,
                                       m, fd.wp, fd.alpha, fd.rn);
  // two rows per thread and step (measured 15% faster than one at a time
  // on the 256^3 workload: more loads in flight per lane)
  if (ta.e12)
    apply_rows_e12<T, 2, FOLD>(t, ta, sm, ql, rl, pnew, w, nreal, sq, swq, sw, fd);
  else
    apply_rows_batched<T, 2, FOLD>(t, ta, sm, ql, rl, pnew, w, nreal, sq, swq, sw, fd);
}

// The residuals of a pass live in the basis, unscaled: r_it in slot it
// (the Ritz step scales slot j by 1 / |r_j|), so the apply reads its r
// there and writes no basis vector.
// FOLD (FP32): the residual update of the previous iteration is formed in
// the staging, r_it = r_{it-1} - alpha w_{it-1} (w_prev: the w buffer of
// the other parity), written to slot it, and the launch adds the sums r.r,
// r.w, w.w (partial slots 3..5) for FIN_APPLYR.  No separate r-update pass
// and one finishing step per iteration.
template <typename T, bool FOLD>
__global__ void __launch_bounds__(RSB_BLOCK) k_lz_apply(lz_args a, const T *__restrict__ pold,
                                                        T *__restrict__ pnew, T *__restrict__ w,
                                                        T *__restrict__ basis, int64_t mpad,
                                                        tiled_args ta, int nlist,
                                                        const T *__restrict__ wprev) {
  __shared__ __attribute__((aligned(16))) T ql[TB_LOCAL];
  // the tile's r (read only to fold the update; see lz_apply_tiled)
  __shared__ __attribute__((aligned(16))) T rl[RSB_TILE];
  tile_t t;
  if (!tile_of(a, LZ_RUNNING, t, nlist)) return;
  const int s = t.s, it = a.iter[s];
  T *cur = basis + (size_t)it * mpad;
  // what the staging reads: r_it, or r_{it-1} to update (FOLD)
  const T *__restrict__ r = (FOLD && it > 0) ? cur - mpad : cur;
  const T beta = (T)SC(s, SC_BETA), m = (T)SC(s, SC_MEANP);
  acc_t<T> sq, swq, sw;
  fold_t<T> fd;
  fd.wp = wprev, fd.rn = it == 0 ? nullptr : cur, fd.alpha = (T)SC(s, SC_ALPHA);
  const int nh = ta.nhalo[t.ti];
  if (nh >= 0) {
    if (it == 0)
      lz_apply_tiled<T, true, FOLD>(a, t, ta, nh, ql, rl, r, pold, pnew, w, beta, m, sq, swq, sw,
                                    fd);
    else
      lz_apply_tiled<T, false, FOLD>(a, t, ta, nh, ql, rl, r, pold, pnew, w, beta, m, sq, swq,
                                     sw, fd);
  } else if (it == 0) {
    lz_apply_rows<T, true, FOLD>(a, t, r, pold, pnew, w, beta, m, ta.slice_off, ta.slice_w,
                                 ta.ell, sq, swq, sw, fd);
  } else {
    lz_apply_rows<T, false, FOLD>(a, t, r, pold, pnew, w, beta, m, ta.slice_off, ta.slice_w,
                                  ta.ell, sq, swq, sw, fd);
  }
  if (FOLD) {
    double v[6] = {sq.value(), swq.value(), sw.value(),
                   fd.rr.value(), fd.rw.value(), fd.ww.value()};
    publish<6>(a, t, v);
  } else {
    double v[3] = {sq.value(), swq.value(), sw.value()};
    publish<3>(a, t, v);
  }
}

// Vertex form of the tiles (tiles.hip, rsb_build_vtiles): the reference's
// gather-scatter form (laplacian.c:159-205), (L q)_e = sum over the slots of
// e of sum over the slots at their vertex v of (q_e - q_e'), evaluated as
// mult(v) (q_e - q_f(v)) - S(v), f(v) the first slot at v and
// S(v) = sum over the slots at v of (q_e' - q_f(v)): every term a difference
// of neighbouring values, as in the neighbour-entry form (summing q itself
// loses the low-frequency part of L q in FP32).  One aligned load per vertex
// fetches its nv window indices (ascending, padded with VT_MAXW); LDS keeps
// S(v) and one 16-bit word f(v) | mult(v) << 12 per vertex; fixed order of
// summation.
struct vtile_args {
  const int *vt_n;
  const int64_t *vt_loff;
  const uint16_t *list, *rowv;
  const int *nhalo;
  const int64_t *halo_off;
  const int *halo;
  int nv;
};

template <typename T, int W>
__device__ inline void vt_sums(const uint16_t *__restrict__ Ls, int nvert, const T *ql, T *S,
                               uint16_t *F) {
  // two vertices per thread and step, both loads issued first
  for (int v0 = threadIdx.x; v0 < nvert; v0 += 2 * blockDim.x) {
    const int v1 = v0 + blockDim.x;
    uint16_t e[2][W];
    if (W == 8) {
      const u32x4 a = __builtin_nontemporal_load((const u32x4 *)(Ls + (int64_t)v0 * 8));
      const u32x4 b = v1 < nvert ? __builtin_nontemporal_load((const u32x4 *)(Ls + (int64_t)v1 * 8))
                                 : (u32x4){0u, 0u, 0u, 0u};
      const unsigned wa[4] = {a.x, a.y, a.z, a.w}, wb[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
      for (int k = 0; k < 4; k++) {
        e[0][2 * k] = (uint16_t)(wa[k] & 0xffffu), e[0][2 * k + 1] = (uint16_t)(wa[k] >> 16);
        e[1][2 * k] = (uint16_t)(wb[k] & 0xffffu), e[1][2 * k + 1] = (uint16_t)(wb[k] >> 16);
      }
    } else {
      const u32x2 a = __builtin_nontemporal_load((const u32x2 *)(Ls + (int64_t)v0 * 4));
      const u32x2 b = v1 < nvert ? __builtin_nontemporal_load((const u32x2 *)(Ls + (int64_t)v1 * 4))
                                 : (u32x2){0u, 0u};
      const unsigned wa[2] = {a.x, a.y}, wb[2] = {b.x, b.y};
#pragma unroll
      for (int k = 0; k < 2; k++) {
        e[0][2 * k] = (uint16_t)(wa[k] & 0xffffu), e[0][2 * k + 1] = (uint16_t)(wa[k] >> 16);
        e[1][2 * k] = (uint16_t)(wb[k] & 0xffffu), e[1][2 * k + 1] = (uint16_t)(wb[k] >> 16);
      }
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int v = u ? v1 : v0;
      if (v >= nvert) break;
      const T ref = ql[e[u][0]];  // every list has at least one slot
      T sum = (T)0;
      int cnt = 0;
#pragma unroll
      for (int k = 0; k < W; k++) {
        const bool real = e[u][k] != VT_MAXW;
        sum += real ? ql[e[u][k]] - ref : (T)0;
        cnt += real;
      }
      S[v] = sum;
      F[v] = (uint16_t)(e[u][0] | (cnt << 12));
    }
  }
}

template <typename T, bool FIRST>
__device__ inline void lz_apply_vertex(const lz_args &a, const tile_t &t, const vtile_args &va,
                                       T *ql, T *S, uint16_t *F, const T *__restrict__ r,
                                       const T *__restrict__ pold, T *__restrict__ pnew,
                                       T *__restrict__ w, T beta, T m, acc_t<T> &sq,
                                       acc_t<T> &swq, acc_t<T> &sw) {
  const int nrows = t.row1 - t.row0;
  const int nreal = min(nrows, t.pstart + t.n - t.row0);
  if (threadIdx.x == 0) ql[VT_MAXW] = (T)0;  // what the lists' padding reads
  stage_window<T, FIRST, false>(t, va.halo + va.halo_off[t.ti], va.nhalo[t.ti], ql, nullptr, r,
                                pold, beta, m);
  const int nvert = va.vt_n[t.ti];
  const uint16_t *Ls = va.list + va.vt_loff[t.ti];
  if (va.nv == 8) vt_sums<T, 8>(Ls, nvert, ql, S, F);
  else vt_sums<T, 4>(Ls, nvert, ql, S, F);
  __syncthreads();
  // the (up to) four rows of a thread: their index words loaded first
  constexpr int R = RSB_TILE / RSB_BLOCK;
  u32x4 pks[R];
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int row = t.row0 + threadIdx.x + k * blockDim.x;
    pks[k] = row < t.row1 ? __builtin_nontemporal_load((const u32x4 *)(va.rowv + (int64_t)row * 8))
                          : (u32x4){0xffffffffu, 0xffffffffu, 0xffffffffu, 0xffffffffu};
  }
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int row = t.row0 + threadIdx.x + k * blockDim.x;
    if (row >= t.row1) continue;
    const int li = row - t.row0;
    const u32x4 pk = pks[k];
    const unsigned id[8] = {pk.x & 0xffffu, pk.x >> 16, pk.y & 0xffffu, pk.y >> 16,
                            pk.z & 0xffffu, pk.z >> 16, pk.w & 0xffffu, pk.w >> 16};
    const T qi = ql[li];
    T sum = (T)0;
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (id[j] != 0xffffu) {
        const unsigned f = F[id[j]];
        sum += (T)(f >> 12) * (qi - ql[f & 0xfffu]) - S[id[j]];
      }
    pnew[row] = qi;
    w[row] = sum;
    if (li < nreal) {
      sq.add(qi);
      swq.dot(sum, qi);
      sw.add(sum);
    }
  }
}

// FP32 only (its LDS: window + per-vertex sums and first-slot / count words
// = 28 KB, five workgroups per CU); a tile without the vertex form (vt_n < 0) takes the
// neighbour entries of the same window.  The level has no wide tiles.
template <typename T>
__global__ void __launch_bounds__(RSB_BLOCK) k_lz_apply_v(lz_args a, const T *__restrict__ pold,
                                                          T *__restrict__ pnew, T *__restrict__ w,
                                                          const T *__restrict__ basis,
                                                          int64_t mpad, vtile_args va,
                                                          tiled_args ta, int nlist) {
  __shared__ __attribute__((aligned(16))) T ql[VT_MAXW + 1];
  __shared__ T S[VT_MAXV];  // the neighbour-entry fallback keeps r of the tile rows here
  __shared__ uint16_t F[VT_MAXV];
  static_assert(VT_MAXV >= RSB_TILE, "the fallback's r of the tile rows lives in S");
  tile_t t;
  if (!tile_of(a, LZ_RUNNING, t, nlist)) return;
  const int s = t.s, it = a.iter[s];
  const T *__restrict__ r = basis + (size_t)it * mpad;  // r_it (its basis slot)
  const T beta = (T)SC(s, SC_BETA), m = (T)SC(s, SC_MEANP);
  acc_t<T> sq, swq, sw;
  if (va.vt_n[t.ti] >= 0) {
    if (it == 0)
      lz_apply_vertex<T, true>(a, t, va, ql, S, F, r, pold, pnew, w, beta, m, sq, swq, sw);
    else
      lz_apply_vertex<T, false>(a, t, va, ql, S, F, r, pold, pnew, w, beta, m, sq, swq, sw);
  } else {
    const int nh = ta.nhalo[t.ti];
    fold_t<T> fd;
    fd.wp = nullptr, fd.rn = nullptr, fd.alpha = (T)0;
    if (it == 0)
      lz_apply_tiled<T, true>(a, t, ta, nh, ql, S, r, pold, pnew, w, beta, m, sq, swq, sw, fd);
    else
      lz_apply_tiled<T, false>(a, t, ta, nh, ql, S, r, pold, pnew, w, beta, m, sq, swq, sw, fd);
  }
  double v[3] = {sq.value(), swq.value(), sw.value()};
  publish<3>(a, t, v);
}

template <typename T>
// r_{it+1} = r_it - alpha w into basis slot it + 1; partial r.r
__global__ void __launch_bounds__(RSB_BLOCK) k_lz_rupdate(lz_args a, T *__restrict__ basis,
                                                          int64_t mpad, const T *__restrict__ w) {
  tile_t t;
  if (!tile_of(a, LZ_RUNNING, t)) return;
  const int s = t.s;
  const T *__restrict__ r = basis + (size_t)a.iter[s] * mpad;
  T *__restrict__ rn = basis + (size_t)(a.iter[s] + 1) * mpad;
  const T alpha = (T)SC(s, SC_ALPHA);
  acc_t<T> acc;
  if constexpr (sizeof(T) == 4) {
    // FP32: four consecutive rows per thread in one 16-byte access each
    // (tile bounds and vector bases are multiples of 64 rows, so a group
    // lies wholly inside or outside the tile)
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    for (int row = t.row0 + 4 * (int)threadIdx.x; row < t.row1; row += 4 * (int)blockDim.x) {
      const f32x4 rv = *(const f32x4 *)(r + row), wv = *(const f32x4 *)(w + row);
      f32x4 x;
      x.x = rsub(rv.x, alpha, wv.x), x.y = rsub(rv.y, alpha, wv.y);
      x.z = rsub(rv.z, alpha, wv.z), x.w = rsub(rv.w, alpha, wv.w);
      *(f32x4 *)(rn + row) = x;
      acc.dot(x.x, x.x), acc.dot(x.y, x.y), acc.dot(x.z, x.z), acc.dot(x.w, x.w);
    }
    double v[1] = {acc.value()};
    publish<1>(a, t, v);
    return;
  }
  // the (up to) four rows of a thread: all loads first
  constexpr int R = RSB_TILE / RSB_BLOCK;
  T rv[R], wv[R];
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int row = t.row0 + threadIdx.x + k * blockDim.x;
    rv[k] = row < t.row1 ? r[row] : (T)0;
    wv[k] = row < t.row1 ? w[row] : (T)0;
  }
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int row = t.row0 + threadIdx.x + k * blockDim.x;
    if (row >= t.row1) continue;
    const T x = rsub(rv[k], alpha, wv[k]);
    rn[row] = x;
    acc.dot(x, x);
  }
  double v[1] = {acc.value()};
  publish<1>(a, t, v);
}

// ---------------------------------------------------------------------------
// Tridiagonal eigen-solve of each finished pass: implicit QL with shifts, the
// steps of fiedler.c:328-432 (FP64, contraction off so every operation rounds
// as written).  One wavefront per segment: every lane runs the same scalar
// recurrence; the diagonal and off-diagonal are held in registers (below) so
// the serial chain never waits on LDS; the plane rotations of the
// eigenvector matrix (in LDS) are spread over the lanes (lane = matrix row,
// each lane touches only its own rows).  The coefficients y of the
// eigenvector with the smallest |eigenvalue| are kept.
#pragma clang fp contract(off)
__device__ inline double sgn_abs(double a, double b) { return b >= 0.0 ? fabs(a) : -fabs(a); }

// d and e live in registers: lane k holds entries k and k + 64 (n <= 128).
// The serial QL chain reads them with readlane (a uniform index), the owning
// lane updates them, and the deflation scan (first m >= l with
// |e_m| / (|d_m| + |d_m+1|) < 1e-12) tests every m at once and takes the
// first hit from a ballot: the same tests, in parallel, give the same m.
__device__ inline double lane_get(double v, int i) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), i);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), i);
  return __longlong_as_double(
      (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned long long)(unsigned)lo));
}
// W words per lane: entries lane (and lane + 64 if W == 2).  Vectors of at
// most 64 entries take W == 1, which leaves no branch in a read or a write.
template <int W>
struct lanes_t {
  double a, b;
  __device__ inline double get(int i) const {
    if (W == 1) return lane_get(a, i);
    return i < RSB_WAVE ? lane_get(a, i) : lane_get(b, i - RSB_WAVE);
  }
  __device__ inline void set(int i, double x, int lane) {
    if (W == 1 || i < RSB_WAVE) a = lane == i ? x : a;
    else b = lane == i - RSB_WAVE ? x : b;
  }
  __device__ inline void load(const double *v, int n, int lane) {
    a = lane < n ? v[lane] : 0.0;
    b = W == 2 && lane + RSB_WAVE < n ? v[lane + RSB_WAVE] : 0.0;
  }
  __device__ inline void store(double *v, int n, int lane) const {
    if (lane < n) v[lane] = a;
    if (W == 2 && lane + RSB_WAVE < n) v[lane + RSB_WAVE] = b;
  }
};

// a / b for |a|, |b| in [2^-400, 2^400]: the operations of the compiler's own
// divide (a reciprocal estimate, two Newton steps, the quotient corrected by
// its exact remainder) without the scaling and special cases it wraps around
// them, so the result is the same correctly rounded quotient.
__device__ inline double div_plain(double a, double b) {
  double y = __builtin_amdgcn_rcp(b);
  y = fmat(y, fmat(-b, y, 1.0), y);
  y = fmat(y, fmat(-b, y, 1.0), y);
  const double q = a * y;
  return fmat(fmat(-b, q, a), y, q);
}
__device__ inline bool in_plain_range(double a) {
  const int ex = (__double2hiint(a) >> 20) & 0x7ff;
  return ex > 1023 - 400 && ex < 1023 + 400;
}
// r = sqrt(x) and 1 / r, both correctly rounded, for x in [1, 2]: Goldschmidt
// steps from the reciprocal square root estimate (the compiler's, without its
// scaling), then the refined estimate of 1 / sqrt(x) corrected twice against
// r: after the first correction it is within an ulp of 1 / r, and a second
// one is then correctly rounded unless r's significand is all ones
// (Markstein, IBM J. Res. Dev. 34, 1990), which r <= sqrt(2) rules out.
__device__ inline void sqrt_rcp_plain(double x, double &r, double &ri) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double e = fmat(-h, g, 0.5);
  g = fmat(g, e, g);
  h = fmat(h, e, h);
  g = fmat(fmat(-g, g, x), h, g);
  g = fmat(fmat(-g, g, x), h, g);
  double z = 2.0 * h;
  z = fmat(z, fmat(-g, z, 1.0), z);
  r = g;
  ri = fmat(z, fmat(-g, z, 1.0), z);
}

// Two wavefronts: the first runs the serial recurrence, whose every step is a
// divide, a square root and a reciprocal one after another, and leaves each
// sweep's rotations in LDS; the second applies them to the eigenvector
// matrix while the first is in its next sweep (one barrier a sweep).  With
// the rotations in the recurrence's own instruction stream, their LDS round
// trips lengthened every step, and branches cost as much again: 1.00 ms per call
// for a pass of 50, now 0.49 (what is left is the latency of ~31 dependent FP64
// operations a step; unrolling it changed nothing).
// z: column i of the matrix at z + i * zp, zp = n rounded up to 64.
struct tqli_shared {
  double cs[2][2][128];  // c and s of a sweep's steps, by buffer
  int l[2], m[2];        // its range; m < 0: no more sweeps
  int failed;
};
__device__ inline int tqli_pitch(int n) { return (n + RSB_WAVE - 1) / RSB_WAVE * RSB_WAVE; }

template <int W>
__device__ void tqli_wave(int n, double *d, double *e, double *z, double *y, double *lam_out,
                          tqli_shared *sh) {
  const int lane = threadIdx.x % RSB_WAVE;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / RSB_WAVE);
  const int zp = tqli_pitch(n);
  for (int i = threadIdx.x; i < n * zp; i += 2 * RSB_WAVE) z[i] = i / zp == i % zp ? 1.0 : 0.0;
  __syncthreads();
  lanes_t<W> D, E;
  if (wave == 1) {
    for (int buf = 0;; buf ^= 1) {
      __syncthreads();
      const int l = sh->l[buf], m = sh->m[buf];
      if (m < 0) break;
      const double *C = sh->cs[buf][0], *S = sh->cs[buf][1];
      for (int k = lane; k < n; k += RSB_WAVE) {
        // z[k][i + 1] carried from step to step, z[k][i] read one step ahead
        double zk1 = z[m * zp + k], zk = z[(m - 1) * zp + k];
        for (int i = m - 1; i >= l; i--) {
          const double next = i > l ? z[(i - 1) * zp + k] : 0.0;
          const double c = C[i + 1], s = S[i + 1];
          z[(i + 1) * zp + k] = s * zk + c * zk1;
          zk1 = c * zk - s * zk1;
          zk = next;
        }
        z[l * zp + k] = zk1;
      }
    }
  } else {
    D.load(d, n, lane);
    E.load(e, n, lane);
    int failed = 0, buf = 0;
    for (int l = 0; l < n && !failed; l++) {
      int sweeps = 0, m;
      while (true) {
        // d[m + 1] next to d[m]: lane 63's neighbour is entry 64
        double dn_a = __shfl_down(D.a, 1, RSB_WAVE);
        double dn_b = 0.0;
        if (W == 2) {
          const double d64 = lane_get(D.b, 0);
          if (lane == RSB_WAVE - 1) dn_a = d64;
          dn_b = __shfl_down(D.b, 1, RSB_WAVE);
        }
        const int ma = lane, mb = lane + RSB_WAVE;
        const bool ta = ma >= l && ma < n - 1 && fabs(E.a) / (fabs(D.a) + fabs(dn_a)) < 1e-12;
        const bool tb = W == 2 && mb >= l && mb < n - 1 && fabs(E.b) / (fabs(D.b) + fabs(dn_b)) < 1e-12;
        const unsigned long long ba = __ballot(ta), bb = __ballot(tb);
        m = ba ? __ffsll((long long)ba) - 1 : bb ? RSB_WAVE + __ffsll((long long)bb) - 1 : n - 1;
        if (m == l) break;
        if (sweeps++ == 30) {
          failed = 1;
          break;
        }
        lanes_t<W> C, S;  // the step's rotation, in the lane of its e[i + 1]
        C.a = C.b = S.a = S.b = 0.0;
        const double dl = D.get(l), el = E.get(l);
        double g = (D.get(l + 1) - dl) / (2.0 * el);
        double r = sqrt(g * g + 1.0);
        double dm = D.get(m);  // d[i + 1] of the step
        g = dm - dl + el / (g + sgn_abs(r, g));
        double s = 1.0, c = 1.0, p = 0.0;
        for (int i = m - 1; i >= l; i--) {
          const double ei = E.get(i), di = D.get(i);
          const double f = s * ei, b = c * ei;
          // the larger of |f|, |g| divides: t = small / large,
          // r = sqrt(t^2 + 1), 1 / r and t / r are the rotation
          const bool fg = fabs(f) >= fabs(g);
          const double big = fg ? f : g, sml = fg ? g : f;
          double t = div_plain(sml, big), ri;
          sqrt_rcp_plain(t * t + 1.0, r, ri);
          if (!(in_plain_range(big) && in_plain_range(sml))) {
            t = sml / big;
            r = sqrt(t * t + 1.0);
            ri = 1.0 / r;
          }
          const double ei1 = big * r, tr = t * ri;
          s = fg ? ri : tr;
          c = fg ? tr : ri;
          g = dm - p;
          dm = di;
          r = (di - g) * s + 2.0 * c * b;
          p = s * r;
          const double di1 = g + p;
          g = c * r - b;
          E.set(i + 1, ei1, lane);
          D.set(i + 1, di1, lane);
          C.set(i + 1, c, lane);
          S.set(i + 1, s, lane);
        }
        C.store(sh->cs[buf][0], n, lane);
        S.store(sh->cs[buf][1], n, lane);
        D.set(l, D.get(l) - p, lane);
        E.set(l, g, lane);
        E.set(m, 0.0, lane);
        if (lane == 0) sh->l[buf] = l, sh->m[buf] = m;
        __syncthreads();
        buf ^= 1;
      }
    }
    if (lane == 0) sh->m[buf] = -1, sh->failed = failed;
    __syncthreads();
  }
  // (the last barrier follows the last sweep's rotations)
  if (wave == 0) {
    const int failed = sh->failed;
    // eigenvalue of smallest magnitude (first on ties, fiedler.c:538-545)
    int imin = 0;
    double emin = fabs(D.get(0));
    for (int i = 1; i < n; i++) {
      const double v = fabs(D.get(i));
      if (v < emin) emin = v, imin = i;
    }
    if (failed) {
      // the reference leaves the rotations untransposed and unnormalised
      for (int j = lane; j < n; j += RSB_WAVE) y[j] = z[j * zp + imin];
    } else {
      // eigenvector imin = column imin of z, normalised (sum in row order)
      lanes_t<W> v, q;
      v.load(z + imin * zp, n, lane);
      q.a = v.a * v.a, q.b = v.b * v.b;
      double nrm = 0.0;
      for (int i = 0; i < n; i++) nrm += q.get(i);
      if (nrm > 0.0) nrm = sqrt(fabs(nrm));
      const double scale = 1.0 / nrm;
      v.a *= scale, v.b *= scale;
      v.store(y, n, lane);
    }
    const double lam = D.get(imin);
    if (lane == 0) *lam_out = lam;
  }
  __syncthreads();
}
// The same QL steps for passes longer than 128 iterations: d and e in LDS
// (every lane computes each update and writes the same value), the
// eigenvector matrix z (n x n, row-major) in global memory, each lane
// rotating its own rows.  Operations and their order are those above, so
// results are bit-identical to it (and to the oracle).
__device__ void tqli_wave_mem(int n, double *d, double *e, double *z, double *y,
                              double *lam_out) {
  const int lane = threadIdx.x;
  for (int64_t i = lane; i < (int64_t)n * n; i += RSB_WAVE) z[i] = 0.0;
  __syncthreads();
  for (int i = lane; i < n; i += RSB_WAVE) z[(int64_t)i * n + i] = 1.0;
  __syncthreads();
  int failed = 0;
  for (int l = 0; l < n && !failed; l++) {
    int sweeps = 0, m;
    while (true) {
      for (m = l; m < n - 1; m++)
        if (fabs(e[m]) / (fabs(d[m]) + fabs(d[m + 1])) < 1e-12) break;
      if (m == l) break;
      if (sweeps++ == 30) {
        failed = 1;
        break;
      }
      const double dl = d[l], el = e[l];
      double g = (d[l + 1] - dl) / (2.0 * el);
      double r = sqrt(g * g + 1.0);
      g = d[m] - dl + el / (g + sgn_abs(r, g));
      double s = 1.0, c = 1.0, p = 0.0;
      for (int i = m - 1; i >= l; i--) {
        const double ei = e[i];
        double f = s * ei, b = c * ei;
        double ei1;
        if (fabs(f) >= fabs(g)) {
          c = g / f;
          r = sqrt(c * c + 1.0);
          ei1 = f * r;
          s = 1.0 / r;
          c = c * s;
        } else {
          s = f / g;
          r = sqrt(s * s + 1.0);
          ei1 = g * r;
          c = 1.0 / r;
          s = s * c;
        }
        g = d[i + 1] - p;
        r = (d[i] - g) * s + 2.0 * c * b;
        p = s * r;
        const double di1 = g + p;
        g = c * r - b;
        e[i + 1] = ei1;
        d[i + 1] = di1;
        for (int k = lane; k < n; k += RSB_WAVE) {
          double *zk = z + (int64_t)k * n;
          const double zk1 = zk[i + 1], zk0 = zk[i];
          zk[i + 1] = s * zk0 + c * zk1;
          zk[i] = c * zk0 - s * zk1;
        }
      }
      d[l] = d[l] - p;
      e[l] = g;
      e[m] = 0.0;
    }
  }
  __syncthreads();  // rows of z written by other lanes are read below
  int imin = 0;
  double emin = fabs(d[0]);
  for (int i = 1; i < n; i++) {
    const double v = fabs(d[i]);
    if (v < emin) emin = v, imin = i;
  }
  if (failed) {
    for (int j = lane; j < n; j += RSB_WAVE) y[j] = z[(int64_t)imin * n + j];
  } else {
    __shared__ double scale;
    if (lane == 0) {
      double nrm = 0.0;
      for (int i = 0; i < n; i++) nrm += z[(int64_t)i * n + imin] * z[(int64_t)i * n + imin];
      if (nrm > 0.0) nrm = sqrt(fabs(nrm));
      scale = 1.0 / nrm;
    }
    __syncthreads();
    for (int j = lane; j < n; j += RSB_WAVE) y[j] = z[(int64_t)j * n + imin] * scale;
  }
  if (lane == 0) *lam_out = d[imin];
  __syncthreads();
}

#pragma clang fp contract(fast)

// Fast variant for the FP32 path: the eigenpair of smallest |eigenvalue| of
// the tridiagonal T directly, instead of all of them.  Eigenvalue by
// multisection on Sturm counts (each of the 64 lanes counts the eigenvalues
// below its own shift; 65 sub-intervals per step), eigenvector by inverse
// iteration with the LDL^T factorisation of T - a I, a the lower end of the
// final interval (Parlett, The Symmetric Eigenvalue Problem, 3.3 and 4.3;
// the count recurrence with the pivot guard of LAPACK dstebz).  Sign: the
// component along the first Lanczos vector (the pass's start) is made
// non-negative.  It agrees with the QL solve to rounding, not bit for bit.
// plain: every squared off-diagonal is in div_plain's range and the pivot
// guard below it.  The count then runs on plain divides without a test in
// its chain, and again in full if some pivot left the range.
template <int W>
__device__ inline int sturm_count(int n, const lanes_t<W> &D, const lanes_t<W> &E2, double x,
                                  double pivmin, bool plain) {
  if (plain) {
    double q = D.get(0) - x;
    bool ok = in_plain_range(q);
    int c = q < 0.0;
    for (int i = 1; i < n; i++) {
      q = (D.get(i) - x) - div_plain(E2.get(i - 1), q);
      ok &= in_plain_range(q);
      c += q < 0.0;
    }
    if (__all(ok)) return c;
  }
  int c = 0;
  double q = D.get(0) - x;
  if (fabs(q) < pivmin) q = -pivmin;
  c += q < 0.0;
  for (int i = 1; i < n; i++) {
    q = (D.get(i) - x) - E2.get(i - 1) / q;
    if (fabs(q) < pivmin) q = -pivmin;
    c += q < 0.0;
  }
  return c;
}

// eigenvalue number j (ascending) in [lo, hi]; returns the final interval
template <int W>
__device__ inline void multisect(int n, const lanes_t<W> &D, const lanes_t<W> &E2, double pivmin,
                                 bool plain, int j, double &lo, double &hi) {
  const int lane = threadIdx.x;
  for (int step = 0; step < 16; step++) {
    const double w = hi - lo;
    if (!(w > 2.0 * DBL_EPSILON * fmax(fabs(lo), fabs(hi)) + pivmin)) break;
    const double x = lo + w * (double)(lane + 1) / (double)(RSB_WAVE + 1);
    const int c = sturm_count<W>(n, D, E2, x, pivmin, plain);
    // lanes whose shift is at or below eigenvalue j: count <= j
    const unsigned long long below = __ballot(c <= j);
    // shifts increase with the lane: the highest such lane is the new lower
    // end, the next lane the new upper end
    const int k = below ? 63 - __clzll((long long)below) : -1;
    const double xk = k >= 0 ? __shfl(x, k, RSB_WAVE) : lo;
    const double xk1 = k + 1 < RSB_WAVE ? __shfl(x, k + 1, RSB_WAVE) : hi;
    lo = xk, hi = xk1;
  }
}

template <int W>
__device__ void eig_min_wave(int n, const double *d, const double *e, double *y,
                             double *lam_out) {
  const int lane = threadIdx.x;
  lanes_t<W> D, E, E2;
  D.load(d, n, lane);
  E.load(e, n - 1, lane);
  E2.a = E.a * E.a, E2.b = E.b * E.b;
  // Gershgorin bounds and the pivot guard
  double glo = DBL_MAX, ghi = -DBL_MAX, emax = 0.0, tnorm = 0.0;
  for (int i = lane; i < n; i += RSB_WAVE) {
    const double r = (i > 0 ? fabs(e[i - 1]) : 0.0) + (i < n - 1 ? fabs(e[i]) : 0.0);
    glo = fmin(glo, d[i] - r), ghi = fmax(ghi, d[i] + r);
    tnorm = fmax(tnorm, fabs(d[i]) + r);
    if (i < n - 1) emax = fmax(emax, e[i] * e[i]);
  }
  for (int o = RSB_WAVE / 2; o > 0; o >>= 1) {
    glo = fmin(glo, __shfl_xor(glo, o, RSB_WAVE));
    ghi = fmax(ghi, __shfl_xor(ghi, o, RSB_WAVE));
    emax = fmax(emax, __shfl_xor(emax, o, RSB_WAVE));
    tnorm = fmax(tnorm, __shfl_xor(tnorm, o, RSB_WAVE));
  }
  const double pivmin = DBL_MIN * fmax(1.0, emax);
  const double span = fmax(ghi - glo, DBL_MIN);
  glo -= 2.0 * DBL_EPSILON * span, ghi += 2.0 * DBL_EPSILON * span;
  const bool plain = __all((lane >= n - 1 || in_plain_range(E2.a)) &&
                           (lane + RSB_WAVE >= n - 1 || in_plain_range(E2.b))) &&
                     pivmin < 0x1p-400;
  // smallest eigenvalue; if it is negative, compare the eigenvalues either
  // side of 0 by magnitude
  double lo = glo, hi = ghi;
  multisect<W>(n, D, E2, pivmin, plain, 0, lo, hi);
  double lam = 0.5 * (lo + hi), shift = lo;
  if (lam < 0.0) {
    const int k = sturm_count<W>(n, D, E2, 0.0, pivmin, plain);
    double l1 = glo, h1 = ghi;
    multisect<W>(n, D, E2, pivmin, plain, k - 1, l1, h1);
    lam = 0.5 * (l1 + h1), shift = l1;
    if (k < n) {
      double l2 = glo, h2 = ghi;
      multisect<W>(n, D, E2, pivmin, plain, k, l2, h2);
      const double lam2 = 0.5 * (l2 + h2);
      if (fabs(lam2) < fabs(lam)) lam = lam2, shift = l2;
    }
  }
  // inverse iteration (two solves): (T - shift I) = L D L^T, a pivot below
  // eps * |T|_inf replaced by +-eps * |T|_inf; each solve is rescaled by its
  // largest entry before normalising.  Entry i of every vector is in lane
  // i % 64; only the pivots, the substitutions and the sum of squares are
  // serial, and those chains read their operands by readlane (on one lane,
  // with every divide in the chain and every operand from LDS, they were
  // half of the kernel's 134 us; now 78 us in all).
  const double tau = DBL_EPSILON * fmax(tnorm, DBL_MIN);
  lanes_t<W> piv, l, x;
  piv.a = piv.b = 1.0;
  double q = D.get(0) - shift;
  if (fabs(q) < tau) q = q < 0.0 ? -tau : tau;
  piv.set(0, q, lane);
  for (int i = 1; i < n; i++) {
    const double di = D.get(i), e2 = E2.get(i - 1);
    double t = div_plain(e2, q);
    if (!(plain && in_plain_range(q))) t = e2 / q;
    q = (di - shift) - t;
    if (fabs(q) < tau) q = q < 0.0 ? -tau : tau;
    piv.set(i, q, lane);
  }
  l.a = E.a / piv.a, l.b = E.b / piv.b;  // l_i = e_i / piv_i
  x.a = x.b = 1.0;
  for (int it = 0; it < 2; it++) {
    // L z = x (unit lower), D w = z, L^T v = w
    double c = x.get(0);
    for (int i = 1; i < n; i++) {
      c = fmat(-l.get(i - 1), c, x.get(i));
      x.set(i, c, lane);
    }
    x.a /= piv.a, x.b /= piv.b;
    c = x.get(n - 1);
    for (int i = n - 2; i >= 0; i--) {
      c = fmat(-l.get(i), c, x.get(i));
      x.set(i, c, lane);
    }
    double amax = fmax(lane < n ? fabs(x.a) : 0.0, lane + RSB_WAVE < n ? fabs(x.b) : 0.0);
    for (int o = RSB_WAVE / 2; o > 0; o >>= 1) amax = fmax(amax, __shfl_xor(amax, o, RSB_WAVE));
    if (!(amax > 0.0) || amax > DBL_MAX) {
      x.a = lane == 0 ? 1.0 : 0.0, x.b = 0.0;
      break;
    }
    x.a /= amax, x.b /= amax;
    double nrm = 0.0;
    for (int i = 0; i < n; i++) {
      const double xi = x.get(i);
      nrm = fmat(xi, xi, nrm);
    }
    nrm = sqrt(nrm);
    int f = 0;
    while (f < n - 1 && x.get(f) == 0.0) f++;
    const double sc = (x.get(f) < 0.0 ? -1.0 : 1.0) / nrm;
    x.a *= sc, x.b *= sc;
  }
  if (lane == 0) *lam_out = lam;
  x.store(y, n, lane);
  __syncthreads();
}

__global__ void __launch_bounds__(RSB_WAVE) k_lz_eigmin(lz_args a) {
  const int s = blockIdx.x;
  if (a.status[s] != LZ_PASSDONE) return;
  extern __shared__ double lds[];
  const int n = a.k[s], M = a.miter_max;
  double *d = lds, *e = d + M;
  const double *Td = a.T + (size_t)s * 2 * M, *Tu = Td + M;
  for (int i = threadIdx.x; i < n; i += RSB_WAVE) {
    d[i] = Td[i];
    e[i] = (i < n - 1) ? Tu[i] : 0.0;
  }
  __syncthreads();
  if (n <= RSB_WAVE) eig_min_wave<1>(n, d, e, a.y + (size_t)s * M, &SC(s, SC_LAMBDA));
  else eig_min_wave<2>(n, d, e, a.y + (size_t)s * M, &SC(s, SC_LAMBDA));
}

__global__ void __launch_bounds__(RSB_WAVE) k_eigmin_test(int n, const double *dd,
                                                          const double *ee, double *y,
                                                          double *lam) {
  extern __shared__ double lds[];
  double *d = lds, *e = d + n;
  for (int i = threadIdx.x; i < n; i += RSB_WAVE) d[i] = dd[i], e[i] = i < n - 1 ? ee[i] : 0.0;
  __syncthreads();
  if (n <= RSB_WAVE) eig_min_wave<1>(n, d, e, y, lam);
  else eig_min_wave<2>(n, d, e, y, lam);
}

__global__ void __launch_bounds__(2 * RSB_WAVE) k_lz_tqli(lz_args a) {
  const int s = blockIdx.x;
  if (a.status[s] != LZ_PASSDONE) return;
  extern __shared__ double lds[];
  __shared__ tqli_shared sh;
  const int n = a.k[s], M = a.miter_max;
  double *d = lds, *e = d + M, *z = e + M;
  const double *Td = a.T + (size_t)s * 2 * M, *Tu = Td + M;
  for (int i = threadIdx.x; i < n; i += 2 * RSB_WAVE) {
    d[i] = Td[i];
    e[i] = (i < n - 1) ? Tu[i] : 0.0;
  }
  __syncthreads();
  if (n <= RSB_WAVE) tqli_wave<1>(n, d, e, z, a.y + (size_t)s * M, &SC(s, SC_LAMBDA), &sh);
  else tqli_wave<2>(n, d, e, z, a.y + (size_t)s * M, &SC(s, SC_LAMBDA), &sh);
}

// Passes longer than 128 iterations (both precisions): segments s0 +
// blockIdx.x, each with its n x n eigenvector matrix at zbuf + blockIdx.x *
// M * M.
__global__ void __launch_bounds__(RSB_WAVE) k_lz_tqli_g(lz_args a, int s0, double *zbuf) {
  const int s = s0 + blockIdx.x;
  if (s >= a.nseg || a.status[s] != LZ_PASSDONE) return;
  extern __shared__ double lds[];
  const int n = a.k[s], M = a.miter_max;
  double *d = lds, *e = d + M;
  const double *Td = a.T + (size_t)s * 2 * M, *Tu = Td + M;
  for (int i = threadIdx.x; i < n; i += RSB_WAVE) {
    d[i] = Td[i];
    e[i] = (i < n - 1) ? Tu[i] : 0.0;
  }
  __syncthreads();
  tqli_wave_mem(n, d, e, zbuf + (size_t)blockIdx.x * M * M, a.y + (size_t)s * M,
                &SC(s, SC_LAMBDA));
}

__global__ void __launch_bounds__(RSB_WAVE) k_tqli_test_g(int n, const double *dd,
                                                          const double *ee, double *y,
                                                          double *lam, double *z) {
  extern __shared__ double lds[];
  double *d = lds, *e = d + n;
  for (int i = threadIdx.x; i < n; i += RSB_WAVE) d[i] = dd[i], e[i] = i < n - 1 ? ee[i] : 0.0;
  __syncthreads();
  tqli_wave_mem(n, d, e, z, y, lam);
}

// Stand-alone tridiagonal solve for the parity tests.
__global__ void __launch_bounds__(2 * RSB_WAVE) k_tqli_test(int n, const double *dd,
                                                        const double *ee, double *y,
                                                        double *lam) {
  extern __shared__ double lds[];
  __shared__ tqli_shared sh;
  double *d = lds, *e = d + n, *z = e + n;
  for (int i = threadIdx.x; i < n; i += 2 * RSB_WAVE) d[i] = dd[i], e[i] = i < n - 1 ? ee[i] : 0.0;
  __syncthreads();
  if (n <= RSB_WAVE) tqli_wave<1>(n, d, e, z, y, lam, &sh);
  else tqli_wave<2>(n, d, e, z, y, lam, &sh);
}

// Ritz vector (fiedler.c:547-553): f = sum_j (r_j / |r_j|) y_j, the basis
// slots holding the residuals r_j unscaled (FP64 accumulation of r_j times
// y_j / |r_j|, j ascending), then its mean (ortho).  Decides restart or
// finish.
template <typename T>
__global__ void __launch_bounds__(RSB_BLOCK) k_lz_ritz(lz_args a, const T *__restrict__ basis,
                                                       int64_t mpad, T *__restrict__ f) {
  tile_t t;
  if (!tile_of(a, LZ_PASSDONE, t)) return;
  const int s = t.s, k = a.k[s];
  const double *y = a.y + (size_t)s * a.miter_max;
  const double *rn = a.rn + (size_t)s * (a.miter_max + 1);
  double v[1] = {0.0};
  if constexpr (sizeof(T) == 4) {
    // FP32: four consecutive rows per thread, one 16-byte load per basis
    // vector, eight vectors in flight (vectors past k read vector k - 1 and
    // are skipped); each row sums j ascending, as below
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    constexpr int U = 8;
    for (int row = t.row0 + 4 * (int)threadIdx.x; row < t.row1; row += 4 * (int)blockDim.x) {
      double x[4] = {0.0, 0.0, 0.0, 0.0};
      for (int j0 = 0; j0 < k; j0 += U) {
        f32x4 b[U];
#pragma unroll
        for (int u = 0; u < U; u++)
          b[u] = *(const f32x4 *)(basis + (size_t)min(j0 + u, k - 1) * mpad + row);
#pragma unroll
        for (int u = 0; u < U; u++)
          if (j0 + u < k) {
            const double yj = y[j0 + u] * rn[j0 + u];
            x[0] += (double)b[u].x * yj, x[1] += (double)b[u].y * yj;
            x[2] += (double)b[u].z * yj, x[3] += (double)b[u].w * yj;
          }
      }
      f32x4 o;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const float xq = row + q - t.pstart < t.n ? (float)x[q] : 0.f;
        o[q] = xq;
        v[0] += (double)xq;
      }
      *(f32x4 *)(f + row) = o;
    }
    publish<1>(a, t, v);
    return;
  }
  // The (up to) four rows of a thread together and eight basis vectors at a
  // time, every load unconditional (rows past the tile read its last row,
  // vectors past k read vector k - 1 and are skipped): 32 loads in flight
  // per lane, no branches between them.  Each row sums j ascending.
  constexpr int R = RSB_TILE / RSB_BLOCK, U = 8;
  int rows[R];
  double x[R];
#pragma unroll
  for (int q = 0; q < R; q++) {
    rows[q] = min(t.row0 + (int)threadIdx.x + q * (int)blockDim.x, t.row1 - 1);
    x[q] = 0.0;
  }
  for (int j0 = 0; j0 < k; j0 += U) {
    T b[U][R];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const T *bj = basis + (size_t)min(j0 + u, k - 1) * mpad;
#pragma unroll
      for (int q = 0; q < R; q++) b[u][q] = bj[rows[q]];
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      if (j0 + u < k) {
        const double yj = y[j0 + u] * rn[j0 + u];
#pragma unroll
        for (int q = 0; q < R; q++) x[q] += (double)b[u][q] * yj;
      }
  }
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int row = t.row0 + (int)threadIdx.x + q * (int)blockDim.x;
    if (row >= t.row1) continue;
    const double xq = row - t.pstart < t.n ? x[q] : 0.0;
    f[row] = (T)xq;
    v[0] += (double)(T)xq;
  }
  publish<1>(a, t, v);
}

// Final normalisation (fiedler.c:606-616) and scatter to compact positions.
template <typename T>
__global__ void __launch_bounds__(RSB_BLOCK) k_lz_finish(lz_args a, int phase,
                                                         const T *__restrict__ f,
                                                         double *__restrict__ fied,
                                                         double *__restrict__ xrow) {
  tile_t t;
  if (!tile_of(a, LZ_FINISHED, t)) return;
  const int s = t.s;
  const double mf = SC(s, SC_MEANF);
  if (phase == 1) {
    const double ni = SC(s, SC_NORMF);
    const int cstart = a.seg[s];
    for (int row = t.row0 + threadIdx.x; row < t.row1; row += blockDim.x) {
      int i = row - t.pstart;
      double x = i < t.n ? ((double)f[row] - mf) * ni : 0.0;
      xrow[row] = x;
      if (i < t.n) fied[cstart + i] = x;
    }
    return;
  }
  double v[1] = {0.0};
  for (int row = t.row0 + threadIdx.x; row < t.row1; row += blockDim.x) {
    int i = row - t.pstart;
    if (i < t.n) {
      double x = (double)f[row] - mf;
      v[0] += x * x;
    }
  }
  publish<1>(a, t, v);
}

// Eigen-residual of the final vector x (FP64): lambda_R = x.Lx, then
// |Lx - lambda_R x| / lambda_R.
__global__ void __launch_bounds__(RSB_BLOCK) k_lz_resid(lz_args a, int phase,
                                                        const double *__restrict__ x,
                                                        const int64_t *__restrict__ slice_off,
                                                        const int *__restrict__ slice_w,
                                                        const uint32_t *__restrict__ ell) {
  tile_t t;
  if (!tile_of(a, LZ_FINISHED, t)) return;
  const int s = t.s;
  const double lam = phase ? SC(s, SC_RES) : 0.0;
  double v[1] = {0.0};
  for (int row = t.row0 + threadIdx.x; row < t.row1; row += blockDim.x) {
    const int sl = row >> 6, lane = row & 63;
    const uint32_t *e = ell + slice_off[sl] + lane;
    const double xi = x[row];
    const int w = slice_w[sl];
    double sum = 0.0;
    // eight entries, then their gathers, in flight
    for (int j0 = 0; j0 < w; j0 += 8) {
      uint32_t q[8];
      double xc[8];
#pragma unroll
      for (int u = 0; u < 8; u++) q[u] = j0 + u < w ? e[(size_t)(j0 + u) * RSB_WAVE] : (uint32_t)row;
#pragma unroll
      for (int u = 0; u < 8; u++) xc[u] = x[q[u] & 0x0fffffffu];
#pragma unroll
      for (int u = 0; u < 8; u++) sum = fmat((double)(q[u] >> 28), xi - xc[u], sum);
    }
    if (phase == 0) v[0] += sum * xi;
    else {
      double d = sum - lam * xi;
      v[0] += d * d;
    }
  }
  publish<1>(a, t, v);
}

// ---------------------------------------------------------------------------
// Segment finalisation: the sums of a segment's tile partials (fixed order)
// and the scalar updates of the phase that produced them.  One workgroup per
// segment; segments not in the phase's state leave at once.
enum {
  FIN_START0 = 0, FIN_START1, FIN_SETUP0, FIN_SETUP1, FIN_APPLY, FIN_RUPDATE, FIN_RITZ,
  FIN_FINISH, FIN_RES0, FIN_RES1, FIN_APPLYR
};

__device__ inline int fin_status(int op) {
  switch (op) {
    case FIN_START0: case FIN_START1: case FIN_SETUP0: case FIN_SETUP1: return LZ_SETUP;
    case FIN_APPLY: case FIN_RUPDATE: case FIN_APPLYR: return LZ_RUNNING;
    case FIN_RITZ: return LZ_PASSDONE;
    default: return LZ_FINISHED;
  }
}

// Totals of NV partial slots (slot k at partial + k * stride) of a segment:
// U tiles per thread in flight (large segments have up to 16k tiles), a
// fixed order of summation (thread t adds tiles t, t + blockDim.x, ... in
// turn, then the block's tree).  Thread 0 holds them.
template <int NV, int U, int NT>
__device__ inline void fin_sums(const double *__restrict__ partial, int stride, int first,
                                int count, double (&tot)[NV], double *red) {
#pragma unroll
  for (int k = 0; k < NV; k++) tot[k] = 0.0;
  for (int i0 = 0; i0 < count; i0 += U * NT) {
    double v[NV][U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + u * NT + (int)threadIdx.x;
      const double *p = partial + first + min(i, count - 1);
#pragma unroll
      for (int k = 0; k < NV; k++) {
        const double x = p[(size_t)k * stride];
        v[k][u] = i < count ? x : 0.0;
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int k = 0; k < NV; k++) tot[k] += v[k][u];
  }
  block_sum<NV, NT / RSB_WAVE>(tot, red);
}

// |r - af w|^2 from the folded apply's sums r.r, r.w, w.w, af = alpha as the
// next launch rounds it, from this iteration's stored r and w, so the value
// does not drift over the iterations.  With rho = |r| / |r - af w| it is off by
// at most 2^-24 (2 rho + 1)^2 relative from the sums (each within 2^-24 of its
// magnitude, |af w| <= |r| + |r - af w|), and by 2^-23 from the rounding of
// the new r: 1e-6 or less where an iteration leaves the residual about as it
// was, as nearly all do.  Errors of the sums' terms cancel mostly: 3e-7 was
// measured at rho = 10, 3e-5 at 100 (1,170 rows; 2e-6 from the stored new r).
__device__ inline double fold_rtr(double alpha, double rr, double rw, double ww) {
  const double af = (double)(float)alpha;
  const double rtr = fmat(af * af, ww, fmat(-2.0 * af, rw, rr));
  return rtr > 0.0 ? rtr : 0.0;
}

// The stop test and the next coefficients after the residual update of
// iteration it, from rtr = r.r of the new residual (fiedler.c:486-509).
__device__ inline void rupdate_step(const lz_args &a, int s, double rtr) {
  const int it = a.iter[s], mi = a.miter[s];
  double rnorm = sqrt(rtr);
  double rtz1 = SC(s, SC_RTZ1), rtz2 = SC(s, SC_RTZ2), beta = SC(s, SC_BETA);
  double pap = SC(s, SC_PAP), pap_old = SC(s, SC_PAPOLD);
  double *Td = a.T + (size_t)s * 2 * a.miter_max, *Tu = Td + a.miter_max;
  if (it == 0) {
    Td[0] = pap / rtz1;
  } else {
    Td[it] = fmat(beta * beta, pap_old, pap) / rtz1;
    Tu[it - 1] = -beta * pap_old / sqrt(rtz2 * rtz1);
  }
  SC(s, SC_RTR) = rtr;
  SC(s, SC_RNORM) = rnorm;
  SC(s, SC_RNI) = 1.0 / rnorm;
  a.rn[(size_t)s * (a.miter_max + 1) + it + 1] = 1.0 / rnorm;
  if (rnorm < SC(s, SC_RTOL) || it + 1 == mi) {
    a.k[s] = it + 1;
    a.status[s] = LZ_PASSDONE;
  } else {
    a.iter[s] = it + 1;
    SC(s, SC_RTZ2) = rtz1;
    SC(s, SC_RTZ1) = rtr;
    SC(s, SC_BETA) = rtr / rtz1;
  }
}

// NT threads per segment: 256, or 512 for the per-iteration sums of levels
// whose segments hold more than LZ_FIN_WIDE tiles (more partials in flight;
// on thousands of small segments the wider workgroup costs more than it
// saves)
template <int NT>
__global__ void __launch_bounds__(NT) k_lz_fin(lz_args a, int op) {
  __shared__ double red[(NT / RSB_WAVE) * 6];
  const int s = a.act_segs ? a.act_segs[blockIdx.x] : blockIdx.x;
  if (a.status[s] != fin_status(op)) return;
  const int first = a.seg_tiles[2 * s], count = a.seg_tiles[2 * s + 1];
  // only the slots the phase wrote are read
  // one pass over the slots the phase wrote (all of them in flight together)
  double tot[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (op == FIN_APPLYR) {
    fin_sums<6, 8, NT>(a.partial, a.pstride, first, count, tot, red);
  } else if (op == FIN_APPLY) {
    double t3[3];
    fin_sums<3, 8, NT>(a.partial, a.pstride, first, count, t3, red);
    tot[0] = t3[0], tot[1] = t3[1], tot[2] = t3[2];
  } else {
    double t1[1];
    fin_sums<1, 8, NT>(a.partial, a.pstride, first, count, t1, red);
    tot[0] = t1[0];
  }
  if (threadIdx.x != 0) return;
  const double n = a.seg[a.nseg + s];
  switch (op) {
    case FIN_START0: SC(s, SC_M0) = tot[0] / n; break;
    case FIN_START1:
      if (a.mode == 2 && a.max_n > 0 && a.seg[a.nseg + s] > a.max_n) {
        // above the size limit: no learned attempt, reference start next
        SC(s, SC_N0) = 0.0;
        SC(s, SC_FALLBACK) = -1.0;
        a.k[s] = a.miter[s];
        a.status[s] = LZ_FINISHED;
      } else if (a.mode == 2 && !(tot[0] > 0.0 && tot[0] < INFINITY)) {
        // constant or non-finite prediction: no pass, straight to the fallback
        SC(s, SC_N0) = 0.0;
        a.k[s] = a.miter[s];
        a.status[s] = LZ_FINISHED;
      } else {
        SC(s, SC_N0) = 1.0 / sqrt(tot[0]);
      }
      break;
    case FIN_SETUP0: SC(s, SC_TMP) = tot[0] / n; break;
    case FIN_SETUP1: {  // fiedler.c:441-456
      double rtr = tot[0], rn = sqrt(rtr);
      SC(s, SC_RTR) = rtr;
      SC(s, SC_RNORM) = rn;
      SC(s, SC_RNORM0) = rn;
      SC(s, SC_RTOL) = rn * a.tol;
      SC(s, SC_RNI) = 1.0 / rn;
      a.rn[(size_t)s * (a.miter_max + 1)] = 1.0 / rn;
      SC(s, SC_RTZ1) = rtr;  // iteration 0: rtz2 = 1 (initial rtz1), rtz1 = rtr
      SC(s, SC_RTZ2) = 1.0;
      SC(s, SC_BETA) = 0.0;
      SC(s, SC_PAP) = 0.0;
      SC(s, SC_MEANP) = 0.0;
      if (a.st0) a.st0[s] = lz_it{rtr, 1.0, 0.0, 0.0, 0.0, 0.0, 0.0, rn * a.tol, -1, a.miter[s]};
      a.iter[s] = 0;
      a.status[s] = LZ_RUNNING;
      break;
    }
    case FIN_APPLY: {  // mean of p, pap = w.(p - mean), alpha (fiedler.c:470-478)
      double mq = tot[0] / n;
      double pap = fmat(-mq, tot[2], tot[1]);
      SC(s, SC_MEANP) = mq;
      SC(s, SC_PAPOLD) = SC(s, SC_PAP);
      SC(s, SC_PAP) = pap;
      SC(s, SC_ALPHA) = SC(s, SC_RTZ1) / pap;
      break;
    }
    case FIN_RUPDATE: rupdate_step(a, s, tot[0]); break;  // tot: r.r
    case FIN_APPLYR: {  // FIN_APPLY, then the update's r.r from the sums r.r, r.w, w.w
      double mq = tot[0] / n;
      double pap = fmat(-mq, tot[2], tot[1]);
      SC(s, SC_MEANP) = mq;
      SC(s, SC_PAPOLD) = SC(s, SC_PAP);
      SC(s, SC_PAP) = pap;
      const double alpha = SC(s, SC_RTZ1) / pap;
      SC(s, SC_ALPHA) = alpha;
      const double rtr = fold_rtr(alpha, tot[3], tot[4], tot[5]);
      SC(s, SC_NFOLD) += 1.0;
      rupdate_step(a, s, rtr);
      break;
    }
    case FIN_RITZ: {  // mean of the Ritz vector; restart or finish (fiedler.c:529-553)
      const int k = a.k[s];
      SC(s, SC_MEANF) = tot[0] / n;
      int np = a.npass[s] + 1;
      a.npass[s] = np;
      a.niter[s] = (np - 1) * a.miter[s] + k;
      const double lam = SC(s, SC_LAMBDA), lprev = SC(s, SC_LAMPREV);
      SC(s, SC_LAMPREV) = lam;
      bool stalled = a.stall > 0.0 && np >= max(2, a.stall_min) &&
                     fabs(lam - lprev) <= a.stall * fabs(lam);
      if (a.plateau > 0.0 && k >= 2) {
        // the Ritz pair's residual |L f - lam f| / (lam |f|) from the Lanczos
        // relation: |t_{k+1,k}| |y_k| / (|y| lam), t_{k+1,k} the next
        // off-diagonal of T, -beta_k pap_{k-1} / sqrt(rtz_{k-1} rtz_k) with
        // beta_k = rtz_k / rtz_{k-1} (the state the last update left)
        const double rk = SC(s, SC_RTR), rk1 = SC(s, SC_RTZ1), pap = SC(s, SC_PAP);
        const double t = (rk / rk1) * pap / sqrt(rk1 * rk);
        const double *y = a.y + (size_t)s * a.miter_max;
        double yy = 0.0;
        for (int j = 0; j < k; j++) yy += y[j] * y[j];
        const double rho = fabs(t * y[k - 1]) / (sqrt(yy) * fabs(lam));
        stalled |= np >= 4 && rho <= a.plateau_max && rho >= a.plateau * SC(s, SC_RHO2);
        SC(s, SC_RHO2) = SC(s, SC_RHO1);
        SC(s, SC_RHO1) = rho;
      }
      if (k == a.miter[s] && np < a.mpass && !stalled) {
        a.status[s] = LZ_SETUP;
      } else {
        a.status[s] = LZ_FINISHED;
      }
      break;
    }
    case FIN_FINISH: SC(s, SC_NORMF) = 1.0 / sqrt(tot[0]); break;
    case FIN_RES0: SC(s, SC_RES) = tot[0]; break;
    case FIN_RES1: SC(s, SC_TMP) = sqrt(tot[0]) / SC(s, SC_RES); break;
  }
}

// ---------------------------------------------------------------------------
// Fused iterations: the finishing step of each reduction is done by the
// launch that needs its result.  Every workgroup of a segment sums the
// segment's partials (the order of k_lz_fin<RSB_BLOCK>, so every workgroup
// gets the same bits) and forms the scalars itself; the workgroup of the
// segment's first tile also records them.  An iteration is then one launch
// with the folded update and two without, instead of two and four, and the
// sums overlap the loads of the window, which do not need them.  Launches
// read one copy of the partials and of the segment state and write the
// other, so no workgroup reads what another of the same launch writes
// (status apart: a segment that stops is recorded there by its first tile,
// and every other workgroup of it leaves either way).
// These launches are bound by their chain of dependent loads: one record per
// tile and one per slice instead of walking five tables, and the sums in the
// shadow of the window, took 250 tiles of quads (FP32, folded) from 11.8 +
// 5.4 us (apply, finishing launch) to 10.3 us an iteration, 184 tiles of
// hexes in FP64 from 13.5 + 4.0 + 2 x 3.75 to 11.6 + 4.1 us.
struct lz_fuse {
  const lz_desc *list;  // tiles of the launch, split over the XCDs as in list_index
  int nlist, per;       // per: grid / LZ_XCDS
  int it;               // iteration of the pass (the same for every running segment)
  const lz_it *st_in;
  lz_it *st_out;
  const double *pa_in;  // partials of the launch before; those of this one go to lz_args.partial
};
// most tiles of a segment: one round of four loads per thread covers the
// partials of an unfolded launch, two rounds of two (of each of six slots)
// those of a folded one from 513 tiles on.  Whole calls at 1,024 / 512 / 256 /
// 0 (separate launches): 1M hexes FP64 78.7 / 80.3 / 82.1 / 86.2 ms, FP32
// 60.9 / 61.3 / 62.4 / 64.6, 2M pipe 702 / 704 / 707 / 739, 260k quads 239 /
// 239 / 239 / 302
#define LZ_FUSE_TILES 1024
// iterations queued between a compaction and the look at its lengths: two of
// 5 to 10 us cover the host's look and its next launches
#define LZ_AHEAD 2

// Scalars after the apply's sums: mean of p, pap, alpha (FIN_APPLY).
__device__ inline void step_apply(lz_it &x, double n, double sq, double swq, double sw) {
  const double mq = sq / n;
  const double pap = fmat(-mq, sw, swq);
  x.meanp = mq;
  x.pap_old = x.pap;
  x.pap = pap;
  x.alpha = x.rtz1 / pap;
}
// The stop test and next coefficients after r.r of iteration x.it
// (rupdate_step on the state record); lead: this workgroup records them.
// Returns false when the pass is over.
__device__ inline bool step_update(const lz_args &a, int s, lz_it &x, double rtr, bool lead,
                                   bool fold) {
  const int it = x.it;
  const double rnorm = sqrt(rtr);
  const bool stop = rnorm < x.rtol || it + 1 == x.mi;
  if (lead) {
    double *Td = a.T + (size_t)s * 2 * a.miter_max, *Tu = Td + a.miter_max;
    if (it == 0) {
      Td[0] = x.pap / x.rtz1;
    } else {
      Td[it] = fmat(x.beta * x.beta, x.pap_old, x.pap) / x.rtz1;
      Tu[it - 1] = -x.beta * x.pap_old / sqrt(x.rtz2 * x.rtz1);
    }
    a.rn[(size_t)s * (a.miter_max + 1) + it + 1] = 1.0 / rnorm;
    if (stop) {
      SC(s, SC_RTR) = rtr;
      SC(s, SC_RNORM) = rnorm;
      SC(s, SC_RNI) = 1.0 / rnorm;
      SC(s, SC_RTZ1) = x.rtz1, SC(s, SC_RTZ2) = x.rtz2, SC(s, SC_BETA) = x.beta;
      SC(s, SC_PAP) = x.pap, SC(s, SC_PAPOLD) = x.pap_old;
      SC(s, SC_MEANP) = x.meanp, SC(s, SC_ALPHA) = x.alpha;
      if (fold) SC(s, SC_NFOLD) += it + 1;
      a.iter[s] = it;
      a.k[s] = it + 1;
      a.status[s] = LZ_PASSDONE;
    }
  }
  if (stop) return false;
  const double rtz1 = x.rtz1;
  x.rtz2 = rtz1;
  x.rtz1 = rtr;
  x.beta = rtr / rtz1;
  return true;
}

struct lz_bc {
  double beta, m, alpha;
  int go;
};
// The finishing step in front of an apply: sums of the launch before, the
// scalars of the next iteration (broadcast through LDS), their record.
// Returns false where the segment's pass is over.
template <bool FOLD>
__device__ inline bool fuse_next(const lz_args &a, const lz_fuse &fu, const lz_desc &d, int status,
                                 double *red, lz_bc *bc) {
  constexpr int NV = FOLD ? 6 : 1;
  double tot[NV];
  lz_it x;
  it_load(x, fu.st_in + d.s);
  fin_sums<NV, FOLD ? 2 : 4, RSB_BLOCK>(fu.pa_in, a.pstride, d.first, d.count, tot, red);
  if (threadIdx.x == 0) {
    const bool run = status == LZ_RUNNING, lead = run && d.ti == d.first;
    double rtr = tot[0];
    if constexpr (FOLD) {
      step_apply(x, (double)d.n, tot[0], tot[1], tot[2]);
      rtr = fold_rtr(x.alpha, tot[3], tot[4], tot[5]);
    }
    const bool go = step_update(a, d.s, x, rtr, lead, FOLD) && run;
    if (go && lead) {
      x.it++;
      it_store(fu.st_out + d.s, x);
    }
    bc->beta = x.beta, bc->m = x.meanp, bc->alpha = x.alpha, bc->go = go;
  }
  __syncthreads();
  return bc->go != 0;
}

__device__ inline tile_t tile_from(const lz_desc &d) {
  tile_t t;
  t.ti = d.ti, t.s = d.s, t.row0 = d.row0, t.row1 = d.row1;
  t.pstart = d.pstart, t.n = d.n, t.first = d.first, t.count = d.count;
  return t;
}

// The window's loads: the thread's own rows and its first halo rows, in
// registers while the sums are formed.  Own rows: four in one access (FP32:
// 4 tid .. + 3), or two pairs (FP64: 2 tid, 2 tid + 512).
template <typename T, bool UPD>
struct window_regs {
  static constexpr int SU = 4;
  typedef T vec __attribute__((ext_vector_type(16 / sizeof(T))));
  static constexpr int V = 16 / sizeof(T), NV = LZ_RPT / V;  // rows per access, accesses
  vec r[NV], p[NV], w[NV];
  int gr[SU];
  T rg[SU], po[SU], wg[SU];
  __device__ inline void load(const tile_t &t, const int *__restrict__ halo, int nh,
                              const T *__restrict__ rr, const T *__restrict__ pold,
                              const T *__restrict__ wp) {
    const int nrows = t.row1 - t.row0;
#pragma unroll
    for (int k = 0; k < SU; k++) {
      const int i = (int)threadIdx.x + k * RSB_BLOCK;
      gr[k] = i < nh ? halo[i] : t.row0;
    }
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const int i = V * ((int)threadIdx.x + k * RSB_BLOCK);
      const int o = t.row0 + (i < nrows ? i : 0);
      r[k] = *(const vec *)(rr + o);
      p[k] = *(const vec *)(pold + o);
      if (UPD) w[k] = *(const vec *)(wp + o);
    }
#pragma unroll
    for (int k = 0; k < SU; k++) {
      rg[k] = rr[gr[k]];
      po[k] = pold[gr[k]];
      wg[k] = UPD ? wp[gr[k]] : (T)0;
    }
  }
  // q = beta (p - m) + r into the window, r of the tile's rows beside it
  // (UPD: r = r - alpha w first, also written to its basis slot rn)
  template <bool KEEP_R>
  __device__ inline void fill(const tile_t &t, const int *__restrict__ halo, int nh, T *ql, T *rl,
                              const T *__restrict__ rr, const T *__restrict__ pold,
                              const T *__restrict__ wp, T beta, T m, T alpha,
                              T *__restrict__ rn) {
    const int nrows = t.row1 - t.row0;
    const int nreal = min(nrows, t.pstart + t.n - t.row0);
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const int i = V * ((int)threadIdx.x + k * RSB_BLOCK);
      if (i >= nrows) continue;
      vec x = r[k], q;
#pragma unroll
      for (int j = 0; j < V; j++) {
        if (UPD) x[j] = rsub(x[j], alpha, w[k][j]);
        q[j] = fmat(beta, p[k][j] - m, x[j]);
        if (i + j >= nreal) q[j] = (T)0;
      }
      if (UPD) *(vec *)(rn + t.row0 + i) = x;
      *(vec *)(ql + i) = q;
      if (KEEP_R) *(vec *)(rl + i) = x;
    }
#pragma unroll
    for (int k = 0; k < SU; k++) {
      const int i = (int)threadIdx.x + k * RSB_BLOCK;
      if (i >= nh) break;
      const T x = UPD ? rsub(rg[k], alpha, wg[k]) : rg[k];
      ql[nrows + i] = fmat(beta, po[k] - m, x);
    }
    for (int i0 = (int)threadIdx.x + SU * RSB_BLOCK; i0 < nh; i0 += SU * RSB_BLOCK) {
#pragma unroll
      for (int k = 0; k < SU; k++) {
        const int i = i0 + k * RSB_BLOCK;
        gr[k] = i < nh ? halo[i] : t.row0;
      }
#pragma unroll
      for (int k = 0; k < SU; k++) {
        rg[k] = rr[gr[k]];
        po[k] = pold[gr[k]];
        wg[k] = UPD ? wp[gr[k]] : (T)0;
      }
#pragma unroll
      for (int k = 0; k < SU; k++) {
        const int i = i0 + k * RSB_BLOCK;
        if (i >= nh) break;
        const T x = UPD ? rsub(rg[k], alpha, wg[k]) : rg[k];
        ql[nrows + i] = fmat(beta, po[k] - m, x);
      }
    }
    __syncthreads();
  }
};

template <typename T, bool FOLD>
__global__ void __launch_bounds__(RSB_BLOCK) k_lz_apply_f(lz_args a, lz_fuse fu,
                                                          const T *__restrict__ pold,
                                                          T *__restrict__ pnew, T *__restrict__ w,
                                                          T *__restrict__ basis, int64_t mpad,
                                                          tiled_args ta,
                                                          const T *__restrict__ wprev) {
  __shared__ __attribute__((aligned(16))) T ql[TB_LOCAL];
  // as in lz_apply_tiled
  constexpr bool KEEP_R = FOLD || sizeof(T) == 4;
  __shared__ __attribute__((aligned(16))) T rl[KEEP_R ? RSB_TILE : 4];
  __shared__ double red[(RSB_BLOCK / RSB_WAVE) * 6];
  __shared__ lz_bc bc;
  const int li = (int)(blockIdx.x % LZ_XCDS) * fu.per + (int)(blockIdx.x / LZ_XCDS);
  if (li >= fu.nlist) return;
  const lz_desc d = fu.list[li];
  // tested with the sums, when the window's loads are on their way (a test
  // here would put a round trip in front of them; they stay in bounds for a
  // segment that has stopped)
  const int status = a.status[d.s];
  const tile_t t = tile_from(d);
  const int it = fu.it, nh = d.nhalo;
  T *cur = basis + (size_t)it * mpad;
  const slice_meta sm = load_meta(t, ta);
  acc_t<T> sq, swq, sw;
  fold_t<T> fd;
  fd.wp = wprev, fd.rn = it == 0 ? nullptr : cur, fd.alpha = (T)0;
  const int nreal = min(t.row1 - t.row0, t.pstart + t.n - t.row0);
  const int *halo = ta.halo + d.halo_off;
  if (it == 0) {
    if (status != LZ_RUNNING) return;
    if (threadIdx.x == 0 && d.ti == d.first) {
      lz_it x;
      it_load(x, fu.st_in + d.s);
      x.it = 0;
      it_store(fu.st_out + d.s, x);
    }
    if (nh >= 0)
      stage_window<T, true, KEEP_R, FOLD>(t, halo, nh, ql, rl, cur, pold, (T)0, (T)0);
    else
      lz_apply_rows<T, true, FOLD>(a, t, cur, pold, pnew, w, (T)0, (T)0, ta.slice_off, ta.slice_w,
                                   ta.ell, sq, swq, sw, fd);
  } else {
    // r_it, or r_{it-1} to update
    const T *__restrict__ r = FOLD ? cur - mpad : cur;
    if (nh >= 0) {
      window_regs<T, FOLD> wr;
      wr.load(t, halo, nh, r, pold, wprev);
      if (!fuse_next<FOLD>(a, fu, d, status, red, &bc)) return;
      wr.template fill<KEEP_R>(t, halo, nh, ql, rl, r, pold, wprev, (T)bc.beta, (T)bc.m,
                             (T)bc.alpha, cur);
    } else {
      if (!fuse_next<FOLD>(a, fu, d, status, red, &bc)) return;
      fd.alpha = (T)bc.alpha;
      lz_apply_rows<T, false, FOLD>(a, t, r, pold, pnew, w, (T)bc.beta, (T)bc.m, ta.slice_off,
                                    ta.slice_w, ta.ell, sq, swq, sw, fd);
    }
  }
  if (nh >= 0) {
    if (ta.e12)
      apply_rows_e12<T, 2, FOLD>(t, ta, sm, ql, rl, pnew, w, nreal, sq, swq, sw, fd);
    else
      apply_rows_batched<T, 2, FOLD>(t, ta, sm, ql, rl, pnew, w, nreal, sq, swq, sw, fd);
  }
  if (FOLD) {
    double v[6] = {sq.value(), swq.value(), sw.value(),
                   fd.rr.value(), fd.rw.value(), fd.ww.value()};
    publish<6>(a, t, v);
  } else {
    double v[3] = {sq.value(), swq.value(), sw.value()};
    publish<3>(a, t, v);
  }
}

// The update r_{it+1} = r_it - alpha w of the fused iterations, with the
// apply's finishing step in front (k_lz_rupdate otherwise).
template <typename T>
__global__ void __launch_bounds__(RSB_BLOCK) k_lz_rupdate_f(lz_args a, lz_fuse fu,
                                                            T *__restrict__ basis, int64_t mpad,
                                                            const T *__restrict__ w) {
  __shared__ double red[(RSB_BLOCK / RSB_WAVE) * 3];
  __shared__ double balpha;
  const int li = (int)(blockIdx.x % LZ_XCDS) * fu.per + (int)(blockIdx.x / LZ_XCDS);
  if (li >= fu.nlist) return;
  const lz_desc d = fu.list[li];
  const int status = a.status[d.s];
  const tile_t t = tile_from(d);
  const T *__restrict__ r = basis + (size_t)fu.it * mpad;
  T *__restrict__ rn = basis + (size_t)(fu.it + 1) * mpad;
  const int nrows = t.row1 - t.row0;
  // the rows of a thread, in the order their squares are summed: four
  // consecutive ones (FP32, one access), or every 256th (FP64)
  constexpr int V = sizeof(T) == 4 ? LZ_RPT : 1, R = LZ_RPT / V;
  typedef T vec __attribute__((ext_vector_type(V)));
  vec rv[R], wv[R];
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int i = V * ((int)threadIdx.x + k * RSB_BLOCK);
    const int o = t.row0 + (i < nrows ? i : 0);
    rv[k] = *(const vec *)(r + o);
    wv[k] = *(const vec *)(w + o);
  }
  lz_it x;
  it_load(x, fu.st_in + d.s);
  double tot[3];
  fin_sums<3, 4, RSB_BLOCK>(fu.pa_in, a.pstride, d.first, d.count, tot, red);
  if (status != LZ_RUNNING) return;
  if (threadIdx.x == 0) {
    step_apply(x, (double)d.n, tot[0], tot[1], tot[2]);
    if (d.ti == d.first) it_store(fu.st_out + d.s, x);
    balpha = x.alpha;
  }
  __syncthreads();
  const T alpha = (T)balpha;
  acc_t<T> acc;
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int i = V * ((int)threadIdx.x + k * RSB_BLOCK);
    if (i >= nrows) continue;
    vec y;
#pragma unroll
    for (int j = 0; j < V; j++) y[j] = rsub(rv[k][j], alpha, wv[k][j]);
    *(vec *)(rn + t.row0 + i) = y;
#pragma unroll
    for (int j = 0; j < V; j++) acc.dot(y[j], y[j]);
  }
  double v[1] = {acc.value()};
  publish<1>(a, t, v);
}

// The finishing step after the last iteration of a pass.
template <bool FOLD>
__global__ void __launch_bounds__(RSB_BLOCK) k_lz_last(lz_args a, lz_fuse fu,
                                                       const int *__restrict__ segs) {
  __shared__ double red[(RSB_BLOCK / RSB_WAVE) * 6];
  __shared__ lz_bc bc;
  lz_desc d;
  d.s = segs[blockIdx.x];
  const int status = a.status[d.s];
  if (status != LZ_RUNNING) return;
  d.first = d.ti = a.seg_tiles[2 * d.s], d.count = a.seg_tiles[2 * d.s + 1];
  d.n = a.seg[a.nseg + d.s];
  fuse_next<FOLD>(a, fu, d, status, red, &bc);
}

__global__ void k_lz_slices(int64_t nslices, const int64_t *__restrict__ off,
                            const int *__restrict__ w, const int *__restrict__ c,
                            slice_rec *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nslices) out[i] = slice_rec{off[i], w[i], c ? c[i] : 0};
}

__global__ void k_lz_desc(lz_args a, int ntiles, const int *__restrict__ nhalo,
                          const int64_t *__restrict__ halo_off, lz_desc *__restrict__ out) {
  const int ti = blockIdx.x * blockDim.x + threadIdx.x;
  if (ti >= ntiles) return;
  lz_desc d;
  d.s = a.tile[3 * ti], d.row0 = a.tile[3 * ti + 1], d.row1 = a.tile[3 * ti + 2];
  d.pstart = a.seg[4 * a.nseg + d.s], d.n = a.seg[a.nseg + d.s];
  d.first = a.seg_tiles[2 * d.s], d.count = a.seg_tiles[2 * d.s + 1];
  d.nhalo = nhalo[ti], d.halo_off = halo_off[ti], d.ti = ti;
  d.pad0 = 0;
  for (int k = 0; k < 4; k++) d.pad[k] = 0;
  out[ti] = d;
}

// Lists of the tiles and segments in a given state (order irrelevant: every
// tile writes its partial at its own index and k_lz_fin sums them in tile
// order).
__global__ void k_lz_compact(lz_args a, int ntiles, int want, int *__restrict__ tiles,
                             int *__restrict__ segs, int *__restrict__ counts,
                             const lz_desc *__restrict__ desc, lz_desc *__restrict__ list) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < ntiles && a.status[a.tile[3 * i]] == want) {
    const int k = atomicAdd(&counts[0], 1);
    tiles[k] = i;
    if (list) list[k] = desc[i];
  }
  if (i < a.nseg && a.status[i] == want) segs[atomicAdd(&counts[1], 1)] = i;
}

// The lists' lengths to the host's pinned ring (ring[2] = 1 once they are
// there), cleared for the next compaction.
__global__ void k_lz_report(int *counts, int *ring) {
  const int n0 = counts[0], n1 = counts[1];
  counts[0] = 0, counts[1] = 0;
  __hip_atomic_store(ring, n0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(ring + 1, n1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(ring + 2, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void k_lz_init_state(lz_args a, int miter_opt) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= a.nseg) return;
  int n = a.seg[a.nseg + s], p = a.seg[2 * a.nseg + s];
  a.status[s] = (p > 1 && n >= 2) ? LZ_SETUP : LZ_IDLE;
  a.miter[s] = n < miter_opt ? n : miter_opt;  // fiedler.c:522
  a.npass[s] = 0, a.niter[s] = 0, a.iter[s] = 0, a.k[s] = 0;
  for (int j = 0; j < LZ_NSC; j++) SC(s, j) = 0.0;
}

// Learned start: segments that missed tol within their passes (k == miter
// on the last pass, as the restart rule of fiedler.c:529-553 reads it) start
// over from the reference start; the iterations spent so far are kept.
__global__ void k_lz_fallback(lz_args a, int *__restrict__ count) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= a.nseg) return;
  if (a.status[s] != LZ_FINISHED || a.k[s] != a.miter[s]) return;
  const bool skipped = SC(s, SC_FALLBACK) < 0.0;  // above the size limit
  SC(s, SC_WARMIT) = skipped ? 0.0 : a.niter[s];
  SC(s, SC_FALLBACK) = skipped ? -1.0 : 1.0;
  SC(s, SC_MEANF) = 0.0;
  a.npass[s] = 0, a.niter[s] = 0, a.iter[s] = 0, a.k[s] = 0;
  a.status[s] = LZ_SETUP;
  atomicAdd(count, 1);
}

// Segments that cannot be bisected spectrally (fewer than 2 elements) keep
// Fiedler value 0.
__global__ void k_lz_zero_small(lz_args a, double *fied) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= a.nseg) return;
  int n = a.seg[a.nseg + s], p = a.seg[2 * a.nseg + s];
  if (p > 1 && n == 1) fied[a.seg[s]] = 0.0;
}

// ---------------------------------------------------------------------------
template <typename T>
static int run_lanczos(rsbgpu *g, int miter_opt, int mpass, double tol, int init_mode,
                       rsbgpu_fiedler_out *out) {
  const int nseg = g->nseg, ntiles = g->ntiles;
  const int64_t mpad = g->mpad;
  int miter_max = 1;
  for (int s = 0; s < nseg; s++)
    if (g->h_p[s] > 1 && g->h_n[s] >= 2) miter_max = std::max(miter_max, std::min(miter_opt, g->h_n[s]));
  // passes of more than 128 iterations take the tridiagonal solve with its
  // eigenvector matrix in global memory (k_lz_tqli_g)
  const bool long_pass = miter_max > 128;
  // buffers
  size_t vb = (size_t)mpad * sizeof(T);
  if (vb > g->vec_bytes) {
    const size_t old = g->vec_bytes;
    size_t got = ~(size_t)0;
    g->vec_bytes = 0;
    for (void **q : {&g->d_p, &g->d_p2, &g->d_w, &g->d_f, &g->d_w2}) {
      size_t one = 0;
      RSB_TRY(rsb_retire(g, *q, old));
      RSB_TRY(rsb_dev_malloc_grown(g, q, vb + 256, old, &one));
      got = std::min(got, one);
    }
    g->vec_bytes = got - 256;
  }
  // the pass's residuals r_0 .. r_miter (the last one written, not used)
  size_t bb = vb * ((size_t)miter_max + 1);
  if (bb > g->basis_bytes) {
    const size_t old = g->basis_bytes;
    size_t got = 0;
    g->basis_bytes = 0;
    RSB_TRY(rsb_retire(g, g->d_basis, old));
    RSB_TRY(rsb_dev_malloc_grown(g, &g->d_basis, bb + 256, old, &got));
    g->basis_bytes = got - 256;
  }
  double *xrow = nullptr;
  RSB_TRY(RSB_SCRATCH(xrow, sizeof(double) * (mpad + 1)));
  lz_state &L = g->lz;
  if (nseg > g->lz_nseg_cap || miter_max > g->lz_miter_cap) {
    // iter, k, npass, niter and miter are carved from the status block
    const size_t os = (size_t)g->lz_nseg_cap, om = (size_t)g->lz_miter_cap;
    g->lz_nseg_cap = g->lz_miter_cap = 0;
    RSB_TRY(rsb_retire(g, L.status, sizeof(int) * os * 6));
    RSB_TRY(rsb_retire(g, L.sc, sizeof(double) * os * LZ_NSC));
    RSB_TRY(rsb_retire(g, L.T, sizeof(double) * os * 2 * om));
    RSB_TRY(rsb_retire(g, L.y, sizeof(double) * os * om));
    RSB_TRY(rsb_retire(g, L.rn, sizeof(double) * os * (om + 1)));
    // the segment count doubles every level
    const size_t cap = nseg <= 4096 && !g->borrowed ? std::max(64, (os ? 4 : 1) * nseg) : nseg;
    RSB_TRY(rsb_dev_malloc((void **)&L.status, sizeof(int) * cap * 6));
    L.iter = L.status + cap, L.k = L.status + 2 * cap, L.npass = L.status + 3 * cap;
    L.niter = L.status + 4 * cap;
    RSB_TRY(rsb_dev_malloc((void **)&L.sc, sizeof(double) * cap * LZ_NSC));
    RSB_TRY(rsb_dev_malloc((void **)&L.T, sizeof(double) * cap * 2 * miter_max));
    RSB_TRY(rsb_dev_malloc((void **)&L.y, sizeof(double) * cap * miter_max));
    RSB_TRY(rsb_dev_malloc((void **)&L.rn, sizeof(double) * cap * ((size_t)miter_max + 1)));
    g->lz_nseg_cap = (int)cap, g->lz_miter_cap = miter_max;
  }
  if (ntiles > g->lz_tile_cap) {
    const size_t old = sizeof(double) * 12 * (size_t)g->lz_tile_cap;
    size_t got = 0;
    g->lz_tile_cap = 0;
    RSB_TRY(rsb_retire(g, L.partial, old));
    RSB_TRY(rsb_dev_malloc_grown(g, (void **)&L.partial, sizeof(double) * 12 * ntiles, old, &got));
    g->lz_tile_cap = (int)(got / (sizeof(double) * 12));
  }
  if (!L.count) RSB_TRY(rsb_dev_malloc((void **)&L.count, sizeof(int)));
  lz_args a;
  a.st0 = nullptr;
  a.act_tiles = nullptr, a.act_segs = nullptr;
  a.seg = g->d_seg, a.tile = g->d_tile, a.seg_tiles = g->d_seg_tiles, a.row_elem = g->d_row_elem;
  a.nseg = nseg;
  a.status = L.status, a.iter = L.iter, a.k = L.k, a.npass = L.npass, a.niter = L.niter;
  a.miter = L.status + 5 * std::max(g->lz_nseg_cap, 1);
  a.sc = L.sc, a.T = L.T, a.y = L.y, a.partial = L.partial, a.rn = L.rn;
  a.mpass = mpass, a.mode = init_mode, a.tol = tol, a.miter_max = miter_max;
  {
    const char *sv = getenv("PARRSB_AMD_LZ_STALL"), *sm = getenv("PARRSB_AMD_LZ_STALL_MIN");
    a.stall = sv ? atof(sv) : 0.0;
    a.stall_min = sm ? atoi(sm) : 2;
    const char *pv = getenv("PARRSB_AMD_LZ_PLATEAU"), *pm = getenv("PARRSB_AMD_LZ_PLATEAU_MAX");
    a.plateau = pv ? atof(pv) : 0.0;
    a.plateau_max = pm ? atof(pm) : 1e-2;
  }
  a.pstride = std::max(g->lz_tile_cap, 1);
  a.max_n = g->lws_max_n;
  T *p = (T *)g->d_p, *p2 = (T *)g->d_p2, *w = (T *)g->d_w, *f = (T *)g->d_f,
    *basis = (T *)g->d_basis;
  hipStream_t st = g->stream;
#define FIN(op)                                           \
  do {                                                    \
    k_lz_fin<RSB_BLOCK><<<nseg, RSB_BLOCK, 0, st>>>(a, (op)); \
    RSB_LAUNCH_CHECK();                                   \
  } while (0)
  // compacted lists of running tiles / segments for the iteration launches
  int *act = nullptr;
  const size_t act_len = (size_t)ntiles + nseg;  // two copies, see compact_start
  RSB_TRY(RSB_SCRATCH(act, sizeof(int) * (2 * act_len + 2)));
  int *act_t = act, *act_s = act + ntiles, *act_n = act + 2 * act_len;
  RSB_TRY(hipMemsetAsync(act_n, 0, sizeof(int) * 2, st));
  int nact[2] = {ntiles, nseg};
  // segments of at most LZ_FUSE_TILES tiles take the fused iterations: every
  // workgroup sums its segment's partials by itself
  int max_seg_tiles = 0;
  for (int q = 0; q < nseg; q++) max_seg_tiles = std::max(max_seg_tiles, g->h_seg_tiles[2 * q + 1]);
  const char *gv = getenv("PARRSB_AMD_LZ_GRAPH");
  const bool use_graph = !g->prof_spmv && gv && atoi(gv) == 1;
  // the vertex form serves the FP32 path (vectors of T = float)
  const bool vform = g->vt_ok && sizeof(T) == 4;
  const char *fuv = getenv("PARRSB_AMD_LZ_FUSE_TILES");
  const int fuse_tiles = fuv ? std::min(atoi(fuv), LZ_FUSE_TILES) : LZ_FUSE_TILES;
  const bool fuse = !vform && !use_graph && max_seg_tiles <= fuse_tiles;
  lz_desc *desc = nullptr, *act_d = nullptr;
  lz_it *stt = nullptr;
  if (fuse && ntiles > 0) {
    RSB_TRY(RSB_SCRATCH(desc, sizeof(lz_desc) * 3 * (size_t)ntiles));
    act_d = desc + ntiles;
    RSB_TRY(RSB_SCRATCH(stt, sizeof(lz_it) * 2 * (size_t)nseg));
    a.st0 = stt + nseg;  // the copy the first launch of a pass reads
    k_lz_desc<<<nblocks(ntiles, 256), 256, 0, st>>>(a, ntiles, g->d_tnhalo, g->d_thalo_off, desc);
    RSB_LAUNCH_CHECK();
  }
  double *const PA[2] = {L.partial, L.partial + (size_t)6 * std::max(g->lz_tile_cap, 1)};
  lz_args ai = a;  // iteration launches over the running lists
  // A compaction is queued by compact_start, into the copy of the lists that
  // no launch reads, and taken up by compact_take once its lengths have
  // arrived in pinned memory.  What is queued in between runs on the lists
  // before (a finished segment's workgroups return at once) and keeps the
  // device busy while the host looks: a copy and a wait after each left it
  // idle for 20 to 45 us, three times a pass.  The graph replays hold the
  // lists' addresses, so they keep one copy and wait.
  int cur = 0;
  auto compact_start = [&](int want) -> int {
    const int to = use_graph ? cur : cur ^ 1;
    __atomic_store_n(g->ring + 2, 0, __ATOMIC_RELEASE);
    k_lz_compact<<<nblocks(std::max(ntiles, nseg), 256), 256, 0, st>>>(
        a, ntiles, want, act + to * act_len, act + to * act_len + ntiles, act_n, desc,
        desc ? desc + (size_t)(to + 1) * ntiles : nullptr);
    k_lz_report<<<1, 1, 0, st>>>(act_n, g->ring);
    RSB_LAUNCH_CHECK();
    return 0;
  };
  auto compact_take = [&]() -> int {
    if (rsb_wait_flag(g, g->ring + 2)) return 2;
    if (!use_graph) cur ^= 1;
    nact[0] = g->ring[0], nact[1] = g->ring[1];
    act_t = act + cur * act_len, act_s = act_t + ntiles;
    if (desc) act_d = desc + (size_t)(cur + 1) * ntiles;
    ai.act_tiles = act_t, ai.act_segs = act_s;
    return 0;
  };
  auto xgrid = [](int n) { return (unsigned)((n + LZ_XCDS - 1) / LZ_XCDS * LZ_XCDS); };
  ai.act_tiles = act_t, ai.act_segs = act_s;
  // The FP64 apply reads the 16-bit entries: with the 12-bit form it took
  // 0.253 against 0.233 ms per launch on the 256^3 box (FP32: 0.163 against
  // 0.177), the class sums in doubles costing more than the bytes they save.
  const bool want12 = sizeof(T) == 4 || g->e12_f64;
  if (want12) {
    const int e12rc = rsb_level_e12(g);
    if (e12rc) return e12rc;
  }
  const bool use12 = want12 && g->e12_ok;
  slice_rec *srec = nullptr;
  RSB_TRY(RSB_SCRATCH(srec, sizeof(slice_rec) * (size_t)std::max<int64_t>(g->nslices, 1)));
  if (ntiles > 0) {
    k_lz_slices<<<nblocks(g->nslices, 256), 256, 0, st>>>(
        g->nslices, use12 ? g->d_off12 : g->d_off16, use12 ? g->d_w12 : g->d_w16,
        use12 ? g->d_c12 : nullptr, srec);
    RSB_LAUNCH_CHECK();
  }
  tiled_args ta{srec,           g->d_slice_off, g->d_slice_w, g->d_ell, g->d_tnhalo,
                g->d_thalo_off, g->d_halo,      g->d_off16,   g->d_w16, g->d_e16,
                use12 ? g->d_e12 : nullptr};
  vtile_args va{g->d_vt_n,  g->d_vt_loff,    g->d_vt_list, g->d_vt_rowv,
                g->d_tnhalo, g->d_thalo_off, g->d_halo,    g->nv};
  // FP32 with the neighbour entries: a pass that starts with at most
  // fold_tiles running tiles folds the r-update into the next apply
  // (k_lz_apply<float, true>, FIN_APPLYR: two launches per iteration instead
  // of four; w alternates between two buffers by iteration parity).
  // On more tiles the extra halo gathers of w outweigh the saved pass.
  // PARRSB_AMD_LZ_FOLD_TILES sets the limit (0: never).
  const char *fev = getenv("PARRSB_AMD_LZ_FOLD_TILES");
  const int fold_tiles = (sizeof(T) == 4 && !vform) ? (fev ? atoi(fev) : LZ_FOLD_TILES) : 0;
  bool fold = false;
  T *const W[2] = {w, (T *)g->d_w2};
  // one iteration (it: the pass iteration, where every running segment is):
  // the apply launch, then the finishing step(s) and the r-update
  // fused launches: which copies of the state and partials they read; they
  // write the other (without the fold: the apply writes copy 0)
  auto fused = [&](int it, int rd, lz_args &af) {
    af = ai;
    af.partial = PA[rd ^ 1];
    return lz_fuse{act_d, nact[0], (nact[0] + LZ_XCDS - 1) / LZ_XCDS, it, stt + (size_t)rd * nseg, stt + (size_t)(rd ^ 1) * nseg,
                   PA[rd]};
  };
  auto apply_launch = [&](int it) {
    T *pold = (it & 1) ? p2 : p, *pnew = (it & 1) ? p : p2;
    const unsigned grid = xgrid(nact[0]);
    if constexpr (sizeof(T) == 4) {  // FP64 passes are never folded
      if (fold && fuse) {
        lz_args af;
        const lz_fuse fu = fused(it, (it + 1) & 1, af);
        k_lz_apply_f<T, true><<<grid, RSB_BLOCK, 0, st>>>(af, fu, pold, pnew, W[it & 1], basis,
                                                          mpad, ta, W[(it + 1) & 1]);
        return;
      }
      if (fold) {
        k_lz_apply<T, true><<<grid, RSB_BLOCK, 0, st>>>(ai, pold, pnew, W[it & 1], basis, mpad, ta,
                                                        nact[0], W[(it + 1) & 1]);
        return;
      }
      if (vform) {
        k_lz_apply_v<float><<<grid, RSB_BLOCK, 0, st>>>(ai, (const float *)pold, (float *)pnew,
                                                        (float *)w, (const float *)basis, mpad, va,
                                                        ta, nact[0]);
        return;
      }
    }
    if (fuse) {
      lz_args af;
      const lz_fuse fu = fused(it, 1, af);
      k_lz_apply_f<T, false><<<grid, RSB_BLOCK, 0, st>>>(af, fu, pold, pnew, w, basis, mpad, ta,
                                                         nullptr);
    } else {
      k_lz_apply<T, false><<<grid, RSB_BLOCK, 0, st>>>(ai, pold, pnew, w, basis, mpad, ta,
                                                       nact[0], nullptr);
    }
  };
  // the iteration sums: wide workgroups where the segments are big
  const bool wide_fin = max_seg_tiles > LZ_FIN_WIDE;
  auto fin_launch = [&](int op) {
    if (wide_fin) k_lz_fin<2 * RSB_BLOCK><<<nact[1], 2 * RSB_BLOCK, 0, st>>>(ai, op);
    else k_lz_fin<RSB_BLOCK><<<nact[1], RSB_BLOCK, 0, st>>>(ai, op);
  };
  auto after_apply = [&](int it) {
    if (fuse) {
      if (fold) return;
      lz_args af;
      const lz_fuse fu = fused(it, 0, af);
      k_lz_rupdate_f<T><<<xgrid(nact[0]), RSB_BLOCK, 0, st>>>(af, fu, basis, mpad, w);
    } else if (fold) {
      fin_launch(FIN_APPLYR);
    } else {
      fin_launch(FIN_APPLY);
      k_lz_rupdate<T><<<nact[0], RSB_BLOCK, 0, st>>>(ai, basis, mpad, w);
      fin_launch(FIN_RUPDATE);
    }
  };

  k_lz_init_state<<<nblocks(nseg, 256), 256, 0, st>>>(a, miter_opt);
  RSB_LAUNCH_CHECK();
  k_lz_zero_small<<<nblocks(nseg, 256), 256, 0, st>>>(a, g->d_fied);
  RSB_LAUNCH_CHECK();
  if (ntiles == 0) {
    return 0;
  }
  // start vector of the segments in LZ_SETUP, normalised into f
  auto start = [&](int mode, const float *sv) -> int {
    a.mode = ai.mode = mode;
    for (int ph = 0; ph < 3; ph++) {
      k_lz_start<T><<<ntiles, RSB_BLOCK, 0, st>>>(a, ph, mode, sv, f);
      RSB_LAUNCH_CHECK();
      if (ph < 2) FIN(ph == 0 ? FIN_START0 : FIN_START1);
    }
    return 0;
  };
  // restarted CG-Lanczos passes of the segments in LZ_SETUP (f holds the
  // normalised start vector; SC_MEANF is 0 for the first pass)
  const size_t tq_lds =
      sizeof(double) * (2 * miter_max + miter_max * ((miter_max + RSB_WAVE - 1) / RSB_WAVE * RSB_WAVE));
  auto passes = [&](int np_max) -> int {
    a.mpass = ai.mpass = np_max;
    // r_0 into basis slot 0
    auto setup = [&]() -> int {
      k_lz_setup<T><<<ntiles, RSB_BLOCK, 0, st>>>(a, 0, f, basis, p);
      RSB_LAUNCH_CHECK();
      FIN(FIN_SETUP0);
      k_lz_setup<T><<<ntiles, RSB_BLOCK, 0, st>>>(a, 1, f, basis, p);
      RSB_LAUNCH_CHECK();
      FIN(FIN_SETUP1);
      return 0;
    };
    // a pass's lists are those of the segments in LZ_SETUP before its setup,
    // which is queued before their lengths are looked at (with no segment
    // left to restart its launches return at the status)
    if (compact_start(LZ_SETUP) || setup() || compact_take()) return 2;
    for (int pass = 0; pass < np_max; pass++) {
      fold = nact[0] <= fold_tiles;
      RSB_TRY(hipEventRecord(g->lz_ev0, st));
      int it, nrec = 0;
      hipGraphExec_t gexec = nullptr;
      int gn[2] = {-1, -1};
      if (g->prof_spmv && (int)g->spmv_ev.size() < 2 * miter_max) {
        size_t old = g->spmv_ev.size();
        g->spmv_ev.resize(2 * miter_max);
        for (size_t q = old; q < g->spmv_ev.size(); q++) RSB_TRY(hipEventCreate(&g->spmv_ev[q]));
      }
      // the running lists are compacted 8 iterations into the pass and then
      // at intervals that double (up to 32) while no segment has finished (a
      // finished segment's tiles only cost launches whose workgroups return
      // at once), and taken up LZ_AHEAD iterations later
      int next_c = 7, step = 8, take_at = -1;
      for (it = 0; it < miter_max; it++) {
        if (nact[0] == 0) break;
        if (use_graph && (it & 7) == 0 && it + 8 < miter_max) {
          // eight iterations as one graph replay (same kernels and grids as
          // the launches below; the grids follow the compacted lists, so
          // the chunk is captured again when they changed)
          if (!gexec || gn[0] != nact[0] || gn[1] != nact[1]) {
            hipGraph_t gr = nullptr;
            RSB_TRY(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
            // (it is a multiple of 8: the chunk's buffer parities are q's)
            for (int q = 0; q < 8; q++) {
              apply_launch(q);
              after_apply(q);
            }
            RSB_TRY(hipStreamEndCapture(st, &gr));
            if (gexec) RSB_TRY(hipGraphExecDestroy(gexec));
            gexec = nullptr;
            RSB_TRY(hipGraphInstantiateWithFlags(&gexec, gr, 0));
            RSB_TRY(hipGraphDestroy(gr));
            gn[0] = nact[0], gn[1] = nact[1];
          }
          RSB_TRY(hipGraphLaunch(gexec, st));
          g->lz_launches += 8;
          it += 7;
          if (it + 1 < miter_max) {
            if (compact_start(LZ_RUNNING) || compact_take()) return 2;
            if (nact[1] == 0) break;
          }
          continue;
        }
        // profiling: every LZ_PROF_EVERY-th launch is bracketed by events (each
        // pair of records costs several microseconds of stream time, so
        // timing every launch slowed the whole call by ~5%)
        const bool samp = g->prof_spmv && (g->spmv_total++ % LZ_PROF_EVERY) == 0;
        if (samp) RSB_TRY(hipEventRecord(g->spmv_ev[2 * nrec], st));
        apply_launch(it);
        if (samp) {
          RSB_TRY(hipEventRecord(g->spmv_ev[2 * nrec + 1], st));
          nrec++;
        }
        after_apply(it);
        RSB_LAUNCH_CHECK();
        g->lz_launches++;
        if (it == next_c && it + 1 + LZ_AHEAD < miter_max) {
          // drop segments that finished their pass from the launch lists
          if (compact_start(LZ_RUNNING)) return 2;
          take_at = it + LZ_AHEAD;
        }
        if (it == take_at) {
          const int before = nact[1];
          if (compact_take()) return 2;
          if (nact[1] == 0) break;
          step = nact[1] == before ? std::min(2 * step, 32) : 8;
          next_c += step;
        }
      }
      if (fuse && nact[1] > 0) {
        // the sums of the last iteration
        lz_args af;
        const lz_fuse fu = fused(miter_max, fold ? (miter_max + 1) & 1 : 1, af);
        if (fold) k_lz_last<true><<<nact[1], RSB_BLOCK, 0, st>>>(af, fu, act_s);
        else k_lz_last<false><<<nact[1], RSB_BLOCK, 0, st>>>(af, fu, act_s);
        RSB_LAUNCH_CHECK();
      }
      RSB_TRY(hipEventRecord(g->lz_ev1, st));
      if (long_pass) {
        // segments in chunks whose matrices take at most 1 GiB together
        const size_t zb = sizeof(double) * (size_t)miter_max * miter_max;
        const int chunk = (int)std::max<size_t>(1, std::min<size_t>(nseg, (1ull << 30) / zb));
        double *zbuf = nullptr;
        RSB_TRY(RSB_SCRATCH(zbuf, zb * (size_t)chunk));
        for (int s0 = 0; s0 < nseg; s0 += chunk) {
          k_lz_tqli_g<<<std::min(chunk, nseg - s0), RSB_WAVE, sizeof(double) * 2 * miter_max,
                        st>>>(a, s0, zbuf);
          RSB_LAUNCH_CHECK();
        }
      } else if (sizeof(T) == 4) {
        k_lz_eigmin<<<nseg, RSB_WAVE, sizeof(double) * 2 * miter_max, st>>>(a);
      } else {
        k_lz_tqli<<<nseg, 2 * RSB_WAVE, tq_lds, st>>>(a);
      }
      RSB_LAUNCH_CHECK();
      k_lz_ritz<T><<<ntiles, RSB_BLOCK, 0, st>>>(a, basis, mpad, f);
      RSB_LAUNCH_CHECK();
      FIN(FIN_RITZ);
      if (compact_start(LZ_SETUP)) return 2;
      if (pass + 1 < np_max && setup()) return 2;
      if (compact_take()) return 2;
      // the pass's events are complete now (one wait per pass end)
      if (gexec) RSB_TRY(hipGraphExecDestroy(gexec));
      float ms = 0.f;
      RSB_TRY(hipEventSynchronize(g->lz_ev1));
      RSB_TRY(hipEventElapsedTime(&ms, g->lz_ev0, g->lz_ev1));
      g->lz_ms += ms;
      for (int q = 0; q < nrec; q++) {
        RSB_TRY(hipEventElapsedTime(&ms, g->spmv_ev[2 * q], g->spmv_ev[2 * q + 1]));
        g->spmv_ms += ms;
      }
      g->spmv_launches += nrec;
      if (nact[1] == 0) break;
    }
    return 0;
  };
  int rc = 0;
  // learned start: nothing to do if no segment is within the size limit
  bool learned_any = false;
  if (init_mode == 2)
    for (int s = 0; s < nseg; s++)
      if (g->h_p[s] > 1 && g->h_n[s] >= 2 && (g->lws_max_n == 0 || g->h_n[s] <= g->lws_max_n))
        learned_any = true;
  if (init_mode == 2 && learned_any) {
    // learned start (per row, written into w, which the passes overwrite
    // only after the start has been normalised into f), then the fallback
    float *srow = (float *)w;
    if ((rc = rsb_lws_predict(g, g->lws_params, g->lws_level, srow))) return rc;
    if ((rc = start(2, srow)) || (rc = passes(std::min(g->lws_passes, mpass)))) return rc;
    RSB_TRY(hipMemsetAsync(L.count, 0, sizeof(int), st));
    k_lz_fallback<<<nblocks(nseg, 256), 256, 0, st>>>(a, L.count);
    RSB_LAUNCH_CHECK();
    int nfb = 0;
    RSB_READ(g, {&nfb, L.count, sizeof(int)});
    if (nfb > 0 && ((rc = start(0, nullptr)) || (rc = passes(mpass)))) return rc;
  } else {
    if ((rc = start(init_mode == 2 ? 0 : init_mode, g->d_start)) || (rc = passes(mpass)))
      return rc;
  }
  k_lz_finish<T><<<ntiles, RSB_BLOCK, 0, st>>>(a, 0, f, g->d_fied, xrow);
  RSB_LAUNCH_CHECK();
  FIN(FIN_FINISH);
  k_lz_finish<T><<<ntiles, RSB_BLOCK, 0, st>>>(a, 1, f, g->d_fied, xrow);
  RSB_LAUNCH_CHECK();
  if (out && out->resid) {
    k_lz_resid<<<ntiles, RSB_BLOCK, 0, st>>>(a, 0, xrow, g->d_slice_off, g->d_slice_w, g->d_ell);
    RSB_LAUNCH_CHECK();
    FIN(FIN_RES0);
    k_lz_resid<<<ntiles, RSB_BLOCK, 0, st>>>(a, 1, xrow, g->d_slice_off, g->d_slice_w, g->d_ell);
    RSB_LAUNCH_CHECK();
    FIN(FIN_RES1);
  }
  // read back per-segment results
  std::vector<int> ni(nseg), np(nseg);
  std::vector<double> sc((size_t)nseg * LZ_NSC);
  RSB_READ(g, {ni.data(), a.niter, sizeof(int) * nseg},
           {np.data(), a.npass, sizeof(int) * nseg},
           {sc.data(), a.sc, sizeof(double) * nseg * LZ_NSC});
  // Algorithmic bytes, per iteration and segment of n rows and nnz
  // off-diagonals: 4(n+1) row pointers + 4 nnz packed entries + 7 s n vector
  // streams for the whole iteration; for k_lz_apply alone 4(n+1) + 4 nnz +
  // 4 s n (p_old and r read once, p_new and w written; r stays in its basis
  // slot).  With the folded update the apply is the iteration: 6 s n (r, w
  // and p_old of the previous iteration read; r, p_new and w written).
  // Counted iterations, real (unpadded) sizes.
  for (int s = 0; s < nseg; s++) {
    const double *scs = &sc[(size_t)s * LZ_NSC];
    ni[s] += (int)scs[SC_WARMIT];
    if (g->h_p[s] > 1 && g->h_n[s] >= 2) {
      double n = g->h_n[s], nz = (double)g->h_seg_nnz[s], sz = sizeof(T);
      const double nf = scs[SC_NFOLD], nu = ni[s] - nf;
      g->lz_bytes += nu * (4 * (n + 1) + 4 * nz + 7 * sz * n) + nf * (4 * (n + 1) + 4 * nz + 6 * sz * n);
      g->spmv_bytes += nu * (4 * (n + 1) + 4 * nz + 4 * sz * n) + nf * (4 * (n + 1) + 4 * nz + 6 * sz * n);
    }
    if (out) {
      if (out->niter) out->niter[s] = ni[s];
      if (out->npass) out->npass[s] = np[s];
      if (out->lambda) out->lambda[s] = sc[(size_t)s * LZ_NSC + SC_LAMBDA];
      if (out->rnorm) {
        out->rnorm[3 * s] = sc[(size_t)s * LZ_NSC + SC_RNORM0];
        out->rnorm[3 * s + 1] = sc[(size_t)s * LZ_NSC + SC_RTOL];
        out->rnorm[3 * s + 2] = sc[(size_t)s * LZ_NSC + SC_RNORM];
      }
      if (out->resid) out->resid[s] = sc[(size_t)s * LZ_NSC + SC_TMP];
      if (out->fallback)
        out->fallback[s] = (init_mode == 2 && !learned_any && g->h_p[s] > 1 && g->h_n[s] >= 2) ||
                                   scs[SC_FALLBACK] < 0.0
                               ? -1
                           : scs[SC_FALLBACK] > 0.0 ? 1 + (int)scs[SC_WARMIT]
                                                    : 0;
    }
  }
  return 0;
}

extern "C" int rsbgpu_set_start(rsbgpu *g, const float *d_start) {
  RSB_TRY(hipSetDevice(g->device));
  RSB_TRY(dev_alloc(g, g->d_start, (size_t)g->nel));
  RSB_TRY(hipMemcpyAsync(g->d_start, d_start, sizeof(float) * (size_t)g->nel,
                         hipMemcpyDeviceToDevice, g->stream));
  return 0;
}

extern "C" int rsbgpu_fiedler(rsbgpu *g, int precision, int max_iter, int max_passes,
                              double tol, int init_mode, rsbgpu_fiedler_out *out) {
  RSB_TRY(hipSetDevice(g->device));
  if (max_iter < 1 || max_passes < 1) RSB_FAIL(3, "rsb_max_iter and rsb_max_passes must be >= 1");
  if (init_mode == 1 && !g->d_start) RSB_FAIL(3, "no start vector set");
  if (init_mode == 2 && !g->lws_params) RSB_FAIL(3, "no warm-start parameters set");
  if (init_mode < 0 || init_mode > 2) RSB_FAIL(3, "unknown init_mode %d", init_mode);
  rsb_phase_begin(g);
  int rc;
  if (precision == 32) rc = run_lanczos<float>(g, max_iter, max_passes, tol, init_mode, out);
  else rc = run_lanczos<double>(g, max_iter, max_passes, tol, init_mode, out);
  rsb_phase_end(g, PH_LANCZOS);
  return rc;
}

static int rsb_test_tridiag(const double *d, const double *e, int n, double *y, double *lam,
                            int fast);

extern "C" int rsbgpu_test_tqli(const double *d, const double *e, int n, double *y,
                                double *lam) {
  return rsb_test_tridiag(d, e, n, y, lam, 0);
}

extern "C" int rsbgpu_test_eigmin(const double *d, const double *e, int n, double *y,
                                  double *lam) {
  return rsb_test_tridiag(d, e, n, y, lam, 1);
}

static int rsb_test_tridiag(const double *d, const double *e, int n, double *y, double *lam,
                            int fast) {
  double *dd = nullptr, *de = nullptr, *dy = nullptr, *dl = nullptr, *dz = nullptr;
  if (n < 1 || n > 4096 || (fast && n > 128)) return 3;
  hipError_t err = rsb_dev_malloc((void **)&dd, sizeof(double) * n);
  if (err == hipSuccess) err = rsb_dev_malloc((void **)&de, sizeof(double) * n);
  if (err == hipSuccess) err = rsb_dev_malloc((void **)&dy, sizeof(double) * n);
  if (err == hipSuccess) err = rsb_dev_malloc((void **)&dl, sizeof(double));
  if (err == hipSuccess) err = hipMemcpy(dd, d, sizeof(double) * n, hipMemcpyHostToDevice);
  if (err == hipSuccess) err = hipMemset(de, 0, sizeof(double) * n);
  if (err == hipSuccess && n > 1)
    err = hipMemcpy(de, e, sizeof(double) * (n - 1), hipMemcpyHostToDevice);
  if (err == hipSuccess) {
    if (fast) {
      k_eigmin_test<<<1, RSB_WAVE, sizeof(double) * 2 * n, 0>>>(n, dd, de, dy, dl);
    } else if (n > 128) {
      err = rsb_dev_malloc((void **)&dz, sizeof(double) * (size_t)n * n);
      if (err == hipSuccess)
        k_tqli_test_g<<<1, RSB_WAVE, sizeof(double) * 2 * n, 0>>>(n, dd, de, dy, dl, dz);
    } else {
      size_t lds = sizeof(double) * (2 * n + n * ((n + RSB_WAVE - 1) / RSB_WAVE * RSB_WAVE));
      k_tqli_test<<<1, 2 * RSB_WAVE, lds, 0>>>(n, dd, de, dy, dl);
    }
    err = hipGetLastError();
  }
  if (err == hipSuccess) err = hipDeviceSynchronize();
  if (err == hipSuccess) err = hipMemcpy(y, dy, sizeof(double) * n, hipMemcpyDeviceToHost);
  if (err == hipSuccess) err = hipMemcpy(lam, dl, sizeof(double), hipMemcpyDeviceToHost);
  if (dd) (void)rsb_dev_free(dd);
  if (de) (void)rsb_dev_free(de);
  if (dy) (void)rsb_dev_free(dy);
  if (dl) (void)rsb_dev_free(dl);
  if (dz) (void)rsb_dev_free(dz);
  return err == hipSuccess ? 0 : 2;
}
