// l2c_fmm.hip -- FMM execute kernels for gfx950 (src/C/leg2cheb.c:1299-1500
// and the near field :236-535), plus the direct O(N^2) kernel (:152-234).
//
// One transform (or one line of a batch) is three launches, both parities in
// every work-group:
//
//   k_up    leaf moments (step 1) on FP64 MFMA and the upward pass (step 2)
//           inside a subtree of 2^gu <= 16 leaf chunks; writes the multipole
//           store for levels >= lu and, for each level l < lu, the subtree
//           root's contribution P(lu-l, .) w_root to its level-l ancestor.  At
//           rank 18 and s <= 64 other work-groups of the same launch do the
//           near field (band_group, FP64 VALU): the raw band sums go to the
//           output, or to the workspace where the output is strided.
//   k_m2l   M2L (step 3) of every block of every level, streaming the M2L
//           matrices (k_m2l_t: block rows in registers, k_m2l: through LDS,
//           k_m2l_mma: FP64 MFMA for many lines; each matrix read once for both
//           parities); blocks above lu first sum the k_up contributions into
//           their multipoles.  HBM-bound.
//   k_far   per subtree of 2^gd leaf chunks: L2L (step 4) down the ancestor
//           chain and the subtree, leaf evaluation (step 5) on FP64 MFMA, added
//           to the band sums, final scaling, one store of the output (which is
//           overwritten, not accumulated).
//
// Other ranks and s > 64: k_up_any, and k_down8r, k_down8 or k_down, which do the
// near field and k_far's work in one launch.
//
// Workspace per line: [multipoles: slot_base(L) x 2M][contributions:
// lu x 2^(lu+2) x 2M][M2L results: slot_base(L) x 2M]; chunk slot
// slot_base(l) + r holds [parity][M].
//
// Kernels are templated on the rank M (MT = M compiled in so that the
// M-loops unroll; MT = 0 reads M at run time).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>

#include "l2c_internal.h"

namespace l2c {

constexpr double kSqrtPi = 1.77245385090551602729816748334;
constexpr double k2Pi = 0.63661977236758134307553505349;  // 2/pi

typedef double d4 __attribute__((ext_vector_type(4)));

// two doubles at any 8-byte boundary, moved as one 16-byte access
typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));
// Buffer descriptor of n doubles at p (both wave-uniform): raw buffer loads
// check each dword against the length and return zero past it.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t line_rsrc(const double *p, int n) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(p), 0, 8 * n, 0x00020000);
}
__device__ __forceinline__ double load_one(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
// The two doubles at byte voff (per lane) + soff (uniform) of the buffer.
__device__ __forceinline__ d2 load_pair(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  const u4 v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
  return __builtin_bit_cast(d2, v);
}

__device__ __forceinline__ void store_pair(d2 v, __amdgpu_buffer_rsrc_t r, int voff) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), r, voff, 0, 0);
}

// How a call's work-groups take its lines, and where the band sums wait for the far
// field: LINES_PLAIN line by line, over the output; LINES_FLAT the same without empty
// groups (k_up); LINES_ACROSS group by group over lines that lie side by side (place);
// LINES_RAW line by line, back to back in the workspace (raw_sums).
enum { LINES_PLAIN = 0, LINES_FLAT = 1, LINES_ACROSS = 2, LINES_RAW = 3 };

// The (group, line) of work-group id of n groups of each of nl lines.  In general
// the groups of a line follow each other.  ACROSS, lines that lie side by side: an HBM
// or L2 line holds one element of each of 8 or 16 of them, so the work-groups of one
// group of all lines run one after the other on one XCD (work-groups go to the eight
// XCDs in turn), each fetching and writing what its neighbours' elements share with
// its own while that is in the XCD's L2.
struct Place {
  unsigned grp, line;
};
template <bool ACROSS>
__device__ __forceinline__ Place place_of(unsigned id, unsigned n, unsigned nl) {
  if (!ACROSS) return {id % n, id / n};
  n *= nl;
  const unsigned t = (id & 7) * (n >> 3) + std::min(id & 7, n & 7) + (id >> 3);
  return {t / nl, t % nl};
}
// that of this work-group in a launch of grid (groups, lines)
template <bool ACROSS>
__device__ __forceinline__ Place place() {
  if (!ACROSS) return {blockIdx.x, blockIdx.y};
  return place_of<true>(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x, gridDim.y);
}

struct WsLayout {
  size_t w, part, m2l, total;
};
__host__ __device__ inline WsLayout ws_layout(const Geo &g) {
  const size_t M2 = 2 * (size_t)g.M;
  WsLayout l;
  l.w = 0;
  l.part = slot_base(g.L) * M2;
  l.m2l = l.part + (size_t)g.lu * ((size_t)4 << g.lu) * M2;
  l.total = l.m2l + slot_base(g.L) * M2;
  return l;
}
size_t ws_doubles(const Geo &g) { return ws_layout(g).total; }

// skewed LDS indices: one pad double every 4 (input) or 8 (Lambda window)
// so that lanes 4 (input) or 8 (Lambda) doubles apart hit distinct banks
__host__ __device__ __forceinline__ int sk4(int c) { return c + (c >> 2); }
__host__ __device__ __forceinline__ int sk8(int k) { return k + (k >> 3); }


// ---------------------------------------------------------------------------
// The near-field band (src/C/leg2cheb.c:236-535) of G = 16 (or 8) leaf chunks, any
// leaf size s <= 64, by the 256 threads of a work-group: rows r of parity sg take
// the columns c = r + t, t < len (2 s - 16 gam for row group gam, shorter in
// the last chunk), y_r = sum H(t - rho) P(2 r0 + sg + t + rho) x(r0 + t).
// Each lane owns 16 rows of one chunk and parity: lane = chunk + G parity + 2 G
// del, row group gam = del, or (G = 16, more than two row groups) 2 p + del; the
// waves split (p, columns).  All lanes of a wave sit at the same t, so H is
// wave-uniform: scalar loads, which the products take as operands; P runs
// through a ring of 16 registers.  Per column a lane reads one x and one P from
// LDS for 16 terms (one multiply and one FMA each), four columns ahead.
//   x, per parity, half index h from the first chunk: h + h / s when 4
//     divides s (one pad per chunk), else h; parity 1 at +nxs, nxs odd when
//     s = 2 mod 4, else G mod 32
//   P, entry m from the first row: m + 2 (m / 2s) for even s (every 2s
//     entries are followed by a copy of the next two), else m
// so that the 32 lanes of half a wave read distinct banks (G = 8: pairs of lanes
// share one of P's), and a lane's four entries are always consecutive (it meets
// a chunk's end only between them, S16: s a multiple of 16, only between trips
// of 16).
// Bound by FP64 issue on large calls (4.6 M vector instructions at N = 2^20,
// s = 64, three quarters of them the products), on one small line by the
// work-group's own chain (window loads 2 us, its trips 1 us each, staging).
// As k_band alone, s = 64: 2^16 10.0 us, 2^20 17.3, 64 lines of 2^18 165; with
// 8 rows a lane, H from LDS and a Lambda window per chunk, s = 16, 32, 64 only,
// 11.3, 18.6 and 212.
constexpr int kBandNT = 256, kBandMaxS = 64;
struct BandLds {
  int nx, pad, nxs, np, pw, PS, CS, total;
};
__host__ __device__ inline BandLds band_lds(const Geo &g, int G) {
  const int s = g.s;
  BandLds d;
  // half indices per parity: the last chunk's columns, to the end of its trips
  // (G = 8: a wave's trips are those of its longest row group)
  d.nx = (G + 1) * s + (G == 8 ? 80 : 32);
  d.pad = (s & 3) == 0;
  const int n = d.nx + (d.pad ? d.nx / s + 1 : 0);
  d.nxs = (s & 3) == 2 ? n | 1 : n + (32 + G - n % 32) % 32;  // G mod 32
  d.pw = 2 * d.nxs;
  d.pw += d.pw & 1;  // 16-byte rows
  d.np = 2 * G * s + (G == 8 ? std::max(s + 64, 148) : s + 64);
  d.np += d.np & 1;
  d.PS = 2 * s + ((s & 1) ? 0 : 2);
  // staging of the sums, [segment][chunk][CS], over the windows
  d.CS = d.PS;
  const int npair = G == 8 ? 1 : (s + 31) / 32;
  // (the unused prefetch behind a last trip may pass the windows' ends)
  d.total = std::max(d.pw + d.np + ((s & 1) ? 0 : 2 * (d.np / (2 * s) + 1)) + 32,
                     (kBandNT / 64 / npair) * G * d.CS);
  return d;
}
inline size_t band_shared_bytes(const Geo &g, int G) { return 8 * (size_t)band_lds(g, G).total; }
inline unsigned band_groups(const Geo &g, int G) {  // work-groups of one line
  return (unsigned)((((size_t)2 << g.L) + G - 1) / G);
}

typedef const __attribute__((address_space(4))) double *kdouble;  // uniform, read-only

// A lane's read pointers into the windows: the next quad of x and of P, and
// the columns to the next chunk end of each (a pad of px or pp doubles then).
struct BandPtr {
  const double *x, *p;
  int lx, lp;
};
constexpr int kBT = 2;  // products in flight before their sums
// One trip of 16 columns from column tb on; X, P of the trip's first quad are
// in XA, PA, and on return those of the next trip's.  The trip's 31 values of
// H are scalar loads (hp: the head, 16 zeros before it), the last eight half a trip
// after the others: all 31 from the start on spilled scalars to scratch in k_up.  KIND 0: as it is; 1:
// columns t >= len read x as zero; 2: that, and the terms left of the diagonal
// (rho > t) are left out, for the trip from column 0.
template <int KIND, bool S16>
__device__ __forceinline__ void band_trip(BandPtr &b, int s1, int s2, kdouble hp, int tb, int len,
                                          double (&pr)[16], double (&XA)[4], double (&PA)[4],
                                          double (&acc)[16]) {
  double XB[4], PB[4], hw[32];
#pragma unroll
  for (int k = 1; k < 24; k++) hw[k] = hp[tb - 16 + k];
  // x of the quad after the current one, P 16 further on
#define QUAD_FETCH(X, P, Q)                                      \
  {                                                              \
    if (!S16 || (Q) == 3) {                                      \
      b.lx -= S16 ? 16 : 4;                                      \
      b.lp -= S16 ? 16 : 4;                                      \
      const bool ox_ = b.lx == 0, op_ = b.lp == 0;               \
      b.x += ox_ ? 5 : 4;                                        \
      b.p += op_ ? 6 : 4;                                        \
      b.lx = ox_ ? s1 : b.lx;                                    \
      b.lp = op_ ? s2 : b.lp;                                    \
    } else {                                                     \
      b.x += 4;                                                  \
      b.p += 4;                                                  \
    }                                                            \
    _Pragma("unroll") for (int k_ = 0; k_ < 4; k_++) {           \
      X[k_] = b.x[k_];                                           \
      P[k_] = b.p[k_];                                           \
    }                                                            \
  }
#define QUAD_STEP(X, P, Q)                                                          \
  _Pragma("unroll") for (int j_ = 0; j_ < 4; j_++) {                                \
    const int k_ = 4 * (Q) + j_;                                                    \
    const double x_ = KIND != 0 ? (tb + k_ < len ? X[j_] : 0.0) : X[j_];            \
    _Pragma("unroll") for (int q_ = 0; q_ < 16 / kBT; q_++) {                       \
      double t_[kBT];                                                               \
      _Pragma("unroll") for (int i_ = 0; i_ < kBT; i_++) {                          \
        const int r_ = kBT * q_ + i_;                                               \
        t_[i_] = KIND != 2 || r_ <= k_ ? hw[16 + k_ - r_] * pr[(k_ + r_) & 15] : 0.0; \
      }                                                                             \
      __builtin_amdgcn_sched_barrier(0);                                            \
      _Pragma("unroll") for (int i_ = 0; i_ < kBT; i_++) {                          \
        const int r_ = kBT * q_ + i_;                                               \
        if (KIND != 2 || r_ <= k_) acc[r_] += t_[i_] * x_;                          \
      }                                                                             \
    }                                                                               \
    pr[k_] = P[j_];                                                                 \
    __builtin_amdgcn_sched_barrier(0);                                              \
  }
  QUAD_FETCH(XB, PB, 0)
  QUAD_STEP(XA, PA, 0)
  QUAD_FETCH(XA, PA, 1)
  {
    int t8 = tb + 8;
    asm volatile("" : "+s"(t8));
#pragma unroll
    for (int k = 0; k < 8; k++) hw[24 + k] = hp[t8 + k];
  }
  QUAD_STEP(XB, PB, 1)
  QUAD_FETCH(XB, PB, 2)
  QUAD_STEP(XA, PA, 2)
  QUAD_FETCH(XA, PA, 3)
  QUAD_STEP(XB, PB, 3)
#undef QUAD_STEP
#undef QUAD_FETCH
}

// Band group grp of the line at src (element stride es, length Nl): the sums
// go to dst (element stride ds), raw (the C2L diagonal included), or with
// the final scaling when scale != 0.
template <bool S16, int G>
__device__ __forceinline__ void band_group(const double *__restrict__ src, size_t es,
                                           double *__restrict__ dst, size_t ds, int Nl,
                                           const Geo &g, int dir, int grp, int scale,
                                           const double *__restrict__ tab,
                                           const double *__restrict__ head, double *sm) {
  const int s = g.s, N = g.N;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const size_t hc0 = (size_t)grp * G * s, row0 = 2 * hc0;
  if (row0 >= (size_t)Nl) return;  // the whole work-group
  const BandLds ly = band_lds(g, G);
  double *xs = sm, *pw = sm + ly.pw;
  const unsigned inv = ((1u << 20) + s - 1) / s;  // h / s = h inv >> 20 for h < 2200
  auto chunk = [&](int h) { return (int)(__umul24(h, inv) >> 20); };
  const bool even = (s & 1) == 0;
  // ---- windows: pairs of P, pairs (2 h, 2 h + 1) of x; past the table's and
  // the line's ends zeros
  constexpr int QX = G == 8 ? 3 : 5;  // ceil(nx / 256), ceil(np / 512) for s = 64
  d2 vp[QX], vx[QX];
  {
    const __amdgpu_buffer_rsrc_t r =
        line_rsrc(tab + row0, (int)std::min<size_t>((size_t)N - row0, ly.np));
#pragma unroll
    for (int q = 0; q < QX; q++) vp[q] = load_pair(r, 16 * tid + 4096 * q, 0);
  }
  if (es == 1) {
    const __amdgpu_buffer_rsrc_t r =
        line_rsrc(src + row0, (int)std::min<size_t>((size_t)Nl - row0, 2 * ly.nx));
#pragma unroll
    for (int q = 0; q < QX; q++) vx[q] = load_pair(r, 16 * tid + 4096 * q, 0);
  } else {
#pragma unroll
    for (int q = 0; q < QX; q++) {
      const size_t i = row0 + 2 * (size_t)(tid + kBandNT * q);
      vx[q].x = src[std::min(i, (size_t)Nl - 1) * es];
      vx[q].y = src[std::min(i + 1, (size_t)Nl - 1) * es];
      if (i >= (size_t)Nl) vx[q].x = 0.0;
      if (i + 1 >= (size_t)Nl) vx[q].y = 0.0;
    }
  }
#pragma unroll
  for (int q = 0; q < QX; q++) {
    const int h = tid + kBandNT * q, c = chunk(h);
    if (2 * h < ly.np) {
      const int a = 2 * h + (even ? 2 * c : 0);
      *reinterpret_cast<d2 *>(pw + a) = vp[q];
      if (even && h == c * s && c > 0) *reinterpret_cast<d2 *>(pw + a - 2) = vp[q];
    }
  }
#pragma unroll
  for (int q = 0; q < QX; q++) {
    const int h = tid + kBandNT * q;
    if (h < ly.nx) {
      const int a = h + (ly.pad ? chunk(h) : 0);
      double x0 = vx[q].x, x1 = vx[q].y;
      if (dir == C2L) {  // v_i = i u_i, v_0 = u_0
        const double i = (double)(row0 + 2 * h);
        x0 *= i == 0.0 ? 1.0 : i;
        x1 *= i + 1.0;
      }
      xs[a] = x0;
      xs[ly.nxs + a] = x1;
    }
  }
  lds_sync();

  // ---- the band
  const int ng = (s + 15) >> 4, npair = G == 8 ? 1 : (ng + 1) >> 1;
  const int lseg = npair == 1 ? 2 : 1, nseg = 1 << lseg;
  const int p = npair == 1 ? 0 : wave & 1, seg = npair == 1 ? wave : wave >> 1;
  double acc[16];
#pragma unroll
  for (int k = 0; k < 16; k++) acc[k] = 0.0;
  {
    const int gl = lane & (G - 1), sg = lane / G & 1, gam = 2 * p + lane / (2 * G);
    const size_t beta = (size_t)grp * G + gl, nLm1 = (size_t)g.nL - 1;
    const size_t r0 = beta * s + 16 * gam, cnt = (N - sg + 1) / 2;
    const size_t cend = beta < nLm1 ? (beta + 2) * s : cnt;
    const int len = 16 * gam < s && r0 < cnt ? (int)(cend - r0) : 0;
    const int T = (2 * s - 32 * p + 15) >> 4;  // trips of the pair's longer group
    const int t0 = 16 * (T * seg >> lseg), t1 = 16 * (T * (seg + 1) >> lseg);
    // columns that every live row of the wave has (none where the chunks'
    // ends differ)
    const bool last = ((size_t)grp + 1) * G > nLm1;
    const int common = last ? 0 : 2 * s - 16 * std::min(G == 8 ? 3 : 2 * p + 1, ng - 1);
    kdouble hp = (kdouble)head;
    double pr[16], XA[4], PA[4];
    const int s1 = ly.pad ? s : 1 << 20, s2 = even ? 2 * s : 1 << 20;
    const int hq = gl * s + 16 * gam + t0, cx = chunk(hq);
    BandPtr b;
    b.x = xs + sg * ly.nxs + hq + (ly.pad ? cx : 0);
    b.lx = ly.pad ? s * (cx + 1) - hq : 1 << 20;
    // entry m = 2 h0 + t + sg of P at column t; its first 16, then the quad after
#pragma unroll
    for (int q = 0; q < 5; q++) {
      const int m = 2 * hq - t0 + 4 * q, c = chunk(m >> 1);
      const double *pm = pw + sg + m + (even ? 2 * c : 0);
#pragma unroll
      for (int k = 0; k < 4; k++) (q < 4 ? pr[4 * q + k] : PA[k]) = pm[k];
      b.p = pm;
      b.lp = even ? 2 * s * (c + 1) - m : 1 << 20;
    }
#pragma unroll
    for (int k = 0; k < 4; k++) XA[k] = b.x[k];
    int tb = t0;
    if (tb == 0 && tb < t1) {
      band_trip<2, S16>(b, s1, s2, hp, tb, len, pr, XA, PA, acc);
      tb = 16;
    }
    for (; tb < t1 && tb + 16 <= common; tb += 16)
      band_trip<0, S16>(b, s1, s2, hp, tb, len, pr, XA, PA, acc);
    for (; tb < t1; tb += 16) band_trip<1, S16>(b, s1, s2, hp, tb, len, pr, XA, PA, acc);
  }
  // the lane's rows again, from a fresh copy of its index (the empty asm hides
  // that it is the one used above, so nothing is held through the trips)
  int ln = lane;
  asm volatile("" : "+v"(ln));
  const int gl = ln & (G - 1), sg = ln / G & 1, gam = 2 * p + ln / (2 * G);
  if (dir == C2L) {
    // less the sum; the C2L diagonal sqrt(pi) an_i v_i (src/C/leg2cheb.c:416)
    const int h0 = gl * s + 16 * gam;
#pragma unroll
    for (int k = 0; k < 16; k++) {
      const int h = h0 + k, c = chunk(h);
      const double d = kSqrtPi * xs[sg * ly.nxs + h + (ly.pad ? c : 0)] *
                       pw[sg + 2 * h + (even ? 2 * c : 0)];
      acc[k] = (seg == 0 ? d : 0.0) - acc[k];
    }
  }
  const bool live = ((size_t)grp * G + gl) * s + 16 * gam < (size_t)(N - sg + 1) / 2;
  lds_sync();  // windows dead: the staging takes their place
  if (live) {
    double *o = sm + (seg * G + gl) * ly.CS + 32 * gam + sg;
#pragma unroll
    for (int k = 0; k < 16; k++)
      if (16 * gam + k < s) o[2 * k] = acc[k];
  }
  lds_sync();
  // ---- the segments' sums, stored
  const int nr = (int)std::min<size_t>((size_t)G * 2 * s, (size_t)Nl - row0);
  auto value = [&](int e) {
    const double *o = sm + e + (even ? 2 * chunk(e >> 1) : 0);
    double v = o[0] + o[G * ly.CS];
    if (nseg == 4) v += o[2 * G * ly.CS] + o[3 * G * ly.CS];
    if (scale) {
      const size_t i = row0 + e;
      if (dir == L2C) {
        v *= k2Pi;
        if (i == 0) v *= 0.5;
      } else {
        v *= (double)i + 0.5;
      }
    }
    return v;
  };
  if (ds == 1) {
    const __amdgpu_buffer_rsrc_t r = line_rsrc(dst + row0, nr);
    for (int e = 2 * tid; e < nr; e += 2 * kBandNT) {
      const d2 v = {value(e), e + 1 < nr ? value(e + 1) : 0.0};
      store_pair(v, r, 8 * e);
    }
  } else {
    for (int e = tid; e < nr; e += kBandNT) dst[(row0 + e) * ds] = value(e);
  }
}

// ---------------------------------------------------------------------------
// k_up_any: the upward pass for ranks other than 18 and leaf sizes above 64.  Grid
// (2^(lu+2), lines), 256 threads.  G = 2^gu <= 16 leaf chunks.
//
// Leaf moments W_par (G x M) = X_par (G x s) T_par (s x M) run on
// v_mfma_f64_16x16x4f64 (A operand: lane l holds A[l%16][l/16]; B: lane l
// holds B[l/16][l%16]; D: lane l, register v holds D[l/16 + 4v][l%16]).
// One wave per (parity, 16-column tile of M).
constexpr int kUpNT = 256;

__host__ __device__ inline int up_xstride(int s) { return s | 1; }  // odd: conflict-free rows
// LDS: input [2][16][xst], moments [16][2][M], parents [8+1][2][M], the
// upward operators U(0), U(1) with rows padded to M+1 (the composite
// operators P are read from L2 by the threads that apply them)
size_t up_shared_bytes(const Geo &g) {
  const size_t M2 = 2 * g.M, Mp = g.M + 1;
  return 8 * (2 * 16 * (size_t)up_xstride(g.s) + 16 * M2 + 9 * M2 + 2 * (size_t)g.M * Mp);
}

// LM: the subtree levels on MFMA (MT > 0; chosen for subtrees of 2^3 and
// 2^4 leaf chunks in calls of up to 8 lines) or on VALU: 2 lines of 70,000 (s = 137)
// 71.3 us against 72.5, 4 of 2^20 (s = 128) 288 against 291, single ones even.  (Its body
// in a function of its own that the kernel calls: four registers spilled to a scratch
// frame, 700,000 (s = 86) 69.2 us against 68.2.)
template <int MT, bool LM>
__global__ void __launch_bounds__(kUpNT) __attribute__((amdgpu_waves_per_eu(4))) k_up_any(
    const double *__restrict__ in, LineMap lm, Geo g, int dir, const double *__restrict__ T,
    const double *__restrict__ U, const double *__restrict__ P, double *__restrict__ wsall,
    size_t wsstride) {
  extern __shared__ double sm[];
  const int M = MT > 0 ? MT : g.M;
  const int s = g.s, L = g.L, M2 = 2 * M, MM = M * M;
  const int G = 1 << g.gu;
  const int j = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const double *src = in + line_off(lm, blockIdx.y);
  const size_t Nl = (size_t)line_len(lm, blockIdx.y, g.N);  // zeros past the line's end
  double *ws = wsall + blockIdx.y * wsstride;
  const WsLayout lay = ws_layout(g);
  double *w = ws + lay.w;
  double *part = ws + lay.part;
  const int xst = up_xstride(s);
  const int Mp = M + 1;
  double *xs = sm;                  // [2][16][xst]
  double *w0 = xs + 2 * 16 * xst;   // [16][2][M]
  double *w1 = w0 + 16 * M2;        // [8+1][2][M]
  double *Ul = w1 + 9 * M2;         // [2][M][M+1]: U(0), U(1)

  // ---- loads, all issued before any use: input, this thread's rows of the
  // upward operators (k = tid % M) and of its composite operator P
  const int nin = G * 2 * s;
  const size_t base = (size_t)j * G * 2 * s;
  double vin[8];
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const int e = q * kUpNT + tid;
    const size_t i = base + e;
    vin[q] = (e < nin && i < Nl) ? src[i * lm.es] : 0.0;
  }
  // B operand of this wave's first MFMA task (16 k-steps = the first 64 rows of T)
  const int ntile = (M + 15) / 16;
  constexpr int QT = 16;
  double tb[QT];
  {
    const int sg = wave / ntile, nt = wave % ntile;
    const int kb = nt * 16 + (lane & 15), ka = lane >> 4;
    const double *tcol = T + (size_t)sg * s * M + kb;
#pragma unroll
    for (int q = 0; q < QT; q++) {
      const int m = 4 * q + ka;
      tb[q] = (wave < 2 * ntile && m < s && kb < M) ? tcol[(size_t)m * M] : 0.0;
    }
  }
  const int ku = tid % M;
  const int np = g.lu * M2;
  // A operand of the upward levels on MFMA (LM): rows rt*16 + (lane %
  // 16) of [U(0) U(1)] (M x 2M), k-steps kk (columns 4 kk + lane / 16), for
  // waves rt < ntile; loaded from HBM with the input, used from registers
  constexpr int QA = LM ? (2 * MT + 3) / 4 : 1;
  double ua[QA];
  if constexpr (LM) {
    const int ra = wave * 16 + (lane & 15);
#pragma unroll
    for (int kk = 0; kk < QA; kk++) {
      const int k = 4 * kk + (lane >> 4);
      const int pu = k < M ? 0 : 1, kc = k - pu * M;
      ua[kk] = (wave < ntile && ra < M && k < M2) ? U[(size_t)pu * MM + (size_t)ra * M + kc] : 0.0;
    }
  }
  // U(0), U(1) in LDS for the VALU levels (M without a compiled kernel),
  // once per work-group; every load of the batch is in flight before the
  // first LDS store
  if constexpr (!LM) {
    const int nop = 2 * MM;
    constexpr int QO = 3;
    double vo[QO];
#pragma unroll
    for (int q = 0; q < QO; q++) {
      const int e = q * kUpNT + tid;
      vo[q] = e < nop ? U[e] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < QO; q++) {
      const int e = q * kUpNT + tid;
      if (e < nop) Ul[(e / M) * Mp + e % M] = vo[q];
    }
    for (int e = QO * kUpNT + tid; e < nop; e += kUpNT) Ul[(e / M) * Mp + e % M] = U[e];
  }
  for (int e0 = 8 * kUpNT; e0 < nin; e0 += kUpNT) {  // rare: G*2s > 2048
    const int e = e0 + tid;
    if (e < nin) {
      const size_t i = base + e;
      const double v = i < Nl ? src[i * lm.es] : 0.0;
      xs[(e & 1) * 16 * xst + (e >> 1) / s * xst + (e >> 1) % s] =
          (dir == C2L && i > 0) ? v * (double)i : v;
    }
  }
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const int e = q * kUpNT + tid;
    if (e < nin) {
      const size_t i = base + e;
      const int h = e >> 1;  // half index inside the subtree
      // v_i = i u_i for C2L (src/C/leg2cheb.c:1325-1335)
      xs[(e & 1) * 16 * xst + (h / s) * xst + (h % s)] =
          (dir == C2L && i > 0) ? vin[q] * (double)i : vin[q];
    }
  }
  // rows G..15 of the MFMA A operand are zero
  for (int e = tid; e < 2 * (16 - G) * xst; e += kUpNT) {
    const int par = e / ((16 - G) * xst), rem = e % ((16 - G) * xst);
    xs[par * 16 * xst + G * xst + rem] = 0.0;
  }
  __syncthreads();

  // ---- step 1 on MFMA: W_par[i][k] = sum_m X_par[i][m] T_par[m][k]
  for (int task = wave; task < 2 * ntile; task += kUpNT / 64) {
    const int sg = task / ntile, nt = task % ntile;
    const int ia = lane & 15, ka = lane >> 4;  // A: row i, k-offset
    const int kb = nt * 16 + (lane & 15);      // B: column k
    const double *xrow = xs + sg * 16 * xst + ia * xst;
    const double *tcol = T + (size_t)sg * s * M + kb;
    d4 acc = {0, 0, 0, 0};
    int m0 = 0;
    if (task == wave) {  // B prefetched for rows < 64; two independent chains
      d4 acc1 = {0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < QT; q += 2) {
        const int m = 4 * q + ka;
        const double a0 = m < s ? xrow[m] : 0.0, a1 = m + 4 < s ? xrow[m + 4] : 0.0;
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, tb[q], acc, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, tb[q + 1], acc1, 0, 0, 0);
      }
      acc += acc1;
      m0 = 4 * QT;
    }
    for (; m0 < s; m0 += 4) {
      const int m = m0 + ka;
      const double a = m < s ? xrow[m] : 0.0;
      const double b = (m < s && kb < M) ? tcol[(size_t)m * M] : 0.0;
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int i = (lane >> 4) + 4 * v;
      if (i < G && kb < M) {
        w0[(i * 2 + sg) * M + kb] = acc[v];
        w[(slot_base(L - 1) + (size_t)j * G + i) * M2 + sg * M + kb] = acc[v];
      }
    }
  }
  __syncthreads();

  // ---- step 2: parent = U0 child0 + U1 child1 inside the subtree.  LM:
  // on v_mfma_f64_16x16x4f64, parents (M x 2n) = [U0 U1] (M x 2M) times the
  // children stacked (2M x 2n), column jc = 2c + parity for parent c (2n <=
  // 16); wave rt < ntile computes row tile rt in two chains of k-steps.
  // Else on VALU, thread (k = tid % M) reading its operator rows from LDS.
  const int npair = kUpNT / M;  // (chunk, parity) pairs handled per sweep
  int n = G;
  if constexpr (LM) {
    const int jc = lane & 15, cc = jc >> 1, sgc = jc & 1;
    for (int lev = L - 2; lev >= g.lu; lev--) {
      n >>= 1;
      if (wave < ntile) {
        d4 D0 = {0, 0, 0, 0}, D1 = {0, 0, 0, 0};
        double bv[QA];
#pragma unroll
        for (int kk = 0; kk < QA; kk++) {
          const int k = 4 * kk + (lane >> 4);
          const int pu = k < M ? 0 : 1, kc = k - pu * M;
          bv[kk] = (jc < 2 * n && k < M2) ? w0[((2 * cc + pu) * 2 + sgc) * M + kc] : 0.0;
        }
#pragma unroll
        for (int kk = 0; kk < QA; kk += 2) {
          D0 = __builtin_amdgcn_mfma_f64_16x16x4f64(ua[kk], bv[kk], D0, 0, 0, 0);
          if (kk + 1 < QA) D1 = __builtin_amdgcn_mfma_f64_16x16x4f64(ua[kk + 1], bv[kk + 1], D1, 0, 0, 0);
        }
        D0 += D1;
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int i = wave * 16 + (lane >> 4) + 4 * v;
          if (i < M && jc < 2 * n) {
            w1[(cc * 2 + sgc) * M + i] = D0[v];
            w[(slot_base(lev) + (size_t)j * n + cc) * M2 + sgc * M + i] = D0[v];
          }
        }
      }
      __syncthreads();
      double *tmp = w0;
      w0 = w1;
      w1 = tmp;
    }
  }
  for (int lev = L - 2; !LM && lev >= g.lu; lev--) {
    n >>= 1;
    if (tid < npair * M) {
      for (int cs = tid / M; cs < 2 * n; cs += npair) {
        const int c = cs >> 1, sg = cs & 1;
        const double *x0 = w0 + (2 * c * 2 + sg) * M;
        const double *x1 = w0 + ((2 * c + 1) * 2 + sg) * M;
        const double *u0 = Ul + ku * Mp, *u1 = Ul + (M + ku) * Mp;
        double a0 = 0, a1 = 0, a2 = 0, a3 = 0;
        if constexpr (MT > 0) {
#pragma unroll
          for (int l = 0; l < MT; l += 2) {
            a0 += u0[l] * x0[l];
            a1 += u1[l] * x1[l];
            if (l + 1 < MT) {
              a2 += u0[l + 1] * x0[l + 1];
              a3 += u1[l + 1] * x1[l + 1];
            }
          }
        } else {
          for (int l = 0; l < M; l++) {
            a0 += u0[l] * x0[l];
            a1 += u1[l] * x1[l];
          }
        }
        const double acc = (a0 + a2) + (a1 + a3);
        w1[(c * 2 + sg) * M + ku] = acc;
        w[(slot_base(lev) + (size_t)j * n + c) * M2 + sg * M + ku] = acc;
      }
    }
    __syncthreads();
    double *tmp = w0;
    w0 = w1;
    w1 = tmp;
  }

  // ---- contributions of the root (level lu, chunk j) to its ancestors:
  // part[l][j] = P(lu-l, j mod 2^(lu-l)) w_root
  for (int task = tid; task < np; task += kUpNT) {
    const int lev = task / M2, o = task % M2, sg = o / M, i = o % M;
    const double *x = w0 + sg * M;
    const int k = g.lu - lev;
    const size_t d = (size_t)j & (((size_t)1 << k) - 1);
    const double *prow = P + ((((size_t)1 << k) - 2) + d) * MM + (size_t)i * M;
    double acc = 0;
#pragma unroll
    for (int l = 0; l < (MT > 0 ? MT : 64); l++) {
      if (MT == 0 && l >= M) break;
      acc += prow[l] * x[l];
    }
    part[((size_t)lev * ((size_t)4 << g.lu) + j) * M2 + o] = acc;
  }
}

// ---------------------------------------------------------------------------
// The upward pass of a subtree of G = 2^gu <= 16 leaf chunks, M = 18 (steps 1
// and 2, src/C/leg2cheb.c:1379-1399), all of it on v_mfma_f64_16x16x4f64 (A
// operand: lane l holds A[l%16][l/16]; B: lane l holds B[l/16][l%16]; D: lane
// l, register v holds D[l/16 + 4v][l%16]):
//   leaf moments W_par (G x M) = X_par (G x s) T_par (s x M), one wave per
//     (parity, 16-column tile of M);
//   parents (M x 2n) = [U0 U1] (M x 2M) times the children stacked (2M x 2n),
//     column 2c + parity for parent c, one wave per 16-row tile;
//   contributions of the root to its ancestors above the subtree.
// Every operand is loaded before any is used; each level leaves through LDS as
// whole vectors.  Bound by latency: one chain of loads, products and barriers
// per work-group.  s = 64: 2^16 5.5 us, 2^20 10.1, 64 lines of 2^18 89; with
// scalar loads, the moments stored a double at a time from the accumulators
// and (more than 8 lines) VALU levels 6.0, 11.8 and 107.  LDS: input [2][16][xst] (xst = 2 mod 4: rows in distinct
// banks), two levels' moments [16 + 8][2][M].
__host__ __device__ inline int up18_xstride(int s) { return s + (6 - (s & 3)) % 4; }
struct Up18Lds {
  int xst, w0, w1, total;
};
__host__ __device__ inline Up18Lds up18_lds(const Geo &g) {
  Up18Lds d;
  d.xst = up18_xstride(g.s);
  d.w0 = 2 * 16 * d.xst;
  d.w1 = d.w0 + 16 * 36;
  d.total = d.w1 + 16 * 36;  // (the levels read 16 chunks, used or not)
  return d;
}
bool up18_eligible(const Geo &g) { return g.M == 18 && g.s <= 64; }
__device__ __forceinline__ void up18_group(const double *__restrict__ in, const LineMap &lm,
                                           const Geo &g, int dir, const double *__restrict__ T,
                                           const double *__restrict__ U,
                                           const double *__restrict__ P,
                                           double *__restrict__ wsall, size_t wsstride, int j,
                                           unsigned line, double *sm) {
  constexpr int M = 18, M2 = 36, MM = M * M;
  const int s = g.s, G = 1 << g.gu;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15, kq = lane >> 4;
  const size_t es = lm.es, base = (size_t)j * G * 2 * s;
  const size_t Nl = (size_t)line_len(lm, line, g.N);  // zeros past the line's end
  const double *src = in + line_off(lm, line) + base * es;
  const int nl = base < Nl ? (int)std::min<size_t>(Nl - base, (size_t)G * 2 * s) : 0;
  double *ws = wsall + line * wsstride;
  const WsLayout lay = ws_layout(g);
  const Up18Lds ly = up18_lds(g);
  double *xs = sm, *w0 = sm + ly.w0, *w1 = sm + ly.w1;

  // ---- loads: input pairs (2 h, 2 h + 1)
  constexpr int QX = 4;  // 16 s / 256 for s = 64
  d2 vx[QX];
  if (es == 1) {
    const __amdgpu_buffer_rsrc_t r = line_rsrc(nl ? src : in, nl);
#pragma unroll
    for (int q = 0; q < QX; q++) vx[q] = load_pair(r, 16 * tid + 4096 * q, 0);
  } else {
#pragma unroll
    for (int q = 0; q < QX; q++) {
      const int e = 2 * (tid + 256 * q);
      vx[q].x = e < nl ? src[(size_t)e * es] : 0.0;
      vx[q].y = e + 1 < nl ? src[(size_t)(e + 1) * es] : 0.0;
    }
  }
  // T, rows 4 q + kq, column kb of this wave's (parity, tile); columns past M
  // lie past the descriptor's end and read zero
  const int sg = wave >> 1, kb = (wave & 1) * 16 + n16;
  constexpr int QT = 16;
  double tb[QT];
  {
    const __amdgpu_buffer_rsrc_t r = line_rsrc(T + (size_t)sg * s * M, s * M);
    const int off = kb < M ? 8 * (kq * M + kb) : 1 << 30;
#pragma unroll
    for (int q = 0; q < QT; q++) tb[q] = load_one(r, off, 4 * M * 8 * q);
  }
  // [U0 U1], rows 16 rt + n16 of waves rt < 2: column k = 4 kk + kq, the
  // second operator from k = M on
  double ua[9];
  {
    const __amdgpu_buffer_rsrc_t r = line_rsrc(U, 2 * MM);
    const int ra = wave * 16 + n16;
    const int o0 = ra < M ? 8 * (ra * M + kq) : 1 << 30, o1 = ra < M ? o0 + 8 * (MM - M) : 1 << 30;
    const int o4 = kq < 2 ? o0 : o1;
#pragma unroll
    for (int kk = 0; kk < 9; kk++) ua[kk] = load_one(r, kk < 4 ? o0 : kk == 4 ? o4 : o1, 32 * kk);
  }
  __builtin_amdgcn_sched_barrier(0);
  const unsigned inv = ((1u << 20) + s - 1) / s;  // h / s = h inv >> 20 for h <= 1024
#pragma unroll
  for (int q = 0; q < QX; q++) {
    const int h = tid + 256 * q;
    if (h < G * s) {
      const int c = (int)(__umul24(h, inv) >> 20);
      double x0 = vx[q].x, x1 = vx[q].y;
      if (dir == C2L) {  // v_i = i u_i, v_0 = u_0 (src/C/leg2cheb.c:1325-1335)
        const double i = (double)(base + 2 * h);
        x0 *= i == 0.0 ? 1.0 : i;
        x1 *= i + 1.0;
      }
      const int a = c * ly.xst + h - c * s;
      xs[a] = x0;
      xs[16 * ly.xst + a] = x1;
    }
  }
  lds_sync();

  // ---- step 1: leaf moments (rows of X past G are not used: each row of a
  // product depends on its own row of A alone)
  {
    const double *xrow = xs + (sg * 16 + n16) * ly.xst + kq;
    d4 D0 = {0, 0, 0, 0}, D1 = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < QT; q += 2) {
      if (4 * q >= s) continue;
      double a0 = xrow[4 * q], a1 = xrow[4 * q + 4];
      if (4 * q + 8 > s) {
        a0 = 4 * q + kq < s ? a0 : 0.0;
        a1 = 4 * q + 4 + kq < s ? a1 : 0.0;
      }
      D0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, tb[q], D0, 0, 0, 0);
      D1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, tb[q + 1], D1, 0, 0, 0);
    }
    D0 += D1;
#pragma unroll
    for (int v = 0; v < 4; v++)
      if (kb < M) w0[(kq + 4 * v) * M2 + sg * M + kb] = D0[v];
  }
  lds_sync();

  // ---- step 2: up the subtree; each level's vectors go out as they lie in LDS
  auto store_level = [&](const double *wl, int lev, int n) {
    double *w = ws + lay.w + (slot_base(lev) + (size_t)j * n) * M2;
    for (int e = tid; e < n * M; e += 256)
      *reinterpret_cast<d2 *>(w + 2 * e) = *reinterpret_cast<const d2 *>(wl + 2 * e);
  };
  store_level(w0, g.L - 1, G);
  int n = G;
  for (int lev = g.L - 2; lev >= g.lu; lev--) {
    n >>= 1;
    if (wave < 2) {
      const int cc = n16 >> 1, sgc = n16 & 1;
      double bv[9];
#pragma unroll
      for (int kk = 0; kk < 9; kk++) {
        const int k = 4 * kk + kq, pu = k < M ? 0 : 1;
        // children of column pair cc of the 8 (past n: values not used)
        bv[kk] = w0[((2 * cc + pu) * 2 + sgc) * M + k - pu * M];
      }
      d4 D0 = {0, 0, 0, 0}, D1 = {0, 0, 0, 0};
#pragma unroll
      for (int kk = 0; kk < 9; kk += 2) {
        D0 = __builtin_amdgcn_mfma_f64_16x16x4f64(ua[kk], bv[kk], D0, 0, 0, 0);
        if (kk + 1 < 9) D1 = __builtin_amdgcn_mfma_f64_16x16x4f64(ua[kk + 1], bv[kk + 1], D1, 0, 0, 0);
      }
      D0 += D1;
      double *o = w1 + n16 * M + wave * 16 + kq;
#pragma unroll
      for (int v = 0; v < 4; v++)
        if (wave * 16 + kq + 4 * v < M && n16 < 2 * n) o[4 * v] = D0[v];
    }
    lds_sync();
    double *tmp = w0;
    w0 = w1;
    w1 = tmp;
    store_level(w0, lev, n);
  }

  // ---- contributions of the root (level lu, chunk j) to its ancestors:
  // part[l][j] = P(lu-l, j mod 2^(lu-l)) w_root
  double *part = ws + lay.part;
  for (int task = tid; task < g.lu * M2; task += 256) {
    const int lev = task / M2, o = task - lev * M2, sgp = o >= M, i = o - sgp * M;
    const int k = g.lu - lev;
    const size_t d = (size_t)j & (((size_t)1 << k) - 1);
    const d2 *prow = reinterpret_cast<const d2 *>(P + ((((size_t)1 << k) - 2) + d) * MM +
                                                  (size_t)i * M);
    const double *x = w0 + sgp * M;
    double a0 = 0, a1 = 0;
#pragma unroll
    for (int l = 0; l < M / 2; l++) {
      const d2 p = prow[l];
      a0 += p.x * x[2 * l];
      a1 += p.y * x[2 * l + 1];
    }
    part[((size_t)lev * ((size_t)4 << g.lu) + j) * M2 + o] = a0 + a1;
  }
}

// The upward pass and, in the same launch, the near-field band, which needs
// nothing of the tree: grid (work-groups, lines, 2) with the band groups at z =
// 0, ahead of the shorter upward groups, or (.., .., 1) for the upward pass
// alone.  The band's products fill the CUs that the upward groups' loads and
// barriers leave idle, and a launch and its tail go: s = 64, k_band and k_up
// apart / together 2^16 15.5 / 10.8 us, 2^20 27.4 / 22.0, 64 lines of 2^18 254 /
// 247.  Band groups behind the upward ones of each line: 256 lines of 2^15 220
// us a call against 188.
//
// Shallow trees (L <= 4) have fewer band groups (nb) than upward ones, and work-groups
// go to the eight XCDs in turn: padded to the upward groups' number, two of four on
// a line of 3300, all of the band would fall to four XCDs.  Their line calls (LINES_FLAT)
// take a grid (nb + upward groups, lines) with the nb groups of every line first and
// none empty: 3000 lines of 3300 (s = 52) 310 -> 211 us (of it 128 the band's and 92 the
// upward groups' in launches of their own), the call 407 -> 301.  So do calls whose
// lines lie side by side (LINES_ACROSS).  LINES_FLAT for all of them costs 0.3 % (the
// division by the group count).
//
// LINES_RAW calls read the strided input twice, for the band and for the moments.  From a
// stride of 8 on (a cache line per element or two) the grid is (.., lines): eight band
// groups, then the upward groups of the same leaf chunks, on the same XCDs, which find
// most of it in their L2.  2^20 at stride 16 k_up 50.8 -> 40.8 us, the call 94 -> 78; at
// stride 2 one after the other is as fast or faster (64 lines of 2^16 113 / 125).
struct BandArgs {
  double *out;  // LINES_RAW: N sums a line
  const double *tab, *head;
  int nb;  // band groups of a line (0: the upward pass alone)
};
template <bool S16, int G, int ORDER>
__global__ void __launch_bounds__(kUpNT) __attribute__((amdgpu_waves_per_eu(4))) k_up(
    const double *__restrict__ in, LineMap lm, Geo g, int dir, const double *__restrict__ T,
    const double *__restrict__ U, const double *__restrict__ P, double *__restrict__ wsall,
    size_t wsstride, BandArgs ba) {
  extern __shared__ double sm[];
  Place w{blockIdx.x, blockIdx.y};
  bool band = blockIdx.z + 1 != gridDim.z;
  if (ORDER == LINES_RAW && ba.nb && gridDim.z == 1) {  // (LINES_RAW, in turn)
    const unsigned r = (4u << g.lu) / ba.nb, per = 8 + 8 * r;
    const unsigned j = blockIdx.x % per, i = blockIdx.x / per * 8 + (j & 7);
    if (i >= (unsigned)ba.nb) return;
    band = j < 8;
    w.grp = band ? i : i * r + (j >> 3) - 1;
  }
  if (ORDER == LINES_FLAT || ORDER == LINES_ACROSS) {
    const unsigned nl = gridDim.y, bands = ba.nb * nl, id = blockIdx.x + gridDim.x * blockIdx.y;
    band = id < bands;
    w = place_of<ORDER == LINES_ACROSS>(band ? id : id - bands, band ? ba.nb : 4u << g.lu, nl);
  }
  if (!band) {
    if ((int)w.grp < 4 << g.lu)
      up18_group(in, lm, g, dir, T, U, P, wsall, wsstride, w.grp, w.line, sm);
  } else {
    const size_t off = line_off(lm, w.line);
    constexpr bool raw = ORDER == LINES_RAW;
    band_group<S16, G>(in + off, lm.es, ba.out + (raw ? (size_t)w.line * g.N : off),
                       raw ? 1 : lm.es, line_len(lm, w.line, g.N), g, dir, w.grp, 0, ba.tab,
                       ba.head, sm);
  }
}

// ---------------------------------------------------------------------------
// k_m2l: M2L of every block (src/C/leg2cheb.c:1419-1435).  Block b of level l
// holds A(b,0), A(b,1), A(b,2); row chunk 2b gets A(b,0) w[2b+2] +
// A(b,1) w[2b+3], row chunk 2b+1 gets A(b,2) w[2b+3]; both parities at once.
// grid: total_blocks(lu) work-groups for the blocks above lu (one each, with
// the multipoles summed from the k_up contributions in a fixed order), then
// one work-group per four blocks below (one block per wave).  256 threads.
constexpr int kM2lNT = 256;
// per wave: three padded matrices, two multipoles, 3M row results
__host__ __device__ inline int m2l_wave_lds(int M) { return 3 * M * (M + 1) + 4 * M + 6 * M; }
// Blocks per work-group below lu: four (one per wave) when four staged blocks
// fit in 64 KiB of LDS (M <= 22), else one block per work-group.
int m2l_bpw(const Geo &g) {
  return 8 * (size_t)(4 * m2l_wave_lds(g.M) + kM2lNT) <= 64 * 1024 ? 4 : 1;
}
size_t m2l_shared_bytes(const Geo &g) {
  return 8 * (size_t)(m2l_bpw(g) * m2l_wave_lds(g.M) + kM2lNT);
}

// Order LDS traffic between lanes of one wave (the wave's DS operations run
// in order; the fences stop the compiler from moving them across).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Evaluate one staged block with the 64 lanes of a wave (WG = false) or the
// whole work-group (WG = true).  Al: [3][M][M+1] (padded rows),
// wl: [chunk 2b+2, 2b+3][parity][M], res: [3M][2] scratch.
template <int MT, bool WG>
__device__ __forceinline__ void m2l_block_compute(const double *Al, const double *wl,
                                                  double *res, int M, int lane,
                                                  double *out_even, double *out_odd) {
  constexpr int step = WG ? kM2lNT : 64;
  for (int row = lane; row < 3 * M; row += step) {
    const int sub = row / M, k = row % M;
    const double *arow = Al + row * (M + 1);
    const double *wv = wl + (sub == 0 ? 0 : 2 * M);
    double o0 = 0, o1 = 0;
#pragma unroll
    for (int l = 0; l < (MT > 0 ? MT : 64); l++) {
      if (MT == 0 && l >= M) break;
      const double a = arow[l];
      o0 += a * wv[l];
      o1 += a * wv[M + l];
    }
    (void)k;
    res[2 * row] = o0;
    res[2 * row + 1] = o1;
  }
  if (WG)
    __syncthreads();
  else
    wave_sync();
  for (int k = lane; k < M; k += step) {
    // row chunk 2b: (A(b,0) w[2b+2]) + (A(b,1) w[2b+3]); row chunk 2b+1: A(b,2) w[2b+3]
    out_even[k] = res[2 * k] + res[2 * (M + k)];
    out_even[M + k] = res[2 * k + 1] + res[2 * (M + k) + 1];
    out_odd[k] = res[2 * (2 * M + k)];
    out_odd[M + k] = res[2 * (2 * M + k) + 1];
  }
}

// Split-form M2L block (precision form 1): record slots in tier order (FP64,
// FP32, BF16), decoded to FP64 into the padded LDS block at pos[slot]; the
// dropped positions (slots past the three tiers) are written as zeros.
struct SplitView {
  const unsigned char *rec;
  const unsigned short *pos;
  int n64, n32, n16, rec_bytes;
};
template <int NTH>
__device__ __forceinline__ void split_unpack(const SplitView &sv, size_t block, int n3, double *Al,
                                             int t) {
  // Every slot reads the aligned 8-byte word holding its value (FP64: the
  // value; FP32: one half; BF16: one quarter), so the loads of a batch carry
  // no branch and all issue before the first LDS store.
  const unsigned char *rb = sv.rec + block * sv.rec_bytes;
  const int n2 = sv.n64 + sv.n32, nt = n2 + sv.n16;
  for (int i0 = 0; i0 < n3; i0 += 8 * NTH) {
    unsigned long long wv[8];
    int d[8], o[8];
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int i = i0 + q * NTH + t;
      d[q] = i < n3 ? (int)sv.pos[i] : -1;
      o[q] = i < sv.n64 ? 8 * i : i < n2 ? 8 * sv.n64 + 4 * (i - sv.n64) : 8 * sv.n64 + 4 * sv.n32 + 2 * (i - n2);
      const int oc = i < nt ? o[q] : 0;  // dropped slots read the record's first word
      wv[q] = *(const unsigned long long *)(rb + (oc & ~7));
    }
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int i = i0 + q * NTH + t;
      const int sh = 8 * (o[q] & 7);
      const double v64 = __longlong_as_double((long long)wv[q]);
      const double v32 = (double)__uint_as_float((unsigned)(wv[q] >> sh));
      const double v16 = (double)__uint_as_float(((unsigned)(wv[q] >> sh) & 0xFFFFu) << 16);
      const double v = i < sv.n64 ? v64 : i < n2 ? v32 : i < nt ? v16 : 0.0;
      if (d[q] >= 0) Al[d[q]] = v;
    }
  }
}

// One block per work-group (B < total_blocks(lu): multipoles summed from the
// k_up contributions; or any block when only one fits the LDS), its lines
// line0 .. line0 + nl - 1.  sm: m2l_wave_lds(M) + kM2lNT doubles.
template <int MT>
__device__ __forceinline__ void m2l_top(const Geo &g, const double *__restrict__ A,
                                        double *__restrict__ wsall, size_t wsstride,
                                        size_t line0, int nl, const SplitView &sv, double *sm,
                                        int B) {
  const int M = MT > 0 ? MT : g.M, M2 = 2 * M, MM = M * M, Mp = M + 1;
  const int tid = threadIdx.x;
  const WsLayout lay = ws_layout(g);
  const int WL = m2l_wave_lds(M);
  int lev = 0;
  while ((int)total_blocks(lev + 1) <= B) lev++;
  const int b = B - (int)total_blocks(lev);
  double *Al = sm, *wl = sm + 3 * M * Mp, *red = sm + WL;
  if (sv.rec) {
    split_unpack<kM2lNT>(sv, (size_t)B, 3 * MM, Al, tid);
  } else {
    const double *Ab = A + (size_t)(3 * total_blocks(lev) + 3 * b) * MM;
    double va[8];
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int e = q * kM2lNT + tid;
      va[q] = e < 3 * MM ? Ab[e] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int e = q * kM2lNT + tid;
      if (e < 3 * MM) Al[(e / M) * Mp + e % M] = va[q];
    }
    for (int e = 8 * kM2lNT + tid; e < 3 * MM; e += kM2lNT) Al[(e / M) * Mp + e % M] = Ab[e];
  }
  const int nw = 2 * M2;  // multipole doubles of chunks 2b+2, 2b+3
  for (int li = 0; li < nl; li++) {
    double *ws = wsall + (line0 + li) * wsstride;
    const double *w = ws + lay.w;
    double *mo = ws + lay.m2l;
    if (lev >= g.lu) {
      const double *wb = w + (slot_base(lev) + 2 * (size_t)b + 2) * M2;
      for (int o = tid; o < nw; o += kM2lNT) wl[o] = wb[o];
    } else {
      const size_t nd = (size_t)1 << (g.lu - lev);
      const int ngrp = std::max(1, kM2lNT / nw);
      for (int o0 = 0; o0 < nw; o0 += kM2lNT) {
        const int o = o0 + tid % std::min(nw, kM2lNT), grp = tid / std::min(nw, kM2lNT);
        double acc = 0;
        if (grp < ngrp && o < nw) {
          const int ci = o / M2, oo = o % M2;
          const double *pp = ws + lay.part +
                             ((size_t)lev * ((size_t)4 << g.lu) + (2 * (size_t)b + 2 + ci) * nd) * M2 + oo;
          for (size_t d0 = grp; d0 < nd; d0 += 8 * (size_t)ngrp) {
            double v[8];
#pragma unroll
            for (int q = 0; q < 8; q++) {
              const size_t d = d0 + (size_t)q * ngrp;
              v[q] = d < nd ? pp[d * M2] : 0.0;
            }
#pragma unroll
            for (int q = 0; q < 8; q++) acc += v[q];
          }
        }
        red[tid] = acc;
        __syncthreads();
        if (tid < std::min(nw, kM2lNT) && o0 + tid < nw) {
          double sum = 0;
          for (int gi = 0; gi < ngrp; gi++) sum += red[gi * std::min(nw, kM2lNT) + tid];
          wl[o0 + tid] = sum;
        }
        __syncthreads();
      }
    }
    __syncthreads();
    m2l_block_compute<MT, true>(Al, wl, wl + nw, M, tid,
                                mo + (slot_base(lev) + 2 * (size_t)b) * M2,
                                mo + (slot_base(lev) + 2 * (size_t)b + 1) * M2);
    __syncthreads();  // wl and the result scratch are reused by the next line
  }
}

template <int MT>
__global__ void __launch_bounds__(kM2lNT) k_m2l(Geo g, const double *__restrict__ A,
                                                double *__restrict__ wsall, size_t wsstride,
                                                int bpw, size_t nlines, int lpb, SplitView sv) {
  extern __shared__ double sm[];
  const int M = MT > 0 ? MT : g.M, M2 = 2 * M, MM = M * M, Mp = M + 1;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const WsLayout lay = ws_layout(g);
  const int ntop = (int)total_blocks(g.lu);
  const int ntot = (int)total_blocks(g.L);
  const int WL = m2l_wave_lds(M);
  // lines line0 .. line0 + nl - 1 share every staged block (the plan's M2L
  // matrices are read once per work-group, not once per line)
  const size_t line0 = (size_t)blockIdx.y * lpb;
  const int nl = (int)std::min<size_t>((size_t)lpb, nlines - line0);

  if ((int)blockIdx.x < ntop || bpw == 1) {
    // ---- one block per work-group: every block above lu (multipoles summed
    // from the k_up contributions), and every block when bpw == 1
    if ((int)blockIdx.x < ntot) m2l_top<MT>(g, A, wsall, wsstride, line0, nl, sv, sm, blockIdx.x);
    return;
  }

  // ---- blocks at levels >= lu: one per wave
  const int B = ntop + ((int)blockIdx.x - ntop) * 4 + wave;
  if (B >= ntot) return;  // no work-group barrier below this point
  int lev = g.lu;
  while ((int)total_blocks(lev + 1) <= B) lev++;
  const int b = B - (int)total_blocks(lev);
  double *Al = sm + wave * WL, *wl = Al + 3 * M * Mp;
  const size_t wofs = lay.w + (slot_base(lev) + 2 * (size_t)b + 2) * M2;  // chunks 2b+2, 2b+3
  const size_t oofs = lay.m2l + (slot_base(lev) + 2 * (size_t)b) * M2;
  // multipoles of the first line; later lines are fetched one line ahead
  const double *wb = wsall + line0 * wsstride + wofs;
  double w0v = lane < 2 * M2 ? wb[lane] : 0.0;  // 2*M2 <= 192
  double w1v = lane + 64 < 2 * M2 ? wb[lane + 64] : 0.0;
  double w2v = lane + 128 < 2 * M2 ? wb[lane + 128] : 0.0;
  if (sv.rec) {
    split_unpack<64>(sv, (size_t)B, 3 * MM, Al, lane);
  } else {
    const double *Ab = A + (size_t)(3 * total_blocks(lev) + 3 * b) * MM;
    constexpr int QA = MT > 0 ? (3 * MT * MT + 63) / 64 : 16;
    double va[QA];
#pragma unroll
    for (int q = 0; q < QA; q++) {
      const int e = q * 64 + lane;
      va[q] = e < 3 * MM ? Ab[e] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < QA; q++) {
      const int e = q * 64 + lane;
      if (e < 3 * MM) Al[(e / M) * Mp + e % M] = va[q];
    }
    for (int e = QA * 64 + lane; e < 3 * MM; e += 64) Al[(e / M) * Mp + e % M] = Ab[e];
  }
  for (int li = 0; li < nl; li++) {
    if (lane < 2 * M2) wl[lane] = w0v;
    if (lane + 64 < 2 * M2) wl[lane + 64] = w1v;
    if (lane + 128 < 2 * M2) wl[lane + 128] = w2v;
    if (li + 1 < nl) {
      const double *wn = wsall + (line0 + li + 1) * wsstride + wofs;
      w0v = lane < 2 * M2 ? wn[lane] : 0.0;
      w1v = lane + 64 < 2 * M2 ? wn[lane + 64] : 0.0;
      w2v = lane + 128 < 2 * M2 ? wn[lane + 128] : 0.0;
    }
    wave_sync();
    double *mo = wsall + (line0 + li) * wsstride + oofs;
    m2l_block_compute<MT, false>(Al, wl, wl + 2 * M2, M, lane, mo, mo + M2);
    wave_sync();  // wl and the result scratch are reused by the next line
  }
}

// M2L of the blocks at levels >= lu, one block per wave, from At (rows across
// lanes): lane r < 3M holds row r of the block (r = sub M + row) in
// registers after M coalesced loads, so no block is staged in LDS and the
// work-group needs only the multipoles' 4M doubles per wave; the rows' sums
// are combined across lanes (chunk 2b: rows of sub 0 plus sub 1; chunk
// 2b+1: sub 2) in the order k_m2l uses, so the results are the same.  The
// first ntop work-groups take the blocks above lu as k_m2l does (one per
// work-group, from A).  Grid (ntop + (ntot - ntop + 3) / 4, line groups),
// kM2lNT threads, 8 (m2l_wave_lds(M) + kM2lNT) bytes of LDS.
template <int MT>
__global__ void __launch_bounds__(kM2lNT) k_m2l_t(Geo g, const double *__restrict__ A,
                                                  const double *__restrict__ At,
                                                  double *__restrict__ wsall, size_t wsstride,
                                                  size_t nlines, int lpb) {
  static_assert(MT > 0 && 3 * MT <= 64, "rows of a block across one wave");
  constexpr int M = MT, M2 = 2 * MT, MM = MT * MT;
  extern __shared__ double sm[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ntop = (int)total_blocks(g.lu), ntot = (int)total_blocks(g.L);
  const size_t line0 = (size_t)blockIdx.y * lpb;
  const int nl = (int)std::min<size_t>((size_t)lpb, nlines - line0);
  if ((int)blockIdx.x < ntop) {
    m2l_top<MT>(g, A, wsall, wsstride, line0, nl, SplitView{}, sm, blockIdx.x);
    return;
  }
  const int B = ntop + ((int)blockIdx.x - ntop) * 4 + wave;
  if (B >= ntot) return;  // no work-group barrier below this point
  int lev = g.lu;
  while ((int)total_blocks(lev + 1) <= B) lev++;
  const int b = B - (int)total_blocks(lev);
  const WsLayout lay = ws_layout(g);
  const size_t wofs = lay.w + (slot_base(lev) + 2 * (size_t)b + 2) * M2;  // chunks 2b+2, 2b+3
  const size_t oofs = lay.m2l + (slot_base(lev) + 2 * (size_t)b) * M2;
  const bool rowl = lane < 3 * M;
  const double *Ab = At + (size_t)B * 3 * MM;
  double a[M];
#pragma unroll
  for (int q = 0; q < M; q++) a[q] = rowl ? Ab[q * 3 * M + lane] : 0.0;
  double *wl = sm + wave * 2 * M2;
  const int sub = lane / M;
  const double *wv = wl + (sub == 0 ? 0 : M2);  // [chunk][parity][M]
  for (int li = 0; li < nl; li++) {
    const double *wb = wsall + (line0 + li) * wsstride + wofs;
    wl[lane] = wb[lane];
    if (lane + 64 < 2 * M2) wl[lane + 64] = wb[lane + 64];
    wave_sync();
    double o0 = 0, o1 = 0;
#pragma unroll
    for (int q = 0; q < M; q++) {
      o0 += a[q] * wv[q];
      o1 += a[q] * wv[M + q];
    }
    const double p0 = __shfl(o0, lane + M, 64), p1 = __shfl(o1, lane + M, 64);
    double *mo = wsall + (line0 + li) * wsstride + oofs;
    if (lane < M) {
      mo[lane] = o0 + p0;
      mo[M + lane] = o1 + p1;
    } else if (lane >= 2 * M && rowl) {
      mo[M2 + lane - 2 * M] = o0;
      mo[M2 + M + lane - 2 * M] = o1;
    }
    wave_sync();  // wl is rewritten for the next line
  }
}

// ---------------------------------------------------------------------------
// k_m2l_mma: M2L of the blocks at levels >= lu for many lines of one plan on
// MFMA, one block per wave, the lines in groups of 8 (16 MFMA columns:
// column n = line (n >> 1), parity n & 1).  A block's three submatrices are
// applied as one stacked operator E (36 x 36): rows 0..17 = [A(b,0) A(b,1)]
// give the M2L vector of chunk 2b, rows 18..35 = [0 A(b,2)] that of chunk
// 2b+1, both from the stacked multipoles S = [w(2b+2); w(2b+3)]
// (src/C/leg2cheb.c:1419-1435).
//   FORM 0: FP64, v_mfma_f64_16x16x4f64 (A lane l: E[l%16][l/16], B lane l:
//           S[l/16][l%16], D lane l reg v: [l/16 + 4v][l%16]); E's fragments
//           stay in registers across the wave's line groups.
//   FORM 2: BF16 slices, v_mfma_f32_16x16x32_bf16 (A lane l elem e:
//           E[l%16][8(l/16)+e], B lane l elem e: S[8(l/16)+e][l%16], D lane l
//           reg v: [4(l/16)+v][l%16]).  Rows of E carry a power-of-two scale
//           from plan time, columns of S one from their largest entry; both
//           are cut into kSlices slices q_i 2^(-8(i+1)) with integers
//           |q_i| <= 256, so every slice is exact in BF16, every product of
//           slices exact in FP32, and the sum over the 36 k of the pairs
//           (i, j) on one anti-diagonal i + j = d exact in one FP32
//           accumulator; anti-diagonals d < kSlices are kept and recombined
//           in FP64.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

// Cut x (|x| < 1) into kSlices integers q_i with x ~ sum q_i 2^(-8(i+1)).
__device__ __forceinline__ void cut_slices(double x, float q[kSlices]) {
#pragma unroll
  for (int i = 0; i < kSlices; i++) {
    const double sc = (double)(1ull << (8 * (i + 1)));
    const double qi = rint(x * sc);
    q[i] = (float)qi;
    x -= qi / sc;  // exact: qi / sc is x rounded to a coarser grid
  }
}

// Plan time (form 2): block B = ntop + blockIdx.x, one wave; lane l writes its
// fragment elements of every (row tile, k-step, slice) and, for l < 48, the
// scale of row l.
__global__ void __launch_bounds__(64) k_slice_A(const double *__restrict__ A, int M, int L, int lu,
                                                unsigned short *__restrict__ q,
                                                double *__restrict__ sc) {
  const int B = (int)total_blocks(lu) + blockIdx.x, l = threadIdx.x;
  int lev = lu;
  while ((int)total_blocks(lev + 1) <= B) lev++;
  const int b = B - (int)total_blocks(lev);
  const size_t MM = (size_t)M * M;
  const double *Ab = A + (3 * total_blocks(lev) + 3 * (size_t)b) * MM;
  auto E = [&](int r, int k) -> double {
    if (r < M) return k < M ? Ab[r * M + k] : (k < 2 * M ? Ab[MM + r * M + (k - M)] : 0.0);
    if (r < 2 * M && k >= M && k < 2 * M) return Ab[2 * MM + (r - M) * M + (k - M)];
    return 0.0;
  };
  auto row_scale = [&](int r) -> double {
    double m = 0.0;
    for (int k = 0; k < 2 * M; k++) m = fmax(m, fabs(E(r, k)));
    if (m == 0.0) return 0.0;
    int e;
    (void)frexp(m, &e);
    return ldexp(1.0, e);  // m < 2^e
  };
  const size_t blk = (size_t)blockIdx.x;
  if (l < 48) sc[blk * 48 + l] = row_scale(l);
  for (int t = 0; t < 3; t++) {
    const int r = 16 * t + (l & 15);
    const double s_r = row_scale(r);
    for (int kk = 0; kk < 2; kk++) {
      float qs[8][kSlices];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const int k = 32 * kk + 8 * (l >> 4) + e;
        cut_slices(s_r > 0 ? E(r, k) / s_r : 0.0, qs[e]);
      }
      for (int i = 0; i < kSlices; i++) {
        unsigned short *dst = q + ((((blk * 3 + t) * 2 + kk) * kSlices + i) * 64 + l) * 8;
#pragma unroll
        for (int e = 0; e < 8; e++) dst[e] = (unsigned short)(__float_as_uint(qs[e][i]) >> 16);
      }
    }
  }
}

// One flat grid: tx ty work-groups for the blocks above lu (tx blocks, their
// multipoles summed from the k_up contributions, ty shares of lpb lines) ahead of
// mx work-groups (four blocks each) per share of the line groups.  As a launch of
// their own (k_m2l) the top blocks took 19 us of 64 lines of 2^18, most of it
// with the chip nearly idle.
struct M2lGrid {
  int tx, ty, lpb, mx;
  SplitView sv;  // of the blocks above lu (precision form 1)
};
template <int FORM>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_m2l_mma(
    Geo g, const double *__restrict__ A, const bf16x8 *__restrict__ Aq,
    const double *__restrict__ Asc, double *__restrict__ wsall, size_t wsstride, size_t nlines,
    int groups_per_wg, M2lGrid mg) {
  extern __shared__ double sm[];
  int bx = (int)blockIdx.x - mg.tx * mg.ty;
  if (bx < 0) {  // a block above lu, lpb lines of it
    const size_t line0 = (size_t)(blockIdx.x / mg.tx) * mg.lpb;
    m2l_top<18>(g, A, wsall, wsstride, line0, (int)std::min<size_t>(mg.lpb, nlines - line0),
                mg.sv, sm, blockIdx.x % mg.tx);
    return;
  }
  const int by = bx / mg.mx;
  bx -= by * mg.mx;
  constexpr int M = 18, M2 = 36, MM = 324, Mp = 19;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntop = (int)total_blocks(g.lu), ntot = (int)total_blocks(g.L);
  const int B = ntop + bx * 4 + wave;
  if (B >= ntot) return;  // no work-group barrier below this point
  int lev = g.lu;
  while ((int)total_blocks(lev + 1) <= B) lev++;
  const int b = B - (int)total_blocks(lev);
  const WsLayout lay = ws_layout(g);
  const size_t sofs = lay.w + (slot_base(lev) + 2 * (size_t)b + 2) * M2;  // S: w(2b+2), w(2b+3)
  const size_t oofs = lay.m2l + (slot_base(lev) + 2 * (size_t)b) * M2;    // out: chunks 2b, 2b+1
  const size_t ngroups = (nlines + 7) / 8;
  const size_t gr0 = (size_t)by * groups_per_wg;
  const size_t gr1 = std::min(ngroups, gr0 + groups_per_wg);
  const int n = lane & 15;
  if (FORM == 0) {
    // the block into this wave's LDS rows, then E's 23 fragments into registers
    double *Al = sm + wave * 3 * M * Mp;
    const double *Ab = A + (size_t)(3 * total_blocks(lev) + 3 * b) * MM;
    constexpr int QA = (3 * MM + 63) / 64;
    double va[QA];
#pragma unroll
    for (int q = 0; q < QA; q++) {
      const int e = q * 64 + lane;
      va[q] = e < 3 * MM ? Ab[e] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < QA; q++) {
      const int e = q * 64 + lane;
      if (e < 3 * MM) Al[(e / M) * Mp + e % M] = va[q];
    }
    wave_sync();
    auto E = [&](int r, int k) -> double {
      if (r < M) return k < M ? Al[r * Mp + k] : Al[(M + r) * Mp + (k - M)];
      if (r < 2 * M && k >= M) return Al[(M + r) * Mp + (k - M)];  // A(b,2) rows
      return 0.0;
    };
    double ea[23];
#pragma unroll
    for (int j = 0; j < 9; j++) {
      const int k = 4 * j + (lane >> 4);
      ea[j] = E(n, k);
      ea[9 + j] = E(16 + n, k);
      if (j >= 4) ea[18 + j - 4] = E(32 + n, k);
    }
    for (size_t gr = gr0; gr < gr1; gr++) {
      const size_t line = gr * 8 + (n >> 1);
      const bool live = line < nlines;
      const double *S = wsall + (live ? line : 0) * wsstride + sofs + (n & 1) * M;
      double bv[9];
#pragma unroll
      for (int j = 0; j < 9; j++) {
        const int k = 4 * j + (lane >> 4);
        bv[j] = live ? S[(k >= M ? M2 : 0) + (k >= M ? k - M : k)] : 0.0;
      }
      d4 D0 = {0, 0, 0, 0}, D1 = D0, D2 = D0;
#pragma unroll
      for (int j = 0; j < 9; j++) {
        D0 = __builtin_amdgcn_mfma_f64_16x16x4f64(ea[j], bv[j], D0, 0, 0, 0);
        D1 = __builtin_amdgcn_mfma_f64_16x16x4f64(ea[9 + j], bv[j], D1, 0, 0, 0);
        if (j >= 4) D2 = __builtin_amdgcn_mfma_f64_16x16x4f64(ea[18 + j - 4], bv[j], D2, 0, 0, 0);
      }
      if (live) {
        double *o = wsall + line * wsstride + oofs + (n & 1) * M;
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int r0 = (lane >> 4) + 4 * v;  // rows of tiles 0, 1, 2: r0, 16 + r0, 32 + r0
          o[r0] = D0[v];                                          // r0 < 16: chunk 2b
          o[16 + r0 < M ? 16 + r0 : M2 + 16 + r0 - M] = D1[v];     // 16..17: 2b; 18..31: 2b+1
          if (32 + r0 < 2 * M) o[M2 + 32 + r0 - M] = D2[v];         // 32..35: 2b+1
        }
      }
    }
  } else {
    const size_t blk = (size_t)(B - ntop);
    const bf16x8 *Ablk = Aq + blk * 3 * 2 * kSlices * 64;
    for (size_t gr = gr0; gr < gr1; gr++) {
      const size_t line = gr * 8 + (n >> 1);
      const bool live = line < nlines;
      const double *S = wsall + (live ? line : 0) * wsstride + sofs + (n & 1) * M;
      // this lane's entries of S: k = 8 (l/16) + e (k-step 0), 32 + 8 (l/16) + e (k-step 1)
      double sv[2][8];
      double mx = 0.0;
#pragma unroll
      for (int kk = 0; kk < 2; kk++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const int k = 32 * kk + 8 * (lane >> 4) + e;
          sv[kk][e] = (live && k < M2) ? S[(k >= M ? M2 : 0) + (k >= M ? k - M : k)] : 0.0;
          mx = fmax(mx, fabs(sv[kk][e]));
        }
      mx = fmax(mx, __shfl_xor(mx, 16));
      mx = fmax(mx, __shfl_xor(mx, 32));
      double s_c = 0.0;
      if (mx > 0) {
        int ex;
        (void)frexp(mx, &ex);
        s_c = ldexp(1.0, ex);
      }
      // the column's slices as B fragments
      bf16x8 bq[2][kSlices];
#pragma unroll
      for (int kk = 0; kk < 2; kk++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
          float qs[kSlices];
          cut_slices(s_c > 0 ? sv[kk][e] / s_c : 0.0, qs);
#pragma unroll
          for (int i = 0; i < kSlices; i++) bq[kk][i][e] = (__bf16)qs[i];
        }
      // one row tile at a time: anti-diagonal accumulators, A's slices
      // fetched per slice (L2-resident), the column's slices kept
      double *o = wsall + line * wsstride + oofs + (n & 1) * M;
      const double *scb = Asc + blk * 48;
#pragma unroll 1
      for (int t = 0; t < 3; t++) {
        f4 acc[kSlices];
#pragma unroll
        for (int d = 0; d < kSlices; d++) acc[d] = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < kSlices; i++) {
          const bf16x8 a0 = Ablk[((t * 2 + 0) * kSlices + i) * 64 + lane];
          const bf16x8 a1 = Ablk[((t * 2 + 1) * kSlices + i) * 64 + lane];
#pragma unroll
          for (int j = 0; j + i < kSlices; j++) {
            acc[i + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, bq[0][j], acc[i + j], 0, 0, 0);
            acc[i + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, bq[1][j], acc[i + j], 0, 0, 0);
          }
        }
        if (live) {
#pragma unroll
          for (int v = 0; v < 4; v++) {
            const int r = 16 * t + 4 * (lane >> 4) + v;
            if (r >= M2) continue;
            double val = 0.0;
#pragma unroll
            for (int d = kSlices - 1; d >= 0; d--) val += ldexp((double)acc[d][v], -8 * (d + 2));
            o[r < M ? r : M2 + r - M] = val * (scb[r] * s_c);
          }
        }
      }
    }
  }
}

// Near-field band for four consecutive half-rows r0..r0+3 of one parity:
// columns c = r0 + t, t < len (len equal for the four rows), term
//   L2C: (a[t-rho] a[r+c+par]) x[c]            (src/C/leg2cheb.c:259,263)
//   C2L: -(dn[t-rho] x[c]) an[r+c+par]  or  -(dn an) x with precompute
//        (src/C/leg2cheb.c:416,426,471-486)
// a[t-rho] sits in a 4-register ring m, a[r+c+par] in a 4-register ring p;
// both rings are indexed by compile-time step numbers, eight steps per trip.
// xsg: parity's input window (skew sk4, origin at the work-group's first
// half-row), aw: Lambda window (skew sk8, origin at row0), hd: band head.
// ALIGNED: rl0 % 4 == 0, so every LDS offset inside a trip is a constant.
// Software-pipelined: the LDS reads of trip b+1 (eight x values, eight head
// values, eight ring refills) are issued before the arithmetic of trip b, so
// LDS latency hides behind 64 FP64 operations.  Reads run at most one trip
// (eight columns) past len, which stays inside the zero-filled windows.
template <int DIR, int PRE, int SG, int ALIGNED>
__device__ __forceinline__ void band_rows(const double *__restrict__ xsg,
                                          const double *__restrict__ aw,
                                          const double *__restrict__ hd, int rl0, int len,
                                          double acc[4]) {
  const int pb = 2 * rl0 + SG;
  int OX[8], OP[12];
  if (ALIGNED) {
#pragma unroll
    for (int k = 0; k < 8; k++) OX[k] = k + (k >> 2);
#pragma unroll
    for (int k = 0; k < 12; k++) OP[k] = k + ((SG + k) >> 3);
  } else {
#pragma unroll
    for (int k = 0; k < 8; k++) OX[k] = sk4(rl0 + k) - sk4(rl0);
#pragma unroll
    for (int k = 0; k < 12; k++) OP[k] = sk8(pb + k) - sk8(pb);
  }
  const double *xb = xsg + sk4(rl0);
  const double *pbp = aw + sk8(pb);
  const double *hb = hd;
  double m[4] = {0, 0, 0, 0};
  double p[4] = {pbp[OP[0]], pbp[OP[1]], pbp[OP[2]], pbp[OP[3]]};
  double a[4] = {acc[0], acc[1], acc[2], acc[3]};
  double XA[8], HA[8], PA[8], XB[8], HB[8], PB[8];
#define L2C_TERM(am, ap, x, acc_)   \
  if (DIR == 0)                     \
    acc_ += ((am) * (ap)) * (x);    \
  else if (PRE)                     \
    acc_ -= ((am) * (ap)) * (x);    \
  else                              \
    acc_ -= ((am) * (x)) * (ap);
#define BAND_STEP(K, XV, HV, PV)                           \
  {                                                        \
    m[(K) & 3] = (HV);                                     \
    const double x_ = (XV);                                \
    L2C_TERM(m[(K) & 3], p[(K) & 3], x_, a[0])             \
    L2C_TERM(m[((K) + 3) & 3], p[((K) + 1) & 3], x_, a[1]) \
    L2C_TERM(m[((K) + 2) & 3], p[((K) + 2) & 3], x_, a[2]) \
    L2C_TERM(m[((K) + 1) & 3], p[((K) + 3) & 3], x_, a[3]) \
    p[(K) & 3] = (PV);                                     \
  }
  // trip t's data: x at xb + 10t, heads at hb + 8t, refills at pbp + 9t
#define LOAD_TRIP(X, H, P, T)                                      \
  _Pragma("unroll") for (int k_ = 0; k_ < 8; k_++) {               \
    X[k_] = xb[10 * (T) + OX[k_]];                                 \
    H[k_] = hb[8 * (T) + k_];                                      \
    P[k_] = pbp[9 * (T) + OP[k_ + 4]];                             \
  }
#define RUN_TRIP(X, H, P)                                                  \
  BAND_STEP(0, X[0], H[0], P[0]) BAND_STEP(1, X[1], H[1], P[1])            \
  BAND_STEP(2, X[2], H[2], P[2]) BAND_STEP(3, X[3], H[3], P[3])            \
  BAND_STEP(4, X[4], H[4], P[4]) BAND_STEP(5, X[5], H[5], P[5])            \
  BAND_STEP(6, X[6], H[6], P[6]) BAND_STEP(7, X[7], H[7], P[7])
  const int nb = len >> 3, rem = len & 7;
  LOAD_TRIP(XA, HA, PA, 0)
  int b = 0;
  for (; b + 2 <= nb; b += 2) {
    LOAD_TRIP(XB, HB, PB, 1)
    RUN_TRIP(XA, HA, PA)
    LOAD_TRIP(XA, HA, PA, 2)
    RUN_TRIP(XB, HB, PB)
    xb += 20;
    pbp += 18;
    hb += 16;
  }
  if (b < nb) {
    RUN_TRIP(XA, HA, PA)
    LOAD_TRIP(XA, HA, PA, 1)
  }
  if (rem) {
    BAND_STEP(0, XA[0], HA[0], PA[0])
    BAND_STEP(1, rem > 1 ? XA[1] : 0.0, HA[1], PA[1])
    BAND_STEP(2, rem > 2 ? XA[2] : 0.0, HA[2], PA[2])
    BAND_STEP(3, rem > 3 ? XA[3] : 0.0, HA[3], PA[3])
    BAND_STEP(4, rem > 4 ? XA[4] : 0.0, HA[4], PA[4])
    BAND_STEP(5, rem > 5 ? XA[5] : 0.0, HA[5], PA[5])
    BAND_STEP(6, rem > 6 ? XA[6] : 0.0, HA[6], PA[6])
  }
#undef RUN_TRIP
#undef LOAD_TRIP
#undef BAND_STEP
#undef L2C_TERM
  acc[0] = a[0];
  acc[1] = a[1];
  acc[2] = a[2];
  acc[3] = a[3];
}

template <int DIR, int PRE>
__device__ __forceinline__ void band_dispatch(int sg, int aligned, const double *xsg,
                                              const double *aw, const double *hd, int rl0,
                                              int len, double acc[4]) {
  if (aligned) {
    if (sg == 0)
      band_rows<DIR, PRE, 0, 1>(xsg, aw, hd, rl0, len, acc);
    else
      band_rows<DIR, PRE, 1, 1>(xsg, aw, hd, rl0, len, acc);
  } else {
    if (sg == 0)
      band_rows<DIR, PRE, 0, 0>(xsg, aw, hd, rl0, len, acc);
    else
      band_rows<DIR, PRE, 1, 0>(xsg, aw, hd, rl0, len, acc);
  }
}


// ---------------------------------------------------------------------------
// k_down: grid (2^(ld+2), lines), 128 threads (2 waves).
constexpr int kR = 4;  // band rows per register block
constexpr int kDownNT = 128;

// LDS plan of k_down (offsets in doubles).  The M2L vectors and the chain
// partial sums are dead once the band phase starts; the output staging
// reuses them.
struct DownLds {
  int xs, aw, cres, mres, qp, out, total;
};
__host__ __device__ inline DownLds down_lds(const Geo &g) {
  const int G = 1 << g.gd, s = g.s, M2 = 2 * g.M;
  DownLds d;
  const int nx = G * s + s + 16;  // half-index window per parity (+ tail)
  const int nxs = nx + (nx >> 2) + 2;
  const int na = 2 * G * s + 2 * s + 32;  // Lambda window (full index)
  const int nas = na + (na >> 3) + 2;
  d.xs = 0;
  d.aw = d.xs + 2 * nxs;
  d.cres = d.aw + nas;
  d.mres = d.cres + (2 * G - 1) * M2;
  d.qp = d.mres + (g.ld + 2 * G - 1) * M2;
  d.out = d.mres;
  d.total = std::max(d.qp + std::max(g.ld, 1) * M2, d.out + 2 * G * s);
  return d;
}
size_t down8_shared_bytes(const Geo &g);
size_t down_shared_bytes(const Geo &g) {
  return g.fast ? down8_shared_bytes(g)
         : g.far ? std::max(far_shared_bytes(g), band_shared_bytes(g, 16))
                 : 8 * (size_t)down_lds(g).total;
}

// Subtree chunk slot cl (level ld + lam, position ci) of work-group Rr:
// slots are level-major, level ld + lam starting at 2^lam - 1.
__device__ __forceinline__ void sub_slot(int cl, int &lam, int &ci) {
  lam = 31 - __builtin_clz(cl + 1);
  ci = cl + 1 - (1 << lam);
}

// Address of M2L vector element e of the work-group's list [chain levels
// 0..ld-1 (ancestors of chunk Rr at level ld)][subtree slots], and whether the
// chunk has an M2L block (the last two chunks of every level have none).
__device__ __forceinline__ size_t m2l_elem(const Geo &g, int Rr, int e, int M2, bool &valid) {
  const int slot = e / M2, o = e - slot * M2;
  int lev;
  size_t r;
  if (slot < g.ld) {
    lev = slot;
    r = (size_t)Rr >> (g.ld - lev);
  } else {
    int lam, ci;
    sub_slot(slot - g.ld, lam, ci);
    lev = g.ld + lam;
    r = ((size_t)Rr << lam) + ci;
  }
  valid = r < ((size_t)4 << lev) - 2;
  return (slot_base(lev) + r) * M2 + o;
}

// Row k of the composite operator Q(ld - lev, Rr mod 2^(ld - lev)) for chain
// task (lev, k) = (task / M, task % M).
// Row k of the chain operator of task (lev, k).  The plan stores each Q
// matrix column-major, so the row's elements are M apart (qrow[l * M]) and
// the M threads of one level, rows k = 0..M-1, read consecutive words.
__device__ __forceinline__ const double *qrow_ptr(const double *Qg, const Geo &g, int Rr, int task,
                                                  int M) {
  const int lev = task / M, k = task - lev * M, kk = g.ld - lev;
  const size_t d = (size_t)Rr & (((size_t)1 << kk) - 1);
  return Qg + ((((size_t)1 << kk) - 2) + d) * (size_t)(M * M) + (size_t)k;
}

// Local expansions (L2L, src/C/leg2cheb.c:1437-1449) of the work-group's
// subtree into cres [slot][parity][M]: the root's c_ld = sum_lev Q(ld - lev,
// .) m2l_lev + m2l_ld replaces the chain c_l = D(r_l & 1) c_(l-1) + m2l_l
// (chunks without an M2L block, the last two of a level and all their
// ancestors, contribute zero exactly as in the chain); then levels
// ld+1..ld+gd: c = D(r & 1) c_parent + m2l.  mres: the M2L vectors in
// m2l_elem order; qp: ld x 2M scratch.  qr: row (tid / M, tid % M) of the
// chain operator when MT > 0 (else read from Qg).  DLDS: the subtree levels
// run on MFMA with D(p) from the LDS copy Dl ([p][k][M + 1], padded rows);
// else on VALU with D(p) row tid % M in d0r/d1r (MT > 0) or from Dg.  Every
// thread of the work-group must call this.
template <int MT, bool DLDS, class Sync>
__device__ __forceinline__ void subtree_locals(const Geo &g, int Rr, int tid, int NT,
                                               const double *mres, double *qp, double *cres,
                                               const double *qr, const double *d0r,
                                               const double *d1r, const double *Qg,
                                               const double *Dg, const double *Dl,
                                               Sync &&sync) {
  const int M = MT > 0 ? MT : g.M, M2 = 2 * M, MM = M * M;
  const int nq = g.ld * M;
  int task0 = tid;
  if (MT > 0 && tid < nq) {  // first task: the operator row is in registers
    const int lev = tid / M, k = tid - lev * M;
    const double *mv = mres + lev * M2;
    double o0 = 0, o1 = 0;
#pragma unroll
    for (int l = 0; l < (MT > 0 ? MT : 1); l++) {
      o0 += qr[l] * mv[l];
      o1 += qr[l] * mv[M + l];
    }
    qp[lev * M2 + k] = o0;
    qp[lev * M2 + M + k] = o1;
    task0 += NT;
  }
  for (int task = task0; task < nq; task += NT) {
    const int lev = task / M, k = task - lev * M;
    const double *mv = mres + lev * M2;
    const double *qrow = qrow_ptr(Qg, g, Rr, task, M);
    double o0 = 0, o1 = 0;
    for (int l = 0; l < M; l++) {
      o0 += qrow[l * M] * mv[l];
      o1 += qrow[l * M] * mv[M + l];
    }
    qp[lev * M2 + k] = o0;
    qp[lev * M2 + M + k] = o1;
  }
  sync();
  for (int o = tid; o < M2; o += NT) {
    // the chain terms in level order; four reads in flight per step
    double v = mres[g.ld * M2 + o];
    int lev = 0;
    for (; lev + 4 <= g.ld; lev += 4) {
      const double q0 = qp[lev * M2 + o], q1 = qp[(lev + 1) * M2 + o];
      const double q2 = qp[(lev + 2) * M2 + o], q3 = qp[(lev + 3) * M2 + o];
      v += q0;
      v += q1;
      v += q2;
      v += q3;
    }
    for (; lev < g.ld; lev++) v += qp[lev * M2 + o];
    cres[o] = v;
  }
  sync();
  if (DLDS) {
    // levels ld+1..ld+gd on v_mfma_f64_16x16x4f64: children of parity p are
    // C (M x n) = D(p) (M x M) C_parents (M x n), n = 2^lam children x 2
    // parities <= 16 columns: column j = child 2(j >> 1) + p, parity j & 1.
    // Work item (p, 16-row tile rt) per wave.
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = NT >> 6;
    const int nrt = (M + 15) >> 4, ksteps = (M + 3) >> 2;
    const int j = lane & 15;
    for (int lam = 1; lam <= g.gd; lam++) {
      const int n = 1 << lam, lev = g.ld + lam;
      const int b0 = n - 1, bp = (n >> 1) - 1;
      for (int item = wave; item < 2 * nrt; item += nw) {
        const int p = item / nrt, rt = item - p * nrt;
        const int ra = rt * 16 + j;  // A row
        d4 D = {0, 0, 0, 0};
        for (int kk = 0; kk < ksteps; kk++) {
          const int k = kk * 4 + (lane >> 4);
          const double a = (ra < M && k < M) ? Dl[(p * M + ra) * (M + 1) + k] : 0.0;
          const double b = (j < n && k < M) ? cres[(bp + (j >> 1)) * M2 + (j & 1) * M + k] : 0.0;
          D = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, D, 0, 0, 0);
        }
        const int c = 2 * (j >> 1) + p, sgc = j & 1;
        const bool valid = j < n && ((size_t)Rr << lam) + c < ((size_t)4 << lev) - 2;
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int row = rt * 16 + (lane >> 4) + 4 * v;
          if (row < M && j < n) {
            const int o = (b0 + c) * M2 + sgc * M + row;
            cres[o] = valid ? D[v] + mres[g.ld * M2 + o] : 0.0;
          }
        }
      }
      sync();
    }
    return;
  }
  const int kd = tid % M, ngrp = NT / M2;
  if (ngrp == 0) {  // fewer threads than 2M: one output per thread and pass, D from memory
    for (int lam = 1; lam <= g.gd; lam++) {
      const int n = 1 << lam, lev = g.ld + lam;
      const int b0 = n - 1, bp = (n >> 1) - 1;
      for (int idx = tid; idx < n * M2; idx += NT) {
        const int ci = idx / M2, oo = idx - ci * M2, sg = oo / M, k = oo - sg * M;
        const size_t r = ((size_t)Rr << lam) + ci;
        double v = 0;
        if (r < ((size_t)4 << lev) - 2) {
          const double *drow = Dg + (r & 1) * MM + (size_t)k * M;
          const double *par = cres + (bp + (ci >> 1)) * M2 + sg * M;
          for (int l = 0; l < M; l++) v += drow[l] * par[l];
          v += mres[(g.ld + b0 + ci) * M2 + oo];
        }
        cres[(b0 + ci) * M2 + oo] = v;
      }
      sync();
    }
    return;
  }
  auto l2l = [&](int p, const double *par) -> double {
    double a0 = 0, a1 = 0;
    if (MT > 0) {
#pragma unroll
      for (int l = 0; l < (MT > 0 ? MT : 1); l += 2) {
        a0 += (p ? d1r[l] : d0r[l]) * par[l];
        if (l + 1 < M) a1 += (p ? d1r[l + 1] : d0r[l + 1]) * par[l + 1];
      }
    } else {
      for (int l = 0; l < M; l++) a0 += Dg[p * MM + kd * M + l] * par[l];
    }
    return a0 + a1;
  };
  for (int lam = 1; lam <= g.gd; lam++) {
    const int n = 1 << lam, lev = g.ld + lam;
    const int b0 = n - 1, bp = (n >> 1) - 1;
    if (tid < ngrp * M2) {
      const int oo = tid % M2, sg = oo / M;
      for (int ci = tid / M2; ci < n; ci += ngrp) {
        const size_t r = ((size_t)Rr << lam) + ci;
        double v = 0;
        if (r < ((size_t)4 << lev) - 2)
          v = l2l((int)(r & 1), cres + (bp + (ci >> 1)) * M2 + sg * M) +
              mres[(g.ld + b0 + ci) * M2 + oo];
        cres[(b0 + ci) * M2 + oo] = v;
      }
    }
    sync();
  }
}

template <int DIR, int PRE, int MT>
__global__ void __launch_bounds__(kDownNT) __attribute__((amdgpu_waves_per_eu(2))) k_down(
    const double *__restrict__ in, double *__restrict__ out, LineMap lm, Geo g, int band_only,
    const double *__restrict__ wsall, size_t wsstride, const double *__restrict__ Dg,
    const double *__restrict__ Qg, const double *__restrict__ Tg, const double *__restrict__ tab,
    const double *__restrict__ htab) {
  extern __shared__ double sm[];
  const int M = MT > 0 ? MT : g.M;
  const int s = g.s, L = g.L, N = g.N, M2 = 2 * M, MM = M * M;
  const int G = 1 << g.gd;
  const int Rr = blockIdx.x;
  const int tid = threadIdx.x, NT = kDownNT;
  const size_t row0 = (size_t)Rr * G * 2 * s;
  if (row0 >= (size_t)N) return;
  const int nr = (int)std::min((size_t)G * 2 * s, (size_t)N - row0);
  const size_t off = line_off(lm, blockIdx.y);
  const double *src = in + off;
  double *dst = out + off;
  const double *ws = wsall + blockIdx.y * wsstride;
  const WsLayout lay = ws_layout(g);
  const double *m2l = ws + lay.m2l;
  const DownLds ld = down_lds(g);
  double *xs = sm + ld.xs;
  const int nxs = (ld.aw - ld.xs) / 2;
  double *aw = sm + ld.aw;
  double *cres = sm + ld.cres;
  double *mres = sm + ld.mres;
  double *qp = sm + ld.qp;
  double *ob = sm + ld.out;

  // ---- phase 0: every load issued before any store; addresses are clamped
  // into range and out-of-range values replaced afterwards, so the loads
  // issue as one straight-line batch
  const int nwin = G * 2 * s + 2 * s + 32;
  constexpr int QW = 10;
  double vx[QW], va[QW];
#pragma unroll
  for (int q = 0; q < QW; q++) {
    const size_t i = std::min(row0 + q * NT + tid, (size_t)N - 1);
    vx[q] = src[i * lm.es];
    va[q] = tab[i];
  }
  // M2L vectors: the ancestor chain (levels 0..ld-1) then the subtree slots
  const int nm = band_only ? 0 : (g.ld + 2 * G - 1) * M2;
  constexpr int QM = 8;
  double vm[QM];
  bool okm[QM];
#pragma unroll
  for (int q = 0; q < QM; q++) {
    const int e = q * NT + tid;
    const size_t a = m2l_elem(g, Rr, e < nm ? e : 0, M2, okm[q]);
    okm[q] = okm[q] && e < nm;
    vm[q] = m2l[okm[q] ? a : 0];
  }
  // ancestor chain in one step: task (lev, k) < ld*M takes row k of the
  // composite operator Q(ld - lev, Rr mod 2^(ld - lev)) from level lev to ld
  const int nq = band_only ? 0 : g.ld * M;
  double qr[MT > 0 ? MT : 1];
  if (MT > 0 && nq > 0) {
    const double *qrow = qrow_ptr(Qg, g, Rr, tid < nq ? tid : 0, M);
#pragma unroll
    for (int l = 0; l < (MT > 0 ? MT : 1); l++) qr[l] = qrow[l * M];
  }
#pragma unroll
  for (int q = 0; q < QW; q++) {
    const int e = q * NT + tid;
    if (e < nwin) {
      const size_t i = row0 + e;
      const double u = i < (size_t)N ? vx[q] : 0.0;
      xs[(e & 1) * nxs + sk4(e >> 1)] = (DIR == 1 && i > 0) ? u * (double)i : u;  // v_i = i u_i
      aw[sk8(e)] = i < (size_t)N ? va[q] : 0.0;
    }
  }
  for (int e = QW * NT + tid; e < nwin; e += NT) {
    const size_t i = row0 + e;
    double v = i < (size_t)N ? src[i * lm.es] : 0.0;
    if (DIR == 1 && i > 0) v *= (double)i;
    xs[(e & 1) * nxs + sk4(e >> 1)] = v;
    aw[sk8(e)] = i < (size_t)N ? tab[i] : 0.0;
  }
#pragma unroll
  for (int q = 0; q < QM; q++) {
    const int e = q * NT + tid;
    if (e < nm) mres[e] = okm[q] ? vm[q] : 0.0;
  }
  for (int e = QM * NT + tid; e < nm; e += NT) {
    bool ok;
    const size_t a = m2l_elem(g, Rr, e, M2, ok);
    mres[e] = ok ? m2l[a] : 0.0;
  }
  // this thread's rows of the two L2L operators (k = tid % M), needed from
  // the subtree pass on; loaded after the window registers are released
  const int kd = tid % M;
  double d0r[MT > 0 ? MT : 1], d1r[MT > 0 ? MT : 1];
  if (MT > 0 && !band_only) {
#pragma unroll
    for (int l = 0; l < (MT > 0 ? MT : 1); l++) {
      d0r[l] = Dg[kd * M + l];
      d1r[l] = Dg[MM + kd * M + l];
    }
  }
  __syncthreads();

  // ---- phase 2: local expansions of the subtree
  if (!band_only)
    subtree_locals<MT, false>(g, Rr, tid, NT, mres, qp, cres, qr, d0r, d1r, Qg, Dg, nullptr,
                             LdsSync{});

  // ---- phase 3: band + leaf evaluation.  Task (chunk, group gam): rows
  // gam*4.. of parity 0, then rows (ngrp-1-gam)*4.. of parity 1, so every
  // thread runs the same number of columns, parity is uniform across a wave
  // in each half, and 16 consecutive lanes take 16 consecutive row groups.
  const int ngrp = (s + kR - 1) / kR;
  const int ntask = G * ngrp;
  const int nLm1 = g.nL - 1;
  const size_t nvalid = ((size_t)2 << L) - 2;
  const size_t c0 = (size_t)Rr * G * s;
  const int aligned = (s & 3) == 0;
  for (int task = tid; task < ntask; task += NT) {
    const int pp = task % ngrp, gch = task / ngrp;
    const size_t beta = (size_t)Rr * G + gch;
    for (int sg = 0; sg < 2; sg++) {
      const int gam = sg == 0 ? pp : ngrp - 1 - pp;
      const int cnt = (N - sg + 1) / 2;  // elements of parity sg
      const size_t cend = beta < (size_t)nLm1 ? (beta + 2) * s : (size_t)cnt;
      const size_t r0 = beta * s + (size_t)gam * kR;
      if (r0 >= (size_t)cnt) continue;
      const int rl0 = (int)(r0 - c0);
      const int len = (int)(cend - r0);
      double acc[kR];
      const double *xsg = xs + sg * nxs;
      if (DIR == 0) {
        acc[0] = acc[1] = acc[2] = acc[3] = 0.0;
      } else {
#pragma unroll
        for (int rho = 0; rho < kR; rho++)
          acc[rho] = kSqrtPi * xsg[sk4(rl0 + rho)] * aw[sk8(2 * (rl0 + rho) + sg)];
      }
      band_dispatch<DIR, PRE>(sg, aligned, xsg, aw, htab, rl0, len, acc);
      // far field: local expansion of leaf chunk beta at the rows' nodes
      double far[kR] = {0, 0, 0, 0};
      if (!band_only && beta < nvalid) {
        const double *c = cres + (G - 1 + gch) * M2 + sg * M;
        if (g.nodal) {
          // Lagrange basis: far = sum_k T_par[m][k] c[k] with the plan's T
#pragma unroll
          for (int rho = 0; rho < kR; rho++) {
            const int ml = min(gam * kR + rho, s - 1);
            const double *tr = Tg + ((size_t)sg * s + ml) * M;
            double f = 0;
            for (int k = 0; k < M; k++) f += tr[k] * c[k];
            far[rho] = f;
          }
        } else {
          // Chebyshev basis: T_k(X) by the three-term recurrence
#pragma unroll
          for (int rho = 0; rho < kR; rho++) {
            const double X = -1 + (double)(2 * (gam * kR + rho) + sg) / (double)s;
            const double X2 = 2 * X;
            double tm = 1, tc = X;
            double f = c[0] + X * c[1];
            for (int k = 2; k < M; k++) {
              const double tn = tc * X2 - tm;
              f += tn * c[k];
              tm = tc;
              tc = tn;
            }
            far[rho] = f;
          }
        }
      }
#pragma unroll
      for (int rho = 0; rho < kR; rho++) {
        const int ml = gam * kR + rho;
        const size_t r = r0 + rho;
        if (ml < s && r < (size_t)cnt) {
          const size_t i = 2 * r + sg;
          double v;
          if (DIR == 0) {
            v = (far[rho] + acc[rho]) * k2Pi;
            if (i == 0) v *= 0.5;
          } else {
            v = (far[rho] + acc[rho]) * ((double)i + 0.5);
          }
          ob[i - row0] = v;
        }
      }
    }
  }
  __syncthreads();
  // ---- phase 4: coalesced store
  for (int e = tid; e < nr; e += NT) dst[(row0 + e) * lm.es] = ob[e];
}

// ---------------------------------------------------------------------------
// k_down8: the downward pass for leaf sizes s = 16, 32, 64 of plans that have
// no k_far (M != 18).  grid
// (2^(ld+2), lines), 64 nw threads with nw = s/16 waves, G = 2^gd <= 16 leaf
// chunks per work-group.
//
// Near field in 8-row register blocks.  Rows of parity sg, chunk g and 8-row
// group gam = 2p + del run over column offsets t in [0, len), len = 2s - 8 gam
// (shorter in the last chunk).  Pair p's columns are cut at ts = s - 8p into
// segment A = [0, ts) and B = [ts, len); wave w runs segment A of pair w and
// segment B of pair nw-1-w, so every wave does 2s - 8(nw-1) columns (8 fewer
// for del = 1).  Lane = g + 16 sg + 32 del: all 64 lanes of a wave sit at the
// same t, so the Toeplitz factor Lambda(t - rho) (dn for C2L) is one uniform
// (scalar) load per column, and the LDS layouts make every lane address of an
// x or Lambda read distinct modulo 32 eight-byte slots:
//   x, per parity, half index h from the work-group start: h + h/s (one pad
//     per chunk; a trip of 8 columns never straddles one), parity 1 at +nxs
//     with nxs = 16 mod 32;
//   Lambda, per chunk g, local index q = 2(r - g s) + sg + t + rho
//     (< 3s + 16): g LW + q with LW = 2 mod 32.
// Far field: the subtree's local expansions evaluated at the leaf nodes on
// v_mfma_f64_16x16x4f64, F_par (s x G) = T_par (s x M) C_par (M x G), added to
// the band sums staged in LDS; then scaling and one coalesced store.
struct Down8Lds {
  int xs, nxs, lw, LW, hd, dl, cres, mres, qp, total;
};
__host__ __device__ inline Down8Lds down8_lds(const Geo &g) {
  const int G = 1 << g.gd, s = g.s, M2 = 2 * g.M;
  Down8Lds d;
  const int nh = (G + 1) * s + 8;  // half indices per parity, one trip of overrun
  const int nhp = nh + nh / s + 1;
  d.xs = 0;
  d.nxs = nhp + (48 - nhp % 32) % 32;  // = 16 mod 32
  d.LW = 3 * s + 16;
  d.LW += (34 - d.LW % 32) % 32;  // = 2 mod 32
  d.lw = d.xs + 2 * d.nxs;
  d.hd = d.lw + G * d.LW;  // band head, 2s + 16
  d.dl = d.hd + 2 * s + 16;  // D(0), D(1) with rows padded to M + 1
  d.cres = d.dl + g.M * M2 + M2;
  d.mres = d.cres + (2 * G - 1) * M2;
  d.qp = d.mres + (g.ld + 2 * G - 1) * M2;
  d.total = d.qp + std::max(g.ld, 1) * M2;
  return d;  // the output staging (2 G s doubles) reuses the x windows
}
size_t down8_shared_bytes(const Geo &g) { return 8 * (size_t)down8_lds(g).total; }
bool down8_eligible(const Geo &g) { return g.s == 16 || g.s == 32 || g.s == 64; }

// One band segment of 8 rows: columns t in [t0, t1) (t0 = 0 or a multiple of
// 8 shared by the wave), software-pipelined half a trip (4 columns) ahead.
// xsg: the lane's parity window; h0: half index of the first row from the
// work-group start; pw: the lane's Lambda window at q = t = 0 of row 0;
// head: the zero-padded band head in LDS (read at wave-uniform addresses:
// keeping it out of scalar memory leaves LDS reads the only users of the
// lgkm counter, so the half-trip prefetch is not drained by scalar waits).
// RAGGED: columns
// t >= len are masked (the last chunk, where len is not a multiple of 8).
template <int DIR, int PRE, bool RAGGED, bool LEAN = false>
__device__ __forceinline__ void band_seg8(const double *__restrict__ xsg,
                                          const double *__restrict__ pw,
                                          const double *__restrict__ head, int h0, int sh,
                                          int t0, int t1, int len, double acc[8]) {
  const int s = 1 << sh;
  const int ntrip = t1 > t0 ? (t1 - t0 + 7) >> 3 : 0;
  if (ntrip == 0) return;
  // ring state at t0: heads Lambda(t0 - 8 + k), refills p(t0 + k)
  double hr[8], pr[8];
  const double *pp = pw + t0;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    hr[k] = t0 >= 8 ? head[t0 - 8 + k] : 0.0;
    pr[k] = pp[k];
  }
  // the trip being fetched: x pointer and position inside its chunk
  int hq = h0 + t0;
  const double *xq = xsg + hq + (hq >> sh);
  int mq = hq & (s - 1);
  const double *hp = head + t0;
  int tt = t0;
  double XA[4], PA[4], HA[4], XB[4], PB[4], HB[4];
  // half H (0: columns 0-3, 1: 4-7) of the current trip
#define FETCH(X, P, H, HALF)                                         \
  _Pragma("unroll") for (int k_ = 0; k_ < 4; k_++) {                 \
    X[k_] = xq[4 * (HALF) + k_];                                     \
    if (RAGGED) X[k_] = tt + 4 * (HALF) + k_ < len ? X[k_] : 0.0;    \
    P[k_] = pp[8 + 4 * (HALF) + k_];                                 \
    H[k_] = hp[4 * (HALF) + k_];                                     \
  }
#define NEXT_TRIP                   \
  {                                 \
    const int pad_ = mq + 8 == s;   \
    mq = pad_ ? 0 : mq + 8;         \
    xq += 8 + pad_;                 \
    pp += 8;                        \
    hp += 8;                        \
    tt += 8;                        \
  }
#define TERM(hv, pv, xv, a)          \
  if (DIR == 0)                      \
    a += ((hv) * (pv)) * (xv);       \
  else if (PRE)                      \
    a -= ((hv) * (pv)) * (xv);       \
  else                               \
    a -= ((hv) * (xv)) * (pv);
  // column t (ring slot K = t mod 8): head Lambda(t) enters slot K, row rho
  // uses Lambda(t - rho) and p(t + rho), then p(t + 8) replaces p(t)
#define STEP(K, X, P, H, J)                                \
  {                                                        \
    hr[K] = H[J];                                          \
    const double x_ = X[J];                                \
    TERM(hr[(K) & 7], pr[(K) & 7], x_, acc[0])             \
    TERM(hr[((K) + 7) & 7], pr[((K) + 1) & 7], x_, acc[1]) \
    TERM(hr[((K) + 6) & 7], pr[((K) + 2) & 7], x_, acc[2]) \
    TERM(hr[((K) + 5) & 7], pr[((K) + 3) & 7], x_, acc[3]) \
    TERM(hr[((K) + 4) & 7], pr[((K) + 4) & 7], x_, acc[4]) \
    TERM(hr[((K) + 3) & 7], pr[((K) + 5) & 7], x_, acc[5]) \
    TERM(hr[((K) + 2) & 7], pr[((K) + 6) & 7], x_, acc[6]) \
    TERM(hr[((K) + 1) & 7], pr[((K) + 7) & 7], x_, acc[7]) \
    pr[K] = P[J];                                          \
    if (LEAN) __builtin_amdgcn_sched_barrier(0);           \
  }
  FETCH(XA, PA, HA, 0)
  for (int b = 0; b < ntrip; b++) {
    FETCH(XB, PB, HB, 1)
    STEP(0, XA, PA, HA, 0) STEP(1, XA, PA, HA, 1) STEP(2, XA, PA, HA, 2) STEP(3, XA, PA, HA, 3)
    NEXT_TRIP
    FETCH(XA, PA, HA, 0)
    STEP(4, XB, PB, HB, 0) STEP(5, XB, PB, HB, 1) STEP(6, XB, PB, HB, 2) STEP(7, XB, PB, HB, 3)
  }
#undef STEP
#undef TERM
#undef NEXT_TRIP
#undef FETCH
}

template <int DIR, int PRE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_down8(
    const double *__restrict__ in, double *__restrict__ out, LineMap lm, Geo g,
    const double *__restrict__ wsall, size_t wsstride, const double *__restrict__ Dg,
    const double *__restrict__ Qg, const double *__restrict__ Tg, const double *__restrict__ tab,
    const double *__restrict__ head) {
  extern __shared__ double sm[];
  const int M = g.M;
  const int s = g.s, N = g.N, M2 = 2 * M, MM = M * M;
  // N: the plan geometry; Nl: this line's length (inputs past it read as zero)
  const int Nl = line_len(lm, blockIdx.y, N);
  const int G = 1 << g.gd, sh = 31 - __builtin_clz(s);
  const int nw = s >> 4, NT = 64 * nw;
  const int Rr = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  // the wave index is wave-uniform; saying so lets the band's column offsets
  // and head loads live in scalar registers
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const size_t row0 = (size_t)Rr * G * 2 * s;
  if (row0 >= (size_t)Nl) return;  // the whole work-group
  const int nr = (int)std::min((size_t)G * 2 * s, (size_t)Nl - row0);
  const size_t hc0 = (size_t)Rr * G * s;  // first half index of the work-group
  const size_t off = line_off(lm, blockIdx.y);
  const double *src = in + off;
  double *dst = out + off;
  const double *m2l = wsall + blockIdx.y * wsstride + ws_layout(g).m2l;
  const Down8Lds ly = down8_lds(g);
  double *xs = sm + ly.xs, *lw = sm + ly.lw, *cres = sm + ly.cres;
  double *mres = sm + ly.mres, *qp = sm + ly.qp, *hd = sm + ly.hd, *dl = sm + ly.dl;
  // output staging after the band: segment A sums in ob (the x windows),
  // segment B sums in ob2 (the Lambda windows); slot of output e: e + e / 2s
  // (one pad per chunk spreads the lanes of every writer over distinct banks)
  double *ob = xs, *ob2 = lw;
  auto slot = [&](int e) { return e + (e >> (sh + 1)); };

  // ---- phase 0: every global load of the kernel issued up front (clamped
  // addresses: one straight-line batch).  The tree operands (M2L vectors, the
  // chain row of Q, D) are needed first; the band windows (x, the Lambda span,
  // the head) stay in flight through the tree pass, whose barriers are
  // LDS-only.
  const int nm = (g.ld + 2 * G - 1) * M2;
  constexpr int QM = 6;
  double vm[QM];
  bool okm[QM];
#pragma unroll
  for (int q = 0; q < QM; q++) {
    const int e = q * NT + tid;
    const size_t a = m2l_elem(g, Rr, e < nm ? e : 0, M2, okm[q]);
    okm[q] = okm[q] && e < nm;
    vm[q] = m2l[okm[q] ? a : 0];
  }
  // keep the tree operands ahead of the windows in the memory pipeline: the
  // stores below then wait for them alone
  __builtin_amdgcn_sched_barrier(0);
  // x: input elements row0 + e, e < nX (both parities interleaved)
  const int nX = 2 * ((G + 1) * s + 8);
  constexpr int QX = 9;  // ceil(nX / NT) for G = 16
  double vx[QX];
  // Lambda: the contiguous span 2 hc0 + e, e < 2Gs + s + 16; element e lies
  // in chunk window e / 2s and, when e mod 2s < s + 16, also in the one before
  const int QL = 3 * s + 16, nLs = 2 * G * s + s + 16;
  constexpr int QLS = 9;  // ceil(nLs / NT) for G = 16
  double vl[QLS];
  const int nhd = 2 * s + 16;  // <= NT
  double vh = 0.0;
#pragma unroll
  for (int q = 0; q < QX; q++)
    vx[q] = src[std::min(row0 + q * NT + tid, (size_t)Nl - 1) * lm.es];
#pragma unroll
  for (int q = 0; q < QLS; q++)
    vl[q] = tab[std::min(2 * hc0 + q * NT + tid, (size_t)N - 1)];
  vh = head[tid < nhd ? tid : 0];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int q = 0; q < QM; q++) {
    const int e = q * NT + tid;
    if (e < nm) mres[e] = okm[q] ? vm[q] : 0.0;
  }
  for (int e = QM * NT + tid; e < nm; e += NT) {
    bool ok;
    const size_t a = m2l_elem(g, Rr, e, M2, ok);
    mres[e] = ok ? m2l[a] : 0.0;
  }
  for (int e = tid; e < 2 * MM; e += NT)
    dl[(e / M) * (M + 1) + e % M] = Dg[e];
  lds_sync();

  // ---- phase 2: local expansions of the subtree
  subtree_locals<0, true>(g, Rr, tid, NT, mres, qp, cres, nullptr, nullptr, nullptr, Qg, Dg, dl,
                            LdsSync{});

  const int ntm = s >> 4, ksteps = (M + 3) >> 2;
  // ---- the band windows
#pragma unroll
  for (int q = 0; q < QX; q++) {
    const int e = q * NT + tid;
    if (e < nX) {
      const size_t i = row0 + e;
      const double u = i < (size_t)Nl ? vx[q] : 0.0;
      const int h = e >> 1;
      xs[(e & 1) * ly.nxs + h + (h >> sh)] = (DIR == 1 && i > 0) ? u * (double)i : u;  // v_i = i u_i
    }
  }
  for (int e = QX * NT + tid; e < nX; e += NT) {
    const size_t i = row0 + e;
    double u = i < (size_t)Nl ? src[i * lm.es] : 0.0;
    if (DIR == 1 && i > 0) u *= (double)i;
    const int h = e >> 1;
    xs[(e & 1) * ly.nxs + h + (h >> sh)] = u;
  }
  auto put_lambda = [&](int e, double v) {
    const int c = e >> (sh + 1), q = e - (c << (sh + 1));
    if (2 * hc0 + e >= (size_t)N) v = 0.0;
    if (c < G) lw[c * ly.LW + q] = v;
    if (c > 0 && q + 2 * s < QL) lw[(c - 1) * ly.LW + q + 2 * s] = v;
  };
#pragma unroll
  for (int q = 0; q < QLS; q++) {
    const int e = q * NT + tid;
    if (e < nLs) put_lambda(e, vl[q]);
  }
  for (int e = QLS * NT + tid; e < nLs; e += NT)
    put_lambda(e, tab[std::min(2 * hc0 + e, (size_t)N - 1)]);
  if (tid < nhd) hd[tid] = vh;
  lds_sync();

  // ---- phase 3: near field.  Lane (chunk gl, parity sg, del); wave:
  // segment A of pair wave, segment B of pair nw-1-wave
  const int gl = lane & 15, sg = (lane >> 4) & 1, del = lane >> 5;
  const int cnt = (N - sg + 1) / 2;  // elements of parity sg
  const size_t beta = (size_t)Rr * G + gl;
  const size_t nLm1 = (size_t)g.nL - 1;
  const size_t cend = beta < nLm1 ? (beta + 2) * s : (size_t)cnt;
  const bool ragged = (size_t)(Rr + 1) * G > nLm1;  // work-group holds the last chunk
  const double *xsg = xs + sg * ly.nxs;
  double accA[8], accB[8];
  int rA = -1, rB = -1;  // first row (half index) of each segment, -1: none
  {
    const int p = wave, gam = 2 * p + del, ts = s - 8 * p;
    const size_t r0 = beta * s + 8 * gam;
    const bool live = gl < G && r0 < (size_t)cnt;
    const int len = live ? (int)(cend - r0) : 0;
    const int h0 = (int)(r0 - hc0);
    const double *pw = lw + gl * ly.LW + 16 * gam + sg;
#pragma unroll
    for (int k = 0; k < 8; k++) accA[k] = 0.0;
    if (live) {
      rA = h0;
      if (DIR == 1) {  // C2L diagonal: sqrt(pi) an_i v_i (src/C/leg2cheb.c:416)
        const double *xr = xsg + h0 + (h0 >> sh);
#pragma unroll
        for (int k = 0; k < 8; k++) accA[k] = kSqrtPi * xr[k] * pw[2 * k];
      }
    }
    if (ragged)
      band_seg8<DIR, PRE, true>(xsg, pw, hd, h0, sh, 0, std::min(ts, len), len, accA);
    else
      band_seg8<DIR, PRE, false>(xsg, pw, hd, h0, sh, 0, ts, len, accA);
  }
  {
    const int p = nw - 1 - wave, gam = 2 * p + del, ts = s - 8 * p;
    const size_t r0 = beta * s + 8 * gam;
    const bool live = gl < G && r0 < (size_t)cnt;
    const int len = live ? (int)(cend - r0) : 0;
    const int h0 = (int)(r0 - hc0);
    const double *pw = lw + gl * ly.LW + 16 * gam + sg;
#pragma unroll
    for (int k = 0; k < 8; k++) accB[k] = 0.0;
    if (live) rB = h0;
    if (ragged)
      band_seg8<DIR, PRE, true>(xsg, pw, hd, h0, sh, ts, len, len, accB);
    else
      band_seg8<DIR, PRE, false>(xsg, pw, hd, h0, sh, ts, len, len, accB);
  }
  lds_sync();  // windows dead: the staging takes their place

  // ---- phase 4: segment A sums to ob, segment B sums to ob2 (each row
  // once in each)
  auto stage = [&](int rl, const double *acc, double *dstg) {
    if (rl < 0) return;
#pragma unroll
    for (int k = 0; k < 8; k++)
      if (hc0 + rl + k < (size_t)cnt) dstg[slot(2 * (rl + k) + sg)] = acc[k];
  };
  stage(rA, accA, ob);
  stage(rB, accB, ob2);
  lds_sync();
  // F_par^T (G x s) = C_par^T (G x M) T_par^T (M x s), tile (parity sgf,
  // rows 16 rt..): A[n][k] = c_k of leaf n, B[k][m] = T_par[16 rt + m][k];
  // lane l then holds leaf l/16 + 4v, row 16 rt + l%16; added into ob.
  const int n = lane & 15;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int tile = wave + j * nw, sgf = tile / ntm, rt = tile - sgf * ntm;
    d4 D = {0, 0, 0, 0};
    for (int kk = 0; kk < ksteps; kk++) {
      const int k = kk * 4 + (lane >> 4);
      const double bv = k < M ? Tg[((size_t)sgf * s + rt * 16 + n) * M + k] : 0.0;
      const double av = (n < G && k < M) ? cres[(G - 1 + n) * M2 + sgf * M + k] : 0.0;
      D = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, D, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int leaf = (lane >> 4) + 4 * v, m = rt * 16 + n;
      const int e = 2 * (leaf * s + m) + sgf;
      if (leaf < G && e < nr) ob[slot(e)] += D[v];
    }
  }
  lds_sync();
  // ---- store: the scaled sum
  for (int e = tid; e < nr; e += NT) {
    const size_t i = row0 + e;
    double v = ob[slot(e)] + ob2[slot(e)];
    if (DIR == 0) {
      v *= k2Pi;
      if (i == 0) v *= 0.5;
    } else {
      v *= (double)i + 0.5;
    }
    dst[i * lm.es] = v;
  }
}

// ---------------------------------------------------------------------------
// k_down8r: k_down8's work (downward pass, near-field band, leaf evaluation;
// src/C/leg2cheb.c:1437-1483 and the band of :236-535) with wave roles.  The
// work-group has 2 s/16 waves: the first s/16 (the tree role) load the M2L
// vectors and operators, run the ancestor chain and the subtree's local
// expansions and evaluate them at the leaf nodes on MFMA (as k_far); the
// others (the band role) load the input and Lambda windows and sum the band,
// one row pair of 8 rows over all its columns per wave.  The roles share no
// LDS and synchronise among themselves with RoleSync; the one hardware
// barrier between them is the join before the scaled sum is stored.  So the
// band's FP64 VALU work overlaps the tree role's loads, LDS round trips and
// dependent MFMA steps inside each work-group, at 128 VGPRs and 78.5 KB of
// LDS (two work-groups, 16 waves, per CU at s = 64).
struct Down8rLds {
  int xs, nxs, lw, LW, hd, cres, dl, mres, qp, obf, ctr, total;
};
__host__ __device__ inline Down8rLds down8r_lds(const Geo &g) {
  const Down8Lds d8 = down8_lds(g);
  const int G = 1 << g.gd, s = g.s, M2 = 2 * g.M;
  Down8rLds d;
  d.xs = d8.xs;
  d.nxs = d8.nxs;
  d.lw = d8.lw;
  d.LW = d8.LW;
  d.hd = d8.hd;
  d.cres = d.hd + 2 * s + 16;
  d.dl = d.cres + (2 * G - 1) * M2;  // D(0), D(1) with rows padded to M + 1
  d.mres = d.dl + g.M * M2 + M2;
  d.qp = d.mres + (g.ld + 2 * G - 1) * M2;
  const int tree_end = d.qp + std::max(g.ld, 1) * M2;
  d.obf = d.dl;  // far-field staging (2 G s + G) over the tree's dead operands
  d.ctr = std::max(tree_end, d.obf + 2 * G * s + G);
  d.total = d.ctr + 1;  // the two roles' barrier counters
  return d;  // the band staging (2 G s + G) reuses the x windows
}
size_t down8r_shared_bytes(const Geo &g) { return 8 * (size_t)down8r_lds(g).total; }

template <int DIR, int PRE>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) k_down8r(
    const double *__restrict__ in, double *__restrict__ out, LineMap lm, Geo g,
    const double *__restrict__ wsall, size_t wsstride, const double *__restrict__ Dg,
    const double *__restrict__ Qg, const double *__restrict__ Tg, const double *__restrict__ tab,
    const double *__restrict__ head, int shift) {
  extern __shared__ double sm[];
  const int M = g.M;
  const int s = g.s, N = g.N, M2 = 2 * M, MM = M * M;
  const int Nl = line_len(lm, blockIdx.y, N);
  const int G = 1 << g.gd, sh = 31 - __builtin_clz(s);
  const int nw = s >> 4, NT = 64 * nw;  // waves and threads of each role
  const int Rr = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool tree = wave < nw;
  const int tid = tree ? (int)threadIdx.x : (int)threadIdx.x - NT;  // index in the role
  const size_t row0 = (size_t)Rr * G * 2 * s;
  if (row0 >= (size_t)Nl) return;  // the whole work-group
  const int nr = (int)std::min((size_t)G * 2 * s, (size_t)Nl - row0);
  const size_t hc0 = (size_t)Rr * G * s;
  const size_t off = line_off(lm, blockIdx.y);
  const double *src = in + off;
  double *dst = out + off;
  // the layout is work-group uniform; its divisions run on the VALU, so its
  // fields are moved to scalar registers rather than held (and spilled) in
  // vector registers through the band loops
  Down8rLds ly = down8r_lds(g);
  ly.nxs = __builtin_amdgcn_readfirstlane(ly.nxs);
  ly.lw = __builtin_amdgcn_readfirstlane(ly.lw);
  ly.LW = __builtin_amdgcn_readfirstlane(ly.LW);
  ly.hd = __builtin_amdgcn_readfirstlane(ly.hd);
  ly.cres = __builtin_amdgcn_readfirstlane(ly.cres);
  ly.dl = __builtin_amdgcn_readfirstlane(ly.dl);
  ly.mres = __builtin_amdgcn_readfirstlane(ly.mres);
  ly.qp = __builtin_amdgcn_readfirstlane(ly.qp);
  ly.obf = __builtin_amdgcn_readfirstlane(ly.obf);
  ly.ctr = __builtin_amdgcn_readfirstlane(ly.ctr);
  double *xs = sm + ly.xs, *lw = sm + ly.lw, *hd = sm + ly.hd;
  double *cres = sm + ly.cres, *dl = sm + ly.dl, *mres = sm + ly.mres, *qp = sm + ly.qp;
  double *ob = xs, *obf = sm + ly.obf;
  int *ctr = reinterpret_cast<int *>(sm + ly.ctr);
  auto slot = [&](int e) { return e + (e >> (sh + 1)); };
  // band lanes (both roles): chunk gl = lane % 16, parity sg = lane / 16 % 2,
  // del = lane / 32; row group gam = 2 p + del of pair p holds rows 8 gam ..
  // 8 gam + 7 of its chunk.  Computed where used, so that nothing of it is
  // live through the tree role's phases.
  // columns [t0, t1) of pair p's row group (t1 < 0: to its end) added to acc
  auto band = [&](int p, int t0, int t1, double acc[8]) {
    const int gl = lane & 15, sg = (lane >> 4) & 1, gam = 2 * p + (lane >> 5);
    const int cnt = (N - sg + 1) / 2;
    const size_t beta = (size_t)Rr * G + gl, nLm1 = (size_t)g.nL - 1;
    const size_t cend = beta < nLm1 ? (beta + 2) * s : (size_t)cnt;
    const size_t r0 = beta * s + 8 * gam;
    const bool live = gl < G && r0 < (size_t)cnt;
    const int len = live ? (int)(cend - r0) : 0;
    const int h0 = (int)(r0 - hc0);
    const double *pw = lw + gl * ly.LW + 16 * gam + sg;
    const double *xsg = xs + sg * ly.nxs;
    const int a0 = std::min(t0, len), a1 = t1 < 0 ? len : std::min(t1, len);
    if ((size_t)(Rr + 1) * G > nLm1)  // the work-group holds the last chunk
      band_seg8<DIR, PRE, true, true>(xsg, pw, hd, h0, sh, a0, a1, len, acc);
    else
      band_seg8<DIR, PRE, false, true>(xsg, pw, hd, h0, sh, a0, a1, len, acc);
  };
  // the sums of pair p's row group of this lane into staging st (= or +=)
  auto stage_group = [&](int p, const double acc[8], double *st, bool add) {
    // a fresh copy of the lane index (the empty asm hides that it equals
    // the one the band used), so that the band's row indices are recomputed
    // here instead of being held in registers through the band
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int gl = ln & 15, sg = (ln >> 4) & 1;
    const int cnt = (N - sg + 1) / 2;
    const size_t r0 = ((size_t)Rr * G + gl) * s + 8 * (2 * p + (ln >> 5));
    if (gl >= G || r0 >= (size_t)cnt) return;
    const int rl = (int)(r0 - hc0);
#pragma unroll
    for (int q = 0; q < 8; q++)
      if (r0 + q < (size_t)cnt) {
        double &o = st[slot(2 * (rl + q) + sg)];
        o = add ? o + acc[q] : acc[q];
      }
  };
  if (threadIdx.x == 0) {
    ctr[0] = 0;
    ctr[1] = 0;
  }
  lds_sync();  // hardware barrier 1 of 2

  if (tree) {
    // the tree role's chain of dependent LDS and MFMA steps is the critical
    // path: its waves issue ahead of the band role's FMA stream
    __builtin_amdgcn_s_setprio(3);
    RoleSync rs{ctr, nw, 0};
    const double *m2l = wsall + blockIdx.y * wsstride + ws_layout(g).m2l;
    const int nm = (g.ld + 2 * G - 1) * M2;
    constexpr int QM = 6;
    double vm[QM];
    bool okm[QM];
#pragma unroll
    for (int q = 0; q < QM; q++) {
      const int e = q * NT + tid;
      const size_t a = m2l_elem(g, Rr, e < nm ? e : 0, M2, okm[q]);
      okm[q] = okm[q] && e < nm;
      vm[q] = m2l[okm[q] ? a : 0];
    }
#pragma unroll
    for (int q = 0; q < QM; q++) {
      const int e = q * NT + tid;
      if (e < nm) mres[e] = okm[q] ? vm[q] : 0.0;
    }
    for (int e = QM * NT + tid; e < nm; e += NT) {
      bool ok;
      const size_t a = m2l_elem(g, Rr, e, M2, ok);
      mres[e] = ok ? m2l[a] : 0.0;
    }
    for (int e = tid; e < 2 * MM; e += NT)
      dl[(e / M) * (M + 1) + e % M] = Dg[e];
    rs();
    subtree_locals<0, true>(g, Rr, tid, NT, mres, qp, cres, nullptr, nullptr, nullptr, Qg, Dg, dl,
                             rs);
    // far field: F_par^T (G x s) = C_par^T (G x M) T_par^T (M x s) on
    // v_mfma_f64_16x16x4f64, two tiles (parity, 16 rows) per wave, written
    // to obf (the chain and subtree operands under it are dead: the last
    // role barrier of subtree_locals is behind every wave)
    const int ntm = s >> 4, ksteps = (M + 3) >> 2;
    const int n = lane & 15;
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int tile = wave + j * nw, sgf = tile / ntm, rt = tile - sgf * ntm;
      d4 D = {0, 0, 0, 0};
      for (int kk = 0; kk < ksteps; kk++) {
        const int k = kk * 4 + (lane >> 4);
        const double bv = k < M ? Tg[((size_t)sgf * s + rt * 16 + n) * M + k] : 0.0;
        const double av = (n < G && k < M) ? cres[(G - 1 + n) * M2 + sgf * M + k] : 0.0;
        D = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, D, 0, 0, 0);
      }
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int leaf = (lane >> 4) + 4 * v, m = rt * 16 + n;
        const int e = 2 * (leaf * s + m) + sgf;
        if (leaf < G && e < nr) obf[slot(e)] = D[v];
      }
    }
    rs();  // far field staged
    // segment B of pair nw - 1 - wave (columns s - 8p - shift onward,
    // k_down8's split moved by shift, a multiple of 8 in [-s, 8 nw]), once
    // the band role has the windows in LDS; added into obf
    const int p = nw - 1 - wave;
    double acc[8];
#pragma unroll
    for (int q = 0; q < 8; q++) acc[q] = 0.0;
    role_wait(ctr + 1, nw);
    band(p, s - 8 * p - shift, -1, acc);
    stage_group(p, acc, obf, true);
    role_arrive(ctr + 1);  // done with the windows
  } else {
    RoleSync rs{ctr + 1, nw, 0};
    // the window phase is address arithmetic and loads: at the default
    // priority its VALU instructions lose issue to the older work-group's
    // band FMAs on the same CU, and the second work-group of a CU gets its
    // windows only when the first one's band is done
    __builtin_amdgcn_s_setprio(2);
    // ---- the windows: x (both parities), the Lambda span, the head
    const int nX = 2 * ((G + 1) * s + 8);
    constexpr int QX = 9;  // ceil(nX / NT) for G = 16, s = 64
    double vx[QX];
    const int QL = 3 * s + 16, nLs = 2 * G * s + s + 16;
    constexpr int QLS = 9;
    double vl[QLS];
    const int nhd = 2 * s + 16;
#pragma unroll
    for (int q = 0; q < QX; q++) vx[q] = src[std::min(row0 + q * NT + tid, (size_t)Nl - 1) * lm.es];
#pragma unroll
    for (int q = 0; q < QLS; q++) vl[q] = tab[std::min(2 * hc0 + q * NT + tid, (size_t)N - 1)];
    double vh[3];
#pragma unroll
    for (int q = 0; q < 3; q++) vh[q] = head[q * NT + tid < nhd ? q * NT + tid : 0];
#pragma unroll
    for (int q = 0; q < QX; q++) {
      const int e = q * NT + tid;
      if (e < nX) {
        const size_t i = row0 + e;
        const double u = i < (size_t)Nl ? vx[q] : 0.0;
        const int h = e >> 1;
        xs[(e & 1) * ly.nxs + h + (h >> sh)] = (DIR == 1 && i > 0) ? u * (double)i : u;
      }
    }
    for (int e = QX * NT + tid; e < nX; e += NT) {
      const size_t i = row0 + e;
      double u = i < (size_t)Nl ? src[i * lm.es] : 0.0;
      if (DIR == 1 && i > 0) u *= (double)i;
      const int h = e >> 1;
      xs[(e & 1) * ly.nxs + h + (h >> sh)] = u;
    }
    auto put_lambda = [&](int e, double v) {
      const int c = e >> (sh + 1), q = e - (c << (sh + 1));
      if (2 * hc0 + e >= (size_t)N) v = 0.0;
      if (c < G) lw[c * ly.LW + q] = v;
      if (c > 0 && q + 2 * s < QL) lw[(c - 1) * ly.LW + q + 2 * s] = v;
    };
#pragma unroll
    for (int q = 0; q < QLS; q++) {
      const int e = q * NT + tid;
      if (e < nLs) put_lambda(e, vl[q]);
    }
    for (int e = QLS * NT + tid; e < nLs; e += NT)
      put_lambda(e, tab[std::min(2 * hc0 + e, (size_t)N - 1)]);
#pragma unroll
    for (int q = 0; q < 3; q++)
      if (q * NT + tid < nhd) hd[q * NT + tid] = vh[q];
    for (int e = 3 * NT + tid; e < nhd; e += NT) hd[e] = head[e];
    rs();

    // ---- segment A of pair wave - nw (columns [0, s - 8p - shift)), then the
    // C2L diagonal (added after the band: zero-started sums keep a single
    // set of accumulators live through the band's two code paths)
    __builtin_amdgcn_s_setprio(0);
    const int p = wave - nw;
    double acc[8];
#pragma unroll
    for (int q = 0; q < 8; q++) acc[q] = 0.0;
    band(p, 0, s - 8 * p - shift, acc);
    if (DIR == 1) {  // C2L diagonal: sqrt(pi) an_i v_i (src/C/leg2cheb.c:416)
      int ln = lane;  // a fresh copy (see stage_group)
      asm volatile("" : "+v"(ln));
      const int gl = ln & 15, sg = (ln >> 4) & 1, gam = 2 * p + (ln >> 5);
      const size_t r0 = ((size_t)Rr * G + gl) * s + 8 * gam;
      if (gl < G && r0 < (size_t)((N - sg + 1) / 2)) {
        const int rl = (int)(r0 - hc0);
        const double *xr = xs + sg * ly.nxs + rl + (rl >> sh);
        const double *pw = lw + gl * ly.LW + 16 * gam + sg;
#pragma unroll
        for (int q = 0; q < 8; q++) acc[q] += kSqrtPi * xr[q] * pw[2 * q];
      }
    }
    // windows dead once both roles' band waves are through: the staging
    // takes their place
    role_arrive(ctr + 1);
    role_wait(ctr + 1, 3 * nw);
    stage_group(p, acc, ob, false);
  }
  lds_sync();  // hardware barrier 2 of 2: the join
  __builtin_amdgcn_s_setprio(0);

  // ---- store: band plus far field, scaled
  for (int e = threadIdx.x; e < nr; e += 2 * NT) {
    const size_t i = row0 + e;
    double v = ob[slot(e)] + obf[slot(e)];
    if (DIR == 0) {
      v *= k2Pi;
      if (i == 0) v *= 0.5;
    } else {
      v *= (double)i + 0.5;
    }
    dst[i * lm.es] = v;
  }
}

// ---------------------------------------------------------------------------
// k_band: the near field by itself, for directM (scaled) and the split
// downward pass (down_split; raw sums, the C2L diagonal included, over the
// output; k_far adds the far field and scales, src/C/leg2cheb.c:1467-1483 and
// the band scaling of :236-535).  Grid (band groups, lines), 256 threads.
template <bool S16, int ORDER>
__global__ void __launch_bounds__(kBandNT) __attribute__((amdgpu_waves_per_eu(4))) k_band(
    const double *__restrict__ in, double *__restrict__ out, LineMap lm, Geo g, int dir, int scale,
    const double *__restrict__ tab, const double *__restrict__ head) {
  extern __shared__ double sm[];
  const Place w = place<ORDER == LINES_ACROSS>();
  constexpr bool raw = ORDER == LINES_RAW;
  const size_t off = line_off(lm, w.line);
  band_group<S16, 16>(in + off, lm.es, out + (raw ? (size_t)w.line * g.N : off), raw ? 1 : lm.es,
                      line_len(lm, w.line, g.N), g, dir, w.grp, scale, tab, head, sm);
}

// ---------------------------------------------------------------------------
// k_far: the downward pass of a subtree of G = 2^gd leaf chunks (any leaf size
// s <= 64, M = 18; src/C/leg2cheb.c:1437-1483): the ancestor chain in one
// step, the subtree's levels and the leaf evaluation on MFMA, added to the raw
// band sums in the output, scaled and stored.  Grid (2^(ld+2), lines), 256
// threads.  Latency-bound: every operand (M2L vectors, chain rows, D and T as
// MFMA fragments, the band sums) is loaded up front, so that the dependent
// steps run from registers and LDS.  s = 64: 2^16 6.7 us, 2^20 12.0, 64 lines of
// 2^18 94; with the operands read as each step needs them 7.8, 13.3 and 130.
constexpr int kFarNT = 256;
struct FarLds {
  int mres, qp, ob, CS, total;
};
__host__ __device__ inline FarLds far_lds(const Geo &g) {
  const int G = 1 << g.gd, s = g.s, M2 = 2 * g.M;
  FarLds d;
  d.mres = (2 * G - 1) * M2;  // after the local expansions [slot][parity][M]
  d.qp = d.mres + (g.ld + 2 * G - 1) * M2;
  d.ob = d.mres;  // far field [leaf][CS], over the dead M2L vectors
  d.CS = 2 * s + ((s & 1) ? 0 : 2);
  d.total = std::max(d.qp + std::max(g.ld, 1) * M2, d.ob + G * d.CS);
  return d;
}
size_t far_shared_bytes(const Geo &g) { return 8 * (size_t)far_lds(g).total; }
bool far_eligible(const Geo &g) { return g.M == 18 && g.s <= kBandMaxS; }

template <int ORDER>
__global__ void __launch_bounds__(kFarNT) __attribute__((amdgpu_waves_per_eu(4))) k_far(
    double *__restrict__ out, const double *__restrict__ raw, LineMap lm, Geo g,
    int dir, const double *__restrict__ wsall, size_t wsstride, const double *__restrict__ Dg, const double *__restrict__ Qg,
    const double *__restrict__ Tg) {
  extern __shared__ double sm[];
  constexpr int M = 18, M2 = 36, MM = M * M;
  const int s = g.s, N = g.N;
  const Place w = place<ORDER == LINES_ACROSS>();
  const int Nl = line_len(lm, w.line, N);
  const int G = 1 << g.gd, Rr = w.grp;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const size_t row0 = (size_t)Rr * G * 2 * s;
  if (row0 >= (size_t)Nl) return;  // the whole work-group
  const int nr = (int)std::min((size_t)G * 2 * s, (size_t)Nl - row0);
  const size_t es = lm.es;
  double *dst = out + line_off(lm, w.line) + row0 * es;
  const double *m2l = wsall + w.line * wsstride + ws_layout(g).m2l;
  const FarLds ly = far_lds(g);
  double *cres = sm, *mres = sm + ly.mres, *qp = sm + ly.qp, *ob = sm + ly.ob;

  // ---- loads.  M2L vectors: slots [chain levels 0..ld-1][subtree, level by
  // level], three slots of 18 pairs a wave; the last two chunks of a level
  // have no M2L block.  Slot r of level lev is chunk slot slot_base(lev) + r =
  // (B >> k) - 4 for the chain (k = ld - lev) and (B << lam) - 4 + ci for chunk
  // ci of subtree level lam, B = slot_base(ld) + 4 + Rr.
  const int nslot = g.ld + 2 * G - 1, sl = lane / 18, o2 = lane - 18 * sl;
  const unsigned B = (4u << g.ld) + Rr;
  auto slot_of = [&](int slot, bool &valid) -> size_t {
    const int cl = slot - g.ld;
    const int lam = cl < 0 ? cl : 31 - __builtin_clz(cl + 1);  // < 0: up the chain
    const int ci = cl < 0 ? 0 : cl + 1 - (1 << lam);
    const size_t c = (lam < 0 ? (size_t)(B >> -lam) : (size_t)B << lam) + ci;
    valid = lane < 54 && slot < nslot && c < ((size_t)8 << (g.ld + lam)) - 2;
    return c - 4;
  };
  constexpr int QM = 4;
  d2 vm[QM];
#pragma unroll
  for (int q = 0; q < QM; q++) {
    bool ok;
    const size_t c = slot_of((4 * q + wave) * 3 + sl, ok);
    const d2 v = *reinterpret_cast<const d2 *>(m2l + (ok ? c * M2 + 2 * o2 : 0));
    vm[q].x = ok ? v.x : 0.0;
    vm[q].y = ok ? v.y : 0.0;
  }
  // chain rows: task (lev, k) = (task / M, task % M), half a row per thread
  const int nq = g.ld * M, half = tid & 1;
  double qr[9];
  {
    const int task = std::min(tid >> 1, std::max(nq - 1, 0));
    const double *qrow = qrow_ptr(Qg, g, Rr, task, M) + half * 9 * M;
#pragma unroll
    for (int l = 0; l < 9; l++) qr[l] = nq > 0 ? qrow[l * M] : 0.0;
  }
  // D(p), rows 16 rt .. of this wave's item (p = wave / 2, rt = wave % 2)
  const int n16 = lane & 15, kq = lane >> 4;
  const int dp = wave >> 1, drt = wave & 1;
  double av[5];
#pragma unroll
  for (int kk = 0; kk < 5; kk++) {
    const int ra = drt * 16 + n16, k = 4 * kk + kq;
    av[kk] = ra < M && k < M ? Dg[dp * MM + ra * M + k] : 0.0;
  }
  // T, rows 16 rt .. of parity sgf, for the tiles wave and wave + 4
  const int ntm = (s + 15) >> 4;
  double tv[2][5];
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int tile = wave + 4 * j, sgf = tile >= ntm, m = (tile - sgf * ntm) * 16 + n16;
#pragma unroll
    for (int kk = 0; kk < 5; kk++) {
      const int k = 4 * kk + kq;
      tv[j][kk] = tile < 2 * ntm && m < s && k < M ? Tg[((size_t)sgf * s + m) * M + k] : 0.0;
    }
  }
  // the band sums this work-group adds to (nr <= 2 G s <= 8 NT)
  d2 vb[4];
  if (ORDER == LINES_RAW || es == 1) {
    const __amdgpu_buffer_rsrc_t r =
        line_rsrc(ORDER == LINES_RAW ? raw + (size_t)w.line * N + row0 : dst, nr);
#pragma unroll
    for (int q = 0; q < 4; q++) vb[q] = load_pair(r, 16 * tid + 4096 * q, 0);
  } else {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int e = 2 * (tid + kFarNT * q);
      vb[q].x = dst[(size_t)std::min(e, nr - 1) * es];
      vb[q].y = dst[(size_t)std::min(e + 1, nr - 1) * es];
    }
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int q = 0; q < QM; q++) {
    const int slot = (4 * q + wave) * 3 + sl;
    if (lane < 54 && slot < nslot) *reinterpret_cast<d2 *>(mres + slot * M2 + 2 * o2) = vm[q];
  }
  for (int s0 = (4 * QM + wave) * 3; s0 < nslot; s0 += 12) {  // (more than 48 slots)
    bool ok;
    const size_t c = slot_of(s0 + sl, ok);
    if (lane < 54 && s0 + sl < nslot) {
      const d2 z = {0.0, 0.0};
      *reinterpret_cast<d2 *>(mres + (s0 + sl) * M2 + 2 * o2) =
          ok ? *reinterpret_cast<const d2 *>(m2l + c * M2 + 2 * o2) : z;
    }
  }
  lds_sync();

  // ---- the subtree root: m2l_ld + sum_lev Q(ld - lev, .) m2l_lev
  for (int t0 = 0; t0 < nq; t0 += kFarNT / 2) {
    const int task = t0 + (tid >> 1);
    if (t0 > 0) {
      const double *qrow = qrow_ptr(Qg, g, Rr, std::min(task, nq - 1), M) + half * 9 * M;
#pragma unroll
      for (int l = 0; l < 9; l++) qr[l] = qrow[l * M];
    }
    const int lev = std::min(task, nq - 1) / M, k = std::min(task, nq - 1) - lev * M;
    const double *mv = mres + lev * M2 + 9 * half;
    double o0 = 0, o1 = 0;
#pragma unroll
    for (int l = 0; l < 9; l++) {
      o0 += qr[l] * mv[l];
      o1 += qr[l] * mv[M + l];
    }
    o0 += __shfl_xor(o0, 1, 64);
    o1 += __shfl_xor(o1, 1, 64);
    if (task < nq) qp[lev * M2 + half * M + k] = half ? o1 : o0;
  }
  lds_sync();
  if (tid < M2) {
    double v = mres[g.ld * M2 + tid];
    for (int lev = 0; lev < g.ld; lev++) v += qp[lev * M2 + tid];
    cres[tid] = v;
  }
  lds_sync();

  // ---- levels ld+1..ld+gd on v_mfma_f64_16x16x4f64: children of parity p are
  // C (M x n) = D(p) (M x M) C_parents (M x n), n = 2^lam children x 2
  // parities <= 16 columns: column j = child 2(j >> 1) + p, parity j & 1
  for (int lam = 1; lam <= g.gd; lam++) {
    const int n = 1 << lam, b0 = n - 1, bp = (n >> 1) - 1, j = n16;
    double bv[5], add[4];
#pragma unroll
    for (int kk = 0; kk < 5; kk++) {
      const int k = 4 * kk + kq;
      bv[kk] = j < n && k < M ? cres[(bp + (j >> 1)) * M2 + (j & 1) * M + k] : 0.0;
    }
    const int c = 2 * (j >> 1) + dp, o = (b0 + c) * M2 + (j & 1) * M + drt * 16 + kq;
    const int nv = drt == 0 ? 4 : (kq < M - 16 ? 1 : 0);  // rows drt 16 + kq + 4 v < M
#pragma unroll
    for (int v = 0; v < 4; v++) add[v] = j < n && v < nv ? mres[g.ld * M2 + o + 4 * v] : 0.0;
    d4 D0 = {0, 0, 0, 0}, D1 = {0, 0, 0, 0};
    D0 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[0], bv[0], D0, 0, 0, 0);
    D1 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[1], bv[1], D1, 0, 0, 0);
    D0 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[2], bv[2], D0, 0, 0, 0);
    D1 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[3], bv[3], D1, 0, 0, 0);
    D0 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[4], bv[4], D0, 0, 0, 0);
    D0 += D1;
    const bool valid = ((size_t)Rr << lam) + c < ((size_t)4 << (g.ld + lam)) - 2;
#pragma unroll
    for (int v = 0; v < 4; v++)
      if (j < n && v < nv) cres[o + 4 * v] = valid ? D0[v] + add[v] : 0.0;
    lds_sync();
  }

  // ---- far field F_par^T (G x s) = C_par^T (G x M) T_par^T (M x s)
#pragma unroll
  for (int t = 0; t < 2; t++) {
    const int tile = wave + 4 * t, sgf = tile >= ntm, rt = tile - sgf * ntm;
    if (tile >= 2 * ntm) continue;
    double cv[5];
#pragma unroll
    for (int kk = 0; kk < 5; kk++) {
      const int k = 4 * kk + kq;
      cv[kk] = n16 < G && k < M ? cres[(G - 1 + n16) * M2 + sgf * M + k] : 0.0;
    }
    d4 D = {0, 0, 0, 0};
#pragma unroll
    for (int kk = 0; kk < 5; kk++) D = __builtin_amdgcn_mfma_f64_16x16x4f64(cv[kk], tv[t][kk], D, 0, 0, 0);
    const int m = rt * 16 + n16;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int leaf = kq + 4 * v;
      if (leaf < G && m < s) ob[leaf * ly.CS + 2 * m + sgf] = D[v];
    }
  }
  lds_sync();
  // ---- the band sums plus the far field, scaled
  const unsigned inv = ((1u << 20) + s - 1) / s;
  const bool even = (s & 1) == 0;
  auto scaled = [&](double v, int e) {
    const size_t i = row0 + e;
    if (dir == C2L) return v * ((double)i + 0.5);
    return i == 0 ? v * k2Pi * 0.5 : v * k2Pi;
  };
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int h = tid + kFarNT * q, e = 2 * h;
    if (e >= nr) continue;
    const double *o = ob + e + (even ? 2 * (int)(__umul24(h, inv) >> 20) : 0);
    const d2 v = {scaled(vb[q].x + o[0], e), scaled(vb[q].y + o[1], e + 1)};
    if (es == 1) {
      store_pair(v, line_rsrc(dst, nr), 16 * h);
    } else {
      dst[(size_t)e * es] = v.x;
      if (e + 1 < nr) dst[(size_t)(e + 1) * es] = v.y;
    }
  }
}

// ---------------------------------------------------------------------------
// direct O(N^2) sums, one row per thread (src/C/leg2cheb.c:152-234).  Grid
// (row blocks, ly, lz): line = blockIdx.z * ly + blockIdx.y, so any number of
// lines runs in one launch (ly <= 65535, the grid's y limit).
__global__ void __launch_bounds__(256) k_direct(const double *__restrict__ in,
                                                double *__restrict__ out, LineMap lm, int N,
                                                int dir, const double *__restrict__ a,
                                                const double *__restrict__ an,
                                                const double *__restrict__ dn, size_t nlines) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t line = (size_t)blockIdx.z * gridDim.y + blockIdx.y;
  if (line >= nlines) return;
  N = line_len(lm, line, N);  // this line's length (tables cover the plan's N)
  if (i >= N) return;
  const size_t off = line_off(lm, line);
  const double *u = in + off;
  const size_t es = lm.es;
  double acc = 0;
  if (dir == L2C) {
    for (int n = 0; n + i < N; n += 2) acc += a[n / 2] * k2Pi * a[n / 2 + i] * u[(size_t)(n + i) * es];
    if (i == 0) acc /= 2;
  } else {
    const double vi = i == 0 ? u[0] : u[(size_t)i * es] * (double)i;
    acc = kSqrtPi * vi * an[i];
    for (int n = 2; n + i < N; n += 2)
      acc -= dn[n / 2] * an[n / 2 + i] * (u[(size_t)(n + i) * es] * (double)(n + i));
    acc *= ((double)i + 0.5);
  }
  out[off + (size_t)i * es] = acc;
}

// k_direct with one wave per output row, for single transforms of larger N
// (one thread per row leaves a few dozen waves, each a serial loop of N/2
// terms): the wave's lanes take every 64th term of the row, in the same
// term order per lane, and add their partial sums across the wave.  Grid
// ((N + 3) / 4, lines): four rows per work-group, line blockIdx.y of lm
// (unpacked maps).
template <int dir, int QR>
__global__ void __launch_bounds__(256) k_direct_rows(const double *__restrict__ in,
                                                     double *__restrict__ out, LineMap lm, int N,
                                                     const double *__restrict__ a,
                                                     const double *__restrict__ an,
                                                     const double *__restrict__ dn) {
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= N) return;  // whole waves: the row index is wave-uniform
  const size_t off = line_off(lm, blockIdx.y);
  const double *u = in + off;
  const size_t es = lm.es;
  // QR terms' loads in flight at once (a term past the end reads the lane's
  // first one and adds nothing), and what the C2L diagonal needs before them.
  // One line (three, a few waves on each SIMD: latency): 1500 4.0 us against 4.25 with
  // one at a time, 2200 5.0 / 5.2, 3072 6.6 / 6.8; four waste more of a row's last
  // batch (2200 5.45, 1000 3.65 / 3.55, though 2500 5.55 / 5.65).  Several lines (one:
  // issue): 30 of 300 4.4 us against 5.8 with four, 2 of 1800 5.7 / 6.6, 8 of 1000 side
  // by side 11.9 / 12.9.
  double ud = 0, pd = 0;
  if (dir == C2L) {
    ud = u[(size_t)i * es];
    pd = an[i];
  }
  const double *Ht = dir == L2C ? a : dn, *Pt = dir == L2C ? a : an;
  double acc = 0;
  for (int k0 = lane + (dir == L2C ? 0 : 1); 2 * k0 + i < N; k0 += 64 * QR) {
    double h[QR], p[QR], x[QR];
#pragma unroll
    for (int q = 0; q < QR; q++) {
      const int k = 2 * (k0 + 64 * q) + i < N ? k0 + 64 * q : k0;
      h[q] = Ht[k];
      p[q] = Pt[k + i];
      x[q] = u[(size_t)(2 * k + i) * es];
    }
#pragma unroll
    for (int q = 0; q < QR; q++) {
      const int n = 2 * (k0 + 64 * q);
      const double t = dir == L2C ? h[q] * k2Pi * p[q] * x[q]
                                  : -(h[q] * p[q] * (x[q] * (double)(n + i)));
      if (n + i < N) acc += t;
    }
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) acc += __shfl_xor(acc, d, 64);
  if (lane == 0) {
    if (dir == L2C) {
      if (i == 0) acc /= 2;
    } else {
      const double vi = i == 0 ? ud : ud * (double)i;
      acc = (kSqrtPi * vi * pd + acc) * ((double)i + 0.5);
    }
    out[off + (size_t)i * es] = acc;
  }
}

// ---------------------------------------------------------------------------
// Direct sums of single transforms (and of line calls of a few lines, one
// line per grid.z) of N above 3072 with the band's register rings
// (src/C/leg2cheb.c:152-234).  Per parity sg the rows r and columns m
// (element 2m + sg) run over [0, R), R = (N - sg + 1) / 2, and
//   y_r = sum_{m >= r} H(m - r) P(m + r + sg) X(m)
// with H = P = Lambda, X = u (L2C), or H = dn (H(0) = 0: the diagonal is
// added after the sum), P = an, X(m) = u_n n (C2L).  A work-group of four
// waves owns 8 G rows of one parity (G groups of 8 rows, 4 / G waves each)
// and stages X, P and H for the columns its rows touch in LDS, in chunks of
// kDbChunk columns (one chunk up to N = 8192); per chunk, lane j of
// the wave for part c of group g takes the columns t = m - r0 in
// [(64c + j) T, (64c + j + 1) T) of the group's 8 rows, T a multiple of 8
// with T/8 odd or two; the 64 lanes' sums are added across the wave, then the
// parts through LDS.  Every window stores index e at e + e/8, so the 64
// lanes' addresses (64 segments of T/8 padded blocks apart) fall in distinct
// banks.  G = 1 (8 rows, four parts) while two work-groups' windows fit a
// CU, else G = 4 (32 rows, one part).  Kernel trace (us), G = 1 / 2 / 4: N =
// 3500 6.4 / 6.4 / 7.0, 4096 7.1 / 7.4 / 7.7, 6000 15.6 / 10.2 / 9.8, 8192
// 20.9 / 12.7 / 11.0 (from 6000 on one work-group per CU: G = 1 then takes
// two rounds, and more rows per work-group load the windows fewer times).
constexpr int kDirectBandMinN = 3072;
// columns per LDS window load: a work-group whose rows touch more columns
// runs them in chunks of this many, the windows reloaded for each
constexpr int kDbChunk = 4096;
__host__ __device__ inline int dband_win(int cols) { return cols + 128; }
__host__ __device__ inline int dband_pad(int e) { return e + (e >> 3); }
size_t dband_shared_bytes(int N) {
  const int w = dband_pad(dband_win(std::min((N + 1) / 2, kDbChunk))) + 1;
  return 8 * (size_t)(3 * w + 24);  // windows, the other parts' row sums (G = 1)
}
// Entries per thread and batch of the window loads: nine where that saves the
// first work-groups a batch (N = 4096 7.0 -> 6.3 us a call, 8192 10.9 -> 10.4), else
// eight (nine: 5000 8.6 -> 8.8, 7000 9.0 -> 9.3)
inline int dband_batch(int N) {
  if ((N + 1) / 2 > kDbChunk) return 8;
  const int w = dband_win((N + 1) / 2);
  return (w + 2303) / 2304 < (w + 2047) / 2048 ? 9 : 8;
}
// G = 1 while two work-groups' windows fit one CU's 160 KB of LDS, else 4
inline int dband_groups(int N) { return dband_shared_bytes(N) <= 80 * 1024 ? 1 : 4; }

// Columns [t0, t1) of the lane's 8 rows, t0 a multiple of 8; xq, pq, hq: the
// padded blocks of X(r0 + t0), P(2 r0 + sg + t0), H(t0), the block before
// hq holding H(t0 - 8 .. t0 - 1) (zero below 0).  Columns t >= len read X as
// zero.  Rings as in band_seg8: slot t mod 8 holds H(t - 8 .. t)
// and P(t .. t + 7); row rho of column t takes H(t - rho) P(t + rho) X(t).
__device__ __forceinline__ void direct_seg8(const double *__restrict__ xq,
                                            const double *__restrict__ pq,
                                            const double *__restrict__ hq, int t0, int t1,
                                            int len, double acc[8]) {
  const int ntrip = t1 > t0 ? (t1 - t0 + 7) >> 3 : 0;
  if (ntrip == 0) return;
  double hr[8], pr[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    hr[k] = hq[k - 9];
    pr[k] = pq[k];
  }
  int tt = t0;
  double XA[4], PA[4], HA[4], XB[4], PB[4], HB[4];
#define DFETCH(X, P, H, HALF)                                       \
  _Pragma("unroll") for (int k_ = 0; k_ < 4; k_++) {                \
    X[k_] = tt + 4 * (HALF) + k_ < len ? xq[4 * (HALF) + k_] : 0.0; \
    P[k_] = pq[9 + 4 * (HALF) + k_];                                \
    H[k_] = hq[4 * (HALF) + k_];                                    \
  }
#define DSTEP(K, X, P, H, J)                                          \
  {                                                                   \
    hr[K] = H[J];                                                     \
    const double x_ = X[J];                                           \
    _Pragma("unroll") for (int r_ = 0; r_ < 8; r_++)                  \
      acc[r_] += (hr[((K) - r_) & 7] * pr[((K) + r_) & 7]) * x_;      \
    pr[K] = P[J];                                                     \
  }
  DFETCH(XA, PA, HA, 0)
  for (int b = 0; b < ntrip; b++) {
    DFETCH(XB, PB, HB, 1)
    DSTEP(0, XA, PA, HA, 0) DSTEP(1, XA, PA, HA, 1) DSTEP(2, XA, PA, HA, 2) DSTEP(3, XA, PA, HA, 3)
    xq += 9;
    pq += 9;
    hq += 9;
    tt += 8;
    DFETCH(XA, PA, HA, 0)
    DSTEP(4, XB, PB, HB, 0) DSTEP(5, XB, PB, HB, 1) DSTEP(6, XB, PB, HB, 2) DSTEP(7, XB, PB, HB, 3)
  }
#undef DSTEP
#undef DFETCH
}

// Grid ((R0 + 8 G - 1) / (8 G), 2, lines) with R0 = (N + 1) / 2, 256
// threads, dband_shared_bytes(N) of LDS; line blockIdx.z of lm (unpacked
// maps).
template <int DIR, int G, int QF>
__global__ void __launch_bounds__(256) k_direct_band(const double *__restrict__ in,
                                                     double *__restrict__ out, LineMap lm, int N,
                                                     const double *__restrict__ a,
                                                     const double *__restrict__ an,
                                                     const double *__restrict__ dn) {
  extern __shared__ double sm[];
  const int sg = blockIdx.y;
  const int R = (N - sg + 1) / 2;
  static_assert(G == 1 || G == 4, "row groups per work-group");
  constexpr int NP = 4 / G;  // parts of each group's columns
  const int Rb = blockIdx.x * 8 * G;
  if (Rb >= R) return;  // the whole work-group
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int span = R - Rb;  // columns Rb .. R - 1
  const int nch = (span + kDbChunk - 1) / kDbChunk;  // column chunks
  const int W = dband_win(std::min(span, kDbChunk)), WP = dband_pad(W) + 1;
  double *xw = sm, *pw = sm + WP, *hw = sm + 2 * WP;
  const size_t off = line_off(lm, blockIdx.z);
  const double *u = in + off;
  const size_t es = lm.es;
  const double *Ht = DIR == 0 ? a : dn;
  const double *Pt = DIR == 0 ? a : an;
  const int nH = DIR == 0 ? N : (N + 1) / 2;  // entries of the H table
  const int g = wave % G, c = wave / G;  // row group, column part
  const int r0 = Rb + 8 * g;
  const bool live = r0 < R;  // (every wave reaches the barriers below)
  const int len = live ? R - r0 : 0;
  double acc[8];
#pragma unroll
  for (int k = 0; k < 8; k++) acc[k] = 0.0;
  for (int ch = 0; ch < nch; ch++) {
    // columns t = m - r0 in [tb, tb + kDbChunk): windows X(Rb + tb + e),
    // P(2 Rb + sg + tb + e), H(tb - 8 + e), e < W, in batches of QF
    // entries per thread, the batch's loads issued before its stores (one
    // entry per trip: 8.6 against 8.2 us at N = 4096; QF = 16 takes 174
    // VGPRs and was slower still)
    const int tb = ch * kDbChunk;
    for (int e0 = tid; e0 < W; e0 += QF * 256) {
      double vx[QF], vp[QF], vh[QF];
#pragma unroll
      for (int k = 0; k < QF; k++) {
        const int e = e0 + k * 256;
        const int m = Rb + tb + e, qi = 2 * Rb + sg + tb + e, hk = tb - 8 + e;
        vx[k] = m < R ? u[(size_t)(2 * m + sg) * es] : 0.0;
        vp[k] = qi < N ? Pt[qi] : 0.0;
        vh[k] = (hk >= 0 && hk < span && hk < nH && !(DIR == 1 && hk == 0)) ? Ht[hk] : 0.0;
      }
#pragma unroll
      for (int k = 0; k < QF; k++) {
        const int e = e0 + k * 256;
        if (e < W) {
          const int pe = dband_pad(e);
          xw[pe] = DIR == 1 ? vx[k] * (double)(2 * (Rb + tb + e) + sg) : vx[k];
          pw[pe] = vp[k];
          hw[pe] = vh[k];
        }
      }
    }
    __syncthreads();
    const int cw = std::min(kDbChunk, span - tb);
    int T8 = (cw + 512 * NP - 1) / (512 * NP);
    // (two: pairs of lanes share a bank, but a trip less than three: N = 4500 8.2 ->
    // 7.7 us)
    if (NP == 1 || T8 != 2) T8 |= 1;
    const int T = 8 * T8;
    const int t0 = tb + (64 * c + lane) * T;
    const int t1 = std::min(std::min(t0 + T, tb + kDbChunk), len);
    if (t0 < t1)  // false for every lane of a wave past the last row
      direct_seg8(xw + dband_pad(8 * g + t0 - tb), pw + dband_pad(16 * g + t0 - tb),
                  hw + dband_pad(t0 - tb + 8), t0, t1, len, acc);
    if (ch + 1 < nch) __syncthreads();  // the next chunk's loads overwrite the windows
  }
  // the 64 lanes' sums of the 8 rows, halving the rows at each of the
  // first three exchanges (lanes with bit 5 set keep rows 4-7, bit 4 the
  // upper two of those four, bit 3 the upper one): 10 exchanges instead of
  // 48, and lane l ends with row l >> 3
  const bool b5 = lane & 32, b4 = lane & 16, b3 = lane & 8;
  double k4[4], k2[2];
#pragma unroll
  for (int j = 0; j < 4; j++)
    k4[j] = (b5 ? acc[j + 4] : acc[j]) + __shfl_xor(b5 ? acc[j] : acc[j + 4], 32, 64);
#pragma unroll
  for (int j = 0; j < 2; j++)
    k2[j] = (b4 ? k4[j + 2] : k4[j]) + __shfl_xor(b4 ? k4[j] : k4[j + 2], 16, 64);
  double v = (b3 ? k2[1] : k2[0]) + __shfl_xor(b3 ? k2[0] : k2[1], 8, 64);
#pragma unroll
  for (int d = 4; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  if constexpr (NP > 1) {
    double *red = sm + 3 * WP;  // [part - 1][group][row]: the other parts' sums
    if (c > 0 && (lane & 7) == 0) red[(c - 1) * 8 * G + 8 * g + (lane >> 3)] = v;
    __syncthreads();
    if (c == 0 && (lane & 7) == 0) {
#pragma unroll
      for (int q = 1; q < NP; q++) v += red[(q - 1) * 8 * G + 8 * g + (lane >> 3)];
    }
  }
  if (c != 0 || !live) return;
  const int r = r0 + (lane >> 3);
  if ((lane & 7) == 0 && r < R) {
    const int i = 2 * r + sg;
    if (DIR == 0) {
      v *= k2Pi;
      if (i == 0) v *= 0.5;
    } else {
      const double vi = i == 0 ? u[0] : u[(size_t)i * es] * (double)i;
      v = (kSqrtPi * vi * an[i] - v) * ((double)i + 0.5);
    }
    out[off + (size_t)i * es] = v;
  }
}

// ---------------------------------------------------------------------------
// Batched lines of the direct path (N <= kDenseMaxN) as dense products on FP64
// MFMA: per parity p, OUT_p (NPP x LT) = K_p (NPP x NPP) IN_p (NPP x LT) for a
// tile of LT lines, K_p upper triangular (the direct sums of
// src/C/leg2cheb.c:152-234 with scaling and C2L weights folded in).
//
// A work-group holds whole lines in LDS [parity][line][c] and every row tile
// of their outputs, so each element is read and written once, and K (NPP <=
// 16 NRM) stays in registers: a wave has a parity and the row tiles w and
// NR-1-w, so that every wave runs the same 4 (NR + 1) k-steps of
// v_mfma_f64_16x16x4f64.  The work-groups stay and walk the line tiles, the
// next tile's inputs in flight in registers during the current one's
// products: HBM-bound.  Row stride 16 NRM + 2 doubles: the writes of contiguous
// lines and the operand reads fall in distinct banks.
//   CONTIG (unit element stride): both parities (NP = 2) of a column move as
//   one 16-byte access, through buffer descriptors of the lines' lengths
//   (reads past the end return zero, writes past it are dropped).
//   Strided lines move 32 lines of one element per half-wave, and their
//   results leave the accumulators as they are (16 lines of one element per
//   store); wide lines then take one parity per work-group (NP = 1), which
//   costs them nothing and leaves three work-groups, out of step with each
//   other, to a CU.
// 65,536 lines, contiguous / strided (us): N = 256 57.5 / 57.7 (4.7 TB/s of
// the 4.9 that a large copy reaches), 160 37.7 / 38.9, 128 24.7 / 24.8 (5.4
// TB/s), 64 17.1 / 13.5; before, one parity after the other through one tile
// with K from L2 for each of them, 83.8 / 71.6, 55.1 / 48.2, 45.6 / 40.8,
// 29.2 / 23.8.  Not staying on the CU (512 threads, K from L2): N = 256
// strided 85.3; staying with both parities of 32 strided lines in one
// work-group of eight waves per CU: 82.6 (its loads, products and stores take
// turns).
template <bool CONTIG, int NRM, int LT, int NP>
__global__ void __launch_bounds__(32 * NRM * NP)
    __attribute__((amdgpu_waves_per_eu(CONTIG && NRM == 8 ? 4 : 3)))
    k_lines_dense(const double *__restrict__ in, double *__restrict__ out, LineMap lm,
                  size_t nlines, int N, int NPP, const double *__restrict__ K) {
  extern __shared__ double sm[];
  constexpr int NW = NRM / 2 * NP, NH = LT / 16;  // waves, 16-line halves
  static_assert(CONTIG ? NP == 2 : LT == 32, "line moves below");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const size_t es = CONTIG ? 1 : lm.es;
  constexpr int KP = 16 * NRM + 2;
  // work items: line tiles, per parity when NP = 1
  const unsigned nitem = (unsigned)((nlines + LT - 1) / LT) * (3 - NP);
  // NP = 1: the grid is even, so a work-group keeps its parity
  const int p = NP == 2 ? wave & 1 : blockIdx.x & 1;
  // start and length of an item's lines (line_off divides), of this item, the
  // next and the one after
  size_t *toff = (size_t *)(sm + NP * LT * KP);
  int *tlen = (int *)(toff + 3 * LT);
  auto offsets = [&](unsigned t, int slot) {
    if (tid >= LT || t >= nitem) return;
    const size_t line = (size_t)(NP == 2 ? t : t >> 1) * LT + tid;
    toff[slot * LT + tid] = line < nlines ? line_off(lm, line) : 0;
    tlen[slot * LT + tid] = line < nlines ? line_len(lm, line, N) : 0;
  };
  unsigned item = blockIdx.x;
  offsets(item, 0);
  offsets(item + gridDim.x, 1);
  const int NR = NPP >> 4, nkt = NPP >> 2;
  // row tiles R0 and R1 of NRM; groups of four k-steps (one 16-column tile):
  // NRM - R0 of R0, then NRM - R1 of R1, columns from the diagonal on.  Tiles
  // past NR read as zero.
  const int R0 = NP == 2 ? wave >> 1 : wave, R1 = NRM - 1 - R0;
  constexpr int NG = NRM + 1;
  double a[NG][4];
  const __amdgpu_buffer_rsrc_t Kr = line_rsrc(K + (size_t)p * NR * nkt * 64, NR * nkt * 64);
#pragma unroll
  for (int g = 0; g < NG; g++) {
    const int row = g < NRM - R0 ? R0 : R1, col = g < NRM - R0 ? R0 + g : R1 + g - (NRM - R0);
    const int base = col < NR ? row * nkt + 4 * col : NR * nkt;
#pragma unroll
    for (int kk = 0; kk < 4; kk++) a[g][kk] = load_one(Kr, 8 * lane + 512 * kk, base * 512);
  }
  // moves of a thread: CONTIG line wave + NW (q / QH), pair lane + 64 (q %
  // QH); else column c0 + cs q (and the half-wave's own parity when NP = 2)
  // of line lane % 32
  constexpr int QH = NRM == 8 ? 2 : 1, QL = LT / NW * QH;
  constexpr int NE = CONTIG ? 2 * QL : 16;
  const int c0 = NP == 2 ? wave : 2 * wave + (lane >> 5);
  constexpr int cs = NP == 2 ? NW : 2 * NW;
  const int i0 = 2 * c0 + (NP == 2 ? lane >> 5 : p);
  double e[NE];
  // buffer descriptor of line l of an item
  auto rsrc = [&](const double *base, int slot, int l) {
    const size_t o = toff[slot * LT + l];
    const size_t ou = (size_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)o) |
                      ((size_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(o >> 32)) << 32);
    return line_rsrc(base + ou, __builtin_amdgcn_readfirstlane(tlen[slot * LT + l]));
  };
  auto fetch = [&](int slot) {
    if constexpr (CONTIG) {
#pragma unroll
      for (int q = 0; q < QL; q++) {
        const d2 t = load_pair(rsrc(in, slot, wave + NW * (q / QH)), 16 * lane + 1024 * (q % QH), 0);
        e[2 * q] = t.x;
        e[2 * q + 1] = t.y;
      }
    } else {
      // (a line past nlines reads line 0 and stores nothing).  One running
      // address: the empty asm keeps the compiler from holding all sixteen
      // steps through the item loop.
      const double *line = in + toff[slot * LT + (lane & 31)], *src = line + (size_t)i0 * es;
      size_t step = 2 * cs * es;
      asm volatile("" : "+s"(step));
      if (N == 32 * NRM) {
#pragma unroll
        for (int q = 0; q < NE; q++, src += step) e[q] = *src;
      } else {
#pragma unroll
        for (int q = 0; q < NE; q++, src += step) {
          const bool ok = i0 + 2 * cs * q < N;
          const double v = *(ok ? src : line);
          e[q] = ok ? v : 0.0;
        }
      }
    }
  };
  auto stage = [&]() {
    if constexpr (CONTIG) {
#pragma unroll
      for (int q = 0; q < QL; q++) {
        const int l = wave + NW * (q / QH), c = lane + 64 * (q % QH);
        if (64 * QH <= 16 * NRM || c < 16 * NRM) {
          sm[l * KP + c] = e[2 * q];
          sm[(LT + l) * KP + c] = e[2 * q + 1];
        }
      }
    } else {
      double *o = sm + ((NP == 2 ? lane >> 5 : 0) * LT + (lane & 31)) * KP + c0;
#pragma unroll
      for (int q = 0; q < NE; q++)
        o[cs * q] = e[q];
    }
  };
  __syncthreads();
  fetch(0);
  stage();
  const d4 z = {0.0, 0.0, 0.0, 0.0};
  double *const mine = sm + ((NP == 2 ? p * LT : 0) + (lane & 15)) * KP + (lane >> 4);
  for (int slot = 0; item < nitem; item += gridDim.x) {
    const int nslot = slot == 2 ? 0 : slot + 1;
    const bool more = item + gridDim.x < nitem;
    __syncthreads();
    if (more) fetch(nslot);
    offsets(item + 2 * gridDim.x, nslot == 2 ? 0 : nslot + 1);
    d4 D[2][NH];  // [row tile][16-line half]
    // (the empty asm keeps the compiler from holding the tests of all four row tile
    // pairs through the item loop: 22 scalars and two vector registers spilled)
    int nr = NR;
    asm volatile("" : "+s"(nr));
    auto products = [&](auto r0) {
      constexpr int r = decltype(r0)::value;
#pragma unroll
      for (int h = 0; h < NH; h++) D[0][h] = D[1][h] = z;
#pragma unroll
      for (int g = 0; g < NG; g++) {
        constexpr int n0 = NRM - r;
        const int col = g < n0 ? r + g : NRM - 1 - r + g - n0;
        if (col >= nr) continue;
        const double *b = mine + 16 * col;
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
          for (int h = 0; h < NH; h++) {
            d4 &d = D[g < n0 ? 0 : 1][h];
            d = __builtin_amdgcn_mfma_f64_16x16x4f64(a[g][kk], b[16 * h * KP + 4 * kk], d, 0, 0, 0);
          }
      }
    };
    constexpr int top = NRM / 2 - 1;  // (waves have R0 <= top)
    if (R0 == 0)
      products(std::integral_constant<int, 0>{});
    else if (R0 == 1)
      products(std::integral_constant<int, std::min(1, top)>{});
    else if (R0 == 2)
      products(std::integral_constant<int, std::min(2, top)>{});
    else
      products(std::integral_constant<int, top>{});
    if constexpr (CONTIG) {
      __syncthreads();  // every wave is done with the input tile
#pragma unroll
      for (int j = 0; j < 2; j++) {
        double *o = mine + 16 * (j ? R1 : R0);
#pragma unroll
        for (int h = 0; h < NH; h++)
#pragma unroll
          for (int v = 0; v < 4; v++) o[16 * h * KP + 4 * v] = D[j][h][v];
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < QL; q++) {
        const int l = wave + NW * (q / QH), c = std::min(lane + 64 * (q % QH), 16 * NRM - 1);
        const d2 t = {sm[l * KP + c], sm[(LT + l) * KP + c]};
        store_pair(t, rsrc(out, slot, l), 16 * lane + 1024 * (q % QH));
      }
    } else {
#pragma unroll
      for (int h = 0; h < NH; h++) {
        const int l = 16 * h + (lane & 15), len = tlen[slot * LT + l];
        size_t step = 8 * es;
        asm volatile("" : "+s"(step));
#pragma unroll
        for (int j = 0; j < 2; j++) {
          const int r0 = 2 * (16 * (j ? R1 : R0) + (lane >> 4)) + p;
          double *dst = out + toff[slot * LT + l] + (size_t)r0 * es;
#pragma unroll
          for (int v = 0; v < 4; v++, dst += step)
            if (r0 + 8 * v < len) *dst = D[j][h][v];
        }
      }
    }
    __syncthreads();  // the tile is free for the next one
    if (more) stage();
    slot = nslot;
  }
}

// the tile [NP][LT][16 NRM + 2], then three items' offsets (size_t) and
// lengths (int)
static size_t dense_shared_bytes(int NRM, int LT, int NP) {
  return 8 * (size_t)NP * LT * (16 * NRM + 2) + 3 * LT * (sizeof(size_t) + sizeof(int));
}

// Batched lines of the direct path with kDenseMaxN < N <= kGemmMaxN: the same
// parity blocks K_p (NPP up to 2048) as a tiled product on FP64 MFMA.  A
// work-group owns 32 pair-rows of both parities for 32 lines (wave: parity
// wave & 1, 16-row tile wave >> 1, two 16-line column tiles) and walks the
// columns c >= its first row in chunks of 64 pairs: the chunk's inputs
// 2c, 2c + 1 of its 32 lines are staged in LDS [parity][line][c], then each
// wave runs v_mfma_f64_16x16x4f64 with A = K_p fragments (global memory,
// L2/MALL-resident) and B = the staged rows.  The next chunk's inputs and
// fragments load into registers during the current chunk's products.
// LDS row stride KC + 2 = 66 doubles: the writes of contiguous lines (lanes
// along c) and the operand reads (16 lines x 2 columns per half-wave, 132
// dwords apart) fall in distinct banks.
// Contiguous lines move both parities of a column as one 16-byte access;
// strided ones 32 lines of one element per half-wave, and their results go
// out of the accumulators as they are (16 lines of one element per store).
// Grid (line tiles, row tiles): the long row tiles are dispatched first, and
// consecutive work-groups share a row tile's K rows.
// Bound by the matrix cores on large calls (4096 lines of 1024 41 TFLOP/s,
// 2048 lines of 3000 54 TFLOP/s of the 72 that a large FP64 product reaches;
// L2 carries 64 KB of fragments and inputs per 128 products of a wave), by
// the chain of chunks, about 1.4 us each, on small ones.  One parity per
// work-group of 64 rows, inputs [c][line] at stride 33 with lanes along c for
// strided lines too, masked fragment loads, measured before it: 1024 lines of
// 1024 24.0 -> 19.4 us, 4096 lines of 2048 212 -> 177, 32 lines of 2048 35 ->
// 27.  Splitting a tile's columns over two or four groups of waves: 4 lines of
// 2048 26 -> 24 us, but 1024 lines of 1024 19.4 -> 20.5 and 25.5.
// Chunks from the last to the diagonal's instead of upwards: a 1200 x 900 array
// through both axes and back 111 -> 96 us (the prefetch behind the last chunk
// falls on lines just read; 97 with the test for NaN and Inf), 2-norm error at N = 2000 3.2-4.6e-16 ->
// 1.7-2.8e-16 (the FMM of the same lines 2.3-7.3e-16).
constexpr int kGemmRT = 32, kGemmLT = 32, kGemmKC = 64, kGemmNT = 256, kGemmKP = kGemmKC + 2;
// The work of tile (bx, by) of the tiled dense product (grid (line tiles,
// row tiles)); k_lines_gemm runs one grid of them, k_lines_gemm_multi the
// grids of several size classes in one launch.
template <bool CONTIG>
__device__ __forceinline__ void lines_gemm_tile(const double *__restrict__ in,
                                                double *__restrict__ out, const LineMap &lm,
                                                size_t nlines, int N, int NPP,
                                                const double *__restrict__ K, unsigned bx,
                                                unsigned by, double *sm) {
  constexpr int KP = kGemmKP, KC = kGemmKC, LT = kGemmLT;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rt = (int)by, p = wave & 1;
  const size_t l0 = (size_t)bx * LT;
  size_t *toff = (size_t *)(sm + 2 * LT * KP);
  int *tlen = (int *)(toff + LT), *flag = tlen + LT;
  if (tid == 0) *flag = 0;
  if (tid < LT) {
    const size_t line = l0 + tid;
    toff[tid] = line < nlines ? line_off(lm, line) : 0;
    tlen[tid] = line < nlines ? line_len(lm, line, N) : 0;
  }
  __syncthreads();
  const int NR = NPP >> 4, nkt = NPP >> 2, R = 2 * rt + (wave >> 1);
  const bool active = R < NR;  // the last row tile may be partly past NPP
  const size_t es = CONTIG ? 1 : lm.es;
  const d4 z = {0.0, 0.0, 0.0, 0.0};
  // sums of the two 16-line halves: each chunk's own, added to the total, from
  // the last column to the diagonal (K falls off away from it, so the large
  // terms come last; one long chain over up to 1024 columns would lose a digit:
  // 2-norm error against double-double sums at N = 2000 1.3-1.8e-15 in one
  // chain)
  d4 D0 = z, D1 = z;
  const double *Bp = sm + (p * LT + (lane & 15)) * KP + (lane >> 4);
  // the fragments of row tile R (zeros past NPP, and for a row tile past it)
  const __amdgpu_buffer_rsrc_t Kr =
      line_rsrc(K + (size_t)(p * NR + (active ? R : 0)) * nkt * 64, active ? 64 * nkt : 0);
  static_assert(KC == 64 && LT == 32 && kGemmRT == 32 && kGemmNT == 256, "thread maps below");
  // staged inputs of this thread in every chunk.  CONTIG: pair c0 + lane of
  // lines 4 q + wave, read through a buffer descriptor of the line's length
  // (reads past its end return zero); else element 2 (c0 + wave + 4 q) +
  // lane / 32 of line lane % 32 (a line past nlines reads line 0 and stores
  // nothing).
  constexpr int QL = CONTIG ? 8 : 1, QE = 16;
  __amdgpu_buffer_rsrc_t src[QL];
  const double *src0 = nullptr;
  if constexpr (CONTIG) {
#pragma unroll
    for (int q = 0; q < QL; q++) {
      const size_t o = toff[4 * q + wave];
      const size_t ou = (size_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)o) |
                        ((size_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(o >> 32)) << 32);
      src[q] = line_rsrc(in + ou, __builtin_amdgcn_readfirstlane(tlen[4 * q + wave]));
    }
  } else {
    src0 = in + toff[lane & 31] + (size_t)(2 * wave + (lane >> 5)) * es;
  }
  double e[QE], a[KC / 4];
  // the loads of chunk c0 (past NPP: zeros).  The empty asm keeps the
  // compiler from carrying one address register per load through the loop.
  auto fetch_in = [&](int c0) {
    asm volatile("" : "+s"(c0));
    if constexpr (CONTIG) {
#pragma unroll
      for (int q = 0; q < QL; q++) {
        const d2 t = load_pair(src[q], 16 * lane, 16 * c0);
        e[2 * q] = t.x;
        e[2 * q + 1] = t.y;
      }
    } else {
      const double *s0 = src0 + (size_t)(2 * c0) * es;
      if (2 * (c0 + KC) <= N) {
#pragma unroll
        for (int q = 0; q < QE; q++) e[q] = s0[(size_t)(8 * q) * es];
      } else {
        const int i0 = 2 * (c0 + wave) + (lane >> 5);
#pragma unroll
        for (int q = 0; q < QE; q++) e[q] = i0 + 8 * q < N ? s0[(size_t)(8 * q) * es] : 0.0;
      }
    }
  };
  auto fragment = [&](int c0, int ks) { return load_one(Kr, 8 * lane + 512 * (ks & 7), 128 * c0 + 512 * (ks & 8)); };
  const int cf = kGemmRT * rt, cl = cf + (NPP - 1 - cf) / KC * KC;  // first and last chunk
  fetch_in(cl);
#pragma unroll
  for (int ks = 0; ks < KC / 4; ks++) a[ks] = fragment(cl, ks);
  // one k-step: its products, then the same step's fragment of chunk cn
  d4 S0, S1;
  auto step = [&](int ks, int cn) {
    const double *b = Bp + 4 * ks;
    S0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ks], b[0], S0, 0, 0, 0);
    S1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ks], b[16 * KP], S1, 0, 0, 0);
    a[ks] = fragment(cn, ks);
    // (the scheduler would gather the loads and hold both chunks' fragments)
    if (ks & 1) __builtin_amdgcn_sched_barrier(0);
  };
  for (int c0 = cl; c0 >= cf; c0 -= KC) {
    if (c0 == cf) {
      bool bad = false;
#pragma unroll
      for (int q = 0; q < QE; q++) bad |= !__builtin_isfinite(e[q]);
      if (bad) *flag = 1;
    }
    if constexpr (CONTIG) {
#pragma unroll
      for (int q = 0; q < QL; q++) {
        sm[(4 * q + wave) * KP + lane] = e[2 * q];
        sm[(LT + 4 * q + wave) * KP + lane] = e[2 * q + 1];
      }
    } else {
#pragma unroll
      for (int q = 0; q < QE; q++)
        sm[((lane >> 5) * LT + (lane & 31)) * KP + wave + 4 * q] = e[q];
    }
    __syncthreads();
    // the next chunk's inputs load during this chunk's products
    int cn = std::max(c0 - KC, cf);
    fetch_in(cn);
    asm volatile("" : "+s"(cn));
    S0 = S1 = z;
    // a NaN or Inf among the diagonal chunk's inputs: the row tile's diagonal
    // block goes term by term, without the zeros below the diagonal
    const bool slow = c0 == cf && __builtin_amdgcn_readfirstlane(*flag) != 0;
#pragma unroll
    for (int ks = KC / 4 - 1; ks >= 8; ks--) step(ks, cn);
    if (!slow || wave < 2) {
#pragma unroll
      for (int ks = 7; ks >= 4; ks--) step(ks, cn);
    }
    // the tile's second row tile starts 16 columns on (K_p is zero before)
    if (c0 != cf || (wave < 2 && !slow)) {
#pragma unroll
      for (int ks = 3; ks >= 0; ks--) step(ks, cn);
    }
    if (slow) {
      const int cb = 16 * (wave >> 1);
      const double *x = sm + (p * LT + (lane & 15)) * KP + cb;
#pragma unroll 1
      for (int c = 15; c >= 0; c--) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int r = (lane >> 4) + 4 * v;
          if (c >= r) {
            const double k = load_one(Kr, 8 * (16 * (c & 3) + r), 512 * ((cf + cb + c) >> 2));
            S0[v] += k * x[c];
            S1[v] += k * x[16 * KP + c];
          }
        }
      }
    }
    D0 += S0;
    D1 += S1;
    __syncthreads();  // the tile is free for the next chunk
  }
  // results: row 16 (wave >> 1) + lane / 16 + 4 v of the tile, line 16 h +
  // lane % 16
  if constexpr (CONTIG) {
    double *o = sm + (p * LT + (lane & 15)) * KP + 16 * (wave >> 1) + (lane >> 4);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      o[4 * v] = D0[v];
      o[4 * v + 16 * KP] = D1[v];
    }
    __syncthreads();
    // pairs 32 rt + lane % 32 of lines 2 wave + lane / 32 + 8 q
    const int r = lane & 31, i = 2 * (kGemmRT * rt + r);
#pragma unroll
    for (int q = 0; q < LT / 8; q++) {
      const int l = 2 * wave + (lane >> 5) + 8 * q, n = tlen[l];
      double *dst = out + toff[l] + i;
      const d2u t = {sm[l * KP + r], sm[(LT + l) * KP + r]};
      if (i + 1 < n)
        *reinterpret_cast<d2u *>(dst) = t;
      else if (i < n)
        dst[0] = t.x;
    }
  } else {
    const int i0 = 2 * (16 * R + (lane >> 4)) + p;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int l = 16 * h + (lane & 15), n = tlen[l];
      double *dst = out + toff[l];
#pragma unroll
      for (int v = 0; v < 4; v++)
        if (active && i0 + 8 * v < n) dst[(size_t)(i0 + 8 * v) * es] = (h ? D1 : D0)[v];
    }
  }
}

template <bool CONTIG>
__global__ void __launch_bounds__(kGemmNT) __attribute__((amdgpu_waves_per_eu(4)))
    k_lines_gemm(const double *__restrict__ in, double *__restrict__ out, LineMap lm,
                 size_t nlines, int N, int NPP, const double *__restrict__ K) {
  extern __shared__ double sm[];
  lines_gemm_tile<CONTIG>(in, out, lm, nlines, N, NPP, K, blockIdx.x, blockIdx.y, sm);
}

// Several size classes of an uneven batch (packed, unit-stride lines) on the
// tiled dense product in one launch: a flat grid over every class's tiles,
// classes in the order given, each class's tiles row tile by row tile (the
// long row tiles first, as in k_lines_gemm's grid).
struct DenseClass {
  const double *K;
  const size_t *off;
  const int *n;
  size_t nlines;
  int N, NPP;
  unsigned bxs, tiles;  // line tiles; bxs x row tiles
};
constexpr int kMaxDenseClasses = 8;
struct DenseClasses {
  DenseClass c[kMaxDenseClasses];
  int count;
};
__global__ void __launch_bounds__(kGemmNT) __attribute__((amdgpu_waves_per_eu(4)))
    k_lines_gemm_multi(const double *__restrict__ in, double *__restrict__ out, DenseClasses dc) {
  extern __shared__ double sm[];
  unsigned t = blockIdx.x;
  int c = 0;
  while (c + 1 < dc.count && t >= dc.c[c].tiles) t -= dc.c[c++].tiles;
  const DenseClass &d = dc.c[c];
  if (t >= d.tiles) return;
  LineMap lm{1, 0, 0, 1, d.off, d.n};
  lines_gemm_tile<true>(in, out, lm, d.nlines, d.N, d.NPP, d.K, t % d.bxs, t / d.bxs, sm);
}

size_t gemm_shared_bytes() {
  return 8 * 2 * (size_t)kGemmLT * kGemmKP + kGemmLT * (sizeof(size_t) + sizeof(int)) +
         sizeof(int);
}

// One transform by direct sums from the Lambda tables a, an, dn (those of a
// direct plan of size N, or of an FMM plan): k_direct_band for N above
// kDirectBandMinN unless band is false (the plan's direct_band), else
// k_direct_rows.  Kernel trace, L2C, k_direct_band /
// k_direct_rows: N = 1024 5.8 / 3.8 us, 4096 8.2 / 9.7 us, 8192 12.2 /
// 27.8 us (below about 3000 the band kernel's window loads and cross-lane
// sums cost more than the row kernel's loads save).
static void launch_direct_one(Prof *prof, int N, size_t dir, const double *a, const double *an,
                              const double *dn, const double *d_in, double *d_out,
                              const LineMap &lm, hipStream_t st, bool band, unsigned nlines = 1) {
  if (N > kDirectBandMinN && band) {
    const int G = dband_groups(N), rows = 8 * G;
    const dim3 grid((unsigned)(((N + 1) / 2 + rows - 1) / rows), 2, nlines);
    const size_t shm = dband_shared_bytes(N);
    const bool nine = dband_batch(N) == 9;
    auto kernel = G == 1 ? (dir == L2C ? (nine ? k_direct_band<0, 1, 9> : k_direct_band<0, 1, 8>)
                                       : (nine ? k_direct_band<1, 1, 9> : k_direct_band<1, 1, 8>))
                         : (dir == L2C ? (nine ? k_direct_band<0, 4, 9> : k_direct_band<0, 4, 8>)
                                       : (nine ? k_direct_band<1, 4, 9> : k_direct_band<1, 4, 8>));
    launch_k(prof, kernel, grid, 256, shm, st, d_in, d_out, lm, N, a, an, dn);
    return;
  }
  auto kernel = nlines > 1 ? (dir == L2C ? k_direct_rows<L2C, 1> : k_direct_rows<C2L, 1>)
                           : (dir == L2C ? k_direct_rows<L2C, 3> : k_direct_rows<C2L, 3>);
  launch_k(prof, kernel, dim3((unsigned)((N + 3) / 4), nlines), 256, 0, st, d_in, d_out, lm, N, a,
           an, dn);
}

// k_direct over nlines lines of map lm (one launch for any number of lines);
// single transforms from kDirectRowsMinN on take launch_direct_one
constexpr int kDirectRowsMinN = 1024;
static void launch_direct(const direct_plan_s *dp, const double *d_in, double *d_out, size_t dir,
                          const LineMap &lm, size_t nlines, hipStream_t st) {
  const int N = (int)dp->N;
  if (nlines == 1 && N >= kDirectRowsMinN) {
    launch_direct_one(dp->prof, N, dir, dp->d_a, dp->d_an, dp->d_dn, d_in, d_out, lm, st,
                      dp->direct_band);
    return;
  }
  const unsigned gy = (unsigned)std::min<size_t>(nlines, dp->lines_y);
  const unsigned gz = (unsigned)((nlines + gy - 1) / gy);
  launch_k(dp->prof, k_direct, dim3((N + 255) / 256, gy, gz), 256, 0, st, d_in, d_out, lm, N,
      (int)dir, dp->d_a, dp->d_an, dp->d_dn, nlines);
}

// Whether a call of nlines lines through direct plan dp takes the tiled dense
// product (k_lines_gemm): the whole-line kernel has the lower cost per line,
// the tiled one more work-groups for a given call, so above N = 32 the tiled
// kernel takes calls of up to kGemmFewLines lines unless the plan's dense_tile
// says otherwise.  Tiled / whole-line (us, contiguous): N = 256 with 1000
// lines 6.2 / 7.3, 4096 lines 8.2 / 8.5 (strided 8.7 / 7.7), 16,384 lines 25.3
// / 20.4; N = 128 with 4096 lines 5.1 / 5.5, 16,384 lines 11.2 / 9.7.
bool dense_tiled(const direct_plan_s *dp, size_t dir, size_t nlines) {
  const int N = (int)dp->N;
  return dp->d_K[dir] && nlines >= 4 &&
         (N > kDenseMaxN || (dp->dense_tile == 2 && N > 32) ||
          (dp->dense_tile == 0 && N > 32 && nlines <= kGemmFewLines));
}

// Packed unit-stride lines of several direct plans in one tiled dense launch.
int run_dense_classes(const DenseItem *items, int count, const double *d_in, double *d_out,
                      size_t dir, hipStream_t st) {
  DenseClasses dc{};
  size_t total = 0;
  for (int i = 0; i < count; i++) {
    if (i >= kMaxDenseClasses) {
      set_error("run_dense_classes: too many classes for one launch");
      return -1;
    }
    const direct_plan_s *dp = items[i].dp;
    DenseClass &c = dc.c[i];
    c.K = dp->d_K[dir];
    c.off = items[i].off;
    c.n = items[i].n;
    c.nlines = items[i].nlines;
    c.N = (int)dp->N;
    c.NPP = dp->NPP;
    c.bxs = (unsigned)((c.nlines + kGemmLT - 1) / kGemmLT);
    c.tiles = c.bxs * (unsigned)((dp->NPP + kGemmRT - 1) / kGemmRT);
    total += c.tiles;
  }
  dc.count = count;
  if (total == 0) return 0;
  k_lines_gemm_multi<<<(unsigned)total, kGemmNT, gemm_shared_bytes(), st>>>(d_in, d_out, dc);
  L2C_HIP(hipGetLastError(), -1);
  return 0;
}

// Lines through the parity blocks K (NPP) of length N on the tiled dense
// product, one launch for any number of lines.
static void launch_lines_gemm(Prof *prof, const double *K, int NPP, int N, const double *d_in,
                              double *d_out, const LineMap &lm, size_t nlines, hipStream_t st) {
  const dim3 grid((unsigned)((nlines + kGemmLT - 1) / kGemmLT),
                  (unsigned)((NPP + kGemmRT - 1) / kGemmRT));
  launch_k(prof, lm.es == 1 ? k_lines_gemm<true> : k_lines_gemm<false>, grid, kGemmNT,
           gemm_shared_bytes(), st, d_in, d_out, lm, nlines, N, NPP, K);
}

// The same on the kernel that holds whole lines (N <= kDenseMaxN).
static void launch_lines_dense(Prof *prof, const double *K, int NPP, int N, const double *d_in,
                               double *d_out, const LineMap &lm, size_t nlines, hipStream_t st) {
  // per_cu: the work-groups that a CU's registers and LDS hold, times 256 CUs
  auto go = [&](auto kern, int NRM, int LT, int NP, int per_cu) {
    const size_t items = (nlines + LT - 1) / LT * (3 - NP);
    launch_k(prof, kern, dim3((unsigned)std::min<size_t>(items, 256 * per_cu)), 32 * NRM * NP,
             dense_shared_bytes(NRM, LT, NP), st, d_in, d_out, lm, nlines, N, NPP, K);
  };
  if (lm.es == 1)
    NPP > 64   ? go(k_lines_dense<true, 8, 16, 2>, 8, 16, 2, 2)
    : NPP > 32 ? go(k_lines_dense<true, 4, 32, 2>, 4, 32, 2, 3)
               : go(k_lines_dense<true, 2, 16, 2>, 2, 16, 2, 8);
  else
    NPP > 64   ? go(k_lines_dense<false, 8, 32, 1>, 8, 32, 1, 3)
    : NPP > 32 ? go(k_lines_dense<false, 4, 32, 2>, 4, 32, 2, 3)
               : go(k_lines_dense<false, 2, 32, 2>, 2, 32, 2, 6);
}

// Batched lines through a direct plan: dense MFMA products when the plan has
// them and the batch is large enough, else one row per thread.
static int launch_direct_lines(const direct_plan_s *dp, const double *d_in, double *d_out,
                               size_t dir, const LineMap &lm, size_t nlines, hipStream_t st) {
  const int N = (int)dp->N;
  if (dense_tiled(dp, dir, nlines)) {
    launch_lines_gemm(dp->prof, dp->d_K[dir], dp->NPP, N, d_in, d_out, lm, nlines, st);
  } else if (dp->d_K[dir] && nlines >= 4) {
    launch_lines_dense(dp->prof, dp->d_K[dir], dp->NPP, N, d_in, d_out, lm, nlines, st);
  } else {
    launch_direct(dp, d_in, d_out, dir, lm, nlines, st);
  }
  L2C_HIP(hipGetLastError(), -1);
  return 0;
}

// ---------------------------------------------------------------------------
// host orchestration

// Whether a call of nlines lines runs its M2L below lu on MFMA (precision
// form 2, or FP64 MFMA for line calls from m2l_mma_lines lines on).
static bool m2l_on_mfma(const fmm_plan_s *p, size_t nlines) {
  if (p->geo.M != 18) return false;
  if (p->precision == 2) return true;
  const int t = p->m2l_mma_lines;
  // (form 1 keeps to its own records up to 31 lines: the bound of 8 was timed
  // against the FP64 matrices)
  const bool mid = p->precision == 0 && p->geo.L >= 8 && p->geo.L <= 10;
  const size_t lines = t >= 0 ? (size_t)t : mid ? 8 : 32;
  return lines > 0 && nlines >= lines;
}
// The work-group geometry of a call: single-line calls take geo1, line
// calls geo (the MFMA M2L forms, whose form-2 tables are cut at geo's lu,
// always take geo).
static const Geo &call_geo(const fmm_plan_s *p, size_t nlines) {
  return nlines == 1 && !m2l_on_mfma(p, nlines) ? p->geo1 : p->geo;
}

// Whether a call's band sums wait for the far field in the workspace, back to back,
// and not in the output (LINES_RAW): where the output's elements lie apart with nothing
// of the call between them (single strided transforms, lines far apart), so that every
// touch of one fetches or writes a cache line.  One transform, s = 64, workspace / output
// (us): 2^20 at stride 16 78 / 123, at 8 62 / 77, at 2 49.5 / 51, 2^18 at 16 33 / 39,
// 2^16 at 16 19 / 22, 20,000 at 8 17.3 / 17.9; 4 lines of 2^20 at 8 245 / 372, 64 of 2^16 at
// 2 113 / 118.  (With the band inside the downward kernel, whose passes over the array are
// two fewer, 2^20 at 16 87, at 8 68, 4 lines at 8 267.)  Lines that lie side by side share
// their cache lines instead (place).
static bool raw_sums(const Geo &g, const LineMap &lm, size_t nlines, bool across) {
  return g.far && lm.es > 1 && !across &&
         (nlines == 1 || band_groups(g, 16) >= 4u << g.lu);  // (else LINES_FLAT)
}

// Workspace for a batch of lines: grown on demand (at least doubling), owned
// by the plan.  Earlier calls may still be running on a caller's stream, so
// the store being replaced is retired, not freed: the plan releases it when
// it is itself freed, and nothing waits here on work of other streams.
// raw: with room for the band sums of every line behind it.
static int ensure_ws(fmm_plan_s *p, size_t nlines, const Geo &g, double **w, bool raw = false) {
  const size_t need = std::max<size_t>(nlines, 1) * (ws_doubles(g) + (raw ? p->N : 0));
  if (p->wl_cap < need) {
    const size_t cap = std::max(need, 2 * p->wl_cap);
    double *nw = nullptr;
    L2C_HIP(hipMalloc(&nw, cap * sizeof(double)), -1);
    if (p->d_wl) p->wl_retired.push_back(p->d_wl);
    p->d_wl = nw;
    p->wl_cap = cap;
  }
  *w = p->d_wl;
  return 0;
}

// k_down8r or k_down8 launch on stream st
static void launch_down8(fmm_plan_s *p, const Geo &g, const double *d_in, double *d_out, size_t dir,
                         const LineMap &lm, size_t nlines, hipStream_t st, double *ws) {
  const size_t wsstride = ws_doubles(g);
  dim3 gd((unsigned)((size_t)4 << g.ld), (unsigned)nlines);
  const size_t shm = down_shared_bytes(g);
  const int nt = 64 * (g.s >> 4);
  const double *tab = dir == L2C ? p->t.a : p->t.an;
  const double *htab = p->t.head[dir];
  prof_begin(p->prof, K_DOWN_BAND, st);
  if (p->down_roles) {
    const size_t shr = down8r_shared_bytes(g);
    const int rsh = std::max(-g.s, std::min(p->roles_shift, 8 * (g.s >> 4))) & ~7;
    if (dir == L2C)
      launch_k(p->prof, k_down8r<0, 0>, gd, 2 * nt, shr, st, d_in, d_out, lm, g, ws, wsstride,
          p->t.D, p->t.Q, p->t.T, tab, htab, rsh);
    else if (p->precompute)
      launch_k(p->prof, k_down8r<1, 1>, gd, 2 * nt, shr, st, d_in, d_out, lm, g, ws, wsstride,
          p->t.D, p->t.Q, p->t.T, tab, htab, rsh);
    else
      launch_k(p->prof, k_down8r<1, 0>, gd, 2 * nt, shr, st, d_in, d_out, lm, g, ws, wsstride,
          p->t.D, p->t.Q, p->t.T, tab, htab, rsh);
  } else if (dir == L2C)
    launch_k(p->prof, k_down8<0, 0>, gd, nt, shm, st, d_in, d_out, lm, g, ws, wsstride,
        p->t.D, p->t.Q, p->t.T, tab, htab);
  else if (p->precompute)
    launch_k(p->prof, k_down8<1, 1>, gd, nt, shm, st, d_in, d_out, lm, g, ws, wsstride,
        p->t.D, p->t.Q, p->t.T, tab, htab);
  else
    launch_k(p->prof, k_down8<1, 0>, gd, nt, shm, st, d_in, d_out, lm, g, ws, wsstride,
        p->t.D, p->t.Q, p->t.T, tab, htab);
  prof_end(p->prof, st);
}

// The split downward pass on st: k_band (before the tree kernels, which it
// does not need), then k_up and k_m2l, then k_far.
static void launch_band(fmm_plan_s *p, const Geo &g, const double *d_in, double *d_out, size_t dir,
                        const LineMap &lm, size_t nlines, hipStream_t st, int order, int scale,
                        int slot) {
  prof_begin(p->prof, slot, st);
  const bool s16 = (g.s & 15) == 0;
  auto kernel =
      order == LINES_ACROSS ? (s16 ? k_band<true, LINES_ACROSS> : k_band<false, LINES_ACROSS>)
      : order == LINES_RAW  ? (s16 ? k_band<true, LINES_RAW> : k_band<false, LINES_RAW>)
                            : (s16 ? k_band<true, LINES_PLAIN> : k_band<false, LINES_PLAIN>);
  launch_k(p->prof, kernel, dim3(band_groups(g, 16), (unsigned)nlines), kBandNT,
           band_shared_bytes(g, 16), st, d_in, d_out, lm, g, (int)dir, scale,
           dir == L2C ? p->t.a : p->t.an, p->t.head[dir]);
  prof_end(p->prof, st);
}

static void launch_far(fmm_plan_s *p, const Geo &g, double *d_out, const double *raw, size_t dir,
                       const LineMap &lm, size_t nlines, hipStream_t st, int order, double *ws,
                       int slot) {
  prof_begin(p->prof, slot, st);
  launch_k(p->prof,
           order == LINES_ACROSS ? k_far<LINES_ACROSS>
           : order == LINES_RAW  ? k_far<LINES_RAW>
                                 : k_far<LINES_PLAIN>,
           dim3((unsigned)((size_t)4 << g.ld), (unsigned)nlines), kFarNT, far_shared_bytes(g), st,
           d_out, raw, lm, g, (int)dir, ws, ws_doubles(g), p->t.D, p->t.Q, p->t.T);
  prof_end(p->prof, st);
}

// Groups of 8 chunks halve a small call's chain of trips (four to two at s =
// 64) and waste a fifth of the lanes' columns: taken while the band's groups of
// 16 leave most of the chip idle, for leaf sizes with more than two row groups.
// us per call, 16 / 8 chunks: one line of 2^13 18.8 / 16.0, 2^16 19.8 / 17.0,
// 200,000 (s = 49) 24.3 / 21.0, 2^18 23.8 / 21.3, 2^19 (256 groups of 16) 33.8 /
// 32.4, 600,000 (512) 39.3 / 41.6, 2^20 44.1 / 45.7; 16 lines of 2^13 (64) 20.3 /
// 17.9, 2 of 2^16 (64) 20.7 / 18.7, 4 of 2^16 (128) 22.0 / 22.8, 12 of 2^14 (96)
// 21.3 / 21.8, 2 of 2^18 (256) 26.0 / 30.8.
static bool band_by_8(const Geo &g, size_t nlines) {
  return g.s > 32 && band_groups(g, 16) * nlines <= (nlines == 1 ? 256 : 64);
}

// The downward pass of a far plan (geo.far): the band inside the k_up launch,
// then k_far; or (down_split 1, and 2 for line calls with L >= 10) a k_band
// launch of its own before k_up.  Per call, s = 64, k_down8r / k_band apart /
// band in the k_up launch (us): one line of 2^11 20.1 / 23.2 / 17.7, 2^16 21.8 /
// 25.5 / 19.3, 2^20 45.1 / 49.7 / 44.2; 16 lines of 2^13 23.6 / 26.7 / 20.3;
// 128 of 2^15 117 / 112 / 104; 64 of 2^18 423 / 387 / 372 (k_down8r: band and
// far field in one work-group of 16 waves, now for other ranks than 18).  The
// band apart wins only below what a call of plain lines reaches (256 lines of
// 2^11 36.9 / 45.5); the batch tuner times both.
static bool use_split(const fmm_plan_s *p, size_t nlines) {
  return p->down_split == 1 || (p->down_split == 2 && nlines > 1 && p->geo.L >= 10);
}

// One execute (or a batch of lines): upward pass, M2L, downward pass, all on st.
template <int MT>
static int launch_fmm_m(fmm_plan_s *p, const Geo &g, const double *d_in, double *d_out,
                        size_t dir, const LineMap &lm, size_t nlines, hipStream_t st,
                        int band_only, double *ws, double *raw = nullptr, bool across = false) {
  const size_t wsstride = ws_doubles(g);
  if (lm.n && !g.fast && !g.far) {  // per-line lengths: not in k_down
    set_error("lines of uneven length need a plan with leaf size s <= 64");
    return -1;
  }
  if (band_only && g.s <= kBandMaxS) {  // directM
    launch_band(p, g, d_in, d_out, dir, lm, nlines, st, LINES_PLAIN, 1, K_DOWN_BAND);
    return 0;
  }
  const bool split = g.far && use_split(p, nlines), fuse = g.far && !split;
  int order = across ? LINES_ACROSS : raw ? LINES_RAW : LINES_PLAIN;
  double *sums = raw ? raw : d_out;  // where the band sums go
  if (split) launch_band(p, g, d_in, sums, dir, lm, nlines, st, order, 0, K_BAND);
  if (!band_only) {
    const bool s16 = (g.s & 15) == 0;
    dim3 gu(4u << g.lu, (unsigned)nlines);
    const bool b8 = fuse && !across && band_by_8(g, nlines);
    const int nb = fuse ? (int)band_groups(g, b8 ? 8 : 16) : 0;
    if (order == LINES_PLAIN && fuse && !b8 && nlines > 1 && (unsigned)nb < gu.x)
      order = LINES_FLAT;
    if (order == LINES_FLAT || order == LINES_ACROSS)
      gu.x += nb;
    else if (fuse && order == LINES_RAW && !b8 && lm.es >= 8)  // in turn
      gu.x = (nb + 7) / 8 * (8 + 8 * (gu.x / nb));
    else if (fuse)
      gu = dim3(std::max(gu.x, (unsigned)nb), gu.y, 2);
    const BandArgs bu{sums, dir == L2C ? p->t.a : p->t.an, p->t.head[dir], nb};
    prof_begin(p->prof, K_UP_SUBTREE, st);
    if (MT == 18 && up18_eligible(g)) {
      const size_t shu = std::max(8 * (size_t)up18_lds(g).total,
                                  fuse ? band_shared_bytes(g, b8 ? 8 : 16) : 0);
      // (calls with lines in turn are past band_by_8's bounds)
      auto kernel =
          order == LINES_ACROSS ? (s16 ? k_up<true, 16, LINES_ACROSS> : k_up<false, 16, LINES_ACROSS>)
          : order == LINES_FLAT ? (s16 ? k_up<true, 16, LINES_FLAT> : k_up<false, 16, LINES_FLAT>)
          : order == LINES_RAW
              ? (b8 ? (s16 ? k_up<true, 8, LINES_RAW> : k_up<false, 8, LINES_RAW>)
                    : (s16 ? k_up<true, 16, LINES_RAW> : k_up<false, 16, LINES_RAW>))
          : b8 ? (s16 ? k_up<true, 8, LINES_PLAIN> : k_up<false, 8, LINES_PLAIN>)
               : (s16 ? k_up<true, 16, LINES_PLAIN> : k_up<false, 16, LINES_PLAIN>);
      launch_k(p->prof, kernel, gu, kUpNT, shu, st, d_in, lm, g, (int)dir, p->t.T, p->t.U, p->t.P,
               ws, wsstride, bu);
    } else if (MT > 0 && g.gu >= 3 && nlines <= 8) {
      launch_k(p->prof, k_up_any<MT, MT != 0>, gu, kUpNT, up_shared_bytes(g), st, d_in, lm, g,
               (int)dir, p->t.T, p->t.U, p->t.P, ws, wsstride);
    } else {
      launch_k(p->prof, k_up_any<MT, false>, gu, kUpNT, up_shared_bytes(g), st, d_in, lm, g,
               (int)dir, p->t.T, p->t.U, p->t.P, ws, wsstride);
    }
    prof_end(p->prof, st);
    const int ntop = (int)total_blocks(g.lu), ntot = (int)total_blocks(g.L);
    const int bpw = m2l_bpw(g);
    const unsigned gx = (unsigned)(ntop + (ntot - ntop + bpw - 1) / bpw);
    // lines per work-group: share each staged block over up to 8 lines while
    // the grid keeps at least ~2048 work-groups
    int lpb = 1;
    while (lpb < 8 && (size_t)gx * ((nlines + 2 * lpb - 1) / (2 * lpb)) >= 2048) lpb *= 2;
    dim3 gm(gx, (unsigned)((nlines + lpb - 1) / lpb));
    prof_begin(p->prof, K_M2L, st);
    const DevTables::Split &sp = p->t.sp[dir];
    const SplitView sv{p->precision == 1 ? sp.rec : nullptr, sp.pos, sp.n64, sp.n32, sp.n16,
                       sp.rec_bytes};
    const bool mma = MT == 18 && m2l_on_mfma(p, nlines);
    if (!mma && MT == 18 && p->t.At[dir] && !sv.rec && bpw == 4) {
      // the same grid; the blocks below lu from At, with the LDS of one
      // staged block (the top blocks') per work-group instead of four
      launch_k(p->prof, k_m2l_t<MT == 18 ? 18 : 1>, gm, kM2lNT,
               8 * (size_t)(m2l_wave_lds(g.M) + kM2lNT), st, g, p->t.A[dir], p->t.At[dir], ws,
               wsstride, nlines, lpb);
    } else if (!mma) {
      launch_k(p->prof, k_m2l<MT>, gm, kM2lNT, m2l_shared_bytes(g), st, g, p->t.A[dir], ws,
          wsstride, bpw, nlines, lpb, sv);
    } else {
      // on MFMA the blocks at levels >= lu, beside them the blocks above lu
      const int nblk = ntot - ntop;
      const unsigned mx = (unsigned)((nblk + 3) / 4);
      const size_t ngroups = (nlines + 7) / 8;
      // line groups per work-group: one while the grid stays small, more so
      // that about 8192 work-groups share the lines
      const size_t gpw = std::max<size_t>(1, (mx * ngroups + 8191) / 8192);
      const M2lGrid mg{ntop, ntop ? (int)gm.y : 0, lpb, (int)mx, sv};
      const dim3 gmm((unsigned)(mg.tx * mg.ty + mx * ((ngroups + gpw - 1) / gpw)));
      const size_t top = 8 * (size_t)(m2l_wave_lds(18) + kM2lNT);
      if (p->precision == 2) {
        const DevTables::Slices &sl = p->t.sl[dir];
        launch_k(p->prof, k_m2l_mma<2>, gmm, 256, top, st, g, p->t.A[dir], (const bf16x8 *)sl.q,
            sl.sc, ws, wsstride, nlines, (int)gpw, mg);
      } else {
        launch_k(p->prof, k_m2l_mma<0>, gmm, 256,
            std::max(top, 4 * 3 * 18 * 19 * sizeof(double)), st, g, p->t.A[dir], nullptr, nullptr,
            ws, wsstride, nlines, (int)gpw, mg);
      }
    }
    prof_end(p->prof, st);
  }
  if (g.far) {
    launch_far(p, g, d_out, raw, dir, lm, nlines, st, order, ws, fuse ? K_DOWN_BAND : K_FAR);
    return 0;
  }
  if (g.fast) {
    launch_down8(p, g, d_in, d_out, dir, lm, nlines, st, ws);
    return 0;
  }
  dim3 gd((unsigned)((size_t)4 << g.ld), (unsigned)nlines);
  const size_t shm = down_shared_bytes(g);
  const double *tab = dir == L2C ? p->t.a : p->t.an;
  const double *htab = p->t.head[dir];
  prof_begin(p->prof, K_DOWN_BAND, st);
  if (dir == L2C)
    launch_k(p->prof, k_down<0, 0, MT>, gd, kDownNT, shm, st, d_in, d_out, lm, g, band_only, ws,
        wsstride, p->t.D, p->t.Q, p->t.T, tab, htab);
  else if (p->precompute)
    launch_k(p->prof, k_down<1, 1, MT>, gd, kDownNT, shm, st, d_in, d_out, lm, g, band_only, ws,
        wsstride, p->t.D, p->t.Q, p->t.T, tab, htab);
  else
    launch_k(p->prof, k_down<1, 0, MT>, gd, kDownNT, shm, st, d_in, d_out, lm, g, band_only, ws,
        wsstride, p->t.D, p->t.Q, p->t.T, tab, htab);
  prof_end(p->prof, st);
  return 0;
}

static int launch_fmm(fmm_plan_s *p, const double *d_in, double *d_out, size_t dir,
                      const LineMap &lm, size_t nlines, hipStream_t st, int band_only,
                      bool across = false) {
  double *ws = nullptr;
  const Geo &g = call_geo(p, nlines);
  bool raw = !band_only && raw_sums(g, lm, nlines, across);
  if (raw && p->wl_cap < nlines * (ws_doubles(g) + p->N)) {
    // nothing is allocated for them in a call that is being captured
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    L2C_HIP(hipStreamIsCapturing(st, &cs), -1);
    raw = cs == hipStreamCaptureStatusNone;
  }
  if (ensure_ws(p, nlines, g, &ws, raw)) return -1;
  double *rw = raw ? ws + nlines * ws_doubles(g) : nullptr;
  const int rc =
      g.M == 18 ? launch_fmm_m<18>(p, g, d_in, d_out, dir, lm, nlines, st, band_only, ws, rw, across)
                : launch_fmm_m<0>(p, g, d_in, d_out, dir, lm, nlines, st, band_only, ws);
  if (rc) return rc;
  L2C_HIP(hipGetLastError(), -1);
  return 0;
}
int run_fmm_launch(fmm_plan_s *p, const double *d_in, double *d_out, size_t dir, size_t stride,
                   hipStream_t st, int band_only) {
  LineMap lm{1, 0, 0, stride};
  if (!band_only && p->N <= (size_t)p->direct_max_n) {
    // small N: the direct sums in one launch (the plan's tables a, an, dn
    // are those of a direct plan of the same N)
    prof_begin(p->prof, K_DIRECT, st);
    launch_direct_one(p->prof, (int)p->N, dir, p->t.a, p->t.an, p->t.dn, d_in, d_out, lm, st,
                      p->direct_band);
    prof_end(p->prof, st);
    L2C_HIP(hipGetLastError(), -1);
    return 0;
  }
  return launch_fmm(p, d_in, d_out, dir, lm, 1, st, band_only);
}
int run_fmm(fmm_plan_s *p, const double *d_in, double *d_out, size_t dir, size_t stride,
            hipStream_t st, int band_only) {
  prof_step(p->prof);
  return run_fmm_launch(p, d_in, d_out, dir, stride, st, band_only);
}

int run_direct(const direct_plan_s *dp, const double *d_in, double *d_out, size_t dir,
               size_t stride, hipStream_t st, size_t precompute) {
  (void)precompute;
  prof_step(dp->prof);
  LineMap lm{1, 0, 0, stride};
  prof_begin(dp->prof, K_DIRECT, st);
  launch_direct(dp, d_in, d_out, dir, lm, 1, st);
  prof_end(dp->prof, st);
  L2C_HIP(hipGetLastError(), -1);
  return 0;
}

// Lines of uneven length packed back to back: line l (l < nlines) starts at
// d_off[l] and has d_n[l] <= plan N elements (unit stride).  FMM plans
// (leaf size 16, 32 or 64) or direct plans (L = 0).
int run_packed(fmm_plan_s *p, const direct_plan_s *dp, const double *d_in, double *d_out,
               size_t dir, size_t nlines, const size_t *d_off, const int *d_n, hipStream_t st) {
  for (size_t l0 = 0; l0 < nlines; l0 += 65535) {
    const size_t nl = std::min<size_t>(65535, nlines - l0);
    LineMap lm{1, 0, 0, 1, d_off + l0, d_n + l0};
    if (dp) {
      if (launch_direct_lines(dp, d_in, d_out, dir, lm, nl, st)) return -1;
    } else {
      if (p->wl_cap < nl * ws_doubles(call_geo(p, nl))) {
        set_error("run_packed: workspace not reserved for this many lines");
        return -1;
      }
      if (launch_fmm(p, d_in, d_out, dir, lm, nl, st, 0)) return -1;
    }
  }
  return 0;
}

// Precision form 2 tables of direction dir: the BF16 slices and row scales of
// every block at levels >= lu (k_slice_A).
int build_slices(fmm_plan_s *p, int dir) {
  const Geo &g = p->geo;
  DevTables::Slices &sl = p->t.sl[dir];
  if (sl.q) return 0;
  const size_t nblk = total_blocks(g.L) - total_blocks(g.lu);
  if (nblk == 0) return 0;
  const size_t nq = nblk * 3 * 2 * kSlices * 64 * 8;
  L2C_HIP(hipMalloc(&sl.q, nq * sizeof(unsigned short)), -1);
  L2C_HIP(hipMalloc(&sl.sc, nblk * 48 * sizeof(double)), -1);
  p->hbm_bytes += nq * sizeof(unsigned short) + nblk * 48 * sizeof(double);
  k_slice_A<<<(unsigned)nblk, 64, 0, p->stream>>>(p->t.A[dir], g.M, g.L, g.lu, sl.q, sl.sc);
  L2C_HIP(hipGetLastError(), -1);
  L2C_HIP(hipStreamSynchronize(p->stream), -1);
  return 0;
}

// Grow the plan's line workspace to nlines lines now (so that later launches,
// graph capture included, never allocate).
int reserve_lines(fmm_plan_s *p, size_t nlines) {
  double *w = nullptr;
  const Geo &g = ws_doubles(p->geo1) > ws_doubles(p->geo) ? p->geo1 : p->geo;
  return ensure_ws(p, std::min<size_t>(nlines, 65535), g, &w);
}

// Whether a line call of nlines lines of FMM plan p runs as direct sums in
// one launch: the plan's small-N route (direct_max_n) while the call holds at
// most direct_line_elems elements, where the FMM's fixed cost of about 22 us
// per call is still the larger.  Per call, FMM / direct (us): N = 2048 with
// 8 lines 21.7 / 16.6 (16 lines 21.8 / 29.0), 4096 with 4 lines 23.1 / 14.3
// (8 lines 23.2 / 23.9), 8192 with 2 lines 24.5 / 19.1 (3 lines 24.6 / 25.9).
static bool direct_lines(const fmm_plan_s *p, size_t nlines) {
  return p->N <= (size_t)p->direct_max_n && nlines * p->N <= (size_t)p->direct_line_elems;
}

// Whether a line call of an FMM plan runs as the tiled dense product on the
// plan's parity blocks (plans of N <= dense_max_n, plain FP64).  The product
// costs N / 2 multiply-adds an element against the FMM's fixed cost per line
// and per call.  Per call, FMM / dense (us, contiguous lines): N = 300 with
// 64 lines 23.6 / 7.7, 4096 lines 298 / 12.4; 512 with 1024 lines 138 / 9.8;
// 1024 with 64 lines 25.6 / 15.1, 4096 lines 567 / 52.6; 1500 with 64 lines
// 27.1 / 21.0, 1024 lines 110 / 33.1; 2048 with 64 lines 24.9 / 26.9, 256
// lines 53.0 / 30.9, 4096 lines 601 / 177.  Above 2048 the blocks would take
// more than 17 MB of HBM per direction for gains that end near N = 4096.
static bool dense_lines(const fmm_plan_s *p, size_t dir, size_t nlines) {
  return p->d_K[dir] && p->precision == 0 && nlines >= (p->N <= 1536 ? 2 : 128);
}

// Whether the FMM kernels of a line call of N elements a line take neighbouring
// lines in turn (place): where a line's neighbour lies nearer than its own next
// element and the call is too large for the caches to keep what the lines share
// from one line's work-groups to the next's.  Lines side by side, group by group /
// line by line, s = 64 unless stated (us): 40 lines of 2^18 307 / 563, 100 807 /
// 1530, 8 of 2^20 245 / 512, 24 of 140,000 (s = 35) 143 / 204, 500 of 33,000 (s =
// 33) 712 / 777, 8 of 2^18 72 / 79; even at 8 of 140,000 57.4 / 57.3 and 24 of
// 70,000 83 / 84; below, the division costs 1 to 2 %: 8 of 2500 18.1 / 17.6, 24 of
// 16,384 31.3 / 31.0.  (With the band inside the downward kernel, whose passes over
// a strided array are two fewer: 400, 1037, 338, 246, 923 and 83.)
static bool lines_across(const LineMap &lm, size_t N, size_t nlines) {
  return nlines > 1 && (lm.n0 > 1 ? lm.ls0 : lm.ls1) < lm.es && N * nlines >= (size_t)1 << 20;
}

int run_lines(fmm_plan_s *p, const double *d_in, double *d_out, size_t dir, size_t nlines,
              size_t n0, size_t ls0, size_t ls1, size_t es, hipStream_t st) {
  prof_step(p->prof);
  LineMap lm{n0 ? n0 : 1, ls0, ls1, es};
  if (p->L == 0) {
    // dense MFMA products when the plan has them (N <= 4096) and there are
    // at least four lines, else one row per thread; either way one launch
    const direct_plan_s *dp = p->dplan;
    prof_begin(dp->prof, K_DIRECT, st);
    const int rc = launch_direct_lines(dp, d_in, d_out, dir, lm, nlines, st);
    prof_end(dp->prof, st);
    return rc;
  }
  if (direct_lines(p, nlines)) {
    prof_begin(p->prof, K_DIRECT, st);
    launch_direct_one(p->prof, (int)p->N, dir, p->t.a, p->t.an, p->t.dn, d_in, d_out, lm, st,
                      p->direct_band, (unsigned)nlines);
    prof_end(p->prof, st);
    L2C_HIP(hipGetLastError(), -1);
    return 0;
  }
  if (dense_lines(p, dir, nlines)) {
    prof_begin(p->prof, K_DIRECT, st);
    launch_lines_gemm(p->prof, p->d_K[dir], p->NPP, (int)p->N, d_in, d_out, lm, nlines, st);
    prof_end(p->prof, st);
    L2C_HIP(hipGetLastError(), -1);
    return 0;
  }
  // lines go in grid.y: at most 65535 per launch, each chunk reusing the
  // front of the plan's line workspace
  const bool across = lines_across(lm, p->N, nlines);
  for (size_t l0 = 0; l0 < nlines; l0 += 65535) {
    lm.l0 = l0;
    if (launch_fmm(p, d_in, d_out, dir, lm, std::min<size_t>(65535, nlines - l0), st, 0, across))
      return -1;
  }
  return 0;
}

// ---------------------------------------------------------------------------
// Workspace of l2c_execute_lines_device_noalloc: a fixed device array, one
// copy per GPU, held until the process ends.  Host code never names it in a
// launch or copy: it passes the per-device address from hipGetSymbolAddress.
constexpr size_t kScratchDoubles = (size_t)4 << 20;  // 32 MiB
static __device__ __align__(256) double scratch[kScratchDoubles];

constexpr int kMaxDevices = 64;
static double *g_scratch[kMaxDevices] = {};
static bool g_scratch_done[kMaxDevices] = {};
static std::mutex g_scratch_mu;

// The scratch address on the current device, looked up once per device (with
// that device current, as the calling thread has it).  nullptr on failure.
static double *scratch_ptr() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    set_error("l2c_execute_lines_device_noalloc: no current device");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_done[dev]) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      set_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
      return nullptr;
    }
    g_scratch[dev] = (double *)ptr;
    g_scratch_done[dev] = true;
  }
  return g_scratch[dev];
}

// Lines through an FMM plan with the fixed scratch as the workspace: as many
// lines per launch as the scratch holds (and at most 65,535), launches in
// order on st, each reusing the scratch front.  Nothing here allocates, and
// nothing in the scratch needs clearing (every element a launch reads was
// written earlier in the same launch sequence).
static int run_lines_scratch(fmm_plan_s *p, double *scr, const double *d_in, double *d_out,
                             size_t dir, size_t nlines, size_t n0, size_t ls0, size_t ls1,
                             size_t es, hipStream_t st) {
  LineMap lm{n0 ? n0 : 1, ls0, ls1, es};
  if (p->L == 0) return launch_direct_lines(p->dplan, d_in, d_out, dir, lm, nlines, st);
  if (direct_lines(p, nlines)) {  // as l2c_execute_lines_device: no workspace
    launch_direct_one(p->prof, (int)p->N, dir, p->t.a, p->t.an, p->t.dn, d_in, d_out, lm, st,
                      p->direct_band, (unsigned)nlines);
    L2C_HIP(hipGetLastError(), -1);
    return 0;
  }
  if (dense_lines(p, dir, nlines)) {  // nor here
    launch_lines_gemm(p->prof, p->d_K[dir], p->NPP, (int)p->N, d_in, d_out, lm, nlines, st);
    L2C_HIP(hipGetLastError(), -1);
    return 0;
  }
  const size_t wsd = std::max(ws_doubles(p->geo), ws_doubles(p->geo1));
  const bool across = lines_across(lm, p->N, nlines);
  const bool raw = raw_sums(p->geo, lm, nlines, across) && wsd + p->N <= kScratchDoubles;
  const size_t per = std::min<size_t>(65535, kScratchDoubles / (wsd + (raw ? p->N : 0)));
  if (per == 0) {
    set_error("l2c_execute_lines_device_noalloc: one line of this plan needs " +
              std::to_string(wsd * sizeof(double)) + " bytes of workspace, more than the " +
              std::to_string(kScratchDoubles * sizeof(double)) + "-byte scratch");
    return -1;
  }
  for (size_t l0 = 0; l0 < nlines; l0 += per) {
    lm.l0 = l0;
    const size_t nl = std::min(per, nlines - l0);
    const Geo &g = call_geo(p, nl);
    double *rw = raw ? scr + nl * wsd : nullptr;
    const int rc = g.M == 18 ? launch_fmm_m<18>(p, g, d_in, d_out, dir, lm, nl, st, 0, scr, rw, across)
                             : launch_fmm_m<0>(p, g, d_in, d_out, dir, lm, nl, st, 0, scr);
    if (rc) return rc;
    L2C_HIP(hipGetLastError(), -1);
  }
  return 0;
}

}  // namespace l2c

using namespace l2c;

extern "C" {

int l2c_execute_lines_device_noalloc(fmm_plan *p, const double *d_in, double *d_out,
                                     size_t direction, size_t nlines, size_t n0, size_t ls0,
                                     size_t ls1, size_t es, void *stream) {
  clear_error();
  if (!p || !d_in || !d_out || direction > 1 || es == 0 || nlines == 0) {
    set_error("l2c_execute_lines_device_noalloc: invalid argument");
    return -1;
  }
  const bool planned = p->L == 0 ? (p->dplan->direction == BOTH || p->dplan->direction == direction)
                                 : p->t.A[direction] != nullptr;
  if (!planned) {
    set_error("l2c_execute_lines_device_noalloc: direction was not planned");
    return -1;
  }
  double *scr = scratch_ptr();
  if (!scr) return -1;
  // no timing events here (their pool would grow by allocation)
  const int cur = p->prof ? p->prof->cur : 0;
  if (p->prof) p->prof->cur = 0;
  const int rc = run_lines_scratch(p, scr, d_in, d_out, direction, nlines, n0, ls0, ls1, es,
                                   stream ? (hipStream_t)stream : p->stream);
  if (p->prof) p->prof->cur = cur;
  return rc;
}

}  // extern "C"
