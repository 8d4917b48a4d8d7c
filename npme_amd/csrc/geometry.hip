// Set-up of one geometry on the device: embedded cell keys, the stable sort
// of the charges by cell, the per-cell ranges, cluster-relative positions,
// spline windows and the per-tile charge lists of spreading and
// interpolation.  Every index is computed with the same FP64 operations as
// the host set-up (no contraction into FMAs), and the sorts are stable, so
// the permutation and every list are bit-identical to the host's; the
// per-charge cell index follows src/PartitionBox.cpp:311-351 and
// src/PartitionEmbeddedBox.cpp:266-455, the spline window
// src/RecSumSupportFunctions.h:123-149.
#include <cstring>
#include <deque>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_reduce.hpp>
#include <rocprim/device/device_scan.hpp>

#include "npme_internal.h"

namespace npme {

// error bits written by the set-up kernels
enum { GEO_ERR_CELL = 1, GEO_ERR_WINDOW = 2, GEO_ERR_FIXED = 4, GEO_LONG_BUCKET = 8 };

__device__ __forceinline__ bool d_coord2cell(double x, double cs, unsigned long ncell,
                                             unsigned long &v)
{
#pragma clang fp contract(off)
  const double tol = 1.0e-14;
  if (x < -tol) return false;
  unsigned long t = (unsigned long)(x / cs);
  if (t > ncell) return false;
  if (t == ncell) {
    if (fabs(x - (double)t * cs) < tol) t--;
    else return false;
  }
  v = t;
  return true;
}

__global__ __launch_bounds__(256) void k_cell_keys(size_t n, const double *__restrict__ coord,
                                                   GeoParams g, int bits, unsigned *__restrict__ key,
                                                   int *__restrict__ slot, int *__restrict__ count,
                                                   int4 *__restrict__ gcell, int *__restrict__ err)
{
#pragma clang fp contract(off)
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  unsigned long a[3] = {0, 0, 0}, b[3] = {0, 0, 0};
  bool ok = true;
  for (int d = 0; d < 3; d++) {
    const double x1 = coord[3 * i + d] + (-g.mn[d]);
    ok = ok && d_coord2cell(x1, g.csA, g.nA[d], a[d]);
    const double x2 = x1 - (double)a[d] * g.csA;
    ok = ok && d_coord2cell(x2, g.csB, g.nP, b[d]);
  }
  if (!ok) {
    atomicOr(err, GEO_ERR_CELL);
    a[0] = a[1] = a[2] = b[0] = b[1] = b[2] = 0;
  }
  const unsigned long Nc = g.nP * g.nP * g.nP;
  const unsigned long tA = (a[0] * g.nA[1] + a[1]) * g.nA[2] + a[2];
  const unsigned k = (unsigned)(tA * Nc + (b[0] * g.nP + b[1]) * g.nP + b[2]);
  key[i] = k;
  // one atomic for the charges of a wavefront that share a cell: atomics on
  // one address are served ~7 ns apart, so 22k charges in a ball of one cell
  // took 146 us with an atomic each
  const int lane = threadIdx.x & 63;
  unsigned long long m = __ballot(1);  // lanes of the same cell
  for (int b2 = 0; b2 < bits; b2++) {  // uniform
    const bool one = (k >> b2) & 1u;
    const unsigned long long ones = __ballot(one);
    m &= one ? ones : ~ones;
  }
  const int lead = __ffsll(m) - 1, before = __popcll(m & ((1ull << lane) - 1));
  int first = 0;
  if (lane == lead) first = atomicAdd(&count[k], __popcll(m));
  slot[i] = __shfl(first, lead) + before;
  gcell[i] = make_int4((int)(a[0] * g.nP + b[0]), (int)(a[1] * g.nP + b[1]),
                       (int)(a[2] * g.nP + b[2]), 0);
}

template <typename K>
__device__ __forceinline__ size_t lower_bound_d(const K *a, size_t n, K v)
{
  size_t lo = 0, hi = n;
  while (lo < hi) {
    const size_t mid = (lo + hi) >> 1;
    if (a[mid] < v) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// Sort by cell.  The keys are dense and a cell holds few charges, so the sort
// is a count of every key (atomics, each charge keeping its arrival number), a
// scan, and a placement at start + arrival; the stable order is restored by
// ranking each charge among its cell's.  That is 5 launches, against 13 to 21
// of a merge sort (600k charges: 260 us, launches of ~6 us with ~5 us between
// them).  Ranking is quadratic in a cell, so cells of more than kRankMax
// charges raise GEO_LONG_BUCKET and the phase is repeated with the radix
// sort.  Set-up of 1M charges, ranked against sorted (the pass up to the
// ranking included): 1,000 a cell 1.83 / 1.98 ms, 2,000 2.12 / 2.17, 4,000
// 2.36 / 2.23; 300k: 0.86 / 0.98, 0.92 / 0.99, 0.98 / 1.00.
constexpr int kRankMax = 2048;

__global__ __launch_bounds__(256) void k_cell_place(size_t n, const unsigned *__restrict__ key,
                                                    const int *__restrict__ slot,
                                                    const int *__restrict__ start, int *__restrict__ tmp)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) tmp[start[key[i]] + slot[i]] = (int)i;
}

// rank of value v among the entries [b, e) of its bucket (distinct values)
__device__ __forceinline__ int bucket_rank(const int *__restrict__ tmp, int b, int e, int v)
{
  int r = 0, f = b;
  for (; f < e && (f & 3); f++) r += tmp[f] < v;
#pragma unroll 8
  for (; f + 4 <= e; f += 4) {
    const int4 t = *reinterpret_cast<const int4 *>(tmp + f);
    r += (t.x < v) + (t.y < v) + (t.z < v) + (t.w < v);
  }
  for (; f < e; f++) r += tmp[f] < v;
  return r;
}

// the stable order: charge i of entry p goes to its bucket's start plus its
// rank, with its cell and its position
__global__ __launch_bounds__(256) void k_cell_rank(size_t n, const int *__restrict__ tmp,
                                                   const unsigned *__restrict__ key,
                                                   const int *__restrict__ start,
                                                   const int4 *__restrict__ gcell,
                                                   const double *__restrict__ coord, int *__restrict__ perm,
                                                   int4 *__restrict__ cellOf, double4 *__restrict__ xs,
                                                   int *__restrict__ err)
{
  const size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const int i = tmp[p];
  const unsigned k = key[i];
  const int b = start[k], e = start[k + 1];
  size_t o = p;
  if (e - b <= kRankMax) o = (size_t)b + bucket_rank(tmp, b, e, i);
  else if (p == (size_t)b) atomicOr(err, GEO_LONG_BUCKET);  // one charge of the cell
  perm[o] = i;
  cellOf[o] = gcell[i];
  xs[o] = make_double4(coord[3 * (size_t)i], coord[3 * (size_t)i + 1], coord[3 * (size_t)i + 2], 0.0);
}

// (start, count) of every cell of the dense cell grid; an empty cell starts
// where its key would be
__global__ __launch_bounds__(256) void k_cell_ranges(long ncell, GeoParams g, const int *__restrict__ start,
                                                     int *__restrict__ cellSE)
{
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  const long g2 = c % g.nb[2], g1 = (c / g.nb[2]) % g.nb[1], g0 = c / ((long)g.nb[1] * g.nb[2]);
  const unsigned long nP = g.nP, Nc = nP * nP * nP;
  const unsigned long a0 = g0 / nP, a1 = g1 / nP, a2 = g2 / nP;
  const unsigned long kc =
      ((a0 * g.nA[1] + a1) * g.nA[2] + a2) * Nc + ((g0 % nP) * nP + (g1 % nP)) * nP + (g2 % nP);
  const int lo = start[kc], hi = start[kc + 1];
  cellSE[2 * c] = lo;
  cellSE[2 * c + 1] = hi - lo;
}

// cell and position of each sorted charge (after the radix sort)
__global__ __launch_bounds__(256) void k_gather_cells(size_t n, const int *__restrict__ perm,
                                                      const int4 *__restrict__ gcell,
                                                      const double *__restrict__ coord,
                                                      int4 *__restrict__ cellOf, double4 *__restrict__ xs)
{
  const size_t s = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const size_t i = (size_t)perm[s];
  cellOf[s] = gcell[i];
  xs[s] = make_double4(coord[3 * i], coord[3 * i + 1], coord[3 * i + 2], 0.0);
}

__global__ __launch_bounds__(256) void k_iota(size_t n, int *__restrict__ v)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = (int)i;
}

// spreading tiles that the window starting at u touches
struct TileRange {
  int lo[3], hi[3];
};
__device__ __forceinline__ TileRange tile_range(const GeoParams &g, int4 u)
{
  TileRange r;
  const int v[3] = {u.x, u.y, u.z};
  for (int d = 0; d < 3; d++) {
    r.lo[d] = v[d] / g.ts[d];
    r.hi[d] = (v[d] + (int)g.Bn - 1) / g.ts[d];
  }
  return r;
}
// interpolation tile of a window start
__device__ __forceinline__ long itile_of(const GeoParams &g, int x, int y, int z)
{
  return ((long)(x / g.TI) * g.nti[1] + y / g.TI) * g.nti[2] + z / g.TI;
}

// per sorted charge: cluster-relative position (FP64 or int32 fixed
// point), spline window start u0 = m0 + N/4 and fractional argument, the
// number of spreading tiles its window touches, and per chunk of 64 charges
// (one wavefront) the smallest and largest window start of each axis
template <bool FP64>
__global__ __launch_bounds__(256) void k_charge_setup(size_t n, const int *__restrict__ perm,
                                                      const double *__restrict__ coord,
                                                      const int4 *__restrict__ cellOf, GeoParams g,
                                                      void *__restrict__ src,
                                                      float4 *__restrict__ srcRes,
                                                      int4 *__restrict__ ms,
                                                      void *__restrict__ frac,
                                                      int *__restrict__ ntile, int4 *__restrict__ chunkBox,
                                                      int *__restrict__ err)
{
#pragma clang fp contract(off)
  const size_t s0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = s0 < n;
  const size_t s = live ? s0 : n - 1;  // a lane past the last repeats it (its box is unchanged)
  const int i = perm[s];
  const int4 gc = cellOf[s];
  const int gcv[3] = {gc.x, gc.y, gc.z};
  double loc[3], fr[3];
  int u0[3];
  int cnt = 1;
  for (int d = 0; d < 3; d++) {
    const double x = coord[3 * (size_t)i + d];
    // the list walk reads positions in one frame (the cells' low corner),
    // the cell-row sum relative to the charge's cluster corner
    loc[d] = g.globalFrame ? x + (-g.mn[d]) : (x + (-g.mn[d])) - (double)(gcv[d] / (int)g.nP) * g.csA;
    const double w = g.NoverL[d] * (x - g.R[d]);
    const long m0 = (w < 0) ? (long)(-w) + 1 : (long)(-w);
    if (m0 < -g.N[d] / 4 || m0 + g.Bn - 1 > g.N[d] / 4 - 1) {
      atomicOr(err, GEO_ERR_WINDOW);
      u0[d] = 0;
      fr[d] = 0;
    } else {
      u0[d] = (int)(m0 + g.N[d] / 4);
      fr[d] = w + (double)m0;
    }
    cnt *= (u0[d] + (int)g.Bn - 1) / g.ts[d] - u0[d] / g.ts[d] + 1;
  }
  ms[s] = make_int4(u0[0], u0[1], u0[2], 0);
  ntile[s] = cnt;
  {
    int lo[3], hi[3];
    for (int d = 0; d < 3; d++) {
      lo[d] = hi[d] = u0[d];
      for (int o = 32; o > 0; o >>= 1) {
        lo[d] = min(lo[d], __shfl_xor(lo[d], o));
        hi[d] = max(hi[d], __shfl_xor(hi[d], o));
      }
    }
    if (live && (threadIdx.x & 63) == 0) {
      chunkBox[2 * (s / 64)] = make_int4(lo[0], lo[1], lo[2], 0);
      chunkBox[2 * (s / 64) + 1] = make_int4(hi[0], hi[1], hi[2], 0);
    }
  }
  if (FP64) {
    ((double4 *)src)[s] = make_double4(loc[0], loc[1], loc[2], 0.0);
    ((double4 *)frac)[s] = make_double4(fr[0], fr[1], fr[2], 0.0);
  } else {
    int v[3];
    float res[3];
    for (int d = 0; d < 3; d++) {
      const double u = loc[d] * g.fxScale;
      const long r = g.globalFrame ? (fabs(u) < 4.0e18 ? llround(u) : 0) : lround(u);
      if (g.globalFrame ? !(fabs(u) < 4.0e18) : (r < -(1L << 20) || r > (1L << g.fxShift) + (1L << 20))) {
        atomicOr(err, GEO_ERR_FIXED);
        v[d] = 0;
      } else {
        // the list walk's frame wraps modulo 2^32
        v[d] = (int)(unsigned)(unsigned long)r;
      }
      res[d] = (float)(u - (double)r);
    }
    ((int4 *)src)[s] = make_int4(v[0], v[1], v[2], 0);
    srcRes[s] = make_float4(res[0], res[1], res[2], 0.0f);
    ((float4 *)frac)[s] = make_float4((float)fr[0], (float)fr[1], (float)fr[2], 0.0f);
  }
}

// (tile, charge) entries of the spreading lists, in charge order
__global__ __launch_bounds__(256) void k_tile_emit(size_t n, const int4 *__restrict__ ms,
                                                   const int *__restrict__ off, GeoParams g,
                                                   unsigned *__restrict__ tkey,
                                                   int *__restrict__ tval)
{
  const size_t s = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const TileRange r = tile_range(g, ms[s]);
  int o = off[s];
  for (int a = r.lo[0]; a <= r.hi[0]; a++)
    for (int b = r.lo[1]; b <= r.hi[1]; b++)
      for (int c = r.lo[2]; c <= r.hi[2]; c++) {
        tkey[o] = (unsigned)(((long)a * g.nt[1] + b) * g.nt[2] + c);
        tval[o] = (int)s;
        o++;
      }
}

// interpolation tile of each charge (the tile holding its window start)
__global__ __launch_bounds__(256) void k_itile_key(size_t n, const int4 *__restrict__ ms,
                                                   GeoParams g, unsigned *__restrict__ key,
                                                   int *__restrict__ val)
{
  const size_t s = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const int4 u = ms[s];
  key[s] = (unsigned)itile_of(g, u.x, u.y, u.z);
  val[s] = (int)s;
}

// Tile lists without a sort: a wavefront per tile (or Q of them, each over a
// contiguous part of the charges) tests the chunks' boxes 64 at a time, then
// the charges of the chunks that reach the tile, and places the hits with a
// ballot, so every list is in charge order.  The sorted charges of a chunk
// are near one another, so a tile opens few chunks.  COUNT writes the hits of
// (tile, part) w, FILL the list at start[w].  A charge belongs to the tile
// when its window [u, u + width) meets the tile's ts points on every axis
// (spreading: width Bn; interpolation: width 1).
struct TileGrid {
  int ts[3], nt[3], width, Q;
};
template <bool FILL>
__global__ __launch_bounds__(256) void k_tile_scan(size_t n, TileGrid g, long nw, const int4 *__restrict__ ms,
                                                   const int4 *__restrict__ chunkBox,
                                                   const int *__restrict__ start, int *__restrict__ out)
{
  const long w = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= nw) return;  // uniform per wavefront
  const int lane = threadIdx.x & 63;
  const int t = (int)(w / g.Q), q = (int)(w - (long)t * g.Q);
  const int tc[3] = {t / (g.nt[1] * g.nt[2]), (t / g.nt[2]) % g.nt[1], t % g.nt[2]};
  int lo[3], hi[3];  // window starts that reach the tile
  for (int d = 0; d < 3; d++) {
    lo[d] = tc[d] * g.ts[d] - (g.width - 1);
    hi[d] = tc[d] * g.ts[d] + g.ts[d] - 1;
  }
  const int nch = (int)((n + 63) / 64), per = (nch + g.Q - 1) / g.Q;
  const int cBeg = q * per, cEnd = min(nch, cBeg + per);
  int k = FILL ? start[w] : 0;
  for (int c0 = cBeg; c0 < cEnd; c0 += 64) {
    const int c = c0 + lane;
    bool hit = false;
    if (c < cEnd) {
      const int4 a = chunkBox[2 * c], b = chunkBox[2 * c + 1];
      hit = a.x <= hi[0] && b.x >= lo[0] && a.y <= hi[1] && b.y >= lo[1] && a.z <= hi[2] && b.z >= lo[2];
    }
    unsigned long long todo = __ballot(hit);
    while (todo) {  // uniform
      // up to four chunks at a time, their loads in flight together
      size_t s[4];
      int4 u[4];
      bool have[4];
#pragma unroll
      for (int v = 0; v < 4; v++) {
        have[v] = todo != 0;
        const int l = have[v] ? __ffsll((unsigned long long)todo) - 1 : 0;
        todo &= todo - 1;  // 0 stays 0
        s[v] = (size_t)(c0 + l) * 64 + lane;
        have[v] = have[v] && s[v] < n;
        u[v] = ms[have[v] ? s[v] : 0];
      }
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const bool in = have[v] && u[v].x >= lo[0] && u[v].x <= hi[0] && u[v].y >= lo[1] && u[v].y <= hi[1] &&
                        u[v].z >= lo[2] && u[v].z <= hi[2];
        const unsigned long long m = __ballot(in);
        if (FILL && in) out[k + __popcll(m & ((1ull << lane) - 1))] = (int)s[v];
        k += __popcll(m);
      }
    }
  }
  if (!FILL && lane == 0) out[w] = k;
}

// first entry of each tile from the starts of its parts
__global__ __launch_bounds__(256) void k_part_starts(long nt, int Q, const int *__restrict__ part,
                                                     int *__restrict__ start)
{
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t <= nt) start[t] = part[t * Q];
}

// the list walk's padding source n (place_sentinel in setup.cpp has the
// reasons).  Mixed: the first of kSentinels candidates, charge 0 moved by
// large odd constants, that no charge comes within thr of on all three axes;
// bad collects the others' bits.
constexpr int kSentinels = 16;
__device__ __forceinline__ int4 sentinel_candidate(int4 c0, int k)
{
  const unsigned m = (unsigned)(k + 1);
  return make_int4((int)((unsigned)c0.x + m * 0x9E3779B9u), (int)((unsigned)c0.y + m * 0x7F4A7C15u),
                   (int)((unsigned)c0.z + m * 0x85EBCA6Bu), 0);
}
__global__ __launch_bounds__(256) void k_sentinel_bad(size_t n, const int4 *__restrict__ src, int thr,
                                                      int *__restrict__ bad)
{
  const size_t s = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const int4 p = src[s], c0 = src[0];
  int b = 0;
#pragma unroll
  for (int k = 0; k < kSentinels; k++) {
    const int4 v = sentinel_candidate(c0, k);
    const int dx = (int)((unsigned)p.x - (unsigned)v.x), dy = (int)((unsigned)p.y - (unsigned)v.y),
              dz = (int)((unsigned)p.z - (unsigned)v.z);
    // the unsigned compare is |d| < thr for any wrapped difference
    const bool near = (unsigned)(dx + thr - 1) < (unsigned)(2 * thr - 1) &&
                      (unsigned)(dy + thr - 1) < (unsigned)(2 * thr - 1) &&
                      (unsigned)(dz + thr - 1) < (unsigned)(2 * thr - 1);
    b |= near ? 1 << k : 0;
  }
  if (b) atomicOr(bad, b);
}
__global__ void k_sentinel_set(size_t n, int4 *__restrict__ src, float4 *__restrict__ res,
                               const int *__restrict__ bad)
{
  int k = 0;
  while (k < kSentinels - 1 && ((bad[0] >> k) & 1)) k++;
  src[n] = sentinel_candidate(src[0], k);
  res[n] = make_float4(0.f, 0.f, 0.f, 0.f);
}
__global__ void k_sentinel_set64(size_t n, double4 *__restrict__ src, double csA)
{
  src[n] = make_double4(-2.0 * csA, -2.0 * csA, -2.0 * csA, 0.0);
}

// start[t] = number of entries with key < t, t = 0..nt
__global__ __launch_bounds__(256) void k_starts(long nt, const unsigned *__restrict__ skey,
                                                size_t m, int *__restrict__ start)
{
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t > nt) return;
  start[t] = (int)lower_bound_d(skey, m, (unsigned)t);
}

// neighbour-list slices of kNlSlice targets: a slice's per-lane length
// comes from its longest list; the scan input is 64 * that length (the last
// slot stays 0 for the total)
__global__ __launch_bounds__(256) void k_slice_len(size_t n, const int *__restrict__ count,
                                                   int *__restrict__ sliceLen,
                                                   long *__restrict__ sliceWords)
{
  const size_t sl = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t nSlices = (n + kNlSlice - 1) / kNlSlice;
  if (sl > nSlices) return;
  if (sl == nSlices) {
    sliceWords[sl] = 0;
    return;
  }
  int m = 0;
  const size_t b = kNlSlice * sl, e = (b + kNlSlice < n) ? b + kNlSlice : n;
  for (size_t s = b; s < e; s++) m = max(m, count[s]);
  const int ml = nlist_lane_len(m);
  sliceLen[sl] = ml;
  sliceWords[sl] = 64L * ml;
}

// zeroes m words (a fill kernel: one launch for the counters of a phase)
__global__ __launch_bounds__(256) void k_zero(size_t m, int *__restrict__ v)
{
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < m) v[i] = 0;
}

__global__ __launch_bounds__(256) void k_sort_coords(size_t n, const int *__restrict__ perm,
                                                     const double *__restrict__ coord,
                                                     double4 *__restrict__ xs)
{
  const size_t s = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const size_t i = (size_t)perm[s];
  xs[s] = make_double4(coord[3 * i], coord[3 * i + 1], coord[3 * i + 2], 0.0);
}

// per cell: count * (charges in the stencil around it), as double
__global__ __launch_bounds__(256) void k_stencil_pairs(long ncell, int nb0, int nb1, int nb2,
                                                       int nN, const int2 *__restrict__ cellSE,
                                                       double *__restrict__ out)
{
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  const int n0 = cellSE[c].y;
  double sum = 0;
  if (n0 > 0) {
    const int g2 = (int)(c % nb2), g1 = (int)((c / nb2) % nb1), g0 = (int)(c / ((long)nb1 * nb2));
    for (int dx = -nN; dx <= nN; dx++)
      for (int dy = -nN; dy <= nN; dy++)
        for (int dz = -nN; dz <= nN; dz++) {
          const int a = g0 + dx, b = g1 + dy, e = g2 + dz;
          if (a < 0 || b < 0 || e < 0 || a >= nb0 || b >= nb1 || e >= nb2) continue;
          sum += (double)cellSE[((long)a * nb1 + b) * nb2 + e].y;
        }
  }
  out[c] = (double)n0 * sum;
}

static dim3 grid_for(size_t n) { return dim3((unsigned)((n + 255) / 256)); }

static int key_bits(unsigned long maxKey)
{
  int b = 1;
  while (b < 64 && (maxKey >> b) != 0) b++;
  return b;
}

// Temporary device storage of a phase, kept until the phase's final
// stream synchronisation: the pool is shared with other streams, so memory
// returns to it only when the work that uses it has finished.
using Keep = std::deque<DevBuf>;
static void keep_or_sync(DevBuf &tmp, Keep *keep, hipStream_t s)
{
  if (keep) {
    keep->emplace_back();
    keep->back().swap(tmp);
  } else {
    NPME_HIP_CHECK(hipStreamSynchronize(s));  // tmp is released on return
  }
}

// stable sort of (key, value) pairs; temporary storage from the pool
template <typename K>
static void sort_pairs(const K *kin, K *kout, const int *vin, int *vout, size_t m, int bits,
                       hipStream_t s, Keep *keep = nullptr)
{
  size_t bytes = 0;
  NPME_HIP_CHECK(rocprim::radix_sort_pairs(nullptr, bytes, kin, kout, vin, vout, m, 0, bits, s));
  DevBuf tmp(bytes);
  NPME_HIP_CHECK(rocprim::radix_sort_pairs(tmp.p, bytes, kin, kout, vin, vout, m, 0, bits, s));
  keep_or_sync(tmp, keep, s);
}

template <typename T, typename S>
static void exclusive_scan(const T *in, S *out, size_t m, hipStream_t s, Keep *keep = nullptr)
{
  size_t bytes = 0;
  NPME_HIP_CHECK(rocprim::exclusive_scan(nullptr, bytes, in, out, (S)0, m, rocprim::plus<S>(), s));
  DevBuf tmp(bytes);
  NPME_HIP_CHECK(rocprim::exclusive_scan(tmp.p, bytes, in, out, (S)0, m, rocprim::plus<S>(), s));
  keep_or_sync(tmp, keep, s);
}

static void throw_geo_err(int e)
{
  if (e & GEO_ERR_CELL) throw Error{NPME_ERR_ARG, "coordinate outside the cell box"};
  if (e & GEO_ERR_WINDOW) throw Error{NPME_ERR_GRID, "spline window outside the compact grid"};
  if (e & GEO_ERR_FIXED) throw Error{NPME_ERR_ARG, "position outside its cluster"};
}

static void zero_words(size_t m, int *v, hipStream_t s)
{
  hipLaunchKernelGGL(k_zero, grid_for(m), dim3(256), 0, s, m, v);
  NPME_HIP_CHECK(hipGetLastError());
}

void geometry_cells_device(const GeoParams &g, size_t n, const double *d_coord, int *d_perm,
                           int4 *d_cellOf, int *d_cellSE, double4 *d_xs, hipStream_t s)
{
  const long ncell = (long)g.nb[0] * g.nb[1] * g.nb[2];
  // counters of every cell key, the closing total, the error word
  DevBuf cnt((ncell + 2) * sizeof(int)), start((ncell + 1) * sizeof(int)), key(n * sizeof(unsigned)),
      slot(n * sizeof(int)), tmp(n * sizeof(int)), gcell(n * sizeof(int4));
  int *count = (int *)cnt.p, *err = count + ncell + 1;
  zero_words((size_t)ncell + 2, count, s);
  hipLaunchKernelGGL(k_cell_keys, grid_for(n), dim3(256), 0, s, n, d_coord, g,
                     key_bits((unsigned long)ncell), (unsigned *)key.p, (int *)slot.p, count, (int4 *)gcell.p, err);
  NPME_HIP_CHECK(hipGetLastError());
  // a charge outside the box gets key 0 and cell 0, so the sort and the
  // ranges stay in bounds; the error is raised after the phase
  Keep keep;
  exclusive_scan((const int *)count, (int *)start.p, (size_t)ncell + 1, s, &keep);
  hipLaunchKernelGGL(k_cell_place, grid_for(n), dim3(256), 0, s, n, (const unsigned *)key.p,
                     (const int *)slot.p, (const int *)start.p, (int *)tmp.p);
  hipLaunchKernelGGL(k_cell_rank, grid_for(n), dim3(256), 0, s, n, (const int *)tmp.p,
                     (const unsigned *)key.p, (const int *)start.p, (const int4 *)gcell.p, d_coord, d_perm,
                     d_cellOf, d_xs, err);
  hipLaunchKernelGGL(k_cell_ranges, grid_for(ncell), dim3(256), 0, s, ncell, g, (const int *)start.p,
                     d_cellSE);
  NPME_HIP_CHECK(hipGetLastError());
  int e = 0;
  NPME_HIP_CHECK(hipMemcpyAsync(&e, err, sizeof(int), hipMemcpyDeviceToHost, s));
  NPME_HIP_CHECK(hipStreamSynchronize(s));
  throw_geo_err(e);
  if (e & GEO_LONG_BUCKET) {
    // thousands of charges in a cell: the stable radix sort
    DevBuf skey(n * sizeof(unsigned)), idx(n * sizeof(int));
    hipLaunchKernelGGL(k_iota, grid_for(n), dim3(256), 0, s, n, (int *)idx.p);
    sort_pairs((const unsigned *)key.p, (unsigned *)skey.p, (const int *)idx.p, d_perm, n,
               key_bits((unsigned long)ncell), s, &keep);
    hipLaunchKernelGGL(k_gather_cells, grid_for(n), dim3(256), 0, s, n, (const int *)d_perm,
                       (const int4 *)gcell.p, d_coord, d_cellOf, d_xs);
    NPME_HIP_CHECK(hipGetLastError());
    NPME_HIP_CHECK(hipStreamSynchronize(s));  // before the scratch returns to the pool
  }
}

// tile lists of up to this much work (tiles times the boxes they test 64 at a
// time, and ~32 opened chunks) are scanned, larger sets sorted: the scan costs
// ~25 instructions a step, twice; the radix sort of 22k charges' 77k entries
// takes 10 launches (100 us; the scan 30 us), that of 600k charges' 2.1M entries
// 120 us.  Whole set-ups, scanned / sorted, by work: 5.7e5 (1M on 256^3) 12.43 /
// 12.59 ms, 6.7e5 (300k on 360^3) 7.00 / 7.03, 9.2e5 (100k on 512^3) 3.71 / 3.67,
// 1.7e6 (300k on 512^3) 7.61 / 7.39, 4.5e6 (1M on 512^3) 14.2 / 13.0; packed sets
// may lose below the line as well (600k in a ball on 256^3, 3.7e5: 1.49 / 1.40)
constexpr double kScanWork = 1.0e6;
static bool scan_tiles(long nt, size_t n) { return (double)nt * ((double)n / 4096.0 + 32.0) <= kScanWork; }

namespace {
// the lists of one tile grid by scanning
struct TileScan {
  TileGrid g;
  size_t n;
  long nt, nw;
  const int4 *ms, *box;
  DevBuf cnt, part;
  TileScan(const int ts[3], const int ntd[3], int width, size_t n_, const int4 *ms_, const int4 *box_)
      : n(n_), ms(ms_), box(box_)
  {
    nt = 1;
    for (int d = 0; d < 3; d++) {
      g.ts[d] = ts[d];
      g.nt[d] = ntd[d];
      nt *= ntd[d];
    }
    g.width = width;
    // parts of a tile: wavefronts for the whole chip (16 a SIMD) of at least 8
    // chunks each, and of at most 256, since all charges may be in one tile
    const long nch = (long)((n + 63) / 64);
    g.Q = (int)std::max({1L, std::min(16384 / nt, (nch + 7) / 8), (nch + 255) / 256});
    nw = nt * g.Q;
    cnt.reset((nw + 1) * sizeof(int));
    part.reset((nw + 1) * sizeof(int));
  }
  const int *total() const { return (const int *)part.p + nw; }
  void count(int *d_start, Keep &keep, hipStream_t s)
  {
    zero_words(1, (int *)cnt.p + nw, s);
    hipLaunchKernelGGL(k_tile_scan<false>, dim3((unsigned)((nw + 3) / 4)), dim3(256), 0, s, n, g, nw, ms, box,
                       (const int *)nullptr, (int *)cnt.p);
    NPME_HIP_CHECK(hipGetLastError());
    exclusive_scan((const int *)cnt.p, (int *)part.p, (size_t)nw + 1, s, &keep);
    hipLaunchKernelGGL(k_part_starts, grid_for(nt + 1), dim3(256), 0, s, nt, g.Q, (const int *)part.p, d_start);
    NPME_HIP_CHECK(hipGetLastError());
  }
  void fill(int *list, hipStream_t s)
  {
    hipLaunchKernelGGL(k_tile_scan<true>, dim3((unsigned)((nw + 3) / 4)), dim3(256), 0, s, n, g, nw, ms, box,
                       (const int *)part.p, list);
    NPME_HIP_CHECK(hipGetLastError());
  }
};
}  // namespace

void geometry_charges_device(const GeoParams &g, bool fp64, size_t n, const double *d_coord,
                             const int *d_perm, const int4 *d_cellOf, void *d_src, void *d_srcRes,
                             int4 *d_ms, void *d_frac, DevBuf &tileStart, DevBuf &tileList,
                             DevBuf &itileStart, DevBuf &itileList, size_t &nTileEntries, bool listSentinel,
                             bool &sentinelPlaced, hipStream_t s)
{
  const long ntiles = (long)g.nt[0] * g.nt[1] * g.nt[2], nit = (long)g.nti[0] * g.nti[1] * g.nti[2];
  const bool scan = scan_tiles(ntiles, n), iscan = scan_tiles(nit, n);
  DevBuf ntile((n + 1) * sizeof(int)), off, box(2 * ((n + 63) / 64) * sizeof(int4));
  // back from this phase in one copy: errors, bad sentinels, list size
  DevBuf backBuf(4 * sizeof(int));
  int *back = (int *)backBuf.p;
  zero_words(4, back, s);
#define NPME_CHARGES(F64)                                                                        \
  hipLaunchKernelGGL(k_charge_setup<F64>, grid_for(n), dim3(256), 0, s, n, d_perm, d_coord, d_cellOf, g, \
                     d_src, (float4 *)d_srcRes, d_ms, d_frac, (int *)ntile.p, (int4 *)box.p, back)
  if (fp64) NPME_CHARGES(true);
  else NPME_CHARGES(false);
#undef NPME_CHARGES
  if (fp64) {
    hipLaunchKernelGGL(k_sentinel_set64, dim3(1), dim3(1), 0, s, n, (double4 *)d_src, g.csA);
  } else {
    // without a list nothing reads source n
    if (listSentinel)
      hipLaunchKernelGGL(k_sentinel_bad, grid_for(n), dim3(256), 0, s, n, (const int4 *)d_src, 1 << 20, back + 1);
    hipLaunchKernelGGL(k_sentinel_set, dim3(1), dim3(1), 0, s, n, (int4 *)d_src, (float4 *)d_srcRes, back + 1);
  }
  NPME_HIP_CHECK(hipGetLastError());
  Keep keep;
  const int wide[3] = {g.TI, g.TI, g.TI};
  TileScan ts(g.ts, g.nt, (int)g.Bn, n, d_ms, (const int4 *)box.p);
  tileStart.reset((ntiles + 1) * sizeof(int));
  itileStart.reset((nit + 1) * sizeof(int));
  itileList.reset(n * sizeof(int));
  const int *total;
  if (scan) {
    ts.count((int *)tileStart.p, keep, s);
    total = ts.total();
  } else {
    off.reset((n + 1) * sizeof(int));
    zero_words(1, (int *)ntile.p + n, s);
    exclusive_scan((const int *)ntile.p, (int *)off.p, n + 1, s, &keep);
    total = (const int *)off.p + n;
  }
  NPME_HIP_CHECK(hipMemcpyAsync(back + 2, total, sizeof(int), hipMemcpyDeviceToDevice, s));
  // the error words come back before any kernel uses the windows as indices
  int b[3] = {0, 0, 0};
  NPME_HIP_CHECK(hipMemcpyAsync(b, back, sizeof(b), hipMemcpyDeviceToHost, s));
  NPME_HIP_CHECK(hipStreamSynchronize(s));
  throw_geo_err(b[0]);
  sentinelPlaced = fp64 || !listSentinel || b[1] != (1 << kSentinels) - 1;
  const size_t m = (size_t)b[2];
  nTileEntries = m;
  tileList.reset(m * sizeof(int));
  DevBuf tk, tv, sk, ik, iv, isk;
  if (scan) {
    ts.fill((int *)tileList.p, s);
  } else {
    // emit (tile, charge) in charge order, stable sort by tile
    tk.reset(m * sizeof(unsigned));
    tv.reset(m * sizeof(int));
    sk.reset(m * sizeof(unsigned));
    hipLaunchKernelGGL(k_tile_emit, grid_for(n), dim3(256), 0, s, n, d_ms, (const int *)off.p, g,
                       (unsigned *)tk.p, (int *)tv.p);
    NPME_HIP_CHECK(hipGetLastError());
    sort_pairs((const unsigned *)tk.p, (unsigned *)sk.p, (const int *)tv.p, (int *)tileList.p, m,
               key_bits((unsigned long)ntiles), s, &keep);
    hipLaunchKernelGGL(k_starts, grid_for(ntiles + 1), dim3(256), 0, s, ntiles, (const unsigned *)sk.p, m,
                       (int *)tileStart.p);
    NPME_HIP_CHECK(hipGetLastError());
  }
  // interpolation lists: one tile per charge
  TileScan its(wide, g.nti, 1, n, d_ms, (const int4 *)box.p);
  if (iscan) {
    its.count((int *)itileStart.p, keep, s);
    its.fill((int *)itileList.p, s);
  } else {
    ik.reset(n * sizeof(unsigned));
    iv.reset(n * sizeof(int));
    isk.reset(n * sizeof(unsigned));
    hipLaunchKernelGGL(k_itile_key, grid_for(n), dim3(256), 0, s, n, d_ms, g, (unsigned *)ik.p, (int *)iv.p);
    NPME_HIP_CHECK(hipGetLastError());
    sort_pairs((const unsigned *)ik.p, (unsigned *)isk.p, (const int *)iv.p, (int *)itileList.p, n,
               key_bits((unsigned long)nit), s, &keep);
    hipLaunchKernelGGL(k_starts, grid_for(nit + 1), dim3(256), 0, s, nit, (const unsigned *)isk.p, n,
                       (int *)itileStart.p);
    NPME_HIP_CHECK(hipGetLastError());
  }
  NPME_HIP_CHECK(hipStreamSynchronize(s));  // before the scratch returns to the pool
}

__global__ __launch_bounds__(256) void k_widen(long m, const int *__restrict__ in,
                                               long *__restrict__ out)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < m) out[i] = in[i];
}

__global__ __launch_bounds__(256) void k_narrow(long m, const long *__restrict__ in,
                                                int *__restrict__ out)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < m) out[i] = (int)in[i];
}

// Cell-row segments of the direct sum without a neighbour list (k_direct):
// per block of 8 sorted targets, the contiguous source ranges of the
// cluster-rows of cells its cutoff sphere can reach, with the same FP64
// decisions (no FMA contraction) as the host build, so the segments are
// identical; COUNT writes the number per block, FILL the segments
// (sB, sE, ax, ay << 16 | az) at segStart[b], and the largest cluster
// offset from a target's cluster goes to maxOff (atomic max).
template <bool FILL>
__global__ __launch_bounds__(256) void k_cell_segments(long nBlocks, size_t n, GeoParams g,
                                                       double Rm,
                                                       const double4 *__restrict__ xs,
                                                       const int4 *__restrict__ cellOf,
                                                       const int2 *__restrict__ cellSE,
                                                       int *__restrict__ count,
                                                       const int *__restrict__ segStart,
                                                       int4 *__restrict__ segs,
                                                       int *__restrict__ maxOff)
{
#pragma clang fp contract(off)
  const long b = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nBlocks) return;
  const int nP = (int)g.nP;
  const double csB = g.csB;
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  int alo[3] = {1 << 30, 1 << 30, 1 << 30}, ahi[3] = {-1, -1, -1};
  const size_t s1 = min(n, (size_t)(8 * b + 8));
  for (size_t s = 8 * b; s < s1; s++) {
    const double4 p = xs[s];
    const int4 c = cellOf[s];
    const double px[3] = {p.x, p.y, p.z};
    const int cc[3] = {c.x, c.y, c.z};
    for (int d = 0; d < 3; d++) {
      const double x = px[d] + (-g.mn[d]);
      lo[d] = fmin(lo[d], x);
      hi[d] = fmax(hi[d], x);
      alo[d] = min(alo[d], cc[d] / nP);
      ahi[d] = max(ahi[d], cc[d] / nP);
    }
  }
  int off = 1, k = 0;
  const int start = FILL ? segStart[b] : 0;
  const int gx0 = max(0, (int)floor((lo[0] - Rm) / csB));
  const int gx1 = min(g.nb[0] - 1, (int)floor((hi[0] + Rm) / csB));
  const int gy0 = max(0, (int)floor((lo[1] - Rm) / csB));
  const int gy1 = min(g.nb[1] - 1, (int)floor((hi[1] + Rm) / csB));
  for (int gx = gx0; gx <= gx1; gx++) {
    const double gapx = fmax(0.0, fmax(gx * csB - hi[0], lo[0] - (gx + 1) * csB));
    if (gapx >= Rm) continue;
    for (int gy = gy0; gy <= gy1; gy++) {
      const double gapy = fmax(0.0, fmax(gy * csB - hi[1], lo[1] - (gy + 1) * csB));
      const double rem = Rm * Rm - gapx * gapx - gapy * gapy;
      if (rem <= 0) continue;
      const double sr = sqrt(rem);
      const int zlo = max(0, (int)floor((lo[2] - sr) / csB));
      const int zhi = min(g.nb[2] - 1, (int)floor((hi[2] + sr) / csB));
      const long row = ((long)gx * g.nb[1] + gy) * g.nb[2];
      for (int az = zlo / nP; az <= zhi / nP; az++) {
        const int z0 = max(zlo, az * nP), z1 = min(zhi, az * nP + nP - 1);
        const int sB = cellSE[row + z0].x;
        const int sE = cellSE[row + z1].x + cellSE[row + z1].y;
        if (sE > sB) {
          if (FILL) segs[start + k] = make_int4(sB, sE, gx / nP, ((gy / nP) << 16) | az);
          k++;
          const int a[3] = {gx / nP, gy / nP, az};
          for (int d = 0; d < 3; d++) off = max(off, max(abs(a[d] - alo[d]), abs(a[d] - ahi[d])));
        }
      }
    }
  }
  if (!FILL) {
    count[b] = k;
    atomicMax(maxOff, off);
  }
}

long cell_segments_device(const GeoParams &g, size_t n, double Rdir, const double4 *d_xs,
                          const int4 *d_cellOf, const int *d_cellSE, int *d_segStart,
                          DevBuf &segs, int &maxOff, hipStream_t s)
{
  const long nBlocks = ((long)n + 7) / 8;
  const double Rm = Rdir * (1.0 + 1.0e-9) + 1.0e-12;
  DevBuf cnt((nBlocks + 1) * sizeof(int)), off(sizeof(int));
  const int one = 1;
  NPME_HIP_CHECK(hipMemcpyAsync(off.p, &one, sizeof(int), hipMemcpyHostToDevice, s));
  NPME_HIP_CHECK(hipMemsetAsync((int *)cnt.p + nBlocks, 0, sizeof(int), s));
  const dim3 grid((unsigned)((nBlocks + 255) / 256));
  hipLaunchKernelGGL(k_cell_segments<false>, grid, dim3(256), 0, s, nBlocks, n, g, Rm, d_xs, d_cellOf,
                     (const int2 *)d_cellSE, (int *)cnt.p, (const int *)nullptr, (int4 *)nullptr,
                     (int *)off.p);
  NPME_HIP_CHECK(hipGetLastError());
  // segment counts in long, so an overflow of the int offsets is seen
  DevBuf wide((nBlocks + 1) * sizeof(long)), start((nBlocks + 1) * sizeof(long));
  hipLaunchKernelGGL(k_widen, grid_for(nBlocks + 1), dim3(256), 0, s, nBlocks + 1,
                     (const int *)cnt.p, (long *)wide.p);
  NPME_HIP_CHECK(hipGetLastError());
  const long total = scan_words_device((const long *)wide.p, (long *)start.p, nBlocks + 1, s);
  NPME_HIP_CHECK(hipMemcpyAsync(&maxOff, off.p, sizeof(int), hipMemcpyDeviceToHost, s));
  NPME_HIP_CHECK(hipStreamSynchronize(s));
  if (total > 0x7fffffffL) throw Error{NPME_ERR_NOMEM, "too many direct-sum segments"};
  hipLaunchKernelGGL(k_narrow, grid_for(nBlocks + 1), dim3(256), 0, s, nBlocks + 1,
                     (const long *)start.p, d_segStart);
  segs.reset(std::max<size_t>((size_t)total, 1) * sizeof(int4));
  hipLaunchKernelGGL(k_cell_segments<true>, grid, dim3(256), 0, s, nBlocks, n, g, Rm, d_xs, d_cellOf,
                     (const int2 *)d_cellSE, (int *)nullptr, (const int *)d_segStart, (int4 *)segs.p,
                     (int *)nullptr);
  NPME_HIP_CHECK(hipGetLastError());
  NPME_HIP_CHECK(hipStreamSynchronize(s));  // before the scratch returns to the pool
  return total;
}

long scan_words_device(const long *d_in, long *d_out, size_t m, hipStream_t s)
{
  exclusive_scan(d_in, d_out, m, s);
  long total = 0;
  NPME_HIP_CHECK(hipMemcpyAsync(&total, d_out + (m - 1), sizeof(long), hipMemcpyDeviceToHost, s));
  NPME_HIP_CHECK(hipStreamSynchronize(s));
  return total;
}

size_t nlist_slices_device(size_t n, const int *d_count, int *d_sliceLen, long *d_sliceStart,
                           hipStream_t s)
{
  const size_t nSlices = (n + kNlSlice - 1) / kNlSlice;
  DevBuf words((nSlices + 1) * sizeof(long));
  hipLaunchKernelGGL(k_slice_len, grid_for(nSlices + 1), dim3(256), 0, s, n, d_count, d_sliceLen,
                     (long *)words.p);
  NPME_HIP_CHECK(hipGetLastError());
  exclusive_scan((const long *)words.p, d_sliceStart, nSlices + 1, s);
  long total = 0;
  NPME_HIP_CHECK(hipMemcpyAsync(&total, d_sliceStart + nSlices, sizeof(long), hipMemcpyDeviceToHost, s));
  NPME_HIP_CHECK(hipStreamSynchronize(s));
  return (size_t)total;
}

// per-axis minimum and maximum of the coordinates: one partial per
// workgroup, then one workgroup over the partials.  Exact; a NaN
// coordinate makes its axis' bounds NaN.
__device__ __forceinline__ double nan_min(double a, double b) { return (a != a || a < b) ? a : b; }
__device__ __forceinline__ double nan_max(double a, double b) { return (a != a || b < a) ? a : b; }

constexpr int BOUNDS_WG = 1024;
__global__ __launch_bounds__(256) void k_coord_bounds(size_t n, const double *__restrict__ coord,
                                                      double *__restrict__ part)
{
  __shared__ double sh[6][256];
  double v[6] = {HUGE_VAL, HUGE_VAL, HUGE_VAL, -HUGE_VAL, -HUGE_VAL, -HUGE_VAL};
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    for (int d = 0; d < 3; d++) {
      const double x = coord[3 * i + d];
      v[d] = nan_min(x, v[d]);
      v[3 + d] = nan_max(x, v[3 + d]);
    }
  for (int d = 0; d < 6; d++) sh[d][threadIdx.x] = v[d];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int d = 0; d < 3; d++) {
        sh[d][threadIdx.x] = nan_min(sh[d][threadIdx.x + w], sh[d][threadIdx.x]);
        sh[3 + d][threadIdx.x] = nan_max(sh[3 + d][threadIdx.x + w], sh[3 + d][threadIdx.x]);
      }
    __syncthreads();
  }
  if (threadIdx.x < 6) part[6 * blockIdx.x + threadIdx.x] = sh[threadIdx.x][0];
}

__global__ __launch_bounds__(256) void k_bounds_final(int np, const double *__restrict__ part,
                                                      double *__restrict__ out)
{
  __shared__ double sh[6][256];
  double v[6] = {HUGE_VAL, HUGE_VAL, HUGE_VAL, -HUGE_VAL, -HUGE_VAL, -HUGE_VAL};
  for (int b = threadIdx.x; b < np; b += blockDim.x)
    for (int d = 0; d < 3; d++) {
      v[d] = nan_min(part[6 * b + d], v[d]);
      v[3 + d] = nan_max(part[6 * b + 3 + d], v[3 + d]);
    }
  for (int d = 0; d < 6; d++) sh[d][threadIdx.x] = v[d];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int d = 0; d < 3; d++) {
        sh[d][threadIdx.x] = nan_min(sh[d][threadIdx.x + w], sh[d][threadIdx.x]);
        sh[3 + d][threadIdx.x] = nan_max(sh[3 + d][threadIdx.x + w], sh[3 + d][threadIdx.x]);
      }
    __syncthreads();
  }
  if (threadIdx.x < 6) out[threadIdx.x] = sh[threadIdx.x][0];
}

size_t coord_bounds_scratch(size_t n)
{
  return (6 * std::min<size_t>(BOUNDS_WG, (n + 255) / 256) + 6) * sizeof(double);
}

void coord_bounds_launch(size_t n, const double *d_coord, double *d_scratch, hipStream_t s)
{
  const int nb = (int)std::min<size_t>(BOUNDS_WG, (n + 255) / 256);
  hipLaunchKernelGGL(k_coord_bounds, dim3(nb), dim3(256), 0, s, n, d_coord, d_scratch);
  hipLaunchKernelGGL(k_bounds_final, dim3(1), dim3(256), 0, s, nb, (const double *)d_scratch,
                     d_scratch + 6 * nb);
  NPME_HIP_CHECK(hipGetLastError());
}

void coord_bounds_device(size_t n, const double *d_coord, double mn[3], double mx[3], hipStream_t s)
{
  const int nb = (int)std::min<size_t>(BOUNDS_WG, (n + 255) / 256);
  DevBuf scratch(coord_bounds_scratch(n));
  coord_bounds_launch(n, d_coord, (double *)scratch.p, s);
  const double *out = (const double *)scratch.p + 6 * nb;
  double v[6];
  NPME_HIP_CHECK(hipMemcpyAsync(v, out, sizeof(v), hipMemcpyDeviceToHost, s));
  NPME_HIP_CHECK(hipStreamSynchronize(s));
  for (int d = 0; d < 3; d++) {
    mn[d] = v[d];
    mx[d] = v[3 + d];
  }
}

// ------------------------------------------------------------------ fine order
// target blocks per cell (64 charges each)
__global__ __launch_bounds__(256) void k_fine_count(long ncell, const int2 *__restrict__ cellSE,
                                                    int *__restrict__ count)
{
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c <= ncell) count[c] = c < ncell ? (cellSE[c].y + 63) / 64 : 0;
}
// a thread per sorted charge, since a cell may hold any number of them (with a
// thread per cell, 1M charges in a ball of 27 cells took 328 us)
__global__ __launch_bounds__(256) void k_fine_blocks(size_t n, int nb1, int nb2, const int4 *__restrict__ cellOf,
                                                     const int2 *__restrict__ cellSE,
                                                     const int *__restrict__ blkStart, int2 *__restrict__ blk)
{
  const size_t s = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const int4 g = cellOf[s];
  const long c = ((long)g.x * nb1 + g.y) * nb2 + g.z;
  const int r = (int)s - cellSE[c].x;
  if (r % 64 == 0) blk[blkStart[c] + r / 64] = make_int2((int)c, r);
}
// sort key: the first charge of the cell (cells keep their order), then the
// Morton index of the position in the cell, 16 steps an axis
__global__ __launch_bounds__(256) void k_fine_keys(size_t n, GeoParams g, const double4 *__restrict__ xs,
                                                   const int4 *__restrict__ cellOf,
                                                   const int2 *__restrict__ cellSE,
                                                   unsigned long *__restrict__ key, int *__restrict__ idx)
{
  const size_t s = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const double4 x = xs[s];
  const int4 c = cellOf[s];
  const double v[3] = {x.x, x.y, x.z};
  const int cc[3] = {c.x, c.y, c.z};
  unsigned m = 0;
  for (int d = 0; d < 3; d++) {
    const double f = (v[d] - g.mn[d] - cc[d] * g.csB) / g.csB * 16.0;
    const int b = min(max((int)f, 0), 15);
    for (int k = 0; k < 4; k++) m |= (unsigned)((b >> k) & 1) << (3 * k + d);
  }
  const long cl = ((long)c.x * g.nb[1] + c.y) * g.nb[2] + c.z;
  key[s] = ((unsigned long)cellSE[cl].x << 12) | m;
  idx[s] = (int)s;
}
// per fine place: the charge, its source entry and residual
__global__ __launch_bounds__(256) void k_fine_order(size_t n, const int *__restrict__ order,
                                                    const int *__restrict__ perm, int *__restrict__ permF)
{
  const size_t f = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (f < n) permF[f] = perm[order[f]];
}
template <typename V>
__global__ __launch_bounds__(256) void k_fine_move(size_t n, const int *__restrict__ order,
                                                   const V *__restrict__ in, V *__restrict__ out)
{
  const size_t f = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (f <= n) out[f] = in[f < n ? (size_t)order[f] : n];
}
// bounding boxes of the groups of 16, relative to the cells' low corner and
// widened by the rounding of positions of this extent to FP32
__global__ __launch_bounds__(256) void k_fine_boxes(long nGroups, GeoParams g, float margin,
                                                    const int2 *__restrict__ blk,
                                                    const int2 *__restrict__ cellSE,
                                                    const int *__restrict__ order,
                                                    const double4 *__restrict__ xs, float4 *__restrict__ box)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nGroups) return;
  const int2 b = blk[i / kFineSub];
  const int2 se = cellSE[b.x];
  const int k0 = b.y + kFineGroup * (int)(i % kFineSub), k1 = min(se.y, k0 + kFineGroup);
  float lo[3] = {1e30f, 1e30f, 1e30f}, hi[3] = {-1e30f, -1e30f, -1e30f};  // empty: in reach of nothing
  for (int k = k0; k < k1; k++) {
    const double4 x = xs[order[se.x + k]];
    const double v[3] = {x.x, x.y, x.z};
    for (int d = 0; d < 3; d++) {
      const float r = (float)(v[d] - g.mn[d]);
      lo[d] = fminf(lo[d], r - margin);
      hi[d] = fmaxf(hi[d], r + margin);
    }
  }
  box[2 * i] = make_float4(lo[0], lo[1], lo[2], 0.f);
  box[2 * i + 1] = make_float4(hi[0], hi[1], hi[2], 0.f);
}

int fine_blocks_device(const GeoParams &g, const int *d_cellSE, DevBuf &blkStart, hipStream_t s)
{
  const long ncell = (long)g.nb[0] * g.nb[1] * g.nb[2];
  DevBuf cnt((ncell + 1) * sizeof(int));
  blkStart.reset((ncell + 1) * sizeof(int));
  hipLaunchKernelGGL(k_fine_count, grid_for(ncell + 1), dim3(256), 0, s, ncell, (const int2 *)d_cellSE,
                     (int *)cnt.p);
  NPME_HIP_CHECK(hipGetLastError());
  exclusive_scan((const int *)cnt.p, (int *)blkStart.p, (size_t)ncell + 1, s);
  int total = 0;
  NPME_HIP_CHECK(hipMemcpyAsync(&total, (int *)blkStart.p + ncell, sizeof(int), hipMemcpyDeviceToHost, s));
  NPME_HIP_CHECK(hipStreamSynchronize(s));
  return total;
}

void fine_order_device(const GeoParams &g, size_t n, int nBlocks, const double4 *d_xs, const int4 *d_cellOf,
                       const int *d_cellSE, const int *d_perm, const int *d_blkStart, int *d_order, int *d_permF,
                       int2 *d_blk, float4 *d_box, hipStream_t s)
{
  const int2 *cse = (const int2 *)d_cellSE;
  DevBuf key(n * sizeof(unsigned long)), skey(n * sizeof(unsigned long)), idx(n * sizeof(int));
  hipLaunchKernelGGL(k_fine_blocks, grid_for(n), dim3(256), 0, s, n, g.nb[1], g.nb[2], d_cellOf, cse, d_blkStart,
                     d_blk);
  hipLaunchKernelGGL(k_fine_keys, grid_for(n), dim3(256), 0, s, n, g, d_xs, d_cellOf, cse,
                     (unsigned long *)key.p, (int *)idx.p);
  NPME_HIP_CHECK(hipGetLastError());
  sort_pairs((const unsigned long *)key.p, (unsigned long *)skey.p, (const int *)idx.p, d_order, n,
             key_bits(((unsigned long)n << 12) | 4095), s);
  hipLaunchKernelGGL(k_fine_order, grid_for(n), dim3(256), 0, s, n, d_order, d_perm, d_permF);
  double extent = 0;
  for (int d = 0; d < 3; d++) extent = std::max(extent, g.nb[d] * g.csB);
  const long ng = (long)kFineSub * nBlocks;
  hipLaunchKernelGGL(k_fine_boxes, grid_for(ng), dim3(256), 0, s, ng, g, (float)(4.0e-7 * extent), d_blk, cse,
                     d_order, d_xs, d_box);
  NPME_HIP_CHECK(hipGetLastError());
  NPME_HIP_CHECK(hipStreamSynchronize(s));  // before the scratch returns to the pool
}

void fine_sources_device(bool fp64, size_t n, const int *d_order, const void *srcS, const void *resS, void *src,
                         void *res, hipStream_t s)
{
  if (fp64) {
    hipLaunchKernelGGL(k_fine_move<double4>, grid_for(n + 1), dim3(256), 0, s, n, d_order,
                       (const double4 *)srcS, (double4 *)src);
  } else {
    hipLaunchKernelGGL(k_fine_move<float4>, grid_for(n + 1), dim3(256), 0, s, n, d_order, (const float4 *)srcS,
                       (float4 *)src);
    hipLaunchKernelGGL(k_fine_move<float4>, grid_for(n + 1), dim3(256), 0, s, n, d_order, (const float4 *)resS,
                       (float4 *)res);
  }
  NPME_HIP_CHECK(hipGetLastError());
  NPME_HIP_CHECK(hipStreamSynchronize(s));  // before the sorted copies return to the pool
}

void sorted_coords_device(size_t n, const int *d_perm, const double *d_coord, double4 *d_xs,
                          hipStream_t s)
{
  hipLaunchKernelGGL(k_sort_coords, grid_for(n), dim3(256), 0, s, n, d_perm, d_coord, d_xs);
  NPME_HIP_CHECK(hipGetLastError());
}

double stencil_candidates_device(const int nb[3], int nNeigh, const int *d_cellSE, hipStream_t s)
{
  const long ncell = (long)nb[0] * nb[1] * nb[2];
  DevBuf per(ncell * sizeof(double)), tot(sizeof(double));
  hipLaunchKernelGGL(k_stencil_pairs, grid_for(ncell), dim3(256), 0, s, ncell, nb[0], nb[1], nb[2],
                     nNeigh, (const int2 *)d_cellSE, (double *)per.p);
  NPME_HIP_CHECK(hipGetLastError());
  size_t bytes = 0;
  NPME_HIP_CHECK(rocprim::reduce(nullptr, bytes, (const double *)per.p, (double *)tot.p, 0.0,
                                 (size_t)ncell, rocprim::plus<double>(), s));
  DevBuf tmp(bytes);
  NPME_HIP_CHECK(rocprim::reduce(tmp.p, bytes, (const double *)per.p, (double *)tot.p, 0.0,
                                 (size_t)ncell, rocprim::plus<double>(), s));
  double v = 0;
  NPME_HIP_CHECK(hipMemcpyAsync(&v, tot.p, sizeof(double), hipMemcpyDeviceToHost, s));
  NPME_HIP_CHECK(hipStreamSynchronize(s));
  return v;
}

}  // namespace npme

namespace npme {
__global__ __launch_bounds__(256) void k_sentinel_near(size_t n, const int4 *__restrict__ src, int4 v,
                                                      int thr, int *__restrict__ hit)
{
  const size_t s = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const int4 p = src[s];
  const int dx = (int)((unsigned)p.x - (unsigned)v.x), dy = (int)((unsigned)p.y - (unsigned)v.y),
            dz = (int)((unsigned)p.z - (unsigned)v.z);
  if (abs(dx) < thr && abs(dy) < thr && abs(dz) < thr) hit[0] = 1;
}

bool sentinel_near_any(size_t n, const void *d_src, int4 v, int thr, hipStream_t s)
{
  DevBuf hit(sizeof(int));
  int h = 0;
  NPME_HIP_CHECK(hipMemsetAsync(hit.p, 0, sizeof(int), s));
  hipLaunchKernelGGL(k_sentinel_near, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n,
                     (const int4 *)d_src, v, thr, (int *)hit.p);
  NPME_HIP_CHECK(hipGetLastError());
  NPME_HIP_CHECK(hipMemcpyAsync(&h, hit.p, sizeof(int), hipMemcpyDeviceToHost, s));
  NPME_HIP_CHECK(hipStreamSynchronize(s));
  return h != 0;
}
}  // namespace npme
