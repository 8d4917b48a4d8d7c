// Batched 1-D FFT passes in LDS for gfx950.
//
// The reciprocal-sum convolution theta = IDFT(G . DFT(Q)) is computed on the
// zero-padded full grid (N1 x N2 x N3) but only the compact quarter-volume
// input and output (M_d = N_d/2 per axis) are ever stored:
//   A  real rows (M3) -> R2C along axis 3, length N3, K3 = N3/2+1 outputs
//   B  columns along axis 2, M2 inputs -> N2 outputs
//   C  columns along axis 1: M1 inputs, forward N1, multiply by G,
//      backward N1, M1 outputs (in place)
//   D  columns along axis 2, N2 inputs -> backward -> M2 outputs
//   E  C2R rows along axis 3, M3 real outputs
// Backward transforms use conj(DFT(conj(x))), so only forward butterflies
// exist.  The twiddle table holds exp(-2 pi i t/N) computed in FP64 on the
// host.
//
// General lengths (7-smooth, even): a Stockham transform of 2 to 4 stages
// with radices up to 16 (make_plan), every stage a switch over compile-time
// butterflies.  A thread owns whole butterflies of one column.  The first
// stage reads global memory straight into its butterflies and the last one
// writes global memory from them, so LDS carries only the exchanges between
// stages (one for two stages, two for three); in the convolution the last
// forward stage, the k-space multiply and the first backward stage are one
// step in registers: the backward transform runs the radices in reverse
// order, so its first butterflies take the rows that the forward transform's
// last ones produced.  Between the read and the write barrier of a stage a
// thread holds its butterflies in registers, so one LDS buffer suffices.
//
// What bounds it: HBM (each pass reads and writes its data once), provided
// enough loads are in flight; the LDS round trips and barriers of a stage
// are the rest, so fewer and larger radices pay.  The earlier form (radices
// 8/4/2/7/5/3, a separate LDS fill, LDS drain and G pass, ~170 VGPRs, 4096
// values a workgroup whatever the length, so 2 to 4 adjacent columns at
// lengths near 1000) took, FP32, passes A/B/C/D/E: 32/60/96/56/31 us on 256 x
// 384 x 500 (now 25/34/56/34/25: 4.4 TB/s in B), 79/124/558/119/77 on 320 x
// 320 x 1152 (now 51/90/201/89/58), 42/85/342/80/41 on 448^3 (now
// 38/65/149/68/43); FP64 120^3 15/14/23/13/14 (now 9/9/13/9/9).  Directions and
// lengths are template arguments: conditions on every stored element had
// cost passes C and D 3 to 9%.
// N = 64 and 512 have kernels of their own (below) with every index a
// compile-time constant.
#include <type_traits>

#include "npme_internal.h"

namespace npme {

template <typename R> struct Cx;
template <> struct Cx<float> { using T = float2; };
template <> struct Cx<double> { using T = double2; };

template <typename T> __device__ __forceinline__ T mk(decltype(T::x) a, decltype(T::x) b)
{
  T r;
  r.x = a;
  r.y = b;
  return r;
}
template <typename T> __device__ __forceinline__ T cadd(T a, T b) { return mk<T>(a.x + b.x, a.y + b.y); }
template <typename T> __device__ __forceinline__ T csub(T a, T b) { return mk<T>(a.x - b.x, a.y - b.y); }
template <typename T> __device__ __forceinline__ T cmul(T a, T b)
{
  return mk<T>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
template <typename T> __device__ __forceinline__ T cconj(T a) { return mk<T>(a.x, -a.y); }
template <typename T> __device__ __forceinline__ T mul_mi(T a) { return mk<T>(a.y, -a.x); }  // * -i

// p[idx] when ok, else zero, with no branch around the load: the index is
// clamped to 0 (p[0] must be readable) and the value selected afterwards.
// A load under a per-lane condition becomes an exec-masked block whose
// result is copied out at once, which waits for that load before the next
// one is issued; with the select, a thread's loads are all in flight together
template <typename T> __device__ __forceinline__ T load_or_zero(const T *p, long idx, bool ok)
{
  const T x = p[ok ? idx : 0];
  return ok ? x : mk<T>(0, 0);
}
constexpr int NT = 256;  // threads per workgroup of the 8^L kernels

// stages of a general plan: radices in forward order; for the forward (F)
// and the reversed (B) order the twiddle stride N / (Ns R) of each stage and
// the multiplier M = ceil(2^22 / Ns) with which j mod Ns is j - ((j M) >> 22)
// Ns (exact for j Ns < 2^22: j and Ns are below 2^11)
struct PlanDev {
  int N, nst;
  int radix[4];
  int strF[4], strB[4];
  unsigned magF[4], magB[4];
};

// ------------------------------------------------------------ small DFTs
// forward: y_k = sum_r x_r exp(-2 pi i r k / R)
template <typename T, int R> struct DFT;

template <typename T> struct DFT<T, 2> {
  __device__ static void run(T *x)
  {
    T a = x[0], b = x[1];
    x[0] = cadd(a, b);
    x[1] = csub(a, b);
  }
};

template <typename T> struct DFT<T, 4> {
  __device__ static void run(T *x)
  {
    T a = cadd(x[0], x[2]), b = csub(x[0], x[2]);
    T c = cadd(x[1], x[3]), d = mul_mi(csub(x[1], x[3]));
    x[0] = cadd(a, c);
    x[2] = csub(a, c);
    x[1] = cadd(b, d);
    x[3] = csub(b, d);
  }
};

template <typename T> struct DFT<T, 8> {
  __device__ static void run(T *x)
  {
    using S = decltype(T::x);
    const S c = (S)0.70710678118654752440;
    T e[4] = {x[0], x[2], x[4], x[6]};
    T o[4] = {x[1], x[3], x[5], x[7]};
    DFT<T, 4>::run(e);
    DFT<T, 4>::run(o);
    T o1 = mk<T>(c * (o[1].x + o[1].y), c * (o[1].y - o[1].x));   // * exp(-i pi/4)
    T o2 = mul_mi(o[2]);                                          // * -i
    T o3 = mk<T>(c * (o[3].y - o[3].x), -c * (o[3].x + o[3].y));  // * exp(-3i pi/4)
    x[0] = cadd(e[0], o[0]);
    x[4] = csub(e[0], o[0]);
    x[1] = cadd(e[1], o1);
    x[5] = csub(e[1], o1);
    x[2] = cadd(e[2], o2);
    x[6] = csub(e[2], o2);
    x[3] = cadd(e[3], o3);
    x[7] = csub(e[3], o3);
  }
};

template <typename T> struct DFT<T, 3> {
  __device__ static void run(T *x)
  {
    using S = decltype(T::x);
    const S s3 = (S)0.86602540378443864676;
    T t1 = cadd(x[1], x[2]);
    T t2 = mk<T>(x[0].x - (S)0.5 * t1.x, x[0].y - (S)0.5 * t1.y);
    T t3 = mk<T>(s3 * (x[1].x - x[2].x), s3 * (x[1].y - x[2].y));
    x[0] = cadd(x[0], t1);
    x[1] = cadd(t2, mul_mi(t3));
    x[2] = csub(t2, mul_mi(t3));
  }
};

// odd radix R = 5, 7: pairwise symmetric form with constant cos/sin
template <int R> struct OddTab;
template <> struct OddTab<5> {
  static constexpr double c[5] = {1.0, 0.30901699437494742410, -0.80901699437494742410,
                                  -0.80901699437494742410, 0.30901699437494742410};
  static constexpr double s[5] = {0.0, 0.95105651629515357212, 0.58778525229247312917,
                                  -0.58778525229247312917, -0.95105651629515357212};
};
template <> struct OddTab<7> {
  static constexpr double c[7] = {1.0, 0.62348980185873353053, -0.22252093395631440429,
                                  -0.90096886790241912624, -0.90096886790241912624,
                                  -0.22252093395631440429, 0.62348980185873353053};
  static constexpr double s[7] = {0.0, 0.78183148246802980871, 0.97492791218182360702,
                                  0.43388373911755812048, -0.43388373911755812048,
                                  -0.97492791218182360702, -0.78183148246802980871};
};

template <typename T, int R> struct DFTOdd {
  __device__ static void run(T *x)
  {
    using S = decltype(T::x);
    constexpr int H = (R - 1) / 2;
    T Sj[H], Dj[H];
#pragma unroll
    for (int j = 1; j <= H; j++) {
      Sj[j - 1] = cadd(x[j], x[R - j]);
      Dj[j - 1] = csub(x[j], x[R - j]);
    }
    T y[R];
    T y0 = x[0];
#pragma unroll
    for (int j = 0; j < H; j++) y0 = cadd(y0, Sj[j]);
    y[0] = y0;
#pragma unroll
    for (int k = 1; k <= H; k++) {
      T A = x[0], B = mk<T>(0, 0);
#pragma unroll
      for (int j = 1; j <= H; j++) {
        const S c = (S)OddTab<R>::c[(j * k) % R], s = (S)OddTab<R>::s[(j * k) % R];
        A.x += c * Sj[j - 1].x;
        A.y += c * Sj[j - 1].y;
        B.x += s * Dj[j - 1].x;
        B.y += s * Dj[j - 1].y;
      }
      y[k] = mk<T>(A.x + B.y, A.y - B.x);      // A - iB
      y[R - k] = mk<T>(A.x - B.y, A.y + B.x);  // A + iB
    }
#pragma unroll
    for (int k = 0; k < R; k++) x[k] = y[k];
  }
};


// cos and sin of 2 pi a / b at compile time (|angle| reduced below pi / 4
// by symmetry is not needed: 24 Taylor terms give FP64 accuracy to |x| <= pi)
constexpr double ct_pi = 3.14159265358979323846;
constexpr double ct_cos(int a, int b)
{
  a %= b;
  if (2 * a > b) a -= b;
  const double x = 2 * ct_pi * a / b;
  double s = 0, t = 1;
  for (int k = 0; k < 24; k++) {
    s += t;
    t *= -x * x / ((2 * k + 1) * (2 * k + 2));
  }
  return s;
}
constexpr double ct_sin(int a, int b)
{
  a %= b;
  if (2 * a > b) a -= b;
  const double x = 2 * ct_pi * a / b;
  double s = 0, t = x;
  for (int k = 0; k < 24; k++) {
    s += t;
    t *= -x * x / ((2 * k + 2) * (2 * k + 3));
  }
  return s;
}

template <typename T, int R> __device__ __forceinline__ void dft_any(T *x);

// R = A B with coprime factors (Good-Thomas): x[(B a + A b) mod R] is a 2-D
// A x B array, X[k] its 2-D transform at (k mod A, k mod B); no twiddles
template <typename T, int A, int B> __device__ __forceinline__ void dft_coprime(T *x)
{
  constexpr int R = A * B;
  T y[B][A];
#pragma unroll
  for (int b = 0; b < B; b++) {
#pragma unroll
    for (int a = 0; a < A; a++) y[b][a] = x[(B * a + A * b) % R];
    dft_any<T, A>(y[b]);
  }
#pragma unroll
  for (int a = 0; a < A; a++) {
    T z[B];
#pragma unroll
    for (int b = 0; b < B; b++) z[b] = y[b][a];
    dft_any<T, B>(z);
#pragma unroll
    for (int b = 0; b < B; b++) y[b][a] = z[b];
  }
#pragma unroll
  for (int k = 0; k < R; k++) x[k] = y[k % B][k % A];
}

template <int R, int I> struct TwConst {
  static constexpr double c = ct_cos(I, R), s = ct_sin(I, R);
};
// x * exp(-2 pi i I / R).  FP32: the low part of a constant is added where it
// exceeds 1e-8.  A rounded constant scales every element it meets alike, so
// its error does not average out as a table's does: with cos(pi/8) off by
// 2.8e-8, V's error on grids with a radix 16 stage was 2 to 8% above that of
// radices up to 8 (1/r, 200 boxes: 144^3 1.01, 256^3 1.08 of it); with the low
// parts it is 0.83 and 0.91 of it, for at most 2% of those passes' time.
template <typename T, int R, int I> __device__ __forceinline__ T mul_root(T x)
{
  using S = decltype(T::x);
  if constexpr (I % R == 0) return x;
  else if constexpr (4 * (I % R) == R) return mul_mi(x);
  else {
    constexpr S c = (S)TwConst<R, I>::c, s = (S)TwConst<R, I>::s;
    if constexpr (sizeof(S) == 4) {
      constexpr S dc = (S)(TwConst<R, I>::c - (double)c), ds = (S)(TwConst<R, I>::s - (double)s);
      constexpr bool lc = dc > 1e-8f || dc < -1e-8f, ls = ds > 1e-8f || ds < -1e-8f;
      S re = x.y * s, im = -x.x * s;
      if constexpr (lc && ls) {
        re = fmaf(x.y, s, fmaf(x.x, dc, x.y * ds));
        im = fmaf(-x.x, s, fmaf(x.y, dc, -x.x * ds));
      } else if constexpr (lc) {
        re = fmaf(x.y, s, x.x * dc);
        im = fmaf(-x.x, s, x.y * dc);
      } else if constexpr (ls) {
        re = fmaf(x.y, s, x.y * ds);
        im = fmaf(-x.x, s, -x.x * ds);
      }
      return mk<T>(fmaf(x.x, c, re), fmaf(x.y, c, im));
    }
    return mk<T>(x.x * c + x.y * s, x.y * c - x.x * s);
  }
}
template <typename T, int A, int K, int B0> __device__ __forceinline__ void root_row(T *y)
{
  // y[k] *= exp(-2 pi i k B0 / (A A)), k = K .. A-1
  if constexpr (K < A) {
    y[K] = mul_root<T, A * A, K * B0>(y[K]);
    root_row<T, A, K + 1, B0>(y);
  }
}
template <typename T, int A, int B0> __device__ __forceinline__ void square_rows(const T *x, T (*y)[A])
{
  if constexpr (B0 < A) {
#pragma unroll
    for (int a = 0; a < A; a++) y[B0][a] = x[A * a + B0];
    dft_any<T, A>(y[B0]);
    root_row<T, A, 1, B0>(y[B0]);
    square_rows<T, A, B0 + 1>(x, y);
  }
}
// R = A^2 (9, 16): Cooley-Tukey with compile-time twiddles
template <typename T, int A> __device__ __forceinline__ void dft_square(T *x)
{
  T y[A][A];
  square_rows<T, A, 0>(x, y);
#pragma unroll
  for (int k1 = 0; k1 < A; k1++) {
    T z[A];
#pragma unroll
    for (int b = 0; b < A; b++) z[b] = y[b][k1];
    dft_any<T, A>(z);
#pragma unroll
    for (int k2 = 0; k2 < A; k2++) x[k1 + A * k2] = z[k2];
  }
}

template <typename T, int R> __device__ __forceinline__ void dft_any(T *x)
{
  if constexpr (R == 5 || R == 7) DFTOdd<T, R>::run(x);
  else if constexpr (R == 6) dft_coprime<T, 2, 3>(x);
  else if constexpr (R == 10) dft_coprime<T, 2, 5>(x);
  else if constexpr (R == 12) dft_coprime<T, 4, 3>(x);
  else if constexpr (R == 9) dft_square<T, 3>(x);
  else if constexpr (R == 16) dft_square<T, 4>(x);
  else DFT<T, R>::run(x);
}

// ------------------------------------------------------------ general stages
// a thread's place: column c of the workgroup, the tj-th of tpc threads of
// that column; row n of the column sits at base + (n << sh) in LDS.  The
// first exchange (written by a first stage of radix R: rows j R + r) leaves
// one row free after every R, so neighbouring threads' writes spread over
// the banks: row n at n + n / R, which stays linear in r for the writer
// (j (R + 1) + r) and for the reader (j + r nb, nb a multiple of R).
struct Place {
  int c, tj, tpc;
  int base, sh;
  __device__ __forceinline__ int at(int n) const { return base + (n << sh); }
};
// rows of a column in LDS: N, and the free rows of the first exchange in
// either direction
__host__ __device__ inline int column_rows(const PlanDev &p)
{
  const int a = p.radix[0], b = p.radix[p.nst - 1];
  return p.N + p.N / (a < b ? a : b);
}

// strided layout: B = 2^lgB columns side by side
__device__ __forceinline__ Place place_cols(int lgB)
{
  Place p;
  p.c = threadIdx.x & ((1 << lgB) - 1);
  p.tj = threadIdx.x >> lgB;
  p.tpc = blockDim.x >> lgB;
  p.base = p.c;
  p.sh = lgB;
  return p;
}
// row layout: C columns one after another, tpc threads each; the threads
// past C tpc have no butterfly
__device__ __forceinline__ Place place_rows(int C, int tpc, int rows)
{
  Place p;
  p.c = threadIdx.x / tpc;
  p.tj = threadIdx.x - p.c * tpc;
  if (p.c >= C) {
    p.c = 0;
    p.tj = 1 << 24;
  }
  p.tpc = tpc;
  p.base = p.c * rows;
  p.sh = 0;
  return p;
}

// butterflies of radix R that one thread holds at a time: up to MV values or
// one butterfly.  With MV >= 14 a column of at most 4095 values needs at most
// 512 threads.
constexpr int bpt_of(int R, int MV) { return R > MV ? 1 : MV / R; }
// columns in FP32: two radix-8 butterflies (fewer, busier threads: pass C at
// 448 points 194 -> 156 us, 280^3 complex 107 -> 82 us against one); in FP64
// two would need more than 128 VGPRs (512-point pass C 434 -> 516 us), and
// row passes are slower with two as well
template <typename Real, bool ROWS> constexpr int hold() { return sizeof(Real) == 4 && !ROWS ? 16 : 14; }

// one call of f(integral_constant<int, R>) for the plan's radix
template <bool EVEN, typename F> __device__ __forceinline__ void with_radix(int R, F &&f)
{
  switch (R) {
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 10: f(std::integral_constant<int, 10>{}); break;
    case 12: f(std::integral_constant<int, 12>{}); break;
    case 16: f(std::integral_constant<int, 16>{}); break;
    default:
      if constexpr (!EVEN) {
        switch (R) {
          case 3: f(std::integral_constant<int, 3>{}); break;
          case 5: f(std::integral_constant<int, 5>{}); break;
          case 7: f(std::integral_constant<int, 7>{}); break;
          case 9: f(std::integral_constant<int, 9>{}); break;
          default: break;
        }
      }
      break;
  }
}

// first stage (Ns = 1): butterfly j takes the elements get(j, r nb), that
// is rows j + r nb with nb = N/R, and writes rows j R + r (with the free
// rows).  HALF: the elements from N/2 on are zero and not read (R is even
// then).  get runs for every slot (butterfly 0 in place of those past the
// last), so no load sits behind a per-lane branch and a thread's loads are
// all in flight together.  INLDS: get reads this column from LDS.
template <typename T, int MV, bool HALF, bool INLDS, typename G>
__device__ __forceinline__ void stage_first(T *lds, const Place &p, int N, int R0, G &&get)
{
  with_radix<HALF>(R0, [&](auto rc) {
    constexpr int R = decltype(rc)::value, BPT = bpt_of(R, MV);
    const int nb = N / R;
    T v[BPT][R];
#pragma unroll
    for (int u = 0; u < BPT; u++) {
      const int j = p.tj + u * p.tpc, jj = j < nb ? j : 0;
#pragma unroll
      for (int r = 0; r < R; r++) v[u][r] = (HALF && r >= R / 2) ? mk<T>(0, 0) : get(jj, r * nb);
    }
    if constexpr (INLDS) __syncthreads();
#pragma unroll
    for (int u = 0; u < BPT; u++) {
      const int j = p.tj + u * p.tpc;
      if (j < nb) {
        dft_any<T, R>(v[u]);
        T *w = lds + p.at(j * (R + 1));
#pragma unroll
        for (int r = 0; r < R; r++) w[r << p.sh] = v[u][r];
      }
    }
  });
  __syncthreads();
}

// inner stage: reads x[j + r nb], nb = N/R, twiddles by w^(r k N/(Ns R)), k
// = j mod Ns, writes y[(j - k) R + k + r Ns]; in LDS, in place.  gap: the
// rows read are those of the first exchange (a free row after every Ns)
template <typename T, int MV>
__device__ __forceinline__ void stage_inner(T *lds, const Place &p, int N, int Rs, int Ns, int str,
                                            unsigned mag, bool gap, const T *tw)
{
  with_radix<false>(Rs, [&](auto rc) {
    constexpr int R = decltype(rc)::value, BPT = bpt_of(R, MV);
    const int nb = N / R;
    const int step = (gap ? nb + nb / Ns : nb) << p.sh;
    T v[BPT][R];
    int q[BPT];  // j / Ns
#pragma unroll
    for (int u = 0; u < BPT; u++) {
      const int j = p.tj + u * p.tpc;
      q[u] = (int)(((unsigned)j * mag) >> 22);
      if (j < nb) {
        const T *x = lds + p.at(gap ? j + q[u] : j);
#pragma unroll
        for (int r = 0; r < R; r++) v[u][r] = x[r * step];
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < BPT; u++) {
      const int j = p.tj + u * p.tpc;
      if (j < nb) {
        const int qN = q[u] * Ns, k = j - qN;
        const T *t = tw;
        const int ks = k * str;
#pragma unroll
        for (int r = 1; r < R; r++) {
          t += ks;
          v[u][r] = cmul(v[u][r], *t);
        }
        dft_any<T, R>(v[u]);
        T *y = lds + p.at(qN * R + k);
#pragma unroll
        for (int r = 0; r < R; r++) y[r * Ns << p.sh] = v[u][r];
      }
    }
  });
  __syncthreads();
}

// rows j + r nb of a last stage (Ns = nb) into v; gap: two-stage plans read
// the first exchange, whose free rows come after every nb
template <typename T, int R>
__device__ __forceinline__ void last_read(const T *lds, const Place &p, int j, int nb, bool gap, T *v)
{
  const T *x = lds + p.at(j);
  const int step = (gap ? nb + 1 : nb) << p.sh;
#pragma unroll
  for (int r = 0; r < R; r++) v[r] = x[r * step];
}
template <typename T, int R> __device__ __forceinline__ void last_dft(const T *tw, int j, T *v)
{
  const T *t = tw;
#pragma unroll
  for (int r = 1; r < R; r++) {
    t += j;
    v[r] = cmul(v[r], *t);
  }
  dft_any<T, R>(v);
}

// last stage (Ns = N/R, so k = j): put(j, low, r nb, value) receives row j +
// r nb; low: r < R/2, for an even radix the rows below N/2 (known at compile
// time).  TOLDS: put writes this column in LDS
template <typename T, int MV, bool TOLDS, typename P>
__device__ __forceinline__ void stage_last(T *lds, const Place &p, int N, int Rs, bool gap, const T *tw, P &&put)
{
  with_radix<false>(Rs, [&](auto rc) {
    constexpr int R = decltype(rc)::value, BPT = bpt_of(R, MV);
    const int nb = N / R;
    T v[BPT][R];
#pragma unroll
    for (int u = 0; u < BPT; u++) {
      const int j = p.tj + u * p.tpc;
      if (j < nb) last_read<T, R>(lds, p, j, nb, gap, v[u]);
    }
    if constexpr (TOLDS) __syncthreads();
#pragma unroll
    for (int u = 0; u < BPT; u++) {
      const int j = p.tj + u * p.tpc;
      if (j < nb) {
        last_dft<T, R>(tw, j, v[u]);
#pragma unroll
        for (int r = 0; r < R; r++) put(j, 2 * r < R, r * nb, v[u][r]);
      }
    }
  });
}

// last forward stage, f(g, value) on its rows with g = pre(j, r nb) (a load
// issued before the stage), first backward stage of the same radix: rows j +
// r N/R in, j R + r (with the free rows) out
template <typename T, int MV, typename GT, typename L, typename F>
__device__ __forceinline__ void stage_turn(T *lds, const Place &p, int N, int Rs, bool gap, const T *tw, L &&pre,
                                           F &&f)
{
  with_radix<false>(Rs, [&](auto rc) {
    constexpr int R = decltype(rc)::value, BPT = bpt_of(R, MV);
    const int nb = N / R;
    T v[BPT][R];
    GT g[BPT][R];
#pragma unroll
    for (int u = 0; u < BPT; u++) {
      const int j = p.tj + u * p.tpc, jj = j < nb ? j : 0;
#pragma unroll
      for (int r = 0; r < R; r++) g[u][r] = pre(jj, r * nb);
    }
#pragma unroll
    for (int u = 0; u < BPT; u++) {
      const int j = p.tj + u * p.tpc;
      if (j < nb) last_read<T, R>(lds, p, j, nb, gap, v[u]);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < BPT; u++) {
      const int j = p.tj + u * p.tpc;
      if (j < nb) {
        last_dft<T, R>(tw, j, v[u]);
#pragma unroll
        for (int r = 0; r < R; r++) v[u][r] = f(g[u][r], v[u][r]);
        dft_any<T, R>(v[u]);
        T *w = lds + p.at(j * (R + 1));
#pragma unroll
        for (int r = 0; r < R; r++) w[r << p.sh] = v[u][r];
      }
    }
  });
  __syncthreads();
}

// the inner stages of a transform, in forward or reversed radix order
template <typename T, int MV>
__device__ __forceinline__ void stages_inner(T *lds, const Place &p, const PlanDev &pl, bool rev, const T *tw)
{
  int Ns = pl.radix[rev ? pl.nst - 1 : 0];
  for (int s = 1; s < pl.nst - 1; s++) {
    const int i = rev ? pl.nst - 1 - s : s;
    stage_inner<T, MV>(lds, p, pl.N, pl.radix[i], Ns, rev ? pl.strB[s] : pl.strF[s],
                rev ? pl.magB[s] : pl.magF[s], s == 1, tw);
    Ns *= pl.radix[i];
  }
}

// the twiddle table, copied into LDS behind the columns (a butterfly reads
// R - 1 of them; from LDS rather than a global load each); ordered by the
// barrier that ends the first stage
template <typename T>
__device__ __forceinline__ const T *twiddles_in(T *lds, int ldsElems, int N, const T *tw)
{
  T *tl = lds + ldsElems;
  for (int i = threadIdx.x; i < N; i += blockDim.x) tl[i] = tw[i];
  return tl;
}

// workgroups are dealt round-robin to the 8 XCDs; remap so each XCD walks a
// contiguous range of columns (adjacent column groups share L2 lines)
__device__ __forceinline__ int xcd_wg()
{
  const int wg = blockIdx.x, nwg = gridDim.x;
  const int x = wg & 7, local = wg >> 3, q = nwg >> 3, r = nwg & 7;
  return x * q + min(x, r) + local;
}

// ------------------------------------------------------------ pass kernels
// generic complex pass.  Column col = o * nInner + i;
// element n at o * outer + i * inner + n * pos (all element counts < 2^31).
struct CGeom {
  int N, Lin, Lout;
  int nCols, nInner, validInner;  // inner index >= validInner: padding column
  int inOuter, inInner, inPos, outOuter, outInner, outPos;
};

// threads of a workgroup at most (FP64 butterflies need twice the registers)
template <typename Real> constexpr int max_threads() { return sizeof(Real) == 4 ? 1024 : 512; }

// which elements of a column a pass reads and keeps, and its direction: FWD
// (pass B; A of complex charges) reads the first N/2 (the rest are zero) and
// keeps all, BACK (D; E) transforms backward, in reversed radix order, and
// keeps the first N/2 (the first radix of a plan is even, the end at which
// half the elements are missing), WHOLE is any forward transform
enum { PASS_FWD, PASS_BACK, PASS_WHOLE };

// strided columns (passes B and D)
template <typename Real, int MODE>
__global__ __launch_bounds__(max_threads<Real>()) void k_fft_cols(CGeom g, PlanDev pl,
                                                                  const typename Cx<Real>::T *tw,
                                                                  const typename Cx<Real>::T *__restrict__ in,
                                                                  typename Cx<Real>::T *__restrict__ out,
                                                                  int lgB)
{
  using T = typename Cx<Real>::T;
  constexpr int MV = hold<Real, false>();
  extern __shared__ char smem_raw[];
  T *lds = reinterpret_cast<T *>(smem_raw);
  const int N = g.N;
  const Place p = place_cols(lgB);
  const int colg = (xcd_wg() << lgB) + p.c;
  const int o0 = colg / g.nInner;
  const bool valid = colg < g.nCols && colg - o0 * g.nInner < g.validInner;
  const int o = valid ? o0 : 0, i = valid ? colg - o0 * g.nInner : 0;
  const T *src = in + ((long)o * g.inOuter + (long)i * g.inInner);
  const T *twl = twiddles_in(lds, column_rows(pl) << lgB, N, tw);
  constexpr bool rev = MODE == PASS_BACK;
  // an invalid column reads column 0 and is not stored
  stage_first<T, MV, MODE == PASS_FWD, false>(lds, p, N, pl.radix[rev ? pl.nst - 1 : 0], [&](int j, int rnb) {
    if constexpr (MODE == PASS_WHOLE) {
      return load_or_zero(src, (long)(j + rnb) * g.inPos, j + rnb < g.Lin);
    } else {
      const T x = (src + (long)j * g.inPos)[(long)rnb * g.inPos];
      return rev ? cconj(x) : x;
    }
  });
  stages_inner<T, MV>(lds, p, pl, rev, twl);
  T *dst = out + ((long)o * g.outOuter + (long)i * g.outInner);
  stage_last<T, MV, false>(lds, p, N, pl.radix[rev ? 0 : pl.nst - 1], pl.nst == 2, twl,
                       [&](int j, bool low, int rnb, T v) {
    const bool keep = MODE == PASS_BACK ? low : MODE == PASS_FWD || j + rnb < g.Lout;
    if (keep && valid) (dst + (long)j * g.outPos)[(long)rnb * g.outPos] = rev ? cconj(v) : v;
  });
}

// contiguous rows (passes A and E of complex charges): C rows a workgroup
template <typename Real, int MODE>
__global__ __launch_bounds__(max_threads<Real>()) void k_fft_rows(CGeom g, PlanDev pl,
                                                                  const typename Cx<Real>::T *tw,
                                                                  const typename Cx<Real>::T *__restrict__ in,
                                                                  typename Cx<Real>::T *__restrict__ out, int C,
                                                                  int tpc)
{
  using T = typename Cx<Real>::T;
  constexpr int MV = hold<Real, true>();
  extern __shared__ char smem_raw[];
  T *lds = reinterpret_cast<T *>(smem_raw);
  const int N = g.N;
  const Place p = place_rows(C, tpc, column_rows(pl));
  const int row = xcd_wg() * C + p.c;
  const bool valid = row < g.nCols;
  const int i = valid ? row : 0;
  const T *src = in + (long)i * g.inInner;
  T *dst = out + (long)i * g.outInner;
  const T *twl = twiddles_in(lds, C * column_rows(pl), N, tw);
  constexpr bool rev = MODE == PASS_BACK;
  stage_first<T, MV, MODE == PASS_FWD, false>(lds, p, N, pl.radix[rev ? pl.nst - 1 : 0], [&](int j, int rnb) {
    if constexpr (MODE == PASS_WHOLE) {
      return load_or_zero(src, j + rnb, j + rnb < g.Lin);
    } else {
      const T x = (src + j)[rnb];
      return rev ? cconj(x) : x;
    }
  });
  stages_inner<T, MV>(lds, p, pl, rev, twl);
  stage_last<T, MV, false>(lds, p, N, pl.radix[rev ? 0 : pl.nst - 1], pl.nst == 2, twl,
                       [&](int j, bool low, int rnb, T v) {
    const bool keep = MODE == PASS_BACK ? low : MODE == PASS_FWD || j + rnb < g.Lout;
    if (keep && valid) (dst + j)[rnb] = rev ? cconj(v) : v;
  });
}

// pass A: two real rows per complex row, R2C by the two-for-one split (Lin
// = N/2 data values a row)
template <typename Real>
__global__ __launch_bounds__(max_threads<Real>()) void k_fft_r2c(int nPairs, int inRow, int outRow,
                                                                 PlanDev pl, const typename Cx<Real>::T *tw,
                                                                 const Real *__restrict__ in,
                                                                 typename Cx<Real>::T *__restrict__ out, int C,
                                                                 int tpc)
{
  using T = typename Cx<Real>::T;
  constexpr int MV = hold<Real, true>();
  extern __shared__ char smem_raw[];
  T *lds = reinterpret_cast<T *>(smem_raw);
  const int N = pl.N;
  const Place p = place_rows(C, tpc, column_rows(pl));
  const int pr = xcd_wg() * C + p.c;
  const bool valid = pr < nPairs;
  const Real *ra = in + (valid ? (long)(2 * pr) * inRow : 0), *rb = ra + inRow;
  const T *twl = twiddles_in(lds, C * column_rows(pl), N, tw);
  stage_first<T, MV, true, false>(lds, p, N, pl.radix[0],
                              [&](int j, int rnb) { return mk<T>((ra + j)[rnb], (rb + j)[rnb]); });
  stages_inner<T, MV>(lds, p, pl, false, twl);
  stage_last<T, MV, true>(lds, p, N, pl.radix[pl.nst - 1], pl.nst == 2, twl,
                      [&](int j, bool, int rnb, T v) { (lds + p.at(j))[rnb] = v; });
  __syncthreads();
  if (!valid) return;
  const Real h = (Real)0.5;
  T *oa = out + (long)(2 * pr) * outRow, *ob = oa + outRow;
  for (int k = p.tj; k <= N / 2; k += tpc) {
    const T z = lds[p.at(k)];
    const T w = cconj(lds[p.at(k == 0 ? 0 : N - k)]);
    const T s = cadd(z, w), d = csub(z, w);
    oa[k] = mk<T>(h * s.x, h * s.y);
    ob[k] = mk<T>(h * d.y, -h * d.x);  // -i d / 2
  }
}

// pass E: Hermitian half rows -> two real rows (backward transform)
template <typename Real>
__global__ __launch_bounds__(max_threads<Real>()) void k_fft_c2r(int nPairs, int inRow, int outRow,
                                                                 PlanDev pl, const typename Cx<Real>::T *tw,
                                                                 const typename Cx<Real>::T *__restrict__ in,
                                                                 Real *__restrict__ out, int C, int tpc)
{
  using T = typename Cx<Real>::T;
  constexpr int MV = hold<Real, true>();
  extern __shared__ char smem_raw[];
  T *lds = reinterpret_cast<T *>(smem_raw);
  const int N = pl.N, h = N / 2;
  const Place p = place_rows(C, tpc, column_rows(pl));
  const int pr = xcd_wg() * C + p.c;
  const bool valid = pr < nPairs;
  const T *ia = in + (valid ? (long)(2 * pr) * inRow : 0), *ib = ia + inRow;
  const T *twl = twiddles_in(lds, C * column_rows(pl), N, tw);
  // each stored element m = 0 .. N/2 of the two Hermitian rows is loaded
  // once and gives both elements n = m and n = N - m of the column:
  // Z = Xa + i Xb (n <= N/2), conj(Xa) + i conj(Xb) above; stored conj(Z).
  // Four elements' loads are in flight together.
  for (int m0 = p.tj; m0 <= h; m0 += 4 * tpc) {
    T a[4], b[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int m = m0 + u * tpc;
      a[u] = ia[m <= h ? m : 0];
      b[u] = ib[m <= h ? m : 0];
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int m = m0 + u * tpc;
      if (m <= h) {
        lds[p.at(m)] = mk<T>(a[u].x - b[u].y, -(a[u].y + b[u].x));
        if (m > 0 && m < h) lds[p.at(N - m)] = mk<T>(a[u].x + b[u].y, a[u].y - b[u].x);
      }
    }
  }
  __syncthreads();
  // reversed radix order: the stage that writes half its elements is the
  // last one
  stage_first<T, MV, false, true>(lds, p, N, pl.radix[pl.nst - 1], [&](int j, int rnb) { return (lds + p.at(j))[rnb]; });
  stages_inner<T, MV>(lds, p, pl, true, twl);
  Real *oa = out + (long)(2 * pr) * outRow, *ob = oa + outRow;
  stage_last<T, MV, false>(lds, p, N, pl.radix[0], pl.nst == 2, twl, [&](int j, bool low, int rnb, T z) {
    if (low && valid) {
      (oa + j)[rnb] = z.x;  // z: conj of the backward transform
      (ob + j)[rnb] = -z.y;
    }
  });
}

// G of pass C.  GM 0: real G at (|k1|, |k2|, k3); GM 1: complex G at
// (|k1|, |k2|, k3 or |k3|) -- the radial kernels, whose grid is even; GM 2:
// complex G at (k1, k2, k3) over the full N1 x N2 x G3 grid (translated
// kernels), where gfl selects k -> -k per axis (bits 1, 2, 4) and the
// conjugate (bit 8).  Layout G[a2][a3 / 8][a1][a3 % 8], a1 over A1 values.
struct GIndex {
  long base;
  int A1;
};
__device__ __forceinline__ int g_neg(int k, int N) { return k ? N - k : 0; }
template <int GM>
__device__ __forceinline__ GIndex g_index(int N, int N2, int Kv, int N3fold, int gfl, bool valid,
                                          int colg, int C3)
{
  const int k2 = valid ? colg / C3 : 0, k3 = valid ? colg - k2 * C3 : 0;
  int a2, a3, G3, A1;
  if constexpr (GM == 2) {
    a2 = (gfl & 2) ? g_neg(k2, N2) : k2;
    a3 = (gfl & 4) ? g_neg(k3, N3fold) : k3;
    G3 = Kv;
    A1 = N;
  } else {
    a2 = (k2 <= N2 / 2) ? k2 : N2 - k2;
    a3 = (N3fold > 0 && k3 > N3fold / 2) ? N3fold - k3 : k3;
    G3 = N3fold > 0 ? (N3fold / 2 + 1) : Kv;
    A1 = N / 2 + 1;
  }
  GIndex r;
  r.base = (((long)a2 * ((G3 + 7) >> 3) + (a3 >> 3)) * A1) * 8 + (a3 & 7);
  r.A1 = A1;
  return r;
}
template <int GM> __device__ __forceinline__ int g_a1(int n, int N, int gfl)
{
  if constexpr (GM == 2) return (gfl & 1) ? g_neg(n, N) : n;
  else return (n <= N / 2) ? n : N - n;
}

// pass C: forward along axis 1 (Lin = N/2 rows of data), X <- X G, backward,
// keep the first N/2 outputs.  Columns c = k2 * C3 + k3.
template <typename Real, int GM>
__global__ __launch_bounds__(max_threads<Real>()) void k_fft_conv(int nCols, int pos, int N2, int gfl, int C3,
                                                                  int Kv, int N3fold, PlanDev pl,
                                                                  const typename Cx<Real>::T *tw, const void *Gv,
                                                                  typename Cx<Real>::T *__restrict__ data, int lgB)
{
  constexpr bool CG = GM > 0;
  using T = typename Cx<Real>::T;
  using GT = typename std::conditional<CG, T, Real>::type;
  constexpr int MV = hold<Real, false>();
  extern __shared__ char smem_raw[];
  T *lds = reinterpret_cast<T *>(smem_raw);
  const int N = pl.N;
  const Place p = place_cols(lgB);
  const int colg = (xcd_wg() << lgB) + p.c;
  // C3: row length of the data (padded); Kv: valid entries of a row
  const bool valid = colg < nCols && colg % C3 < Kv;
  T *col = data + (valid ? colg : 0);
  const T *twl = twiddles_in(lds, column_rows(pl) << lgB, N, tw);
  const GIndex gi = g_index<GM>(N, N2, Kv, N3fold, gfl, valid, colg, C3);
  const GT *Gp = reinterpret_cast<const GT *>(Gv) + gi.base;
  // an invalid column reads column 0 and is not stored
  stage_first<T, MV, true, false>(lds, p, N, pl.radix[0],
                              [&](int j, int rnb) { return (col + (long)j * pos)[(long)rnb * pos]; });
  stages_inner<T, MV>(lds, p, pl, false, twl);
  // times G, conjugated for the backward transform
  auto load_g = [&](int j, int rnb) {
    GT gv = Gp[g_a1<GM>(j + rnb, N, gfl) * 8];
    if constexpr (GM == 2)
      if (gfl & 8) gv = cconj(gv);
    return gv;
  };
  stage_turn<T, MV, GT>(lds, p, N, pl.radix[pl.nst - 1], pl.nst == 2, twl, load_g, [&](GT gv, T x) {
    if constexpr (CG) return cconj(cmul(x, gv));
    else return mk<T>(gv * x.x, -gv * x.y);
  });
  stages_inner<T, MV>(lds, p, pl, true, twl);
  stage_last<T, MV, false>(lds, p, N, pl.radix[0], pl.nst == 2, twl, [&](int j, bool low, int rnb, T v) {
    if (low && valid) (col + (long)j * pos)[(long)rnb * pos] = cconj(v);
  });
}

// ------------------------------------------------------------ N = 8^L passes
// Strided passes (B, C, D) for N = 8^L (64, 512) with every index known at
// compile time: 4096 / N columns per workgroup, each thread owns two
// radix-8 butterflies of one column per stage.  The first stage reads its
// eight inputs straight from global memory (rows j + r N/8; with HIN only
// the first N/2 rows are non-zero, so four of them) and the last stage
// writes straight to global memory, so LDS carries only the L-1 exchanges
// between stages.  In the convolution the outputs of the forward transform's
// last stage are exactly the inputs of the backward transform's first stage
// for the same thread (rows j + r N/8), so the k-space multiply and the
// conjugation happen in registers between the two transforms.
template <typename T> __device__ __forceinline__ void dft8_half(T *x)
{
  // DFT8 of (x0, x1, x2, x3, 0, 0, 0, 0)
  using S = decltype(T::x);
  const S c = (S)0.70710678118654752440;
  // even part DFT4(x0, x2, 0, 0) = (x0 + x2, x0 - i x2, x0 - x2, x0 + i x2)
  const T e0 = cadd(x[0], x[2]), e2 = csub(x[0], x[2]);
  const T e1 = cadd(x[0], mul_mi(x[2])), e3 = csub(x[0], mul_mi(x[2]));
  const T o0 = cadd(x[1], x[3]), o2 = csub(x[1], x[3]);
  const T o1 = cadd(x[1], mul_mi(x[3])), o3 = csub(x[1], mul_mi(x[3]));
  const T t1 = mk<T>(c * (o1.x + o1.y), c * (o1.y - o1.x));   // * exp(-i pi/4)
  const T t2 = mul_mi(o2);                                    // * -i
  const T t3 = mk<T>(c * (o3.y - o3.x), -c * (o3.x + o3.y));  // * exp(-3i pi/4)
  x[0] = cadd(e0, o0);
  x[4] = csub(e0, o0);
  x[1] = cadd(e1, t1);
  x[5] = csub(e1, t1);
  x[2] = cadd(e2, t2);
  x[6] = csub(e2, t2);
  x[3] = cadd(e3, t3);
  x[7] = csub(e3, t3);
}

// the twiddle table: in LDS behind the columns in FP32 (FP64 columns fill 64
// KB and read it from global memory)
template <typename T> __device__ __forceinline__ const T *twiddles8(T *lds, int ldsElems, int N, const T *tw)
{
  if constexpr (sizeof(T) == 8) return twiddles_in(lds, ldsElems, N, tw);
  else return tw;
}

template <int L> struct P8 {
  static constexpr int N = L == 2 ? 64 : 512;
  static constexpr int NB = N / 8;          // butterflies per column and stage
  static constexpr int LGB = L == 2 ? 6 : 3;  // columns per workgroup: 4096 / N
  static constexpr int B = 1 << LGB;
  static constexpr int TPC = NT / B;        // threads per column
  static constexpr int BPT = NB / TPC;      // butterflies per thread
};

// LDS slot of (row, column c) of a radix-8 workgroup: rows of B columns.
// For the 512-point FP32 kernels a row (8 columns of 8 bytes) covers half of
// the LDS banks, and which half follows the row's parity; the first stage's
// writes of one wavefront go to rows 8 apart, all of one parity, so the rows
// of every odd group of 8 are stored pairwise swapped (row ^ 1): the
// wavefront's writes then alternate halves.  The other stages access whole
// groups of 8 consecutive rows, which the swap only permutes.
template <typename T, int L> constexpr bool lds_swap8() { return L == 3 && sizeof(T) == 8; }
template <typename T, int L> __device__ __forceinline__ int slot8(int row, int c)
{
  using P = P8<L>;
  if constexpr (lds_swap8<T, L>()) return ((row ^ ((row >> 3) & 1)) << P::LGB) + c;
  else return (row << P::LGB) + c;
}
// LDS elements of the columns (the twiddle table follows them)
template <typename T, int L> constexpr int lds_elems8() { return P8<L>::N << P8<L>::LGB; }

// middle stage NS of a column: read x[j + r NB], twiddle, DFT8, write
// y[(j - k) 8 + k + r NS] (LDS index * B + c), with a barrier between the
// reads and the writes
template <typename T, int L, int NS>
__device__ __forceinline__ void mid8(T *lds, int c, int tj, const T *tw)
{
  using P = P8<L>;
  T v[P::BPT][8];
#pragma unroll
  for (int u = 0; u < P::BPT; u++) {
    const int j = tj + u * P::TPC;
#pragma unroll
    for (int r = 0; r < 8; r++) v[u][r] = lds[slot8<T, L>(j + r * P::NB, c)];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < P::BPT; u++) {
    const int j = tj + u * P::TPC, k = j & (NS - 1);
    constexpr int stride = P::N / (8 * NS);
#pragma unroll
    for (int r = 1; r < 8; r++) v[u][r] = cmul(v[u][r], tw[r * k * stride]);
    DFT<T, 8>::run(v[u]);
    const int o = (j - k) * 8 + k;
#pragma unroll
    for (int r = 0; r < 8; r++) lds[slot8<T, L>(o + r * NS, c)] = v[u][r];
  }
  __syncthreads();
}

// last stage (NS = NB): k = j, outputs rows j + r NB, kept in registers
template <typename T, int L>
__device__ __forceinline__ void last8(T *lds, int c, int tj, const T *tw, T (*v)[8])
{
  using P = P8<L>;
#pragma unroll
  for (int u = 0; u < P::BPT; u++) {
    const int j = tj + u * P::TPC;
#pragma unroll
    for (int r = 0; r < 8; r++) v[u][r] = lds[slot8<T, L>(j + r * P::NB, c)];
  }
#pragma unroll
  for (int u = 0; u < P::BPT; u++) {
    const int j = tj + u * P::TPC;
#pragma unroll
    for (int r = 1; r < 8; r++) v[u][r] = cmul(v[u][r], tw[r * j]);
    DFT<T, 8>::run(v[u]);
  }
}

// first stage (NS = 1) from registers holding rows j + r NB: DFT8, write
// y[8 j + r]
template <typename T, int L, bool HALF>
__device__ __forceinline__ void first8(T *lds, int c, int tj, T (*v)[8])
{
  using P = P8<L>;
#pragma unroll
  for (int u = 0; u < P::BPT; u++) {
    const int j = tj + u * P::TPC;
    if constexpr (HALF) dft8_half(v[u]);
    else DFT<T, 8>::run(v[u]);
#pragma unroll
    for (int r = 0; r < 8; r++) lds[slot8<T, L>(8 * j + r, c)] = v[u][r];
  }
  __syncthreads();
}

// the transform of one column after its first stage: stages 1 .. L-1
template <typename T, int L>
__device__ __forceinline__ void rest8(T *lds, int c, int tj, const T *tw, T (*v)[8])
{
  if constexpr (L == 3) mid8<T, L, 8>(lds, c, tj, tw);
  last8<T, L>(lds, c, tj, tw, v);
}

// element r NB rows on from a thread's first one: the rows' offset is uniform
// (scalar registers), the thread's own in 32 bits for FP32 (the passes bound
// a column's elements to 2^31 over N / 2 rows, so N / 8 rows stay below 4 GB),
// which costs no vector instruction per access; 64 bits for FP64
template <typename Real> using LaneOff = typename std::conditional<sizeof(Real) == 4, unsigned, size_t>::type;
template <typename T, typename O> __device__ __forceinline__ T *row_at(T *base, long rows, O lane)
{
  return reinterpret_cast<T *>(reinterpret_cast<char *>(base + rows) + lane);
}
template <typename T, typename O> __device__ __forceinline__ const T *row_at(const T *base, long rows, O lane)
{
  return reinterpret_cast<const T *>(reinterpret_cast<const char *>(base + rows) + lane);
}

// passes B (HIN: the first half of the rows non-zero, all stored) and D
// (BACK: backward, the first half stored), and whole forward columns: column
// o * nInner + i, element n at o * outer + i * inner + n * pos.  These passes
// are bound by instruction issue rather than by HBM or LDS (512 points FP32:
// smaller working sets that stay in the memory-side cache, or half the LDS
// traffic with 16 x 32 points, are no faster), so direction and lengths are
// template arguments and row offsets scalar: 643 -> 564 vector instructions
// per 16 elements in B, none of them 64-bit multiplies, 86 -> 79 us at 512^3
// (D 91 -> 89; FP64, bound by HBM, unchanged).
template <typename Real, int L, bool HIN, bool BACK>
__global__ __launch_bounds__(NT) void k_fft8_cols(CGeom g, const typename Cx<Real>::T *tw,
                                                  const typename Cx<Real>::T *__restrict__ in,
                                                  typename Cx<Real>::T *__restrict__ out)
{
  using T = typename Cx<Real>::T;
  using P = P8<L>;
  extern __shared__ char smem_raw[];
  T *lds = reinterpret_cast<T *>(smem_raw);
  const int c = threadIdx.x & (P::B - 1), tj = threadIdx.x >> P::LGB;
  // the workgroup's first column (uniform) and this thread's
  const int colg0 = xcd_wg() << P::LGB, colg = colg0 + c;
  const int of = colg0 / g.nInner, inf = colg0 - of * g.nInner;
  const int o0 = colg / g.nInner;
  const bool valid = colg < g.nCols && colg - o0 * g.nInner < g.validInner;
  // a column past the last takes the first one's place and is not stored
  const int o = valid ? o0 : of, i = valid ? colg - o0 * g.nInner : inf;
  using Off = LaneOff<Real>;
  const T *src = in + ((long)of * g.inOuter + (long)inf * g.inInner);
  T *dst = out + ((long)of * g.outOuter + (long)inf * g.outInner);
  const Off sl = (Off)((o - of) * g.inOuter + (i - inf) * g.inInner + tj * g.inPos) * (Off)sizeof(T);
  const Off dl = (Off)((o - of) * g.outOuter + (i - inf) * g.outInner + tj * g.outPos) * (Off)sizeof(T);
  const T *twl = twiddles8<T>(lds, lds_elems8<T, L>(), P::N, tw);
  T v[P::BPT][8];
#pragma unroll
  for (int u = 0; u < P::BPT; u++) {
#pragma unroll
    for (int r = 0; r < 8; r++) {
      if (HIN && r >= 4) {
        v[u][r] = mk<T>(0, 0);
      } else {
        const T x = *row_at(src, (long)(u * P::TPC + r * P::NB) * g.inPos, sl);
        v[u][r] = BACK ? cconj(x) : x;
      }
    }
  }
  // the barrier of first8 also orders the twiddle copy before its use
  first8<T, L, HIN>(lds, c, tj, v);
  rest8<T, L>(lds, c, tj, twl, v);
  if (!valid) return;
#pragma unroll
  for (int u = 0; u < P::BPT; u++) {
#pragma unroll
    for (int r = 0; r < (BACK ? 4 : 8); r++)
      *row_at(dst, (long)(u * P::TPC + r * P::NB) * g.outPos, dl) = BACK ? cconj(v[u][r]) : v[u][r];
  }
}

// pass C: forward along axis 1 (the first N/2 rows non-zero), times G,
// backward, the first N/2 rows kept; columns c = k2 * C3 + k3, Kv valid k3
template <typename Real, int L, int GM>
__global__ __launch_bounds__(NT) void k_fft8_conv(int nCols, int pos, int N2, int gfl, int C3, int Kv,
                                                  int N3fold, const typename Cx<Real>::T *tw,
                                                  const void *Gv,
                                                  typename Cx<Real>::T *__restrict__ data)
{
  constexpr bool CG = GM > 0;
  using T = typename Cx<Real>::T;
  using P = P8<L>;
  constexpr int N = P::N;
  extern __shared__ char smem_raw[];
  T *lds = reinterpret_cast<T *>(smem_raw);
  const int c = threadIdx.x & (P::B - 1), tj = threadIdx.x >> P::LGB;
  const int colg0 = xcd_wg() << P::LGB, colg = colg0 + c;
  const bool valid = colg < nCols && colg % C3 < Kv;
  // a column past the last takes the first one's place and is not stored
  using Off = LaneOff<Real>;
  T *col = data + colg0;  // uniform; plus the thread's column and first row
  const Off cl = ((Off)(valid ? c : 0) + (Off)tj * (Off)pos) * (Off)sizeof(T);
  const T *twl = twiddles8<T>(lds, lds_elems8<T, L>(), N, tw);
  // the G values of the thread's rows, fetched up front
  const GIndex gi = g_index<GM>(N, N2, Kv, N3fold, gfl, valid, colg, C3);
  using GT = typename std::conditional<CG, T, Real>::type;
  GT gv[P::BPT][8];
  T v[P::BPT][8];
#pragma unroll
  for (int u = 0; u < P::BPT; u++) {
    const int j = tj + u * P::TPC;
#pragma unroll
    for (int r = 0; r < 8; r++) {
      const int n = j + r * P::NB;
      gv[u][r] = reinterpret_cast<const GT *>(Gv)[(long)g_a1<GM>(n, N, gfl) * 8 + gi.base];
      if constexpr (GM == 2)
        if (gfl & 8) gv[u][r] = cconj(gv[u][r]);
      // rows below N / 2 hold data
      v[u][r] = r < 4 ? *row_at(col, (long)(u * P::TPC + r * P::NB) * pos, cl) : mk<T>(0, 0);
    }
  }
  first8<T, L, true>(lds, c, tj, v);
  rest8<T, L>(lds, c, tj, twl, v);
  // times G, conjugated for the backward transform (rows j + r NB)
#pragma unroll
  for (int u = 0; u < P::BPT; u++)
#pragma unroll
    for (int r = 0; r < 8; r++) {
      if constexpr (CG) v[u][r] = cconj(cmul(v[u][r], gv[u][r]));
      else v[u][r] = mk<T>(gv[u][r] * v[u][r].x, -gv[u][r] * v[u][r].y);
    }
  __syncthreads();  // every thread has read the last forward stage
  first8<T, L, false>(lds, c, tj, v);
  rest8<T, L>(lds, c, tj, twl, v);
  if (!valid) return;
#pragma unroll
  for (int u = 0; u < P::BPT; u++) {
#pragma unroll
    for (int r = 0; r < 4; r++) *row_at(col, (long)(u * P::TPC + r * P::NB) * pos, cl) = cconj(v[u][r]);
  }
}

// set-up: even extension of a compact line (length N/2+1) to length N,
// forward DFT, folded back to the compact line, in place (FP64).  PAIR: real
// lines 2c and 2c + 1 share one complex transform z = a + i b; the transform
// of a real even line is real, so A = Re Z and B = Im Z.
template <bool PAIR>
__global__ __launch_bounds__(max_threads<double>()) void k_fft_even(int nCols, int nInner, int outer, int inner,
                                                                    int pos, PlanDev pl, const double2 *tw,
                                                                    void *__restrict__ data, int lgB)
{
  using E = typename std::conditional<PAIR, double, double2>::type;
  constexpr int MV = hold<double, false>();
  extern __shared__ char smem_raw[];
  double2 *lds = reinterpret_cast<double2 *>(smem_raw);
  const int N = pl.N, h = N / 2;
  const Place p = place_cols(lgB);
  const int cg = (xcd_wg() << lgB) + p.c;
  const int ca = PAIR ? 2 * cg : cg, cb = ca + 1;
  const bool va = ca < nCols, vb = PAIR && cb < nCols;
  auto line_of = [&](int c) {
    const int o = c / nInner, i = c - o * nInner;
    return static_cast<E *>(data) + ((long)o * outer + (long)i * inner);
  };
  E *la = line_of(va ? ca : 0), *lb = line_of(vb ? cb : 0);
  const double2 *twl = twiddles_in(lds, column_rows(pl) << lgB, N, tw);
  stage_first<double2, MV, false, false>(lds, p, N, pl.radix[0], [&](int j, int rnb) {
    const int n = j + rnb;
    const long k = (long)((n <= h) ? n : N - n) * pos;
    // without a second line: zero, not line 0, which its own workgroup is
    // rewriting (a changing b is not even, and would show in Re Z)
    if constexpr (PAIR) {
      const double b = lb[k];
      return mk<double2>(la[k], vb ? b : 0.0);
    }
    else return la[k];
  });
  stages_inner<double2, MV>(lds, p, pl, false, twl);
  stage_last<double2, MV, true>(lds, p, N, pl.radix[pl.nst - 1], pl.nst == 2, twl,
                            [&](int j, bool, int rnb, double2 v) { (lds + p.at(j))[rnb << p.sh] = v; });
  __syncthreads();
  if (!va) return;
  for (int n = p.tj; n <= h; n += p.tpc) {
    double2 v = lds[p.at(n)];
    if (n != 0 && n != h) {
      const double2 w = lds[p.at(N - n)];
      v = mk<double2>(0.5 * (v.x + w.x), 0.5 * (v.y + w.y));
    }
    if constexpr (PAIR) {
      la[(long)n * pos] = v.x;
      if (vb) lb[(long)n * pos] = v.y;
    } else {
      la[(long)n * pos] = v;
    }
  }
}

// ------------------------------------------------------------ host side
static PlanDev to_dev(const FFTPlan1D &p)
{
  if (p.nst < 2 || p.nst > 4) throw Error{NPME_ERR_GRID, "FFT length without a plan"};
  PlanDev d{};
  d.N = p.N;
  d.nst = p.nst;
  for (int i = 0; i < p.nst; i++) d.radix[i] = p.radix[i];
  for (int rev = 0; rev < 2; rev++) {
    int Ns = 1;
    for (int s = 0; s < p.nst; s++) {
      const int R = p.radix[rev ? p.nst - 1 - s : s];
      (rev ? d.strB : d.strF)[s] = p.N / (Ns * R);
      (rev ? d.magB : d.magF)[s] = ((1u << 22) + Ns - 1) / Ns;
      Ns *= R;
    }
  }
  return d;
}

// threads a column needs: every stage's N / R butterflies in bpt_of(R)
// rounds
static int threads_per_column(const FFTPlan1D &p, int MV)
{
  int t = 1;
  for (int i = 0; i < p.nst; i++) {
    const int nb = p.N / p.radix[i], b = bpt_of(p.radix[i], MV);
    t = std::max(t, (nb + b - 1) / b);
  }
  return t;
}

struct FftLaunch {
  int lgB, C, tpc, T;  // columns a workgroup (2^lgB strided, C rows), threads a column, threads
  size_t lds;
};

// LDS of a workgroup: half a CU's 160 KB, so that two share a CU (long
// columns: all of it)
constexpr size_t kFftLds = 80 * 1024, kFftLdsMax = 160 * 1024;
// a launch should have this many workgroups (four for each of 256 CUs)
// before workgroups are made wider.  Sum of the passes, us, by lines of 512 /
// 1,024 / 2,048 / 8,192: 1/r 96^3 39.2 / 40.5 / 40.4 / 40.4, 280^3 120.6 / 120.2 /
// 124.8 / 129.1; FP64 96^3 42.6 / 45.7 / 45.7 / 45.6, 360^3 410 / 410 / 408 / 434
// (small grids would take 512, large ones lose from 2,048 on)
constexpr long kFftWide = 1024;

// strided columns: 16 adjacent columns for short lengths where there are
// enough of them, else 8 (64 bytes of FP32 complex values a row, half a cache
// line; 8 and 4 in FP64), fewer only where LDS or the threads of a workgroup
// do not allow them
static FftLaunch launch_cols(const FFTPlan1D &p, bool fp64, long nCols)
{
  const int es = fp64 ? 16 : 8, maxT = fp64 ? 512 : 1024;
  const int MV = fp64 ? hold<double, false>() : hold<float, false>();
  const int tmin = threads_per_column(p, MV), rows = column_rows(to_dev(p));
  const int lgMin = fp64 ? 2 : 3;
  for (int lgB = lgMin + (p.N <= 256 && nCols >= (kFftWide << (lgMin + 1)) ? 1 : 0); lgB >= 0; lgB--) {
    FftLaunch c{};
    c.lgB = lgB;
    const int B = 1 << lgB;
    c.T = (B * tmin + 63) / 64 * 64;
    c.tpc = c.T / B;
    c.lds = ((size_t)rows * B + p.N) * es;
    if (c.T <= maxT && c.lds <= (lgB > 0 ? kFftLds : kFftLdsMax)) return c;
  }
  throw Error{NPME_ERR_UNSUPPORTED, "FFT length " + std::to_string(p.N) + " does not fit a workgroup"};
}

// contiguous rows: about 256 threads a workgroup, fewer where the rows would
// not give enough workgroups
static FftLaunch launch_rows(const FFTPlan1D &p, bool fp64, long nRows)
{
  const int es = fp64 ? 16 : 8, rows = column_rows(to_dev(p));
  FftLaunch c{};
  c.tpc = threads_per_column(p, fp64 ? hold<double, true>() : hold<float, true>());
  c.C = (int)std::max(1L, std::min(256L / c.tpc, nRows / kFftWide));
  while (c.C > 1 && ((size_t)rows * c.C + p.N) * es > kFftLds / 2) c.C--;
  c.T = (c.C * c.tpc + 63) / 64 * 64;
  c.lds = ((size_t)rows * c.C + p.N) * es;
  if (c.T > (fp64 ? 512 : 1024) || c.lds > kFftLdsMax)
    throw Error{NPME_ERR_UNSUPPORTED, "FFT length " + std::to_string(p.N) + " does not fit a workgroup"};
  return c;
}

// LDS of a radix-8 pass (N = 64 or 512): the columns, plus the twiddle
// table in FP32
static size_t pass_lds8(int N, bool fp64)
{
  return (size_t)(4096) * (fp64 ? 16 : 8) + (fp64 ? 0 : (size_t)N * 8);
}

// L when N = 8^L with L in {2, 3}, else 0
static int pow8_level(const FFTPlan1D &p) { return p.N == 64 ? 2 : p.N == 512 ? 3 : 0; }

static void check_int(long v, const char *what)
{
  if (v < 0 || v > 0x7fffffffL) throw Error{NPME_ERR_UNSUPPORTED, std::string(what) + " exceeds 2^31 elements"};
}

void fft_pass_complex(bool fp64, const PassGeom &g, const FFTPlan1D &plan, const void *tw,
                      const void *in, void *out, bool backward, hipStream_t s, bool pow8)
{
  const bool rows = (g.inPos == 1 && g.outPos == 1);
  CGeom c;
  c.N = g.N;
  c.Lin = g.Lin;
  c.Lout = g.Lout;
  c.nCols = (int)g.nCols;
  c.nInner = (int)g.nInner;
  c.validInner = g.validInner < 0 ? (int)g.nInner : (int)g.validInner;
  c.inOuter = (int)g.inOuter;
  c.inInner = (int)g.inInner;
  c.inPos = (int)g.inPos;
  c.outOuter = (int)g.outOuter;
  c.outInner = (int)g.outInner;
  c.outPos = (int)g.outPos;
  check_int(g.nCols * std::max<long>(1, g.N), "FFT pass");
  const int L8 = pow8 ? pow8_level(plan) : 0;
  const int mode = backward ? PASS_BACK : 2 * g.Lin == g.N && g.Lout == g.N ? PASS_FWD : PASS_WHOLE;
  if (backward && (g.Lin != g.N || 2 * g.Lout != g.N))
    throw Error{NPME_ERR_ARG, "backward pass: all of a column in, half of it out"};
  // whole transforms are the kernel grid's, in FP64
  if (mode == PASS_WHOLE && !fp64) throw Error{NPME_ERR_ARG, "whole forward transforms run in FP64"};
  const bool half8 = 2 * g.Lin == g.N, full8 = g.Lin == g.N;
  if (!rows && L8 > 0 && (backward ? full8 && 2 * g.Lout == g.N : (half8 || full8) && g.Lout == g.N)) {
    // N = 8^L: the compile-time kernel (4096 / N columns per workgroup)
    const dim3 grid((unsigned)((g.nCols + (4096 / g.N) - 1) / (4096 / g.N)));
    const size_t sh8 = pass_lds8(g.N, fp64);
#define NPME_F8(R, LV, H, BK)                                                                  \
  hipLaunchKernelGGL((k_fft8_cols<R, LV, H, BK>), grid, dim3(NT), sh8, s, c,                   \
                     (const typename Cx<R>::T *)tw, (const typename Cx<R>::T *)in,            \
                     (typename Cx<R>::T *)out)
#define NPME_F8L(R, LV)                                                                        \
  do {                                                                                         \
    if (backward) NPME_F8(R, LV, false, true);                                                 \
    else if (half8) NPME_F8(R, LV, true, false);                                               \
    else if constexpr (sizeof(R) == 8) NPME_F8(R, LV, false, false);                           \
  } while (0)
    if (fp64) {
      if (L8 == 2) NPME_F8L(double, 2);
      else NPME_F8L(double, 3);
    } else {
      if (L8 == 2) NPME_F8L(float, 2);
      else NPME_F8L(float, 3);
    }
#undef NPME_F8
#undef NPME_F8L
    NPME_HIP_CHECK(hipGetLastError());
    return;
  }
  const PlanDev pd = to_dev(plan);
#define NPME_FFTC(R, H)                                                                        \
  do {                                                                                         \
    if (rows)                                                                                  \
      hipLaunchKernelGGL((k_fft_rows<R, H>), grid, dim3(l.T), l.lds, s, c, pd,                 \
                         (const typename Cx<R>::T *)tw, (const typename Cx<R>::T *)in,        \
                         (typename Cx<R>::T *)out, l.C, l.tpc);                                 \
    else                                                                                       \
      hipLaunchKernelGGL((k_fft_cols<R, H>), grid, dim3(l.T), l.lds, s, c, pd,                 \
                         (const typename Cx<R>::T *)tw, (const typename Cx<R>::T *)in,        \
                         (typename Cx<R>::T *)out, l.lgB);                                      \
  } while (0)
  const FftLaunch l = rows ? launch_rows(plan, fp64, g.nCols) : launch_cols(plan, fp64, g.nCols);
  const int per = rows ? l.C : 1 << l.lgB;
  const dim3 grid((unsigned)((g.nCols + per - 1) / per));
#define NPME_FFTM(R)                                                                           \
  do {                                                                                         \
    if (mode == PASS_FWD) NPME_FFTC(R, PASS_FWD);                                              \
    else if (mode == PASS_BACK) NPME_FFTC(R, PASS_BACK);                                       \
    else if constexpr (sizeof(R) == 8) NPME_FFTC(R, PASS_WHOLE);                               \
  } while (0)
  if (fp64) NPME_FFTM(double);
  else NPME_FFTM(float);
#undef NPME_FFTM
#undef NPME_FFTC
  NPME_HIP_CHECK(hipGetLastError());
}

void fft_pass_r2c_rows(bool fp64, int N, int Lin, long nRows, long inRowStride,
                       long outRowStride, const FFTPlan1D &plan, const void *tw, const void *in,
                       void *out, hipStream_t s)
{
  check_int(nRows * std::max(inRowStride, outRowStride), "FFT pass");
  if (2 * Lin != N || plan.N != N) throw Error{NPME_ERR_ARG, "R2C pass: rows of N/2 values"};
  const int nPairs = (int)(nRows / 2);
  const FftLaunch l = launch_rows(plan, fp64, nPairs);
  const dim3 grid((unsigned)((nPairs + l.C - 1) / l.C));
#define NPME_R2C(R)                                                                            \
  hipLaunchKernelGGL((k_fft_r2c<R>), grid, dim3(l.T), l.lds, s, nPairs, (int)inRowStride,      \
                     (int)outRowStride, to_dev(plan), (const typename Cx<R>::T *)tw,           \
                     (const R *)in, (typename Cx<R>::T *)out, l.C, l.tpc)
  if (fp64) NPME_R2C(double);
  else NPME_R2C(float);
#undef NPME_R2C
  NPME_HIP_CHECK(hipGetLastError());
}

void fft_pass_c2r_rows(bool fp64, int N, int Lout, long nRows, long inRowStride,
                       long outRowStride, const FFTPlan1D &plan, const void *tw, const void *in,
                       void *out, hipStream_t s)
{
  check_int(nRows * std::max(inRowStride, outRowStride), "FFT pass");
  if (plan.N != N || 2 * Lout != N) throw Error{NPME_ERR_ARG, "C2R pass: rows of N/2 values"};
  const int nPairs = (int)(nRows / 2);
  const FftLaunch l = launch_rows(plan, fp64, nPairs);
  const dim3 grid((unsigned)((nPairs + l.C - 1) / l.C));
#define NPME_C2R(R)                                                                            \
  hipLaunchKernelGGL((k_fft_c2r<R>), grid, dim3(l.T), l.lds, s, nPairs, (int)inRowStride, \
                     (int)outRowStride, to_dev(plan), (const typename Cx<R>::T *)tw,           \
                     (const typename Cx<R>::T *)in, (R *)out, l.C, l.tpc)
  if (fp64) NPME_C2R(double);
  else NPME_C2R(float);
#undef NPME_C2R
  NPME_HIP_CHECK(hipGetLastError());
}

void fft_pass_convolve(bool fp64, bool complexG, int N, int Lin, long nCols, long pos_stride,
                       int N2, int G2, long C3, long Kv, const FFTPlan1D &plan, const void *tw,
                       const void *G, void *data, hipStream_t s, bool pow8, bool fullG, int gflags)
{
  // C3: entries per axis-2 row in the data (padded), Kv of them valid.
  // complexG: complex charges and kernel, the axis-3 index runs over
  // N3 = Kv (folded to |k3| for a radial kernel's G); else the R2C data of
  // real charges, k3 in [0, Kv).  fullG: G is complex over the full grid
  // (GM 2), for either data; the k3 reversal (gflags bit 4) needs complex
  // data.
  (void)G2;
  check_int(nCols * (long)Lin, "FFT pass");
  const int gm = fullG ? 2 : complexG ? 1 : 0;
  if (fullG && !complexG && (gflags & 4))
    throw Error{NPME_ERR_UNSUPPORTED, "axis-3 reversal of G needs complex data"};
  if (2 * Lin != N || plan.N != N) throw Error{NPME_ERR_ARG, "convolution pass: columns of N/2 values"};
  // the axis-3 length of complex data (0 for the R2C data of real kernels)
  const int N3fold = complexG ? (int)Kv : 0;
  const int L8 = pow8 ? pow8_level(plan) : 0;
  if (L8 > 0) {
    const dim3 grid((unsigned)((nCols + (4096 / N) - 1) / (4096 / N)));
    const size_t sh8 = pass_lds8(N, fp64);
#define NPME_C8(R, LV, GMV)                                                                    \
  hipLaunchKernelGGL((k_fft8_conv<R, LV, GMV>), grid, dim3(NT), sh8, s, (int)nCols,           \
                     (int)pos_stride, N2, gflags, (int)C3, (int)Kv, N3fold,                     \
                     (const typename Cx<R>::T *)tw, G, (typename Cx<R>::T *)data)
#define NPME_C8L(R, GMV)                                                                       \
  do {                                                                                         \
    if (L8 == 2) NPME_C8(R, 2, GMV);                                                           \
    else NPME_C8(R, 3, GMV);                                                                   \
  } while (0)
#define NPME_C8G(R)                                                                            \
  do {                                                                                         \
    if (gm == 2) NPME_C8L(R, 2);                                                               \
    else if (gm == 1) NPME_C8L(R, 1);                                                          \
    else NPME_C8L(R, 0);                                                                       \
  } while (0)
    if (fp64) NPME_C8G(double);
    else NPME_C8G(float);
#undef NPME_C8
#undef NPME_C8L
#undef NPME_C8G
    NPME_HIP_CHECK(hipGetLastError());
    return;
  }
  const FftLaunch l = launch_cols(plan, fp64, nCols);
  const dim3 grid((unsigned)((nCols + (1 << l.lgB) - 1) >> l.lgB));
#define NPME_CONV(R, GMV)                                                                      \
  hipLaunchKernelGGL((k_fft_conv<R, GMV>), grid, dim3(l.T), l.lds, s, (int)nCols,              \
                     (int)pos_stride, N2, gflags, (int)C3, (int)Kv, N3fold, to_dev(plan),       \
                     (const typename Cx<R>::T *)tw, G, (typename Cx<R>::T *)data, l.lgB)
#define NPME_CONVG(R)                                                                          \
  do {                                                                                         \
    if (gm == 2) NPME_CONV(R, 2);                                                              \
    else if (gm == 1) NPME_CONV(R, 1);                                                         \
    else NPME_CONV(R, 0);                                                                      \
  } while (0)
  if (fp64) NPME_CONVG(double);
  else NPME_CONVG(float);
#undef NPME_CONVG
#undef NPME_CONV
  NPME_HIP_CHECK(hipGetLastError());
}

template <bool PAIR>
static void pass_even(int N, long nCols, long nInner, long outer, long inner, long pos,
                      const FFTPlan1D &plan, const void *tw, void *data, hipStream_t s)
{
  check_int(nCols * (long)(N / 2 + 1), "FFT pass");
  const long cols = PAIR ? (nCols + 1) / 2 : nCols;
  const FftLaunch l = launch_cols(plan, true, cols);
  const dim3 grid((unsigned)((cols + (1 << l.lgB) - 1) >> l.lgB));
  hipLaunchKernelGGL(k_fft_even<PAIR>, grid, dim3(l.T), l.lds, s, (int)nCols, (int)nInner, (int)outer,
                     (int)inner, (int)pos, to_dev(plan), (const double2 *)tw, data, l.lgB);
  NPME_HIP_CHECK(hipGetLastError());
}

void fft_pass_even_real(int N, long nCols, long nInner, long outer, long inner, long pos,
                        const FFTPlan1D &plan, const void *tw, double *data, hipStream_t s)
{
  pass_even<true>(N, nCols, nInner, outer, inner, pos, plan, tw, data, s);
}

void fft_pass_even(int N, long nCols, long nInner, long outer, long inner, long pos,
                   const FFTPlan1D &plan, const void *tw, void *data, hipStream_t s)
{
  pass_even<false>(N, nCols, nInner, outer, inner, pos, plan, tw, data, s);
}

}  // namespace npme
