// The field-level FFT reconstructions on half spectra, in few passes over memory
// (pyrecon/iterative_fft.py:30-82, pyrecon/plane_parallel_fft.py:41-55,
// pyrecon/iterative_fft_particle.py:104-118).
//
// The reference transforms real meshes with numpy's c2c FFT, multiplies the spectrum by a function
// of k, transforms back and keeps the real part; with a local line of sight one iteration does that
// six times.  Here:
//   * A real mesh has a Hermitian spectrum: only kz <= n2 / 2 is kept, in rows of `pitch` elements
//     (whole 128-byte lines).  Two real rows go through one complex transform along z.
//   * Taking the real part of c2c's result keeps the Hermitian part of the product, that is
//     (F(k) d(k) + conj(F(-k) d(-k))) / 2 with -k in the FFT's own numbering, where the Nyquist
//     wavenumber of an even axis is its own negative.  The factors below are that half-sum: an odd
//     power of a Nyquist component appears only together with another one.
//   * k_a k_b / k^2 splits into 1 / k^2 and a product of powers of kx, ky and kz.  The x pass
//     transforms forward, divides by k^2 and goes back with kx^0, kx^1, kx^2 without leaving the
//     workgroup (1 mesh read, 3 written).  x and y are constant along z: the y pass transforms the
//     six products, times x_a x_b, and adds those of one power of z, three fields written where the
//     three read were; the z pass transforms those and adds them times 1, z, z^2 in registers.
// Bound: HBM, with the LDS exchanges and the FP64 butterflies close behind.  One iteration with a
// local line of sight moves 19 meshes (z and y forward 2 + 2, x pass 1 + 3, y 3 + 3, z 3 + 2); six
// fields between y and z (in slabs, for their size) made it 25, one c2c transform per term with separate
// operators 120.  At 384^3 in FP64 the three iterations and the displacements take 10.8 ms, 12.9 with six
// fields, 63.3 that way; 512^3 23.6 and 27.9.  Passes at 384^3: z and y forward 0.16 and 0.18 ms (5.5 and
// 5.1 TB/s), x 0.67 ms (2.7 TB/s, four transforms), y 1.34 ms (six transforms: 0.22 ms each, the FP64
// arithmetic and LDS of one with two workgroups a CU), z with the sums 0.67 ms (3.4 TB/s; 1.5 for six).
#include <cmath>

#include "prh_fft.hpp"

namespace prh {

// Radix sequence with the fewest passes: twos in eights, a two moved to a five (radix 10) or a
// three (radix 6) where that saves a pass.
bool line_plan(size_t n, LinePlan& P) {
  if (n < 2 || n > static_cast<size_t>(kLineMax)) return false;
  int c2 = 0, c3 = 0, c5 = 0, c7 = 0;
  size_t m = n;
  for (; m % 2 == 0; m /= 2) c2++;
  for (; m % 3 == 0; m /= 3) c3++;
  for (; m % 5 == 0; m /= 5) c5++;
  for (; m % 7 == 0; m /= 7) c7++;
  if (m != 1) return false;
  int rads[kLinePasses + 2], nr = 0;
  int lone = c2 % 3;  // twos that do not fill an eight
  int tens = 0, sixes = 0;
  if (lone && lone <= c5) tens = lone;
  else if (lone && lone <= c3) sixes = lone;
  lone -= tens + sixes;
  for (int i = 0; i < c2 / 3; i++) rads[nr++] = 8;
  if (lone == 2) rads[nr++] = 4;
  if (lone == 1) rads[nr++] = 2;
  for (int i = 0; i < c5; i++) rads[nr++] = i < tens ? 10 : 5;
  for (int i = 0; i < c3; i++) rads[nr++] = i < sixes ? 6 : 3;
  for (int i = 0; i < c7; i++) rads[nr++] = 7;
  if (nr > kLinePasses) return false;
  P.n = static_cast<int>(n);
  P.npass = nr;
  P.ntw = 0;
  auto magic = [](int d) { return d > 1 ? static_cast<unsigned>((1ULL << 32) / d + 1) : 0u; };
  int ns = 1;
  for (int i = 0; i < nr; i++) {
    LinePass& S = P.pass[i];
    S.rad = rads[i];
    S.ns = ns;
    S.m = P.n / S.rad;
    S.tw = P.ntw;
    if (ns > 1) P.ntw += (S.rad - 1) * ns;
    S.div_ns = magic(ns);
    S.div_m = magic(S.m);
    ns *= S.rad;
  }
  return true;
}

namespace {

constexpr int kPowers = 3;  // a local line of sight: fields of z^0, z^1 and z^2

// Shape, wavenumbers and line of sight of a call.
struct SpecShape {
  int n[3];
  int nzc, pitch;   // kept elements of a z row, and its length in memory
  double val[3];    // k_i = 2 pi (f val_i), numpy's fftfreq
  double los[3];
  double beta, norm;
};

__device__ __forceinline__ double wave(int i, int n, double val) {
  const int f = i < (n - 1) / 2 + 1 ? i : i - n;
  constexpr double twopi = 2 * 3.141592653589793;
  return twopi * (static_cast<double>(f) * val);
}
__device__ __forceinline__ bool nyquist(int i, int n) { return 2 * i == n; }

template <typename R>
__device__ __forceinline__ Cx<R> scaled(Cx<R> v, double s) {
  return {static_cast<R>(static_cast<double>(v.re) * s), static_cast<R>(static_cast<double>(v.im) * s)};
}

// The thread index, as a value the compiler cannot carry over from one round of a loop to the next:
// what is worked out from it (wavenumbers, coordinates of every element held) is worked out again
// instead of being kept in registers.
__device__ __forceinline__ int hidden(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

template <typename R>
__device__ __forceinline__ Cx<R>* stage_twiddles(Cx<R>* at, const Cx<R>* __restrict__ tw, int n) {
  for (int k = threadIdx.x; k < n; k += blockDim.x) at[k] = tw[k];
  return at;
}

// ---- z ---------------------------------------------------------------------

// Real rows -> half spectra, `nl` pairs of rows a block.  Z = a + i b is
// transformed and split: A[k] = (Z[k] + conj Z[n-k]) / 2, B[k] = (Z[k] - conj Z[n-k]) / 2i.
template <typename R>
__global__ __launch_bounds__(1024) void k_rows_forward(const R* __restrict__ mesh, Cx<R>* __restrict__ spec,
                                                      LinePlan P, const Cx<R>* __restrict__ tw, int nl,
                                                      unsigned div_nzc, int nzc, int pitch, int nrows) {
  extern __shared__ double smem[];
  Cx<R>* buf = reinterpret_cast<Cx<R>*>(smem);
  const int n = P.n;
  const int held = (nl * n + 15) & ~15;
  LineFft<R, false> L{buf, stage_twiddles(buf + held, tw, P.ntw), n, nl, 0, static_cast<int>(blockDim.x), static_cast<int>(threadIdx.x)};
  const int pair0 = blockIdx.x * nl;
  L.template run<false, false, true>(
      P,
      [&](int line, int e) {
        const int row = 2 * (pair0 + line);
        const R* a = mesh + static_cast<size_t>(row) * n + e;
        return Cx<R>{row < nrows ? a[0] : R(0), row + 1 < nrows ? a[n] : R(0)};
      },
      [](int, int, Cx<R>) {});
  const int total = nl * nzc;
  for (int t = threadIdx.x; t < total; t += blockDim.x) {
    const int line = quotient(t, div_nzc), k = t - line * nzc;
    const int row = 2 * (pair0 + line);
    if (row >= nrows) break;
    const Cx<R> z = buf[L.slot(line, k)], c = buf[L.slot(line, k == 0 ? 0 : n - k)];
    Cx<R>* out = spec + static_cast<size_t>(row) * pitch + k;
    out[0] = {R(0.5) * (z.re + c.re), R(0.5) * (z.im - c.im)};
    if (row + 1 < nrows) out[pitch] = {R(0.5) * (z.im + c.im), R(0.5) * (c.re - z.re)};
  }
}

struct RealGeom {
  double o[3], c[3];  // mesh coordinates o + c j
};

enum RowsOut { kRowsStore = 0, kRowsMinus = 1, kRowsMinusLocal = 2 };

// Half spectra -> real rows (the real part of the c2c result: the imaginary parts of the elements
// that are their own conjugates are dropped).
//   kRowsStore: field blockIdx.y of `fields` to out[blockIdx.y].
//   kRowsMinus: out = base - factor t.
//   kRowsMinusLocal: out = base - factor (t_0 + z t_1 + z^2 t_2) / |x|^2, the three fields one after
//     another through the same registers.
template <typename R>
struct RowsArgs {
  const Cx<R>* field[kPowers];
  R* out[3];
  const R* base;
  int nrows;
  double factor;
  RealGeom G;
};

template <typename R, int MODE>
__global__ __launch_bounds__(1024) void k_rows_inverse(RowsArgs<R> A, LinePlan P, const Cx<R>* __restrict__ tw,
                                                      int nl, unsigned div_nzc, unsigned div_n, SpecShape S) {
  extern __shared__ double smem[];
  Cx<R>* buf = reinterpret_cast<Cx<R>*>(smem);
  const int n = P.n;
  const int held = (nl * n + 15) & ~15;
  LineFft<R, false> L{buf, stage_twiddles(buf + held, tw, P.ntw), n, nl, 0, static_cast<int>(blockDim.x), static_cast<int>(threadIdx.x)};
  const int pair0 = blockIdx.x * nl;
  constexpr int NF = MODE == kRowsMinusLocal ? kPowers : 1;
  constexpr int kSum = MODE == kRowsMinusLocal ? LineTile<R>::held : 1;
  double sum_a[kSum], sum_b[kSum];
#pragma unroll
  for (int i = 0; i < kSum; i++) sum_a[i] = 0., sum_b[i] = 0.;
  const int total = nl * S.nzc;
#pragma unroll 1
  for (int f = 0; f < NF; f++) {
    const Cx<R>* __restrict__ field = A.field[MODE == kRowsStore ? blockIdx.y : f];
    L.tid = hidden(threadIdx.x);
    if (f > 0) __syncthreads();
    // the kept half of a thread's elements; fewer at a time beside the sums of the three fields
    constexpr int kBatch = MODE == kRowsMinusLocal ? LineTile<R>::held / 4 + 1 : LineTile<R>::held / 2 + 1;
    for (int t0 = L.tid; t0 < total; t0 += kBatch * L.nt) {
      Cx<R> a[kBatch], b[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; i++) {
        const int t = t0 + i * L.nt;
        const int line = quotient(t, div_nzc), k = t - line * S.nzc;
        // a row past the end reads the last one; its result is not used
        const int ra = min(2 * (pair0 + line), A.nrows - 1), rb = min(2 * (pair0 + line) + 1, A.nrows - 1);
        const Cx<R>* in = field + k;
        a[i] = in[static_cast<size_t>(ra) * S.pitch];
        b[i] = in[static_cast<size_t>(rb) * S.pitch];
      }
#pragma unroll
      for (int i = 0; i < kBatch; i++) {
        const int t = t0 + i * L.nt;
        if (t >= total) continue;
        const int line = quotient(t, div_nzc), k = t - line * S.nzc;
        if (k == 0 || 2 * k == n) {
          buf[L.slot(line, k)] = {a[i].re, b[i].re};
        } else {
          buf[L.slot(line, k)] = {a[i].re - b[i].im, a[i].im + b[i].re};
          buf[L.slot(line, n - k)] = {a[i].re + b[i].im, b[i].re - a[i].im};
        }
      }
    }
    __syncthreads();
    if constexpr (MODE == kRowsStore) {
      R* __restrict__ out = A.out[blockIdx.y];
      L.template run<true, true, false>(
          P, [](int, int) { return Cx<R>{R(0), R(0)}; },
          [&](int line, int e, Cx<R> v) {
            const int row = 2 * (pair0 + line);
            const size_t at = static_cast<size_t>(row) * n + e;
            if (row < A.nrows) out[at] = v.re;
            if (row + 1 < A.nrows) out[at + n] = v.im;
          });
    } else if constexpr (MODE == kRowsMinus) {
      L.template run<true, true, false>(
          P, [](int, int) { return Cx<R>{R(0), R(0)}; },
          [&](int line, int e, Cx<R> v) {
            const int row = 2 * (pair0 + line);
            const size_t at = static_cast<size_t>(row) * n + e;
            if (row < A.nrows)
              A.out[0][at] = static_cast<R>(static_cast<double>(A.base[at]) - A.factor * static_cast<double>(v.re));
            if (row + 1 < A.nrows)
              A.out[0][at + n] =
                  static_cast<R>(static_cast<double>(A.base[at + n]) - A.factor * static_cast<double>(v.im));
          });
    } else {
      L.template run<true, true, true>(P, [](int, int) { return Cx<R>{R(0), R(0)}; }, [](int, int, Cx<R>) {});
#pragma unroll
      for (int i = 0; i < LineTile<R>::held; i++) {
        int line, e;
        L.element(i, div_n, line, e);
        const Cx<R> v = buf[L.slot(line, e)];
        const double z = A.G.o[2] + A.G.c[2] * static_cast<double>(e);
        const double w = f == 0 ? 1. : f == 1 ? z : z * z;
        sum_a[i] += w * static_cast<double>(v.re);
        sum_b[i] += w * static_cast<double>(v.im);
      }
    }
  }
  if constexpr (MODE == kRowsMinusLocal) {
#pragma unroll
    for (int i = 0; i < LineTile<R>::held; i++) {
      int line, e;
      if (!L.element(i, div_n, line, e)) continue;
      const int row = 2 * (pair0 + line);
      if (row >= A.nrows) continue;
      const unsigned ra = row, rb = ra + 1;
      const unsigned ia = ra / S.n[1], ib = rb / S.n[1];
      const double xa = A.G.o[0] + A.G.c[0] * static_cast<double>(ia);
      const double ya = A.G.o[1] + A.G.c[1] * static_cast<double>(ra - ia * S.n[1]);
      const double xb = A.G.o[0] + A.G.c[0] * static_cast<double>(ib);
      const double yb = A.G.o[1] + A.G.c[1] * static_cast<double>(rb - ib * S.n[1]);
      const double z = A.G.o[2] + A.G.c[2] * static_cast<double>(e);
      const size_t at = static_cast<size_t>(row) * n + e;
      A.out[0][at] = static_cast<R>(static_cast<double>(A.base[at]) -
                                    A.factor * (sum_a[i] / (xa * xa + ya * ya + z * z)));
      if (row + 1 < A.nrows)
        A.out[0][at + n] = static_cast<R>(static_cast<double>(A.base[at + n]) -
                                          A.factor * (sum_b[i] / (xb * xb + yb * yb + z * z)));
    }
  }
}

// ---- y ---------------------------------------------------------------------

// In place along y: planes blockIdx.z of the spectrum (or of spec[blockIdx.y] each).
template <typename R, bool INV>
__global__ __launch_bounds__(1024) void k_columns(Cx<R>* s0, Cx<R>* s1, Cx<R>* s2, LinePlan P,
                                                 const Cx<R>* __restrict__ tw, int lw, int pitch) {
  extern __shared__ double smem[];
  Cx<R>* buf = reinterpret_cast<Cx<R>*>(smem);
  const int n = P.n;
  const int W = 1 << lw;
  LineFft<R, true> L{buf, stage_twiddles(buf + (n + 1) * W, tw, P.ntw), n, W, lw, static_cast<int>(blockDim.x), static_cast<int>(threadIdx.x)};
  Cx<R>* spec = blockIdx.y == 0 ? s0 : blockIdx.y == 1 ? s1 : s2;
  Cx<R>* base = spec + static_cast<size_t>(blockIdx.z) * n * pitch + blockIdx.x * W;
  L.template run<INV, false, false>(
      P,
      [&](int line, int e) { return base[static_cast<size_t>(e) * pitch + line]; },
      [&](int line, int e, Cx<R> v) { base[static_cast<size_t>(e) * pitch + line] = v; });
}

// A local line of sight: the sum over the pairs of axes of x_a x_b t_ab, grouped by its power of z, from
// X_p = IFFT_x(kx^p d).  With t_ab along z still to be transformed,
//   u = 0: x^2 t_xx + 2 x y t_xy + y^2 t_yy    from X2, ky X1, ky^2 X0, to where X2 was
//   u = 1: kz (2 x t_xz + 2 y t_yz)            from X1, ky X0, to where X1 was
//   u = 2: kz^2 t_zz                           from X0, in place
// Elements with a Nyquist component (the header's half-sum):
//   xy at ky Nyquist and xz at kz Nyquist keep the kx Nyquist term alone, whose transform along x is
//   (-1)^x times its value; the x pass leaves those values in edge_y[kz] and edge_z[ky].
//   yz at kz Nyquist keeps the ky Nyquist term alone.
// A block owns its lines of the three arrays: the later outputs read them again, from L2.
template <typename R>
__global__ __launch_bounds__(1024) void k_columns_local(Cx<R>* x0, Cx<R>* x1, Cx<R>* x2, const Cx<R>* __restrict__ edge_y,
                                                       const Cx<R>* __restrict__ edge_z, LinePlan P,
                                                       const Cx<R>* __restrict__ tw, int lw, SpecShape S, RealGeom G) {
  extern __shared__ double smem[];
  Cx<R>* buf = reinterpret_cast<Cx<R>*>(smem);
  const int n = P.n;
  const int W = 1 << lw;
  LineFft<R, true> L{buf, stage_twiddles(buf + (n + 1) * W, tw, P.ntw), n, W, lw, static_cast<int>(blockDim.x), static_cast<int>(threadIdx.x)};
  const int ix = blockIdx.y, kz0 = blockIdx.x * W;
  const size_t row = static_cast<size_t>(S.pitch), first = static_cast<size_t>(ix) * n * row + kz0;
  const double x = G.o[0] + G.c[0] * static_cast<double>(ix);
  const double sign = ix & 1 ? -1. : 1.;
  const double knx = S.n[0] % 2 ? 0. : sign * wave(S.n[0] / 2, S.n[0], S.val[0]);
  constexpr int kBatch = LineTile<R>::held / 2;
  double sum_re[LineTile<R>::held], sum_im[LineTile<R>::held];
#pragma unroll 1
  for (int t = 0; t < 6; t++) {
    // output u, power o of y (and of ky), power p of x (and of kx)
    const int u = t < 3 ? 0 : t < 5 ? 1 : 2, o = t < 3 ? t : t < 5 ? t - 3 : 0, p = 2 - u - o;
    const Cx<R>* in = (p == 0 ? x0 : p == 1 ? x1 : x2) + first;
    L.tid = hidden(threadIdx.x);
    // a few elements at a time beside the sums
#pragma unroll 1
    for (int i0 = 0; i0 < LineTile<R>::held; i0 += kBatch) {
      Cx<R> d[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; i++) {
        int line, e;
        L.element(i0 + i, 0, line, e);
        d[i] = in[e * row + line];
      }
      if (i0 == 0) __syncthreads();
#pragma unroll
      for (int i = 0; i < kBatch; i++) {
        int line, e;
        if (!L.element(i0 + i, 0, line, e)) continue;
        const bool nyz = nyquist(kz0 + line, S.n[2]), nyy = nyquist(e, n);
        const double ky = wave(e, n, S.val[1]), kz = wave(kz0 + line, S.n[2], S.val[2]);
        Cx<R> v = d[i];
        double s = o == 0 ? 1. : o == 1 ? ky : ky * ky;
        if (u == 1 && o == 1 && nyz != nyy) s = 0.;
        if (u == 1 && o == 0 && nyz) {
          s = knx;
          if (knx != 0.) v = edge_z[e];
        }
        if (u == 0 && o == 1 && nyy) {
          s = kz0 + line < S.nzc ? knx * ky : 0.;
          if (s != 0.) v = edge_y[kz0 + line];
        }
        if (u > 0) s *= u == 1 ? kz : kz * kz;
        buf[L.slot(line, e)] = s == 0. ? Cx<R>{R(0), R(0)} : scaled(v, s);
      }
    }
    __syncthreads();
    L.template run<true, true, true>(P, [](int, int) { return Cx<R>{R(0), R(0)}; }, [](int, int, Cx<R>) {});
    const double xs = p == 0 ? 1. : p == 1 ? x : x * x;
    const double twice = t == 0 || t == 2 || t == 5 ? 1. : 2.;
    Cx<R>* out = (u == 0 ? x2 : u == 1 ? x1 : x0) + first;
#pragma unroll
    for (int i = 0; i < LineTile<R>::held; i++) {
      int line, e;
      const bool ok = L.element(i, 0, line, e);
      const double y = G.o[1] + G.c[1] * static_cast<double>(e);
      const double w = twice * xs * (o == 0 ? 1. : o == 1 ? y : y * y);
      const Cx<R> v = buf[L.slot(line, e)];
      const double re = w * static_cast<double>(v.re), im = w * static_cast<double>(v.im);
      sum_re[i] = o == 0 ? re : sum_re[i] + re;
      sum_im[i] = o == 0 ? im : sum_im[i] + im;
      if (ok && p == 0) out[e * row + line] = {static_cast<R>(sum_re[i]), static_cast<R>(sum_im[i])};
    }
  }
}

// ---- x ---------------------------------------------------------------------

enum XMode { kXLocal = 0, kXGlobal = 1, kXGrad = 2, kXPlane = 3 };

// Forward along x, d = spectrum / k^2 (0 at k = 0) times 1 / N, and back with
//   kXLocal:  kx^0, kx^1 (without the Nyquist term), kx^2   -> out[0..2], edge values aside
//   kXGlobal: (k . los)^2                                   -> out[0]
//   kXGrad:   i kx, i ky, i kz                              -> out[0..2]
//   kXPlane:  the same over 1 + beta (k . los)^2 / k^2      -> out[0..2]
// out[0] may be the input: a block owns its lines and has read them before it writes any.
template <typename R, int MODE>
__global__ __launch_bounds__(1024) void k_pencils(const Cx<R>* spec, Cx<R>* out0, Cx<R>* out1, Cx<R>* out2,
                                                 Cx<R>* __restrict__ edge_y, Cx<R>* __restrict__ edge_z,
                                                 LinePlan P, const Cx<R>* __restrict__ tw, int lw, SpecShape S) {
  extern __shared__ double smem[];
  Cx<R>* buf = reinterpret_cast<Cx<R>*>(smem);
  const int n = P.n;
  const int W = 1 << lw;
  LineFft<R, true> L{buf, stage_twiddles(buf + (n + 1) * W, tw, P.ntw), n, W, lw, static_cast<int>(blockDim.x), static_cast<int>(threadIdx.x)};
  const int iy = blockIdx.y, kz0 = blockIdx.x * W;
  const size_t es = static_cast<size_t>(S.n[1]) * S.pitch;
  const size_t base = static_cast<size_t>(iy) * S.pitch + kz0;
  const double ky = wave(iy, S.n[1], S.val[1]);
  const bool nyy = nyquist(iy, S.n[1]);
  L.template run<false, false, true>(
      P, [&](int line, int e) { return spec[base + e * es + line]; }, [](int, int, Cx<R>) {});
  Cx<R> d[LineTile<R>::held];
#pragma unroll
  for (int i = 0; i < LineTile<R>::held; i++) {
    int line, e;
    if (!L.element(i, 0, line, e)) continue;
    const double kx = wave(e, n, S.val[0]), kz = wave(kz0 + line, S.n[2], S.val[2]);
    const double k2 = kx * kx + ky * ky + kz * kz;
    d[i] = scaled(buf[L.slot(line, e)], (e | iy | (kz0 + line)) == 0 ? 0. : S.norm / k2);
    if (MODE == kXLocal && nyquist(e, n) && kz0 + line < S.nzc) {
      if (nyy) edge_y[kz0 + line] = d[i];
      if (nyquist(kz0 + line, S.n[2])) edge_z[iy] = d[i];
    }
  }
  constexpr int NO = MODE == kXGlobal ? 1 : 3;
#pragma unroll 1
  for (int o = 0; o < NO; o++) {
    Cx<R>* out = o == 0 ? out0 : o == 1 ? out1 : out2;
    L.tid = hidden(threadIdx.x);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < LineTile<R>::held; i++) {
      int line, e;
      if (!L.element(i, 0, line, e)) continue;
      const double kx = wave(e, n, S.val[0]);
      const bool nyx = nyquist(e, n);
      Cx<R> v;
      if constexpr (MODE == kXLocal) {
        v = o == 0 ? d[i] : scaled(d[i], o == 2 ? kx * kx : nyx ? 0. : kx);
      } else {
        const int iz = kz0 + line;
        const double kz = wave(iz, S.n[2], S.val[2]);
        const bool nyz = nyquist(iz, S.n[2]);
        // line-of-sight component of the Nyquist wavenumbers and of the others
        double ln = 0., lo = 0.;
        if constexpr (MODE != kXGrad) {
          (nyx ? ln : lo) += kx * S.los[0];
          (nyy ? ln : lo) += ky * S.los[1];
          (nyz ? ln : lo) += kz * S.los[2];
        }
        if constexpr (MODE == kXGlobal) {
          v = scaled(d[i], ln * ln + lo * lo);
        } else {
          const double ka = o == 0 ? kx : o == 1 ? ky : kz;
          const bool nya = o == 0 ? nyx : o == 1 ? nyy : nyz;
          double s = nya ? 0. : ka;
          if constexpr (MODE == kXPlane) {
            const double k2 = kx * kx + ky * ky + kz * kz;
            const double up = (ln + lo) * (ln + lo), dn = (ln - lo) * (ln - lo);
            double g = (e | iy | iz) == 0 ? 0. : 1. / (1. + S.beta * (up / k2));
            if (nyx || nyy || nyz) {
              const double h = 1. / (1. + S.beta * (dn / k2));
              g = nya ? 0.5 * (g - h) : 0.5 * (g + h);
              s = ka;
            }
            s *= g;
          }
          v = scaled(d[i], s);
          v = Cx<R>{-v.im, v.re};
        }
      }
      buf[L.slot(line, e)] = v;
    }
    __syncthreads();
    L.template run<true, true, false>(
        P, [](int, int) { return Cx<R>{R(0), R(0)}; },
        [&](int line, int e, Cx<R> v) { out[base + e * es + line] = v; });
  }
}

// ---- host ------------------------------------------------------------------

struct Layout {
  LinePlan P[3];
  int nzc = 0, pitch = 0;
  size_t elems = 0;     // one half spectrum
};

template <typename R>
bool layout(const size_t* n, Layout& L) {
  for (int d = 0; d < 3; d++)
    if (!line_plan(n[d], L.P[d])) return false;
  constexpr int W = LineTile<R>::lines;
  L.nzc = static_cast<int>(n[2]) / 2 + 1;
  L.pitch = (L.nzc + W - 1) / W * W;
  L.elems = n[0] * n[1] * L.pitch;
  return true;
}

size_t edge_elems(const Layout& L, const size_t* n) { return (L.nzc + n[1] + 15) / 16 * 16; }

// Complex elements of scratch: spectra, and for a local line of sight the edge values.
size_t scratch_elems(const Layout& L, const size_t* n, int spectra, bool local) {
  return spectra * L.elems + (local ? edge_elems(L, n) : 0);
}

template <typename R>
SpecShape spec_shape(const Layout& L, const size_t* n, const R* boxsize, const double* los, double beta) {
  SpecShape S;
  double cells = 1.;
  for (int d = 0; d < 3; d++) {
    S.n[d] = static_cast<int>(n[d]);
    // d = boxsize / nmesh in float64 and val = 1 / (n d), as numpy.fft.fftfreq
    const double cell = static_cast<double>(boxsize[d]) / static_cast<double>(S.n[d]);
    S.val[d] = 1.0 / (static_cast<double>(S.n[d]) * cell);
    S.los[d] = los ? los[d] : 0.;
    cells *= static_cast<double>(S.n[d]);
  }
  S.nzc = L.nzc;
  S.pitch = L.pitch;
  S.beta = beta;
  S.norm = 1. / cells;
  return S;
}

template <typename K>
int allow_lds(K kernel, size_t bytes) {
  if (bytes > 65536)
    PRH_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                static_cast<int>(bytes)));
  return PRH_OK;
}

unsigned magic_of(int d) { return d > 1 ? static_cast<unsigned>((1ULL << 32) / d + 1) : 0u; }

template <typename R>
struct Call {
  prh_workspace* ws;
  Layout L;
  SpecShape S;
  hipStream_t s;
  const Cx<R>* tw(int d) const { return static_cast<const Cx<R>*>(ws->smooth.pass_tw[d]); }

  // a launch that moves `meshes` half spectra (or real meshes), under the transform timer
  template <class F>
  int timed(double meshes, F&& launch) const {
    timer_before(PRH_TIMER_FFT_PASS, s);
    PRH_TRY(launch());
    PRH_LAUNCHED();
    timer_after(PRH_TIMER_FFT_PASS, s,
                meshes * static_cast<double>(S.n[0]) * S.n[1] * S.n[2] * sizeof(R));
    return PRH_OK;
  }

  // mesh -> half spectrum, transformed along z and y
  int forward_zy(const R* mesh, Cx<R>* spec) const {
    PRH_TRY(timed(2, [&]() {
      const LineRows B = line_rows<R>(L.P[2]);
      const int nrows = S.n[0] * S.n[1];
      auto* k = &k_rows_forward<R>;
      PRH_TRY(allow_lds(k, B.lds));
      k<<<ceil_div((nrows + 1) / 2, B.nl), B.threads, B.lds, s>>>(mesh, spec, L.P[2], tw(2), B.nl, magic_of(S.nzc),
                                                                  S.nzc, S.pitch, nrows);
      return PRH_OK;
    }));
    return columns<false>(1, spec, spec, spec);
  }

  template <bool INV>
  int columns(int count, Cx<R>* s0, Cx<R>* s1, Cx<R>* s2) const {
    return timed(2. * count, [&]() {
      const LineCols B = line_cols<R>(L.P[1]);
      const dim3 grid(S.pitch >> B.lw, count, S.n[0]);
      auto* k = &k_columns<R, INV>;
      PRH_TRY(allow_lds(k, B.lds));
      k<<<grid, B.threads, B.lds, s>>>(s0, s1, s2, L.P[1], tw(1), B.lw, S.pitch);
      return PRH_OK;
    });
  }

  template <int MODE>
  int pencils(const Cx<R>* spec, Cx<R>* o0, Cx<R>* o1, Cx<R>* o2, Cx<R>* edge_y, Cx<R>* edge_z) const {
    return timed(MODE == kXGlobal ? 2 : 4, [&]() {
      const LineCols B = line_cols<R>(L.P[0]);
      const dim3 grid(S.pitch >> B.lw, S.n[1]);
      auto* k = &k_pencils<R, MODE>;
      PRH_TRY(allow_lds(k, B.lds));
      k<<<grid, B.threads, B.lds, s>>>(spec, o0, o1, o2, edge_y, edge_z, L.P[0], tw(0), B.lw, S);
      return PRH_OK;
    });
  }

  template <int MODE>
  int rows(const RowsArgs<R>& A, int fields) const {
    const double meshes = MODE == kRowsStore ? 2. * fields : MODE == kRowsMinus ? 3. : kPowers + 2.;
    return timed(meshes, [&]() {
      const LineRows B = line_rows<R>(L.P[2]);
      auto* k = &k_rows_inverse<R, MODE>;
      PRH_TRY(allow_lds(k, B.lds));
      const dim3 grid(ceil_div((A.nrows + 1) / 2, B.nl), MODE == kRowsStore ? fields : 1);
      k<<<grid, B.threads, B.lds, s>>>(A, L.P[2], tw(2), B.nl, magic_of(S.nzc), magic_of(S.n[2]), S);
      return PRH_OK;
    });
  }
};

template <typename R>
int open_call(Call<R>& C, prh_workspace* ws, const size_t* nmesh, const R* boxsize, const double* los,
              double beta, void* stream) {
  if (!(ws->flags & PRH_WS_FFT) || !ws->smooth.have) {
    set_error("workspace was built without Fourier tables for this shape (PRH_WS_FFT)");
    return PRH_ERR_STATE;
  }
  if (ws->dtype != Tag<R>::code) {
    set_error("workspace precision does not match the mesh");
    return PRH_ERR_ARG;
  }
  for (int d = 0; d < 3; d++)
    if (ws->n[d] != nmesh[d]) {
      set_error("workspace mesh does not match nmesh");
      return PRH_ERR_CAPACITY;
    }
  if (!layout<R>(nmesh, C.L)) {
    set_error("half-spectrum transforms take axes of 2 to %d cells with factors 2, 3, 5 and 7", kLineMax);
    return PRH_ERR_ARG;
  }
  C.ws = ws;
  C.s = as_stream(stream);
  C.S = spec_shape<R>(C.L, nmesh, boxsize, los, beta);
  return PRH_OK;
}

int scratch_bytes(const size_t* nmesh, int dtype, int kind, size_t* bytes) {
  if (!nmesh || !bytes || kind < 0 || kind > 2 || (dtype != PRH_F32 && dtype != PRH_F64)) return PRH_ERR_ARG;
  Layout L;
  const bool ok = dtype == PRH_F64 ? layout<double>(nmesh, L) : layout<float>(nmesh, L);
  *bytes = 0;
  if (!ok) return PRH_OK;
  const size_t elems = scratch_elems(L, nmesh, kind == PRH_SPECTRAL_GLOBAL ? 1 : 3, kind == PRH_SPECTRAL_LOCAL);
  *bytes = elems * 2 * static_cast<size_t>(dtype);
  return PRH_OK;
}

template <typename R>
int do_iterate(prh_workspace* ws, const R* src, const R* delta, R* out, const size_t* nmesh, const R* boxsize,
               const R* boxcenter, const double* los, double factor, void* scratch, size_t nscratch,
               void* stream) {
  if (!ws || !src || !delta || !out || !nmesh || !boxsize || !boxcenter || !scratch) return PRH_ERR_ARG;
  Call<R> C;
  PRH_TRY(open_call<R>(C, ws, nmesh, boxsize, los, 0., stream));
  const Layout& L = C.L;
  const SpecShape& S = C.S;
  if (nscratch < scratch_elems(L, nmesh, los ? 1 : 3, !los) * sizeof(Cx<R>)) {
    set_error("scratch of %zu bytes is too small", nscratch);
    return PRH_ERR_CAPACITY;
  }
  Cx<R>* spec = static_cast<Cx<R>*>(scratch);
  RowsArgs<R> A = {};
  A.out[0] = out;
  A.base = delta;
  A.factor = factor;
  for (int d = 0; d < 3; d++) {
    // MeshInfo.offset in the mesh dtype (mesh.py:462-465); cellsize in float64
    A.G.o[d] = static_cast<double>(static_cast<R>(boxcenter[d] - boxsize[d] / R(2)));
    A.G.c[d] = static_cast<double>(boxsize[d]) / static_cast<double>(S.n[d]);
  }
  PRH_TRY(C.forward_zy(src, spec));
  if (los) {
    PRH_TRY((C.template pencils<kXGlobal>(spec, spec, spec, spec, nullptr, nullptr)));
    PRH_TRY((C.template columns<true>(1, spec, spec, spec)));
    A.field[0] = spec;
    A.nrows = S.n[0] * S.n[1];
    return C.template rows<kRowsMinus>(A, 1);
  }
  Cx<R>*x1 = spec + L.elems, *x2 = x1 + L.elems, *edge_y = x2 + L.elems, *edge_z = edge_y + L.nzc;
  PRH_TRY((C.template pencils<kXLocal>(spec, spec, x1, x2, edge_y, edge_z)));
  PRH_TRY(C.timed(6, [&]() {
    const LineCols B = line_cols<R>(L.P[1]);
    const dim3 grid(S.pitch >> B.lw, S.n[0]);
    auto* k = &k_columns_local<R>;
    PRH_TRY(allow_lds(k, B.lds));
    k<<<grid, B.threads, B.lds, C.s>>>(spec, x1, x2, edge_y, edge_z, L.P[1], C.tw(1), B.lw, S, A.G);
    return PRH_OK;
  }));
  A.field[0] = x2;
  A.field[1] = x1;
  A.field[2] = spec;
  A.nrows = S.n[0] * S.n[1];
  return C.template rows<kRowsMinusLocal>(A, kPowers);
}

template <typename R>
int do_displacements(prh_workspace* ws, const R* delta, R* psi0, R* psi1, R* psi2, const size_t* nmesh,
                     const R* boxsize, const double* los, double beta, void* scratch, size_t nscratch,
                     void* stream) {
  if (!ws || !delta || !psi0 || !psi1 || !psi2 || !nmesh || !boxsize || !scratch) return PRH_ERR_ARG;
  Call<R> C;
  PRH_TRY(open_call<R>(C, ws, nmesh, boxsize, los, beta, stream));
  const Layout& L = C.L;
  const SpecShape& S = C.S;
  if (nscratch < scratch_elems(L, nmesh, 3, false) * sizeof(Cx<R>)) {
    set_error("scratch of %zu bytes is too small", nscratch);
    return PRH_ERR_CAPACITY;
  }
  Cx<R>*x0 = static_cast<Cx<R>*>(scratch), *x1 = x0 + L.elems, *x2 = x1 + L.elems;
  PRH_TRY(C.forward_zy(delta, x0));
  if (los)
    PRH_TRY((C.template pencils<kXPlane>(x0, x0, x1, x2, nullptr, nullptr)));
  else
    PRH_TRY((C.template pencils<kXGrad>(x0, x0, x1, x2, nullptr, nullptr)));
  RowsArgs<R> A = {};
  A.field[0] = x0, A.field[1] = x1, A.field[2] = x2;
  A.out[0] = psi0, A.out[1] = psi1, A.out[2] = psi2;
  A.nrows = S.n[0] * S.n[1];
  PRH_TRY((C.template columns<true>(3, x0, x1, x2)));
  return C.template rows<kRowsStore>(A, 3);
}

}  // namespace
}  // namespace prh

using namespace prh;

extern "C" {

int prh_spectral_scratch(const size_t* nmesh, int dtype, int kind, size_t* bytes) {
  return scratch_bytes(nmesh, dtype, kind, bytes);
}
int prh_spectral_iterate_f32(prh_workspace* ws, const float* src, const float* delta, float* out, const size_t* nmesh,
                             const float* boxsize, const float* boxcenter, const double* los, double factor,
                             void* scratch, size_t nscratch, void* stream) {
  return do_iterate<float>(ws, src, delta, out, nmesh, boxsize, boxcenter, los, factor, scratch, nscratch, stream);
}
int prh_spectral_iterate_f64(prh_workspace* ws, const double* src, const double* delta, double* out, const size_t* nmesh,
                             const double* boxsize, const double* boxcenter, const double* los, double factor,
                             void* scratch, size_t nscratch, void* stream) {
  return do_iterate<double>(ws, src, delta, out, nmesh, boxsize, boxcenter, los, factor, scratch, nscratch, stream);
}
int prh_spectral_displacements_f32(prh_workspace* ws, const float* delta, float* psi0, float* psi1, float* psi2,
                                   const size_t* nmesh, const float* boxsize, const double* los, double beta,
                                   void* scratch, size_t nscratch, void* stream) {
  return do_displacements<float>(ws, delta, psi0, psi1, psi2, nmesh, boxsize, los, beta, scratch, nscratch, stream);
}
int prh_spectral_displacements_f64(prh_workspace* ws, const double* delta, double* psi0, double* psi1, double* psi2,
                                   const size_t* nmesh, const double* boxsize, const double* los, double beta,
                                   void* scratch, size_t nscratch, void* stream) {
  return do_displacements<double>(ws, delta, psi0, psi1, psi2, nmesh, boxsize, los, beta, scratch, nscratch, stream);
}

}  // extern "C"
