// Transforms of lines of up to kLineMax elements whose factors are 2, 3, 5 and 7, held by a
// workgroup: Stockham passes of radix 8, 10, 7, 6, 5, 4, 3, 2 with the butterflies in registers and
// one LDS exchange between passes.
//
// The first pass takes its inputs from a callback and the last one hands its results to a callback,
// both in registers, so that plain reads from and writes to global memory need no extra trip through
// LDS; either end can be left in LDS instead, for callers that work on the elements in between.
// (Every radix has its copy of the callbacks: long ones belong in a loop over LDS.)
//
// Two layouts of a tile of lines:
//   kAcross: elements of a line are far apart and neighbouring lines adjacent (x and y axes).  Lanes
//     run along the lines first; LDS is [element][line] with kTileLines lines, one 128-byte row per
//     element, which uses every bank once whatever rows a wavefront touches.
//   kAlong: the elements of a line are contiguous (z axis).  Lanes run along the elements; LDS is
//     [line][element] with the low three index bits XOR-ed by the next three.
#pragma once

#include "prh_workspace.hpp"

namespace prh {

template <typename R>
struct Cx {
  R re, im;
};

template <typename R>
__device__ __forceinline__ Cx<R> cmul(Cx<R> a, Cx<R> b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}

constexpr int kLineMax = 1024;
constexpr int kLinePasses = 10;

// One pass: radix, span ns of the sub-transforms done so far, butterflies m = n / rad of a line, start
// of its twiddles, and the multipliers that divide by ns and m (floor(2^32 / d) + 1; exact for the
// small numerators used here).  The twiddles of a pass, exp(-2 pi i r k / (ns rad)) for r = 1 .. rad - 1,
// k < ns, lie k first: neighbouring butterflies read neighbouring values.  (One table of the n-th roots
// read with a stride r n / (ns rad) puts them on a few LDS banks: 646 instead of 523 us for 512-cell
// rows along z of 512^3 in FP64.)
struct LinePass {
  int rad, ns, m, tw;
  unsigned div_ns, div_m;
};

struct LinePlan {
  int n, npass, ntw;
  LinePass pass[kLinePasses];
};

// False when `n` is outside what these kernels take: 2 to kLineMax, factors 2, 3, 5 and 7.
bool line_plan(size_t n, LinePlan& P);

__device__ __forceinline__ int quotient(int t, unsigned magic) {
  return static_cast<int>(__umulhi(static_cast<unsigned>(t), magic));
}

template <typename R>
struct LineTile {
  static constexpr int lines = 128 / static_cast<int>(sizeof(Cx<R>));  // lines of a 128-byte row
  static constexpr int held = 64 / static_cast<int>(sizeof(R));        // elements a thread holds at most
};

// Butterflies of one pass that a thread takes: few enough for 96 registers of FP64 values and their
// twiddles, so that five wavefronts fit a SIMD.
template <typename R, int RAD>
constexpr int kFlies = (RAD >= 5 ? 1 : RAD >= 3 ? 2 : 4) * 8 / static_cast<int>(sizeof(R));

// ---- small DFTs in registers, forward exp(-2 pi i / n) or (INV) conjugate ----

template <bool INV, typename R>
__device__ __forceinline__ Cx<R> mul_mi(Cx<R> a) {  // a * (-i), inverse a * (+i)
  return INV ? Cx<R>{-a.im, a.re} : Cx<R>{a.im, -a.re};
}
template <typename R>
__device__ __forceinline__ Cx<R> cadd(Cx<R> a, Cx<R> b) { return {a.re + b.re, a.im + b.im}; }
template <typename R>
__device__ __forceinline__ Cx<R> csub(Cx<R> a, Cx<R> b) { return {a.re - b.re, a.im - b.im}; }

template <bool INV, typename R>
__device__ __forceinline__ void dft2r(Cx<R>& a, Cx<R>& b) {
  const Cx<R> t = a;
  a = cadd(t, b);
  b = csub(t, b);
}

template <bool INV, typename R>
__device__ __forceinline__ void dft3r(Cx<R>& a, Cx<R>& b, Cx<R>& c) {
  constexpr R h = R(0.86602540378443864676);  // sin(2 pi / 3)
  const Cx<R> s = cadd(b, c), d = csub(b, c);
  const Cx<R> m = {a.re - R(0.5) * s.re, a.im - R(0.5) * s.im};
  const Cx<R> r = mul_mi<INV>(Cx<R>{h * d.re, h * d.im});
  a = cadd(a, s);
  b = cadd(m, r);
  c = csub(m, r);
}

template <bool INV, typename R>
__device__ __forceinline__ void dft4r(Cx<R>& a, Cx<R>& b, Cx<R>& c, Cx<R>& d) {
  const Cx<R> s02 = cadd(a, c), d02 = csub(a, c), s13 = cadd(b, d), r = mul_mi<INV>(csub(b, d));
  a = cadd(s02, s13);
  c = csub(s02, s13);
  b = cadd(d02, r);
  d = csub(d02, r);
}

template <bool INV, typename R>
__device__ __forceinline__ void dft5r(Cx<R>& a, Cx<R>& b, Cx<R>& c, Cx<R>& d, Cx<R>& e) {
  constexpr R c1 = R(0.30901699437494742410), c2 = R(-0.80901699437494742410);
  constexpr R s1 = R(0.95105651629515357212), s2 = R(0.58778525229247312917);
  const Cx<R> p1 = cadd(b, e), q1 = csub(b, e), p2 = cadd(c, d), q2 = csub(c, d);
  const Cx<R> m1 = {a.re + (c1 * p1.re + c2 * p2.re), a.im + (c1 * p1.im + c2 * p2.im)};
  const Cx<R> m2 = {a.re + (c2 * p1.re + c1 * p2.re), a.im + (c2 * p1.im + c1 * p2.im)};
  const Cx<R> r1 = mul_mi<INV>(Cx<R>{s1 * q1.re + s2 * q2.re, s1 * q1.im + s2 * q2.im});
  const Cx<R> r2 = mul_mi<INV>(Cx<R>{s2 * q1.re - s1 * q2.re, s2 * q1.im - s1 * q2.im});
  a = cadd(a, cadd(p1, p2));
  b = cadd(m1, r1);
  e = csub(m1, r1);
  c = cadd(m2, r2);
  d = csub(m2, r2);
}

template <int RAD, bool INV, typename R>
__device__ __forceinline__ void dft_small(Cx<R>* v) {
  if constexpr (RAD == 2) {
    dft2r<INV>(v[0], v[1]);
  } else if constexpr (RAD == 3) {
    dft3r<INV>(v[0], v[1], v[2]);
  } else if constexpr (RAD == 4) {
    dft4r<INV>(v[0], v[1], v[2], v[3]);
  } else if constexpr (RAD == 5) {
    dft5r<INV>(v[0], v[1], v[2], v[3], v[4]);
  } else if constexpr (RAD == 6) {
    // 2 x 3: even and odd inputs, X_k = E_k + w6^k O_k, X_{k+3} = E_k - w6^k O_k
    constexpr R h = R(0.86602540378443864676);
    Cx<R> e0 = v[0], e1 = v[2], e2 = v[4], o0 = v[1], o1 = v[3], o2 = v[5];
    dft3r<INV>(e0, e1, e2);
    dft3r<INV>(o0, o1, o2);
    o1 = cmul(o1, Cx<R>{R(0.5), INV ? h : -h});
    o2 = cmul(o2, Cx<R>{R(-0.5), INV ? h : -h});
    v[0] = cadd(e0, o0), v[3] = csub(e0, o0);
    v[1] = cadd(e1, o1), v[4] = csub(e1, o1);
    v[2] = cadd(e2, o2), v[5] = csub(e2, o2);
  } else if constexpr (RAD == 7) {
    // symmetric and antisymmetric parts of the pairs (q, 7 - q)
    constexpr R c1 = R(0.62348980185873353053), c2 = R(-0.22252093395631440429),
                c3 = R(-0.90096886790241912624);
    constexpr R s1 = R(0.78183148246802980871), s2 = R(0.97492791218182360702),
                s3 = R(0.43388373911755812048);
    const Cx<R> a = v[0];
    Cx<R> p[3], q[3];
#pragma unroll
    for (int k = 0; k < 3; k++) p[k] = cadd(v[1 + k], v[6 - k]), q[k] = csub(v[1 + k], v[6 - k]);
    constexpr R C[3][3] = {{c1, c2, c3}, {c2, c3, c1}, {c3, c1, c2}};
    constexpr R S[3][3] = {{s1, s2, s3}, {s2, -s3, -s1}, {s3, -s1, s2}};
    v[0] = cadd(a, cadd(p[0], cadd(p[1], p[2])));
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const Cx<R> m = {a.re + (C[k][0] * p[0].re + C[k][1] * p[1].re + C[k][2] * p[2].re),
                       a.im + (C[k][0] * p[0].im + C[k][1] * p[1].im + C[k][2] * p[2].im)};
      const Cx<R> r = mul_mi<INV>(Cx<R>{S[k][0] * q[0].re + S[k][1] * q[1].re + S[k][2] * q[2].re,
                                        S[k][0] * q[0].im + S[k][1] * q[1].im + S[k][2] * q[2].im});
      v[1 + k] = cadd(m, r);
      v[6 - k] = csub(m, r);
    }
  } else if constexpr (RAD == 8) {
    // 2 x 4: sums give the even outputs, rotated differences the odd ones
    constexpr R h = R(0.70710678118654752440);
    Cx<R> a[4], b[4];
#pragma unroll
    for (int k = 0; k < 4; k++) a[k] = cadd(v[k], v[k + 4]), b[k] = csub(v[k], v[k + 4]);
    b[1] = cmul(b[1], Cx<R>{h, INV ? h : -h});
    b[2] = mul_mi<INV>(b[2]);
    b[3] = cmul(b[3], Cx<R>{-h, INV ? h : -h});
    dft4r<INV>(a[0], a[1], a[2], a[3]);
    dft4r<INV>(b[0], b[1], b[2], b[3]);
#pragma unroll
    for (int k = 0; k < 4; k++) v[2 * k] = a[k], v[2 * k + 1] = b[k];
  } else {
    static_assert(RAD == 10, "radix");
    // 2 x 5: X_2m from the sums, X_{2m+1} from the differences times w10^k
    constexpr R ca = R(0.80901699437494742410), sa = R(0.58778525229247312917);
    constexpr R cb = R(0.30901699437494742410), sb = R(0.95105651629515357212);
    Cx<R> a[5], b[5];
#pragma unroll
    for (int k = 0; k < 5; k++) a[k] = cadd(v[k], v[k + 5]), b[k] = csub(v[k], v[k + 5]);
    b[1] = cmul(b[1], Cx<R>{ca, INV ? sa : -sa});
    b[2] = cmul(b[2], Cx<R>{cb, INV ? sb : -sb});
    b[3] = cmul(b[3], Cx<R>{-cb, INV ? sb : -sb});
    b[4] = cmul(b[4], Cx<R>{-ca, INV ? sa : -sa});
    dft5r<INV>(a[0], a[1], a[2], a[3], a[4]);
    dft5r<INV>(b[0], b[1], b[2], b[3], b[4]);
#pragma unroll
    for (int k = 0; k < 5; k++) v[2 * k] = a[k], v[2 * k + 1] = b[k];
  }
}

template <int N>
struct Int {
  static constexpr int value = N;
};

template <class F>
__device__ __forceinline__ void with_radix(int rad, F&& f) {
  switch (rad) {
    case 8: f(Int<8>{}); break;
    case 4: f(Int<4>{}); break;
    case 2: f(Int<2>{}); break;
    case 6: f(Int<6>{}); break;
    case 3: f(Int<3>{}); break;
    case 5: f(Int<5>{}); break;
    case 10: f(Int<10>{}); break;
    default: f(Int<7>{}); break;
  }
}

// The block has threads for every pass: kFlies butterflies each (line_threads).
template <typename R, bool ACROSS>
struct LineFft {
  Cx<R>* buf;
  const Cx<R>* tw;
  int n;
  int nl;   // lines of the tile: kAcross a power of two
  int lw;   // its logarithm (kAcross)
  int nt, tid;

  __device__ __forceinline__ int slot(int line, int e) const {
    if (ACROSS) return ((e ^ (((e >> 2) ^ (e >> 3)) & 1)) << lw) + line;
    const int i = line * n + e;
    return i ^ ((i >> 4) & 15) ^ ((i >> 3) & 8);
  }

  // Butterfly f of this thread.
  __device__ __forceinline__ bool where(const LinePass& P, int f, int& line, int& j) const {
    const int t = tid + f * nt;
    if (ACROSS) {
      line = t & (nl - 1);
      j = t >> lw;
    } else {
      line = P.m > 1 ? quotient(t, P.div_m) : t;
      j = t - line * P.m;
    }
    return ACROSS ? j < P.m : line < nl;
  }

  // Element i (below LineTile<R>::held) of this thread in the order of memory, for loops over the
  // tile; (0, 0) where it has none, so that a loop that loads and uses elements need not branch
  // around each load (and wait for it before the next).
  __device__ __forceinline__ bool element(int i, unsigned div_n, int& line, int& e) const {
    const int t = tid + i * nt;
    if (ACROSS) {
      line = t & (nl - 1);
      e = t >> lw;
    } else {
      line = quotient(t, div_n);
      e = t - line * n;
    }
    const bool ok = ACROSS ? e < n : line < nl;
    if (!ok) line = e = 0;
    return ok;
  }

  // All passes of one direction.  ld(line, e) gives element e of a line, st(line, e, value) takes
  // it.  IN_LDS: the input lies in buf (after a barrier) and ld is not used.  OUT_LDS: the result is
  // left in buf, behind a barrier, and st is not used.
  template <bool INV, bool IN_LDS, bool OUT_LDS, class Load, class Store>
  __device__ __forceinline__ void run(const LinePlan& plan, Load&& ld, Store&& st) const {
    for (int p = 0; p < plan.npass; p++) {
      const LinePass P = plan.pass[p];
      with_radix(P.rad, [&](auto rc) {
        constexpr int RAD = decltype(rc)::value;
        constexpr int F = kFlies<R, RAD>;
        Cx<R> v[F * RAD];
#pragma unroll
        for (int f = 0; f < F; f++) {
          int line, j;
          if (!where(P, f, line, j)) continue;
          if (!IN_LDS && p == 0) {
#pragma unroll
            for (int r = 0; r < RAD; r++) v[f * RAD + r] = ld(line, j + r * P.m);
          } else {
#pragma unroll
            for (int r = 0; r < RAD; r++) v[f * RAD + r] = buf[slot(line, j + r * P.m)];
          }
        }
#pragma unroll
        for (int f = 0; f < F; f++) {
          int line, j;
          if (!where(P, f, line, j)) continue;
          if (P.ns > 1) {
            const Cx<R>* root = tw + P.tw + (j - quotient(j, P.div_ns) * P.ns);
#pragma unroll
            for (int r = 1; r < RAD; r++) {
              Cx<R> w = root[(r - 1) * P.ns];
              if (INV) w.im = -w.im;
              v[f * RAD + r] = cmul(v[f * RAD + r], w);
            }
          }
          dft_small<RAD, INV>(v + f * RAD);
        }
        if (OUT_LDS || p + 1 < plan.npass) {
          __syncthreads();
#pragma unroll
          for (int f = 0; f < F; f++) {
            int line, j;
            if (!where(P, f, line, j)) continue;
            const int q = P.ns > 1 ? quotient(j, P.div_ns) : j;
            const int e = q * P.ns * (RAD - 1) + j;  // q ns rad + (j - q ns)
#pragma unroll
            for (int r = 0; r < RAD; r++) buf[slot(line, e + r * P.ns)] = v[f * RAD + r];
          }
          __syncthreads();
        } else {
#pragma unroll
          for (int f = 0; f < F; f++) {
            int line, j;
            if (!where(P, f, line, j)) continue;
#pragma unroll
            for (int r = 0; r < RAD; r++) st(line, j + r * P.m, v[f * RAD + r]);
          }
        }
      });
    }
  }
};

// Threads for a tile of `lines` lines: every pass's butterflies, kFlies a thread, and the elements.
template <typename R>
inline int line_threads(const LinePlan& P, int lines) {
  int need = (lines * P.n + LineTile<R>::held - 1) / LineTile<R>::held;
  for (int i = 0; i < P.npass; i++) {
    const int rad = P.pass[i].rad;
    const int flies = rad >= 5 ? kFlies<R, 5> : rad >= 3 ? kFlies<R, 3> : kFlies<R, 2>;
    const int t = (lines * P.pass[i].m + flies - 1) / flies;
    need = t > need ? t : need;
  }
  return (need + 63) / 64 * 64;
}

struct LineCols {
  int lw, threads;
  size_t lds;
};

// Tile of kAcross lines: 128-byte rows, 64-byte ones for lines that would need more than 1024 threads.
template <typename R>
LineCols line_cols(const LinePlan& P) {
  int lw = sizeof(R) == 8 ? 3 : 4;
  if (line_threads<R>(P, 1 << lw) > 1024) lw--;
  return {lw, line_threads<R>(P, 1 << lw),
          sizeof(Cx<R>) * ((static_cast<size_t>(P.n + 1) << lw) + static_cast<size_t>(P.ntw))};
}

struct LineRows {
  int nl, threads;
  size_t lds;
};
// Pairs of rows: as many as 256 threads take.  Blocks of a multiple of four wavefronts share the
// four SIMDs evenly; five pairs of 384 elements on five wavefronts left half of the slots empty
// (2.2 against 1.35 ms for six fields of 384^3).
template <typename R>
LineRows line_rows(const LinePlan& P) {
  int nl = 256 * LineTile<R>::held / P.n;
  if (nl < 1) nl = 1;
  while (nl > 1 && line_threads<R>(P, nl) > 256) nl--;
  return {nl, line_threads<R>(P, nl), sizeof(Cx<R>) * (((nl * P.n + 15) & ~15) + static_cast<size_t>(P.ntw))};
}

}  // namespace prh
