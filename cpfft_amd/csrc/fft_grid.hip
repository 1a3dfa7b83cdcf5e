// fft_grid.hip -- G_K_dF (src/G_K_dF.f:11-87) and the CG iteration around it
// for the grid edges that fft_pencil.hip's plans do not cover: 16, 32 and 48
// with compile-time plans, every other edge (prime factors up to 13) with a
// plan read at run time; and tangent_homo's solves at 64 and 96.
//
// Up to edge 126 one component of an x slab (N z lines of N points, or their
// half spectrum) fits the LDS of a CU, and an application is three kernels:
//   k_fwd    per (x, component): K4:F contraction (ddot42n order,
//            G_K_dF.f:241-268), z and y transforms; in a CG iteration first
//            the convergence test of the previous iteration, the direction
//            p = r + beta p and the p.(K4:p) partial sums
//   k_mid    x transform, Green projection of a tensor row, x inverse; in a
//            CG iteration an extra block forms alpha meanwhile
//   k_inv    per (x, component): y and z inverse, with the x, r update and
//            the r.r partial sums
// Above it z, y and x have kernels of their own (k_zf, k_y, k_x, k_y, k_zi).
// At these sizes a launch and the gap after it cost as much as the work
// (16^3: seven kernels an iteration took 29 us, three take 18), so the nine
// right-hand sides of tangent_homo also share every launch.
//
// Half spectrum of a right-hand side: [c][x][kz][y] (slabs), or T1[c][kz][L]
// with L = x N + y the line index and T2[c][kz][y][x].  Two real lines share
// one complex FFT.  For even N the textbook operator removes the Nyquist
// planes, so plane kz = N/2 is neither stored nor transformed.
//
// In LDS a line's elements are contiguous and rows have an odd stride;
// consecutive threads take consecutive lines, so reads and writes of a
// transform fall on distinct banks without padding.
#include <algorithm>

#include "kernels.h"

// No implicit contraction into FMAs: the order and rounding of every
// transform and sum is the same in all instantiations and block sizes.  The
// transforms' FMAs are written out.
#pragma clang fp contract(off)

namespace cpfft {
namespace gp {

// x / d for 0 <= x, d < 2^16
struct Div {
  unsigned d, m;
  __host__ __device__ explicit Div(unsigned dd = 1) : d(dd), m(dd > 1 ? 0xFFFFFFFFu / dd + 1u : 0u) {}
  __device__ __forceinline__ int operator()(int x) const {
    return d == 1u ? x : (int)__umulhi((unsigned)x, m);
  }
};

constexpr int kMaxE = 8;    // elements per thread of a transform, at most
constexpr int kSlabN = 126; // largest edge of the slab kernels: N (N/2 + 1) <= kMaxE * 1024
constexpr int kML = 8;      // x lines per component and block of k_mid (128-byte runs)
constexpr int kMaxSt = 8;
// Kernels' NC: the edge, or a plan read at run time.  Radices 11 and 13 take
// more registers than 1024 threads have (24 to 96 bytes a lane go to scratch),
// so the edges without these factors have instantiations without them: no
// scratch, a solve at 45^3 3.21 ms instead of 3.35.
constexpr int kAnyRadix = 0, kSmooth = -1;
inline bool smooth(int N) { return N <= kSlabN && N % 11 != 0 && N % 13 != 0; }

struct Grid {
  int N, NZ, nzk, NN;  // edge, N/2+1, planes kept, lines N*N
  int TL, nzb;         // lines per block of the z passes, their blocks
  int gamma_mode;
  bool pair;           // k_mid leaves u, not F (see there)
  long V, S1;
  Div dN;
  int nst;
  int rad[kMaxSt];
  Div dNs[kMaxSt];
};

// ---------------------------------------------------------------- transforms
__device__ __forceinline__ cplx cadd(cplx a, cplx b) { return cplx{a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ cplx csub(cplx a, cplx b) { return cplx{a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ cplx cmul(cplx a, cplx b) {
  return cplx{fma(a.re, b.re, -(a.im * b.im)), fma(a.re, b.im, a.im * b.re)};
}
template <bool FWD>
__device__ __forceinline__ cplx mul_mi(cplx a) {  // by -i forward, +i inverse
  return FWD ? cplx{a.im, -a.re} : cplx{-a.im, a.re};
}
template <bool FWD>
__device__ __forceinline__ cplx twid(const cplx* tw, int e) {
  cplx w = tw[e];
  if (!FWD) w.im = -w.im;
  return w;
}

// cos and sin of 2 pi k / R for k <= R/2
template <int R>
struct Root;
template <>
struct Root<3> {
  static constexpr double c[2] = {1.0, -0.5}, s[2] = {0.0, 0.866025403784438646764};
};
template <>
struct Root<5> {
  static constexpr double c[3] = {1.0, 0.309016994374947424102, -0.809016994374947424102};
  static constexpr double s[3] = {0.0, 0.951056516295153572116, 0.587785252292473129169};
};
template <>
struct Root<6> {
  static constexpr double c[4] = {1.0, 0.5, -0.5, -1.0};
  static constexpr double s[4] = {0.0, 0.866025403784438646764, 0.866025403784438646764, 0.0};
};
template <>
struct Root<7> {
  static constexpr double c[4] = {1.0, 0.623489801858733530525, -0.222520933956314404289,
                                  -0.900968867902419126236};
  static constexpr double s[4] = {0.0, 0.781831482468029808708, 0.974927912181823607018,
                                  0.433883739117558120476};
};
template <>
struct Root<9> {
  static constexpr double c[5] = {1.0, 0.766044443118978035202, 0.173648177666930348852, -0.5,
                                  -0.939692620785908384054};
  static constexpr double s[5] = {0.0, 0.642787609686539326323, 0.984807753012208059367,
                                  0.866025403784438646764, 0.342020143325668733044};
};
template <>
struct Root<10> {
  static constexpr double c[6] = {1.0, 0.809016994374947424102, 0.309016994374947424102,
                                  -0.309016994374947424102, -0.809016994374947424102, -1.0};
  static constexpr double s[6] = {0.0, 0.587785252292473129169, 0.951056516295153572116,
                                  0.951056516295153572116, 0.587785252292473129169, 0.0};
};
template <>
struct Root<11> {
  static constexpr double c[6] = {1.0, 0.841253532831181168862, 0.415415013001886425529,
                                  -0.142314838273285140444, -0.654860733945285064057,
                                  -0.95949297361449738989};
  static constexpr double s[6] = {0.0, 0.540640817455597582108, 0.909631995354518371412,
                                  0.989821441880932732376, 0.755749574354258283774,
                                  0.281732556841429697711};
};
template <>
struct Root<13> {
  static constexpr double c[7] = {1.0, 0.8854560256532098959, 0.568064746731155802512,
                                  0.120536680255323053349, -0.35460488704253562597,
                                  -0.748510748171101098635, -0.970941817426052027157};
  static constexpr double s[7] = {0.0, 0.464723172043768545656, 0.82298386589365639458,
                                  0.992708874098053992801, 0.93501624268541482344,
                                  0.663122658240795202377, 0.239315664287557767149};
};
template <int R>
__device__ __forceinline__ constexpr double rc(int e) {
  return Root<R>::c[e <= R / 2 ? e : R - e];
}
template <int R>
__device__ __forceinline__ constexpr double rs(int e) {
  return e <= R / 2 ? Root<R>::s[e] : -Root<R>::s[R - e];
}

// in-register DFT of size R
template <int R, bool FWD>
__device__ __forceinline__ void dft(cplx* x) {
  if constexpr (R == 2) {
    const cplx a = x[0], b = x[1];
    x[0] = cadd(a, b);
    x[1] = csub(a, b);
  } else if constexpr (R == 4) {
    const cplx b0 = cadd(x[0], x[2]), b1 = csub(x[0], x[2]), b2 = cadd(x[1], x[3]);
    const cplx b3 = mul_mi<FWD>(csub(x[1], x[3]));
    x[0] = cadd(b0, b2);
    x[1] = cadd(b1, b3);
    x[2] = csub(b0, b2);
    x[3] = csub(b1, b3);
  } else if constexpr (R == 8) {
    cplx e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
    dft<4, FWD>(e);
    dft<4, FWD>(o);
    const double h = 0.70710678118654752440;  // sqrt(2)/2
    const cplx s1 = FWD ? cplx{o[1].re + o[1].im, o[1].im - o[1].re}
                        : cplx{o[1].re - o[1].im, o[1].re + o[1].im};
    const cplx s3 = FWD ? cplx{o[3].im - o[3].re, -(o[3].re + o[3].im)}
                        : cplx{-(o[3].re + o[3].im), o[3].re - o[3].im};
    const cplx w2 = mul_mi<FWD>(o[2]);
    x[0] = cadd(e[0], o[0]);
    x[4] = csub(e[0], o[0]);
    x[1] = cplx{fma(h, s1.re, e[1].re), fma(h, s1.im, e[1].im)};
    x[5] = cplx{fma(-h, s1.re, e[1].re), fma(-h, s1.im, e[1].im)};
    x[2] = cadd(e[2], w2);
    x[6] = csub(e[2], w2);
    x[3] = cplx{fma(h, s3.re, e[3].re), fma(h, s3.im, e[3].im)};
    x[7] = cplx{fma(-h, s3.re, e[3].re), fma(-h, s3.im, e[3].im)};
  } else if constexpr (R == 6 || R == 9 || R == 10) {
    // R = A B: DFTs of size B over x[n + A m], twiddles, DFTs of size A
    constexpr int A = R == 9 ? 3 : 2, B = R / A;
    cplx y[A][B];
#pragma unroll
    for (int n = 0; n < A; ++n) {
#pragma unroll
      for (int m = 0; m < B; ++m) y[n][m] = x[n + A * m];
      dft<B, FWD>(y[n]);
      if (n > 0)
#pragma unroll
        for (int k = 1; k < B; ++k)
          y[n][k] = cmul(y[n][k], cplx{rc<R>(n * k), FWD ? -rs<R>(n * k) : rs<R>(n * k)});
    }
#pragma unroll
    for (int k = 0; k < B; ++k) {
      cplx z[A];
#pragma unroll
      for (int n = 0; n < A; ++n) z[n] = y[n][k];
      dft<A, FWD>(z);
#pragma unroll
      for (int n = 0; n < A; ++n) x[k + B * n] = z[n];
    }
  } else {
    // odd prime: X_q, X_{R-q} = C_q -+ i S_q from sums and differences of
    // x_t and x_{R-t}
    constexpr int H = R / 2;
    cplx a[H + 1], d[H + 1];
    cplx s0 = x[0];
#pragma unroll
    for (int t = 1; t <= H; ++t) {
      a[t] = cadd(x[t], x[R - t]);
      d[t] = csub(x[t], x[R - t]);
      s0 = cadd(s0, a[t]);
    }
    const cplx x0 = x[0];
    x[0] = s0;
#pragma unroll
    for (int q = 1; q <= H; ++q) {
      cplx C = x0, S{0.0, 0.0};
#pragma unroll
      for (int t = 1; t <= H; ++t) {
        const double c = rc<R>((q * t) % R), s = rs<R>((q * t) % R);
        C = cplx{fma(c, a[t].re, C.re), fma(c, a[t].im, C.im)};
        S = cplx{fma(s, d[t].re, S.re), fma(s, d[t].im, S.im)};
      }
      // forward X_q = C - i S: (C.re + S.im, C.im - S.re)
      const cplx u{C.re + S.im, C.im - S.re}, v{C.re - S.im, C.im + S.re};
      x[q] = FWD ? u : v;
      x[R - q] = FWD ? v : u;
    }
  }
}

// One in-place Stockham pass of radix R over nl lines of length N: a thread
// reads its butterflies (MB at most) into registers, the block
// synchronises, the results go back.
template <int R, int MB, bool FWD, class LB>
__device__ __forceinline__ void stage(cplx* buf, const cplx* tw, int N, int Ns, Div dNs, int nl,
                                      Div dnl, LB lb, int es) {
  const int nb = N / R, tot = nl * nb, ts = N / (Ns * R), T = blockDim.x;
  cplx x[MB][R];
#pragma unroll
  for (int u = 0; u < MB; ++u) {
    const int b = threadIdx.x + u * T;
    if (b < tot) {
      const int j = dnl(b), line = b - j * nl;
      const cplx* s = buf + lb(line) + j * es;
#pragma unroll
      for (int t = 0; t < R; ++t) x[u][t] = s[t * nb * es];
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < MB; ++u) {
    const int b = threadIdx.x + u * T;
    if (b < tot) {
      const int j = dnl(b), line = b - j * nl;
      int o = j * R;
      if (Ns > 1) {
        const int h = dNs(j), k = j - h * Ns;
        o = h * Ns * R + k;
#pragma unroll
        for (int t = 1; t < R; ++t) x[u][t] = cmul(x[u][t], twid<FWD>(tw, t * k * ts));
      }
      dft<R, FWD>(x[u]);
      cplx* d = buf + lb(line) + o * es;
#pragma unroll
      for (int q = 0; q < R; ++q) d[q * Ns * es] = x[u][q];
    }
  }
  __syncthreads();
}

// radices of the compile-time edges
constexpr int ct_radix(int n, int st) {
  return n == 16 ? (st == 0 ? 4 : st == 1 ? 4 : 0)
       : n == 32 ? (st == 0 ? 8 : st == 1 ? 4 : 0)
       : n == 48 ? (st == 0 ? 8 : st == 1 ? 6 : 0)
       : n == 64 ? (st == 0 ? 8 : st == 1 ? 8 : 0)
       : n == 96 ? (st == 0 ? 6 : st == 1 ? 4 : st == 2 ? 4 : 0) : 0;
}
template <int NC, bool FWD, int ME, class LB, int ST = 0, int NS = 1>
__device__ __forceinline__ void fft_ct(cplx* buf, const cplx* tw, int nl, Div dnl, LB lb, int es) {
  constexpr int R = ct_radix(NC, ST);
  if constexpr (R > 0) {
    stage<R, (ME + R - 1) / R, FWD>(buf, tw, NC, NS, Div(NS), nl, dnl, lb, es);
    fft_ct<NC, FWD, ME, LB, ST + 1, NS * R>(buf, tw, nl, dnl, lb, es);
  }
}
// unscaled FFT of nl lines in place; at most ME elements per thread.  Starts
// with the lines written (the caller synchronises before), ends synchronised.
template <int NC, bool FWD, int ME, class LB>
__device__ __forceinline__ void fft(cplx* buf, const cplx* tw, const Grid& g, int nl, LB lb, int es) {
  const Div dnl(nl);
  if constexpr (NC > 0) {
    fft_ct<NC, FWD, ME>(buf, tw, nl, dnl, lb, es);
  } else {
    int Ns = 1;
    for (int st = 0; st < g.nst; ++st) {
      const int r = g.rad[st];
#define CPFFT_STAGE(R)                                                                    \
  case R:                                                                                 \
    stage<R, (ME + R - 1) / R, FWD>(buf, tw, g.N, Ns, g.dNs[st], nl, dnl, lb, es);        \
    break;
      switch (r) {
        CPFFT_STAGE(2) CPFFT_STAGE(3) CPFFT_STAGE(4) CPFFT_STAGE(5) CPFFT_STAGE(6)
        CPFFT_STAGE(7) CPFFT_STAGE(8) CPFFT_STAGE(9) CPFFT_STAGE(10)
        default: break;
      }
      if constexpr (NC == kAnyRadix) {
        switch (r) {
          CPFFT_STAGE(11) CPFFT_STAGE(13)
          default: break;
        }
      }
#undef CPFFT_STAGE
      Ns *= r;
    }
  }
}

template <int NC>
__device__ __forceinline__ int edge(const Grid& g) {
  return NC > 0 ? NC : g.N;
}
template <int NC>
__device__ __forceinline__ Div divN(const Grid& g) {
  if constexpr (NC > 0) return Div(NC);
  return g.dN;
}
template <int NC>
__device__ __forceinline__ void load_tw(cplx* tw, const cplx* __restrict__ twg, int N) {
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twg[i];
}

// sum over a wave, valid in every lane
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// per right-hand side pointers of a launch
struct Ptr {
  double* p[9];
};

// ---------------------------------------------------------------- arguments
struct FwdArgs {
  Ptr F;                 // operand (!DIR), or the direction of the last iteration (DIR)
  long fs;               // !HASK: stride of F's components
  Ptr r, pn;             // DIR: residual, new direction
  const double* K4;
  cplx* T1;
  long ts;               // spectrum entries per right-hand side
  const cplx* tw;
  int nrhs;
  // DIR
  const CGScalars* old;  // state before this iteration (!DIR: finished systems are skipped)
  CGScalars* nw;         // state of this iteration (may be old when !chk)
  const double* rrp;     // chk: r.r partial sums of the previous iteration
  int nrr;
  int chk;               // test convergence first
  const double* dc;      // with m: voxel sums, running means (launch_cg_check)
  double* m;
  double scale;
  double* pqp;           // p.(K4:p) partial sums
};
struct MidArgs {
  cplx* T1;
  cplx* T2;          // five-kernel path
  long ts;
  const cplx* tw;
  CGScalars* cs;     // nullptr: no CG; else blocks of finished systems return
  const double* pqp; // alpha is formed from npq partial sums
  int npq;
  double* dc;        // voxel sums of the nine components (9 per right-hand side)
};
struct InvArgs {
  const cplx* T1;
  long ts;
  const cplx* tw;
  Ptr out;             // MODE 0, 1, 3
  Ptr pd, r, x;        // MODE 1: pd; MODE 2: r, with x.p[rhs] also pd and x
  double* part;        // MODE 1, 2, 3: partial sums
  const CGScalars* cs; // nullptr: no CG
};

// ------------------------------------------------------- steps of the blocks
// Block -> (run of points, components, right-hand side).  The blocks of a run
// read the same F (or r, p) and, for several right-hand sides, the same K4;
// they are placed on one XCD (blocks go to the eight XCDs in turn), next to
// each other, so that its L2 serves all but the first.
struct Where {
  int tile, rhs, c0;
};
template <int CPB>
__device__ __forceinline__ Where where(int nrhs) {
  constexpr int NCB = 9 / CPB;
  const int loc = blockIdx.x >> 3, per = NCB * nrhs, tq = loc / per, i = loc - tq * per;
  const int rhs = i / NCB;
  return Where{tq * 8 + (int)(blockIdx.x & 7), rhs, (i - rhs * NCB) * CPB};
}

// Start of a CG iteration's first kernel: with chk the test of the previous
// iteration, repeated by every block from the r.r partial sums (in
// ordered_sum's order; a few thousand values from L2 at most, instead of a
// launch) and kept by the first one.  Returns whether the system is done.
__device__ __forceinline__ bool cg_begin(const FwdArgs& a, int rhs, bool first, double& beta) {
  __shared__ double s_beta;
  __shared__ int s_done;
  if (threadIdx.x < 64) {
    CGScalars c = a.old[rhs];
    if (a.chk && c.done == 0) {
      const double* part = a.rrp + (long)rhs * a.nrr;
      double acc[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        acc[q] = 0.0;
        for (int i = threadIdx.x + 64 * q; i < a.nrr; i += 256) acc[q] += part[i];
      }
      const double rr1 = wave_sum((acc[0] + acc[2]) + (acc[1] + acc[3]));
      if (threadIdx.x == 0) {
        if (first && a.m)
          for (int k = 0; k < 9; ++k) a.m[9 * rhs + k] += c.alpha * (a.dc[9 * rhs + k] * a.scale);
        cg_check(&c, rr1);
      }
    }
    if (threadIdx.x == 0) {
      if (first && a.nw != a.old) a.nw[rhs] = c;
      s_beta = c.beta;
      s_done = c.done;
    }
  }
  __syncthreads();
  beta = s_beta;
  return s_done != 0;
}

// What components c0 .. c0 + CPB of K4:F (or of F, !HASK) at a voxel are formed
// from; DIR: F is the last direction.  Fetched apart from their use: the first
// point's travel while the kernel still reads the state of the iteration.
template <bool HASK, bool DIR, int CPB>
struct Point {
  double k[HASK ? CPB : 1][9], f[9], r[9];
};
template <bool HASK, bool DIR, int CPB>
__device__ __forceinline__ void fetch_point(const FwdArgs& a, int rhs, int c0, long e, long V,
                                            Point<HASK, DIR, CPB>& p) {
  const double* F = a.F.p[rhs];
  if constexpr (HASK) {
    // uniform bases and one 32-bit offset (8 V < 2^32 at these edges): 27
    // loads without 27 addresses in vector registers
    const unsigned o = 8u * (unsigned)e;
    auto ld = [&](const double* base) {
      return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(base) + o);
    };
#pragma unroll
    for (int j = 0; j < CPB; ++j)
#pragma unroll
      for (int d = 0; d < 9; ++d) p.k[j][d] = ld(a.K4 + (9 * (c0 + j) + d) * V);
    if constexpr (DIR) {
      const double* R = a.r.p[rhs];
#pragma unroll
      for (int d = 0; d < 9; ++d) p.r[d] = ld(R + d * V);
    }
#pragma unroll
    for (int d = 0; d < 9; ++d) p.f[d] = ld(F + d * V);
  } else {
#pragma unroll
    for (int j = 0; j < CPB; ++j) p.f[j] = F[(c0 + j) * a.fs + e];
  }
}
// (K4:F)_c of components c0 .. c0 + CPB at voxel e (or F_c without K4); DIR:
// F is the new direction r + beta F, its components stored, fc its value there
template <bool HASK, bool DIR, int CPB>
__device__ __forceinline__ void use_point(const FwdArgs& a, int rhs, int c0, long e, long V,
                                          double beta, const Point<HASK, DIR, CPB>& p,
                                          double (&v)[CPB], double (&fc)[CPB]) {
  if constexpr (HASK) {
    double f[9];
    if constexpr (DIR) {
#pragma unroll
      for (int d = 0; d < 9; ++d) f[d] = p.r[d];
      if (beta != 0.0) {
#pragma unroll
        for (int d = 0; d < 9; ++d) f[d] = f[d] + beta * p.f[d];
      }
    } else {
#pragma unroll
      for (int d = 0; d < 9; ++d) f[d] = p.f[d];
    }
#pragma unroll
    for (int j = 0; j < CPB; ++j) {
      v[j] = ddot42n_row(p.k[j], f);
      if constexpr (DIR) {
#pragma unroll
        for (int d = 0; d < 9; ++d) fc[j] = (d == c0 + j) ? f[d] : fc[j];
        a.pn.p[rhs][(c0 + j) * V + e] = fc[j];
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < CPB; ++j) v[j] = p.f[j];
  }
}

// The points e0 + p, p < npts, of a run (line p / N, z = p mod N) into the
// line pairs of buf; DIR: the sums of v fc to pq[j * pqs] (each thread its
// points in turn, then the block).  pt: with AHEAD the operands of point tid,
// already fetched.  Ends synchronised.
template <int NC, bool HASK, bool DIR, int CPB, bool AHEAD>
__device__ __forceinline__ void load_lines(const Grid& g, const FwdArgs& a, int rhs, int c0,
                                           long e0, int npts, int nl, double beta, cplx* buf,
                                           double* pq, long pqs, Point<HASK, DIR, CPB>& pt) {
  __shared__ double wsum[CPB][16];
  const int N = edge<NC>(g), LS = N | 1, LP = (nl + 1) >> 1, T = blockDim.x, tid = threadIdx.x;
  const Div dN = divN<NC>(g);
  double* bd = reinterpret_cast<double*>(buf);
  double acc[CPB];
#pragma unroll
  for (int j = 0; j < CPB; ++j) acc[j] = 0.0;
  for (int p = tid; p < npts; p += T) {
    double v[CPB], fc[CPB];
    if (!AHEAD) fetch_point<HASK, DIR, CPB>(a, rhs, c0, e0 + p, g.V, pt);
    use_point<HASK, DIR, CPB>(a, rhs, c0, e0 + p, g.V, beta, pt, v, fc);
    if (AHEAD && p + T < npts) fetch_point<HASK, DIR, CPB>(a, rhs, c0, e0 + p + T, g.V, pt);
    const int l = dN(p), z = p - l * N;
#pragma unroll
    for (int j = 0; j < CPB; ++j) {
      bd[2 * ((j * LP + (l >> 1)) * LS + z) + (l & 1)] = v[j];
      if constexpr (DIR) acc[j] += v[j] * fc[j];
    }
  }
  if constexpr (DIR) {
    if (pq) {
#pragma unroll
      for (int j = 0; j < CPB; ++j) {
        const double w = wave_sum(acc[j]);
        if ((tid & 63) == 0) wsum[j][tid >> 6] = w;
      }
    }
  }
  if (nl & 1)  // the last line has no partner
    for (int i = tid; i < CPB * N; i += T) {
      const int j = dN(i), z = i - j * N;
      bd[2 * ((j * LP + LP - 1) * LS + z) + 1] = 0.0;
    }
  __syncthreads();
  if constexpr (DIR) {
    if (pq && tid < CPB) {
      double s = wsum[tid][0];
      for (int k = 1; k < T >> 6; ++k) s += wsum[tid][k];
      pq[tid * pqs] = s;
    }
  }
}

// Z = FFT(a + i b): A_k = (Z_k + conj Z_{N-k})/2, B_k = -i (Z_k - conj Z_{N-k})/2
__device__ __forceinline__ void unpack(const cplx* line, int k, int N, cplx& A, cplx& B) {
  const cplx zk = line[k], zn = line[k == 0 ? 0 : N - k];
  A = cplx{0.5 * (zk.re + zn.re), 0.5 * (zk.im - zn.im)};
  B = cplx{0.5 * (zk.im + zn.im), -0.5 * (zk.re - zn.re)};
}
// and back: Z_k = A_k + i B_k, with A_{N-k} = conj A_k
__device__ __forceinline__ void pack(cplx* line, int k, int N, int NZ, cplx A, cplx B) {
  line[k] = cplx{A.re - B.im, A.im + B.re};
  if (k >= 1 && N - k >= NZ) line[N - k] = cplx{A.re + B.im, B.re - A.im};
}

// The transformed lines of a run back to voxels (times 1/N^3).  MODE 0: out =
// the transform.  1: also the partial sum of pd . out.  2: the transform q is
// not stored; r -= alpha q, with x also x += alpha pd, and the partial sum
// of the new r . r.  3: out = minus the transform and the partial sum of its
// square.  Sums as in load_lines.
struct Fetched {
  double p[2], r[2], x[2];
};
template <int MODE>
__device__ __forceinline__ void fetch(const InvArgs& a, int rhs, long i, bool in, int j, Fetched& f) {
  const bool xu = MODE == 2 && a.x.p[rhs] != nullptr;
  f.p[j] = in && (MODE == 1 || xu) ? a.pd.p[rhs][i] : 0.0;
  f.r[j] = in && MODE == 2 ? a.r.p[rhs][i] : 0.0;
  f.x[j] = in && xu ? a.x.p[rhs][i] : 0.0;
}
template <int NC, int MODE>
__device__ __forceinline__ void store_lines(const Grid& g, const InvArgs& a, int rhs, long e0,
                                            int npts, const cplx* buf, Fetched& f, double* part) {
  __shared__ double wsum[16];
  const int N = edge<NC>(g), LS = N | 1, T = blockDim.x, tid = threadIdx.x;
  const Div dN = divN<NC>(g);
  const double sc = 1.0 / (double)g.V;
  const double al = MODE == 2 ? a.cs[rhs].alpha : 0.0;
  const bool xu = MODE == 2 && a.x.p[rhs] != nullptr;
  double acc = 0.0;
  for (int b0 = 0; b0 < npts; b0 += 2 * T) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int p = b0 + j * T + tid;
      if (p < npts) {
        const int l = dN(p), z = p - l * N;
        const cplx v = buf[(l >> 1) * LS + z];
        const double q = ((l & 1) ? v.im : v.re) * sc;
        const long i = e0 + p;
        if constexpr (MODE == 2) {
          if (xu) a.x.p[rhs][i] = f.x[j] + al * f.p[j];
          const double rn = f.r[j] - al * q;
          a.r.p[rhs][i] = rn;
          acc += rn * rn;
        } else {
          a.out.p[rhs][i] = MODE == 3 ? -q : q;
          acc += MODE == 3 ? q * q : q * f.p[j];
        }
      }
      if (b0 + 2 * T < npts) fetch<MODE>(a, rhs, e0 + p + 2 * T, p + 2 * T < npts, j, f);
    }
  }
  if constexpr (MODE > 0) {
    acc = wave_sum(acc);
    if ((tid & 63) == 0) wsum[tid >> 6] = acc;
    __syncthreads();
    if (tid == 0) {
      double s = wsum[0];
      for (int k = 1; k < T >> 6; ++k) s += wsum[k];
      *part = s;
    }
  }
}

// components 3 row .. 3 row + 2 at frequency (x, y, kz) from the same three;
// the operations and operands are project9's
__device__ __forceinline__ void project_row(int N, int gamma_mode, int x, int y, int kz,
                                            const cplx A[3], cplx o[3]) {
  const bool even = (N & 1) == 0;
  const int fx = x <= N / 2 ? x : x - N, fy = y <= N / 2 ? y : y - N;
  o[0] = o[1] = o[2] = cplx{0.0, 0.0};
  if (gamma_mode == 0 && even) {
    double q1[3], q2[3], s1, s2;
    proj_vectors(N, gamma_mode, x, y, kz, q1, q2);
    proj_weights(N, gamma_mode, x, y, kz, s1, s2);
    if (s1 != 0.0) {
      const cplx aq = gamma_aq(q1, A);
#pragma unroll
      for (int j = 0; j < 3; ++j) gamma_term(aq, q1[j], s1, o[j]);
    }
    if (s2 != 0.0) {
      const cplx aq = gamma_aq(q2, A);
#pragma unroll
      for (int j = 0; j < 3; ++j) gamma_term(aq, q2[j], s2, o[j]);
    }
  } else if (!(even && (2 * abs(fx) == N || 2 * abs(fy) == N || 2 * kz == N))) {
    const double q[3] = {(double)fx, (double)fy, (double)kz};
    const double qq = q[0] * q[0] + q[1] * q[1] + q[2] * q[2];
    if (qq > 1e-10) {
      const double s = 1.0 / qq;
      const cplx aq = gamma_aq(q, A);
#pragma unroll
      for (int j = 0; j < 3; ++j) gamma_term(aq, q[j], s, o[j]);
    }
  }
}

// alpha = rr / p.q from the partial sums, by one wave
__device__ __forceinline__ void form_alpha(const MidArgs& a, int rhs) {
  const double* part = a.pqp + (long)rhs * a.npq;
  double acc = 0.0;
  int i = threadIdx.x;
  for (; i + 7 * 64 < a.npq; i += 8 * 64) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = part[i + 64 * u];
#pragma unroll
    for (int u = 0; u < 8; ++u) acc += v[u];
  }
  for (; i < a.npq; i += 64) acc += part[i];
  acc = wave_sum(acc);
  if (threadIdx.x == 0) a.cs[rhs].alpha = a.cs[rhs].rr / acc;
}

// ------------------------------------------------------------- slab kernels
// k_fwd: block = (x, component, right-hand side); blockIdx.x as where().
// One buffer: the line pairs [m][z], after the z transforms (through
// registers) the half spectrum [kz][y].  One component a block: three (F read
// three times instead of nine) took as long for one system at 32^3 and 48^3.
// The blocks of a slab share F through their XCD's L2 (798 B a voxel are
// fetched at 32^3, 855 at 90^3, 865 at 126^3, of the 792 that K4, r and p are),
// but with the contraction in it the kernel is slower than fft_pencil.hip's
// pass A from 64^3 on (56 against 41 us): loads, transforms and stores of a
// block follow one another, and from 64^3 its threads and LDS leave room for
// one block a CU, so the stream stops meanwhile (2.6 TB/s at 90^3).
template <int NC, int ME, bool HASK, bool DIR, bool AHEAD>
__global__ __launch_bounds__(1024) void k_fwd(Grid g, FwdArgs a) {
  extern __shared__ cplx lds[];
  const Where w = where<1>(a.nrhs);
  const int N = edge<NC>(g), LS = N | 1, NN = N * N, T = blockDim.x, tid = threadIdx.x;
  if (w.tile >= N) return;
  const int x = w.tile, nzk = g.nzk, LP = (N + 1) >> 1;
  cplx* tw = lds;
  cplx* buf = lds + N;
  Point<HASK, DIR, 1> pt;
  if (AHEAD && tid < NN) fetch_point<HASK, DIR, 1>(a, w.rhs, w.c0, (long)x * NN + tid, g.V, pt);
  load_tw<NC>(tw, a.tw, N);
  double beta = 0.0;
  if constexpr (DIR) {
    if (cg_begin(a, w.rhs, x == 0 && w.c0 == 0, beta)) return;
  } else {
    if (a.old && a.old[w.rhs].done) return;
  }
  load_lines<NC, HASK, DIR, 1, AHEAD>(g, a, w.rhs, w.c0, (long)x * NN, NN, N, beta, buf,
                               DIR && a.pqp ? a.pqp + ((long)w.rhs * 9 + w.c0) * N + x : nullptr, N,
                               pt);
  auto lb = [&](int l) { return l * LS; };
  fft<NC, true, ME>(buf, tw, g, LP, lb, 1);
  {
    constexpr int MQ = ME / 2 + 1;  // pairs per thread
    cplx A[MQ], B[MQ];
    const Div dLP(LP);
    const int tot = LP * nzk;
#pragma unroll
    for (int u = 0; u < MQ; ++u) {
      const int q = tid + u * T;
      if (q < tot) {
        const int k = dLP(q), m = q - k * LP;
        unpack(buf + m * LS, k, N, A[u], B[u]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < MQ; ++u) {
      const int q = tid + u * T;
      if (q < tot) {
        const int k = dLP(q), m = q - k * LP;
        cplx* d = buf + k * LS + 2 * m;
        d[0] = A[u];
        if (2 * m + 1 < N) d[1] = B[u];
      }
    }
    __syncthreads();
  }
  fft<NC, true, ME>(buf, tw, g, nzk, lb, 1);
  const int M = nzk * N;
  const Div dN = divN<NC>(g);
  cplx* o = a.T1 + w.rhs * a.ts + ((long)w.c0 * N + x) * M;
  for (int i = tid; i < M; i += T) {
    const int k = dN(i), y = i - k * N;
    o[i] = buf[k * LS + y];
  }
}

// k_mid: kML consecutive (kz, y) lines of one tensor row; grid
// (ceil(nzk N / kML) (+1), 3, nrhs), block 0 forms alpha when a.pqp.
// PAIR (textbook operator: F_j = q_j u with u = (q . A) / |q|^2): q_y and q_z
// are constant along an x line, so the line q_y A_y + q_z A_z is transformed
// instead of two, and u instead of F_y and F_z, which k_inv forms: two lines a
// row each way for three, and two written.  Nine systems at 96^3 68.7 -> 62.5
// ms, 32^3 3.29 -> 3.09, one at 48^3 2.08 -> 2.02.  The reference's operator
// keeps the order of its sums also for odd N, where it would save as much
// (45^3 3.11 -> 3.04): a solve to a tolerance below the rounding floor, as the
// reference's example deck asks for, takes another number of iterations there.
template <int NC, bool PAIR>
__global__ __launch_bounds__(1024) void k_mid(Grid g, MidArgs a) {
  extern __shared__ cplx lds[];
  constexpr int NL = PAIR ? 2 : 3;  // x lines per (kz, y), as mid_lines
  const int rhs = blockIdx.z, row = blockIdx.y, tid = threadIdx.x, T = blockDim.x;
  int tile = blockIdx.x;
  if (a.cs) {
    if (a.cs[rhs].done) return;
    if (a.pqp) {
      if (tile == 0) {
        if (row == 0 && tid < 64) form_alpha(a, rhs);
        return;
      }
      --tile;
    }
  }
  const int N = edge<NC>(g), LS = N | 1, M = g.nzk * N;
  const int m0 = tile * kML, nm = min(kML, M - m0);
  const Div dN = divN<NC>(g);
  cplx* tw = lds;
  cplx* buf = lds + N;
  load_tw<NC>(tw, a.tw, N);
  cplx* T1 = a.T1 + rhs * a.ts + (long)(3 * row) * N * M + m0;
  auto lb = [&](int l) { return l * LS; };
  if constexpr (PAIR) {
    const long cst = (long)N * M;
    const bool even = (N & 1) == 0;
    // T is a multiple of kML: a thread's points have one line t
    const int t = tid & (kML - 1), kz = dN(m0 + t), y = m0 + t - kz * N;
    const int fy = y <= N / 2 ? y : y - N;
    const double qy = fy, qz = kz;
    for (int i = tid; i < N * kML; i += T) {
      const int x = i / kML;
      if (t < nm) {
        const cplx* s = T1 + (long)x * M + t;
        const cplx A0 = s[0], A1 = s[cst], A2 = s[2 * cst];
        buf[t * LS + x] = A0;
        buf[(kML + t) * LS + x] = cplx{qy * A1.re + qz * A2.re, qy * A1.im + qz * A2.im};
      }
    }
    if (a.dc && m0 == 0 && tid < 64) {  // before the sums are overwritten
      double s1 = 0.0, s2 = 0.0;
      for (int x = tid; x < N; x += 64) {
        s1 += T1[cst + (long)x * M].re;
        s2 += T1[2 * cst + (long)x * M].re;
      }
      s1 = wave_sum(s1);
      s2 = wave_sum(s2);
      if (tid == 0) {
        a.dc[9 * rhs + 3 * row + 1] = s1;
        a.dc[9 * rhs + 3 * row + 2] = s2;
      }
    }
    __syncthreads();
    fft<NC, true, 4>(buf, tw, g, NL * kML, lb, 1);
    if (a.dc && m0 == 0 && tid == 0) a.dc[9 * rhs + 3 * row] = buf[0].re;
    const bool nyq = even && (2 * abs(fy) == N || 2 * kz == N);
    for (int i = tid; i < N * kML; i += T) {
      const int x = i / kML;
      if (t >= nm) continue;
      const int fx = x <= N / 2 ? x : x - N;
      const double qx = fx, qq = qx * qx + qy * qy + qz * qz;
      cplx *b = buf + t * LS + x, *u = b + kML * LS;
      cplx v{0.0, 0.0};
      if (!(nyq || (even && 2 * abs(fx) == N)) && qq > 1e-10) {
        const double s = 1.0 / qq;
        v = cplx{s * (qx * b->re + u->re), s * (qx * b->im + u->im)};
      }
      *b = cplx{qx * v.re, qx * v.im};
      *u = v;
    }
  } else {
    const int tot = 3 * N * kML;
    for (int i = tid; i < tot; i += T) {
      const int t = i & (kML - 1), cx = i / kML, c = dN(cx), x = cx - c * N;
      if (t < nm) buf[(c * kML + t) * LS + x] = T1[(long)cx * M + t];
    }
    __syncthreads();
    fft<NC, true, 4>(buf, tw, g, NL * kML, lb, 1);
    if (a.dc && m0 == 0) {
      if (tid < 3) a.dc[9 * rhs + 3 * row + tid] = buf[tid * kML * LS].re;
      __syncthreads();
    }
    for (int i = tid; i < N * kML; i += T) {
      const int t = i & (kML - 1), x = i / kML;
      if (t >= nm) continue;
      const int kz = dN(m0 + t), y = m0 + t - kz * N;
      cplx* b = buf + t * LS + x;
      const cplx A[3] = {b[0], b[kML * LS], b[2 * kML * LS]};
      cplx o[3];
      project_row(N, g.gamma_mode, x, y, kz, A, o);
      b[0] = o[0];
      b[kML * LS] = o[1];
      b[2 * kML * LS] = o[2];
    }
  }
  __syncthreads();
  fft<NC, false, 4>(buf, tw, g, NL * kML, lb, 1);
  for (int i = tid; i < NL * N * kML; i += T) {
    const int t = i & (kML - 1), cx = i / kML, c = dN(cx), x = cx - c * N;
    if (t < nm) T1[(long)cx * M + t] = buf[(c * kML + t) * LS + x];
  }
}

// k_inv: block = (x, component, right-hand side); grid (N, 9, nrhs).  With
// g.pair component 3 i + j > 3 i is q_j u_i, u_i in place 3 i + 1.
template <int NC, int ME, int MODE>
__global__ __launch_bounds__(1024) void k_inv(Grid g, InvArgs a) {
  extern __shared__ cplx lds[];
  const int rhs = blockIdx.z, c = blockIdx.y, x = blockIdx.x, tid = threadIdx.x, T = blockDim.x;
  if (a.cs && a.cs[rhs].done) return;
  const int N = edge<NC>(g), LS = N | 1, NN = N * N, nzk = g.nzk, M = nzk * N, LP = (N + 1) >> 1;
  const Div dN = divN<NC>(g);
  cplx* tw = lds;
  cplx* buf = lds + N;
  load_tw<NC>(tw, a.tw, N);
  const int j3 = g.pair ? c % 3 : 0;
  const cplx* s = a.T1 + rhs * a.ts + ((long)(c - (j3 == 2)) * N + x) * M;
  for (int i = tid; i < M; i += T) {
    const int k = dN(i), y = i - k * N;
    cplx v = s[i];
    if (j3 > 0) {
      const double q = j3 == 2 ? k : y <= N / 2 ? y : y - N;
      v = cplx{q * v.re, q * v.im};
    }
    buf[k * LS + y] = v;
  }
  // the vector values of this thread's first points travel meanwhile
  const long e0 = c * g.V + (long)x * NN;
  Fetched f;
#pragma unroll
  for (int j = 0; j < 2; ++j) fetch<MODE>(a, rhs, e0 + tid + j * T, tid + j * T < NN, j, f);
  __syncthreads();
  auto lb = [&](int l) { return l * LS; };
  fft<NC, false, ME>(buf, tw, g, nzk, lb, 1);
  {
    constexpr int MQ = ME / 2 + 1;
    cplx A[MQ], B[MQ];
    const Div dLP(LP);
#pragma unroll
    for (int u = 0; u < MQ; ++u) {
      const int q = tid + u * T;
      if (q < LP * nzk) {
        const int k = dLP(q), m = q - k * LP;
        const cplx* b = buf + k * LS + 2 * m;
        A[u] = b[0];
        B[u] = 2 * m + 1 < N ? b[1] : cplx{0.0, 0.0};
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < MQ; ++u) {
      const int q = tid + u * T;
      if (q < LP * nzk) {
        const int k = dLP(q), m = q - k * LP;
        pack(buf + m * LS, k, N, g.NZ, A[u], B[u]);
      }
    }
    if (nzk < g.NZ)  // the removed Nyquist plane
      for (int m = tid; m < LP; m += T) buf[m * LS + N / 2] = cplx{0.0, 0.0};
    __syncthreads();
  }
  fft<NC, false, ME>(buf, tw, g, LP, lb, 1);
  store_lines<NC, MODE>(g, a, rhs, e0, NN, buf, f, a.part + ((long)rhs * 9 + c) * N + x);
}

// ------------------------------------------------------ CG update of p.q
// x += alpha p, r -= alpha q with alpha = rr / p.q from the inverse pass's
// partial sums (every block forms it, the first keeps it), and the r.r
// partial sums; grid (blocks, nrhs).  For the reference's operator, where p.q
// is not known before q.
constexpr int kStepRun = 2048;  // elements per block, more above 1024 blocks
struct StepArgs {
  Ptr p, q, x, r;
  const double* pqp;
  int npq;
  CGScalars* cs;
  double* rrp;
};
static int step_blocks(long V) { return (int)std::min(1024L, (9 * V + kStepRun - 1) / kStepRun); }
__global__ __launch_bounds__(256) void k_step(long n, StepArgs a) {
  __shared__ double s_al, wsum[4];
  const int rhs = blockIdx.y, tid = threadIdx.x;
  if (a.cs[rhs].done) return;
  if (tid < 64) {
    const double* part = a.pqp + (long)rhs * a.npq;
    double acc = 0.0;
    for (int i = tid; i < a.npq; i += 64) acc += part[i];
    acc = wave_sum(acc);
    if (tid == 0) {
      s_al = a.cs[rhs].rr / acc;
      if (blockIdx.x == 0) a.cs[rhs].alpha = s_al;
    }
  }
  __syncthreads();
  const double al = s_al;
  const long chunk = (n + gridDim.x - 1) / gridDim.x;
  const long lo = blockIdx.x * chunk, hi = min(n, lo + chunk);
  const double *P = a.p.p[rhs], *Q = a.q.p[rhs];
  double *X = a.x.p[rhs], *R = a.r.p[rhs];
  double acc = 0.0;
  for (long i = lo + tid; i < hi; i += 4 * 256) {
    double pv[4], qv[4], xv[4], rv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const long e = i + u * 256;
      const bool in = e < hi;
      qv[u] = in ? Q[e] : 0.0;
      rv[u] = in ? R[e] : 0.0;
      pv[u] = in && X ? P[e] : 0.0;
      xv[u] = in && X ? X[e] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const long e = i + u * 256;
      if (e >= hi) break;
      if (X) X[e] = xv[u] + al * pv[u];
      const double rn = rv[u] - al * qv[u];
      R[e] = rn;
      acc += rn * rn;
    }
  }
  acc = wave_sum(acc);
  if ((tid & 63) == 0) wsum[tid >> 6] = acc;
  __syncthreads();
  if (tid == 0) a.rrp[(long)rhs * gridDim.x + blockIdx.x] = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
}

// ---------------------------------------------------- edges above kSlabN
// k_zf: TL lines, three components, one right-hand side; T1[c][kz][L]
template <bool HASK, bool DIR>
__global__ __launch_bounds__(256) void k_zf(Grid g, FwdArgs a) {
  constexpr int CPB = 3;
  extern __shared__ cplx lds[];
  const Where w = where<CPB>(a.nrhs);
  if (w.tile >= g.nzb) return;
  const int N = g.N, LS = N | 1;
  const int L0 = w.tile * g.TL, nl = min(g.TL, g.NN - L0), LP = (nl + 1) >> 1;
  cplx* tw = lds;
  cplx* buf = lds + N;
  Point<HASK, DIR, CPB> pt;
  load_tw<kAnyRadix>(tw, a.tw, N);
  double beta = 0.0;
  if constexpr (DIR) {
    if (cg_begin(a, w.rhs, w.tile == 0 && w.c0 == 0, beta)) return;
  }
  load_lines<kAnyRadix, HASK, DIR, CPB, false>(
      g, a, w.rhs, w.c0, (long)L0 * N, nl * N, nl, beta, buf,
      DIR && a.pqp ? a.pqp + ((long)w.rhs * 9 + w.c0) * g.nzb + w.tile : nullptr, g.nzb,
      pt);
  fft<kAnyRadix, true, kMaxE>(buf, tw, g, CPB * LP, [&](int l) { return l * LS; }, 1);
  const Div dLP(LP);
#pragma unroll
  for (int j = 0; j < CPB; ++j) {
    cplx* T1 = a.T1 + w.rhs * a.ts + (long)(w.c0 + j) * g.NZ * g.NN + L0;
    for (int q = threadIdx.x; q < LP * g.nzk; q += 256) {
      const int k = dLP(q), m = q - k * LP;
      cplx A, B;
      unpack(buf + (j * LP + m) * LS, k, N, A, B);
      cplx* o = T1 + (long)k * g.NN + 2 * m;
      o[0] = A;
      if (2 * m + 1 < nl) o[1] = B;
    }
  }
}

constexpr int kTX = 8;  // x lines per block of k_y: 128-byte transposed runs

// FWD: T1[c][kz][x][y] -> T2[c][kz][y][x]; inverse: T2 -> T1.
// grid (ceil(N / kTX), nzk, 9 nrhs)
template <bool FWD>
__global__ __launch_bounds__(256) void k_y(Grid g, MidArgs a) {
  extern __shared__ cplx lds[];
  const int rhs = blockIdx.z / 9, c = blockIdx.z - 9 * rhs, kz = blockIdx.y;
  if (a.cs && a.cs[rhs].done) return;
  const int N = g.N, LS = N | 1, x0 = blockIdx.x * kTX, nx = min(kTX, N - x0);
  cplx* tw = lds;
  cplx* buf = lds + N;
  load_tw<kAnyRadix>(tw, a.tw, N);
  const long plane = rhs * a.ts + ((long)c * g.NZ + kz) * g.NN;
  const Div dnx(nx);
  if constexpr (FWD) {
    for (int i = threadIdx.x; i < nx * N; i += 256) {
      const int t = g.dN(i), y = i - t * N;
      buf[t * LS + y] = a.T1[plane + (long)x0 * N + i];
    }
  } else {
    for (int i = threadIdx.x; i < nx * N; i += 256) {
      const int y = dnx(i), t = i - y * nx;
      buf[t * LS + y] = a.T2[plane + (long)y * N + x0 + t];
    }
  }
  __syncthreads();
  fft<kAnyRadix, FWD, kMaxE>(buf, tw, g, nx, [&](int l) { return l * LS; }, 1);
  if constexpr (FWD) {
    for (int i = threadIdx.x; i < nx * N; i += 256) {
      const int y = dnx(i), t = i - y * nx;
      a.T2[plane + (long)y * N + x0 + t] = buf[t * LS + y];
    }
  } else {
    for (int i = threadIdx.x; i < nx * N; i += 256) {
      const int t = g.dN(i), y = i - t * N;
      a.T1[plane + (long)x0 * N + i] = buf[t * LS + y];
    }
  }
}

// y lines per block of k_x: 3 YB lines of length N, kMaxE elements a thread
__host__ __device__ inline int x_lines(int N) {
  const int t = kMaxE * 256 / (3 * N);
  return t < 1 ? 1 : t > 8 ? 8 : t;
}

// x transforms, projection and inverse of one tensor row, in place in T2.
// grid (ceil(N / YB), nzk, 3 nrhs)
__global__ __launch_bounds__(256) void k_x(Grid g, MidArgs a) {
  extern __shared__ cplx lds[];
  const int rhs = blockIdx.z / 3, row = blockIdx.z - 3 * rhs, kz = blockIdx.y;
  if (a.cs && a.cs[rhs].done) return;
  const int N = g.N, LS = N | 1, YB = x_lines(N), y0 = blockIdx.x * YB, ny = min(YB, N - y0);
  cplx* tw = lds;
  cplx* buf = lds + N;
  load_tw<kAnyRadix>(tw, a.tw, N);
  const long cst = (long)g.NZ * g.NN;
  cplx* T2 = a.T2 + rhs * a.ts + ((long)(3 * row) * g.NZ + kz) * g.NN + (long)y0 * N;
#pragma unroll
  for (int c = 0; c < 3; ++c)
    for (int i = threadIdx.x; i < ny * N; i += 256) {
      const int t = g.dN(i), x = i - t * N;
      buf[(c * ny + t) * LS + x] = T2[c * cst + i];
    }
  __syncthreads();
  auto lb = [&](int l) { return l * LS; };
  fft<kAnyRadix, true, kMaxE>(buf, tw, g, 3 * ny, lb, 1);
  if (a.dc && kz == 0 && y0 == 0) {
    if (threadIdx.x < 3) a.dc[9 * rhs + 3 * row + threadIdx.x] = buf[threadIdx.x * ny * LS].re;
    __syncthreads();
  }
  for (int i = threadIdx.x; i < ny * N; i += 256) {
    const int t = g.dN(i), x = i - t * N;
    cplx* b = buf + t * LS + x;
    const cplx A[3] = {b[0], b[ny * LS], b[2 * ny * LS]};
    cplx o[3];
    project_row(N, g.gamma_mode, x, y0 + t, kz, A, o);
    b[0] = o[0];
    b[ny * LS] = o[1];
    b[2 * ny * LS] = o[2];
  }
  __syncthreads();
  fft<kAnyRadix, false, kMaxE>(buf, tw, g, 3 * ny, lb, 1);
#pragma unroll
  for (int c = 0; c < 3; ++c)
    for (int i = threadIdx.x; i < ny * N; i += 256) {
      const int t = g.dN(i), x = i - t * N;
      T2[c * cst + i] = buf[(c * ny + t) * LS + x];
    }
}

// grid (nzb, 9, nrhs)
template <int MODE>
__global__ __launch_bounds__(256) void k_zi(Grid g, InvArgs a) {
  extern __shared__ cplx lds[];
  const int rhs = blockIdx.z, c = blockIdx.y, tile = blockIdx.x, tid = threadIdx.x;
  if (a.cs && a.cs[rhs].done) return;
  const int N = g.N, LS = N | 1;
  const int L0 = tile * g.TL, nl = min(g.TL, g.NN - L0), npts = nl * N, LP = (nl + 1) >> 1;
  const long e0 = (long)L0 * N + c * g.V;
  cplx* tw = lds;
  cplx* buf = lds + N;
  load_tw<kAnyRadix>(tw, a.tw, N);
  const cplx* T1 = a.T1 + rhs * a.ts + (long)c * g.NZ * g.NN + L0;
  const Div dLP(LP);
  for (int q = tid; q < LP * g.nzk; q += 256) {
    const int k = dLP(q), m = q - k * LP;
    const cplx* s = T1 + (long)k * g.NN + 2 * m;
    pack(buf + m * LS, k, N, g.NZ, s[0], 2 * m + 1 < nl ? s[1] : cplx{0.0, 0.0});
  }
  if (g.nzk < g.NZ)  // the removed Nyquist plane
    for (int m = tid; m < LP; m += 256) buf[m * LS + N / 2] = cplx{0.0, 0.0};
  Fetched f;
#pragma unroll
  for (int j = 0; j < 2; ++j) fetch<MODE>(a, rhs, e0 + tid + j * 256, tid + j * 256 < npts, j, f);
  __syncthreads();
  fft<kAnyRadix, false, 4>(buf, tw, g, LP, [&](int l) { return l * LS; }, 1);
  store_lines<kAnyRadix, MODE>(g, a, rhs, e0, npts, buf, f,
                       a.part + ((long)rhs * 9 + c) * g.nzb + tile);
}

// ------------------------------------------------------------------- host
// fewest radices whose product is N, then the smallest sum
static void plan(int n, int* best, int& nb, int* cur, int nc, int from) {
  static const int R[11] = {13, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};
  if (n == 1) {
    int sb = 0, sc = 0;
    for (int i = 0; i < nb; ++i) sb += best[i];
    for (int i = 0; i < nc; ++i) sc += cur[i];
    if (nb == 0 || nc < nb || (nc == nb && sc < sb)) {
      nb = nc;
      for (int i = 0; i < nc; ++i) best[i] = cur[i];
    }
    return;
  }
  if (nc == kMaxSt) return;
  for (int i = from; i < 11; ++i)
    if (n % R[i] == 0) {
      cur[nc] = R[i];
      plan(n / R[i], best, nb, cur, nc + 1, i);
    }
}

// x lines per (kz, y) and tensor row (see k_mid)
static int mid_lines(int N, int gamma_mode) { return N <= kSlabN && gamma_mode == 1 ? 2 : 3; }

static Grid make_grid(const SpecGeom& s) {
  Grid g;
  g.N = s.N;
  g.NZ = s.Nz;
  g.nzk = s.gamma_mode == 1 && s.N % 2 == 0 ? s.Nz - 1 : s.Nz;
  g.NN = s.N * s.N;
  g.gamma_mode = s.gamma_mode;
  g.pair = mid_lines(s.N, s.gamma_mode) == 2;
  g.V = s.V;
  g.S1 = s.S1;
  g.dN = Div(s.N);
  // above kSlabN: at most 512 complex elements of a component per block, but
  // two lines
  const int lp = 512 / s.N;
  g.TL = 2 * (lp < 1 ? 1 : lp);
  g.nzb = s.N <= kSlabN ? s.N : (g.NN + g.TL - 1) / g.TL;
  int cur[kMaxSt], nb = 0;
  plan(s.N, g.rad, nb, cur, 0, 0);
  g.nst = nb;
  int ns = 1;
  for (int i = 0; i < nb; ++i) {
    g.dNs[i] = Div(ns);
    ns *= g.rad[i];
  }
  return g;
}

static int up64(int n) { return (n + 63) / 64 * 64; }
// Threads of the slab kernels.  The transforms need a quarter of the half
// spectrum's elements (candidate kFew); a lone system's blocks do not fill
// the chip, and each thread waits for its voxels one after the other, so up
// to 512 threads take one each (solve 32^3 1.33 -> 1.20 ms, 45^3 3.21 -> 3.14;
// 768 are slower: one block a CU).  Several systems with the contraction in
// the kernel keep the few: their blocks fill the chip and 384 or 512 threads
// are fewer waves (nine at 32^3: 3.3 ms with 192 threads, 3.9 with 512).
constexpr int kFew = -1;
static int slab_threads(int N, int i) {
  const int t = std::min(1024, up64((N * (N / 2 + 1) + 3) / 4));
  return i == kFew ? t : i == 1 ? std::min(1024, 2 * t) : std::max(t, std::min(512, up64(N * N)));
}
// of k_mid, for its nl lines of N points per (kz, y)
static int mid_threads(int N, int nl, int i) {
  return up64(nl * kML * N / (N < 32 || i == 1 ? 2 : 4)) * (N < 32 && i == 1 ? 2 : 1);
}
// elements per thread the runtime plans allow for: four up to edge 88
constexpr int kE4N = 88;  // 88 * 45 <= 4 * 1024

// more than 64 KiB of dynamic LDS has to be asked for
template <class K>
static void allow_lds(K kernel, size_t bytes) {
  if (bytes > 65536)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}
static size_t lds_slab(int N) { return ((size_t)N + (size_t)(N / 2 + 1) * (N | 1)) * sizeof(cplx); }
static size_t lds_lines(int N, int lines) {
  return ((size_t)N + (size_t)lines * (N | 1)) * sizeof(cplx);
}

// The first point's operands ahead of the rest need some 40 registers more:
// for a lone system, where a block's own latency counts (16^3 0.75 -> 0.69 ms);
// several systems' blocks do better with more waves a SIMD (nine at 32^3 3.28
// against 3.38), and radices 11 and 13 leave no registers for it.
template <int NC, int ME, bool HASK, bool DIR>
static void fwd_slab(const Grid& g, const FwdArgs& a, int threads, hipStream_t s) {
  constexpr bool ahead = HASK && NC != kAnyRadix;
  // several systems have the contraction in this kernel below edge 40 only
  constexpr bool several = !ahead || (DIR && NC != 48 && ME != kMaxE);
  auto k = k_fwd<NC, ME, HASK, DIR, !several>;
  if constexpr (ahead && several) {
    if (a.nrhs == 1) k = k_fwd<NC, ME, HASK, DIR, true>;
  }
  const size_t lds = lds_slab(g.N);
  allow_lds(k, lds);
  k<<<8 * ((g.N + 7) / 8) * 9 * a.nrhs, threads, lds, s>>>(g, a);
}

template <int NC, bool HASK, bool DIR>
static void forward(const Grid& g, const FwdArgs& a, int cand, hipStream_t s) {
  const int t = slab_threads(g.N, cand);
  if constexpr (NC == kAnyRadix) {
    if (g.N > kSlabN) {
      k_zf<HASK, DIR><<<8 * ((g.nzb + 7) / 8) * 3 * a.nrhs, 256,
                        lds_lines(g.N, 3 * (g.TL / 2)), s>>>(g, a);
      return;
    }
  }
  if constexpr (NC <= 0) {
    if (g.N > kE4N) return fwd_slab<NC, kMaxE, HASK, DIR>(g, a, t, s);
  }
  fwd_slab<NC, NC == 96 ? 5 : 4, HASK, DIR>(g, a, t, s);
}

// Edges of fft_pencil.hip: only tangent_homo's systems come here, with the
// textbook operator and K4:p formed by a launch of its own
constexpr bool tangent_only(int NC) { return NC == 64 || NC == 96; }

template <int NC>
static void middle(const Grid& g, const MidArgs& a, int nrhs, int cand, hipStream_t s) {
  if (NC != kAnyRadix || g.N <= kSlabN) {
    const int tiles = (g.nzk * g.N + kML - 1) / kML;
    const dim3 grid(tiles + (a.pqp ? 1 : 0), 3, nrhs);
    const int nl = mid_lines(g.N, g.gamma_mode);
    auto k = k_mid<NC, true>;
    if constexpr (!tangent_only(NC))
      if (!g.pair) k = k_mid<NC, false>;
    k<<<grid, mid_threads(g.N, nl, cand), lds_lines(g.N, nl * kML), s>>>(g, a);
  } else if constexpr (NC == kAnyRadix) {
    const int yb = x_lines(g.N);
    if (a.pqp) launch_cg_alpha(a.pqp, a.npq, a.cs, s, nrhs, a.npq);
    const dim3 gy((g.N + kTX - 1) / kTX, g.nzk, 9 * nrhs);
    k_y<true><<<gy, 256, lds_lines(g.N, kTX), s>>>(g, a);
    k_x<<<dim3((g.N + yb - 1) / yb, g.nzk, 3 * nrhs), 256, lds_lines(g.N, 3 * yb), s>>>(g, a);
    k_y<false><<<gy, 256, lds_lines(g.N, kTX), s>>>(g, a);
  }
}

template <int NC, int ME, int MODE>
static void inv_slab(const Grid& g, const InvArgs& a, int nrhs, int threads, hipStream_t s) {
  auto k = k_inv<NC, ME, MODE>;
  const size_t lds = lds_slab(g.N);
  allow_lds(k, lds);
  k<<<dim3(g.N, 9, nrhs), threads, lds, s>>>(g, a);
}
template <int NC, int MODE>
static void inverse(const Grid& g, const InvArgs& a, int nrhs, int cand, hipStream_t s) {
  const int t = slab_threads(g.N, cand);
  if constexpr (NC == kAnyRadix) {
    if (g.N > kSlabN) {
      k_zi<MODE><<<dim3(g.nzb, 9, nrhs), 256, lds_lines(g.N, g.TL / 2), s>>>(g, a);
      return;
    }
  }
  if constexpr (NC <= 0) {
    if (g.N > kE4N) return inv_slab<NC, kMaxE, MODE>(g, a, nrhs, t, s);
  }
  inv_slab<NC, NC == 96 ? 5 : 4, MODE>(g, a, nrhs, t, s);
}

// spectrum entries per right-hand side; above kSlabN T2 follows T1
static long spec_stride(const Grid& g) { return (g.N <= kSlabN ? 9 : 18) * g.S1; }

struct Args {
  FwdArgs f{};
  MidArgs m{};
  InvArgs i{};
  Args(const Grid& g, const double* K4, cplx* spec, const cplx* tw, int nrhs) {
    f.fs = g.V;
    f.K4 = K4;
    f.T1 = spec;
    f.nrhs = nrhs;
    m.T1 = spec;
    m.T2 = spec + 9 * g.S1;
    i.T1 = spec;
    f.ts = m.ts = i.ts = spec_stride(g);
    f.tw = m.tw = i.tw = tw;
  }
};

template <int NC>
static void run_gkdf(const SpecGeom& sg, const double* F, const double* K4, double* out,
                     cplx* spec, const cplx* tw, hipStream_t s) {
  const Grid g = make_grid(sg);
  Args a(g, K4, spec, tw, 1);
  a.f.F.p[0] = const_cast<double*>(F);
  a.i.out.p[0] = out;
  if (K4)
    forward<NC, true, false>(g, a.f, sg.tune.a, s);
  else
    forward<NC, false, false>(g, a.f, sg.tune.a0, s);
  middle<NC>(g, a.m, 1, sg.tune.c, s);
  inverse<NC, 0>(g, a.i, 1, sg.tune.b, s);
}

// Shape of the x pass in a solve.  At 64 and 96 the context's shapes are those
// of fft_pencil.hip's passes, so the default.  (The forward pass of several
// systems always takes its default: the best for one system can be the worse
// for nine, at 48^3 5.87 instead of 5.49 ms a tangent.)
static int mid_shape(const SpecGeom& sg) { return gkdf_grid_edge(sg.N) ? sg.tune.c : 0; }

template <int NC>
static void run_cg(const SpecGeom& sg, const GridCG& c, int part, hipStream_t s) {
  const Grid g = make_grid(sg);
  const int np = 9 * g.nzb;
  const bool plain = c.out[0] != nullptr;  // p.q from the inverse pass
  const int ct = c.nrhs > 1 && !c.q[0] ? kFew : 0;
  Args a(g, c.K4, c.spec, c.tw, c.nrhs);
  for (int k = 0; k < c.nrhs; ++k) {
    a.f.F.p[k] = c.p_old[k];
    a.f.pn.p[k] = a.i.pd.p[k] = c.p_new[k];
    a.f.r.p[k] = a.i.r.p[k] = c.r[k];
    a.i.x.p[k] = c.x[k];
    a.i.out.p[k] = c.out[k];
  }
  a.f.old = c.cs_old;
  a.f.nw = a.m.cs = c.cs_new;
  a.i.cs = c.cs_new;
  a.f.rrp = c.rr;
  a.f.nrr = plain ? step_blocks(g.V) : np;
  a.f.chk = c.chk;
  a.f.dc = a.m.dc = c.dc;
  a.f.m = c.m;
  a.f.scale = c.scale;
  a.f.pqp = plain ? nullptr : c.pq;
  a.m.pqp = a.f.pqp;
  a.m.npq = c.q[0] ? c.npq : np;
  a.i.part = plain ? c.pq : c.rr;
  if (part == 0) {
    if (c.q[0]) {
      for (int k = 0; k < c.nrhs; ++k) a.f.F.p[k] = const_cast<double*>(c.q[k]);
      forward<NC, false, false>(g, a.f, 0, s);
    } else if constexpr (!tangent_only(NC)) {
      forward<NC, true, true>(g, a.f, ct, s);
    }
    middle<NC>(g, a.m, c.nrhs, mid_shape(sg), s);
  } else if (part == 1) {
    if (!plain)
      inverse<NC, 2>(g, a.i, c.nrhs, ct, s);
    else if constexpr (!tangent_only(NC))
      inverse<NC, 1>(g, a.i, c.nrhs, ct, s);
  } else if (plain) {
    StepArgs t{};
    t.p = a.i.pd;
    t.q = a.i.out;
    t.x = a.i.x;
    t.r = a.i.r;
    t.pqp = c.pq;
    t.npq = np;
    t.cs = c.cs_new;
    t.rrp = c.rr;
    k_step<<<dim3(a.f.nrr, c.nrhs), 256, 0, s>>>(9 * g.V, t);
  }
}

template <int NC>
static void run_homo_rhs(const SpecGeom& sg, const double* K4, int i0, int n, double* const* r,
                         cplx* spec, const cplx* tw, double* rr, hipStream_t s) {
  const Grid g = make_grid(sg);
  Args a(g, nullptr, spec, tw, n);
  a.f.fs = 9 * g.V;  // column i of K4: rows i, 9 + i, ...
  a.i.part = rr;
  for (int k = 0; k < n; ++k) {
    a.f.F.p[k] = const_cast<double*>(K4) + (long)(i0 + k) * g.V;
    a.i.out.p[k] = r[k];
  }
  forward<NC, false, false>(g, a.f, 0, s);
  middle<NC>(g, a.m, n, mid_shape(sg), s);
  inverse<NC, 3>(g, a.i, n, 0, s);
}

template <int NC>
static void run_pass(const SpecGeom& sg, int pass, int v, const double* F, const double* K4,
                     cplx* spec, const cplx* tw, hipStream_t s) {
  const Grid g = make_grid(sg);
  Args a(g, K4, spec, tw, 1);
  a.f.F.p[0] = const_cast<double*>(F);
  // the inverse pass writes behind the spectrum
  a.i.out.p[0] = reinterpret_cast<double*>(spec + 9 * g.S1);
  switch (pass) {
    case 0: forward<NC, true, false>(g, a.f, v, s); break;
    case 1: forward<NC, false, false>(g, a.f, v, s); break;
    case 2: inverse<NC, 0>(g, a.i, 1, v, s); break;
    default: middle<NC>(g, a.m, 1, v, s); break;
  }
}

}  // namespace gp

// ---- interface (kernels.h)
bool gkdf_slab_edge(int N) { return N <= gp::kSlabN; }
bool gkdf_grid_edge(int N) { return !(N == 64 || N == 96 || N == 128 || N == 256); }

#define CPFFT_EDGE(call, large)     \
  switch (g.N) {                    \
    default:                        \
      if (gp::smooth(g.N))          \
        gp::call<gp::kSmooth> CPFFT_ARGS; \
      else                          \
        gp::call<gp::kAnyRadix> CPFFT_ARGS; \
      break;                        \
    case 16: gp::call<16> CPFFT_ARGS; break; \
    case 32: gp::call<32> CPFFT_ARGS; break; \
    case 48: gp::call<48> CPFFT_ARGS; break; \
    large                           \
  }
// with the edges of tangent_only
#define CPFFT_EDGE_ALL(call)                         \
  CPFFT_EDGE(call, case 64: gp::call<64> CPFFT_ARGS; break; \
             case 96: gp::call<96> CPFFT_ARGS; break;)

void launch_cg_grid(const SpecGeom& g, const GridCG& c, int part, hipStream_t s) {
#define CPFFT_ARGS (g, c, part, s)
  CPFFT_EDGE_ALL(run_cg)
#undef CPFFT_ARGS
}

void launch_homo_rhs_grid(const SpecGeom& g, const double* K4, int i0, int n, double* const* r,
                          cplx* spec, const cplx* tw, double* rr, hipStream_t s) {
#define CPFFT_ARGS (g, K4, i0, n, r, spec, tw, rr, s)
  CPFFT_EDGE_ALL(run_homo_rhs)
#undef CPFFT_ARGS
}

void launch_gkdf_grid(const SpecGeom& g, const double* F, const double* K4, double* out,
                      cplx* spec, const cplx* tw, hipStream_t s) {
#define CPFFT_ARGS (g, F, K4, out, spec, tw, s)
  CPFFT_EDGE(run_gkdf, )
#undef CPFFT_ARGS
}
int grid_parts(int N) {
  SpecGeom s{};
  s.N = N;
  s.Nz = N / 2 + 1;
  return 9 * gp::make_grid(s).nzb;
}
int grid_rr_parts(int N, bool projection) {
  return projection ? grid_parts(N) : gp::step_blocks((long)N * N * N);
}
// The test inside the next iteration's first kernel costs every block the
// sum of these values (9 N up to kSlabN); above, a launch of its own is cheaper.
bool grid_fused_check(int N) { return grid_parts(N) <= 2304; }
long grid_spec_len(const SpecGeom& g) { return gp::spec_stride(gp::make_grid(g)); }

int grid_candidate(int N, int gamma_mode, int pass, int v) {
  if (N != 16 && N != 32 && N != 48) return 0;
  if (v < 0 || v > 1) return 0;
  return (pass == 3 ? gp::mid_threads(N, gp::mid_lines(N, gamma_mode), v) : gp::slab_threads(N, v)) / 64;
}
void launch_grid_pass(const SpecGeom& g, int pass, int v, const double* F, const double* K4,
                      cplx* spec, const cplx* tw, hipStream_t s) {
#define CPFFT_ARGS (g, pass, v, F, K4, spec, tw, s)
  switch (g.N) {
    case 16: gp::run_pass<16> CPFFT_ARGS; break;
    case 32: gp::run_pass<32> CPFFT_ARGS; break;
    default: gp::run_pass<48> CPFFT_ARGS; break;
  }
#undef CPFFT_ARGS
}

}  // namespace cpfft
