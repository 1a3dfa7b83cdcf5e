// cpfft_kernels.hip -- CDNA4 (gfx950) kernels of the CPFFT solver step.
//
//  * BLAS-1 and reductions for CG, Newton norms and volume averages
//    (FFT_nr3.f:85-147, tangent_homo.f:62-66): deterministic two-stage
//    block reductions (fixed order, no floating-point atomics).
//  * drive_eps_sig (src/drive_eps_sig.f:16-339): one thread per voxel,
//    body in mm10_core.h.
#include <type_traits>

#include "../../include/cpfft.h"
#include "green.h"
#include "kernels.h"

namespace cpfft {

static constexpr int kBlock = 256;

// ------------------------------------------------------------- operator
const char* make_spec_geom(int N, int gamma_mode, SpecGeom& g) {
  g = SpecGeom{};
  g.N = N;
  g.Nz = N / 2 + 1;
  g.V = (long)N * N * N;
  g.S1 = (long)N * N * g.Nz;
  g.gamma_mode = gamma_mode;
  if (gkdf_grid_edge(N)) {
    if (N > 227) return "no grid edge above 227 but 256 is served";
    int m = N;
    for (int p : {2, 3, 5, 7, 11})
      while (m % p == 0) m /= p;
    if (m > 13) return "N has a prime factor above 13, or 13 twice";
  }
  return nullptr;
}

void launch_gkdf(const SpecGeom& g, const double* F, const double* K4, double* out, cplx* spec,
                 const cplx* tw, hipStream_t s) {
  if (gkdf_grid_edge(g.N))
    launch_gkdf_grid(g, F, K4, out, spec, tw, s);
  else
    launch_gkdf_pencil(g, F, K4, out, spec, tw, s);
}

// ------------------------------------------------------------ reductions
static constexpr int kRedBlocks = 1024;

int reduce_partials_count(long) { return kRedBlocks * 9; }

// halving-tree sum over a block of kBlock threads (tree_sum0), valid in
// thread 0; the closing barrier lets a caller reuse sh in a loop
__device__ inline double block_sum(double v, double* sh) {
  const double r = tree_sum0<kBlock>(v, sh);
  __syncthreads();
  return r;
}

// fixed partition: block b handles the contiguous range [b*chunk, (b+1)*chunk)
__global__ __launch_bounds__(kBlock) void k_dot_part(const double* __restrict__ x,
                                                     const double* __restrict__ y, long n,
                                                     double* __restrict__ part) {
  __shared__ double sh[kBlock];
  long chunk = (n + gridDim.x - 1) / gridDim.x;
  long a = blockIdx.x * chunk, b = min(n, a + chunk);
  double acc = 0.0;
  for (long i = a + threadIdx.x; i < b; i += blockDim.x) acc += x[i] * y[i];
  double s = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ __launch_bounds__(kBlock) void k_sum_parts(const double* __restrict__ part, int np,
                                                      int nres, double* __restrict__ out) {
  __shared__ double sh[kBlock];
  for (int r = 0; r < nres; ++r) {
    double acc = 0.0;
    for (int i = threadIdx.x; i < np; i += blockDim.x) acc += part[r * np + i];
    double s = block_sum(acc, sh);
    if (threadIdx.x == 0) out[r] = s;
  }
}

void launch_dot(const double* x, const double* y, long n, double* partials, double* d_out,
                hipStream_t s) {
  k_dot_part<<<kRedBlocks, kBlock, 0, s>>>(x, y, n, partials);
  k_sum_parts<<<1, kBlock, 0, s>>>(partials, kRedBlocks, 1, d_out);
}

// mean of each of the 9 components: partial sums per component
__global__ __launch_bounds__(kBlock) void k_sum9_part(const double* __restrict__ x, long V,
                                                      double* __restrict__ part) {
  __shared__ double sh[kBlock];
  long chunk = (V + gridDim.x - 1) / gridDim.x;
  long a = blockIdx.x * chunk, b = min(V, a + chunk);
  for (int c = 0; c < 9; ++c) {
    double acc = 0.0;
    for (long i = a + threadIdx.x; i < b; i += blockDim.x) acc += x[c * V + i];
    double s = block_sum(acc, sh);
    if (threadIdx.x == 0) part[c * gridDim.x + blockIdx.x] = s;
  }
}

__global__ void k_scale9(double* out, double sc) {
  if (threadIdx.x < 9) out[threadIdx.x] *= sc;
}

void launch_mean9(const double* x, long V, double* partials, double* d_out, hipStream_t s) {
  k_sum9_part<<<kRedBlocks, kBlock, 0, s>>>(x, V, partials);
  k_sum_parts<<<1, kBlock, 0, s>>>(partials, kRedBlocks, 9, d_out);
  k_scale9<<<1, 64, 0, s>>>(d_out, 1.0 / (double)V);
}

// tangent_homo's end: means of the 81 rows of K4, kMeanBlocks partial sums
// a row, then one wave a row
static constexpr int kMeanBlocks = 64;
__global__ __launch_bounds__(kBlock) void k_sum81_part(const double* __restrict__ K4, long V,
                                                       double* __restrict__ part) {
  __shared__ double sh[kBlock];
  const double* x = K4 + blockIdx.y * V;
  const long chunk = (V + gridDim.x - 1) / gridDim.x;
  const long a = blockIdx.x * chunk, b = min(V, a + chunk);
  double acc = 0.0;
  for (long i = a + threadIdx.x; i < b; i += kBlock) acc += __builtin_nontemporal_load(x + i);
  const double s = tree_sum0<kBlock>(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.y * kMeanBlocks + blockIdx.x] = s;
}
__global__ __launch_bounds__(64) void k_mean81(const double* __restrict__ part, double sc,
                                               const double* __restrict__ m,
                                               double* __restrict__ out) {
  const int row = blockIdx.x, j = row / 9, i = row - 9 * j;
  const double s = tree_sum0<64>(part[row * kMeanBlocks + threadIdx.x], nullptr);
  if (threadIdx.x == 0) out[row] = s * sc + m[9 * i + j];
}
void launch_mean81(const double* K4, long V, const double* m, double* partials, double* out,
                   hipStream_t s) {
  static_assert(81 * kMeanBlocks <= 9 * kRedBlocks, "partial sums buffer");
  k_sum81_part<<<dim3(kMeanBlocks, 81), kBlock, 0, s>>>(K4, V, partials);
  k_mean81<<<81, 64, 0, s>>>(partials, 1.0 / (double)V, m, out);
}

// --------------------------------------------------------------- BLAS-1
__global__ void k_axpy(long n, double a, const double* __restrict__ x, double* __restrict__ y) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    y[i] = y[i] + a * x[i];
}
__global__ void k_scal(long n, double a, double* __restrict__ x) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    x[i] = a * x[i];
}
__global__ void k_copy(long n, const double* __restrict__ x, double* __restrict__ y) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    y[i] = x[i];
}
struct V9 {
  double v[9];
};
__global__ void k_fill9(long V, V9 v, double* __restrict__ x) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < 9 * V; i += (long)gridDim.x * blockDim.x)
    x[i] = v.v[i / V];
}
__global__ void k_fill(long n, double v, double* __restrict__ x) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    x[i] = v;
}
__global__ void k_state_init(long V, int W, double tt0, double* __restrict__ st) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < (long)W * V;
       i += (long)gridDim.x * blockDim.x) {
    const long w = i / V;
    double v = 0.0;
    if (w == CPFFT_W_RP + 0 || w == CPFFT_W_RP + 4 || w == CPFFT_W_RP + 8) v = 1.0;
    if (w == CPFFT_W_TT) v = tt0;
    st[i] = v;
  }
}
__global__ void k_gather_col(long V, int col, const double* __restrict__ K4, double* __restrict__ C) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < 9 * V; i += (long)gridDim.x * blockDim.x) {
    long j = i / V, e = i - j * V;
    C[i] = K4[(9 * j + col) * V + e];
  }
}
static inline unsigned grid_for(long n) {
  long g = (n + kBlock - 1) / kBlock;
  return (unsigned)(g > 8192 ? 8192 : (g < 1 ? 1 : g));
}

void launch_axpy(long n, double a, const double* x, double* y, hipStream_t s) {
  k_axpy<<<grid_for(n), kBlock, 0, s>>>(n, a, x, y);
}
void launch_scal(long n, double a, double* x, hipStream_t s) {
  k_scal<<<grid_for(n), kBlock, 0, s>>>(n, a, x);
}
void launch_copy(long n, const double* x, double* y, hipStream_t s) {
  k_copy<<<grid_for(n), kBlock, 0, s>>>(n, x, y);
}
void launch_fill9(long V, const double* v9, double* x, hipStream_t s) {
  V9 v;
  for (int i = 0; i < 9; ++i) v.v[i] = v9[i];
  k_fill9<<<grid_for(9 * V), kBlock, 0, s>>>(V, v, x);
}
void launch_fill(long n, double v, double* x, hipStream_t s) {
  k_fill<<<grid_for(n), kBlock, 0, s>>>(n, v, x);
}
__global__ void k_fill_f32(long n, float v, float* __restrict__ x) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    x[i] = v;
}
void launch_fill_f32(long n, float v, float* x, hipStream_t s) {
  k_fill_f32<<<grid_for(n), kBlock, 0, s>>>(n, v, x);
}
void launch_state_init(long V, int W, double tt0, double* state, hipStream_t s) {
  k_state_init<<<grid_for((long)W * V), kBlock, 0, s>>>(V, W, tt0, state);
}
void launch_gather_k4_col(long V, int i, const double* K4, double* C, hipStream_t s) {
  k_gather_col<<<grid_for(9 * V), kBlock, 0, s>>>(V, i, K4, C);
}
// ------------------------------------------------- device-scalar CG
// Start of a solve: x = 0, r = b (and p = b), partial sums of b.b over the
// contiguous ranges of k_dot_part
template <bool P>
__global__ __launch_bounds__(kBlock) void k_cg_start(long n, const double* __restrict__ b,
                                                     double* __restrict__ x,
                                                     double* __restrict__ r,
                                                     double* __restrict__ p,
                                                     double* __restrict__ part) {
  __shared__ double sh[kBlock];
  const long chunk = (n + gridDim.x - 1) / gridDim.x;
  const long lo = blockIdx.x * chunk, hi = min(n, lo + chunk);
  double acc = 0.0;
  for (long i = lo + threadIdx.x; i < hi; i += kBlock) {
    const double v = b[i];
    x[i] = 0.0;
    r[i] = v;
    if constexpr (P) p[i] = v;
    acc += v * v;
  }
  const double s = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}
// block b: system b; told: with one system, host memory that receives
// 2 seq + (whether the right-hand side vanishes)
__global__ __launch_bounds__(kBlock) void k_cg_init(const double* __restrict__ part, int np,
                                                    double tol, int maxit, int zero_code,
                                                    CGScalars* __restrict__ cs,
                                                    double* __restrict__ m, long long* told,
                                                    long long seq) {
  __shared__ double sh[kBlock];
  const double bb = ordered_sum<kBlock>(part + (long)blockIdx.x * np, np, sh);
  if (m && threadIdx.x < 9) m[9 * blockIdx.x + threadIdx.x] = 0.0;
  if (threadIdx.x == 0) {
    CGScalars c{};
    c.rr = bb;
    c.n2b = sqrt(bb);
    c.tolb = tol * c.n2b;
    c.tol = tol;
    c.resnorm = c.n2b;
    c.maxit = maxit;
    c.done = c.n2b <= 2.220446049250313e-16 ? zero_code : 0;
    cs[blockIdx.x] = c;
    if (told)
      __hip_atomic_store(told, 2 * seq + (c.done != 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}
void launch_cg_start(long n, const double* b, double* x, double* r, double* p, double* partials,
                     hipStream_t s) {
  if (p)
    k_cg_start<true><<<kRedBlocks, kBlock, 0, s>>>(n, b, x, r, p, partials);
  else
    k_cg_start<false><<<kRedBlocks, kBlock, 0, s>>>(n, b, x, r, p, partials);
}
int cg_start_parts() { return kRedBlocks; }
void launch_cg_init(const double* part, int np, double tol, int maxit, int zero_code,
                    CGScalars* cs, double* m, int nsys, hipStream_t s, long long* told,
                    long long seq) {
  k_cg_init<<<nsys, kBlock, 0, s>>>(part, np, tol, maxit, zero_code, cs, m, told, seq);
}
// alpha = rr / (p.q) from the partial sums (same order as k_sum_parts)
// block b serves system b: partial sums part + b pstride, scalars cs + b
__global__ __launch_bounds__(kBlock) void k_cg_alpha(const double* __restrict__ part, int np,
                                                     CGScalars* __restrict__ cs, long pstride) {
  cs += blockIdx.x;
  part += blockIdx.x * pstride;
  if (cs->done) return;
  __shared__ double sh[kBlock];
  const double pq = ordered_sum<kBlock>(part, np, sh);
  if (threadIdx.x == 0) cs->alpha = cs->rr / pq;
}

template <bool XUPD>
__global__ __launch_bounds__(kBlock) void k_cg_update_s(long n, const CGScalars* __restrict__ cs,
                                                        const double* __restrict__ p,
                                                        const double* __restrict__ q,
                                                        double* __restrict__ x,
                                                        double* __restrict__ r,
                                                        double* __restrict__ part) {
  if (cs->done) return;
  const double a = cs->alpha;
  __shared__ double sh[kBlock];
  long chunk = (n + gridDim.x - 1) / gridDim.x;
  long lo = blockIdx.x * chunk, hi = min(n, lo + chunk);
  double acc = 0.0;
  // four elements per pass with their loads issued together (more bytes in
  // flight per wave); the sum keeps the element order
  long i = lo + threadIdx.x;
  for (; i + 3 * kBlock < hi; i += 4 * kBlock) {
    double pv[4], qv[4], xv[4], rv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if constexpr (XUPD) {
        pv[u] = p[i + u * kBlock];
        xv[u] = x[i + u * kBlock];
      }
      qv[u] = q[i + u * kBlock];
      rv[u] = r[i + u * kBlock];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if constexpr (XUPD) x[i + u * kBlock] = xv[u] + a * pv[u];
      const double ri = rv[u] - a * qv[u];
      r[i + u * kBlock] = ri;
      acc += ri * ri;
    }
  }
  for (; i < hi; i += kBlock) {
    if constexpr (XUPD) x[i] = x[i] + a * p[i];
    double ri = r[i] - a * q[i];
    r[i] = ri;
    acc += ri * ri;
  }
  double s = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}
// |r| test from the r.r partial sums (FFT_nr3.f:304-306); with m, first
// m[c] += alpha * dc[c] * scale (this iteration's alpha)
// block b serves system b (part + b pstride, cs + b, dc and m + 9 b)
__global__ __launch_bounds__(kBlock) void k_cg_check(const double* __restrict__ part, int np,
                                                     CGScalars* __restrict__ cs,
                                                     const double* __restrict__ dc,
                                                     double* __restrict__ m, double scale,
                                                     long pstride) {
  cs += blockIdx.x;
  part += blockIdx.x * pstride;
  if (dc) dc += 9 * blockIdx.x;
  if (m) m += 9 * blockIdx.x;
  if (cs->done) return;
  __shared__ double sh[kBlock];
  const double rr1 = ordered_sum<kBlock>(part, np, sh);
  if (threadIdx.x == 0) {
    if (m)
      for (int c = 0; c < 9; ++c) m[c] += cs->alpha * (dc[c] * scale);
    cg_check(cs, rr1);
  }
}
void launch_cg_update_check(long n, CGScalars* cs, const double* p, const double* q, double* x,
                            double* r, double* partials, hipStream_t s, bool xupd,
                            const double* dc, double* m, double scale) {
  if (xupd)
    k_cg_update_s<true><<<kRedBlocks, kBlock, 0, s>>>(n, cs, p, q, x, r, partials);
  else
    k_cg_update_s<false><<<kRedBlocks, kBlock, 0, s>>>(n, cs, p, q, x, r, partials);
  k_cg_check<<<1, kBlock, 0, s>>>(partials, kRedBlocks, cs, dc, m, scale, 0);
}
void launch_cg_alpha(const double* part, int np, CGScalars* cs, hipStream_t s, int nsys,
                     long pstride) {
  k_cg_alpha<<<nsys, kBlock, 0, s>>>(part, np, cs, pstride);
}
void launch_cg_check(const double* part, int np, CGScalars* cs, hipStream_t s, const double* dc,
                     double* m, double scale, int nsys, long pstride) {
  k_cg_check<<<nsys, kBlock, 0, s>>>(part, np, cs, dc, m, scale, pstride);
}

// ------------------------------------------ multi-RHS K4 contraction
// q_i = K4 : p_i for the right-hand sides i < nrhs whose solve is still
// running (tangent_homo's nine solves share K4, which is read once).
// First p_i = r_i + beta p_i.
__global__ __launch_bounds__(kBlock) void k_k4_contract_multi(long V, const double* __restrict__ K4,
                                                              Ptr9 pp, const CGScalars* __restrict__ cs,
                                                              int nrhs, Ptr9r rr,
                                                              double* __restrict__ pqpart) {
  const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const bool valid = e < V;  // no early return: pqpart sums use a block barrier
  bool any = false;
  for (int i = 0; i < nrhs; ++i) any |= cs[i].done == 0;
  if (!any) return;  // the same in every thread of the launch
  double k[81];
#pragma unroll
  for (int j = 0; j < 81; ++j) k[j] = valid ? __builtin_nontemporal_load(K4 + j * V + e) : 0.0;
  // r and p of right-hand side i in buffer i % 2: those of the next running
  // one are loaded before the current one is computed and stored, so their
  // latency overlaps the work (the done flags are the same in every thread)
  auto running = [&](int i) { return i < nrhs && cs[i].done == 0; };
  double rb[2][9], pb[2][9];
  auto load = [&](int i, double (&r9)[9], double (&p9)[9]) {
#pragma unroll
    for (int c = 0; c < 9; ++c) {
      r9[c] = valid ? __builtin_nontemporal_load(rr.r[i] + c * V + e) : 0.0;
      p9[c] = valid ? __builtin_nontemporal_load(pp.p[i] + c * V + e) : 0.0;
    }
  };
  // pqpart: per right-hand side, the wave sums of p_i . (K4:p_i)
  __shared__ double wred[9][kBlock / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (running(0)) load(0, rb[0], pb[0]);
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    if (i + 1 < 9 && running(i + 1)) load(i + 1, rb[(i + 1) & 1], pb[(i + 1) & 1]);
    if (!running(i)) continue;
    double f[9];
    const double beta = cs[i].beta;
    double* pw = const_cast<double*>(pp.p[i]);
#pragma unroll
    for (int c = 0; c < 9; ++c) {
      // (the first direction is r, whatever p holds)
      f[c] = beta == 0.0 ? rb[i & 1][c] : rb[i & 1][c] + beta * pb[i & 1][c];
      if (valid) __builtin_nontemporal_store(f[c], pw + c * V + e);
    }
    double pq = 0.0;
#pragma unroll
    for (int r = 0; r < 9; ++r) {
      const double q = ddot42n_row(k + 9 * r, f);
      if (valid) __builtin_nontemporal_store(q, pp.q[i] + r * V + e);
      pq += q * f[r];
    }
    if (pqpart) {
      // butterfly over the wave: every lane ends with the same sum
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) pq += __shfl_xor(pq, off);
      if (lane == 0) wred[i][wave] = pq;
    }
  }
  if (pqpart) {
    __syncthreads();
    const int i = threadIdx.x;
    if (running(i))
      pqpart[(long)i * gridDim.x + blockIdx.x] = (wred[i][0] + wred[i][1]) + (wred[i][2] + wred[i][3]);
  }
}

int k4_contract_multi_blocks(long V) { return (int)((V + kBlock - 1) / kBlock); }

void launch_k4_contract_multi(long V, const double* K4, const Ptr9& pp, const CGScalars* cs,
                              int nrhs, hipStream_t s, const Ptr9r& rr, double* pqpart) {
  k_k4_contract_multi<<<(unsigned)k4_contract_multi_blocks(V), kBlock, 0, s>>>(V, K4, pp, cs, nrhs,
                                                                              rr, pqpart);
}

// ------------------------------------------------------- stress update
// One thread per voxel, one wave per block.  Bound by FP64 issue and the
// latency of a single wave per SIMD: the Newton iteration's 7x7 system and
// the slip sums take 512 registers a lane (two waves would spill more than a
// kilobyte a lane and run 1.7 times as long).  So what is not needed is left
// out of each instantiation: EXPL the explicit update of iteration 0, WARM
// the warm-start candidates, MatParamsInt the calls to pow; scratch falls from 640
// to 148 bytes a lane (with the candidates 512, and 720 with the general
// parameters, which always have them).  At 128^3, about five local iterations
// a voxel: 3.31 ms for fcc (60% of a wave's cycles issue a vector instruction,
// 28% wait) against 5.83 with the stages of the local solve, their line
// searches and the general parameters inlined one after another and slip
// systems taken one at a time.  The candidates' registers cost what they save:
// from the previous iterate 2.86 ms a call against 2.75 over load steps 6 to 25
// of the 128^3 workload, with 1.68 local iterations a voxel instead of 3.01.
template <int NS, bool EXPL, bool WARM, class MP>
__global__ __launch_bounds__(64) void k_drive_eps_sig(long V, MP P,
                                                      const Orient<NS>* __restrict__ orients,
                                                      const int32_t* __restrict__ oid, int step,
                                                      const double* __restrict__ Fn,
                                                      const double* __restrict__ Fn1,
                                                      const double* __restrict__ sn,
                                                      double* __restrict__ snp1,
                                                      double* __restrict__ Pn1,
                                                      double* __restrict__ tan6,
                                                      const float* __restrict__ ws,
                                                      int warm_prev,
                                                      long long* __restrict__ counters) {
  const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
  Counters cnt{0, 0, 0, 0, 0, 0};
  if (e < V) {
    const Orient<NS>& o = orients[oid[e]];
    // this step's previous global iterate (stress, slip resistance), read
    // before the update overwrites it
    double xp[7];
    if (WARM && warm_prev) {
#pragma unroll
      for (int k = 0; k < 6; ++k) xp[k] = snp1[k * V + e];
      xp[6] = snp1[15 * V + e];
    }
    voxel_update<NS, EXPL, WARM>(
        P, o, step,
        [&](int which, int c) { return which ? Fn1[c * V + e] : Fn[c * V + e]; },
        [&](int w) { return sn[w * V + e]; },
        [&](int w, double v) { snp1[w * V + e] = v; },
        [&](int c, double v) { Pn1[c * V + e] = v; },
        [&](int c, double v) { tan6[c * V + e] = v; }, cnt, ws ? ws + e : nullptr, V,
        warm_prev ? xp : nullptr);
  }
  // wavefront-level sums of the counters, one integer atomic per wavefront
  long long c[6] = {cnt.pred_it, cnt.upd_it, cnt.cuts, cnt.failed, cnt.ls_evals, cnt.ws_fallback};
  for (int k = 0; k < 6; ++k) {
    long long v = c[k];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if ((threadIdx.x & 63) == 0 && v) atomicAdd((unsigned long long*)&counters[k], (unsigned long long)v);
  }
  // local iterations the wavefront issues: 64 lanes times its slowest lane's
  // count (counters[6]; against counters[0] + counters[1], the lanes' own
  // iterations, it measures the divergence of the local solves)
  long long m = cnt.pred_it + cnt.upd_it;
  for (int off = 32; off > 0; off >>= 1) m = max(m, (long long)__shfl_xor(m, off, 64));
  if ((threadIdx.x & 63) == 0 && m) atomicAdd((unsigned long long*)&counters[6], (unsigned long long)(64 * m));
}

// K4 = dP/dF from the tangent of k_drive_eps_sig (cep2A)
__global__ __launch_bounds__(64) void k_cep2A(long V, const double* __restrict__ Fn,
                                              const double* __restrict__ Fn1,
                                              const double* __restrict__ snp1,
                                              const double* __restrict__ tan6,
                                              double* __restrict__ K4) {
  const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (e >= V) return;
  double t6[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) t6[k] = snp1[k * V + e];
  voxel_dPdF([&](int which, int c) { return which ? Fn1[c * V + e] : Fn[c * V + e]; }, t6,
             [&](int c) { return tan6[c * V + e]; },
             [&](int c, double v) { K4[c * V + e] = v; });
}

template <int NS>
void launch_drive_eps_sig(long V, const MatParams& P, const Orient<NS>* orients,
                          const int32_t* orient_id, int step, int iter, const double* Fn,
                          const double* Fn1, const double* sn, double* snp1, double* Pn1,
                          double* tan6, double* K4, const float* ws, int warm_prev,
                          long long* counters, hipStream_t s) {
  const int bs = 64;
  unsigned g = (unsigned)((V + bs - 1) / bs);
  auto update = [&](auto expl, auto warm, auto params) {
    k_drive_eps_sig<NS, decltype(expl)::value, decltype(warm)::value><<<g, bs, 0, s>>>(
        V, params, orients, orient_id, step, Fn, Fn1, sn, snp1, Pn1, tan6, ws, warm_prev, counters);
  };
  const std::true_type yes;
  const std::false_type no;
  // (other materials' Newton iterations have one form, with the candidates)
  const bool simple = P.int_rate && P.m_is_one, warm = ws || warm_prev;
  if (iter == 0)
    update(yes, no, P);
  else if (simple && !warm)
    update(no, no, MatParamsInt{P});
  else if (simple)
    update(no, yes, MatParamsInt{P});
  else
    update(no, yes, P);
  k_cep2A<<<g, bs, 0, s>>>(V, Fn, Fn1, snp1, tan6, K4);
}

// ----------------------------------------------- warm-start features
// rows r < nrows of voxels e = e0 + r * stride: raw network inputs into
// X[r][18 + 2 NS]; with T != nullptr also the converged slip increments of
// state n+1, as u_s (slip_to_u), into T[r][NS] (training pairs)
template <int NS>
__global__ __launch_bounds__(64) void k_mlp_features(long V, MatParams P,
                                                     const Orient<NS>* __restrict__ orients,
                                                     const int32_t* __restrict__ oid, int step,
                                                     const double* __restrict__ Fn,
                                                     const double* __restrict__ Fn1,
                                                     const double* __restrict__ sn,
                                                     const double* __restrict__ snp1, long e0,
                                                     long stride, long nrows,
                                                     float* __restrict__ X, float* __restrict__ T) {
  constexpr int NIN = 18 + 2 * NS;
  const long r = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (r >= nrows) return;
  const long e = e0 + r * stride;
  if (e >= V) return;
  float f[NIN];
  voxel_features<NS>(P, orients[oid[e]], step,
                     [&](int which, int c) { return which ? Fn1[c * V + e] : Fn[c * V + e]; },
                     [&](int w) { return sn[w * V + e]; }, f);
  for (int k = 0; k < NIN; ++k) X[r * NIN + k] = f[k];
  if (T) {
    const double dg = P.alter_mode ? P.eps_dot_0_y * P.dt : 1.0;
    for (int k = 0; k < NS; ++k) T[r * NS + k] = (float)slip_to_u(P, dg, snp1[(23 + k) * V + e]);
  }
}

// every voxel's network inputs, normalised ((x - mean) / sd, nrm =
// [mean | sd]) and rounded to BF16, into Xv[e][NINP] with the pad columns
// zero: the A operand of the inference kernel
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even (inputs are finite)
  return (uint16_t)(u >> 16);
}
template <int NS>
__global__ __launch_bounds__(64) void k_mlp_features_norm(long V, MatParams P,
                                                          const Orient<NS>* __restrict__ orients,
                                                          const int32_t* __restrict__ oid,
                                                          int step, const double* __restrict__ Fn,
                                                          const double* __restrict__ Fn1,
                                                          const double* __restrict__ sn,
                                                          const float* __restrict__ nrm, int ninp,
                                                          uint16_t* __restrict__ Xv) {
  constexpr int NIN = 18 + 2 * NS;
  const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (e >= V) return;
  float f[NIN];
  voxel_features<NS>(P, orients[oid[e]], step,
                     [&](int which, int c) { return which ? Fn1[c * V + e] : Fn[c * V + e]; },
                     [&](int w) { return sn[w * V + e]; }, f);
  uint16_t* x = Xv + e * ninp;
  // NIN is even; compile-time indexes keep f in registers
#pragma unroll
  for (int k = 0; k < NIN; k += 2) {
    const uint16_t lo = f32_to_bf16((f[k] - nrm[k]) / nrm[NIN + k]);
    const uint16_t hi = f32_to_bf16((f[k + 1] - nrm[k + 1]) / nrm[NIN + k + 1]);
    *reinterpret_cast<uint32_t*>(x + k) = (uint32_t)lo | ((uint32_t)hi << 16);
  }
  for (int k = NIN; k < ninp; k += 2) *reinterpret_cast<uint32_t*>(x + k) = 0u;
}

template <int NS>
void launch_mlp_features(long V, const MatParams& P, const Orient<NS>* orients, const int32_t* oid,
                         int step, const double* Fn, const double* Fn1, const double* sn,
                         const double* snp1, long e0, long stride, long nrows, float* X, float* T,
                         hipStream_t s) {
  k_mlp_features<NS><<<(unsigned)((nrows + 63) / 64), 64, 0, s>>>(
      V, P, orients, oid, step, Fn, Fn1, sn, snp1, e0, stride, nrows, X, T);
}
template <int NS>
void launch_mlp_features_norm(long V, const MatParams& P, const Orient<NS>* orients,
                              const int32_t* oid, int step, const double* Fn, const double* Fn1,
                              const double* sn, const float* nrm, int ninp, uint16_t* Xv,
                              hipStream_t s) {
  k_mlp_features_norm<NS><<<(unsigned)((V + 63) / 64), 64, 0, s>>>(V, P, orients, oid, step, Fn,
                                                                   Fn1, sn, nrm, ninp, Xv);
}
#define CPFFT_INST_FEATURES(NS)                                                                  \
  template void launch_mlp_features<NS>(long, const MatParams&, const Orient<NS>*, const int32_t*, \
                                        int, const double*, const double*, const double*,         \
                                        const double*, long, long, long, float*, float*,          \
                                        hipStream_t);                                             \
  template void launch_mlp_features_norm<NS>(long, const MatParams&, const Orient<NS>*,           \
                                             const int32_t*, int, const double*, const double*,   \
                                             const double*, const float*, int, uint16_t*,         \
                                             hipStream_t);
CPFFT_INST_FEATURES(12)
CPFFT_INST_FEATURES(24)
#undef CPFFT_INST_FEATURES

template void launch_drive_eps_sig<12>(long, const MatParams&, const Orient<12>*, const int32_t*,
                                       int, int, const double*, const double*, const double*,
                                       double*, double*, double*, double*, const float*, int,
                                       long long*, hipStream_t);
template void launch_drive_eps_sig<24>(long, const MatParams&, const Orient<24>*, const int32_t*,
                                       int, int, const double*, const double*, const double*,
                                       double*, double*, double*, double*, const float*, int,
                                       long long*, hipStream_t);
template void launch_drive_eps_sig<48>(long, const MatParams&, const Orient<48>*, const int32_t*,
                                       int, int, const double*, const double*, const double*,
                                       double*, double*, double*, double*, const float*, int,
                                       long long*, hipStream_t);

}  // namespace cpfft
