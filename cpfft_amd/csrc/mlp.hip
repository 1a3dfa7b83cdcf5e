// mlp.hip -- the learned warm start of the per-voxel Newton solve: a
// nin -> 128 -> 128 -> nout tanh network (nin = 18 + 2 ns, nout = ns for a
// crystal of ns slip systems) trained and evaluated with BF16 matrix-core
// (MFMA) products and FP32 accumulation.  It has no counterpart in
// the reference; it only supplies the starting point of mm10_solve
// (mm10_a.f:2945-3023), whose FP64 Newton iteration and tolerances are
// unchanged.
//
// A training step is two launches.  k_mlp_step takes 32 rows per block
// through the forward pass, the loss and the backward pass without leaving
// the CU, the activations in LDS, the tanh values that the backward pass
// needs in the registers of the lanes that made them, and writes what the
// weight gradients read with the rows contiguous.  k_mlp_grad gives each
// 16 x 16 tile of a weight gradient to one wave, which sums over all rows in
// order, and applies Adam to it.  A step on 4096 rows takes 33 us (20 + 13)
// where one launch per product and reduction took 505 us, 381 of them in the
// three weight gradients (6 to 64 waves, two-byte loads across the rows).
#include "mlp.h"

#include <algorithm>
#include <type_traits>

namespace cpfft {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float f) {
  // round to nearest even (inputs are finite)
  uint32_t u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__global__ void k_to_bf16(long n, const float* __restrict__ x, uint16_t* __restrict__ y) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    y[i] = f2bf(x[i]);
}

// ---- column statistics of the log ------------------------------------------
// mean and standard deviation of each column of X [rows][cx] and T
// [rows][ct] (cx + ct <= 96), two passes with FP64 accumulation; a zero
// deviation is replaced by 1.  A block takes a run of consecutive rows, so
// the loads are contiguous (one block per column read one float per 168
// bytes: 137 us a pass pair, at 65536 rows of 42 + 12).
static constexpr int kStatCols = 96, kStatGroups = 10, kStatT = kStatCols * kStatGroups;

// part[block][c] = sum over the block's rows of x (PASS 0) or (x - mean)^2
template <int PASS>
__global__ __launch_bounds__(kStatT) void k_colstats(long rows, long per, int cx, int ct,
                                                     const float* __restrict__ X,
                                                     const float* __restrict__ T,
                                                     const double* __restrict__ sums,
                                                     double* __restrict__ part) {
  __shared__ double sh[kStatGroups][kStatCols];
  const int c = threadIdx.x % kStatCols, g = threadIdx.x / kStatCols;
  const long r0 = blockIdx.x * per, r1 = min(rows, r0 + per);
  double acc = 0.0;
  if (c < cx + ct) {
    const float* p = c < cx ? X + c : T + (c - cx);
    const int ld = c < cx ? cx : ct;
    const double mu = PASS ? sums[c] / (double)rows : 0.0;
    for (long r = r0 + g; r < r1; r += kStatGroups) {
      const double d = p[r * ld] - mu;
      acc += PASS ? d * d : d;
    }
  }
  sh[g][c] = acc;
  __syncthreads();
  if (g == 0) {
    for (int k = 1; k < kStatGroups; ++k) acc += sh[k][c];
    part[(long)blockIdx.x * kStatCols + c] = acc;
  }
}
// sums over the blocks; PASS 1 also writes mean and deviation
template <int PASS>
__global__ __launch_bounds__(kStatT) void k_colstats_sum(int nb, long rows, int cx, int ct,
                                                         const double* __restrict__ part,
                                                         double* __restrict__ sums,
                                                         float* __restrict__ norm) {
  __shared__ double sh[kStatGroups][kStatCols];
  const int c = threadIdx.x % kStatCols, g = threadIdx.x / kStatCols;
  double acc = 0.0;
  for (int b = g; b < nb; b += kStatGroups) acc += part[(long)b * kStatCols + c];
  sh[g][c] = acc;
  __syncthreads();
  if (g != 0 || c >= cx + ct) return;
  for (int k = 1; k < kStatGroups; ++k) acc += sh[k][c];
  if (PASS == 0) {
    sums[c] = acc;
  } else {
    const double v = sqrt(acc / (double)rows);
    float* mean = c < cx ? norm + c : norm + 2 * cx + (c - cx);
    float* sd = c < cx ? norm + cx + c : norm + 2 * cx + ct + (c - cx);
    *mean = (float)(sums[c] / (double)rows);
    *sd = v > 0.0 ? (float)v : 1.0f;
  }
}

__device__ __forceinline__ uint32_t mix32(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352du;
  x ^= x >> 15;
  x *= 0x846ca68bu;
  x ^= x >> 16;
  return x;
}

static unsigned grid1(long n) {
  long g = (n + 255) / 256;
  return (unsigned)(g > 4096 ? 4096 : (g < 1 ? 1 : g));
}

// ---- packed BF16 weights of the training step ------------------------------
// Every product below reads its weight operand as 16-byte runs along K:
// W1 [128][ninp], W2 [128][128], W2^T [128][128], W3 [noutp][128] and W3^T
// [128][32], the padding zero.
struct PackOff {
  long w1, w2, w2t, w3, w3t, end;
};
__host__ __device__ inline PackOff pack_off(int ninp, int noutp) {
  PackOff o;
  o.w1 = 0;
  o.w2 = o.w1 + (long)kMlpHid * ninp;
  o.w2t = o.w2 + (long)kMlpHid * kMlpHid;
  o.w3 = o.w2t + (long)kMlpHid * kMlpHid;
  o.w3t = o.w3 + (long)noutp * kMlpHid;
  o.end = o.w3t + (long)kMlpHid * 32;
  return o;
}
inline int nout_pad(int nout) { return (nout + 15) / 16 * 16; }
long mlp_pack_len(const MlpDims& d) { return pack_off(mlp_nin_pad(d.nin), nout_pad(d.nout)).end; }

// parameter i (flat FP32 index) into its packed places
__device__ __forceinline__ void pack_param(long i, float w, const MlpDims& d, const PackOff& o,
                                           int ninp, uint16_t* __restrict__ pk) {
  const uint16_t b = f2bf(w);
  if (i < d.offB1) {
    const int u = (int)(i / d.nin), k = (int)(i - (long)u * d.nin);
    pk[o.w1 + (long)u * ninp + k] = b;
  } else if (i >= d.offW2 && i < d.offB2) {
    const int q = (int)(i - d.offW2), u = q / kMlpHid, k = q % kMlpHid;
    pk[o.w2 + q] = b;
    pk[o.w2t + (long)k * kMlpHid + u] = b;
  } else if (i >= d.offW3 && i < d.offB3) {
    const int q = (int)(i - d.offW3), u = q / kMlpHid, k = q % kMlpHid;
    pk[o.w3 + q] = b;
    pk[o.w3t + (long)k * 32 + u] = b;
  }
}
__global__ __launch_bounds__(256) void k_pack(MlpDims d, int ninp, int noutp,
                                              const float* __restrict__ params,
                                              uint16_t* __restrict__ pk) {
  const PackOff o = pack_off(ninp, noutp);
  const long i = blockIdx.x * 256L + threadIdx.x;
  if (i < d.nparam) pack_param(i, params[i], d, o, ninp, pk);
}
__global__ __launch_bounds__(256) void k_zero_u16(long n, uint16_t* __restrict__ p) {
  const long i = blockIdx.x * 256L + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ---- forward and backward pass of 32 rows ----------------------------------
// Rows either come from the log (count > 0: drawn with replacement by a hash
// of (seed, step, row), normalised) or are Xf, Tf themselves.  Yout != nullptr:
// only the forward pass, Y [rows][nout].  Products are
// v_mfma_f32_16x16x16_bf16 in ascending K with the weights as the A operand:
// lane l supplies A row l%16 and B column l%16 at k = 4*(l/16)..+3 and holds
// C rows 4*(l/16)..+3 of column l%16.  Wave w owns units 16w..16w+15.  BF16
// rounding points: inputs, weights, hidden activations and back-propagated
// errors; bias, tanh, its derivative and every sum in FP32, the loss in FP64.
// Bound by latency (one block per CU, five dependent products); 32 rows give
// a batch of 4096 128 blocks.  For the gradients it leaves the BF16 operands
// in the order in which k_mlp_grad's lanes read them (grad_at) and the FP32
// errors with the rows contiguous (leading dimension ld, a multiple of 32;
// rows past the batch hold zero errors).
static constexpr int kSR = 32;              // rows per block
static constexpr int kST = 512;             // threads: 8 waves
static constexpr int kRS = kMlpHid + 8;     // [row][unit] stride
static constexpr int kTS = kSR + 8;         // [unit][row] stride

// what the weight gradients read: BF16 X^T, H1^T, H2^T, dY^T, dZ2^T, dZ1^T
// (at these unit offsets) and FP32 dY^T, dZ2^T, dZ1^T ([unit][ld])
struct GradRows {
  int x, h1, h2, dy, dz2, dz1, end;  // BF16 units
  int fy, f2, f1, fend;              // FP32 units
};
__host__ __device__ inline GradRows grad_rows(int ninp, int noutp) {
  GradRows g;
  g.x = 0;
  g.h1 = g.x + ninp;
  g.h2 = g.h1 + kMlpHid;
  g.dy = g.h2 + kMlpHid;
  g.dz2 = g.dy + noutp;
  g.dz1 = g.dz2 + kMlpHid;
  g.end = g.dz1 + kMlpHid;
  g.fy = 0;
  g.f2 = g.fy + noutp;
  g.f1 = g.f2 + kMlpHid;
  g.fend = g.f1 + kMlpHid;
  return g;
}
// Place of (unit, row) in the BF16 operands: 16 units by 32 rows are one
// contiguous kilobyte, a lane's 16 bytes its operands of two MFMA steps.
// (As plain [unit][ld] rows a wave's load touched sixteen rows 8 KB apart,
// and the gradients of 4096 rows took 59 us instead of 13 us.)
__device__ __forceinline__ long grad_at(int ld, int unit, int row) {
  const int lane = (unit & 15) + 16 * ((row & 15) >> 2);
  return (((long)(unit >> 4) * (ld >> 5) + (row >> 5)) * 64 + lane) * 8 + ((row >> 4) & 1) * 4 +
         (row & 3);
}
inline int row_ld(int rows) { return (rows + kSR - 1) / kSR * kSR; }

template <int NINP, int NOUTP>
__global__ __launch_bounds__(kST) void k_mlp_step(int rows, int ld, MlpDims d, long count,
                                                  uint32_t seed, uint32_t step,
                                                  const float* __restrict__ Xf,
                                                  const float* __restrict__ Tf,
                                                  const float* __restrict__ nrm,
                                                  const uint16_t* __restrict__ pk,
                                                  const float* __restrict__ params,
                                                  uint16_t* __restrict__ gT,
                                                  float* __restrict__ fT,
                                                  double* __restrict__ lpart,
                                                  float* __restrict__ Yout) {
  constexpr int XS = NINP + 8;
  // H1 and dZ2 share a buffer: dZ2 is written two barriers after the last
  // read of H1
  __shared__ __align__(16) uint16_t X[kSR * XS];
  __shared__ __align__(16) uint16_t sB[kSR * kRS];
  __shared__ __align__(16) uint16_t H2[kSR * kRS];
  __shared__ __align__(16) uint16_t dY[kSR * 40];
  __shared__ __align__(16) uint16_t T[kMlpHid * kTS];  // transposing buffer
  __shared__ double lsum[4];
  uint16_t *H1 = sB, *dZ2 = sB;
  const PackOff o = pack_off(NINP, NOUTP);
  const GradRows q = grad_rows(NINP, NOUTP);
  const int nin = d.nin, nout = d.nout;
  const int r0 = blockIdx.x * kSR;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int li = lane & 15, kg = lane >> 4;
  auto src_row = [&](int r) -> long {
    const uint32_t h = mix32(seed * 0x9e3779b9u ^ mix32(step * 0x85ebca6bu ^ (uint32_t)(r0 + r)));
    return (long)(h % (uint32_t)count);
  };
  for (int i = threadIdx.x; i < kSR * NINP; i += kST) {
    const int r = i / NINP, c = i - r * NINP;
    float v = 0.0f;
    if (c < nin && r0 + r < rows)
      v = count > 0 ? (Xf[src_row(r) * nin + c] - nrm[c]) / nrm[nin + c]
                    : Xf[(long)(r0 + r) * nin + c];
    const uint16_t b = f2bf(v);
    X[r * XS + c] = b;
    T[c * kTS + r] = b;
  }
  for (int i = threadIdx.x; i < kSR * 40; i += kST) dY[i] = 0;
  // n units of the transposing buffer to unit u0 of gT, 16 bytes a thread
  auto flush = [&](int n, int u0) {
    for (int i = threadIdx.x; i < n * (kSR / 8); i += kST) {
      const int u = (i >> 6) * 16 + (i & 15), g = (i >> 4) & 3;
      const uint2 lo = *reinterpret_cast<const uint2*>(T + u * kTS + 4 * g);
      const uint2 hi = *reinterpret_cast<const uint2*>(T + u * kTS + 16 + 4 * g);
      *reinterpret_cast<u32x4*>(gT + grad_at(ld, u0 + u, r0 + 4 * g)) = u32x4{lo.x, lo.y, hi.x, hi.y};
    }
  };
  __syncthreads();
  if (!Yout) flush(NINP, q.x);
  auto lv = [](const uint16_t* p) { return *reinterpret_cast<const bf16x4*>(p); };
  // four consecutive units of one row: [row][unit] and the transposing buffer
  auto put = [&](uint16_t* R, int row, int u, const float v[4]) {
    uint16_t b[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) b[j] = f2bf(v[j]);
    if (R)
      *reinterpret_cast<uint2*>(R + row * kRS + u) =
          uint2{(uint32_t)b[0] | ((uint32_t)b[1] << 16), (uint32_t)b[2] | ((uint32_t)b[3] << 16)};
#pragma unroll
    for (int j = 0; j < 4; ++j) T[(u + j) * kTS + row] = b[j];
  };
  const int u0 = 16 * w + 4 * kg;  // this lane's units u0..u0+3
  // acc[rt] += A B^T over K for the two row tiles: A row 16 w + li at Ag, B
  // rows in LDS
  auto product = [&](auto K_, const uint16_t* Ag, const uint16_t* Bs, int bs, f32x4 (&acc)[2]) {
    constexpr int K = decltype(K_)::value;
    bf16x4 a[K / 16];
#pragma unroll
    for (int ks = 0; ks < K / 16; ++ks) a[ks] = lv(Ag + ks * 16 + kg * 4);
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      acc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < K / 16; ++ks)
        acc[rt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
            a[ks], lv(Bs + (16 * rt + li) * bs + ks * 16 + kg * 4), acc[rt], 0, 0, 0);
    }
  };
  using std::integral_constant;
  float h1[2][4], h2[2][4];
  f32x4 acc[2];
  product(integral_constant<int, NINP>{}, pk + o.w1 + (16 * w + li) * NINP, X, XS, acc);
  __syncthreads();  // X^T has left the transposing buffer
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
#pragma unroll
    for (int j = 0; j < 4; ++j) h1[rt][j] = tanhf(acc[rt][j] + params[d.offB1 + u0 + j]);
    put(H1, 16 * rt + li, u0, h1[rt]);
  }
  __syncthreads();
  if (!Yout) flush(kMlpHid, q.h1);
  product(integral_constant<int, kMlpHid>{}, pk + o.w2 + (16 * w + li) * kMlpHid, H1, kRS, acc);
  __syncthreads();
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
#pragma unroll
    for (int j = 0; j < 4; ++j) h2[rt][j] = tanhf(acc[rt][j] + params[d.offB2 + u0 + j]);
    put(H2, 16 * rt + li, u0, h2[rt]);
  }
  __syncthreads();
  if (!Yout) flush(kMlpHid, q.h2);
  // output layer and the loss: wave w < 2 NOUTP/16 takes row tile w % 2 of
  // output tile w / 2
  if (w < NOUTP / 8) {
    const int rt = w & 1, ot = w >> 1;
    f32x4 ac = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < kMlpHid / 16; ++ks)
      ac = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
          lv(pk + o.w3 + (16 * ot + li) * kMlpHid + ks * 16 + kg * 4),
          lv(H2 + (16 * rt + li) * kRS + ks * 16 + kg * 4), ac, 0, 0, 0);
    const int r = 16 * rt + li, row = r0 + r;
    const float sc = 2.0f / (float)((long)rows * nout);
    const long src = count > 0 ? src_row(r) : row;
    double ls = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = 16 * ot + 4 * kg + j;
      float g = 0.0f;
      if (n < nout && row < rows) {
        const float y = ac[j] + params[d.offB3 + n];
        if (Yout) {
          Yout[(long)row * nout + n] = y;
        } else {
          const float t = count > 0 ? (Tf[src * nout + n] - nrm[2 * nin + n]) / nrm[2 * nin + nout + n]
                                    : Tf[src * nout + n];
          const float e = y - t;
          ls += (double)e * e;
          g = sc * e;
        }
      }
      if (!Yout) {
        const uint16_t b = f2bf(g);
        dY[r * 40 + n] = b;
        gT[grad_at(ld, q.dy + n, row)] = b;
        fT[(long)(q.fy + n) * ld + row] = g;
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ls += __shfl_xor(ls, off);
    if (lane == 0) lsum[w] = ls;
  }
  if (Yout) return;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = lsum[0];
    for (int k = 1; k < NOUTP / 8; ++k) s += lsum[k];
    lpart[blockIdx.x] = s;
  }
  // dZ2 = (dY W3) (1 - H2^2)
  product(integral_constant<int, NOUTP>{}, pk + o.w3t + (16 * w + li) * 32, dY, 40, acc);
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = acc[rt][j];
      const float h = h2[rt][j];
      v[j] *= 1.0f - h * h;
      fT[(long)(q.f2 + u0 + j) * ld + r0 + 16 * rt + li] = v[j];
    }
    put(dZ2, 16 * rt + li, u0, v);
  }
  __syncthreads();
  flush(kMlpHid, q.dz2);
  // dZ1 = (dZ2 W2) (1 - H1^2)
  product(integral_constant<int, kMlpHid>{}, pk + o.w2t + (16 * w + li) * kMlpHid, dZ2, kRS, acc);
  __syncthreads();
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = acc[rt][j];
      const float h = h1[rt][j];
      v[j] *= 1.0f - h * h;
      fT[(long)(q.f1 + u0 + j) * ld + r0 + 16 * rt + li] = v[j];
    }
    put(nullptr, 16 * rt + li, u0, v);
  }
  __syncthreads();
  flush(kMlpHid, q.dz1);
}

// ---- weight gradients and Adam ---------------------------------------------
// Block b < nb_tiles: four 16 x 16 tiles of the weight gradients, one per
// wave, each summed over all rows in ascending order with
// v_mfma_f32_16x16x16_bf16; the operands of sixteen steps are loaded ahead
// of their products.  The other blocks: one bias gradient each, 256 row classes
// in order, then a halving tree.  Both orders are fixed by the sizes alone.
// ADAM: the Adam update (Kingma & Ba 2015) of the FP32 master weights and
// their packed BF16 copies (no block reads weights here); else grads.
// Bound by the chain of ld / 16 dependent MFMAs: 13 us for 4096 rows.
template <int NINP, int NOUTP, bool ADAM>
__global__ __launch_bounds__(256) void k_mlp_grad(int ld, MlpDims d, int nb_tiles,
                                                  const uint16_t* __restrict__ gT,
                                                  const float* __restrict__ fT,
                                                  float* __restrict__ grads,
                                                  float* __restrict__ wt, float* __restrict__ m,
                                                  float* __restrict__ v, uint16_t* __restrict__ pk,
                                                  float lr, float b1, float b2, float eps, float c1,
                                                  float c2) {
  const GradRows q = grad_rows(NINP, NOUTP);
  auto done = [&](long i, float gi) {
    if constexpr (ADAM) {
      const float mi = b1 * m[i] + (1.f - b1) * gi;
      const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
      m[i] = mi;
      v[i] = vi;
      const float wn = wt[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
      wt[i] = wn;
      pack_param(i, wn, d, pack_off(NINP, NOUTP), NINP, pk);
    } else {
      grads[i] = gi;
    }
  };
  if ((int)blockIdx.x >= nb_tiles) {  // bias gradients: b3, b2, b1
    __shared__ float sh[256];
    int c = (int)blockIdx.x - nb_tiles;
    long i;
    int row;
    if (c < d.nout) {
      row = q.fy + c;
      i = d.offB3 + c;
    } else if ((c -= d.nout) < kMlpHid) {
      row = q.f2 + c;
      i = d.offB2 + c;
    } else {
      c -= kMlpHid;
      row = q.f1 + c;
      i = d.offB1 + c;
    }
    const float* p = fT + (long)row * ld;
    float acc = 0.f;
    for (int r = threadIdx.x; r < ld; r += 256) acc += p[r];
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
      if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
      __syncthreads();
    }
    if (threadIdx.x == 0) done(i, sh[0]);
    return;
  }
  constexpr int H16 = kMlpHid / 16, T3 = NOUTP / 16 * H16, T2 = H16 * H16, T1 = H16 * (NINP / 16);
  const int lane = threadIdx.x & 63;
  const int li = lane & 15, kg = lane >> 4;
  int t = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
  if (t >= T3 + T2 + T1) return;
  int ra, rb, mt, nt, cols, rowsm;  // operand units, tile position, matrix shape
  long off;
  if (t < T2) {
    mt = t / H16;
    nt = t - mt * H16;
    ra = q.dz2 + 16 * mt;
    rb = q.h1 + 16 * nt;
    cols = kMlpHid;
    rowsm = kMlpHid;
    off = d.offW2;
  } else if ((t -= T2) < T1) {
    mt = t / (NINP / 16);
    nt = t - mt * (NINP / 16);
    ra = q.dz1 + 16 * mt;
    rb = q.x + 16 * nt;
    cols = d.nin;
    rowsm = kMlpHid;
    off = d.offW1;
  } else {
    t -= T1;
    mt = t / H16;
    nt = t - mt * H16;
    ra = q.dy + 16 * mt;
    rb = q.h2 + 16 * nt;
    cols = kMlpHid;
    rowsm = d.nout;
    off = d.offW3;
  }
  const u32x4* A = reinterpret_cast<const u32x4*>(gT + grad_at(ld, ra, 0)) + lane;
  const u32x4* B = reinterpret_cast<const u32x4*>(gT + grad_at(ld, rb, 0)) + lane;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const int nk = ld >> 5;  // pairs of steps
  constexpr int U = 8;
  u32x4 a[2][U], b[2][U];
  auto load = [&](u32x4 (&x)[U], u32x4 (&y)[U], int k) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const long i = (long)(k + u < nk ? k + u : nk - 1) * 64;
      x[u] = A[i];
      y[u] = B[i];
    }
  };
  auto mul = [&](const u32x4 (&x)[U], const u32x4 (&y)[U], int k) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k + u >= nk) break;
      acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
          __builtin_bit_cast(bf16x4, uint2{x[u].x, x[u].y}),
          __builtin_bit_cast(bf16x4, uint2{y[u].x, y[u].y}), acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
          __builtin_bit_cast(bf16x4, uint2{x[u].z, x[u].w}),
          __builtin_bit_cast(bf16x4, uint2{y[u].z, y[u].w}), acc, 0, 0, 0);
    }
  };
  load(a[0], b[0], 0);
  for (int k = 0; k < nk; k += 2 * U) {
    load(a[1], b[1], k + U);
    mul(a[0], b[0], k);
    load(a[0], b[0], k + 2 * U);
    mul(a[1], b[1], k + U);
  }
  const int col = 16 * nt + li;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = 16 * mt + 4 * kg + j;
    if (r < rowsm && col < cols) done(off + (long)r * cols + col, acc[j]);
  }
}

// ------------------------------------------------------------- host side
void mlp_weights_to_bf16(const MlpBuffers& b, hipStream_t s) {
  k_to_bf16<<<grid1(b.d.nparam), 256, 0, s>>>(b.d.nparam, b.params, b.pbf);
}

void mlp_pack_weights(const MlpBuffers& b, hipStream_t s) {
  const int ninp = mlp_nin_pad(b.d.nin), noutp = nout_pad(b.d.nout);
  const long n = mlp_pack_len(b.d);
  k_zero_u16<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(n, b.pk);
  k_pack<<<(unsigned)((b.d.nparam + 255) / 256), 256, 0, s>>>(b.d, ninp, noutp, b.params, b.pk);
}

int mlp_row_blocks(int rows) { return (rows + kSR - 1) / kSR; }
long mlp_grad_bf16(const MlpDims& d, int rows) {
  return (long)grad_rows(mlp_nin_pad(d.nin), nout_pad(d.nout)).end * row_ld(rows);
}
long mlp_grad_f32(const MlpDims& d, int rows) {
  return (long)grad_rows(mlp_nin_pad(d.nin), nout_pad(d.nout)).fend * row_ld(rows);
}

template <int NINP, int NOUTP>
static void launch_step(const MlpBuffers& b, int rows, long count, uint32_t seed, uint32_t step,
                        const float* X, const float* T, float* Y, hipStream_t s) {
  k_mlp_step<NINP, NOUTP><<<(unsigned)mlp_row_blocks(rows), kST, 0, s>>>(
      rows, row_ld(rows), b.d, count, seed, step, X, T, b.norm, b.pk, b.params, b.gT, b.fT, b.part,
      Y);
}
template <int NINP, int NOUTP, bool ADAM>
static void launch_grad(const MlpBuffers& b, int rows, float lr, float c1, float c2,
                        hipStream_t s) {
  const int h16 = kMlpHid / 16;
  const int tiles = h16 * (NOUTP / 16 + h16 + NINP / 16), nbt = (tiles + 3) / 4;
  k_mlp_grad<NINP, NOUTP, ADAM><<<(unsigned)(nbt + 2 * kMlpHid + b.d.nout), 256, 0, s>>>(
      row_ld(rows), b.d, nbt, b.gT, b.fT, b.grads, b.params, b.m, b.v, b.pk, lr, 0.9f, 0.999f,
      1e-8f, c1, c2);
}
// the two network sizes: fcc (42 inputs, 12 outputs) and bcc24 (66, 24)
static bool small_net(const MlpDims& d) { return mlp_nin_pad(d.nin) == 64 && d.nout <= 16; }

void mlp_forward(const MlpBuffers& b, int rows, const float* Xf, float* Y, hipStream_t s) {
  if (small_net(b.d))
    launch_step<64, 16>(b, rows, 0, 0, 0, Xf, nullptr, Y, s);
  else
    launch_step<96, 32>(b, rows, 0, 0, 0, Xf, nullptr, Y, s);
}

void mlp_grad(const MlpBuffers& b, int rows, const float* Xf, const float* Tf, hipStream_t s) {
  if (small_net(b.d)) {
    launch_step<64, 16>(b, rows, 0, 0, 0, Xf, Tf, nullptr, s);
    launch_grad<64, 16, false>(b, rows, 0.f, 0.f, 0.f, s);
  } else {
    launch_step<96, 32>(b, rows, 0, 0, 0, Xf, Tf, nullptr, s);
    launch_grad<96, 32, false>(b, rows, 0.f, 0.f, 0.f, s);
  }
}

void mlp_train_step(const MlpBuffers& b, int rows, long count, uint32_t seed, uint32_t step,
                    float lr, long t, hipStream_t s) {
  const float c1 = 1.f - powf(0.9f, (float)t), c2 = 1.f - powf(0.999f, (float)t);
  if (small_net(b.d)) {
    launch_step<64, 16>(b, rows, count, seed, step, b.logX, b.logT, nullptr, s);
    launch_grad<64, 16, true>(b, rows, lr, c1, c2, s);
  } else {
    launch_step<96, 32>(b, rows, count, seed, step, b.logX, b.logT, nullptr, s);
    launch_grad<96, 32, true>(b, rows, lr, c1, c2, s);
  }
}

// blocks of the column statistics: 64 rows or more each, at most 256
static int stat_blocks(long rows) { return (int)std::max(1L, std::min(256L, rows / 64)); }
long mlp_stat_doubles() { return 257L * kStatCols; }

void mlp_stats(const MlpBuffers& b, long count, hipStream_t s) {
  const MlpDims& d = b.d;
  const int nb = stat_blocks(count);
  const long per = (count + nb - 1) / nb;
  double* sums = b.stat + 256L * kStatCols;
  static_assert(18 + 3 * kMlpMaxOut <= kStatCols, "columns of the log");
  k_colstats<0><<<nb, kStatT, 0, s>>>(count, per, d.nin, d.nout, b.logX, b.logT, nullptr, b.stat);
  k_colstats_sum<0><<<1, kStatT, 0, s>>>(nb, count, d.nin, d.nout, b.stat, sums, nullptr);
  k_colstats<1><<<nb, kStatT, 0, s>>>(count, per, d.nin, d.nout, b.logX, b.logT, sums, b.stat);
  k_colstats_sum<1><<<1, kStatT, 0, s>>>(nb, count, d.nin, d.nout, b.stat, sums, b.norm);
}

// ------------------------------------------------------------ inference
// One launch over all voxels.  The block stages the BF16 weights (rows
// padded by eight elements against LDS bank conflicts) and the FP32 biases
// and output normalisation in LDS; each wavefront then takes 16 voxels at a
// time through the three layers with v_mfma_f32_16x16x32_bf16, the weights
// as the A operand (rows = output units) and the activations as the B
// operand (columns = the 16 voxels).  Lane l supplies A row l%16 and B
// column l%16 at k = 8*(l/16)..+7 of each K step of 32, and holds C rows
// 4*(l/16)..+3 of column l%16.  So after a layer, lane l holds units
// 16t + 4g + j (g = l/16, j < 4) of tile t for voxel l%16, and the eight
// values of tiles 2s and 2s+1 are that lane's B operand of the next layer's
// K step s, once the K index of the next weights is permuted the same way:
// position 8g + 4h + j of K step s is unit 32s + 16h + 4g + j.  The
// weights are stored permuted in LDS, the activations never leave the
// registers.  The rounding points are those of k_mlp_step: FP32 bias and
// tanh, BF16 hidden activations, FP32 output.
static constexpr int kIW = 8;               // wavefronts per inference block
static constexpr int kHS = kMlpHid + 8;     // padded row of W2, W3

// the unit at K position p (< 128) of the permuted order
__device__ __forceinline__ int perm_k(int p) {
  const int s = p >> 5, q = p & 31, g = q >> 3, h = (q >> 2) & 1, j = q & 3;
  return 32 * s + 16 * h + 4 * g + j;
}

template <int NINP, int NOUTP>
__global__ __launch_bounds__(64 * kIW) void k_mlp_infer(long V, int nin, int nout,
                                                        const uint16_t* __restrict__ Xv,
                                                        const uint16_t* __restrict__ pbf,
                                                        const float* __restrict__ params,
                                                        MlpDims d, const float* __restrict__ nrm,
                                                        float* __restrict__ ws) {
  constexpr int S1 = NINP + 8;
  __shared__ __align__(16) uint16_t W1[kMlpHid * S1];
  __shared__ __align__(16) uint16_t W2[kMlpHid * kHS];   // K permuted
  __shared__ __align__(16) uint16_t W3[NOUTP * kHS];     // K permuted
  __shared__ float b1[kMlpHid], b2[kMlpHid], b3[NOUTP], mt[NOUTP], st[NOUTP];
  const int T = 64 * kIW;
  for (int i = threadIdx.x; i < kMlpHid * S1; i += T) {
    const int n = i / S1, k = i - n * S1;
    W1[i] = k < nin ? pbf[d.offW1 + (long)n * nin + k] : 0;
  }
  for (int i = threadIdx.x; i < kMlpHid * kHS; i += T) {
    const int n = i / kHS, k = i - n * kHS;
    W2[i] = k < kMlpHid ? pbf[d.offW2 + (long)n * kMlpHid + perm_k(k)] : 0;
  }
  for (int i = threadIdx.x; i < NOUTP * kHS; i += T) {
    const int n = i / kHS, k = i - n * kHS;
    W3[i] = (n < nout && k < kMlpHid) ? pbf[d.offW3 + (long)n * kMlpHid + perm_k(k)] : 0;
  }
  for (int i = threadIdx.x; i < kMlpHid; i += T) {
    b1[i] = params[d.offB1 + i];
    b2[i] = params[d.offB2 + i];
  }
  for (int i = threadIdx.x; i < NOUTP; i += T) {
    b3[i] = i < nout ? params[d.offB3 + i] : 0.f;
    mt[i] = i < nout ? nrm[2 * nin + i] : 0.f;
    st[i] = i < nout ? nrm[2 * nin + nout + i] : 0.f;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int li = lane & 15, kg = lane >> 4;
  const long nrb = (V + 15) / 16;
  for (long rb = (long)blockIdx.x * kIW + w; rb < nrb; rb += (long)gridDim.x * kIW) {
    const long r = rb * 16 + li;  // this lane's voxel (B column)
    // layer 1: B = the voxel's inputs straight from HBM
    bf16x8 x1[NINP / 32];
#pragma unroll
    for (int ks = 0; ks < NINP / 32; ++ks) {
      if (r < V) {
        x1[ks] = *reinterpret_cast<const bf16x8*>(Xv + r * NINP + ks * 32 + kg * 8);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) x1[ks][j] = (__bf16)0.0f;
      }
    }
    // a layer's output as the next layer's B operand: K step s packs tiles
    // 2s (elements 0-3) and 2s+1 (elements 4-7), two BF16 per 32-bit word
    u32x4 h[kMlpHid / 32];
    // bias, tanh and BF16 rounding of tile t's four values, packed in pairs
    auto act = [&](f32x4 acc, const float* bias, int t, uint32_t* p) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const float v0 = tanhf(acc[2 * q] + bias[16 * t + 4 * kg + 2 * q]);
        const float v1 = tanhf(acc[2 * q + 1] + bias[16 * t + 4 * kg + 2 * q + 1]);
        p[q] = (uint32_t)f2bf(v0) | ((uint32_t)f2bf(v1) << 16);
      }
    };
#pragma unroll
    for (int s2 = 0; s2 < kMlpHid / 32; ++s2) {
      f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < NINP / 32; ++ks) {
        const bf16x8 a0 = *reinterpret_cast<const bf16x8*>(W1 + (32 * s2 + li) * S1 + ks * 32 + kg * 8);
        const bf16x8 a1 = *reinterpret_cast<const bf16x8*>(W1 + (32 * s2 + 16 + li) * S1 + ks * 32 + kg * 8);
        acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, x1[ks], acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, x1[ks], acc1, 0, 0, 0);
      }
      uint32_t p[4];
      act(acc0, b1, 2 * s2, p);
      act(acc1, b1, 2 * s2 + 1, p + 2);
      h[s2] = u32x4{p[0], p[1], p[2], p[3]};
      // keep the scheduler from hoisting every tile's weight loads (the
      // registers they would hold cost occupancy)
      __builtin_amdgcn_sched_barrier(0);
    }
    // layer 2
    u32x4 h2[kMlpHid / 32];
#pragma unroll
    for (int s2 = 0; s2 < kMlpHid / 32; ++s2) {
      f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < kMlpHid / 32; ++ks) {
        const bf16x8 a0 = *reinterpret_cast<const bf16x8*>(W2 + (32 * s2 + li) * kHS + ks * 32 + kg * 8);
        const bf16x8 a1 = *reinterpret_cast<const bf16x8*>(W2 + (32 * s2 + 16 + li) * kHS + ks * 32 + kg * 8);
        const bf16x8 b = __builtin_bit_cast(bf16x8, h[ks]);
        acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b, acc1, 0, 0, 0);
      }
      uint32_t p[4];
      act(acc0, b2, 2 * s2, p);
      act(acc1, b2, 2 * s2 + 1, p + 2);
      h2[s2] = u32x4{p[0], p[1], p[2], p[3]};
      __builtin_amdgcn_sched_barrier(0);
    }
    // layer 3 and the output normalisation
#pragma unroll
    for (int jt = 0; jt < NOUTP / 16; ++jt) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < kMlpHid / 32; ++ks) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(W3 + (16 * jt + li) * kHS + ks * 32 + kg * 8);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, h2[ks]), acc, 0, 0, 0);
      }
      if (r < V) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int n = 16 * jt + 4 * kg + j;
          if (n < nout) ws[n * V + r] = (acc[j] + b3[n]) * st[n] + mt[n];
        }
      }
    }
  }
}

void mlp_infer(const MlpBuffers& b, long V, hipStream_t s) {
  const unsigned g = 512;  // two blocks per CU (their weights fit the LDS); each loops over row blocks
  const MlpDims& d = b.d;
  if (mlp_nin_pad(d.nin) == 64 && d.nout <= 16)
    k_mlp_infer<64, 16><<<g, 64 * kIW, 0, s>>>(V, d.nin, d.nout, b.Xv, b.pbf, b.params, d, b.norm,
                                                b.ws);
  else
    k_mlp_infer<96, 32><<<g, 64 * kIW, 0, s>>>(V, d.nin, d.nout, b.Xv, b.pbf, b.params, d, b.norm,
                                                b.ws);
}

}  // namespace cpfft
