// kernels.h -- launch wrappers for the CDNA4 kernels (defined in
// cpfft_kernels.hip), called by the context code in cpfft_api.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "cg_device.h"
#include "cpfft_common.h"
#include "green.h"
#include "mm10_core.h"
#include "mlp.h"

namespace cpfft {

// Launch shapes chosen by the autotuner, as candidate indices (0 = the
// default shape).  fft_pencil.hip: a, a0 pass A with / without K4, b the y
// passes, c pass C.  fft_grid.hip (16, 32, 48): a, a0 k_fwd with / without
// K4, b k_inv (where they form no CG sum), c k_mid.  All
// candidates compute bit-identical results.
struct PencilTune {
  int a = 0, a0 = 0, b = 0, c = 0;
};
constexpr int kPencilCands = 5;  // candidate indices per pass are below this

struct SpecGeom {
  int N, Nz;        // grid edge, number of z frequencies kept (N/2+1)
  long V;           // N^3
  long S1;          // complex entries per spectral component: N*N*Nz
  int gamma_mode;   // 0 reference operator, 1 textbook projection
  const int* skip;  // fft_pencil.hip: if non-null and *skip != 0, every block returns at once
  PencilTune tune;  // launch shapes
};

// Geometry of the operator for edge N and Gamma variant gamma_mode.  Returns
// nullptr, or why N cannot be served.
const char* make_spec_geom(int N, int gamma_mode, SpecGeom& g);

// Displacement reconstruction (f2disp.hip): the cosine table (of
// f2disp_cos_doubles(N) doubles) once, then u (device, [3 (N+1)^3]
// node-major) from F; work holds f2disp_scratch_doubles(N) doubles and must
// not overlap u.
size_t f2disp_scratch_doubles(int N);
size_t f2disp_cos_doubles(int N);
void launch_f2disp_cos(int N, double* C, hipStream_t s);
void launch_f2disp(int N, const double* F, const double len[3], const double* C, double* work,
                   double* u, hipStream_t s);

// Gamma:(K4:F) or Gamma:F (K4 == nullptr).  spec: 2*9*S1 complex scratch.
// tw: the N twiddles exp(-2 pi i k/N).  fft_pencil.hip for N = 64, 96, 128,
// 256, fft_grid.hip for every other edge.
// CG work fused into the operator's passes (fft_pencil.hip):
// dir_p != nullptr: pass A first sets dir_p = dir_r + cs->beta * dir_p (the
//   CG direction, F must be dir_p) and transforms the new direction;
// dot_p != nullptr: pass D writes per-block partial sums of dot_p . out
//   into dot_part (gkdf_dot_parts(N) values, fixed order);
// dc != nullptr: pass C stores the voxel sums of the nine components of its
//   input (F, or K4:F) in dc[0..9);
// pq_part != nullptr (with dir_p): pass A writes the partial sums of
//   p . (K4:p) over each pencil pair (y, y+1) of each x into
//   pq_part[x*N/2 + y/2] (N*N/2 values, the same under every tile).  For a
//   symmetric projection G (the textbook operator) and p in its range, as
//   every CG direction of a right-hand side G(.) is, p . G(K4:p) equals
//   p . (K4:p), so pass D then needs no dot product.
// alpha_np > 0: right after pass A, alpha = cs->rr / (sum of the alpha_np
//   partial sums in pq_part);
// upd_r != nullptr (alpha already in cs): pass D does not store the
//   transform q but updates upd_r -= alpha q, with upd_x != nullptr also
//   upd_x += alpha dir_p, and writes per-block partial sums of the new
//   upd_r . upd_r into rr_part (gkdf_dot_parts(N) values).
struct CGFuse {
  double* dir_p;
  const double* dir_r;
  CGScalars* cs;
  const double* dot_p;
  double* dot_part;
  double* dc;
  double* pq_part;
  int alpha_np;
  double* upd_r;
  double* upd_x;
  double* rr_part;
};

void launch_gkdf(const SpecGeom& g, const double* F, const double* K4, double* out, cplx* spec,
                 const cplx* tw, hipStream_t s);
// ---- fft_grid.hip
// whether edge N is served there; whether by the slab kernels, which serve
// launch_cg_grid with q and launch_homo_rhs_grid for N = 64 and 96 too
bool gkdf_grid_edge(int N);
bool gkdf_slab_edge(int N);
void launch_gkdf_grid(const SpecGeom& g, const double* F, const double* K4, double* out,
                      cplx* spec, const cplx* tw, hipStream_t s);
// One CG iteration of nrhs systems (at most nine) that share K4.
// part 0: the forward pass (with chk first the convergence test of the
//   previous iteration, as launch_cg_check does it; p_new = r + beta p_old;
//   K4:p_new and its product with p_new) and the passes up to the projected
//   spectrum, alpha among them;
// part 1: the inverse pass: r -= alpha q, where x[i] != nullptr also
//   x += alpha p_new, and the r.r partial sums;
// part 2: nothing.
// out[0] != nullptr instead (the reference's operator): part 0 forms no
//   alpha; part 1 stores q in out with the p.q partial sums; part 2 forms alpha
//   and updates r and x.
// cs_old is the state before the iteration, cs_new the one after chk; they
// may be the same array when !chk.  p_old and p_new are different fields.
struct GridCG {
  int nrhs;
  double *p_old[9], *p_new[9], *r[9], *x[9], *out[9];
  const double* q[9];  // q[0] != nullptr: K4:p_new, formed by the caller (part 0 then neither
  int npq;             // tests nor forms the direction) with npq values of pq per system
  const double* K4;
  cplx* spec;  // nrhs * grid_spec_len entries
  const cplx* tw;
  CGScalars *cs_old, *cs_new;
  int chk;
  double *pq, *rr;  // partial sums: nrhs * grid_parts(N), nrhs * grid_rr_parts(N, out[0] == nullptr)
  double *dc, *m;   // as launch_cg_check, nine values per system (or nullptr)
  double scale;
};
void launch_cg_grid(const SpecGeom& g, const GridCG& c, int part, hipStream_t s);
// r[i] = -G(K4:E_i) for the unit tensors E_i, i0 <= i < i0 + n, with the r.r
// partial sums in rr (tangent_homo's right-hand sides)
void launch_homo_rhs_grid(const SpecGeom& g, const double* K4, int i0, int n, double* const* r,
                          cplx* spec, const cplx* tw, double* rr, hipStream_t s);
int grid_parts(int N);
int grid_rr_parts(int N, bool projection);
bool grid_fused_check(int N);  // whether chk may be used at this edge
long grid_spec_len(const SpecGeom& g);
// autotuner support for N = 16, 32, 48 (see pencil_candidate)
int grid_candidate(int N, int gamma_mode, int pass, int v);
void launch_grid_pass(const SpecGeom& g, int pass, int v, const double* F, const double* K4,
                      cplx* spec, const cplx* tw, hipStream_t s);

// ---- fft_pencil.hip
// returns false (and launches nothing) when N has no compile-time plan
bool launch_gkdf_pencil(const SpecGeom& g, const double* F, const double* K4, double* out,
                        cplx* spec, const cplx* tw, hipStream_t s, const CGFuse* fuse = nullptr);
// number of partial sums pass D writes for a fused dot product
int gkdf_dot_parts(int N);
// autotuner support: the value (pencils or lines per block) of candidate
// `variant` of pass `pass` (0 A with K4, 1 A without, 2 B, 3 C) for edge N,
// 0 if there is none; and one pass launched by itself with that candidate
int pencil_candidate(int N, int pass, int variant);
bool launch_pencil_pass(const SpecGeom& g, int pass, int variant, const double* F,
                        const double* K4, cplx* spec, const cplx* tw, hipStream_t s);

// alpha = rr / sum(part[0..np)) (p.q partial sums); for nsys systems at
// once, system b reading part + b pstride and cs[b] (one block each)
void launch_cg_alpha(const double* part, int np, CGScalars* cs, hipStream_t s, int nsys = 1,
                     long pstride = 0);
// convergence test and beta from the r.r partial sums part[0..np); with
// m != nullptr also m[c] += alpha * dc[c] * scale for c < 9 (the running sum
// over iterations of alpha times the mean of K4:p); nsys systems as for
// launch_cg_alpha, with dc and m advanced by 9 per system
void launch_cg_check(const double* part, int np, CGScalars* cs, hipStream_t s,
                     const double* dc = nullptr, double* m = nullptr, double scale = 0.0,
                     int nsys = 1, long pstride = 0);
// x += alpha p (xupd; without it x and p are not touched); r -= alpha q
// with the r.r partial sums, then the convergence test and beta (no p.q, no
// direction update)
void launch_cg_update_check(long n, CGScalars* cs, const double* p, const double* q, double* x,
                            double* r, double* partials, hipStream_t s, bool xupd = true,
                            const double* dc = nullptr, double* m = nullptr,
                            double scale = 0.0);

// x = 0, r = b, with p != nullptr also p = b, and the partial sums of b.b
// (start of a CG solve); then launch_cg_init with np = cg_start_parts()
void launch_cg_start(long n, const double* b, double* x, double* r, double* p, double* partials,
                     hipStream_t s);
int cg_start_parts();
// state of nsys solves about to start, from the partial sums of b.b (np per
// system): done = zero_code where |b| vanishes (FFT_nr3.f:254-262); with
// m != nullptr its nine values per system are cleared; with told != nullptr
// (pinned host memory, one system) *told = 2 seq + (whether |b| vanishes)
void launch_cg_init(const double* part, int np, double tol, int maxit, int zero_code,
                    CGScalars* cs, double* m, int nsys, hipStream_t s, long long* told = nullptr,
                    long long seq = 0);
// out[9 j + i] = mean of row 9 j + i of K4 + m[9 i + j] (tangent_homo's end:
// the mean of K4:(E_i + x_i))
void launch_mean81(const double* K4, long V, const double* m, double* partials, double* out,
                   hipStream_t s);

// up to nine field pointers (multi-RHS solves)
struct Ptr9 {
  const double* p[9];
  double* q[9];
};
// for every i < nrhs with cs[i].done == 0: the direction p_i = r_i +
// cs[i].beta p_i, then q_i = K4 : p_i (ddot42n)
struct Ptr9r {
  const double* r[9];
};
// pqpart != nullptr: also p_i . (K4:p_i) of each running right-hand side,
// per block, at pqpart[i * k4_contract_multi_blocks(V) + block].
void launch_k4_contract_multi(long V, const double* K4, const Ptr9& pp, const CGScalars* cs,
                              int nrhs, hipStream_t s, const Ptr9r& rr,
                              double* pqpart = nullptr);
int k4_contract_multi_blocks(long V);

// reductions: result -> d_out[0..nres) on device (two-stage, fixed order)
void launch_dot(const double* x, const double* y, long n, double* partials, double* d_out,
                hipStream_t s);
void launch_mean9(const double* x, long V, double* partials, double* d_out, hipStream_t s);
void launch_axpy(long n, double a, const double* x, double* y, hipStream_t s);
void launch_scal(long n, double a, double* x, hipStream_t s);
void launch_copy(long n, const double* x, double* y, hipStream_t s);
void launch_fill9(long V, const double* v9_host, double* x, hipStream_t s);
// x[0..n) = v (a store, unlike a scaling by zero, which keeps NaN or Inf)
void launch_fill(long n, double v, double* x, hipStream_t s);
void launch_fill_f32(long n, float v, float* x, hipStream_t s);
// initial material state [W][V] (mm10_init_cc_hist0, mm10_a.f:473-573, with
// mm10_init_voche, :2042-2055): zero, except Rp = I and tau_tilde = tt0
void launch_state_init(long V, int W, double tt0, double* state, hipStream_t s);
// C[j] = K4[(9 j + i) rows] copy (tangent_homo column i)
void launch_gather_k4_col(long V, int i, const double* K4, double* C, hipStream_t s);

// per-voxel update: stress update (state n+1, P, material tangent into
// tan6 [36][V]) followed by its pull-back to K4 = dP/dF
// ws: predicted slip increments [NS][V] for the warm start, or nullptr;
// warm_prev != 0: the state n+1 the call overwrites (this step's previous
// global iterate) is a warm-start candidate too
template <int NS>
void launch_drive_eps_sig(long V, const MatParams& P, const Orient<NS>* orients,
                          const int32_t* orient_id, int step, int iter, const double* Fn,
                          const double* Fn1, const double* sn, double* snp1, double* Pn1,
                          double* tan6, double* K4, const float* ws, int warm_prev,
                          long long* counters, hipStream_t s);

// warm-start network inputs of voxels e0 + r*stride (r < nrows) into
// X[r][18 + 2 NS]; with T also their converged slip increments (state n+1)
template <int NS>
void launch_mlp_features(long V, const MatParams& P, const Orient<NS>* orients, const int32_t* oid,
                         int step, const double* Fn, const double* Fn1, const double* sn,
                         const double* snp1, long e0, long stride, long nrows, float* X, float* T,
                         hipStream_t s);
// every voxel's inputs normalised with nrm ([mean | sd]) as BF16 rows of
// ninp columns (zero-padded) into Xv
template <int NS>
void launch_mlp_features_norm(long V, const MatParams& P, const Orient<NS>* orients,
                              const int32_t* oid, int step, const double* Fn, const double* Fn1,
                              const double* sn, const float* nrm, int ninp, uint16_t* Xv,
                              hipStream_t s);

int reduce_partials_count(long n);

// error text for cpfft_last_error (of the calling thread)
void set_last_error(const char* what);
// cpfft_gkdf_noalloc's scratch: the device address of the current GPU's
// copy of its static array (resolved on the first call per device; also
// from cpfft_create).  0, or a negative code with the error text set.
int noalloc_scratch_current_device(cplx** out);

}  // namespace cpfft
