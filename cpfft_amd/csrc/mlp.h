// mlp.h -- buffers and launchers of the warm-start network (mlp.hip) and of
// the per-voxel feature / warm-start kernels (cpfft_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cpfft {

constexpr int kMlpHid = 128;
constexpr int kMlpMaxOut = 24;  // slip systems of the largest set the warm start serves

// Sizes of the network for a crystal of ns slip systems: nin = 18 + 2 ns
// inputs (see voxel_features), nout = ns outputs.  Flat FP32 parameter
// vector [W1 (128 x nin) | b1 | W2 (128 x 128) | b2 | W3 (nout x 128) | b3],
// W rows the output units; normalisation [mean_x | sd_x | mean_t | sd_t].
struct MlpDims {
  int nin = 0, nout = 0;
  long offW1 = 0, offB1 = 0, offW2 = 0, offB2 = 0, offW3 = 0, offB3 = 0, nparam = 0;
  int nnorm = 0;
};
inline MlpDims mlp_dims(int ns) {
  MlpDims d;
  d.nin = 18 + 2 * ns;
  d.nout = ns;
  d.offW1 = 0;
  d.offB1 = d.offW1 + (long)kMlpHid * d.nin;
  d.offW2 = d.offB1 + kMlpHid;
  d.offB2 = d.offW2 + (long)kMlpHid * kMlpHid;
  d.offW3 = d.offB2 + kMlpHid;
  d.offB3 = d.offW3 + (long)d.nout * kMlpHid;
  d.nparam = d.offB3 + d.nout;
  d.nnorm = 2 * d.nin + 2 * d.nout;
  return d;
}
// inputs padded for the inference kernel's K steps of 32
inline int mlp_nin_pad(int nin) { return (nin + 31) / 32 * 32; }

struct MlpBuffers {
  MlpDims d;
  float* params = nullptr;  // FP32 master weights
  uint16_t* pbf = nullptr;  // BF16 copy used by the GEMMs
  float* grads = nullptr;
  float* m = nullptr;       // Adam moments
  float* v = nullptr;
  float* norm = nullptr;
  float* logX = nullptr;    // logged raw features [cap][nin]
  float* logT = nullptr;    // logged converged slip increments [cap][nout]
  long cap = 0;
  int rows = 0;             // batch capacity of the training buffers
  float* Xf = nullptr;      // [rows][nin] normalised FP32 inputs staged from the host
  float* Tb = nullptr;      // [rows][nout] normalised targets
  float* Y = nullptr;       // [rows][nout] network outputs
  uint16_t* pk = nullptr;   // packed BF16 weights of the training step (mlp_pack_len)
  uint16_t* gT = nullptr;   // operands of the weight gradients (mlp_grad_bf16)
  float* fT = nullptr;      // back-propagated errors for the bias gradients (mlp_grad_f32)
  double* part = nullptr;   // loss partial sums [mlp_row_blocks(rows)]
  double* stat = nullptr;   // column statistics (mlp_stat_doubles)
  uint16_t* Xv = nullptr;   // normalised BF16 inputs of every voxel [V][mlp_nin_pad(nin)]
  float* ws = nullptr;      // predicted slip increments for the warm start [nout][V]
};

// BF16 copy of the weights for the inference kernel (pbf)
void mlp_weights_to_bf16(const MlpBuffers& b, hipStream_t s);
// packed BF16 copies for the training step (pk); mlp_train_step keeps them
// current, so once before the first step after a change of params
long mlp_pack_len(const MlpDims& d);
void mlp_pack_weights(const MlpBuffers& b, hipStream_t s);
// rows per launch are split into blocks of 32, each with a partial loss
int mlp_row_blocks(int rows);
long mlp_grad_bf16(const MlpDims& d, int rows);
long mlp_grad_f32(const MlpDims& d, int rows);
// Y[rows][nout] = network(Xf) (normalised units)
void mlp_forward(const MlpBuffers& b, int rows, const float* Xf, float* Y, hipStream_t s);
// gradient of mean((Y - T)^2) over rows x nout into b.grads, partial sums of
// (Y - T)^2 into b.part[0..mlp_row_blocks(rows))
void mlp_grad(const MlpBuffers& b, int rows, const float* Xf, const float* Tf, hipStream_t s);
// one Adam step (step number t, learning rate lr) on rows drawn from the
// log's first count pairs; partial losses as mlp_grad's
void mlp_train_step(const MlpBuffers& b, int rows, long count, uint32_t seed, uint32_t step,
                    float lr, long t, hipStream_t s);
long mlp_stat_doubles();
void mlp_stats(const MlpBuffers& b, long count, hipStream_t s);
// Inference over all voxels in one launch: ws[k][e] = the network's output
// k for the normalised inputs Xv[e] (row stride mlp_nin_pad(nin)),
// denormalised (the weights must be in pbf).  BF16 operands, FP32
// accumulation, the rounding points of mlp_forward.
void mlp_infer(const MlpBuffers& b, long V, hipStream_t s);

}  // namespace cpfft
