// Internal state of a cloudsc_mlp_t, shared by the MLP and the surrogate translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

namespace mlp {
typedef __bf16 bf16;
}  // namespace mlp

struct cloudsc_mlp {
  int nl = 0;                   // number of linear layers (hidden layers + 1)
  std::vector<int> din, dout;   // per layer
  int max_batch = 0;
  long step = 0;
  // per layer
  std::vector<float*> w, b, mw, vw, mb, vb, gw, gb;
  std::vector<mlp::bf16*> wb;
  // per hidden layer l (0..nl-2): Z_l (fp32), A_l (mlp::bf16) -- A_l is the input of layer l+1
  std::vector<float*> z;
  std::vector<mlp::bf16*> a;
  mlp::bf16 *g0 = nullptr, *g1 = nullptr;  // gradient ping-pong buffers
  float* y = nullptr;           // output [max_batch x n_out]
  float* loss = nullptr;        // device scalar
  float* ws = nullptr;          // partial products of split weight-gradient contractions
  size_t ws_elems = 0;
  std::vector<void*> allocs;
};

namespace mlp {
// Forward pass over M rows of x (bf16 [M x n_in]) into y (fp32 [M x n_out]); with a target t (fp32 [M x n_out]) it
// keeps what backward needs and forms the loss weighted by wgt.
hipError_t forward(cloudsc_mlp* m, const bf16* x, int M, float* y, const float* t, const float* wgt, hipStream_t s);
// cloudsc_mlp_train_step without the transposed input.
int train_step(cloudsc_mlp* m, const bf16* x, const float* t, const float* wgt, int M, float lr, hipStream_t s);
}  // namespace mlp
