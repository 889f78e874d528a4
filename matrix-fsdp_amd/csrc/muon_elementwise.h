// Element-wise stages of the Muon update: momentum, norm, scale + transpose, parameter update.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mfsdp {

constexpr int kMuonMaxPartials = 1 << 18;  // upper bound on the workgroups of a matrix in the momentum kernel (one partial sum each)
constexpr int kMaxMuonGroup = 32;          // matrices one launch carries by value in its kernel arguments

// One matrix of a launch.  `same` / `trans` receive the scaled update and its transpose: rows x cols with ld_same, cols x
// rows with ld_trans, both zero up to the next multiples of 64; either may be null.
struct MuonMatrix {
  const void* grad;
  void* buf;         // momentum buffer
  uint16_t* xraw;    // rows x cols unscaled bf16 update
  uint16_t* same;
  uint16_t* trans;
  float* partials;   // sums of squares, one per workgroup of the momentum kernel; 16-byte aligned
  int n_partials;
  int rows, cols;
  int ld_same, ld_trans;
};

struct MuonMatrices {
  int n = 0;
  float* norms = nullptr;  // one per matrix
  MuonMatrix m[kMaxMuonGroup];
};

// Workgroups (and partial sums) of a matrix of `numel` elements in muon_momentum.
int muon_momentum_partials(int64_t numel);

// buf <- lerp(buf, g, 1-mu); xraw <- bf16(nesterov ? lerp(g, buf, mu) : buf); partial sums of squares of every matrix
// (without momentum: xraw <- bf16(g)).
int muon_momentum(const MuonMatrices& g, int dtype, double momentum, int nesterov, bool with_momentum, hipStream_t stream);

// same[r][c] = bf16(x[r][c] / norm), trans[c][r] = same[r][c], with norm = max(bf16(sqrt(sum of the partials)), bf16(eps)).
int muon_scale_transpose(const MuonMatrices& g, float eps, hipStream_t stream);

// p <- p*decay - adj_lr * O (torch/optim/_muon.py:313-315).
int muon_apply(void* param, int dtype, const void* ortho, int rows, int cols, int ldo, float decay, float neg_lr,
               hipStream_t stream);

int muon_extract(void* out, const void* ortho, int rows, int cols, int ldo, hipStream_t stream);

// out <- bf16(scale * in), numel a multiple of 8 and both pointers 16-byte aligned.
int muon_scale_bf16(void* out, const void* in, int64_t numel, float scale, hipStream_t stream);

}  // namespace mfsdp
