// bf16 MFMA GEMM used by the Newton-Schulz iteration (gfx950).  Internal to libmfsdp_hip.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mfsdp {

// One product C = bf16( alpha * (P * Q^T) + beta * D ), fp32 accumulation.
//   P: M x K row-major (ldp), Q: N x K row-major (ldq), D / C: M x N row-major (ldd / ldc).
//   K is a multiple of 64.  M and N are what the result needs; tiles cover them rounded up to a tile, so the memory
//   behind C, CT, D, P and Q must hold rows and columns up to the next multiple of 256.  What lies beyond M and N in the
//   operands may be anything: it only reaches results beyond M and N, which nobody reads (K never extends into them).
//   D may be null (beta ignored); with D, Q must hold its transpose: Q[n][k] == D[k][n] for k < K, where K covers M
//   (whole tiles pick their D values out of the Q slabs on their way through LDS; the fix-up of K-split pieces reads D
//   itself).  CT, when non-null, also receives the transpose: CT[n][m] = C[m][n] (ldct); with kGemmSkipC only CT is written.
// Parameter update in the epilogue (the last product of a Muon step): when update_param is set, nothing is stored to
// C / CT; every element o = bf16(alpha P Q^T + beta D) of the M x N result instead goes into
//     param <- round(param * update_decay) + update_neg_lr * o        (torch/optim/_muon.py:313-315)
// on the contiguous row-major parameter (M x N, or N x M with kGemmUpdateTransposed).  General products only.
//
// kGemmQColumns: Q is given as K x N row-major (ldq), rows beyond M taken as zero, K spanning M, at most kMaxQColumnsElements of
// it; general products on 256 tiles (gemm_plan takes no others for them).  D is then the same matrix.
enum GemmFlags {
  kGemmSkipC = 1,
  kGemmUpdateTransposed = 2,
  kGemmQColumns = 4,
};
struct GemmProblem {
  const void* P;
  const void* Q;
  const void* D;
  void* C;
  void* CT;
  void* update_param;
  int M, N, K;
  int ldp, ldq, ldd, ldc, ldct;
  float update_decay, update_neg_lr;
  int flags;
  // filled by the launch: K pieces per split tile, first partial tile of the problem in the scratch
  int splits, partial_base;
};

constexpr int kMaxGemmLeading = 1 << 22;  // largest leading dimension of P and Q: a tile's rows are reached by 31-bit byte offsets
constexpr int64_t kMaxQColumnsElements = (1 << 30) - 1;  // M rounded up to whole tiles times ldq: 31-bit byte offsets again
constexpr int kMaxGemmGroup = 32;  // problems one launch carries by value in its kernel arguments

// Products of one launch.  symmetric: every P*Q^T is known to be symmetric (M == N); only tiles on or below the diagonal
// are computed and each off-diagonal tile is also written mirrored into C.
struct GemmGroup {
  int n = 0;
  float alpha = 1.0f, beta = 0.0f;
  int symmetric = 0;
  int update_dtype = 0;  // of the parameters (MFSDP_F32 / MFSDP_BF16)
  int shared = 0;        // other matrices' products run beside this launch of one problem on other streams: a symmetric product
                         // then takes the 256 x 256 tiles even where their triangle fills only part of the CUs
  GemmProblem problem[kMaxGemmGroup];
};

// Device scratch for the K-split pieces of the last partial round of tiles (fp32 partial tiles).
struct GemmScratch {
  void* partials = nullptr;
  int64_t partials_bytes = 0;
};
constexpr int64_t kGemmPartialsBytes = 64ll << 20;

// Tile variants: 1 = 256 x 256 tile / 8 waves / one workgroup per CU, 2 = 128 x 128 tile / 4 waves / two per CU,
// 4 = 64 x 64 tile / K cut among 8 waves, 3 = whichever is expected to be faster for the launch at hand.
struct GemmTuning {
  int general_variant = 3;
  int symmetric_variant = 3;
  int group_m = 4;            // general products: tile rows walked together (the workgroups of one XCD share their P panels)
  int split_remainder = 1;    // split the tiles of the last partial round along K
  int max_splits = 16;
};
void set_gemm_tuning(const GemmTuning& tuning);
GemmTuning get_gemm_tuning();

// Flops the kernels execute for these products with the current tuning: 2 * tile area * K per computed tile (a symmetric
// product computes the tiles on or below the diagonal only).
int64_t gemm_nt_executed_flops(const GemmGroup& group);

// How a launch runs: tile variant, the problems in launch order (longest K first), how many of a problem's tiles are cut
// along K and into how many pieces.  It depends on the sizes only: one plan serves every iteration of a step.
struct GemmPlan {
  int variant = 0;
  double us = 0.0;  // expected
  int order[kMaxGemmGroup];
  int split_tiles[kMaxGemmGroup], splits[kMaxGemmGroup];  // by position in `order`
};
GemmPlan gemm_plan(const GemmGroup& group, const GemmScratch& scratch);
bool on_256_tiles(const GemmPlan& plan);

// Enqueues the products on `stream` as one launch (and a fix-up launch when tiles are split along K); returns an MFSDP_*
// status.  `plan` is gemm_plan's for a group of these sizes.
int gemm_nt_bf16(const GemmGroup& group, const GemmPlan& plan, const GemmScratch& scratch, hipStream_t stream);

}  // namespace mfsdp
