// Owner-rank Muon update of one matrix: momentum -> Newton-Schulz (bf16 MFMA GEMMs) -> parameter update.
//
// The iteration keeps X (m x n, m <= n) and, where that is faster (stores_transposes), X^T (n x m), so that all three
// products of a step are K-contiguous "NT" GEMMs; elsewhere the update product reads X by columns:
//     A  = X X^T                    P = Q = X          (symmetric: lower-triangle tiles, mirrored store)
//     B  = b A + c A A = b A + c A A^T   P = Q = A     (symmetric)
//     X' = a X + B X                P = B, Q = X^T or X     (writes X' and, where kept, X'^T)
// Every product is rounded to bf16, as the reference's bf16 addmm / mm do.  Buffers are padded to multiples of 256 so
// the GEMM needs no edge handling; what a product reads beyond a matrix's sides along K is zero.
//
// A step's matrices do not depend on each other: up to 32 of them go through every stage as ONE launch (momentum, norm,
// scale + transpose, three products per iteration), so that small matrices fill the machine together and a step costs
// 2 or 3 + 3 x steps launches instead of that many per matrix.
#include "mfsdp_common.h"
#include "muon_elementwise.h"
#include "muon_gemm.h"

#include <algorithm>
#include <cmath>
#include <memory>
#include <new>

namespace mfsdp {
namespace {

constexpr int64_t kPad = 256;
constexpr int64_t kAlign = 256;  // byte alignment of every workspace region
constexpr int kTileK = 64;       // K of every product is rounded up to this: the operands are zero up to there

int64_t round_up(int64_t v, int64_t to) { return (v + to - 1) / to * to; }

// One matrix in the workspace.  Leading dimensions are padded to multiples of 256, so that tiles of every variant stay
// inside the buffers; only the part up to the next multiples of 64 is ever read as an operand's K or defined at all.
struct Matrix {
  int rows, cols;          // of the parameter
  int m, n, mp, np;        // short / long side and their padded sizes
  bool tall;               // rows > cols: the iteration runs on the transpose
  bool keeps_xt;           // X^T is stored beside X, see stores_transposes
  uint16_t* X[2];          // mp x np
  uint16_t* XT[2];         // np x mp
  uint16_t* A;             // mp x mp
  uint16_t* B;             // mp x mp
  int64_t bytes;
  uint16_t* xraw() const { return X[1]; }  // rows x cols unscaled bf16 update
};

bool plan_matrix(int64_t rows, int64_t cols, char* base, Matrix* w) {
  if (rows <= 0 || cols <= 0 || rows > (1 << 30) || cols > (1 << 30)) return false;
  w->rows = static_cast<int>(rows);
  w->cols = static_cast<int>(cols);
  w->tall = rows > cols;
  w->keeps_xt = true;
  w->m = static_cast<int>(std::min(rows, cols));
  w->n = static_cast<int>(std::max(rows, cols));
  w->mp = static_cast<int>(round_up(w->m, kPad));
  w->np = static_cast<int>(round_up(w->n, kPad));
  const int64_t x_bytes = round_up(static_cast<int64_t>(w->mp) * w->np * 2, kAlign);
  const int64_t a_bytes = round_up(static_cast<int64_t>(w->mp) * w->mp * 2, kAlign);
  int64_t off = 0;
  auto take = [&](int64_t bytes) { char* r = base ? base + off : nullptr; off += bytes; return reinterpret_cast<uint16_t*>(r); };
  w->X[0] = take(x_bytes);
  w->X[1] = take(x_bytes);
  w->XT[0] = take(x_bytes);
  w->XT[1] = take(x_bytes);
  w->A = take(a_bytes);
  w->B = take(a_bytes);
  w->bytes = off;
  return true;
}

// Behind the matrices of a launch: their norms and the scratch of the products.
constexpr int64_t kSharedBytes = kAlign + kGemmPartialsBytes;
static_assert(kMaxMuonGroup <= kMaxGemmGroup && kMaxMuonGroup * sizeof(float) <= kAlign, "a group travels through both kinds of launch");
// the sums of squares of the momentum kernel are consumed by the norm before the first product runs
static_assert(kMuonMaxPartials % 4 == 0 && static_cast<int64_t>(kMaxMuonGroup) * kMuonMaxPartials * 4 <= kGemmPartialsBytes,
              "the partial sums borrow the products' scratch");

// Most workspace a group is given beyond what its largest matrix needs anyway: three 12288 x 4096 matrices.
constexpr int64_t kGroupBytes = 1344ll << 20;

// Does the triangle of 256 x 256 tiles of the matrix's symmetric products occupy three quarters of the CUs?  Such a matrix
// goes through the stages on its own: others beside it would cost their workspace and gain next to nothing (15360 x 5120
// and 5120 x 13824 in bf16 together 11.14 ms with 1.4 GiB, one after the other 11.27 ms with 0.75 GiB).
bool fills_machine(const Matrix& w, int cus) {
  const int t = (w.m + 255) / 256;
  return 4 * (t * (t + 1) / 2) >= 3 * cus;
}

// A group of matrices that go through every stage of the update together, one launch per stage.
struct Group {
  int n = 0;
  Matrix w[kMaxMuonGroup];
  void* param[kMaxMuonGroup];
  float decay[kMaxMuonGroup], neg_lr[kMaxMuonGroup];
  MuonMatrices elementwise;
  GemmScratch scratch;
};

void finish_group(Group* g, char* shared) {
  g->elementwise.n = g->n;
  g->elementwise.norms = reinterpret_cast<float*>(shared);
  g->scratch.partials = shared + kAlign;
  g->scratch.partials_bytes = kGemmPartialsBytes;
  float* partials = static_cast<float*>(g->scratch.partials);
  for (int i = 0; i < g->n; ++i) {
    const Matrix& w = g->w[i];
    MuonMatrix& m = g->elementwise.m[i];
    m.xraw = w.xraw();
    // the input is rows x cols; the iteration wants the short side first
    m.same = w.tall ? w.XT[0] : w.X[0];
    m.trans = w.tall ? w.X[0] : w.XT[0];
    m.ld_same = w.tall ? w.mp : w.np;
    m.ld_trans = w.tall ? w.np : w.mp;
    m.rows = w.rows;
    m.cols = w.cols;
    m.n_partials = muon_momentum_partials(static_cast<int64_t>(w.rows) * w.cols);
    m.partials = partials;
    partials += round_up(m.n_partials, 4);  // the norm reads groups of four
  }
}

// The size of the update product.
void update_size(const Matrix& w, GemmProblem* p) {
  p->M = w.m;
  p->N = w.n;
  p->K = static_cast<int>(round_up(w.m, kTileK));
}

// Does the group store X^T beside X?  The update product can take X itself (kGemmQColumns), and the epilogues of the update
// products and the scale kernel then store one orientation of X instead of two; its walk over X is some percent slower, which
// weighs the more the longer K is, and the stores weigh the less the more rounds of tiles they spread over.
// Whole step with X^T -> without, us: 24 of 1536x1024 1248 -> 1089, a hidden2048 layer 2048 -> 1841, six of 1536x4096 in bf16 1355
// -> 1213, 3072x12288 2105 -> 1891, 5120x15360 5863 -> 5740.  It is left out
// * on 256 tiles (on 128 ones 1024x2048 226 -> 251, 1000x3000 with four smaller 316 -> 331; 64 tiles read their operands
//   straight into registers, K-contiguous);
// * where the tiles fill more than a round, so that their stores compete (200 tiles 777 -> 793; 320 1063 -> 1030, 352 1294 -> 1261);
// * up to an X of 192 MiB, about the largest that was measured to gain (200 MiB in one matrix 7494 -> 7475);
// * where kGemmQColumns takes X padded to whole tiles, which a few rows of 4 Mi elements exceed (kMaxQColumnsElements);
// * for one matrix with a short side of up to 5632 (5632x9000 4305 -> 4222, 5632x14000 6118 -> 6129; 5888x8000 4257 -> 4406,
//   8192x8192 8509 -> 8795, 10240x10240 17431 -> 18139);
// * for several where X, A and B, what an iteration hands to the next, stay within the memory-side cache of 256 MB beside what else
//   passes through it: 201e6 bytes 2440 -> 2374 (4096x4096*2), 216e6 2645 -> 2651 (3328x4160*3), 226e6 2531 -> 2461
//   (3072x3072*4); 253e6 3160 -> 3226 (3700x4000*3), 256e6 3045 -> 3128 (3200x3600*4), 327e6 4496 -> 4562 (4096x5120*3);
// * beyond that for short sides of up to 1700 (1700x1700*18 2346 -> 2333, 1536x4096*16 3314 -> 3203; 1800x1800*14 2265 -> 2303)
//   and, where X is at least twice A, of up to 2560 (2560x5120*6 4015 -> 3865, 2304x6912*5 3093 -> 3019; 2816x5632*5 3972 ->
//   4021, and with X less than twice A 2304x2880*12 3891 -> 3958).
constexpr int64_t kOneOrientationBytes = 192ll << 20;
bool stores_transposes(const Group& group) {
  GemmGroup g;
  int64_t x = 0, a = 0, tiles = 0, padded = 0;  // x, a: bytes of every X and A
  int side = 0;
  g.n = group.n;
  for (int i = 0; i < g.n; ++i) {
    const Matrix& w = group.w[i];
    g.problem[i] = GemmProblem{};
    update_size(w, &g.problem[i]);
    x += static_cast<int64_t>(w.m) * w.n * 2;
    a += static_cast<int64_t>(w.m) * w.m * 2;
    tiles += static_cast<int64_t>((w.m + 255) / 256) * ((w.n + 255) / 256);
    padded = std::max(padded, static_cast<int64_t>(w.mp) * w.np);
    side = std::max(side, w.m);
  }
  const bool gains = g.n == 1 ? side <= 5632 : x + 2 * a <= 230'000'000 || side <= 1700 || (side <= 2560 && x >= 2 * a);
  return !gains || x > kOneOrientationBytes || padded > kMaxQColumnsElements || 4 * tiles < 5 * device_cu_count() ||
         !on_256_tiles(gemm_plan(g, group.scratch));
}

void choose_transposes(Group* group, int steps) {
  if (steps == 0 || stores_transposes(*group)) return;  // without a product the result is taken from either
  for (int i = 0; i < group->n; ++i) {
    Matrix& w = group->w[i];
    w.keeps_xt = false;
    (w.tall ? group->elementwise.m[i].same : group->elementwise.m[i].trans) = nullptr;
  }
}

// Newton-Schulz on the updates already sitting in xraw with their partial sums of squares.  With `update_dtype` >= 0 and
// at least one step the last product writes the parameters themselves; otherwise O is left in X[steps & 1] (wide) or
// XT[steps & 1] (tall).
int run_newton_schulz(Group& group, float a, float b, float c, int steps, float eps, bool shared, int update_dtype, hipStream_t stream) {
  choose_transposes(&group, steps);
  if (int rc = muon_scale_transpose(group.elementwise, eps, stream)) return rc;
  GemmGroup g;
  g.n = group.n;
  GemmPlan gram, poly, update;  // made in the first iteration
  for (int s = 0; s < steps; ++s) {
    const int cur = s & 1, nxt = cur ^ 1;
    g.alpha = 1.0f; g.beta = 0.0f; g.symmetric = 1; g.shared = shared;
    for (int i = 0; i < group.n; ++i) {
      const Matrix& w = group.w[i];
      GemmProblem& p = g.problem[i] = GemmProblem{};
      p.P = w.X[cur]; p.Q = w.X[cur]; p.C = w.A;
      p.M = w.m; p.N = w.m; p.K = static_cast<int>(round_up(w.n, kTileK));
      p.ldp = w.np; p.ldq = w.np; p.ldc = w.mp;
    }
    if (s == 0) gram = gemm_plan(g, group.scratch);
    if (int rc = gemm_nt_bf16(g, gram, group.scratch, stream)) return rc;
    if (c == 0.0f) {
      // addmm with alpha = 0 leaves beta * A (the product is not formed at all, torch/optim/_muon.py:61 with a
      // quadratic polynomial); the GEMM's D path needs alpha != 0 (it adds (beta / alpha) D to the accumulators)
      for (int i = 0; i < group.n; ++i)
        if (int rc = muon_scale_bf16(group.w[i].B, group.w[i].A, static_cast<int64_t>(group.w[i].mp) * group.w[i].mp, b, stream)) return rc;
    } else {
      g.alpha = c; g.beta = b;
      for (int i = 0; i < group.n; ++i) {
        const Matrix& w = group.w[i];
        GemmProblem& p = g.problem[i] = GemmProblem{};
        p.P = w.A; p.Q = w.A; p.D = w.A; p.C = w.B;  // A is symmetric: D^T is Q
        p.M = w.m; p.N = w.m; p.K = static_cast<int>(round_up(w.m, kTileK));
        p.ldp = w.mp; p.ldq = w.mp; p.ldd = w.mp; p.ldc = w.mp;
      }
      if (s == 0) poly = gemm_plan(g, group.scratch);
      if (int rc = gemm_nt_bf16(g, poly, group.scratch, stream)) return rc;
    }
    g.alpha = 1.0f; g.beta = a; g.symmetric = 0; g.shared = 0;
    for (int i = 0; i < group.n; ++i) {
      const Matrix& w = group.w[i];
      GemmProblem& p = g.problem[i] = GemmProblem{};
      p.P = w.B; p.Q = w.XT[cur]; p.D = w.X[cur]; p.C = w.X[nxt]; p.CT = w.XT[nxt];  // Q = X^T
      update_size(w, &p);
      p.ldp = w.mp; p.ldq = w.mp; p.ldd = w.np; p.ldc = w.np; p.ldct = w.mp;
      if (!w.keeps_xt) {
        p.Q = w.X[cur];
        p.ldq = w.np;
        p.flags |= kGemmQColumns;
        if (s + 1 < steps) p.CT = nullptr;
      }
      if (s + 1 == steps) {  // the last step only has to leave O in the parameter's orientation
        if (w.tall) p.flags |= kGemmSkipC;
        else p.CT = nullptr;
        if (update_dtype >= 0) {  // ... or take it straight into the parameter: O is never stored
          g.update_dtype = update_dtype;
          p.update_param = group.param[i];
          p.update_decay = group.decay[i];
          p.update_neg_lr = group.neg_lr[i];
          if (w.tall) p.flags |= kGemmUpdateTransposed;
        }
      }
    }
    if (s == 0) update = gemm_plan(g, group.scratch);
    if (int rc = gemm_nt_bf16(g, update, group.scratch, stream)) return rc;
  }
  return MFSDP_OK;
}

const uint16_t* result_of(const Matrix& w, int steps) { return w.tall ? w.XT[steps & 1] : w.X[steps & 1]; }

// everything that can be refused is refused before the first kernel is enqueued (a step must not be left half applied)
int check_iteration(float a, float b, float c, int steps) {
  if (!std::isfinite(a) || !std::isfinite(b) || !std::isfinite(c) || (c != 0.0f && !std::isfinite(b / c)))
    return fail(MFSDP_ERR_INVALID, "Newton-Schulz coefficients must be finite (and b / c representable), got (%g, %g, %g)", a, b, c);
  if (steps < 0 || steps >= 100) return fail(MFSDP_ERR_INVALID, "Number of steps must be less than 100 for computational efficiency");
  return MFSDP_OK;
}

int check_matrix(int64_t rows, int64_t cols, int steps, Matrix* w) {
  if (!plan_matrix(rows, cols, nullptr, w))
    return fail(MFSDP_ERR_INVALID, "Input tensor gradient must be a 2D matrix with positive sizes, got %lld x %lld",
                static_cast<long long>(rows), static_cast<long long>(cols));
  if (steps > 0 && w->np > kMaxGemmLeading)  // of the products' operands; without a product there is no limit
    return fail(MFSDP_ERR_UNSUPPORTED, "leading dimensions beyond 2^22 elements, got %lld x %lld", static_cast<long long>(rows), static_cast<long long>(cols));
  return MFSDP_OK;
}

int check_workspace(const void* workspace, int64_t have, int64_t need) {
  if (workspace == nullptr || have < need)
    return fail(MFSDP_ERR_INVALID, "workspace of %lld bytes needed, got %lld", static_cast<long long>(need), static_cast<long long>(have));
  if (reinterpret_cast<uintptr_t>(workspace) % kAlign) return fail(MFSDP_ERR_INVALID, "workspace must be %lld-byte aligned", static_cast<long long>(kAlign));
  return MFSDP_OK;
}

// What the matrices of one step have in common.
struct StepArgs {
  int dtype;
  double momentum;
  int nesterov;
  float a, b, c;
  int steps;
  float eps;
  bool shared;
};

int check_step(const StepArgs& s) {
  if (int rc = check_iteration(s.a, s.b, s.c, s.steps)) return rc;
  if (s.dtype != MFSDP_F32 && s.dtype != MFSDP_BF16) return fail(MFSDP_ERR_INVALID, "dtype must be f32 or bf16");
  if (!(s.momentum >= 0.0)) return fail(MFSDP_ERR_INVALID, "momentum should be >= 0 but is: %g", s.momentum);
  return MFSDP_OK;
}

int check_tensors(const void* param, const void* grad, const void* buf, int dtype, double lr, double weight_decay) {
  if (!param || !grad || !buf) return fail(MFSDP_ERR_INVALID, "null tensor pointer");
  const uintptr_t elem = dtype == MFSDP_F32 ? 4 : 2;
  if ((reinterpret_cast<uintptr_t>(param) | reinterpret_cast<uintptr_t>(grad) | reinterpret_cast<uintptr_t>(buf)) % elem)
    return fail(MFSDP_ERR_INVALID, "tensor pointers must be aligned to their elements");
  if (!(lr >= 0.0)) return fail(MFSDP_ERR_INVALID, "Learning rate should be >= 0 but is: %g", lr);
  if (!(weight_decay >= 0.0)) return fail(MFSDP_ERR_INVALID, "weight decay should be >= 0 but is: %g", weight_decay);
  return MFSDP_OK;
}

// the host scalars are doubles, as in Python: 1 - lr * wd and -adjusted_lr are rounded to fp32 once, where the tensor
// operation takes them
void add_to_group(Group* g, const Matrix& w, void* param, const void* grad, void* buf, double lr, double weight_decay, double adjusted_lr) {
  g->w[g->n] = w;
  g->param[g->n] = param;
  g->decay[g->n] = static_cast<float>(1.0 - lr * weight_decay);
  g->neg_lr[g->n] = static_cast<float>(-adjusted_lr);
  g->elementwise.m[g->n].grad = grad;
  g->elementwise.m[g->n].buf = buf;
  ++g->n;
}

int run_step(Group* g, char* shared, const StepArgs& s, hipStream_t stream) {
  finish_group(g, shared);
  if (int rc = muon_momentum(g->elementwise, s.dtype, s.momentum, s.nesterov, true, stream)) return rc;
  if (int rc = run_newton_schulz(*g, s.a, s.b, s.c, s.steps, s.eps, s.shared, s.dtype, stream)) return rc;
  if (s.steps > 0) return MFSDP_OK;  // the last product has updated the parameters
  for (int i = 0; i < g->n; ++i) {
    const Matrix& w = g->w[i];
    if (int rc = muon_apply(g->param[i], s.dtype, result_of(w, 0), w.rows, w.cols, w.tall ? w.mp : w.np, g->decay[i], g->neg_lr[i], stream)) return rc;
  }
  return MFSDP_OK;
}

// A matrix of a call that waits for its group.
struct Pending {
  bool alone;  // see fills_machine
  int64_t bytes;
  int64_t job;
};

// The matrices of a call.  Without host memory for them `data` is null: nothing of this may throw out of an extern "C" function.
struct PendingList {
  explicit PendingList(int64_t n) : data(new (std::nothrow) Pending[n]), cus(device_cu_count()) {}
  void add(const Matrix& w) {
    data[size] = Pending{fills_machine(w, cus), w.bytes, size};
    ++size;
  }
  // Those that go alone first, then the largest first, so that a group holds matrices of like size; equals in the order given.
  void sort() {
    std::sort(data.get(), data.get() + size, [](const Pending& x, const Pending& y) {
      return x.alone != y.alone ? x.alone : x.bytes != y.bytes ? x.bytes > y.bytes : x.job < y.job;
    });
  }
  // The group that starts at `first` ends before the returned position: as many as one launch carries and `room` holds, at
  // least one.
  int64_t group_end(int64_t first, int64_t room, int64_t* bytes) const {
    int64_t end = first + 1;
    *bytes = data[first].bytes;
    while (!data[first].alone && end < size && end - first < kMaxMuonGroup && *bytes + data[end].bytes <= room) *bytes += data[end++].bytes;
    return end;
  }
  std::unique_ptr<Pending[]> data;
  int64_t size = 0;
  int cus;
};

int out_of_host_memory(int64_t n) { return fail(MFSDP_ERR_UNSUPPORTED, "out of host memory for %lld matrices", static_cast<long long>(n)); }

// Flops the products of one Newton-Schulz step of `n` matrices that share their launches execute.
int64_t executed_flops(const Matrix* w, int n, bool shared) {
  GemmGroup gram, poly, update;
  gram.n = poly.n = update.n = n;
  gram.symmetric = poly.symmetric = 1;
  gram.shared = poly.shared = shared;
  auto size = [](GemmProblem* p, int rows, int cols, int k) {
    *p = GemmProblem{};
    p->M = rows;
    p->N = cols;
    p->K = static_cast<int>(round_up(k, kTileK));
  };
  for (int i = 0; i < n; ++i) {
    size(&gram.problem[i], w[i].m, w[i].m, w[i].n);
    size(&poly.problem[i], w[i].m, w[i].m, w[i].m);
    size(&update.problem[i], w[i].m, w[i].n, w[i].m);
  }
  return gemm_nt_executed_flops(gram) + gemm_nt_executed_flops(poly) + gemm_nt_executed_flops(update);
}

}  // namespace
}  // namespace mfsdp

using namespace mfsdp;

extern "C" int64_t mfsdp_muon_workspace_bytes(int64_t rows, int64_t cols) {
  Matrix w;
  return plan_matrix(rows, cols, nullptr, &w) ? w.bytes + kSharedBytes : 0;
}

extern "C" int64_t mfsdp_muon_many_workspace_bytes(int64_t n, const int64_t* rows, const int64_t* cols) {
  if (n <= 0 || rows == nullptr || cols == nullptr) return 0;
  PendingList order(n);
  if (!order.data) return out_of_host_memory(n), 0;
  for (int64_t i = 0; i < n; ++i) {
    Matrix w;
    if (!plan_matrix(rows[i], cols[i], nullptr, &w)) return 0;
    order.add(w);
  }
  order.sort();
  int64_t largest = 0;
  for (int64_t next = 0; next < n;) {
    int64_t bytes = 0;
    next = order.group_end(next, kGroupBytes, &bytes);
    largest = std::max(largest, bytes);
  }
  return largest + kSharedBytes;
}

extern "C" int64_t mfsdp_muon_executed_flops(int64_t rows, int64_t cols, int steps, int flags) {
  Matrix w;
  if (steps < 0 || !plan_matrix(rows, cols, nullptr, &w)) return 0;
  return steps * executed_flops(&w, 1, (flags & MFSDP_MUON_SHARED_MACHINE) != 0);
}

extern "C" int64_t mfsdp_muon_many_executed_flops(int64_t n, const int64_t* rows, const int64_t* cols, int steps, int64_t workspace_bytes) {
  if (n <= 0 || rows == nullptr || cols == nullptr || steps < 0) return 0;
  PendingList order(n);
  if (!order.data) return out_of_host_memory(n), 0;
  for (int64_t i = 0; i < n; ++i) {
    Matrix w;
    if (!plan_matrix(rows[i], cols[i], nullptr, &w) || w.bytes + kSharedBytes > workspace_bytes) return 0;
    order.add(w);
  }
  order.sort();
  int64_t flops = 0;
  for (int64_t next = 0; next < n;) {
    Matrix w[kMaxMuonGroup];
    int64_t bytes = 0;
    int count = 0;
    for (const int64_t end = order.group_end(next, workspace_bytes - kSharedBytes, &bytes); next < end; ++next)
      plan_matrix(rows[order.data[next].job], cols[order.data[next].job], nullptr, &w[count++]);
    flops += executed_flops(w, count, false);
  }
  return steps * flops;
}

extern "C" int mfsdp_newton_schulz(const void* update, int update_dtype, int64_t rows, int64_t cols, float a, float b, float c,
                                   int steps, float eps, void* out_bf16, void* workspace, int64_t workspace_bytes, void* stream) {
  Group g;
  if (int rc = check_iteration(a, b, c, steps)) return rc;
  if (int rc = check_matrix(rows, cols, steps, &g.w[0])) return rc;
  if (int rc = check_workspace(workspace, workspace_bytes, g.w[0].bytes + kSharedBytes)) return rc;
  if (update_dtype != MFSDP_F32 && update_dtype != MFSDP_BF16) return fail(MFSDP_ERR_INVALID, "update dtype must be f32 or bf16");
  if (!update || !out_bf16) return fail(MFSDP_ERR_INVALID, "null tensor pointer");
  if (reinterpret_cast<uintptr_t>(update) % (update_dtype == MFSDP_F32 ? 4 : 2)) return fail(MFSDP_ERR_INVALID, "update must be aligned to its elements");
  hipStream_t s = as_stream(stream);
  char* base = static_cast<char*>(workspace);
  Matrix w;
  plan_matrix(rows, cols, base, &w);
  add_to_group(&g, w, nullptr, update, nullptr, 0.0, 0.0, 0.0);
  finish_group(&g, base + w.bytes);
  if (int rc = muon_momentum(g.elementwise, update_dtype, 0.0, 0, false, s)) return rc;
  if (int rc = run_newton_schulz(g, a, b, c, steps, eps, false, -1, s)) return rc;
  return muon_extract(out_bf16, result_of(w, steps), w.rows, w.cols, w.tall ? w.mp : w.np, s);
}

extern "C" int mfsdp_muon_step_ex(void* param, const void* grad, void* momentum_buf, int dtype, int64_t rows, int64_t cols, double lr,
                                  double weight_decay, double momentum, int nesterov, float a, float b, float c, int steps, float eps,
                                  double adjusted_lr, int flags, void* workspace, int64_t workspace_bytes, void* stream) {
  const StepArgs s{dtype, momentum, nesterov, a, b, c, steps, eps, (flags & MFSDP_MUON_SHARED_MACHINE) != 0};
  Matrix w;
  if (int rc = check_step(s)) return rc;
  if (int rc = check_matrix(rows, cols, steps, &w)) return rc;
  if (int rc = check_workspace(workspace, workspace_bytes, w.bytes + kSharedBytes)) return rc;
  if (int rc = check_tensors(param, grad, momentum_buf, dtype, lr, weight_decay)) return rc;
  if (flags & ~MFSDP_MUON_SHARED_MACHINE) return fail(MFSDP_ERR_INVALID, "unknown flags 0x%x", flags);
  char* base = static_cast<char*>(workspace);
  plan_matrix(rows, cols, base, &w);
  Group g;
  add_to_group(&g, w, param, grad, momentum_buf, lr, weight_decay, adjusted_lr);
  return run_step(&g, base + w.bytes, s, as_stream(stream));
}

extern "C" int mfsdp_muon_step(void* param, const void* grad, void* momentum_buf, int dtype, int64_t rows, int64_t cols, double lr,
                               double weight_decay, double momentum, int nesterov, float a, float b, float c, int steps, float eps,
                               double adjusted_lr, void* workspace, int64_t workspace_bytes, void* stream) {
  return mfsdp_muon_step_ex(param, grad, momentum_buf, dtype, rows, cols, lr, weight_decay, momentum, nesterov, a, b, c, steps, eps,
                            adjusted_lr, 0, workspace, workspace_bytes, stream);
}

extern "C" int mfsdp_muon_step_many(int64_t n, const mfsdp_muon_job* jobs, int dtype, double momentum, int nesterov, float a, float b,
                                    float c, int steps, float eps, void* workspace, int64_t workspace_bytes, void* stream) {
  if (n < 0 || (n > 0 && jobs == nullptr)) return fail(MFSDP_ERR_INVALID, "jobs is null or n negative");
  if (n == 0) return MFSDP_OK;
  const StepArgs s{dtype, momentum, nesterov, a, b, c, steps, eps, false};
  if (int rc = check_step(s)) return rc;
  PendingList order(n);
  if (!order.data) return out_of_host_memory(n);
  int64_t largest = 0;
  for (int64_t i = 0; i < n; ++i) {
    Matrix w;
    if (int rc = check_matrix(jobs[i].rows, jobs[i].cols, steps, &w)) return rc;
    if (int rc = check_tensors(jobs[i].param, jobs[i].grad, jobs[i].momentum_buf, dtype, jobs[i].lr, jobs[i].weight_decay)) return rc;
    order.add(w);
    largest = std::max(largest, w.bytes);
  }
  if (int rc = check_workspace(workspace, workspace_bytes, largest + kSharedBytes)) return rc;
  order.sort();
  char* base = static_cast<char*>(workspace);
  for (int64_t next = 0; next < n;) {
    Group g;
    int64_t bytes = 0, used = 0;
    for (const int64_t end = order.group_end(next, workspace_bytes - kSharedBytes, &bytes); next < end; ++next) {
      const mfsdp_muon_job& job = jobs[order.data[next].job];
      Matrix w;
      plan_matrix(job.rows, job.cols, base + used, &w);
      add_to_group(&g, w, job.param, job.grad, job.momentum_buf, job.lr, job.weight_decay, job.adjusted_lr);
      used += w.bytes;
    }
    if (int rc = run_step(&g, base + used, s, as_stream(stream))) return rc;
  }
  return MFSDP_OK;
}

extern "C" int mfsdp_gemm_nt_bf16(const void* p, const void* q, void* c, int m, int n, int k, void* partials, int64_t partials_bytes, void* stream) {
  if (m % 256 || n % 256) return fail(MFSDP_ERR_INVALID, "mfsdp_gemm_nt_bf16: M=%d and N=%d must be multiples of 256", m, n);
  GemmGroup g;
  g.n = 1;
  GemmProblem& a = g.problem[0] = GemmProblem{};
  a.P = p; a.Q = q; a.C = c;
  a.M = m; a.N = n; a.K = k;
  a.ldp = k; a.ldq = k; a.ldc = n;
  GemmScratch scratch;
  scratch.partials = partials;
  scratch.partials_bytes = partials ? partials_bytes : 0;
  return gemm_nt_bf16(g, gemm_plan(g, scratch), scratch, as_stream(stream));
}

extern "C" void mfsdp_set_muon_tuning(int general_variant, int symmetric_variant, int group_m, int split_remainder,
                                      int max_splits) {
  GemmTuning t = get_gemm_tuning();
  if (general_variant > 0) t.general_variant = general_variant;
  if (symmetric_variant > 0) t.symmetric_variant = symmetric_variant;
  if (group_m > 0) t.group_m = group_m;
  if (split_remainder > 0) t.split_remainder = split_remainder == 1;
  if (max_splits > 0) t.max_splits = max_splits;
  set_gemm_tuning(t);
}
