// The host side of the training path: output allocation, argument checks and
// launches of libmingru_hip's entry points on torch tensors, one Python call
// per operation or per block pass.
//
// Why: a block of the bf16 training path issues 9 to 16 launches forward and
// backward. Issued one by one from Python (ctypes call, torch.empty, stride
// and pointer reads, about 9 us each) they took 180 to 340 us of host time,
// more than the GPU time of every block up to about 2000 rows and half of a
// training step's; from here a launch costs 2 to 3 us. The maths stays in the
// kernels and autograd stays in Python (blocks.py, linear.py, norm.py,
// scan.py): these functions are the bodies of its Functions.
//
// Every function takes the handle of the current HIP stream and launches on
// it; outputs and workspaces come from torch's caching allocator, so nothing
// outlives a call here. The GIL is released while a call runs.

#include <torch/extension.h>

#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>
#include <vector>

#include "mingru_hip.h"

namespace {

using at::Tensor;
typedef std::optional<Tensor> Opt;

struct MgError : std::runtime_error {
  using std::runtime_error::runtime_error;
};
py::object* g_error = nullptr;  // gruboros_amd._lib.MingruHipError

[[noreturn]] void fail(const std::string& m) { throw MgError(m); }
void check(int rc, const char* what) {
  if (rc) fail(std::string(what) + " failed (code " + std::to_string(rc) + "): " + mg_last_error());
}

constexpr float kEps = 1.1920928955078125e-07f;  // torch.finfo(float32).eps, nn.RMSNorm's for fp32

int code(const Tensor& t) {
  if (t.scalar_type() == at::kFloat) return MG_F32;
  if (t.scalar_type() == at::kBFloat16) return MG_BF16;
  fail(std::string("unsupported dtype ") + c10::toString(t.scalar_type()) +
       ": the MI355X kernels take float32 and bfloat16 (cast a float16 model with .to(torch.bfloat16) instead)");
}
void need_cuda(const Tensor& t) {
  if (!t.is_cuda())
    fail("libmingru_hip kernels run on the GPU only; got a tensor on " + t.device().str() +
         ". There is no CPU path in the product; the CPU restatement of the reference lives in oracle/ for tests.");
}
Tensor make(at::IntArrayRef size, at::ScalarType type, const Tensor& like) {
  return at::empty(size, like.options().dtype(type).requires_grad(false));
}
Tensor bytes(size_t n, const Tensor& like) { return make({static_cast<int64_t>(n)}, at::kByte, like); }
// Pointers for the kernels: every tensor is checked to be on the GPU, and the
// fp32 ones to be fp32, where its pointer is taken.
void* ptr(const Tensor& t) {
  need_cuda(t);
  return t.data_ptr();
}
void* ptr(const Opt& t) { return t ? ptr(*t) : nullptr; }
float* fp(const Tensor& t) {
  if (t.scalar_type() != at::kFloat) fail(std::string("expected a float32 tensor, got ") + c10::toString(t.scalar_type()));
  return static_cast<float*>(ptr(t));
}
float* fp(const Opt& t) { return t ? fp(*t) : nullptr; }
// a dense vector of n fp32 values (a bias, a norm weight)
float* vec(const Tensor& t, int64_t n, const char* name) {
  if (t.numel() != n || !t.is_contiguous()) fail(std::string(name) + ": expected " + std::to_string(n) + " contiguous float32 values");
  return fp(t);
}
int16_t* h16(const Tensor& t) { return static_cast<int16_t*>(ptr(t)); }
void* st(int64_t stream) { return reinterpret_cast<void*>(stream); }
bool deterministic() { return at::globalContext().deterministicAlgorithms(); }

int64_t row_stride(const Tensor& t, const char* name) {
  if (t.dim() != 2 || t.stride(1) != 1) {
    std::string s = std::string(name) + ": expected a 2-D tensor with unit inner stride, got shape ";
    for (int64_t i = 0; i < t.dim(); ++i) s += std::to_string(t.size(i)) + (i + 1 < t.dim() ? "x" : "");
    fail(s);
  }
  return t.stride(0);
}

// A matrix operand of a product: rows x cols exactly, so that a launch reads and writes inside it
// (the C ABI sees leading dimensions only).
const Tensor& extent(const Tensor& t, int64_t rows, int64_t cols, const char* name) {
  if (t.dim() != 2 || t.size(0) != rows || t.size(1) != cols) {
    std::string s = std::string(name) + ": expected [" + std::to_string(rows) + ", " + std::to_string(cols) + "], got [";
    for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
    fail(s + "]");
  }
  return t;
}

// Rows per launch of a row-parallel product over n rows whose operands take
// `row_bytes` per row at most: each operand then spans under 2 GiB, mg_gemm's
// buffer range with 256 rows of slack; a multiple of 256.
int64_t row_step(int64_t n, int64_t row_bytes) {
  int64_t r = ((int64_t(1) << 31) - 1) / std::max<int64_t>(row_bytes, 1) - 257;
  r = std::max<int64_t>(256, r / 256 * 256);
  return n <= r ? n : r;
}

// A 2-D bf16 operand or output as the entry points take it.
struct Mat {
  void* p;
  int64_t ld;
  int64_t esize;
  Mat rows(int64_t r0) const { return {static_cast<char*>(p) + r0 * ld * esize, ld, esize}; }
  Mat cols(int64_t c0) const { return {static_cast<char*>(p) + c0 * esize, ld, esize}; }
};
Mat mat(const Tensor& t, const char* name) { return {ptr(t), row_stride(t, name), int64_t(t.element_size())}; }

// ------------------------------------------------------------------ products

void gemm(int al, Mat a, int bl, Mat b, int64_t M, int64_t N, int64_t K, int epi, const float* bias, void* aux,
          int64_t ldaux, int c_dtype, Mat c, int flags, const Tensor& like, int64_t stream) {
  if (deterministic()) flags |= MG_GEMM_DETERMINISTIC;
  const size_t wsb = mg_gemm_workspace_bytes(al, bl, M, N, K, epi, c_dtype, flags);
  Tensor ws;
  if (wsb) ws = bytes(wsb, like);
  check(mg_gemm(al, a.p, a.ld, bl, b.p, b.ld, M, N, K, epi, bias, aux, ldaux, c_dtype, c.p, c.ld, flags,
                wsb ? ptr(ws) : nullptr, wsb, st(stream)),
        "mg_gemm");
}

// x w^T (+ bias, + GELU with the pre-activation kept) [N, O], bf16; x [N, K], w [O, K]
Tensor linear_fwd(const Tensor& x, const Tensor& w, const float* bias, const Tensor* pre, int64_t stream) {
  const int64_t n = x.size(0), k = x.size(1), o = extent(w, w.size(0), k, "w").size(0);
  Tensor y = make({n, o}, at::kBFloat16, x);
  const Mat xm = mat(x, "x"), wm = mat(w, "w"), ym = mat(y, "y");
  const int epi = pre ? MG_EPI_BIAS_GELU : bias ? MG_EPI_BIAS : MG_EPI_NONE;
  const int64_t step = row_step(n, 2 * std::max(xm.ld, o));
  for (int64_t r = 0; r < n; r += step)
    gemm(MG_KCONTIG, xm.rows(r), MG_KCONTIG, wm, std::min(n - r, step), o, k, epi, bias, pre ? h16(*pre) + r * o : nullptr,
         pre ? o : 0, MG_BF16, ym.rows(r), 0, x, stream);
  return y;
}

// out[N, O] = x w^T to fp32 accuracy from hi/lo pairs x [N, 2K], w [O, 2K]
void linear_fwd_hilo(Mat x, Mat w, int64_t n, int64_t o, int64_t k, int c_dtype, Mat out, const Tensor& like,
                     int64_t stream) {
  const int64_t step = row_step(n, std::max(2 * x.ld, out.ld * out.esize));
  for (int64_t r = 0; r < n; r += step)
    gemm(MG_KCONTIG, x.rows(r), MG_KCONTIG, w, std::min(n - r, step), o, k, MG_EPI_NONE, nullptr, nullptr, 0, c_dtype,
         out.rows(r), MG_GEMM_HILO, like, stream);
}

// dy w [N, K] for dy [N, O] bf16, w [O, K] bf16: bf16 rounded stochastically, or fp32
Tensor linear_dx(const Tensor& dy, const Tensor& w, bool f32, int64_t stream) {
  const int64_t n = dy.size(0), o = dy.size(1), k = extent(w, o, w.size(-1), "w").size(1);
  Tensor dx = make({n, k}, f32 ? at::kFloat : at::kBFloat16, dy);
  const Mat dm = mat(dy, "dy"), wm = mat(w, "w"), xm = mat(dx, "dx");
  const int64_t step = row_step(n, std::max(2 * dm.ld, k * xm.esize));
  for (int64_t r = 0; r < n; r += step)
    gemm(MG_KCONTIG, dm.rows(r), MG_MNCONTIG, wm, std::min(n - r, step), k, o, MG_EPI_NONE, nullptr, nullptr, 0,
         f32 ? MG_F32 : MG_BF16, xm.rows(r), f32 ? 0 : MG_GEMM_STOCHASTIC, dy, stream);
  return dx;
}

// dy^T x [M, N] fp32 for dy [rows, M], x [rows, N] bf16: a new tensor, or added into `into`
Tensor linear_dw(Mat dy, Mat x, int64_t n, int64_t m, int64_t k, const Opt& into, const Tensor& like, int64_t stream) {
  Tensor out = into ? *into : make({m, k}, at::kFloat, like);
  const Mat om = mat(out, "dW");
  const int64_t step = row_step(n, 2 * std::max(dy.ld, x.ld));
  for (int64_t r = 0; r < n; r += step)
    gemm(MG_MNCONTIG, dy.rows(r), MG_MNCONTIG, x.rows(r), m, k, std::min(n - r, step), MG_EPI_NONE, nullptr, nullptr, 0,
         MG_F32, om, into || r ? MG_GEMM_ACCUMULATE : 0, like, stream);
  return out;
}

// Two weight gradients over the same rows in one launch (mg_gemm_wgrad_pair), each
// a new tensor or (both) added into into0 and into1; over 2 GiB one at a time.
std::pair<Tensor, Tensor> linear_dw_pair(Mat dy0, Mat x0, int64_t m0, int64_t k0, Mat dy1, Mat x1, int64_t m1, int64_t k1,
                                         int64_t n, const Opt& into0, const Opt& into1, const Tensor& like,
                                         int64_t stream) {
  const bool acc = into0 && into1;
  if (row_step(n, 2 * std::max(std::max(dy0.ld, x0.ld), std::max(dy1.ld, x1.ld))) < n)
    return {linear_dw(dy0, x0, n, m0, k0, acc ? into0 : Opt(), like, stream),
            linear_dw(dy1, x1, n, m1, k1, acc ? into1 : Opt(), like, stream)};
  Tensor o0 = acc ? *into0 : make({m0, k0}, at::kFloat, like), o1 = acc ? *into1 : make({m1, k1}, at::kFloat, like);
  const int flags = (acc ? MG_GEMM_ACCUMULATE : 0) | (deterministic() ? MG_GEMM_DETERMINISTIC : 0);
  const size_t wsb = mg_gemm_wgrad_pair_workspace_bytes(m0, k0, m1, k1, n, flags);
  Tensor ws;
  if (wsb) ws = bytes(wsb, like);
  check(mg_gemm_wgrad_pair(dy0.p, dy0.ld, x0.p, x0.ld, m0, k0, fp(o0), o0.stride(0), dy1.p, dy1.ld, x1.p, x1.ld, m1, k1,
                           fp(o1), o1.stride(0), n, flags, wsb ? ptr(ws) : nullptr, wsb, st(stream)),
        "mg_gemm_wgrad_pair");
  return {o0, o1};
}

// dX = dy w and the weight gradients of `dws` (dy_i [n, m_i], x_i [n, k_i] over the same n
// rows; each a new tensor or added into `into`) in one launch where they share one
// (mg_gemm_group); nullopt otherwise.
struct DW {
  Mat dy, x;
  int64_t m, k;
  Opt into;
};
std::optional<std::vector<Tensor>> group(const Tensor& dy, const Tensor& w, const std::vector<DW>& dws, int64_t stream) {
  const int64_t n = dy.size(0), o = dy.size(1), k = extent(w, o, w.size(-1), "w").size(1);
  const Mat dm = mat(dy, "dy"), wm = mat(w, "w");
  // One weight gradient beside dX needs 512 rows and 16 tiles with it: below, the launch saved is less
  // than the partials cost (us, apart -> together: 279 rows, 512 x 1024, 18.2 -> 21.2; 25 rows, 1024 x
  // 2048, accumulated, 18.5 -> 19.8; 1919 rows, 256 x 512, 23.6 -> 25.8; 1194 rows, 1024 x
  // 2048, accumulated, 49 -> 36).
  const auto tiles = [](int64_t r, int64_t c) { return ((r + 255) / 256) * ((c + 255) / 256); };
  if (dws.size() == 1 && (n < 512 || tiles(n, k) + tiles(dws[0].m, dws[0].k) < 16)) return std::nullopt;
  const auto span = [](int64_t rows, int64_t ld) { return (rows + 512) * ld * 2 < (int64_t(1) << 31); };
  bool ok = span(n, dm.ld) && span(o, wm.ld) && (dws.size() == 1 || dws.size() == 2);
  mg_gemm_desc d[3] = {{dm.p, wm.p, nullptr, dm.ld, wm.ld, k, int(n), int(k), int(o), 0}};
  for (size_t i = 0; ok && i < dws.size(); ++i) {
    const DW& q = dws[i];
    ok = span(n, q.dy.ld) && span(n, q.x.ld);
    d[i + 1] = {q.dy.p, q.x.p, nullptr, q.dy.ld, q.x.ld, q.k, int(q.m), int(q.k), int(n), q.into ? 1 : 0};
  }
  const int count = 1 + int(dws.size()), flags = deterministic() ? MG_GEMM_DETERMINISTIC : 0;
  if (!ok || !mg_gemm_group_fits(d, count, flags)) return std::nullopt;
  std::vector<Tensor> out{make({n, k}, at::kBFloat16, dy)};
  d[0].C = ptr(out[0]);
  for (size_t i = 0; i < dws.size(); ++i) {
    out.push_back(dws[i].into ? *dws[i].into : make({dws[i].m, dws[i].k}, at::kFloat, dy));
    d[i + 1].C = ptr(out.back());
    d[i + 1].ldc = out.back().stride(0);
  }
  const size_t wsb = mg_gemm_group_workspace_bytes(d, count, flags);
  Tensor ws;
  if (wsb) ws = bytes(wsb, dy);
  check(mg_gemm_group(d, count, flags, wsb ? ptr(ws) : nullptr, wsb, st(stream)), "mg_gemm_group");
  return out;
}

// mg_gemm_f32 on raw operands
void gemm_f32_raw(int al, const float* a, int64_t lda, int bl, const float* b, int64_t ldb, int64_t M, int64_t N, int64_t K,
                  int epi, const float* bias, float* aux, float* c, int64_t ldc, int flags, const Tensor& like, int64_t stream) {
  const size_t wsb = mg_gemm_f32_workspace_bytes(M, N, K, flags);
  Tensor ws;
  if (wsb) ws = bytes(wsb, like);
  check(mg_gemm_f32(al, a, lda, bl, b, ldb, M, N, K, epi, bias, aux, aux ? N : 0, c, ldc, flags, wsb ? ptr(ws) : nullptr, wsb,
                    st(stream)),
        "mg_gemm_f32");
}

// sum_k A(m, k) B(k, n) (+ bias) in fp32, into `out` or a new tensor
Tensor gemm_f32(const Tensor& a, int al, const Tensor& b, int bl, int64_t M, int64_t N, int64_t K, const Opt& out_,
                const Opt& bias, int flags, int64_t stream) {
  need_cuda(a);
  need_cuda(b);
  if (a.scalar_type() != at::kFloat || b.scalar_type() != at::kFloat) fail("mg_gemm_f32 operands must be float32");
  Tensor out = out_ ? *out_ : make({M, N}, at::kFloat, a);
  extent(a, al == MG_KCONTIG ? M : K, al == MG_KCONTIG ? K : M, "A");
  extent(b, bl == MG_KCONTIG ? N : K, bl == MG_KCONTIG ? K : N, "B");
  extent(out, M, N, "C");
  const Mat am = mat(a, "A"), bm = mat(b, "B"), om = mat(out, "C");
  gemm_f32_raw(al, static_cast<float*>(am.p), am.ld, bl, static_cast<float*>(bm.p), bm.ld, M, N, K,
               bias ? MG_EPI_BIAS : MG_EPI_NONE, bias ? vec(*bias, N, "bias") : nullptr, nullptr, fp(out), om.ld, flags, a, stream);
  return out;
}

Tensor column_sum(const Tensor& x, int64_t stream);

// The fp32 FeedForward: (pre or none, act, y) of rows x [N, D]; pre kept with `train`.
std::tuple<Opt, Tensor, Tensor> ff_f32_forward(const Tensor& x, const Tensor& w1, const Tensor& b1, const Tensor& w2,
                                               const Tensor& b2, bool train, int64_t stream) {
  const int64_t N = x.size(0), D = x.size(1), F = w1.size(0), O = w2.size(0);
  extent(w1, F, D, "w1");
  extent(w2, O, F, "w2");
  const int flags = deterministic() ? MG_GEMM_DETERMINISTIC : 0;
  Opt pre;
  if (train) pre = make({N, F}, at::kFloat, x);
  Tensor act = make({N, F}, at::kFloat, x), y = make({N, O}, at::kFloat, x);
  gemm_f32_raw(MG_KCONTIG, fp(x), row_stride(x, "x"), MG_KCONTIG, fp(w1), row_stride(w1, "w1"), N, F, D, MG_EPI_BIAS_GELU,
               vec(b1, F, "b1"), fp(pre), fp(act), F, flags, x, stream);
  gemm_f32_raw(MG_KCONTIG, fp(act), F, MG_KCONTIG, fp(w2), row_stride(w2, "w2"), N, O, F, MG_EPI_BIAS, vec(b2, O, "b2"), nullptr,
               fp(y), O, flags, x, stream);
  return {pre, act, y};
}

// (dx or none, dW1, db1, dW2, db2 or none each) for a contiguous dy [N, O]
std::tuple<Opt, Opt, Opt, Opt, Opt> ff_f32_backward(const Tensor& x, const Tensor& pre, const Tensor& act, const Tensor& w1,
                                                    const Tensor& w2, const Tensor& dy, bool want_x, bool want_w1, bool want_b1,
                                                    bool want_w2, bool want_b2, int64_t stream) {
  const int64_t N = x.size(0), D = x.size(1), F = pre.size(1), O = dy.size(1);
  extent(w1, F, D, "w1");
  extent(w2, O, F, "w2");
  extent(pre, N, F, "pre");
  extent(act, N, F, "act");
  extent(dy, N, O, "dy");
  const int flags = deterministic() ? MG_GEMM_DETERMINISTIC : 0;
  Opt dx, dw1, db1, dw2, db2;
  const int64_t ldx = row_stride(x, "x"), ld1 = row_stride(w1, "w1"), ld2 = row_stride(w2, "w2");
  if (want_w2) {
    dw2 = make({O, F}, at::kFloat, x);
    gemm_f32_raw(MG_MNCONTIG, fp(dy), O, MG_MNCONTIG, fp(act), F, O, F, N, MG_EPI_NONE, nullptr, nullptr, fp(dw2), F, flags, x,
                 stream);
  }
  if (want_b2) db2 = column_sum(dy, stream);
  if (want_x || want_w1 || want_b1) {
    Tensor dpre = make({N, F}, at::kFloat, x);  // dy W2 * gelu'(pre)
    gemm_f32_raw(MG_KCONTIG, fp(dy), O, MG_MNCONTIG, fp(w2), ld2, N, F, O, MG_EPI_GELU_GRAD, nullptr, fp(pre), fp(dpre), F, flags,
                 x, stream);
    if (want_b1) db1 = column_sum(dpre, stream);
    if (want_w1) {
      dw1 = make({F, D}, at::kFloat, x);
      gemm_f32_raw(MG_MNCONTIG, fp(dpre), F, MG_MNCONTIG, fp(x), ldx, F, D, N, MG_EPI_NONE, nullptr, nullptr, fp(dw1), D, flags, x,
                   stream);
    }
    if (want_x) {
      dx = make({N, D}, at::kFloat, x);
      gemm_f32_raw(MG_KCONTIG, fp(dpre), F, MG_MNCONTIG, fp(w1), ld1, N, D, F, MG_EPI_NONE, nullptr, nullptr, fp(dx), D, flags, x,
                   stream);
    }
  }
  return {dx, dw1, db1, dw2, db2};
}

// ------------------------------------------------------------------ norm

typedef std::tuple<Opt, Tensor, Tensor, Opt> NormOut;

// (x + delta or none, y, rstd, pair or none) of rows x [..., D]; with_lo: y is the first half of pair
NormOut norm_fwd(const Tensor& x, const Opt& delta, const Tensor& w, bool bf16, bool with_lo, int64_t stream) {
  const int64_t D = x.size(-1), N = x.numel() / std::max<int64_t>(D, 1);
  if (delta && delta->numel() != x.numel()) fail("delta: expected as many values as x has");
  Opt pair, x_out;
  Tensor y;
  if (with_lo) {
    std::vector<int64_t> s = x.sizes().vec();
    s.back() = 2 * D;
    pair = make(s, at::kBFloat16, x);
    y = pair->narrow(-1, 0, D);
  } else {
    y = make(x.sizes(), bf16 ? at::kBFloat16 : at::kFloat, x);
  }
  Tensor rstd = make({N}, at::kFloat, x);
  if (delta) x_out = make(x.sizes(), at::kFloat, x);
  check(mg_add_rmsnorm_fwd(fp(x), delta ? code(*delta) : 0, ptr(delta), vec(w, D, "norm weight"), fp(x_out), bf16 || with_lo ? MG_BF16 : MG_F32,
                           ptr(y), with_lo ? h16(*pair) + D : nullptr, with_lo ? 2 * D : D, fp(rstd), N, D, kEps, st(stream)),
        "mg_add_rmsnorm_fwd");
  return {x_out, y, rstd, pair};
}

// (dx, ddelta or none, dw); dy contiguous or none (zero); dy_scale a device scalar or none
std::tuple<Opt, Opt, Tensor> norm_bwd(const Tensor& xn, const Tensor& w, const Tensor& rstd, const Opt& dy_, const Opt& dres_,
                                      bool want_dx, int delta_type, const Opt& dy_scale_, int64_t stream) {
  const int64_t D = xn.size(-1), N = xn.numel() / std::max<int64_t>(D, 1);
  Tensor dy = dy_ ? dy_->contiguous() : at::zeros(xn.sizes(), xn.options().dtype(at::kFloat));
  Opt dres, dx, dd, scale;
  if (dres_) dres = dres_->to(at::kFloat).contiguous();
  if (dy_scale_) scale = dy_scale_->detach().to(xn.device(), at::kFloat).reshape({1});
  if (want_dx) dx = make(xn.sizes(), at::kFloat, xn);
  if (delta_type >= 0) dd = make(xn.sizes(), delta_type == MG_BF16 ? at::kBFloat16 : at::kFloat, xn);
  Tensor dw = make({D}, at::kFloat, xn);
  const size_t wsb = mg_add_rmsnorm_bwd_workspace_bytes(N, D);
  Tensor ws = bytes(wsb, xn);
  if (dy.numel() != xn.numel() || (dres && dres->numel() != xn.numel())) fail("norm gradient: expected as many values as x has");
  check(mg_add_rmsnorm_bwd_scaled(fp(xn), vec(w, D, "norm weight"), vec(rstd, N, "rstd"), code(dy), ptr(dy), fp(scale), fp(dres), fp(dx),
                                  std::max(delta_type, 0), ptr(dd), fp(dw), N, D, ptr(ws), wsb, st(stream)),
        "mg_add_rmsnorm_bwd");
  return {dx, dd, dw};
}

// ------------------------------------------------------------------ scan

// hidden and gate [B, T, Di] with unit inner stride and shared strides, as raw pointers
struct HG {
  int dtype;
  char *hidden, *gate;
  int64_t sb, ld;
  int64_t B, T, Di;
};
HG split(const Tensor& hg) {  // [B, T, 2 Di] (or [N, 2 Di] with B, T set by the caller), contiguous
  const int64_t Di = hg.size(-1) / 2;
  char* p = static_cast<char*>(ptr(hg));
  return {code(hg), p, p + Di * hg.element_size(), hg.dim() == 3 ? hg.size(1) * 2 * Di : 0, 2 * Di,
          hg.dim() == 3 ? hg.size(0) : 0, hg.dim() == 3 ? hg.size(1) : 0, Di};
}
HG two(const Tensor& hidden, const Tensor& gate) {
  return {code(hidden), static_cast<char*>(ptr(hidden)), static_cast<char*>(ptr(gate)), hidden.stride(0),
          hidden.stride(1), hidden.size(0), hidden.size(1), hidden.size(2)};
}

// (h, h_last, ckpt or none)
std::tuple<Tensor, Tensor, Opt> scan_fwd_hg(const HG& s, const Opt& h0, at::ScalarType out, bool need_ckpt, const Tensor& ws,
                                            const Tensor& like, int64_t stream) {
  Tensor h = make({s.B, s.T, s.Di}, out, like), last = make({s.B, 1, s.Di}, at::kFloat, like);
  Opt ckpt;
  if (need_ckpt && out != at::kFloat)
    ckpt = make({static_cast<int64_t>(mg_scan_ckpt_elems(s.B, s.T, s.Di))}, at::kFloat, like);
  check(mg_scan_fwd(s.dtype, s.hidden, s.gate, s.sb, s.ld, fp(h0), code(h), ptr(h), h.stride(0), h.stride(1), fp(last),
                    fp(ckpt), s.B, s.T, s.Di, ptr(ws), ws.numel(), st(stream)),
        "mg_scan_fwd");
  return {h, last, ckpt};
}

// dhidden and dgate into d (a layout like s), returns dh0 or none
Opt scan_bwd_hg(const HG& s, const Opt& h0, const Opt& h, const Opt& ckpt, const Opt& dh_, const Opt& dlast_, const HG& d,
                bool want_dh0, const Tensor& ws, const Tensor& like, int64_t stream) {
  const at::ScalarType hd = h ? h->scalar_type() : at::kFloat;
  Tensor dh;
  if (!dh_)
    dh = at::zeros({s.B, s.T, s.Di}, like.options().dtype(hd));
  else if (dh_->scalar_type() != hd || dh_->stride(-1) != 1 || dh_->stride(0) % 4 || dh_->stride(1) % 4)
    dh = dh_->to(hd).contiguous();
  else
    dh = *dh_;
  Opt dlast, dh0;
  if (dlast_) dlast = dlast_->reshape({s.B, s.Di}).to(at::kFloat).contiguous();
  if (want_dh0) dh0 = make({s.B, 1, s.Di}, at::kFloat, like);
  check(mg_scan_bwd(s.dtype, s.hidden, s.gate, s.sb, s.ld, fp(h0), hd == at::kFloat ? MG_F32 : MG_BF16, ptr(h),
                    h ? h->stride(0) : 0, h ? h->stride(1) : 0, fp(ckpt), ptr(dh), dh.stride(0), dh.stride(1), fp(dlast),
                    d.hidden, d.gate, d.sb, d.ld, fp(dh0), s.B, s.T, s.Di, ptr(ws), ws.numel(), st(stream)),
        "mg_scan_bwd");
  return dh0;
}

std::tuple<Tensor, Tensor, Opt> scan_fwd(const Tensor& hidden, const Tensor& gate, const Opt& h0, bool bf16_out, bool need_ckpt,
                                         const Tensor& ws, int64_t stream) {
  return scan_fwd_hg(two(hidden, gate), h0, bf16_out ? at::kBFloat16 : at::kFloat, need_ckpt, ws, hidden, stream);
}
Opt scan_bwd(const Tensor& hidden, const Tensor& gate, const Opt& h0, const Opt& h, const Opt& ckpt, const Opt& dh,
             const Opt& dlast, const Tensor& dhidden, const Tensor& dgate, bool want_dh0, const Tensor& ws, int64_t stream) {
  return scan_bwd_hg(two(hidden, gate), h0, h, ckpt, dh, dlast, two(dhidden, dgate), want_dh0, ws, hidden, stream);
}
// (x_out, h_last, ckpt): x_out = res + h
std::tuple<Tensor, Tensor, Tensor> scan_fwd_residual_hg(const HG& s, const Opt& h0, const Tensor& res_, const Tensor& ws,
                                                        int64_t stream) {
  const Tensor res = res_.contiguous();
  Tensor x = make({s.B, s.T, s.Di}, at::kFloat, res), last = make({s.B, 1, s.Di}, at::kFloat, res);
  Tensor ckpt = make({static_cast<int64_t>(mg_scan_ckpt_elems(s.B, s.T, s.Di))}, at::kFloat, res);
  check(mg_scan_fwd_residual(s.dtype, s.hidden, s.gate, s.sb, s.ld, fp(h0), fp(res), fp(x), x.stride(0), x.stride(1), fp(last),
                             fp(ckpt), s.B, s.T, s.Di, ptr(ws), ws.numel(), st(stream)),
        "mg_scan_fwd_residual");
  return {x, last, ckpt};
}

std::tuple<Tensor, Tensor, Tensor> scan_fwd_residual(const Tensor& hidden, const Tensor& gate, const Opt& h0, const Tensor& res,
                                                     const Tensor& ws, int64_t stream) {
  return scan_fwd_residual_hg(two(hidden, gate), h0, res, ws, stream);
}

// ------------------------------------------------------------------ blocks

// MinGRUBlock.forward (blocks.py). x, pending [N, D] rows of [B, T, D]; w_pair, w_bf16:
// to_hidden_and_gate's hi/lo pair [2 Di, 2 D] and bf16 copy; to_pair: to_out's pair or none.
// Returns (x1 or none, rstd, pair, hg, h or none, h_last, out or none, h_pair or none, ckpt or
// none): without to_out, `out` is x1 + h (`residual`) or h; with it, to_out's fp32 output.
typedef std::tuple<Opt, Tensor, Tensor, Tensor, Opt, Tensor, Tensor, Opt, Opt> GruOut;
GruOut gru_forward(const Tensor& x, const Opt& pending, const Tensor& w_norm, const Tensor& w_pair, const Tensor& w_bf16,
                   const Opt& to_pair, const Opt& h0, int64_t B, int64_t T, bool residual, bool one_launch, const Tensor& ws,
                   int64_t stream) {
  const int64_t N = x.size(0), D = x.size(1), Di = w_pair.size(0) / 2;
  if (N != B * T) fail("x: expected B * T rows");
  extent(w_pair, 2 * Di, 2 * D, "w_pair");
  extent(w_bf16, 2 * Di, D, "w_bf16");
  if (to_pair) extent(*to_pair, D, 2 * Di, "to_out's pair");
  else if (residual && Di != D) fail("without to_out the scan's width is x's");
  if (h0) vec(*h0, B * Di, "h0");
  auto [x_out, n, rstd, pair] = norm_fwd(x, pending, w_norm, true, true, stream);
  Tensor hg = make({N, 2 * Di}, at::kBFloat16, x);
  const Mat pm = mat(*pair, "pair"), wm = mat(w_pair, "w_pair"), hm = mat(hg, "hg");
  const auto span = [](int64_t rows, int64_t ld) { return (rows + 256) * ld * 2 < (int64_t(1) << 31); };
  const bool pair_ok = one_launch && wm.ld % 8 == 0 && wm.ld >= 2 * D && reinterpret_cast<uintptr_t>(wm.p) % 16 == 0 &&
                       span(N, pm.ld) && span(2 * Di, wm.ld);
  if (pair_ok && !deterministic() && mg_gemm_hilo_cols_fits(N, 2 * Di, D, Di)) {  // (its sum order is its own)
    check(mg_gemm_hilo_cols(pm.p, pm.ld, wm.p, wm.ld, N, 2 * Di, D, Di, hm.p, hm.ld, st(stream)), "mg_gemm_hilo_cols");
  } else if (pair_ok && D % 128 == 0 && Di % 256 == 0) {
    check(mg_gemm_hilo_prefix(pm.p, pm.ld, wm.p, wm.ld, N, 2 * Di, D, Di, hm.p, hm.ld, st(stream)), "mg_gemm_hilo_prefix");
  } else {
    linear_fwd_hilo(pm, wm, N, Di, D, MG_BF16, hm, x, stream);  // minGRU.py:45, hidden half
    const Mat wb = mat(w_bf16, "w_hg");                          // gate half
    const int64_t step = row_step(N, 2 * std::max(pm.ld, hm.ld));
    for (int64_t r = 0; r < N; r += step)
      gemm(MG_KCONTIG, pm.rows(r), MG_KCONTIG, wb.rows(Di), std::min(N - r, step), Di, D, MG_EPI_NONE, nullptr, nullptr, 0,
           MG_BF16, hm.rows(r).cols(Di), 0, x, stream);
  }
  HG s = split(hg);
  s.B = B, s.T = T, s.sb = T * 2 * Di;
  const Tensor& x1 = x_out ? *x_out : x;
  if (!to_pair && residual) {
    auto [x2, last, ckpt] = scan_fwd_residual_hg(s, h0, x1.view({B, T, D}), ws, stream);
    return {x_out, rstd, *pair, hg, std::nullopt, last, x2, std::nullopt, ckpt};
  }
  if (!to_pair) {
    auto [h, last, none] = scan_fwd_hg(s, h0, at::kFloat, false, ws, x, stream);
    return {x_out, rstd, *pair, hg, h, last, h, std::nullopt, std::nullopt};
  }
  Tensor h_pair = make({N, 2 * Di}, at::kBFloat16, x), last = make({B, 1, Di}, at::kFloat, x);
  Tensor out = make({N, D}, at::kFloat, x), ckpt = make({static_cast<int64_t>(mg_scan_ckpt_elems(B, T, Di))}, at::kFloat, x);
  check(mg_scan_fwd_pair(s.hidden, s.gate, s.sb, s.ld, fp(h0), ptr(h_pair), fp(last), fp(ckpt), B, T, Di, ptr(ws), ws.numel(),
                         st(stream)),
        "mg_scan_fwd_pair");
  linear_fwd_hilo(mat(h_pair, "h_pair"), mat(*to_pair, "to_pair"), N, D, Di, MG_F32, mat(out, "out"), x, stream);
  return {x_out, rstd, *pair, hg, std::nullopt, last, out.view({B, T, D}), h_pair, ckpt};
}

// MinGRUBlock.backward. dx1: the gradient of the residual stream [B, T, D] or none; dout: of
// to_out's output (with h_pair) or of h. into_hg / into_to: .grad tensors that the weight
// gradients are added into (then none is returned for them).
// Returns (dx, dpending or none, dw_norm, dW_hg or none, dh0 or none, dW_to or none).
typedef std::tuple<Tensor, Opt, Tensor, Opt, Opt, Opt> GruGrads;
GruGrads gru_backward(const Tensor& xn, const Tensor& w_norm, const Tensor& rstd, const Tensor& pair, const Tensor& hg,
                      const Opt& h, const Opt& h0, const Tensor& w_bf16, const Opt& ckpt, const Opt& h_pair, const Opt& to_bf16,
                      const Opt& dx1, const Opt& dout, const Opt& dlast, int64_t B, int64_t T, bool has_pending, bool want_hg,
                      bool want_to, bool want_dh0, bool pair_launch, const Opt& into_hg, const Opt& into_to, const Tensor& ws,
                      int64_t stream) {
  const int64_t N = xn.size(0), D = xn.size(1), Di = hg.size(1) / 2;
  extent(hg, N, 2 * Di, "hg");
  extent(pair, N, 2 * D, "pair");
  extent(w_bf16, 2 * Di, D, "w_bf16");
  if (h_pair) extent(*h_pair, N, 2 * Di, "h_pair");
  if (to_bf16) extent(*to_bf16, D, Di, "to_out's weight");
  Opt dh, dW_to, dW_hg, dh0;
  Tensor dob;
  if (ckpt && !h_pair) {
    dh = dx1;  // x_next = x1 + h: h and the residual get the same gradient
  } else if (dout && h_pair) {
    const Tensor d = dout->reshape({N, D}).to(at::kFloat).contiguous();
    dob = make({N, D}, at::kBFloat16, xn);
    check(mg_round_bf16_sr(fp(d), d.numel(), ptr(dob), 0x3c1d, st(stream)), "mg_round_bf16_sr");
    dh = linear_dx(dob, *to_bf16, true, stream).view({B, T, Di});
    if (want_to && !want_hg) {
      Tensor g = linear_dw(mat(dob, "dout"), mat(*h_pair, "h_pair"), N, D, Di, into_to, xn, stream);
      if (!into_to) dW_to = g;
    }
  } else if (dout) {
    dh = dout->to(at::kFloat);
  }
  Tensor dhg = make({N, 2 * Di}, at::kBFloat16, xn);
  if (!dh && !dlast) {
    dhg.zero_();
    if (want_dh0) dh0 = at::zeros_like(*h0);
  } else {
    HG s = split(hg), d = split(dhg);
    s.B = B, s.T = T, s.sb = d.sb = T * 2 * Di;
    dh0 = scan_bwd_hg(s, h0, h, ckpt, dh, dlast, d, want_dh0, ws, xn, stream);
  }
  Tensor dn;
  const Mat dm = mat(dhg, "dhg"), nm = mat(pair, "pair");
  const bool both = want_hg && want_to && h_pair && dout;
  if (want_hg) {
    std::vector<DW> dws{{dm, nm, 2 * Di, D, into_hg}};
    if (both) dws.push_back({mat(dob, "dout"), mat(*h_pair, "h_pair"), D, Di, into_to});
    if (auto g = group(dhg, w_bf16, dws, stream)) {
      dn = (*g)[0];
      if (!into_hg) dW_hg = (*g)[1];
      if (both && !into_to) dW_to = (*g)[2];
    }
  }
  if (!dn.defined()) {
    dn = linear_dx(dhg, w_bf16, false, stream);
    if (both && pair_launch) {
      // to_out's and to_hidden_and_gate's weight gradients in one launch
      const bool into = into_to && into_hg;
      auto [g_to, g_hg] = linear_dw_pair(mat(dob, "dout"), mat(*h_pair, "h_pair"), D, Di, dm, nm, 2 * Di, D, N,
                                         into ? into_to : Opt(), into ? into_hg : Opt(), xn, stream);
      if (!into) dW_to = g_to, dW_hg = g_hg;
    } else {
      if (both) {
        Tensor g = linear_dw(mat(dob, "dout"), mat(*h_pair, "h_pair"), N, D, Di, into_to, xn, stream);
        if (!into_to) dW_to = g;
      }
      if (want_hg) {
        Tensor g = linear_dw(dm, nm, N, 2 * Di, D, into_hg, xn, stream);
        if (!into_hg) dW_hg = g;
      }
    }
  }
  Opt dres;
  if (dx1) dres = dx1->reshape({N, D});
  auto [dx, dpend, dw] = norm_bwd(xn, w_norm, rstd, dn, dres, true, has_pending ? MG_BF16 : -1, std::nullopt, stream);
  return {*dx, dpend, dw, dW_hg, dh0, dW_to};
}

// FFBlock.forward: (x2 or none, n2, rstd, pre, act, pending) of rows x1 [N, D] (+ out).
typedef std::tuple<Opt, Tensor, Tensor, Tensor, Tensor, Tensor> FFOut;
FFOut ff_forward(const Tensor& x1, const Opt& out, const Tensor& w_norm, const Tensor& w1, const Tensor& b1, const Tensor& w2,
                 const Tensor& b2, int64_t stream) {
  extent(w1, w1.size(0), x1.size(1), "w1");
  extent(w2, w2.size(0), w1.size(0), "w2");
  auto [x2, n2, rstd, none] = norm_fwd(x1, out, w_norm, true, false, stream);
  Tensor pre = make({x1.size(0), w1.size(0)}, at::kBFloat16, x1);
  Tensor act = linear_fwd(n2, w1, vec(b1, w1.size(0), "b1"), &pre, stream);     // pre = n2 W1^T + b1, act = gelu(pre)
  Tensor pend = linear_fwd(act, w2, vec(b2, w2.size(0), "b2"), nullptr, stream);  // act W2^T + b2
  return {x2, n2, rstd, pre, act, pend};
}

// (dpre, db1, db2): the GELU backward and both bias gradients (mg_ff_bias_bwd)
std::tuple<Tensor, Tensor, Tensor> ff_bias_bwd(const Tensor& dact, const Tensor& pre, const Tensor& dy, int64_t stream) {
  const int64_t N = pre.size(0), C1 = pre.size(1), C2 = dy.size(1);
  Tensor dpre = make({N, C1}, at::kBFloat16, pre), db1 = make({C1}, at::kFloat, pre), db2 = make({C2}, at::kFloat, pre);
  const size_t wsb = mg_ff_bias_bwd_workspace_bytes(N, C1, C2);
  Tensor ws = bytes(wsb, pre);
  check(mg_ff_bias_bwd(code(dact), ptr(dact), row_stride(dact, "dact"), ptr(pre), row_stride(pre, "pre"), ptr(dpre), C1,
                       fp(db1), N, C1, ptr(dy), row_stride(dy, "dy"), fp(db2), C2, ptr(ws), wsb, st(stream)),
        "mg_ff_bias_bwd");
  return {dpre, db1, db2};
}

// FFBlock.backward for a bf16 contiguous dpend [N, D]: (dx, dw_norm, dW1 or none, db1, dW2 or
// none, db2), the weight gradients added into into1 / into2 where given.
typedef std::tuple<Tensor, Tensor, Opt, Tensor, Opt, Tensor> FFGrads;
FFGrads ff_backward(const Tensor& x2, const Tensor& w_norm, const Tensor& rstd, const Tensor& n2, const Tensor& pre,
                    const Tensor& act, const Tensor& w1, const Tensor& w2, const Opt& dx2, const Tensor& dp, bool pair_launch,
                    const Opt& into1, const Opt& into2, int64_t stream) {
  const int64_t N = x2.size(0), D = x2.size(1), F = pre.size(1);
  extent(n2, N, D, "n2");
  extent(act, N, F, "act");
  extent(dp, N, D, "dpend");
  Tensor dact = linear_dx(dp, w2, false, stream);
  auto [dpre, db1, db2] = ff_bias_bwd(dact, pre, dp, stream);
  const Mat dpm = mat(dp, "dpend"), am = mat(act, "act"), dm = mat(dpre, "dpre"), nm = mat(n2, "n2");
  Tensor dn2;
  Opt dW1, dW2;
  if (auto g = group(dpre, w1, {{dpm, am, D, F, into2}, {dm, nm, F, D, into1}}, stream)) {
    dn2 = (*g)[0];
    if (!into2) dW2 = (*g)[1];
    if (!into1) dW1 = (*g)[2];
  } else {
    dn2 = linear_dx(dpre, w1, false, stream);
    if (pair_launch) {
      const bool into = into1 && into2;
      auto [g2, g1] = linear_dw_pair(dpm, am, D, F, dm, nm, F, D, N, into ? into2 : Opt(), into ? into1 : Opt(), x2, stream);
      if (!into) dW1 = g1, dW2 = g2;
    } else {
      Tensor g2 = linear_dw(dpm, am, N, D, F, into2, x2, stream), g1 = linear_dw(dm, nm, N, F, D, into1, x2, stream);
      if (!into1) dW1 = g1;
      if (!into2) dW2 = g2;
    }
  }
  Opt dres;
  if (dx2) dres = dx2->reshape({N, D});
  auto [dx, none, dw] = norm_bwd(x2, w_norm, rstd, dn2, dres, true, -1, std::nullopt, stream);
  return {*dx, dw, dW1, db1, dW2, db2};
}

// FinalNormCE.forward: (loss, x + pending or none, embed, rstd, dlogits); w bf16 [V, D]
std::tuple<Tensor, Opt, Tensor, Tensor, Tensor> head_forward(const Tensor& x, const Opt& pending, const Tensor& w_norm,
                                                             const Tensor& w, const Tensor& labels, int64_t stream) {
  const int64_t N = x.size(0), D = x.size(1), V = extent(w, w.size(0), D, "w").size(0);
  if (labels.scalar_type() != at::kLong || labels.numel() != N || !labels.is_contiguous())
    fail("labels: expected one contiguous int64 value per row");
  auto [x_out, embed, rstd, none] = norm_fwd(x, pending, w_norm, true, false, stream);
  Tensor dl = make({N, V}, at::kBFloat16, x), part = make({mg_logits_cross_entropy_partials(N)}, at::kFloat, x);
  check(mg_logits_cross_entropy(ptr(embed), D, ptr(w), row_stride(w, "w"), static_cast<int64_t*>(ptr(labels)), ptr(dl), V,
                                fp(part), nullptr, N, D, V, static_cast<float>(1.0 / N), st(stream)),
        "mg_logits_cross_entropy");
  return {part.sum() / N, x_out, embed, rstd, dl};
}

// FinalNormCE.backward: (dx, dpending or none, dw_norm, dW or none); g: the loss's gradient
std::tuple<Tensor, Opt, Tensor, Opt> head_backward(const Tensor& xn, const Tensor& w_norm, const Tensor& rstd,
                                                   const Tensor& embed, const Tensor& dl, const Tensor& w, const Tensor& g,
                                                   bool has_pending, bool want_w, int64_t stream) {
  Tensor de = linear_dx(dl, w, true, stream);  // fp32, unscaled
  Opt dW;
  if (want_w) {
    dW = linear_dw(mat(dl, "dlogits"), mat(embed, "embed"), xn.size(0), dl.size(1), embed.size(1), std::nullopt, xn, stream);
    dW->mul_(g);  // the loss's upstream scale, in fp32; no host sync
  }
  auto [dx, dpend, dw] = norm_bwd(xn, w_norm, rstd, de, std::nullopt, true, has_pending ? MG_BF16 : -1, g, stream);
  return {*dx, dpend, dw, dW};
}

// One layer of the no-grad forward of a model whose activations and parameters share a dtype
// (bf16: generate.py's cast; fp32), reference mingru/minLM.py:119-130: x [N, D] fp32 residual
// stream, pending [N, D] or none; norm weights and biases fp32. Returns (x2, pending, h_last), x2
// without the new pending; nullopt where a width or layout is not the kernels'. The scan writes what
// the next product reads (bf16 h), or adds its state to the residual stream itself (no to_out), and
// the GELU is the first product's epilogue.
std::optional<std::tuple<Tensor, Tensor, Tensor>> infer_layer(const Tensor& x, const Opt& pending, const Tensor& w_norm,
                                                              const Tensor& w_hg, const Opt& w_to, const Tensor& w_ff,
                                                              const Tensor& w1, const Tensor& b1, const Tensor& w2,
                                                              const Tensor& b2, const Opt& h0, int64_t B, int64_t T,
                                                              const Tensor& ws, int64_t stream) {
  const int64_t N = x.size(0), D = x.size(1), Di = w_hg.size(0) / 2, F = w1.size(0);
  const bool f32 = w_hg.scalar_type() == at::kFloat;
  for (const Tensor* w : {&w_hg, &w1, &w2, w_to ? &*w_to : &w_hg})
    if (w->scalar_type() != w_hg.scalar_type() || w->dim() != 2 || w->stride(1) != 1 || w->size(0) % 8 || w->size(1) % 8 ||
        w->stride(0) % 8 || reinterpret_cast<uintptr_t>(w->data_ptr()) % 16)
      return std::nullopt;
  for (const Tensor* t : {&w_hg, &w1, &w2, w_to ? &*w_to : &w_hg, &w_norm, &w_ff, &b1, &b2})
    if (t->device() != x.device()) return std::nullopt;
  if (N < 1 || D > 4096 || Di % 8 || (w_to && (w_to->size(0) != D || w_to->size(1) != Di)) || (!w_to && Di != D) ||
      w_hg.size(1) != D || w1.size(1) != D || w2.size(0) != D || w2.size(1) != F || w_norm.numel() != D || w_ff.numel() != D ||
      b1.numel() != F || b2.numel() != D || x.stride(1) != 1 || x.stride(0) != D)
    return std::nullopt;
  const int flags = deterministic() ? MG_GEMM_DETERMINISTIC : 0;
  const auto linear = [&](const Tensor& a, const Tensor& w) {
    if (!f32) return linear_fwd(a, w, nullptr, nullptr, stream);
    Tensor y = make({a.size(0), w.size(0)}, at::kFloat, a);
    gemm_f32_raw(MG_KCONTIG, fp(a), a.stride(0), MG_KCONTIG, fp(w), w.stride(0), a.size(0), w.size(0), w.size(1), MG_EPI_NONE,
                 nullptr, nullptr, fp(y), w.size(0), flags, a, stream);
    return y;
  };
  auto [x1_, n, rstd, none] = norm_fwd(x, pending, w_norm, !f32, false, stream);
  Tensor x1 = x1_ ? *x1_ : x, hg = linear(n, w_hg), x2, n2, last;
  HG s = split(hg);
  s.B = B, s.T = T, s.sb = T * 2 * Di;
  if (w_to) {
    auto [h, l, no_ckpt] = scan_fwd_hg(s, h0, f32 ? at::kFloat : at::kBFloat16, false, ws, x, stream);
    auto [x2_, n2_, r2, none2] = norm_fwd(x1, linear(h.view({N, Di}), *w_to), w_ff, !f32, false, stream);
    x2 = *x2_, n2 = n2_, last = l;
  } else {
    auto [xr, l, ckpt] = scan_fwd_residual_hg(s, h0, x1.view({B, T, D}), ws, stream);
    x2 = xr.view({N, D}), last = l;
    n2 = std::get<1>(norm_fwd(x2, std::nullopt, w_ff, !f32, false, stream));
  }
  if (f32) return std::make_tuple(x2, std::get<2>(ff_f32_forward(n2, w1, b1, w2, b2, false, stream)), last);
  Tensor pre = make({N, F}, at::kBFloat16, x);  // (the epilogue rounds it to bf16; its values are not used)
  Tensor act = linear_fwd(n2, w1, vec(b1, F, "b1"), &pre, stream);
  return std::make_tuple(x2, linear_fwd(act, w2, vec(b2, D, "b2"), nullptr, stream), last);
}

// Column sums of a 2-D fp32 or bf16 tensor with unit inner stride, fp32.
Tensor column_sum(const Tensor& x, int64_t stream) {
  const int64_t N = x.size(0), C = x.size(1);
  Tensor out = make({C}, at::kFloat, x);
  const size_t wsb = mg_column_sum_workspace_bytes(N, C);
  Tensor ws = bytes(wsb, x);
  check(mg_column_sum(code(x), ptr(x), x.stride(0), N, C, fp(out), ptr(ws), wsb, st(stream)), "mg_column_sum");
  return out;
}

}  // namespace

PYBIND11_MODULE(_native, m) {
  typedef py::call_guard<py::gil_scoped_release> nogil;
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const MgError& e) {
      PyErr_SetString(g_error ? g_error->ptr() : PyExc_RuntimeError, e.what());
    }
  });
  m.def("set_error", [](py::object e) { g_error = new py::object(std::move(e)); });
  m.def("gemm_f32", &gemm_f32, nogil());
  m.def("ff_f32_forward", &ff_f32_forward, nogil());
  m.def("ff_f32_backward", &ff_f32_backward, nogil());
  m.def("norm_fwd", &norm_fwd, nogil());
  m.def("norm_bwd", &norm_bwd, nogil());
  m.def("scan_fwd", &scan_fwd, nogil());
  m.def("scan_fwd_residual", &scan_fwd_residual, nogil());
  m.def("scan_bwd", &scan_bwd, nogil());
  m.def("gru_forward", &gru_forward, nogil());
  m.def("gru_backward", &gru_backward, nogil());
  m.def("ff_forward", &ff_forward, nogil());
  m.def("ff_backward", &ff_backward, nogil());
  m.def("ff_bias_bwd", &ff_bias_bwd, nogil());
  m.def("head_forward", &head_forward, nogil());
  m.def("head_backward", &head_backward, nogil());
  m.def("infer_layer", &infer_layer, nogil());
  m.def("column_sum", &column_sum, nogil());
}
