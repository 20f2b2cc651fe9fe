// The host side of the hot calls in native code: each function here allocates a call's outputs and temporaries and
// issues its launches through the C-ABI of libmxfp8_mlp.so (include/mxfp8_mlp.h), in one step from Python.
//
// Why: at a few thousand tokens and below a pass is bound by the host.  The launches themselves cost about 3 us each
// on the host; the Python around them (an allocation 1.7 us, address and stride lookups, ctypes conversions and
// structures) cost two to three times as much again.  Same launches in the same order on the same stream as the
// Python wrappers of _native.py, so the same bits; temporaries that no tensor has to name and that live as long as each
// other share one allocation, cut into 256-byte aligned pieces (the caching allocator hands the memory on only to later
// work of the same stream).  A pass holds no more memory at its peak than with one tensor for each: 142336 tokens,
// 2048 x 6144, rank 16, 5.87 GB forward and 4.26 GB backward (6.17 and 5.18 GB with one allocation for all).  Shapes, dtypes and strides that the callers do not check themselves are
// checked here; an error of the library raises _native.NativeError with its message.  Every function runs without the
// interpreter's lock, as a ctypes call does: a launch may wait for room in the stream's queue, and other Python threads
// go on meanwhile.  Nothing below touches a Python object.
// Counterpart of the Python glue of /root/reference/scripts/fused_mlp.py:262-336, mxfp8.py:78-293 and
// fused_linear.py:219-279.
#include <torch/extension.h>

#include <algorithm>
#include <array>
#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/mxfp8_mlp.h"
#include "gemm_shape.h"

namespace py = pybind11;
using at::Tensor;
using OptT = std::optional<Tensor>;

namespace {

constexpr auto kF8 = at::kFloat8_e4m3fn, kE8 = at::kFloat8_e8m0fnu, kBF = at::kBFloat16, kF32 = at::kFloat;

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
int64_t scale_numel(int64_t rows, int64_t cols) { return cdiv(rows, 128) * (cols / 128) * 512; }
int64_t tiled_rows(int64_t r) { return cdiv(r, 16) * 16; }
int64_t ft_rows(int64_t r) { return cdiv(r, 32) * 32; }

PyObject* g_error = nullptr;  // _native.NativeError

struct NativeError : std::runtime_error {  // becomes g_error in Python
  using std::runtime_error::runtime_error;
};
[[noreturn]] void raise(const std::string& msg) { throw NativeError(msg); }
void ok(int rc, const char* name) {
  if (rc) raise(std::string(name) + " failed with code " + std::to_string(rc) + ": " + mxfp8_last_error());
}
void gpu(const Tensor& t, const char* what) {
  if (!t.is_cuda())
    raise(std::string(what) + ": tensors must be on the GPU (the MXFP8 path has no CPU implementation)");
}
void* stm(int64_t s) { return reinterpret_cast<void*>(s); }
void* ptr(const Tensor& t) { return t.data_ptr(); }
void* ptr(const OptT& t) { return t ? t->data_ptr() : nullptr; }
float* fptr(const Tensor& t) { return static_cast<float*>(t.data_ptr()); }

Tensor empty(at::IntArrayRef shape, at::ScalarType dt, const Tensor& like) {
  return at::empty(shape, like.options().dtype(dt).requires_grad(false));
}

// One allocation for temporaries with one life: sizes are taken first (take), addresses once it is made (at).  drop()
// hands the memory back for what is allocated next: the work is ordered by the stream, so its last reader may still run.
struct Arena {
  int64_t total = 0;
  Tensor buf;
  int64_t take(int64_t bytes) {
    const int64_t off = total;
    total += cdiv(bytes, 256) * 256;
    return off;
  }
  void make(const Tensor& like) { buf = empty({total}, at::kByte, like); }
  void drop() { buf.reset(); }
  void* at(int64_t off) const { return static_cast<char*>(buf.data_ptr()) + off; }
  float* f(int64_t off) const { return static_cast<float*>(at(off)); }
};

// ------------------------------------------------------------------ single calls
std::tuple<Tensor, Tensor> quant_rows(const Tensor& x, int64_t stream) {
  gpu(x, "mxfp8_quant_rows");
  const int64_t R = x.size(0), K = x.size(1);
  Tensor q = empty({R, K}, kF8, x), s = empty({scale_numel(R, K)}, kE8, x);
  if (R) ok(mxfp8_quant_rows(ptr(x), R, K, x.stride(0), ptr(q), K, ptr(s), K / 128, 0, stm(stream)), "mxfp8_quant_rows");
  return {q, s};
}

std::tuple<Tensor, Tensor> quant_tiled(const Tensor& x, int64_t stream) {
  gpu(x, "mxfp8_quant_tiled");
  const int64_t R = x.size(0), K = x.size(1);
  Tensor q = empty({tiled_rows(R), K}, kF8, x), s = empty({scale_numel(R, K)}, kE8, x);
  if (R) ok(mxfp8_quant_tiled(ptr(x), R, K, x.stride(0), ptr(q), ptr(s), stm(stream)), "mxfp8_quant_tiled");
  return {q, s};
}

std::tuple<Tensor, Tensor, Tensor, OptT> quant_lora(const Tensor& x, const Tensor& w, double scale, bool out_t,
                                                    int64_t stream) {
  gpu(x, "mxfp8_quant_lora");
  const int64_t R = x.size(0), K = x.size(1), rp = w.size(0), tpad = cdiv(R, 128) * 128;
  Tensor q = empty({tiled_rows(R), K}, kF8, x), s = empty({scale_numel(R, K)}, kE8, x), out = empty({R, rp}, kBF, x);
  OptT outT;
  if (out_t) outT = empty({rp, tpad}, kBF, x);
  ok(mxfp8_quant_lora(ptr(x), R, K, x.stride(0), ptr(q), ptr(s), ptr(w), rp, (float)scale, ptr(out), ptr(outT), tpad,
                      stm(stream)),
     "mxfp8_quant_lora");
  return {q, s, out, outT};
}

// mxfp8.mx_mm for the shapes without a workspace (every layout but the explicit 8-wave one)
Tensor gemm(const Tensor& q, const Tensor& s, const Tensor& w, const Tensor& ws, const OptT& out_, const OptT& P,
            const OptT& Q, double alpha, int64_t layout, int64_t M, int64_t stream) {
  gpu(q, "mxfp8_gemm_nt");
  const int64_t N = w.size(0), K = q.size(1);
  Tensor out = out_ ? *out_ : empty({layout & MXFP8_GEMM_C_FT ? ft_rows(M) : M, N}, kBF, q);
  if (M)
    ok(mxfp8_gemm_nt(ptr(q), ptr(s), q.stride(0), ptr(w), ptr(ws), w.stride(0), M, N, K, ptr(out), out.stride(0), ptr(P),
                     P ? P->stride(0) : 0, ptr(Q), Q ? Q->stride(0) : 0, P ? P->size(1) : 0, (float)alpha, layout, nullptr,
                     0, stm(stream)),
       "mxfp8_gemm_nt");
  return out;
}

std::vector<Tensor> gemm_seg(const Tensor& q, const Tensor& s, const Tensor& w, const Tensor& ws,
                             const std::vector<int64_t>& widths, const OptT& P, const OptT& Q, double alpha,
                             int64_t layout, int64_t M, const std::vector<int64_t>& rcols, int64_t r, int64_t stream) {
  gpu(q, "mxfp8_gemm_nt_seg");
  const int64_t N = w.size(0), K = q.size(1), n = (int64_t)widths.size();
  TORCH_CHECK(n >= 1 && n <= 4, "gemm_seg: 1 to 4 outputs");
  std::vector<Tensor> outs;
  int64_t col0[4], ld[4], c0 = 0;
  void* p[4];
  for (int64_t k = 0; k < n; ++k) {
    outs.push_back(empty({M, widths[k]}, kBF, q));
    col0[k] = c0;
    ld[k] = widths[k];
    p[k] = ptr(outs.back());
    c0 += widths[k];
  }
  TORCH_CHECK(c0 == N && (rcols.empty() || (int64_t)rcols.size() == n), "gemm_seg: widths must sum to N");
  if (M)
    ok(mxfp8_gemm_nt_seg(ptr(q), ptr(s), q.stride(0), ptr(w), ptr(ws), w.stride(0), M, N, K, n, col0, p, ld, ptr(P),
                         P ? P->stride(0) : 0, ptr(Q), Q ? Q->stride(0) : 0, P ? (rcols.empty() ? P->size(1) : r) : 0,
                         rcols.empty() ? nullptr : rcols.data(), (float)alpha, layout, stm(stream)),
       "mxfp8_gemm_nt_seg");
  return outs;
}

// The rule by which the library takes a GEMM's workgroup shape: (shape, shape of the rows from tail_row on, tail_row).
std::tuple<std::string, std::optional<std::string>, int64_t> gemm_shape(int64_t M, int64_t N, int64_t K, int64_t kind,
                                                                        int64_t cus) {
  TORCH_CHECK(M > 0 && N > 0 && K > 0 && M < (1LL << 30) && N < (1LL << 30) && K < (1LL << 30) && N % 128 == 0 &&
                  K % 128 == 0 && kind >= 0 && kind <= mxk::kGemmSeg && cus > 0 && cus < (1 << 20),
              "gemm_shape: bad size or kind");
  const auto name = [](mxk::ShapeId id) {
    const auto& c = mxk::kCost[(int)id];
    return std::to_string(c.bm) + "x" + std::to_string(c.bn);
  };
  const mxk::Pick p = mxk::pick_shape(M, N, K, (int)cus, (mxk::GemmKind)kind);
  return {name(p.shape), p.tail_row ? std::optional<std::string>(name(p.tail)) : std::nullopt, p.tail_row};
}

using TnJob = std::tuple<Tensor, Tensor, Tensor, double, bool>;  // x, p, out, scale, transpose

Tensor gemm_tn(const Tensor& q, const Tensor& s, const Tensor& w, const Tensor& ws, const Tensor& P, const Tensor& Q,
               double alpha, int64_t layout, int64_t M, const std::vector<TnJob>& jobs, const Tensor& part,
               int64_t stream) {
  gpu(q, "mxfp8_gemm_nt_tn");
  const int64_t N = w.size(0), K = q.size(1), n = (int64_t)jobs.size();
  TORCH_CHECK(n >= 1 && n <= MXFP8_LORA_TN_MAX_JOBS, "gemm_tn: 1 to ", MXFP8_LORA_TN_MAX_JOBS, " reductions");
  mxfp8_lora_tn_job table[MXFP8_LORA_TN_MAX_JOBS];
  const int64_t T = std::get<0>(jobs[0]).size(0), Kt = std::get<0>(jobs[0]).size(1);
  const int64_t chunks = mxfp8_lora_tn_chunks(T, Kt);
  int64_t ranks = 0;
  for (int64_t k = 0; k < n; ++k) {
    const auto& [x, p, o, sc, tr] = jobs[k];
    table[k] = {ptr(x), x.stride(0), ptr(p), p.size(1), (float)sc, tr, o.scalar_type() == kF32, ptr(o)};
    ranks += p.size(1);
  }
  if (part.numel() < chunks * ranks * Kt) raise("lora_tn_batch: partial buffer too small");
  Tensor out = empty({layout & MXFP8_GEMM_C_FT ? ft_rows(M) : M, N}, kBF, q);
  ok(mxfp8_gemm_nt_tn(ptr(q), ptr(s), q.stride(0), ptr(w), ptr(ws), w.stride(0), M, N, K, ptr(out), out.stride(0), ptr(P),
                      P.stride(0), ptr(Q), Q.stride(0), P.size(1), (float)alpha, layout, table, n, T, Kt, chunks,
                      fptr(part), stm(stream)),
     "mxfp8_gemm_nt_tn");
  return out;
}

Tensor res_lora(const Tensor& x, const Tensor& y, const Tensor& xa, const Tensor& B, double scale, int64_t stream) {
  gpu(x, "mxfp8_res_lora");
  Tensor out = at::empty_like(x);
  if (x.size(0))
    ok(mxfp8_res_lora(ptr(x), ptr(y), ptr(xa), xa.stride(0), ptr(B), x.size(0), x.size(1), B.size(1), (float)scale,
                      ptr(out), stm(stream)),
       "mxfp8_res_lora");
  return out;
}

// mxfp8.lora_bwd / lora_bwd_batch of a group's MX layers (one common rank): codes of every dy side by side in q (in the
// MX-tiled layout, the same bytes in the order that the dx GEMM streams), each layer's d(xa) in its columns of dS, and
// the layers' dB.
std::tuple<OptT, OptT, std::vector<Tensor>> group_lora_bwd(const std::vector<Tensor>& dys, const Tensor& xS,
                                                           const std::vector<Tensor>& Bs,
                                                           const std::vector<int64_t>& cols,
                                                           const std::vector<double>& scales, const Tensor& dS,
                                                           bool need_q, int64_t stream) {
  const int64_t n = (int64_t)dys.size();
  TORCH_CHECK(n >= 1 && n <= MXFP8_LORA_BWD_MAX_JOBS && (int64_t)Bs.size() == n && (int64_t)cols.size() == n &&
                  (int64_t)scales.size() == n && dys[0].size(0) > 0,
              "group_lora_bwd: 1 to 8 layers, T > 0");
  const int64_t T = dys[0].size(0), R = Bs[0].size(1);
  TORCH_CHECK(xS.scalar_type() == kBF && dS.scalar_type() == kBF && xS.stride(1) == 1 && dS.stride(1) == 1 &&
                  xS.size(0) == T && dS.size(0) == T,
              "group_lora_bwd: xS and dS [T, *] bf16 with unit column stride");
  for (int64_t k = 0; k < n; ++k) {
    const int64_t N = dys[k].size(1);
    TORCH_CHECK(dys[k].scalar_type() == kBF && dys[k].size(0) == T && dys[k].stride(1) == 1 && N % 128 == 0 &&
                    Bs[k].is_contiguous() && Bs[k].size(0) == N && Bs[k].size(1) == R && Bs[k].scalar_type() == kBF,
                "group_lora_bwd: dy [T, N] bf16 with unit column stride, N % 128 == 0, and B [N, r] bf16 contiguous");
    TORCH_CHECK(cols[k] >= 0 && cols[k] + R <= xS.size(1) && cols[k] + R <= dS.size(1),
                "group_lora_bwd: columns ", cols[k], " to ", cols[k] + R, " of xS and dS");
  }
  gpu(dys[0], "mxfp8_lora_bwd");
  int64_t sum_n = 0;
  for (const auto& d : dys) sum_n += d.size(1);
  OptT q, s;
  if (need_q) {
    q = empty({tiled_rows(T), sum_n}, kF8, dys[0]);
    s = empty({scale_numel(T, sum_n)}, kE8, dys[0]);
  }
  const int64_t chunks = mxfp8_lora_bwd_batch_chunks(T, sum_n);
  Arena a;
  int64_t pdx[MXFP8_LORA_BWD_MAX_JOBS], pdb[MXFP8_LORA_BWD_MAX_JOBS];
  std::vector<Tensor> dbs;
  for (int64_t k = 0; k < n; ++k) {
    const int64_t N = dys[k].size(1);
    pdx[k] = a.take(N / 128 * T * R * 4);
    pdb[k] = a.take(chunks * N * R * 4);
    dbs.push_back(empty({N, R}, kF32, dys[k]));
  }
  a.make(dys[0]);
  auto* xs = static_cast<uint16_t*>(xS.data_ptr());
  auto* ds = static_cast<uint16_t*>(dS.data_ptr());
  mxfp8_lora_bwd_job jobs[MXFP8_LORA_BWD_MAX_JOBS];
  int64_t tile = 0;
  for (int64_t k = 0; k < n; ++k) {
    const int64_t N = dys[k].size(1);
    jobs[k] = {ptr(dys[k]), N,         dys[k].stride(0), need_q ? tile : 0, xs + cols[k], xS.stride(0), ptr(Bs[k]),
               (float)scales[k], ds + cols[k], dS.stride(0), fptr(dbs[k]), a.f(pdx[k]), a.f(pdb[k])};
    tile += N / 128;
  }
  ok(mxfp8_lora_bwd_batch(jobs, n, T, R, ptr(q), need_q ? sum_n : 0, ptr(s), need_q ? sum_n / 128 : 0, need_q, stm(stream)),
     "mxfp8_lora_bwd_batch");
  return {q, s, dbs};
}

// ------------------------------------------------------------------ the fused MLP
// A weight's codes have as many columns as the product sums over: the adapters of a layer may fit where its base weight
// does not, and the kernels would read past it.
void check_cols(const char* what, const Tensor& w, int64_t k) {
  TORCH_CHECK(w.dim() == 2 && w.size(1) == k, what, " of ", w.sizes(), ", a product over ", k, " columns");
}

// Every bf16 form of the step's LoRA weights (fused_mlp._prep): S, ST, bg, bu, bgT, buT, ad, adT, bd, bdT.
std::vector<Tensor> mlp_forms(const std::array<Tensor, 6>& w, int64_t stream) {
  gpu(w[0], "mxfp8_lora_prep");
  std::array<Tensor, 6> f;
  for (int i = 0; i < 6; ++i) f[i] = w[i].detach().to(kF32).contiguous();
  const Tensor &Ag = f[0], &Bg = f[1], &Au = f[2], &Bu = f[3], &Ad = f[4], &Bd = f[5];
  const int64_t R = Ag.size(0), K = Ag.size(1), N = Bg.size(0);
  const std::array<std::array<int64_t, 2>, 10> sh = {{{2 * R, K}, {K, 2 * R}, {N, R}, {N, R}, {R, N}, {R, N}, {R, N},
                                                      {N, R}, {K, R}, {R, K}}};
  std::vector<Tensor> o;
  for (const auto& d : sh) o.push_back(empty({d[0], d[1]}, kBF, Ag));
  ok(mxfp8_lora_prep(fptr(Ag), fptr(Au), fptr(Bg), fptr(Bu), fptr(Ad), fptr(Bd), R, K, N, ptr(o[0]), ptr(o[1]), ptr(o[2]),
                     ptr(o[3]), ptr(o[4]), ptr(o[5]), ptr(o[6]), ptr(o[7]), ptr(o[8]), ptr(o[9]), stm(stream)),
     "mxfp8_lora_prep");
  return o;
}

// fused_mlp._MLP.forward with its default switches, after the weight forms: (y, xs, gu).  fold_sum: the largest T * R
// whose xS_down partials the down GEMM's launch sums.
std::tuple<Tensor, Tensor, Tensor> mlp_forward(const Tensor& x, const Tensor& S, const Tensor& bg, const Tensor& bu,
                                               const Tensor& ad, const Tensor& bd, const Tensor& wf, const Tensor& wfs,
                                               const Tensor& wd, const Tensor& wds, double s_g, double s_u, double s_d,
                                               int64_t fold_sum, int64_t stream) {
  const int64_t T = x.size(0), K = x.size(1), R = ad.size(0), N = ad.size(1);
  check_cols("mlp_forward: gate|up weight", wf, K);
  check_cols("mlp_forward: down weight", wd, N);
  gpu(x, "mxfp8_gemm_swiglu_fwd");
  Tensor xs = empty({T, 2 * R}, kBF, x), gu = empty({ft_rows(T), 2 * N}, kBF, x), y;
  const int64_t parts = 2 * N / 128;
  const bool fold = R == 16 && T * R <= fold_sum;
  // a: the codes of x, dropped after the gate|up GEMM; b: the codes of h; the xS_down partials and their sum in b where the
  // down GEMM makes it, else the partials in c, dropped after their sum
  Arena a, b, c;
  Arena& p = fold ? b : c;
  const int64_t q = a.take(tiled_rows(T) * K), s = a.take(scale_numel(T, K));
  const int64_t qh = b.take(tiled_rows(T) * N), sh = b.take(scale_numel(T, N)), part = p.take(parts * T * R * 4),
                xsd_b = fold ? b.take(T * R * 2) : 0;
  a.make(x);
  b.make(x);
  if (!fold) c.make(x);
  ok(mxfp8_quant_lora(ptr(x), T, K, x.stride(0), a.at(q), a.at(s), ptr(S), 2 * R, 1.f, ptr(xs), nullptr,
                      cdiv(T, 128) * 128, stm(stream)),
     "mxfp8_quant_lora");
  ok(mxfp8_gemm_swiglu_fwd(a.at(q), a.at(s), ptr(wf), ptr(wfs), T, N, K, ptr(xs), ptr(bg), ptr(bu), ptr(ad), R,
                           (float)s_g, (float)s_u, ptr(gu), b.at(qh), b.at(sh), p.f(part), stm(stream)),
     "mxfp8_gemm_swiglu_fwd");
  a.drop();
  Tensor xsd;
  if (!fold) {
    xsd = empty({T, R}, kBF, x);
    ok(mxfp8_sum_parts(c.f(part), parts, T * R, 1.f, ptr(xsd), 1, stm(stream)), "mxfp8_sum_parts");
    c.drop();
  }
  y = empty({T, wd.size(0)}, kBF, x);
  const int64_t lay = MXFP8_GEMM_A_TILED | MXFP8_GEMM_B_TILED | MXFP8_GEMM_B_PI;
  if (fold)
    ok(mxfp8_gemm_nt_sum(b.at(qh), b.at(sh), N, ptr(wd), ptr(wds), N, T, wd.size(0), N, ptr(y), y.stride(0), b.f(part),
                         parts, 1.f, b.at(xsd_b), ptr(bd), bd.stride(0), R, (float)s_d, lay, -1, stm(stream)),
       "mxfp8_gemm_nt_sum");
  else
    ok(mxfp8_gemm_nt(b.at(qh), b.at(sh), N, ptr(wd), ptr(wds), N, T, wd.size(0), N, ptr(y), y.stride(0), ptr(xsd), R,
                     ptr(bd), bd.stride(0), R, (float)s_d, lay, nullptr, 0, stm(stream)),
       "mxfp8_gemm_nt");
  return {y, xs, gu};
}

// The same without the output (a checkpoint's recompute): (xs, gu).
std::tuple<Tensor, Tensor> mlp_graph(const Tensor& x, const Tensor& S, const Tensor& w, const Tensor& ws, int64_t N,
                                     int64_t stream) {
  const int64_t T = x.size(0), K = x.size(1), rp = S.size(0);
  check_cols("mlp_graph: gate|up weight", w, K);
  gpu(x, "mxfp8_gemm_nt");
  Tensor xs = empty({T, rp}, kBF, x), gu = empty({ft_rows(T), 2 * N}, kBF, x);
  Arena a;
  const int64_t q = a.take(tiled_rows(T) * K), s = a.take(scale_numel(T, K));
  a.make(x);
  ok(mxfp8_quant_lora(ptr(x), T, K, x.stride(0), a.at(q), a.at(s), ptr(S), rp, 1.f, ptr(xs), nullptr,
                      cdiv(T, 128) * 128, stm(stream)),
     "mxfp8_quant_lora");
  ok(mxfp8_gemm_nt(a.at(q), a.at(s), K, ptr(w), ptr(ws), K, T, 2 * N, K, ptr(gu), 2 * N, nullptr, 0, nullptr, 0, 0, 1.f,
                   MXFP8_GEMM_A_TILED | MXFP8_GEMM_B_TILED | MXFP8_GEMM_C_FT, nullptr, 0, stm(stream)),
     "mxfp8_gemm_nt");
  return {xs, gu};
}

// fused_mlp._MLP.backward with its default switches: (dx or None, dA [2R, K], dB_g, dB_u, dA_d, dB_d).  f: S, ST, bg,
// bu, bgT, buT, ad, adT, bd, bdT (mlp_forms); wt: W_downᵀ in the dgrad row order; wx: W_guᵀ in the pi_col order.
std::tuple<OptT, Tensor, Tensor, Tensor, Tensor, Tensor> mlp_backward(
    const Tensor& dy, const Tensor& x, const Tensor& xs, const Tensor& gu, const std::vector<Tensor>& f, const Tensor& wt,
    const Tensor& wts, const Tensor& wx, const Tensor& wxs, double s_g, double s_u, double s_d, int64_t SB, int64_t CG,
    bool wide, bool need_x, bool fp32_a, bool fp32_bd, int64_t stream) {
  TORCH_CHECK(f.size() == 10, "mlp_backward: ten weight forms");
  const Tensor &ST = f[1], &bg = f[2], &bu = f[3], &bgT = f[4], &buT = f[5], &ad = f[6], &adT = f[7], &bdT = f[9];
  const int64_t T = dy.size(0), K = x.size(1), R = ad.size(0), N = ad.size(1), tpad = cdiv(T, 128) * 128;
  check_cols("mlp_backward: down weight", wt, dy.size(1));
  check_cols("mlp_backward: gate|up weight", wx, 2 * N);
  gpu(dy, "mxfp8_mlp_bwd");
  const int64_t nsb = cdiv(tpad, SB), n_dxa = N / (wide ? 256 : 128), chunks = mxfp8_lora_tn_chunks(T, K);
  // m: dhm, dropped after the backward kernel; a, dropped after the finish: the codes of dy (read by the dh GEMM) under the
  // partials (written after it); b: the codes of dg | du, and dxd and the transposed operands (read by the backward
  // kernel) under the finish's results; c: the token reductions' partials, made when a is gone
  Arena m, a, b, c;
  const int64_t dhm = m.take(ft_rows(T) * N * 2);
  const int64_t qd = a.take(tiled_rows(T) * dy.size(1)), sd = a.take(scale_numel(T, dy.size(1))), end_a = a.total;
  a.total = 0;
  const int64_t dxa_p = a.take(n_dxa * T * 3 * R * 4), dbg_p = a.take(nsb * N * R * 4), dbu_p = a.take(nsb * N * R * 4),
                dad_p = a.take(nsb * R * N * 4);
  a.total = std::max(a.total, end_a);
  const int64_t qg = need_x ? b.take(tiled_rows(T) * 2 * N) : 0, sg = need_x ? b.take(scale_numel(T, 2 * N)) : 0,
                under_b = b.total;
  const int64_t dxd = b.take(T * R * 2), dxdT = b.take(R * tpad * 2), xsT = b.take(2 * R * tpad * 2), end_b = b.total;
  b.total = under_b;
  const int64_t dxa = b.take(T * 2 * R * 2), xsd = b.take(T * R * 2);
  b.total = std::max(b.total, end_b);
  const int64_t part = c.take(chunks * 3 * R * K * 4);
  a.make(dy);
  m.make(dy);
  b.make(dy);
  void* const st = stm(stream);
  ok(mxfp8_quant_lora_tp(ptr(dy), T, dy.size(1), dy.stride(0), a.at(qd), a.at(sd), ptr(bdT), R, (float)s_d, b.at(dxd),
                         b.at(dxdT), tpad, ptr(xs), xs.stride(0), 2 * R, b.at(xsT), st),
     "mxfp8_quant_lora_tp");
  const int64_t tt = MXFP8_GEMM_A_TILED | MXFP8_GEMM_B_TILED;
  ok(mxfp8_gemm_nt(a.at(qd), a.at(sd), dy.size(1), ptr(wt), ptr(wts), dy.size(1), T, N, dy.size(1), m.at(dhm), N, nullptr,
                   0, nullptr, 0, 0, 1.f, tt | MXFP8_GEMM_C_FT | MXFP8_GEMM_B_PI, nullptr, 0, st),
     "mxfp8_gemm_nt");
  ok(mxfp8_mlp_bwd(ptr(gu), ptr(xs), b.at(xsT), m.at(dhm), b.at(dxd), b.at(dxdT), ptr(bg), ptr(bu), ptr(bgT), ptr(buT),
                   ptr(ad), ptr(adT), T, N, R, (float)s_g, (float)s_u, SB, CG, need_x ? b.at(qg) : nullptr,
                   need_x ? b.at(sg) : nullptr, a.f(dxa_p), a.f(dbg_p), a.f(dbu_p), a.f(dad_p), nullptr,
                   1 | 2 | (wide ? 4 : 0), st),
     "mxfp8_mlp_bwd");
  m.drop();
  Tensor dBg = empty({N, R}, kF32, dy), dBu = empty({N, R}, kF32, dy), dAd = empty({R, N}, kF32, dy);
  ok(mxfp8_mlp_bwd_finish(a.f(dxa_p), a.f(dbg_p), a.f(dbu_p), a.f(dad_p), n_dxa, nsb, T, N, R, (float)s_g, (float)s_u,
                          b.at(dxa), b.at(xsd), fptr(dBg), fptr(dBu), fptr(dAd), st),
     "mxfp8_mlp_bwd_finish");
  a.drop();
  c.make(dy);
  Tensor dA = empty({2 * R, K}, fp32_a ? kF32 : kBF, dy), dBd = empty({K, R}, fp32_bd ? kF32 : kBF, dy);
  const mxfp8_lora_tn_job jobs[2] = {{ptr(dy), dy.stride(0), b.at(xsd), R, (float)s_d, 1, fp32_bd, ptr(dBd)},
                                     {ptr(x), x.stride(0), b.at(dxa), 2 * R, 1.f, 0, fp32_a, ptr(dA)}};
  const bool fold = need_x && R == 16;
  if (!fold) ok(mxfp8_lora_tn_batch(jobs, 2, T, K, chunks, c.f(part), st), "mxfp8_lora_tn_batch");
  OptT dx;
  if (need_x) {
    dx = empty({T, K}, kBF, dy);
    const int64_t lay = tt | MXFP8_GEMM_B_PI;
    if (fold)
      ok(mxfp8_gemm_nt_tn(b.at(qg), b.at(sg), 2 * N, ptr(wx), ptr(wxs), 2 * N, T, K, 2 * N, ptr(dx), K, b.at(dxa), 2 * R,
                          ptr(ST), ST.stride(0), 2 * R, 1.f, lay, jobs, 2, T, K, chunks, c.f(part), st),
         "mxfp8_gemm_nt_tn");
    else
      ok(mxfp8_gemm_nt(b.at(qg), b.at(sg), 2 * N, ptr(wx), ptr(wxs), 2 * N, T, K, 2 * N, ptr(dx), K, b.at(dxa), 2 * R,
                       ptr(ST), ST.stride(0), 2 * R, 1.f, lay, nullptr, 0, st),
         "mxfp8_gemm_nt");
  }
  return {dx, dA, dBg, dBu, dAd, dBd};
}

}  // namespace

PYBIND11_MODULE(_mxhost, m) {
  m.def("set_error", [](py::object e) {
    Py_XINCREF(e.ptr());
    Py_XDECREF(g_error);
    g_error = e.ptr();
  });
  py::register_local_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const NativeError& e) {
      PyErr_SetString(g_error ? g_error : PyExc_RuntimeError, e.what());
    }
  });
  m.def("abi_version", [] { return MXFP8_MLP_ABI_VERSION; });
  const auto def = [&m](const char* name, auto f) { m.def(name, f, py::call_guard<py::gil_scoped_release>()); };
  def("quant_rows", &quant_rows);
  def("quant_tiled", &quant_tiled);
  def("quant_lora", &quant_lora);
  def("gemm", &gemm);
  def("gemm_shape", &gemm_shape);
  def("gemm_seg", &gemm_seg);
  def("gemm_tn", &gemm_tn);
  def("res_lora", &res_lora);
  def("group_lora_bwd", &group_lora_bwd);
  def("mlp_forms", &mlp_forms);
  def("mlp_forward", &mlp_forward);
  def("mlp_graph", &mlp_graph);
  def("mlp_backward", &mlp_backward);
}
