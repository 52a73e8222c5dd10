// One checkpointed decoder layer's forward, and its recompute plus backward, as
// one call each: the launches of femtotron_amd/fused_layer.py's layer_forward and
// layer_backward in the same order, from C++.
//
// At a few hundred tokens the layer's 30-40 kernels take less time than Python
// needs to issue them (2048-wide bf16 layer at 256 tokens: 358 us of kernels, 688
// us of wall time): every op costs its tensors, its checks and a foreign call.
// Here a call costs its argument block, and every intermediate lies in one
// workspace (377 us).  Layouts and arithmetic are those of the entry points called.
#include <algorithm>

#include "fh_common.hpp"

namespace {

using fh::fail;

// Byte offsets of consecutive 256-byte aligned buffers.
struct Arena {
  size_t at = 0;
  size_t take(size_t bytes) {
    const size_t off = at;
    at += (bytes + 255) & ~size_t(255);
    return off;
  }
};

struct Sizes {
  int64_t T, H, F, hq, hkv, nqkv;
  size_t e;  // bytes per element
  explicit Sizes(const fh_layer& l)
      : T(l.batch * l.seq_len), H(l.hidden), F(l.ffn), hq(l.n_heads * l.head_dim), hkv(l.n_kv_heads * l.head_dim),
        nqkv(hq + 2 * hkv), e(l.dt == FH_BF16 ? 2 : 4) {}
  size_t mat(int64_t cols) const { return static_cast<size_t>(T) * cols * e; }
};

int check_layer(const fh_layer* l) {
  FH_REQUIRE(l != nullptr, "layer: null argument block");
  FH_REQUIRE(l->dt == FH_BF16 || l->dt == FH_F32, "layer: dtype must be FH_BF16 or FH_F32");
  FH_REQUIRE(l->batch > 0 && l->seq_len > 0 && l->hidden > 0 && l->ffn > 0 && l->n_heads > 0 && l->n_kv_heads > 0 &&
                 l->head_dim > 0,
             "layer: sizes must be positive");
  return FH_OK;
}

size_t gemm_ws(const fh_layer& l, int op, int64_t m, int64_t n, int64_t k) {
  return l.dt == FH_BF16 ? fh_gemm_bf16_any_k_workspace_size(op, m, n, k) : 0;
}

int gemm(const fh_layer& l, int op, const void* a, int64_t lda, const void* b, int64_t ldb, void* c, int64_t ldc,
         const void* residual, int64_t m, int64_t n, int64_t k, void* ws, hipStream_t s) {
  return l.dt == FH_BF16 ? fh_gemm_bf16_any_k(op, a, lda, b, ldb, c, ldc, residual, ldc, m, n, k, ws, s)
                         : fh_gemm_f32(op, a, lda, b, ldb, c, ldc, residual, ldc, m, n, k, s);
}

// Workspace of the forward products (q/k/v, o, gate/up, down).
size_t forward_gemm_ws(const fh_layer& l, const Sizes& z) {
  return std::max(std::max(gemm_ws(l, FH_GEMM_NT, z.T, z.nqkv, z.H), gemm_ws(l, FH_GEMM_NT, z.T, z.H, z.hq)),
                  std::max(gemm_ws(l, FH_GEMM_NT, z.T, 2 * z.F, z.H), gemm_ws(l, FH_GEMM_NT, z.T, z.H, z.F)));
}

struct FwdPlan {
  size_t y, qkv, o, a, p, gu, ws, total;
};

// y holds RMSNorm1's output, then RMSNorm2's; p takes the place of qkv, o and a.
FwdPlan fwd_plan(const fh_layer& l) {
  const Sizes z(l);
  FwdPlan f{};
  Arena ar;
  f.y = ar.take(z.mat(z.H));
  f.gu = ar.take(z.mat(2 * z.F));
  f.p = ar.at;
  f.qkv = ar.take(z.mat(z.nqkv));
  f.o = ar.take(z.mat(z.hq));
  f.a = ar.take(z.mat(z.H));
  if (ar.at - f.p < z.mat(z.F)) ar.take(z.mat(z.F) - (ar.at - f.p));
  f.ws = ar.take(forward_gemm_ws(l, z));
  f.total = ar.at;
  return f;
}

// The last three weight gradients as one group (bf16).
void fill_group(const Sizes& z, fh_gemm_problem (&g)[3]) {
  g[0] = fh_gemm_problem{nullptr, z.H, nullptr, z.F, nullptr, z.F, nullptr, z.F, z.H, z.F};         // down
  g[1] = fh_gemm_problem{nullptr, z.H, nullptr, z.hq, nullptr, z.hq, nullptr, z.hq, z.H, z.hq};     // o
  g[2] = fh_gemm_problem{nullptr, z.nqkv, nullptr, z.H, nullptr, z.H, nullptr, z.H, z.nqkv, z.H};  // q/k/v
}

struct BwdPlan {
  size_t y1, rstd1, qkv, o, lse, h, rstd2, zz, gu, dp, dgu, a, t, dh, dqkv, ws, total;
};

// a (the o projection) lies where dgu will be; t (dz, then dO, then dy1), dh and
// dqkv take gu's place once the SwiGLU backward has read it.
BwdPlan bwd_plan(const fh_layer& l) {
  const Sizes z(l);
  BwdPlan b{};
  Arena ar;
  b.y1 = ar.take(z.mat(z.H));
  b.rstd1 = ar.take(static_cast<size_t>(z.T) * 4);
  b.qkv = ar.take(z.mat(z.nqkv));
  b.o = ar.take(z.mat(z.hq));
  b.lse = ar.take(static_cast<size_t>(z.T) * l.n_heads * 4);
  b.h = ar.take(z.mat(z.H));
  b.rstd2 = ar.take(static_cast<size_t>(z.T) * 4);
  b.zz = ar.take(z.mat(z.H));
  b.gu = b.t = ar.at;
  ar.take(z.mat(std::max(z.H, z.hq)));
  b.dh = ar.take(z.mat(z.H));
  b.dqkv = ar.take(z.mat(z.nqkv));
  if (ar.at - b.gu < z.mat(2 * z.F)) ar.take(z.mat(2 * z.F) - (ar.at - b.gu));
  b.dp = ar.take(z.mat(z.F));
  b.dgu = b.a = ar.take(z.mat(std::max(2 * z.F, z.H)));
  size_t ws = forward_gemm_ws(l, z);
  ws = std::max(ws, gemm_ws(l, FH_GEMM_NN, z.T, z.F, z.H));
  ws = std::max(ws, gemm_ws(l, FH_GEMM_TN, 2 * z.F, z.H, z.T));
  ws = std::max(ws, gemm_ws(l, FH_GEMM_NN, z.T, z.H, 2 * z.F));
  ws = std::max(ws, gemm_ws(l, FH_GEMM_NN, z.T, z.hq, z.H));
  ws = std::max(ws, gemm_ws(l, FH_GEMM_NN, z.T, z.H, z.nqkv));
  if (l.dt == FH_BF16) {
    fh_gemm_problem g[3];
    fill_group(z, g);
    ws = std::max(ws, fh_gemm_bf16_grouped_any_k_workspace_size(FH_GEMM_TN, 3, g, z.T));
  }
  ws = std::max(ws, fh_rmsnorm_bwd_workspace_size(z.T, z.H));
  ws = std::max(ws, fh_attn_bwd_call_workspace_size(l.dt, l.batch, l.seq_len, l.n_heads, l.n_kv_heads, l.head_dim));
  b.ws = ar.take(ws);
  b.total = ar.at;
  return b;
}

#define FH_TRY(call)          \
  do {                        \
    if (int e_ = (call)) return e_; \
  } while (0)

// q/k/v projection, RoPE (k by a pass, q as attention loads it) and attention.
int qkv_attention(const fh_layer& l, const Sizes& z, const void* y, char* qkv, void* o, float* lse, bool keep,
                  void* ws, hipStream_t s) {
  FH_TRY(gemm(l, FH_GEMM_NT, y, z.H, l.wqkv, z.H, qkv, z.nqkv, nullptr, z.T, z.nqkv, z.H, ws, s));
  char* k = qkv + z.hq * z.e;
  char* v = k + z.hkv * z.e;
  FH_TRY(fh_rope_fwd(l.dt, k, z.nqkv, z.T, l.seq_len, l.n_kv_heads, l.head_dim, l.cos, l.sin, l.cos_per_token, s));
  return fh_attn_fwd_rope(l.dt, qkv, z.nqkv, k, z.nqkv, v, z.nqkv, o, z.hq, lse, keep ? qkv : nullptr,
                          keep ? z.nqkv : 0, l.batch, l.seq_len, l.n_heads, l.n_kv_heads, l.head_dim, l.scale, l.cos,
                          l.sin, l.cos_per_token, s);
}

}  // namespace

extern "C" size_t fh_layer_workspace_size(const fh_layer* layer, int backward) {
  if (check_layer(layer)) return 0;
  return backward ? bwd_plan(*layer).total : fwd_plan(*layer).total;
}

extern "C" int fh_layer_fwd(const fh_layer* layer, const void* x, void* out, void* workspace, hipStream_t s) {
  FH_TRY(check_layer(layer));
  FH_REQUIRE(x && out && workspace && fh::aligned16(workspace), "layer_fwd: null or misaligned buffer");
  FH_REQUIRE(out != x, "layer_fwd: out must not be x");
  const fh_layer& l = *layer;
  const Sizes z(l);
  const FwdPlan f = fwd_plan(l);
  char* w = static_cast<char*>(workspace);
  FH_TRY(fh_rmsnorm_fwd(l.dt, x, l.w1, w + f.y, nullptr, z.T, z.H, l.eps1, s));
  FH_TRY(qkv_attention(l, z, w + f.y, w + f.qkv, w + f.o, nullptr, false, w + f.ws, s));
  FH_TRY(gemm(l, FH_GEMM_NT, w + f.o, z.hq, l.wo, z.hq, w + f.a, z.H, nullptr, z.T, z.H, z.hq, w + f.ws, s));
  FH_TRY(fh_add_rmsnorm_fwd(l.dt, x, w + f.a, l.w2, out, w + f.y, nullptr, z.T, z.H, l.eps2, s));
  FH_TRY(gemm(l, FH_GEMM_NT, w + f.y, z.H, l.wgu, z.H, w + f.gu, 2 * z.F, nullptr, z.T, 2 * z.F, z.H, w + f.ws, s));
  FH_TRY(fh_swiglu_fwd(l.dt, w + f.gu, w + f.gu + z.F * z.e, 2 * z.F, w + f.p, z.F, z.T, z.F, s));
  return gemm(l, FH_GEMM_NT, w + f.p, z.F, l.wd, z.F, out, z.H, out, z.T, z.H, z.F, w + f.ws, s);
}

extern "C" int fh_layer_bwd(const fh_layer* layer, const void* x, const void* dout, void* dx, void* dwqkv, void* dwo,
                            void* dwgu, void* dwd, void* dw1, void* dw2, int accumulate, void* workspace,
                            hipStream_t s) {
  FH_TRY(check_layer(layer));
  FH_REQUIRE(x && dout && dx && dwqkv && dwo && dwgu && dwd && dw1 && dw2 && workspace && fh::aligned16(workspace),
             "layer_bwd: null or misaligned buffer");
  const fh_layer& l = *layer;
  FH_REQUIRE(accumulate == 0 || l.dt == FH_BF16, "layer_bwd: gradients accumulate in bf16 only");
  const Sizes z(l);
  const BwdPlan b = bwd_plan(l);
  char* w = static_cast<char*>(workspace);
  void* ws = w + b.ws;
  float* rstd1 = reinterpret_cast<float*>(w + b.rstd1);
  float* rstd2 = reinterpret_cast<float*>(w + b.rstd2);
  float* lse = reinterpret_cast<float*>(w + b.lse);
  auto into = [&](int bit, void* g) -> const void* { return accumulate & bit ? g : nullptr; };

  // The recompute, up to the gate/up projection.
  FH_TRY(fh_rmsnorm_fwd(l.dt, x, l.w1, w + b.y1, rstd1, z.T, z.H, l.eps1, s));
  FH_TRY(qkv_attention(l, z, w + b.y1, w + b.qkv, w + b.o, lse, true, ws, s));
  FH_TRY(gemm(l, FH_GEMM_NT, w + b.o, z.hq, l.wo, z.hq, w + b.a, z.H, nullptr, z.T, z.H, z.hq, ws, s));
  FH_TRY(fh_add_rmsnorm_fwd(l.dt, x, w + b.a, l.w2, w + b.h, w + b.zz, rstd2, z.T, z.H, l.eps2, s));
  FH_TRY(gemm(l, FH_GEMM_NT, w + b.zz, z.H, l.wgu, z.H, w + b.gu, 2 * z.F, nullptr, z.T, 2 * z.F, z.H, ws, s));

  // MLP; the SwiGLU backward writes the product p over dp.
  char* dp = w + b.dp;
  char* dgu = w + b.dgu;
  FH_TRY(gemm(l, FH_GEMM_NN, dout, z.H, l.wd, z.F, dp, z.F, nullptr, z.T, z.F, z.H, ws, s));
  FH_TRY(fh_swiglu_bwd(l.dt, dp, z.F, w + b.gu, w + b.gu + z.F * z.e, 2 * z.F, dgu, dgu + z.F * z.e, 2 * z.F, dp, z.F,
                       z.T, z.F, s));
  FH_TRY(gemm(l, FH_GEMM_TN, dgu, 2 * z.F, w + b.zz, z.H, dwgu, z.H, into(FH_LAYER_DWGU, dwgu), 2 * z.F, z.H, z.T, ws,
              s));
  FH_TRY(gemm(l, FH_GEMM_NN, dgu, 2 * z.F, l.wgu, z.H, w + b.t, z.H, nullptr, z.T, z.H, 2 * z.F, ws, s));
  FH_TRY(fh_rmsnorm_bwd(l.dt, w + b.t, w + b.h, l.w2, rstd2, dout, w + b.dh, dw2, ws, z.T, z.H, l.eps2, s));

  // Attention.
  FH_TRY(gemm(l, FH_GEMM_NN, w + b.dh, z.H, l.wo, z.hq, w + b.t, z.hq, nullptr, z.T, z.hq, z.H, ws, s));
  char* q = w + b.qkv;
  char* dq = w + b.dqkv;
  const size_t ko = z.hq * z.e, vo = (z.hq + z.hkv) * z.e;
  FH_TRY(fh_attn_bwd_rope(l.dt, q, z.nqkv, q + ko, z.nqkv, q + vo, z.nqkv, w + b.o, z.hq, w + b.t, z.hq, lse, dq,
                          z.nqkv, dq + ko, z.nqkv, dq + vo, z.nqkv, ws, l.batch, l.seq_len, l.n_heads, l.n_kv_heads,
                          l.head_dim, l.scale, l.cos, l.sin, l.cos_per_token, s));
  fh_gemm_problem g[3];
  fill_group(z, g);
  g[0].a = dout, g[0].b = dp, g[0].c = dwd, g[0].residual = into(FH_LAYER_DWD, dwd);
  g[1].a = w + b.dh, g[1].b = w + b.o, g[1].c = dwo, g[1].residual = into(FH_LAYER_DWO, dwo);
  g[2].a = dq, g[2].b = w + b.y1, g[2].c = dwqkv, g[2].residual = into(FH_LAYER_DWQKV, dwqkv);
  if (l.dt == FH_BF16) {
    FH_TRY(fh_gemm_bf16_grouped_any_k(FH_GEMM_TN, 3, g, z.T, ws, s));
  } else {
    for (const fh_gemm_problem& p : g)
      FH_TRY(fh_gemm_f32(FH_GEMM_TN, p.a, p.lda, p.b, p.ldb, p.c, p.ldc, nullptr, 0, p.m, p.n, z.T, s));
  }
  FH_TRY(gemm(l, FH_GEMM_NN, dq, z.nqkv, l.wqkv, z.H, w + b.t, z.H, nullptr, z.T, z.H, z.nqkv, ws, s));
  return fh_rmsnorm_bwd(l.dt, w + b.t, x, l.w1, rstd1, w + b.dh, dx, dw1, ws, z.T, z.H, l.eps1, s);
}
