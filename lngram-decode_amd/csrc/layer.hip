// The memory layer's launches behind one call: RouteNgramMemoryV2.forward after the router
// (ffnmem/memory/lngram_v2.py:1361-1407) and memory_step (ffnmem/infer.py:152-182), each the same
// entry points and shapes as their op-by-op forms, with the intermediates in one workspace.  A layer
// of a few hundred tokens is 5 to 9 launches of 3-20 us each; launched one by one from Python, with a
// tensor allocated for every result, they took 90-140 us of host time (200-token prefill, 4 x 128 tiny
// fp32 layer, 4 x 5 cached step).
#include "common.h"

namespace lng {

// cache[b, p0 + i, r] = codes[b, i, r] (as uint8)
__global__ __launch_bounds__(256) void k_put_codes(const void* __restrict__ codes, int dt, int64_t total, int64_t nR,
                                                   int64_t seq_stride, int64_t p0R, uint8_t* __restrict__ cache) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= total) return;
  uint8_t c;
  if (dt == LNG_U8)
    c = static_cast<const uint8_t*>(codes)[i];
  else if (dt == LNG_I32)
    c = static_cast<uint8_t>(static_cast<const int32_t*>(codes)[i]);
  else
    c = static_cast<uint8_t>(static_cast<const int64_t*>(codes)[i]);
  cache[i / nR * seq_stride + p0R + i % nR] = c;
}

namespace {

struct Layout {
  size_t at = 0;
  size_t take(int64_t bytes) {
    const size_t p = at;
    at += (static_cast<size_t>(bytes) + 255) & ~size_t{255};
    return p;
  }
};

struct Dims {
  int64_t es, inner, kvi, dt;
  explicit Dims(const lng_memory_layer& L)
      : es(dtype_size(L.dtype)), inner(int64_t{L.q_heads} * L.head_dim), kvi(int64_t{L.kv_heads} * L.head_dim),
        dt(int64_t{L.n_orders} * L.mem_dim) {}
};

bool row_stats(const lng_memory_layer& L, const Dims& d) {  // the short conv takes the projection's row statistics
  return L.dtype == LNG_BF16 && L.conv_k == 4 && L.conv_dilation == 3 && L.hidden % 8 == 0 && L.hidden <= 2048 &&
         d.inner % 32 == 0;
}

struct Fwd {  // workspace offsets of one forward
  size_t q, head, mixed, rowsq = 0, norm = 0, tokens = 0, tokens_n = 0, kv = 0, total;
  Fwd(const lng_memory_layer& L, const Dims& d, int64_t M) {
    Layout w;
    q = w.take(M * d.inner * d.es);
    head = w.take(M * d.inner * d.es);
    mixed = w.take(M * L.hidden * d.es);
    if (row_stats(L, d)) rowsq = w.take(int64_t{lng_linear_rowsq_partials(L.hidden)} * M * 4);
    if (!L.fused) {
      norm = w.take(M * L.hidden * d.es);
      tokens = w.take(M * L.routes * d.dt * d.es);
      tokens_n = w.take(M * L.routes * d.dt * d.es);
      kv = w.take(M * L.routes * 2 * d.kvi * d.es);
    }
    total = w.at;
  }
};

// The query heads span the width (the fused readout reads h by rows of as many elements as q).
bool layer_ok(const lng_memory_layer* L) {
  return L && (L->dtype == LNG_BF16 || L->dtype == LNG_F32) && L->hidden > 0 && L->routes > 0 && L->n_orders >= 1 &&
         L->n_orders <= 4 && L->mem_dim > 0 && L->q_heads > 0 && L->kv_heads > 0 && L->head_dim > 0 &&
         L->q_heads % L->kv_heads == 0 && int64_t{L->q_heads} * L->head_dim == L->hidden && L->conv_k > 0 &&
         L->conv_dilation > 0 && L->w_q && L->q_norm && L->kv && L->mem_norm && L->w_o && L->conv_norm && L->conv_w &&
         (!L->fused || (L->dtype == LNG_BF16 && L->n_orders == 2 && L->orders[0] == 2 && L->orders[1] == 3 &&
                        L->mem_dim == 128 && L->bits == 4 && L->q_heads == 16 && L->kv_heads == 4 && L->head_dim == 64));
}

}  // namespace
}  // namespace lng

using namespace lng;

#define TRY(call)                   \
  do {                              \
    if (int rc = (call)) return rc; \
  } while (0)

extern "C" {

size_t lng_memory_layer_size(void) { return sizeof(lng_memory_layer); }

size_t lng_memory_forward_workspace_bytes(const lng_memory_layer* L, int64_t B, int64_t T) {
  if (!layer_ok(L) || B < 0 || T < 0) return 0;
  return Fwd(*L, Dims(*L), B * T).total;
}

int lng_memory_forward(const lng_memory_layer* L, const void* h, const void* codes, int codes_dtype, int64_t B, int64_t T,
                       void* workspace, size_t workspace_bytes, void* out, void* stream) {
  if (!layer_ok(L) || B < 0 || T < 0) return fail(LNG_E_ARG, "memory_forward: bad layer or shape");
  const int64_t M = B * T;
  if (M == 0) return LNG_OK;
  if (!h || !codes || !workspace || !out) return fail(LNG_E_ARG, "memory_forward: null buffer");
  if (L->fused && codes_dtype != LNG_U8) return fail(LNG_E_DTYPE, "memory_forward: the fused readout takes uint8 codes");
  const Dims d(*L);
  const Fwd w(*L, d, M);
  if (workspace_bytes < w.total) return fail(LNG_E_ARG, "memory_forward: workspace too small");
  char* ws = static_cast<char*>(workspace);
  void *q = ws + w.q, *head = ws + w.head, *mixed = ws + w.mixed;
  if (L->fused) {
    const bool scaled = lng_linear_rowscale_ok(M, d.inner, L->hidden) != 0;
    if (scaled)
      TRY(lng_linear_rowscale(h, L->w_q, M, d.inner, L->hidden, L->q_eps, q, stream));
    else
      TRY(lng_linear(h, L->w_q, L->dtype, M, d.inner, L->hidden, q, stream));
    TRY(lng_memory_readout_fused(q, scaled ? nullptr : h, L->q_eps, static_cast<const uint8_t*>(codes), B, T, L->routes,
                                 L->tables[0], L->tables[1], L->kv, L->mem_norm, L->mem_eps, L->scale, L->sink_logit,
                                 head, stream));
  } else {
    void *norm = ws + w.norm, *tokens = ws + w.tokens, *tokens_n = ws + w.tokens_n, *kv = ws + w.kv;
    TRY(lng_rmsnorm(h, L->q_norm, L->dtype, M, L->hidden, L->q_eps, LNG_NORM_FUSED, norm, stream));
    TRY(lng_linear(norm, L->w_q, L->dtype, M, d.inner, L->hidden, q, stream));
    TRY(lng_route_tokens(codes, codes_dtype, B, T, L->routes, 0, L->routes, L->orders, L->n_orders, L->bits, L->tables,
                         L->dtype, L->mem_dim, nullptr, nullptr, 0, tokens, stream));
    TRY(lng_rmsnorm(tokens, L->mem_norm, L->dtype, M * L->routes, static_cast<int32_t>(d.dt), L->mem_eps, LNG_NORM_FUSED,
                    tokens_n, stream));
    TRY(lng_linear(tokens_n, L->kv, L->dtype, M * L->routes, 2 * d.kvi, d.dt, kv, stream));
    const int64_t st[3] = {L->routes * 2 * d.kvi, L->head_dim, 2 * d.kvi};
    TRY(lng_sink_attention_strided(q, kv, static_cast<char*>(kv) + d.kvi * d.es, L->dtype, M, L->kv_heads,
                                   L->q_heads / L->kv_heads, L->routes, L->head_dim, st, st, L->scale, L->sink_logit,
                                   head, stream));
  }
  if (row_stats(*L, d)) {
    float* rowsq = reinterpret_cast<float*>(ws + w.rowsq);
    TRY(lng_linear_rowsq(head, L->w_o, M, L->hidden, d.inner, mixed, rowsq, stream));
    return lng_causal_conv_rowsq(mixed, rowsq, lng_linear_rowsq_partials(L->hidden), L->conv_norm, L->conv_w, B, T,
                                 L->hidden, L->conv_k, L->conv_dilation, L->conv_eps, 1, out, stream);
  }
  TRY(lng_linear(head, L->w_o, L->dtype, M, L->hidden, d.inner, mixed, stream));
  return lng_causal_conv(mixed, L->conv_norm, L->conv_w, L->dtype, B, T, L->hidden, L->conv_k, L->conv_dilation,
                         L->conv_eps, 1, out, stream);
}

int lng_memory_step(const lng_memory_layer* L, const void* h, const void* codes, int codes_dtype, int64_t B, int64_t n,
                    int64_t pos0, uint8_t* code_cache, void* conv_cache, int64_t max_len, void* workspace,
                    size_t workspace_bytes, void* out, void* stream) {
  if (!layer_ok(L) || !L->fused || B < 0 || n < 0 || pos0 < 0 || pos0 + n > max_len || B * n > 64 || L->hidden % 32)
    return fail(LNG_E_ARG, "memory_step: a fused layer, B * n <= 64 new positions inside the caches");
  if (codes_dtype != LNG_U8 && codes_dtype != LNG_I32 && codes_dtype != LNG_I64)
    return fail(LNG_E_DTYPE, "memory_step: codes u8, i32 or i64");
  const int64_t M = B * n;
  if (M == 0) return LNG_OK;
  if (!h || !codes || !code_cache || !conv_cache || !workspace || !out)
    return fail(LNG_E_ARG, "memory_step: null buffer");
  const Dims d(*L);
  const size_t half = (static_cast<size_t>(M * d.inner * d.es) + 255) & ~size_t{255};
  if (workspace_bytes < 2 * half) return fail(LNG_E_ARG, "memory_step: workspace smaller than two query rows a position");
  void *q = workspace, *head = static_cast<char*>(workspace) + half;
  const int64_t nR = n * L->routes;
  k_put_codes<<<static_cast<unsigned>(cdiv(B * nR, 256)), 256, 0, as_stream(stream)>>>(
      codes, codes_dtype, B * nR, nR, max_len * L->routes, pos0 * L->routes, code_cache);
  TRY(check_launch("memory_step (codes)"));
  TRY(lng_linear(h, L->w_q, L->dtype, M, d.inner, L->hidden, q, stream));
  TRY(lng_memory_readout_fused_at(q, h, L->q_eps, code_cache, B, n, L->routes, max_len, pos0, nullptr, L->tables[0],
                                  L->tables[1], L->kv, L->mem_norm, L->mem_eps, L->scale, L->sink_logit, head, stream));
  TRY(lng_linear_at(head, L->w_o, M, L->hidden, d.inner, n, max_len, pos0, nullptr, conv_cache, stream));
  return lng_causal_conv_at(conv_cache, L->conv_norm, L->conv_w, L->dtype, B, max_len, pos0 + n, pos0, nullptr, n,
                            L->hidden, L->conv_k, L->conv_dilation, L->conv_eps, 1, out, stream);
}

}  // extern "C"
