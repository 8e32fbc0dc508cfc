// Table gradient of one order's lookup by listed windows: the embedding backward behind the
// surrogate's pass-through (ffnmem/memory/lngram_v2.py:1084-1092, :454) without atomics on memory.
//
// A route's block of the table has S = 2^(bits*order) rows, and W = B*T positions each name one of
// them (or none).  Three kernels:
//   k_tg_keys   the address of every (position, route) as a route-major uint16 row (0xFFFF: no
//               gradient), through 64 x 64 LDS tiles so that codes are read along routes and keys
//               written along positions;
//   k_tg_sort   one block per route: a counting sort of its W keys with the S counters in LDS;
//               start[r][S + 1] and the positions in key order, perm[r][W];
//   k_tg_sum    one 16-lane group per table row: sums the row's gradient rows in fp32 registers and
//               writes the row once, in the table's dtype (zeros where no window names it).
// Bound: the gradient rows read once (W * R * D elements) and the table written once.  The atomic
// form (k_table_grad) adds W * R * D fp32 values one atomic each into a cleared fp32 table, which the
// caller then rounds: 10.5 ms an order at 8 x 2048 positions, 184 routes, D 128, bf16, whatever the
// order.  Serves the training lookups that lng_lookup_grad does not (other widths, dtypes and orders).
// The order of a row's sum varies between calls (sort_windows).
#include "window_sort.h"

namespace lng {


constexpr int TG_LONG = 1024;        // a row of more windows than this is summed by its whole block

struct TgWs {  // byte offsets in the workspace
  size_t keys, start, perm, total;
  int64_t kstride;  // uint16 elements of a route's row of keys
};
static size_t tg_al(size_t x) { return (x + 255) & ~size_t{255}; }
static TgWs tg_layout(int64_t W, int32_t R, int64_t S) {
  TgWs w{};
  w.kstride = (W + 63) / 64 * 64;
  w.keys = 0;
  w.start = tg_al(static_cast<size_t>(R) * w.kstride * 2);
  w.perm = w.start + tg_al(static_cast<size_t>(R) * (S + 1) * 4);
  w.total = w.perm + tg_al(static_cast<size_t>(R) * W * 4);
  return w;
}

struct TgArgs {
  const void* grad;  // rows of D elements, grad_stride elements apart, in (b, t, r) order
  int64_t grad_stride;
  const void* codes;
  int codes_dt;
  const uint8_t* valid;
  int64_t W, T;
  int32_t R, order, bits, shift;  // shift = bits * order
  int64_t kstride;
};

__device__ __forceinline__ uint32_t tg_code(const void* p, int dt, int64_t i, uint32_t mask) {
  if (dt == LNG_U8) return static_cast<const uint8_t*>(p)[i] & mask;
  if (dt == LNG_I32) return static_cast<uint32_t>(static_cast<const int32_t*>(p)[i]) & mask;
  return static_cast<uint32_t>(static_cast<const int64_t*>(p)[i]) & mask;
}

__global__ __launch_bounds__(256) void k_tg_keys(TgArgs a, uint16_t* __restrict__ keys) {
  __shared__ uint16_t tile[64][66];
  const int64_t w0 = static_cast<int64_t>(blockIdx.x) * 64;
  const int r0 = blockIdx.y * 64;
  const uint32_t mask = (1u << a.bits) - 1;
  for (int i = threadIdx.x; i < 64 * 64; i += 256) {
    const int wl = i >> 6, rl = i & 63;
    const int64_t w = w0 + wl;
    const int r = r0 + rl;
    uint32_t key = WIN_DEAD;
    if (w < a.W && r < a.R && w % a.T >= a.order - 1 && (a.valid == nullptr || a.valid[w])) {
      key = 0;
      for (int k = 0; k < a.order; ++k)
        key |= tg_code(a.codes, a.codes_dt, (w - (a.order - 1) + k) * a.R + r, mask) << (k * a.bits);
    }
    tile[wl][rl] = static_cast<uint16_t>(key);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 64 * 64; i += 256) {
    const int rl = i >> 6, wl = i & 63;
    if (r0 + rl < a.R) keys[(r0 + rl) * a.kstride + w0 + wl] = tile[wl][rl];  // w0 + wl < kstride
  }
}

__global__ __launch_bounds__(1024) void k_tg_sort(TgArgs a, const uint16_t* __restrict__ keys,
                                                  uint32_t* __restrict__ start, uint32_t* __restrict__ perm) {
  extern __shared__ uint32_t cnt[];  // [S + 16]
  const int64_t r = blockIdx.x, S = int64_t{1} << a.shift;
  sort_windows(keys + r * a.kstride, a.kstride, static_cast<int>(S), 0, start + r * (S + 1), perm + r * a.W, cnt);
}

template <typename TM, int V>
__device__ __forceinline__ void tg_load(const TM* p, float (&v)[V]) {
  if constexpr (sizeof(TM) * V >= 16) {  // whole 16-byte pieces (the host checks base and stride)
    constexpr int E = 16 / sizeof(TM);
#pragma unroll
    for (int c = 0; c < V / E; ++c) {
      const u32x4 w = reinterpret_cast<const u32x4*>(p)[c];
      const TM* e = reinterpret_cast<const TM*>(&w);
#pragma unroll
      for (int j = 0; j < E; ++j) v[c * E + j] = to_f32(e[j]);
    }
  } else {
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = to_f32(p[j]);
  }
}

// Eight gradient rows of a group are in flight at once: order 3 has 4 windows a row and order 2 has
// 64 at 16384 positions, and a group's next request does not wait for its last sum.
template <typename TM, typename TO, int V>
__global__ __launch_bounds__(256) void k_tg_sum(TgArgs a, const uint32_t* __restrict__ start,
                                                const uint32_t* __restrict__ perm, TO* __restrict__ out) {
  constexpr int D = 16 * V, U = V >= 16 ? 4 : 8;
  __shared__ float red[16][D];
  __shared__ uint32_t lng_lo[16], lng_hi[16];
  __shared__ int any_long;
  const int tid = threadIdx.x, grp = tid >> 4, l = tid & 15;
  const int64_t S = int64_t{1} << a.shift;
  const int64_t rows = S * a.R;
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * 16, row = row0 + grp;
  if (tid == 0) any_long = 0;
  __syncthreads();
  const TM* grad = static_cast<const TM*>(a.grad);
  // the sum over perm entries lo, lo + step .. of route r (step 1, or the 16 groups' share of a long row)
  auto sum = [&](int64_t r, uint32_t lo, uint32_t hi, float (&acc)[V]) {
    const uint32_t* pm = perm + r * a.W;
    for (uint32_t j = lo; j < hi; j += 16) {
      const uint32_t mine = j + l < hi ? pm[j + l] : 0;
      const int m = static_cast<int>(hi - j < 16 ? hi - j : 16);
      for (int k = 0; k < m; k += U) {
        float g[U][V];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t w = static_cast<uint32_t>(__shfl(static_cast<int>(mine), k + u, 16));
          if (k + u < m) {
            tg_load<TM, V>(grad + (w * a.R + r) * a.grad_stride + l * V, g[u]);
          } else {
#pragma unroll
            for (int v = 0; v < V; ++v) g[u][v] = 0.f;
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int v = 0; v < V; ++v) acc[v] += g[u][v];
      }
    }
  };
  auto store = [&](int64_t rw, const float (&acc)[V]) {
    TO* o = out + rw * D + l * V;
    TO t[V];
#pragma unroll
    for (int v = 0; v < V; ++v) t[v] = from_f32<TO>(acc[v]);
#pragma unroll
    for (int v = 0; v < V; ++v) o[v] = t[v];
  };
  if (row < rows) {
    const int64_t r = row >> a.shift;
    const uint32_t* st = start + r * (S + 1) + (row & (S - 1));
    const uint32_t lo = st[0], hi = st[1];
    if (hi - lo <= TG_LONG) {
      float acc[V];
#pragma unroll
      for (int v = 0; v < V; ++v) acc[v] = 0.f;
      sum(r, lo, hi, acc);
      store(row, acc);
    } else if (l == 0) {
      any_long = 1;
    }
    if (l == 0) {
      lng_lo[grp] = lo;
      lng_hi[grp] = hi;
    }
  } else if (l == 0) {
    lng_lo[grp] = lng_hi[grp] = 0;
  }
  __syncthreads();
  if (!any_long) return;  // the whole block
  for (int g = 0; g < 16; ++g) {
    const uint32_t lo = lng_lo[g], hi = lng_hi[g];
    if (hi - lo <= TG_LONG) continue;  // the whole block
    const uint32_t share = (hi - lo + 15) / 16;
    const uint32_t b = lo + grp * share;
    float acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = 0.f;
    if (b < hi) sum((row0 + g) >> a.shift, b, b + share < hi ? b + share : hi, acc);
#pragma unroll
    for (int v = 0; v < V; ++v) red[grp][l * V + v] = acc[v];
    __syncthreads();
    if (tid < D) {
      float s = 0.f;
      for (int k = 0; k < 16; ++k) s += red[k][tid];
      out[(row0 + g) * D + tid] = from_f32<TO>(s);
    }
    __syncthreads();
  }
}

template <typename TM, typename TO>
static int tg_sum_launch(const TgArgs& a, int32_t D, const uint32_t* start, const uint32_t* perm, void* out,
                         hipStream_t s) {
  const unsigned blocks = static_cast<unsigned>(cdiv(static_cast<int64_t>(a.R) << a.shift, 16));
  TO* o = static_cast<TO*>(out);
  switch (D) {
    case 32: k_tg_sum<TM, TO, 2><<<blocks, 256, 0, s>>>(a, start, perm, o); break;
    case 64: k_tg_sum<TM, TO, 4><<<blocks, 256, 0, s>>>(a, start, perm, o); break;
    case 128: k_tg_sum<TM, TO, 8><<<blocks, 256, 0, s>>>(a, start, perm, o); break;
    default: k_tg_sum<TM, TO, 16><<<blocks, 256, 0, s>>>(a, start, perm, o); break;
  }
  return check_launch("k_tg_sum");
}

}  // namespace lng

using namespace lng;

// Shapes the listed form serves: the route's counters in LDS, positions and rows in 32 bits.
static bool tg_ok(int64_t B, int64_t T, int32_t R, int32_t order, int32_t bits) {
  if (B < 0 || T < 0 || R <= 0 || order < 1 || bits < 1 || bits > 8 || bits * order > 13) return false;
  return B * T < (int64_t{1} << 31) - 64 && (static_cast<int64_t>(R) << (bits * order)) < (int64_t{1} << 31);
}

extern "C" size_t lng_table_grad_workspace_bytes(int64_t B, int64_t T, int32_t R, int32_t order, int32_t bits) {
  if (!tg_ok(B, T, R, order, bits)) return 0;
  return tg_layout(B * T, R, int64_t{1} << (bits * order)).total;
}

extern "C" int lng_table_grad_rows(const void* grad_memory, int mem_dtype, int64_t grad_stride, const void* codes,
                                   int codes_dtype, const uint8_t* valid_mask, int64_t B, int64_t T, int32_t R,
                                   int32_t route_start, int32_t mem_dim, int32_t order, int32_t bits,
                                   int64_t table_rows, void* workspace, size_t workspace_bytes, void* table_grad,
                                   int out_dtype, void* stream) {
  if (!tg_ok(B, T, R, order, bits) || route_start < 0)
    return fail(LNG_E_ARG, "table_grad_rows: shape outside lng_table_grad_workspace_bytes' range");
  if (mem_dtype != LNG_F32 && mem_dtype != LNG_BF16) return fail(LNG_E_DTYPE, "table_grad_rows: memory f32 or bf16");
  if (out_dtype != LNG_F32 && out_dtype != LNG_BF16) return fail(LNG_E_DTYPE, "table_grad_rows: gradient f32 or bf16");
  if (codes_dtype != LNG_U8 && codes_dtype != LNG_I32 && codes_dtype != LNG_I64)
    return fail(LNG_E_DTYPE, "table_grad_rows: codes u8, i32 or i64");
  if (mem_dim != 32 && mem_dim != 64 && mem_dim != 128 && mem_dim != 256)
    return fail(LNG_E_ARG, "table_grad_rows: mem_dim must be 32, 64, 128 or 256");
  const int shift = bits * order;
  if (table_rows < ((static_cast<int64_t>(route_start) + R) << shift))
    return fail(LNG_E_ARG, "table_grad_rows: table has fewer rows than (route_start + R) * 2^(bits*order)");
  const int64_t W = B * T;
  if (!table_grad || !workspace || (W > 0 && (!grad_memory || !codes)))
    return fail(LNG_E_ARG, "table_grad_rows: null buffer");
  const int es = dtype_size(mem_dtype);
  if (grad_stride < mem_dim || (grad_stride * es) % 16 || (reinterpret_cast<uintptr_t>(grad_memory) & 15) ||
      (reinterpret_cast<uintptr_t>(table_grad) & 15) || (reinterpret_cast<uintptr_t>(workspace) & 15))
    return fail(LNG_E_ARG, "table_grad_rows: gradient rows, table and workspace must be 16-byte aligned");
  const int64_t S = int64_t{1} << shift;
  const TgWs w = tg_layout(W, R, S);
  if (workspace_bytes < w.total)
    return fail(LNG_E_ARG, "table_grad_rows: workspace smaller than lng_table_grad_workspace_bytes");
  hipStream_t s = as_stream(stream);
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  uint16_t* keys = reinterpret_cast<uint16_t*>(ws + w.keys);
  uint32_t* start = reinterpret_cast<uint32_t*>(ws + w.start);
  uint32_t* perm = reinterpret_cast<uint32_t*>(ws + w.perm);
  const TgArgs a{grad_memory, grad_stride, codes, codes_dtype, valid_mask, W, T, R, order, bits, shift, w.kstride};
  if (W > 0) k_tg_keys<<<dim3(static_cast<unsigned>(w.kstride / 64), static_cast<unsigned>(cdiv(R, 64))), 256, 0, s>>>(a, keys);
  k_tg_sort<<<static_cast<unsigned>(R), 1024, static_cast<size_t>(S + 16) * 4, s>>>(a, keys, start, perm);
  char* out = static_cast<char*>(table_grad) +
              (static_cast<int64_t>(route_start) << shift) * mem_dim * dtype_size(out_dtype);
  if (mem_dtype == LNG_BF16)
    return out_dtype == LNG_BF16 ? tg_sum_launch<bf16, bf16>(a, mem_dim, start, perm, out, s)
                                 : tg_sum_launch<bf16, float>(a, mem_dim, start, perm, out, s);
  return out_dtype == LNG_BF16 ? tg_sum_launch<float, bf16>(a, mem_dim, start, perm, out, s)
                               : tg_sum_launch<float, float>(a, mem_dim, start, perm, out, s);
}
