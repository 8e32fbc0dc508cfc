// Backward of the training lookup at the SB shape (bf16 tables of orders 2 and 3 with rows of 128,
// 4-bit codes, approximate surrogate): both orders' route-logit gradients and table gradients from one
// reading of the memory gradient (_LngramSurrogate, ffnmem/memory/lngram_v2.py:430-447, and the
// embedding backward of its lookup, :1084-1092).
//
// A position's windows are named by the position that ends them.  For each order, a route's windows
// are sorted by the table row they read (window_sort.h); a wave takes 64 consecutive windows of a
// route's list, 16 at a time, and all the windows of one row at once:
//   scores   C[m][n] = T_m . g_n, a 16x16x128 bf16 matrix product as four of 32 features added
//            pairwise (relative error of the gradient against fp64 8.85e-8; as one chain 9.55e-8,
//            order by order 9.07e-8): T_m the row with address bit m flipped (m < 4 order) and T_12 the
//            row itself, g_n the windows' gradient rows.  The result holds a window's four flips of digit e in one lane, which subtracts the looked-up
//            row's product and stores them to plane e of the workspace;
//   row sum  the gradient rows, staged in LDS, are also summed in fp32 with two features a lane; a
//            complete row is stored once, rounded once; a row cut by the wave's ends leaves fp32
//            partial sums in the workspace, which k_lg_merge adds up (and clears the rows that no
//            window names).
// k_lg_out sums each output's windows in the reference's order (digit ascending) and applies the
// slope.  A route's blocks run on one XCD, whose L2 holds the route's table rows.
// Least traffic: the gradient read once (1.54 GB at 8 x 2048 positions, 184 routes) and the scores
// written and read once (482 MB).  Measured there: k_lg_main 545 us for order 3 and 224 us for order 2,
// k_lg_out 85, the lists 56, k_lg_merge 50; the order-by-order kernels took 1.9 ms (two copies of the
// gradient's halves, surrogate 498 + 60 and 316, table gradients 600).  k_lg_main<3> waits on its table
// rows: an XCD's 512 waves work on as many routes at once as it takes to fill them, 1 MB of rows each,
// beside the gradient's and the scores' streams in its 4 MB L2.  Chunks of 128 windows keep four routes
// in flight (574 and 240 us, 59 % of L2 requests miss), of 64 two; with 48 and 32 the rows cut by chunk
// ends cost more than that gives (+12 and +24 us over all).  Rows requested two runs ahead gave nothing
// (578).  Operands loaded straight into their lanes, 64 bytes of 16 rows an instruction, took 659 and
// 278 us: a row is loaded by 16 lanes and staged.
#include "window_sort.h"

namespace lng {

constexpr int LG_CHUNK = 64;  // windows of a wave, an entry a lane

// A staged tile: 16 rows of 16 16-byte pieces, piece p of row n in slot p ^ lg_swz(n).  Rows are loaded
// and stored by 16 lanes each (whole lines) and read as matrix operands by lane (n, kg) in pieces
// lg_piece(kg, s): either way the 16 lanes that one LDS pass serves (0-7 with 16-23, ..) hit 16 slots.
__device__ __forceinline__ int lg_swz(int n) { return ((n & 1) << 3) | (n >> 1); }
__device__ __forceinline__ int lg_piece(int kg, int s) { return ((kg & 1) << 2) | ((kg >> 1) << 3) | s; }

struct LgOrder {  // one order's buffers
  const bf16* table;       // the first route's first row
  const uint8_t* valid;    // [W] or null
  const uint32_t* start;   // [R][S + 1]
  const uint32_t* perm;    // [R][W]: position << shift | address
  float* scores;           // [order][R][W][4], or null: no route-logit gradient wanted
  float* part;             // [R][chunks][2][128] fp32: sums of the chunk's first and last row where cut
  bf16* out;               // [R << shift][128], or null: no table gradient wanted
};
struct LgArgs {
  const bf16* grad;        // rows of 2 x 128, gstride elements apart
  int64_t gstride;
  LgOrder o[2];            // orders 2 and 3
  int32_t W, T, R, chunks;
};

struct LgWs {
  size_t keys[2], start[2], perm[2], scores[2], part[2], total;
  int64_t kstride;
};
static size_t lg_al(size_t x) { return (x + 255) & ~size_t{255}; }
static LgWs lg_layout(int64_t W, int64_t R) {
  LgWs w{};
  size_t at = 0;
  auto take = [&](size_t n) {
    const size_t p = at;
    at += lg_al(n);
    return p;
  };
  w.kstride = (W + 63) / 64 * 64;
  const size_t chunks = static_cast<size_t>((W + LG_CHUNK - 1) / LG_CHUNK);
  for (int i = 0; i < 2; ++i) {
    const size_t S = size_t{1} << (4 * (i + 2));
    w.keys[i] = take(static_cast<size_t>(R) * w.kstride * 2);
    w.start[i] = take(static_cast<size_t>(R) * (S + 1) * 4);
    w.perm[i] = take(static_cast<size_t>(R) * W * 4);
    w.scores[i] = take(static_cast<size_t>(i + 2) * R * W * 16);
    w.part[i] = take(static_cast<size_t>(R) * chunks * 2 * 128 * 4);
  }
  w.total = at;
  return w;
}

__device__ __forceinline__ uint32_t lg_code(const void* p, int dt, int64_t i) {
  if (dt == LNG_U8) return static_cast<const uint8_t*>(p)[i] & 15;
  if (dt == LNG_I32) return static_cast<uint32_t>(static_cast<const int32_t*>(p)[i]) & 15;
  return static_cast<uint32_t>(static_cast<const int64_t*>(p)[i]) & 15;
}

// Route-major keys of both orders from one reading of the codes, through 64 x 64 LDS tiles.
__global__ __launch_bounds__(256) void k_lg_keys(LgArgs a, const void* __restrict__ codes, int codes_dt, int64_t kstride,
                                                 uint16_t* __restrict__ keys2, uint16_t* __restrict__ keys3) {
  __shared__ uint16_t tile[2][64][66];
  const int w0 = blockIdx.x * 64, r0 = blockIdx.y * 64;
  const int rl = threadIdx.x & 63, r = r0 + rl;
#pragma unroll 4
  for (int k = 0; k < 16; ++k) {
    const int wl = __builtin_amdgcn_readfirstlane(4 * k + (static_cast<int>(threadIdx.x) >> 6)), w = w0 + wl;
    uint32_t k2 = WIN_DEAD, k3 = WIN_DEAD;
    if (w < a.W && r < a.R) {
      const int t = w % a.T;
      const int64_t i = static_cast<int64_t>(w) * a.R + r;
      const uint32_t c0 = lg_code(codes, codes_dt, i);
      const uint32_t c1 = t >= 1 ? lg_code(codes, codes_dt, i - a.R) : 0;
      const uint32_t c2 = t >= 2 ? lg_code(codes, codes_dt, i - 2 * static_cast<int64_t>(a.R)) : 0;
      if (t >= 1 && (a.o[0].valid == nullptr || a.o[0].valid[w])) k2 = c1 | (c0 << 4);
      if (t >= 2 && (a.o[1].valid == nullptr || a.o[1].valid[w])) k3 = c2 | (c1 << 4) | (c0 << 8);
    }
    tile[0][wl][rl] = static_cast<uint16_t>(k2);
    tile[1][wl][rl] = static_cast<uint16_t>(k3);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 64 * 64; i += 256) {
    const int rr = i >> 6, wl = i & 63;
    if (r0 + rr >= a.R) continue;
    const int64_t at = (r0 + rr) * kstride + w0 + wl;
    keys2[at] = tile[0][wl][rr];
    keys3[at] = tile[1][wl][rr];
  }
}

__global__ __launch_bounds__(1024) void k_lg_sort(const uint16_t* __restrict__ keys2, const uint16_t* __restrict__ keys3,
                                                  int64_t kstride, int64_t W, uint32_t* __restrict__ start2,
                                                  uint32_t* __restrict__ start3, uint32_t* __restrict__ perm2,
                                                  uint32_t* __restrict__ perm3) {
  __shared__ uint32_t cnt[4096 + 16];
  const int64_t r = blockIdx.x;
  const bool three = blockIdx.y != 0;
  const int shift = three ? 12 : 8;
  const int64_t S = int64_t{1} << shift;
  sort_windows((three ? keys3 : keys2) + r * kstride, kstride, static_cast<int>(S), shift,
               (three ? start3 : start2) + r * (S + 1), (three ? perm3 : perm2) + r * W, cnt);
}

template <int ORDER>
__global__ __launch_bounds__(256) void k_lg_main(LgArgs a) {
  constexpr int SH = 4 * ORDER;
  constexpr uint32_t AM = (1u << SH) - 1;
  __shared__ __attribute__((aligned(16))) char stage[4][2][4096];
  const LgOrder& o = a.o[ORDER - 2];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int col = lane & 15, kg = lane >> 4;
  const int xcd = blockIdx.x & 7, k8 = blockIdx.x >> 3;
  const int bpr = (a.chunks + 3) / 4;  // blocks of a route
  const int r = (k8 / bpr) * 8 + xcd;
  const int c = (k8 % bpr) * 4 + wave;
  if (r >= a.R || c >= a.chunks) return;  // the whole wave; the block has no barrier
  const uint32_t* st = o.start + static_cast<int64_t>(r) * ((1 << SH) + 1);
  const int total = static_cast<int>(st[1 << SH]);
  const int lo = c * LG_CHUNK, nw = min(LG_CHUNK, total - lo);
  if (nw <= 0) return;
  const uint32_t* pm = o.perm + static_cast<int64_t>(r) * a.W;
  const uint32_t ent = pm[lo + min(lane, nw - 1)];  // the chunk's entries
  const bf16* grad = a.grad + (ORDER - 2) * 128 + static_cast<int64_t>(r) * a.gstride + col * 8;
  const int64_t wstride = static_cast<int64_t>(a.R) * a.gstride;
  const bf16* table = o.table + (static_cast<int64_t>(r) << SH) * 128 + col * 8;
  float* part = o.part + (static_cast<int64_t>(r) * a.chunks + c) * 256;
  bf16* out = o.out == nullptr ? nullptr : o.out + (static_cast<int64_t>(r) << SH) * 128;
  float* scores = o.scores == nullptr
                      ? nullptr
                      : o.scores + (static_cast<int64_t>(kg < ORDER ? kg : 0) * a.R + r) * a.W * int64_t{4};
  char* gst = stage[wave][0];
  char* tst = stage[wave][1];
  auto at = [&](int q) {  // entry q of the chunk (q may differ between lanes)
    return static_cast<uint32_t>(__shfl(static_cast<int>(ent), q));
  };
  // 16 rows into registers, 4 a load and 16 lanes a row: the gradients of windows 16 b ..; the table rows
  // of one address (row m has address bit m flipped, rows 4 ORDER .. 15 are the row itself)
  auto load_grad = [&](int b, u32x4 (&g)[4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      g[k] = *reinterpret_cast<const u32x4*>(grad + static_cast<int64_t>(at(16 * b + 4 * k + kg) >> SH) * wstride);
  };
  auto load_rows = [&](uint32_t row, u32x4 (&t)[4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int m = 4 * k + kg;
      t[k] = *reinterpret_cast<const u32x4*>(table + static_cast<int64_t>(row ^ (m < SH ? 1u << m : 0u)) * 128);
    }
  };
  auto put = [&](char* buf, const u32x4 (&x)[4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int n = 4 * k + kg;
      *reinterpret_cast<u32x4*>(buf + n * 256 + ((col ^ lg_swz(n)) << 4)) = x[k];
    }
  };
  auto frag = [&](const char* buf, int s) {
    return *reinterpret_cast<const bf16x8*>(buf + col * 256 + ((lg_piece(kg, s) ^ lg_swz(col)) << 4));
  };
  // the open row and its sum over this chunk (features 2 lane, 2 lane + 1)
  uint32_t cur = 0xFFFFFFFF;
  float s0 = 0.f, s1 = 0.f;
  auto flush = [&]() {
    if (out == nullptr || cur == 0xFFFFFFFF) return;
    const int b = static_cast<int>(st[cur]), e = static_cast<int>(st[cur + 1]);
    if (b < lo || e > lo + nw) {  // cut: the first slot when an earlier chunk began the row
      reinterpret_cast<float2*>(part + (b < lo ? 0 : 128))[lane] = float2{s0, s1};
    } else {
      reinterpret_cast<bf16x2*>(out + static_cast<int64_t>(cur) * 128)[lane] =
          bf16x2{static_cast<bf16>(s0), static_cast<bf16>(s1)};
    }
  };
  const int nb = (nw + 15) / 16;
  u32x4 g[4], t[4];
  uint32_t trow = __builtin_amdgcn_readfirstlane(ent) & AM;  // the row that t holds
  bool fresh = true;                                            // t is not staged yet
  load_grad(0, g);
  if (scores != nullptr) load_rows(trow, t);
  for (int b = 0; b < nb; ++b) {
    const uint32_t e = at(16 * b + col), addr = e & AM;  // this lane's column
    const int n = min(16, nw - 16 * b);                  // columns of this batch
    __builtin_amdgcn_wave_barrier();
    put(gst, g);
    __builtin_amdgcn_wave_barrier();
    if (b + 1 < nb) load_grad(b + 1, g);
    bf16x8 gf[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) gf[s] = frag(gst, s);
    for (int i = 0; i < n;) {
      const uint32_t row = __builtin_amdgcn_readlane(addr, i);
      const int j = i + __builtin_popcountll(__ballot(addr == row && col >= i && col < n) & 0xFFFF);
      if (scores != nullptr) {
        if (fresh) {
          __builtin_amdgcn_wave_barrier();
          put(tst, t);
          __builtin_amdgcn_wave_barrier();
          fresh = false;
        }
        // the next row's table rows are requested under this one's products
        const int q = 16 * b + j;
        if (q < nw) {
          const uint32_t nxt = __builtin_amdgcn_readlane(ent, q) & AM;
          if (nxt != trow) {
            load_rows(nxt, t);
            trow = nxt;
            fresh = true;
          }
        }
        f32x4 c4[4];
#pragma unroll
        for (int s = 0; s < 4; ++s)
          c4[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(tst, s), gf[s], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        const f32x4 cc = (c4[0] + c4[1]) + (c4[2] + c4[3]);
        const float here = __shfl(cc[0], 48 + col);
        f32x4 sc;
#pragma unroll
        for (int k = 0; k < 4; ++k) sc[k] = (cc[k] - here) * (((row >> (4 * kg + k)) & 1) ? -1.f : 1.f);
        if (kg < ORDER && col >= i && col < j) reinterpret_cast<f32x4*>(scores)[e >> SH] = sc;
      }
      if (out != nullptr) {
        if (row != cur) {
          flush();
          cur = row;
          s0 = s1 = 0.f;
        }
        for (int k = i; k < j; ++k) {
          const uint32_t v =
              *reinterpret_cast<const uint32_t*>(gst + k * 256 + (((lane >> 2) ^ lg_swz(k)) << 4) + (lane & 3) * 4);
          s0 += __builtin_bit_cast(float, v << 16);
          s1 += __builtin_bit_cast(float, v & 0xFFFF0000u);
        }
      }
      i = j;
    }
  }
  flush();
}

// Rows cut by chunks: the chunk that a cut row begins in adds its part and the following chunks' in
// order.  Rows that no window names are cleared.  A block takes 256 rows and a share of the chunks; both
// orders in one launch (50 us at 8 x 2048; one after the other 62, each waiting on dependent loads).
template <int ORDER>
__device__ __forceinline__ void lg_merge(const LgArgs& a) {
  constexpr int SH = 4 * ORDER;
  const LgOrder& o = a.o[ORDER - 2];
  if (o.out == nullptr) return;
  const int r = blockIdx.y;
  const uint32_t* st = o.start + static_cast<int64_t>(r) * ((1 << SH) + 1);
  bf16* out = o.out + (static_cast<int64_t>(r) << SH) * 128;
  const int grp = threadIdx.x >> 4, l = threadIdx.x & 15;
  for (int i = grp; i < 256 && blockIdx.x < (1 << SH) / 256; i += 16) {
    const int row = blockIdx.x * 256 + i;
    if (st[row] == st[row + 1]) reinterpret_cast<u32x4*>(out + static_cast<int64_t>(row) * 128)[l] = u32x4{0u, 0u, 0u, 0u};
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int total = static_cast<int>(st[1 << SH]);
  const uint32_t* pm = o.perm + static_cast<int64_t>(r) * a.W;
  for (int c = blockIdx.x * 4 + wave; c < a.chunks; c += gridDim.x * 4) {
    const int lo = c * LG_CHUNK, hi = lo + LG_CHUNK;
    if (hi >= total) break;  // the last chunk cuts no row
    const int row = static_cast<int>(pm[hi - 1] & ((1u << SH) - 1));
    const int b = static_cast<int>(st[row]), e = static_cast<int>(st[row + 1]);
    if (b < lo || e <= hi) continue;  // began in an earlier chunk, or ends here
    const float2* p = reinterpret_cast<const float2*>(o.part + (static_cast<int64_t>(r) * a.chunks + c) * 256);
    float2 s = p[64 + lane];
    for (int k = c + 1; k * LG_CHUNK < e; ++k) {
      const float2 q = p[static_cast<int64_t>(k - c) * 128 + lane];
      s.x += q.x;
      s.y += q.y;
    }
    const bf16x2 v{static_cast<bf16>(s.x), static_cast<bf16>(s.y)};
    reinterpret_cast<bf16x2*>(out + static_cast<int64_t>(row) * 128)[lane] = v;
  }
}
__global__ __launch_bounds__(256) void k_lg_merge(LgArgs a) {
  if (blockIdx.z != 0)
    lg_merge<3>(a);
  else
    lg_merge<2>(a);
}

// grad_q[b, t, r, k] = the orders' sums, each slope * (((0 + S0(t)[k]) + S1(t)[k]) + ..) in the output's
// type, Se(t) the digit-e scores of the window whose digit e is position t (it ends at t + order - 1 -
// e); 0 for a window without a gradient.  64 positions x 16 routes a block: scores read along
// positions, outputs written along routes through LDS.
template <typename TO>
__global__ __launch_bounds__(256) void k_lg_out(LgArgs a, const void* __restrict__ q, int q_dt, float temperature,
                                                float alpha, TO* __restrict__ out) {
  __shared__ f32x4 tile[2][64][17];
  const int bt0 = blockIdx.x * 64, r0 = blockIdx.y * 16, tid = threadIdx.x;
  const bool active = alpha != 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int p = k * 256 + tid, rl = p >> 6, bl = p & 63;
    const int r = r0 + rl, bt = bt0 + bl;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int order = i + 2;
      f32x4 acc{0.f, 0.f, 0.f, 0.f};
      if (active && r < a.R && bt < a.W) {
        const int t = bt % a.T;
        const f32x4* sp = reinterpret_cast<const f32x4*>(a.o[i].scores);
#pragma unroll
        for (int e = 0; e < 3; ++e) {
          if (e >= order) break;
          const int d = order - 1 - e;  // the window ends d positions on
          const bool live = t + d < a.T && t >= e && (a.o[i].valid == nullptr || a.o[i].valid[bt + d]);
          const f32x4 v = live ? sp[(static_cast<int64_t>(e) * a.R + r) * a.W + bt + d] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[j] += v[j];
        }
      }
      tile[i][bl][rl] = acc;
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int p = k * 256 + tid, bl = p >> 4, rl = p & 15;
    const int r = r0 + rl, bt = bt0 + bl;
    if (r >= a.R || bt >= a.W) continue;
    const f32x4 a2 = tile[0][bl][rl], a3 = tile[1][bl][rl];
    const int64_t i = static_cast<int64_t>(bt) * a.R + r;
    f32x4 res{0.f, 0.f, 0.f, 0.f};
    if (active) {
      f32x4 qv;
      if (q_dt == LNG_BF16) {
        const bf16x4 qh = reinterpret_cast<const bf16x4*>(q)[i];
#pragma unroll
        for (int j = 0; j < 4; ++j) qv[j] = static_cast<float>(qh[j]);
      } else {
        qv = reinterpret_cast<const f32x4*>(q)[i];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float pr = 1.f / (1.f + expf(-(temperature * qv[j])));
        const float slope = alpha * pr * (1.f - pr);
        res[j] = round_to<TO>(a2[j] * slope) + round_to<TO>(a3[j] * slope);
      }
    }
    if constexpr (sizeof(TO) == 2) {
      bf16x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = static_cast<bf16>(res[j]);
      reinterpret_cast<bf16x4*>(out)[i] = v;
    } else {
      reinterpret_cast<f32x4*>(out)[i] = res;
    }
  }
}

}  // namespace lng

using namespace lng;

// positions in 20 bits beside a 12-bit address, scores in 31-bit row indices
static bool lg_ok(int64_t B, int64_t T, int32_t R, int32_t mem_dim, int32_t bits, int mem_dtype, int exact) {
  return mem_dtype == LNG_BF16 && !exact && mem_dim == 128 && bits == 4 && R > 0 && R <= 256 && B > 0 && T > 0 &&
         B * T < (int64_t{1} << 20);
}

extern "C" size_t lng_lookup_grad_workspace_bytes(int64_t B, int64_t T, int32_t R, int32_t mem_dim, int32_t bits,
                                                  int mem_dtype, int exact) {
  return lg_ok(B, T, R, mem_dim, bits, mem_dtype, exact) ? lg_layout(B * T, R).total : 0;
}

extern "C" int lng_lookup_grad(const void* grad_memory, int mem_dtype, int64_t grad_stride, const void* q_logits,
                               int q_dtype, const void* codes, int codes_dtype, const void* table2,
                               const void* table3, int64_t table2_rows, int64_t table3_rows, const uint8_t* valid2,
                               const uint8_t* valid3, int64_t B, int64_t T, int32_t R, int32_t route_start,
                               int32_t mem_dim, int32_t bits, float temperature, float scale, void* workspace,
                               size_t workspace_bytes, void* grad_q, int out_dtype, void* grad_table2,
                               void* grad_table3, void* stream) {
  if (!lg_ok(B, T, R, mem_dim, bits, mem_dtype, 0) || route_start < 0)
    return fail(LNG_E_ARG, "lookup_grad: shape outside lng_lookup_grad_workspace_bytes' range");
  if ((q_dtype != LNG_F32 && q_dtype != LNG_BF16) || (out_dtype != LNG_F32 && out_dtype != LNG_BF16))
    return fail(LNG_E_DTYPE, "lookup_grad: logits and gradient f32 or bf16");
  if (codes_dtype != LNG_U8 && codes_dtype != LNG_I32 && codes_dtype != LNG_I64)
    return fail(LNG_E_DTYPE, "lookup_grad: codes u8, i32 or i64");
  if (!grad_memory || !q_logits || !codes || !table2 || !table3 || !workspace)
    return fail(LNG_E_ARG, "lookup_grad: null buffer");
  const int64_t top = static_cast<int64_t>(route_start) + R;
  if (table2_rows < (top << 8) || table3_rows < (top << 12))
    return fail(LNG_E_ARG, "lookup_grad: a table has fewer rows than (route_start + R) * 2^(bits*order)");
  auto al = [](const void* p, uintptr_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; };
  if (grad_stride < 2 * mem_dim || grad_stride % 8 || !al(grad_memory, 16) || !al(table2, 16) || !al(table3, 16) ||
      !al(workspace, 256) || !al(q_logits, q_dtype == LNG_BF16 ? 8 : 16) || !al(grad_q, out_dtype == LNG_BF16 ? 8 : 16) ||
      !al(grad_table2, 16) || !al(grad_table3, 16))
    return fail(LNG_E_ARG, "lookup_grad: rows, tables, logits and gradients must be 16-byte aligned (bf16 logits and "
                           "their gradient 8), the workspace 256-byte");
  const LgWs w = lg_layout(B * T, R);
  if (workspace_bytes < w.total)
    return fail(LNG_E_ARG, "lookup_grad: workspace smaller than lng_lookup_grad_workspace_bytes");
  hipStream_t s = as_stream(stream);
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  const float alpha = static_cast<float>(static_cast<double>(scale) * temperature);
  const bool want_q = grad_q != nullptr && temperature != 0.f && scale != 0.f;
  LgArgs a{};
  a.grad = static_cast<const bf16*>(grad_memory);
  a.gstride = grad_stride;
  a.W = static_cast<int32_t>(B * T);
  a.T = static_cast<int32_t>(T);
  a.R = R;
  a.chunks = static_cast<int32_t>(cdiv(B * T, LG_CHUNK));
  for (int i = 0; i < 2; ++i) {
    const int64_t first = static_cast<int64_t>(route_start) << (4 * (i + 2));
    void* gt = i ? grad_table3 : grad_table2;
    a.o[i] = LgOrder{static_cast<const bf16*>(i ? table3 : table2) + first * 128, i ? valid3 : valid2,
                     reinterpret_cast<uint32_t*>(ws + w.start[i]), reinterpret_cast<uint32_t*>(ws + w.perm[i]),
                     want_q ? reinterpret_cast<float*>(ws + w.scores[i]) : nullptr,
                     reinterpret_cast<float*>(ws + w.part[i]),
                     gt == nullptr ? nullptr : static_cast<bf16*>(gt) + first * 128};
  }
  uint16_t* k2 = reinterpret_cast<uint16_t*>(ws + w.keys[0]);
  uint16_t* k3 = reinterpret_cast<uint16_t*>(ws + w.keys[1]);
  k_lg_keys<<<dim3(static_cast<unsigned>(w.kstride / 64), static_cast<unsigned>(cdiv(R, 64))), 256, 0, s>>>(
      a, codes, codes_dtype, w.kstride, k2, k3);
  k_lg_sort<<<dim3(static_cast<unsigned>(R), 2), 1024, 0, s>>>(
      k2, k3, w.kstride, B * T, reinterpret_cast<uint32_t*>(ws + w.start[0]), reinterpret_cast<uint32_t*>(ws + w.start[1]),
      reinterpret_cast<uint32_t*>(ws + w.perm[0]), reinterpret_cast<uint32_t*>(ws + w.perm[1]));
  const unsigned blocks = static_cast<unsigned>(8 * cdiv(R, 8) * cdiv(a.chunks, 4));
  if (want_q || grad_table2) k_lg_main<2><<<blocks, 256, 0, s>>>(a);
  if (want_q || grad_table3) k_lg_main<3><<<blocks, 256, 0, s>>>(a);
  if (grad_table2 || grad_table3) k_lg_merge<<<dim3(16, static_cast<unsigned>(R), 2), 256, 0, s>>>(a);
  if (grad_q) {
    const dim3 og(static_cast<unsigned>(cdiv(a.W, 64)), static_cast<unsigned>(cdiv(R, 16)));
    const float al_ = want_q ? alpha : 0.f;
    if (out_dtype == LNG_BF16)
      k_lg_out<bf16><<<og, 256, 0, s>>>(a, q_logits, q_dtype, temperature, al_, static_cast<bf16*>(grad_q));
    else
      k_lg_out<float><<<og, 256, 0, s>>>(a, q_logits, q_dtype, temperature, al_, static_cast<float*>(grad_q));
  }
  return check_launch("lookup_grad");
}
