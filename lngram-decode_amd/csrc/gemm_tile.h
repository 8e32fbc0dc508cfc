// GEMM tiles: bf16 projections between the skinny kernel's rows and the one-tile-per-CU kernels', and fp32.
//
// y[m, n] = sum_k x[m, k] * w[n, k]: a block of WN x WM waves computes BN (w rows) x BM (x rows), wave
// (wn, wm) its BN/WN x BM/WM part in 16x16 fragments, accumulating in K order whatever the tile, so the
// results equal the other kernels' (bf16: 16x16x32 products; fp32: 16x16x4 products, bit for bit four
// fmaf in K order).  K advances 128 bytes a stage through a ring of SLOTS LDS stages filled by buffer
// loads straight into LDS; rows past N or M lie outside the buffers and read as zero.
#pragma once

#include "common.h"

namespace lng {

template <typename T, int BN, int BM, int WN, int WM, int SLOTS>
struct TileGemm {
  static constexpr int NWAVE = WN * WM, NT = 64 * NWAVE;
  static constexpr int K_ST = 128 / sizeof(T);          // k of a stage: 64 bf16 or 32 fp32
  static constexpr int PE = 16 / sizeof(T);             // elements of a piece
  typedef T Frag __attribute__((ext_vector_type(PE)));  // an operand lane's share of 4 pieces' k
  static constexpr int ROWS = BN + BM;                  // LDS rows of a stage, w's first
  static constexpr int FN = BN / WN / 16, FM = BM / WM / 16;
  static constexpr int LOADS = ROWS / 8 / NWAVE;        // 8 rows an instruction
  static constexpr int W_LOADS = BN / 8 / NWAVE;
  static constexpr int LDS_ELEMS = SLOTS * ROWS * K_ST;
  static_assert(ROWS % (8 * NWAVE) == 0 && BN % (8 * NWAVE) == 0 && BN % (16 * WN) == 0 && BM % (16 * WM) == 0, "tile split");
  static_assert((SLOTS - 2) * LOADS <= 60, "vmcnt");

  f32x4 acc[FN][FM];
  float xss[FM];  // XRMS: sum of squares of x row 16 j + (lane & 15)

  // piece p of row r is in slot p ^ swz(r): a pass of 16-byte reads (bf16) or a 4-byte read of 16 rows x 16
  // bytes (fp32) meets each bank once
  __device__ __forceinline__ static int swz(int r) { return (sizeof(T) == 2 ? r : r >> 1) & 7; }
  // a lane's operand of half h of a stage, row r: bf16 piece 4 h + psel; fp32 element psel of each of the
  // pieces 4 h .., so that product e takes k 4 e .. 4 e + 3 of the 16
  __device__ __forceinline__ static Frag operand(const T* st, int r, int h, int psel, int sw) {
    const T* row = st + r * K_ST;
    if constexpr (sizeof(T) == 2) {
      return *reinterpret_cast<const Frag*>(row + PE * ((4 * h + psel) ^ sw));
    } else {
      Frag v;
#pragma unroll
      for (int e = 0; e < PE; ++e) v[e] = row[PE * ((4 * h + e) ^ sw) + psel];
      return v;
    }
  }
  __device__ __forceinline__ static f32x4 mma(Frag a, Frag b, f32x4 c) {
    if constexpr (sizeof(T) == 2) {
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    } else {
#pragma unroll
      for (int e = 0; e < PE; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
      return c;
    }
  }

  // waits until at most `left` later stages of this wave's loads are in flight
  __device__ __forceinline__ static void wait(int left) {
    if (left >= SLOTS - 2)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SLOTS - 2) * LOADS) : "memory");
    else if (SLOTS > 3 && left == 1)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

  template <bool XRMS>
  __device__ __forceinline__ void run(T* ring, const T* W, const T* X, int64_t N, int64_t M, int64_t K, int64_t n0,
                                      int64_t m0) {
    static_assert(SLOTS >= 2 && SLOTS <= 4, "wait()");
    constexpr int ES = sizeof(T);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int wn = wave % WN, wm = wave / WN;
    const int nk = static_cast<int>(K / K_ST);
    auto clip = [](int64_t b) { return static_cast<int>(b < 0x7fffffffll ? b : 0x7fffffffll); };
    const __amdgpu_buffer_rsrc_t wrs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(W + n0 * K), 0, clip((N - n0) * K * ES), BUF_DW3);
    const __amdgpu_buffer_rsrc_t xrs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(X + m0 * K), 0, clip((M - m0) * K * ES), BUF_DW3);
    // load d of this wave covers stage rows (d NWAVE + wave) 8 ..: the first W_LOADS are w's
    uint32_t voff[LOADS];
#pragma unroll
    for (int d = 0; d < LOADS; ++d) {
      const int r = (d * NWAVE + wave) * 8 + (lane >> 3);
      const int64_t rr = r < BN ? r : r - BN;
      voff[d] = static_cast<uint32_t>((rr * K + PE * ((lane & 7) ^ swz(r))) * ES);
    }
    auto issue = [&](int kt, int to_slot) {
      T* dst = ring + to_slot * ROWS * K_ST;
#pragma unroll
      for (int d = 0; d < LOADS; ++d) {
        auto* to = (__attribute__((address_space(3))) void*)(dst + (d * NWAVE + wave) * 8 * K_ST);
        const uint32_t off = voff[d] + static_cast<uint32_t>(kt) * 128;
        if (d < W_LOADS)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, to, 16, off, 0, 0, 0);
        else
          __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, to, 16, off, 0, 0, 0);
      }
    };
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < FM; ++j) xss[j] = 0.f;
    const int rsel = lane & 15, psel = lane >> 4;
    for (int s = 0; s < SLOTS - 1 && s < nk; ++s) issue(s, s);
    auto stage = [&](int kt, int slot) {
      wait(nk - 1 - kt);
      // stage kt has landed for every wave, and every wave has read the slot of stage kt - 1 (no release
      // fence: it would wait for the stages in flight)
      __builtin_amdgcn_s_barrier();
      if (kt + SLOTS - 1 < nk) issue(kt + SLOTS - 1, (slot + SLOTS - 1) % SLOTS);
      const T* st = ring + slot * ROWS * K_ST;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        Frag b[FM];
#pragma unroll
        for (int j = 0; j < FM; ++j)
          b[j] = operand(st, BN + wm * (BM / WM) + j * 16 + rsel, h, psel, swz(rsel));
        Frag a[FN];
#pragma unroll
        for (int i = 0; i < FN; ++i) a[i] = operand(st, wn * (BN / WN) + i * 16 + rsel, h, psel, swz(rsel));
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
          for (int j = 0; j < FM; ++j) acc[i][j] = mma(a[i], b[j], acc[i][j]);
        if constexpr (XRMS) {
          // a row's sum in two chains, its even and its odd pieces in order, as the lanes of
          // k_gemm_proj_bf16's 32x32x16 fragments form it: lane groups 0, 1 and 2, 3 exchange pieces and
          // take one of two row fragments each (of a last single one, the same)
#pragma unroll
          for (int j = 0; j < FM; j += 2) {
            const u32x4 lo = __builtin_bit_cast(u32x4, b[j]), hi = __builtin_bit_cast(u32x4, b[j + 1 < FM ? j + 1 : j]);
            uint32_t pc[2][4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const auto r = __builtin_amdgcn_permlane32_swap(lo[q], hi[q], false, false);
              pc[0][q] = r[0];
              pc[1][q] = r[1];
            }
#pragma unroll
            for (int half = 0; half < 2; ++half)
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                const bf16x2 v = __builtin_bit_cast(bf16x2, pc[half][q]);
                xss[j] = __builtin_amdgcn_fdot2_f32_bf16(v, v, xss[j], false);
              }
          }
        }
      }
    };
    // the slots in turn, so that each is a constant offset of the operands' addresses (fp32, 200 x 256 x
    // 1024: 14.8 -> 9.7 us; bf16, 200 x 1024 x 1024: 5.0 -> 4.0)
    int kt = 0;
    for (; kt + SLOTS <= nk; kt += SLOTS) {
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) stage(kt + s, s);
    }
#pragma unroll
    for (int s = 0; s < SLOTS - 1; ++s)
      if (kt + s < nk) stage(kt + s, s);
    if constexpr (XRMS) {
#pragma unroll
      for (int j = 0; j < FM; j += 2) {
        xss[j] += __shfl_xor(xss[j], 16, 64);  // the row's other pieces
        if (j + 1 < FM) {
          const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, xss[j]),
                                                          __builtin_bit_cast(uint32_t, xss[j]), false, false);
          const uint32_t r0 = r[0], r1 = r[1];  // (a bit cast of the element itself takes element 0)
          xss[j] = __builtin_bit_cast(float, r0);
          xss[j + 1] = __builtin_bit_cast(float, r1);
        }
      }
    }
  }
};

}  // namespace lng
