// The kernel definitions of the dense W4A8-iu8 GEMMs, as macros over the bodies in iu8_gemm.h and
// iu8_pf32.h: one place for the argument lists (crates/saber-kernels/src/abi.rs:3349-3372) shared by
// the product object `macaq_iu8` and the parity suite's accumulator taps (`iu8_taps`).
#pragma once
#include "iu8_gemm.h"
#include "iu8_pf32.h"
#include "iu8_pf_law.h"
#include "iu8_stream.h"

#define IU8_DEC(name, TM, W8, NT, KW, WPB, D, ALDS, ACC)                                                         \
  extern "C" __global__ __launch_bounds__(WPB * 64) void name(                                                    \
      const unsigned char *__restrict__ a, const unsigned char *__restrict__ w, const float *__restrict__ as,     \
      const float *__restrict__ ws, int *__restrict__ decode_partial, int *__restrict__ decode_counter,           \
      unsigned short *__restrict__ c, int m, int n, int k) {                                                       \
    static_assert(ALDS > 0 ? TM == 1 : WPB == KW, "staged rows are one row tile; a streamed cell's waves its k-waves"); \
    if constexpr (ALDS == 0) {                                                                                      \
      iu8_stream_cells<TM, W8, NT, KW, D, ACC>(a, w, as, ws, decode_partial, decode_counter, c, m, n, k,            \
                                               iu8_blk_of_grid(), (int)gridDim.x);                                  \
    } else {                                                                                                       \
      iu8_dec_body<W8, NT, KW, WPB, D, ALDS, ACC>(a, w, as, ws, decode_partial, decode_counter, c,              \
                                                      iu8_rows{nullptr, 0, m}, n, k);                               \
    }                                                                                                              \
  }

// The workgroup's r-th thin tile (its column block), -1: none. The order of the workgroups is iu8_dense_tile_at's.
static __device__ __forceinline__ int iu8_thin_tile_at(const iu8_pf_plan &p, int r, int gx) {
  const int G = gridDim.x, w = blockIdx.x, at = (G & 7) == 0 ? (w & 7) * (G >> 3) + (w >> 3) : w;
  if (p.own_wgs > 0 && at >= p.rem) {
    const int j = at - p.rem + r * p.own_wgs;
    if (r < p.own) return j < gx ? j : -1;
    r -= p.own;
  }
  // the rest by all, the last workgroups first: the first ones have a quarter tile more
  const int j = p.own * p.own_wgs + (G - 1 - at) + r * G;
  return j < gx ? j : -1;
}

// Persistent launch: gridDim.x workgroups (one or OCC a CU) walk the tiles of the m x n output.
//
// The 256 x 256 cell's last round and its ragged rows (iu8_pf_law.h): a thin last round is cut into quarter tiles on the
// 128 x 128 cell, which take 0.42 (one round) or 0.84 (two) of a big tile's time, and a few rows past the last whole 256 run as
// thin tiles on a 128 x 256 cell whose waves skip row blocks without a row. Same bytes: every output element is one exact
// integer sum and one epilogue, whichever cell computes it.
#define IU8_PF32(name, W8, WMW, WNW, TM, TN, ACC, ST, OCC, DEEP, KW)                                                    \
  extern "C" __global__ __launch_bounds__(WMW * WNW * KW * 64)                                                    \
      __attribute__((amdgpu_waves_per_eu(WMW * WNW * KW * OCC / 4, WMW * WNW * KW * OCC / 4))) void name(          \
      const unsigned char *__restrict__ a, const unsigned char *__restrict__ w, const float *__restrict__ as,     \
      const float *__restrict__ ws, unsigned short *__restrict__ c, int m, int n, int k) {                         \
    constexpr int BM = WMW * TM * 32, BN = WNW * TN * 32;                                                          \
    constexpr bool TAIL = WMW == 2 && WNW == 4 && TM == 4 && TN == 2 && !ACC && !DEEP;                             \
    const int gx = (n + BN - 1) / BN, gy = (m + BM - 1) / BM;                                                      \
    const iu8_rows R{nullptr, 0, m};                                                                               \
    if constexpr (TAIL) {                                                                                          \
      constexpr int LB = iu8_pf32_lds_bytes<W8, WMW, WNW, TM, TN, ST>(), LS = iu8_pf32_lds_bytes<W8, 4, 2, 1, 2, 3>();\
      constexpr int LT = iu8_pf32_lds_bytes<W8, 1, 8, 4, 1, 3, iu8_pf32_stashes<true, 1, 8, 4, 1>()>();            \
      constexpr int LM = LB > LS ? LB : LS;                                                                        \
      __shared__ __attribute__((aligned(1024))) iu8_u8 lds[LM > LT ? LM : LT];                                     \
      const int G = gridDim.x;                                                                                     \
      const iu8_pf_plan plan = G == 256 ? iu8_pf_plan256(m, gx, 256, k, W8) : iu8_pf_plan256(m, gx, G, k, W8);        \
      iu8_pf32_run<W8, WMW, WNW, TM, TN, ACC, ST, DEEP, false, false, true>(                                       \
          a, as, c, n, k,                                                                                          \
          [&](int r, iu8_tile &t) {                                                                                \
            int bx, by;                                                                                            \
            if ((plan.tail && r >= plan.q) || !iu8_dense_tile_at(r, gx, plan.gy, bx, by)) return false;            \
            t = iu8_tile{R, by * BM, bx * (BN / 16), w, ws, by * gx + bx};                                         \
            return true;                                                                                           \
          },                                                                                                       \
          nullptr, nullptr, lds);                                                                                  \
      if (plan.tail) {                                                                                             \
        __syncthreads();                                                                                           \
        iu8_pf32_run<W8, 4, 2, 1, 2, ACC, 3, false, false, false, true>(                                           \
            a, as, c, n, k,                                                                                        \
            [&](int r, iu8_tile &t) {                                                                              \
              const int j = (int)blockIdx.x + r * G;                                                               \
              if (j >= 4 * plan.rem) return false;                                                                 \
              int bx, by;                                                                                          \
              iu8_dense_tile_of(plan.q * G + (j >> 2), gx, plan.gy, bx, by);                                       \
              t = iu8_tile{R, by * BM + ((j >> 1) & 1) * 128, (bx * BN + (j & 1) * 128) / 16, w, ws, 0};           \
              return true;                                                                                         \
            },                                                                                                     \
            nullptr, nullptr, lds);                                                                                \
      }                                                                                                            \
      if (plan.thin) {                                                                                             \
        __syncthreads();                                                                                           \
        iu8_pf32_run<W8, 1, 8, 4, 1, ACC, 3, false, true, false, true>(                                            \
            a, as, c, n, k,                                                                                        \
            [&](int r, iu8_tile &t) {                                                                              \
              const int j = iu8_thin_tile_at(plan, r, gx);                                                         \
              if (j < 0) return false;                                                                             \
              t = iu8_tile{R, plan.gy * BM, j * (BN / 16), w, ws, 0};                                              \
              return true;                                                                                         \
            },                                                                                                     \
            nullptr, nullptr, lds);                                                                                \
      }                                                                                                            \
    } else {                                                                                                       \
      iu8_pf32_run<W8, WMW, WNW, TM, TN, ACC, ST, DEEP, false, false, false, false, false, KW>(a, as, c, n, k, [&](int r, iu8_tile &t) { \
        int bx, by;                                                                                                \
        if (!iu8_dense_tile_at(r, gx, gy, bx, by)) return false;                                                   \
        t = iu8_tile{R, by * BM, bx * (BN / 16), w, ws, by * gx + bx};                                             \
        return true;                                                                                               \
      });                                                                                                          \
    }                                                                                                              \
  }
