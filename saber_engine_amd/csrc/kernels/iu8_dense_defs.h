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

// The form a cell of BM x BN rows and columns, OCC workgroups a CU, takes on a short K: wave tiles, stages and k-waves (the launch,
// its threads and its tiles are the cell's own). Most cells have one form: a second one costs 128 x 256 and 128 x 320 (three
// stages for four below K = 3,072) 3-7 % of the time of their long K, and gives them 1-3 % of the short one's.
template <bool W8, int BM, int BN, int OCC>
struct iu8_pf_short {
  static constexpr bool HAS = false;
};
// W4 128 x 128, two k-waves and five stages (iu8_pf32.h): their meeting, some 1 us a tile, and the stages to fill are more than the
// halved reads save on a few K steps. us, cold weights, 4 x 2 wave tiles of one wave and three stages / k-waves: 512 rows of
// 7168 x 1024 8.7 / 9.8, 768 of 5120 x 2048 12.5 / 13.3, 96 of 28672 x 2048 13.5 / 15.0, 430 of 7728 x 384 6.6 / 7.5; over 63 shapes the
// k-waves are 16 % slower below K = 512, 12 % below 1,024, 9 % below 2,048. From K = 2,176 they gain: 71 rows of 18048 x 2432
// 13.6 / 12.7, 700 of 4096 x 4096 19.4 / 17.9; 46 shapes of 4,096-6,143 7 %, 38 from 9,000 14 %.
template <>
struct iu8_pf_short<false, 128, 128, 1> {
  static constexpr bool HAS = true;
  static constexpr int WMW = 4, WNW = 2, TM = 1, TN = 2, ST = 3, KW = 1;
  static constexpr bool DEEP = false;
  static __device__ __forceinline__ bool takes(int k, int) { return k <= 2048; }
};
// Int8 weights 128 x 128, four stages: three up to K = 2,048, and up to 6,143 on a count of tiles that leaves the order by XCD
// (iu8_dense_tile_at), where the fourth makes neighbours' loads miss each other in the L2. us on three / four: 143 rows of 14352 x
// 1664 13.0 / 15.5, of 14208 x 3840 21.9 / 26.0, 584 of 6256 x 1152 12.0 / 13.6, 638 of 5312 x 256 6.2 / 6.5; 415 of 6832 x 2688 16.2 /
// 14.7, 304 of 9872 x 9856 53.4 / 48.0.
template <>
struct iu8_pf_short<true, 128, 128, 1> {
  static constexpr bool HAS = true;
  static constexpr int WMW = 4, WNW = 2, TM = 1, TN = 2, ST = 3, KW = 1;
  static constexpr bool DEEP = false;
  static __device__ __forceinline__ bool takes(int k, int wgs) { return k <= 2048 || (k < 6144 && wgs % 8 != 0); }
};
// W4 64 x 64, two k-waves: the deep form of one wave a wave tile up to K = 512, where the k-waves' meeting and their fuller prologue are what a
// launch is. us, deep / k-waves: 600 rows of 4096 x 128 6.1 / 6.5, 200 of 4096 x 128 3.5 / 3.6; over 140 shapes the k-waves are 3 % slower at K = 128, 2 %
// at 256, level at 384 and 512, 2 % faster at 640, 5 % at 1,536, 9 % at 3,072 and 15 % past 8,192.
template <>
struct iu8_pf_short<false, 64, 64, 2> {
  static constexpr bool HAS = true;
  static constexpr int WMW = 2, WNW = 2, TM = 1, TN = 1, ST = 6, KW = 1;
  static constexpr bool DEEP = true;
  static __device__ __forceinline__ bool takes(int k, int) { return k <= 512; }
};
// Int8 weights 64 x 64, five stages: four below K = 3,072. us on four / five: 511 rows of 2784 x 256 4.6 / 5.0, 675 of 2096 x 1024 8.4 /
// 8.9, 2,025 of 560 x 2304 10.4 / 10.7; 89 of 2112 x 5376 13.7 / 12.5, 142 of 1648 x 8960 20.8 / 17.7. (Between 1,536 and 3,071 the
// two are level on the whole: 160-256 tiles gain up to 6 %, more than 256 lose up to 6 %.)
template <>
struct iu8_pf_short<true, 64, 64, 2> {
  static constexpr bool HAS = true;
  static constexpr int WMW = 2, WNW = 2, TM = 1, TN = 1, ST = 4, KW = 1;
  static constexpr bool DEEP = true;
  static __device__ __forceinline__ bool takes(int k, int) { return k < 3072; }
};

// The tiles of a dense launch on the cell, or on its form for a short K.
template <bool W8, int WMW, int WNW, int TM, int TN, bool ACC, int ST, int OCC, bool DEEP, int KW>
static __device__ __forceinline__ void iu8_pf32_dense(const unsigned char *__restrict__ a, const unsigned char *__restrict__ w,
                                                      const float *__restrict__ as, const float *__restrict__ ws,
                                                      unsigned short *__restrict__ c, int m, int n, int k) {
  constexpr int BM = WMW * TM * 32, BN = WNW * TN * 32;
  const int gx = (n + BN - 1) / BN, gy = (m + BM - 1) / BM;
  const iu8_rows R{nullptr, 0, m};
  auto tile_at = [&](int r, iu8_tile &t) {
    int bx, by;
    if (!iu8_dense_tile_at(r, gx, gy, bx, by)) return false;
    t = iu8_tile{R, by * BM, bx * (BN / 16), w, ws, by * gx + bx};
    return true;
  };
  using S = iu8_pf_short<W8, BM, BN, OCC>;
  if constexpr (S::HAS) {
    static_assert(S::WMW * S::TM * 32 == BM && S::WNW * S::TN * 32 == BN && S::WMW * S::WNW * S::KW == WMW * WNW * KW, "one launch");
    constexpr int L = iu8_pf32_lds_bytes<W8, WMW, WNW, TM, TN, ST>();
    static_assert(iu8_pf32_lds_bytes<W8, S::WMW, S::WNW, S::TM, S::TN, S::ST>() <= L, "the short form runs in the cell's stages");
    __shared__ __attribute__((aligned(1024))) iu8_u8 lds[L];
    if (S::takes(k, (int)gridDim.x))
      iu8_pf32_run<W8, S::WMW, S::WNW, S::TM, S::TN, ACC, S::ST, S::DEEP, false, false, true, false, false, S::KW>(a, as, c, n, k, tile_at, nullptr, nullptr, lds);
    else
      iu8_pf32_run<W8, WMW, WNW, TM, TN, ACC, ST, DEEP, false, false, true, false, false, KW>(a, as, c, n, k, tile_at, nullptr, nullptr, lds);
  } else {
    iu8_pf32_run<W8, WMW, WNW, TM, TN, ACC, ST, DEEP, false, false, false, false, false, KW>(a, as, c, n, k, tile_at);
  }
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
      iu8_pf32_dense<W8, WMW, WNW, TM, TN, ACC, ST, OCC, DEEP, KW>(a, w, as, ws, c, m, n, k);                       \
    }                                                                                                              \
  }
