// The streamed cells (5 to 96 rows): the weights of a block of NT 16-row tiles and, beside them, the rows' codes go
// straight from memory / L2 into registers, K dealt to the KW k-waves of a workgroup in 128-deep steps. Operand orders and
// the contract: iu8_common.h; the staged and the grouped decode cells: iu8_gemm.h.
//
// What bounds it. A CU's vector-memory path hands its waves' loads back in order (measured: waves reading data that lies in
// L2 get 112 bytes a ns alone and 29 beside waves that stream from memory at 27), so the rows' bytes cost a CU as much as
// the weights' own: (rows + columns / 2) x K bytes at some 53 a ns. A wider block divides the rows' share by its columns as
// long as a block a CU is left; more steps in flight than two do not help (a path that is full already).
#pragma once
#include "iu8_gemm.h"
#include "iu8_stream_law.h"

// LDS of a cell: the waves' partials of PASSES groups of NTP column tiles, one after the other (at most LDSK KiB), and the scales.
template <int TM, int NT, int KW, int LDSK>
struct iu8_stream_geo {
  static constexpr int FIT = LDSK / (KW * TM), PASSES = (NT + FIT - 1) / FIT, NTP = (NT + PASSES - 1) / PASSES;
  static constexpr int RED = KW * TM * NTP * 1024, BYTES = RED + (NT * 16 + TM * 16) * 4;
  static_assert(FIT > 0 && NT * 16 <= KW * 64 && TM * 16 <= KW * 64, "one column tile's partials fit, a thread a scale");
};

// EXACT: how the last steps are issued. Every load of the ring stands where the compiler can count those in flight at each
// consume (under a test it waits for all of them). EXACT: one straight-line tail a remainder, a pointer a lane; else one loop
// whose issue past a wave's last step reads the matrix's first fragment, which is cached, and drops it, on wave-uniform bases.
// The first asks for no byte too many, the second keeps the addresses out of vector registers and the unpack out of the tail's
// common head; which is faster differs by cell. us, loop / exact: W4 5 rows of 5120 x 5120 5.6 / 5.1, 20 rows 7.1 / 6.5, 64 rows of
// 4096 x 4096 7.5 / 7.1, 45 rows of 34816 x 5120 22.0 / 21.3; W8 16 rows of 5120 x 6144 9.6 / 8.4; the other way W8 64 rows 12.6 / 12.9, W4
// 72 rows of 20480 x 5120 21.4 / 22.7, W8 45 rows of 20480 x 5120 22.4 / 23.7.
template <int TM, bool W8, int NT, int KW, int D, bool ACC, int LDSK, bool EXACT, bool SHORT = false>
__device__ __forceinline__ void iu8_stream_body(iu8_u8 *__restrict__ lds, const iu8_u8 *__restrict__ A, const iu8_u8 *__restrict__ W,
                                                const float *__restrict__ as, const float *__restrict__ ws, int *__restrict__ P,
                                                int *__restrict__ cnt, void *__restrict__ Cv, int M, int N, int K, const iu8_blk B) {
  using geo = iu8_stream_geo<TM, NT, KW, LDSK>;
  constexpr int WSTEP = W8 ? 2048 : 1024, WV = W8 ? 2 : 1;  // bytes of a 16-row weight tile a step, 16-byte loads a lane
  constexpr int BN = NT * 16, PASSES = geo::PASSES, NTP = geo::NTP;
  constexpr int ITEMS = TM * NTP, NI = (ITEMS + KW - 1) / KW;  // 16 x 16 tiles of a group's output; a wave sums and stores NI
  int *s_red = (int *)lds;
  float *s_sc = (float *)(lds + geo::RED);
  __shared__ int s_last;

  const int tid = threadIdx.x, lane = tid & 63, wk = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntiles = N >> 4, steps = K >> 7, ktiles = K >> 6;
  const int Z = B.Z, z = B.z, spb = (steps + Z - 1) / Z;
  const int s_lo = z * spb, s_hi = min(steps, s_lo + spb);
  const int nt0 = B.bx * NT, ml = lane & 15, lg = lane >> 4;
  // this wave's steps: s_lo + wk + t * KW, t in [0, T)
  const int T = s_lo + wk < s_hi ? (s_hi - s_lo - wk + KW - 1) / KW : 0;

  // wave-uniform bases and 32-bit lane offsets: no address arithmetic in vector registers
  const unsigned lane16 = lane * 16;
  const iu8_u8 *wb[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) wb[j] = W + (size_t)min(nt0 + j, ntiles - 1) * steps * WSTEP;  // past N: the last tile, not stored
  unsigned ao[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    // a lane past the live rows reads the last live row again (a line its load touches anyway); its output is not stored
    const int ar = min(i * 16 + ml, M - 1);
    ao[i] = (unsigned)((ar >> 4) * ktiles * 1024 + ((ar & 15) + 16 * lg) * 16);
  }
  // the epilogue's scales are requested in front of everything else and wait in registers: asked for behind the last K
  // step they are one or two memory latencies on the launch
  const float pre_ws = ws[min(B.bx * BN + tid, N - 1)], pre_as = as[min(tid, M - 1)];

  iu8_v4i acc[TM][NT];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = iu8_v4i{0, 0, 0, 0};
  // (the fences below keep a slot's re-issue behind its own consume and in front of the next slot's)
  iu8_v4u ring[D][NT][WV];
  iu8_v4i ringa[D][TM][2];
  auto consume = [&](int slot) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      iu8_v4i w0, w1;
      if constexpr (W8) {
        w0 = (iu8_v4i)ring[slot][j][0];
        w1 = (iu8_v4i)ring[slot][j][WV - 1];
      } else {
        iu8_unpack_w4(ring[slot][j][0], w0, w1);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[i][j] = iu8_mfma(w0, ringa[slot][i][0], acc[i][j]);
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[i][j] = iu8_mfma(w1, ringa[slot][i][1], acc[i][j]);
    }
  };
  if constexpr (EXACT) {
    // the wave's first step of every tile, a pointer a lane
    const iu8_u8 *wp[NT], *ap[TM];
#pragma unroll
    for (int j = 0; j < NT; ++j) wp[j] = wb[j] + (size_t)(s_lo + wk) * WSTEP + lane16;
#pragma unroll
    for (int i = 0; i < TM; ++i) ap[i] = A + (size_t)(s_lo + wk) * 2048 + ao[i];
    auto issue = [&](int slot, int t) {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int v = 0; v < WV; ++v) ring[slot][j][v] = iu8_ldg_nt(wp[j] + (size_t)t * (KW * WSTEP) + v * 1024);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) ringa[slot][i][h] = *(const iu8_v4i *)(ap[i] + ((size_t)t * (2 * KW) + h) * 1024);
    };
    if (T > 0) {
#pragma unroll
      for (int i = 0; i < D; ++i) issue(i, min(i, T - 1));
    }
    int t0 = 0;
    for (; t0 + 2 * D <= T; t0 += D) {
#pragma unroll
      for (int i = 0; i < D; ++i) {
        consume(i);
        __builtin_amdgcn_sched_barrier(0);
        issue(i, t0 + i + D);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    const int rest = T - t0;  // up to 2D - 1 steps left, min(rest, D) of them in the ring
#pragma unroll
    for (int e = 0; e < D; ++e) {
      if (rest - D != e) continue;  // rest = D + e: e more steps to issue
#pragma unroll
      for (int i = 0; i < D; ++i) {
        consume(i);
        __builtin_amdgcn_sched_barrier(0);
        if (i < e) issue(i, t0 + i + D);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < e; ++i) consume(i);
    }
    if (rest < D) {
#pragma unroll
      for (int i = 0; i < D; ++i)
        if (i < rest) consume(i);
    }
  } else {
    auto issue = [&](int slot, int t) {
      const bool live = t < T;
      const int s = live ? s_lo + wk + t * KW : 0;
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int v = 0; v < WV; ++v) ring[slot][j][v] = iu8_ldg_nt((live ? wb[j] : W) + (size_t)s * WSTEP + v * 1024 + lane16);
      const iu8_u8 *ab = A + (size_t)s * 2048;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) ringa[slot][i][h] = *(const iu8_v4i *)(ab + h * 1024 + ao[i]);
    };
    // SHORT, a symbol's own cell, which the law takes at any K: a wave without a step asks for nothing. The matrix's first fragment,
    // read by every such wave of the grid, is one line of one channel (W8, 33 rows of 8192 x 256 / 384 / 640 4.8 / 5.0 / 5.5 -> 3.6 /
    // 4.1 / 4.5 us). The wider cells start at a K that gives every wave a step.
    if (!SHORT || T > 0) {
#pragma unroll
      for (int i = 0; i < D; ++i) {
        issue(i, i);
        __builtin_amdgcn_sched_barrier(0);
      }
      int t0 = 0;
      for (; t0 + D < T; t0 += D) {
#pragma unroll
        for (int i = 0; i < D; ++i) {
          consume(i);
          __builtin_amdgcn_sched_barrier(0);
          issue(i, t0 + i + D);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
#pragma unroll
      for (int i = 0; i < D; ++i) {
        if (t0 + i < T) consume(i);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // ---- the k-waves' partials meet in LDS (exact int32 adds), and every wave sums and stores its share of the block's
  // items: with wave 0 doing all of it behind scales asked for only here, the end of a launch was a chain of memory
  // latencies (figures: iu8_variants.def).
  if (tid < BN) s_sc[tid] = iu8_wsu<W8>(&pre_ws, 0);
  if (tid < TM * 16) s_sc[BN + tid] = pre_as;
  // item u of group p: the lane's row and first of four columns
  struct at_t {
    int m, n, col;  // col: of the block's columns
    bool live;
  };
  auto at = [&](int p, int u) {
    const int item = wk + u * KW, j = p * NTP + item % NTP, col = j * 16 + lg * 4;
    const at_t t{(item / NTP) * 16 + ml, B.bx * BN + col, col, true};
    return at_t{t.m, t.n, t.col, item < ITEMS && j < NT && t.m < M && t.n < N};
  };
  iu8_v4i sum[PASSES][NI];
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    if (p) __syncthreads();
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < NTP; ++j)
        if (p * NTP + j < NT) *(iu8_v4i *)&s_red[((wk * TM + i) * NTP + j) * 256 + lane * 4] = acc[i][p * NTP + j];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      sum[p][u] = iu8_v4i{0, 0, 0, 0};
      if (wk + u * KW < ITEMS) {
#pragma unroll
        for (int q = 0; q < KW; ++q) sum[p][u] += *(const iu8_v4i *)&s_red[(q * ITEMS + wk + u * KW) * 256 + lane * 4];
      }
    }
  }
  auto store = [&](int p, int u) {
    const at_t t = at(p, u);
    if (!t.live) return;
    if constexpr (ACC) {
      *(iu8_v4i *)((int *)Cv + (size_t)t.m * N + t.n) = sum[p][u];
    } else {
      const float am = s_sc[BN + t.m];
      unsigned h[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) h[r] = iu8_bf16_bits(iu8_epi(sum[p][u][r], am, s_sc[t.col + r]));
      *(iu8_v2u *)((unsigned short *)Cv + (size_t)t.m * N + t.n) = iu8_v2u{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
    }
  };
  if (Z == 1) {
#pragma unroll
    for (int p = 0; p < PASSES; ++p)
#pragma unroll
      for (int u = 0; u < NI; ++u) store(p, u);
    return;
  }

  // ---- grid-level split of K: partials to `decode_partial`, quad-major ([N / 4][M][4 columns] a share: a wave's store and
  // load of an item are four runs of 256 bytes), the last-arriving workgroup of this column block adds the others' to its own
  // and runs the epilogue; the counter is left at zero.
  auto part = [&](int q, int m, int n) { return &P[(((size_t)q * (N >> 2) + (n >> 2)) * M + m) * 4]; };
#pragma unroll
  for (int p = 0; p < PASSES; ++p)
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      const at_t t = at(p, u);
      if (t.live) iu8_store_through(part(z, t.m, t.n), sum[p][u]);
    }
  iu8_stores_done();
  __syncthreads();
  const iu8_arrival arrival = iu8_arrival_of(B.bx, Z, iu8_stream_shared_words(W8, TM, K));
  int *const word = &cnt[arrival.word];
  if (tid == 0) s_last = arrival.last((unsigned)iu8_arrive(word, (int)arrival.one()), Z);
  __syncthreads();
  if (!s_last) return;
  if (tid == 0) iu8_arrive(word, (int)(0u - arrival.all(Z)));
  constexpr int SH = PASSES * NI <= 2 ? 3 : PASSES * NI <= 9 ? 2 : 1;  // shares asked for at a time
  for (int q0 = 1; q0 < Z; q0 += SH) {
    iu8_v4i v[SH][PASSES][NI];
#pragma unroll
    for (int s = 0; s < SH; ++s)
      if (q0 + s < Z) {
        const int q = z + q0 + s < Z ? z + q0 + s : z + q0 + s - Z;
#pragma unroll
        for (int p = 0; p < PASSES; ++p)
#pragma unroll
          for (int u = 0; u < NI; ++u) {
            const at_t t = at(p, u);
            v[s][p][u] = iu8_load_through(part(q, min(t.m, M - 1), min(t.n, N - 4)));  // (no such item: some entry, dropped)
          }
      }
#pragma unroll
    for (int s = 0; s < SH; ++s)
      if (q0 + s < Z) {
#pragma unroll
        for (int p = 0; p < PASSES; ++p)
#pragma unroll
          for (int u = 0; u < NI; ++u) sum[p][u] += v[s][p][u];
      }
  }
#pragma unroll
  for (int p = 0; p < PASSES; ++p)
#pragma unroll
    for (int u = 0; u < NI; ++u) store(p, u);
}

// A symbol's two cells in one LDS block. The launch's own grid says which runs: 64-column blocks where `nblk` blocks of the
// symbol's own width would not reach the last column (iu8_stream_law.h is the host's rule for it). So the arrivals are counted
// by the grid's blocks (iu8_arrival_of: in no more words than blocks), and a grid laid out in the symbol's own blocks stays right where the rule has changed since.
template <int TM, bool W8, int NT, int KW, int D, bool ACC>
__device__ __forceinline__ void iu8_stream_cells(const iu8_u8 *__restrict__ A, const iu8_u8 *__restrict__ W, const float *__restrict__ as,
                                                 const float *__restrict__ ws, int *__restrict__ P, int *__restrict__ cnt,
                                                 void *__restrict__ Cv, int M, int N, int K, const iu8_blk B, int nblk) {
  constexpr int LDSK = 72;  // two workgroups a CU
  constexpr int NW = IU8_STREAM_WIDE_NT;
  constexpr int OWN = iu8_stream_geo<TM, NT, KW, LDSK>::BYTES, WIDE = iu8_stream_geo<TM, NW, KW, LDSK>::BYTES;
  __shared__ __attribute__((aligned(16))) iu8_u8 lds[KW == 8 && WIDE > OWN ? WIDE : OWN];
  if constexpr (KW == 8) {
    if (nblk < (N + NT * 16 - 1) / (NT * 16)) {
      iu8_stream_body<TM, W8, NW, KW, 1, ACC, LDSK, TM <= 2>(lds, A, W, as, ws, P, cnt, Cv, M, N, K, B);
      return;
    }
  }
  iu8_stream_body<TM, W8, NT, KW, D, ACC, LDSK, !(W8 && TM >= 3), true>(lds, A, W, as, ws, P, cnt, Cv, M, N, K, B);
}
