// The attention output gate's Hadamard-basis int8 producer for gfx950: the code object
// `attn_glue_hadi8`, standing in for the reference's object of the same name
// (crates/saber-kernels/hip/attn_glue_hadi8.hip, symbol crates/saber-kernels/src/macaq_iu8.rs:870)
// with the same kernel symbol and kernarg layout (`had_t` last).
//
//   attn_gate_quant_hadi8_t256_tiled1   v = bf16(core * bf16(sigmoid(gate))), the o_proj's A producer.
//       core bf16 [rows, n]; gate is the projection's [q | gate] block, row stride `gs`, head stride
//       2*hd, the gate half at +hd (crates/saber-kernels/src/abi.rs:2683-2694); n <= 6144.
//
// Then u = v * t, x = H32 u per 32-block, x * (1/sqrt(32)), and the per-token int8 law on x; codes
// in the gfx950 A fragment order. sigmoid = 1 / (1 + expf(-g)) is rounded to bf16 before use, so the
// device's expf shows only through a bf16 -> bf16 function (glue_sigmoid_bf16, iu8_had.h), which a
// tap kernel of the test-only object `iu8_taps` tables.
#include "iu8_had.h"

// `lut` (the table form, may be null): bf16(sigmoid) of every bf16 pattern as attn_gate_sigmoid_bf16_table wrote
// it; the gate is then read from the table's middle in LDS (iu8_had.h) instead of computed.
template <bool LUT, int T = 256, int MG = HAD_MAXG>
static __device__ __forceinline__ void attn_gate_body(const unsigned short *__restrict__ core,
                                                      const unsigned short *__restrict__ gate, unsigned char *__restrict__ q,
                                                      float *__restrict__ scale, int n, int hd, int gs,
                                                      const float *__restrict__ had_t,
                                                      const unsigned short *__restrict__ lut) {
#pragma clang fp contract(off)
  const int row = had_row(), tid = threadIdx.x, NV = n >> 3;
  core += (size_t)row * n, gate += (size_t)row * gs;
  __shared__ __attribute__((aligned(16))) unsigned short s_lut[LUT ? 2 * HAD_LUT_N : 8];
  // one group a thread (few rows): the row's pieces and signs are requested with the table, in front of its barrier (6,144
  // wide, table form, at 1 / 16 / 45 / 200 rows 4.36 / 4.63 / 4.77 / 5.59 -> 3.65 / 3.93 / 4.07 / 4.89 us, with the shorter
  // lane stages, roundings and table addresses of iu8_had.h, which take 777 / 2,048 rows from 13.7 / 19.1 to 12.6 / 18.1)
  constexpr bool EARLY = T == 1024 && MG == 1;
  iu8_v4u rc[EARLY ? MG : 1], rg[EARLY ? MG : 1];
  iu8_v4f t_lo, t_hi;
  auto pieces = [&](int g, iu8_v4u &c, iu8_v4u &a) {
    const int e = g << 3, h = e / hd, o = e - h * hd;
    c = *(const iu8_v4u *)(core + e), a = *(const iu8_v4u *)(gate + (size_t)h * 2 * hd + hd + o);
  };
  if constexpr (EARLY) {
#pragma unroll
    for (int i = 0; i < MG; ++i) pieces(min(tid + i * T, NV - 1), rc[i], rg[i]);
    const float *t8 = had_t + 8 * min(tid, NV - 1);
    t_lo = *(const iu8_v4f *)t8, t_hi = *(const iu8_v4f *)(t8 + 4);
  }
  if constexpr (LUT) {
    had_lut_copy<unsigned short, T> tb;
    tb.request(lut, tid);
    tb.commit(s_lut, tid);
    __syncthreads();
  }
  float sv[MG][8];
#pragma unroll
  for (int i = 0; i < MG; ++i) {
    const int g = tid + i * T;
    if (g >= NV) continue;
    iu8_v4u c, a;
    if constexpr (EARLY) c = rc[i], a = rg[i];
    else pieces(g, c, a);
    float vc[8], vg[8];
    had_unpack8(c, vc);
    if constexpr (LUT) {
      unsigned t[4];
      bool far;
      had_lut8(s_lut, a, t, far);
      had_unpack8(iu8_v4u{t[0], t[1], t[2], t[3]}, vg);
      if (__builtin_expect(far, 0)) {
        asm volatile("");  // stays a branch (iu8_code4_rcp has the reason)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const unsigned b = j & 1 ? a[j >> 1] >> 16 : a[j >> 1] & 0xFFFFu;
          if (!had_lut_inside(b)) vg[j] = glue_sigmoid_bf16(iu8_bf16_f32((unsigned short)b));
        }
      }
    } else {
      had_unpack8(a, vg);
#pragma unroll
      for (int j = 0; j < 8; ++j) vg[j] = glue_sigmoid_bf16(vg[j]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) sv[i][j] = vc[j] * vg[j];
    had_bf16_round(sv[i]);
    if constexpr (EARLY) had32(sv[i], t_lo, t_hi, tid);
    else had32(sv[i], had_t + 8 * g, tid);
  }
  had_tail<T>(sv, NV, q, scale, row, n);
}
extern "C" __global__ __launch_bounds__(256) void attn_gate_quant_hadi8_t256_tiled1(
    const unsigned short *__restrict__ core, const unsigned short *__restrict__ gate, unsigned char *__restrict__ q,
    float *__restrict__ scale, int n, int hd, int gs, const float *__restrict__ had_t) {
  attn_gate_body<false>(core, gate, q, scale, n, hd, gs, had_t, nullptr);
}
// the table form (no counterpart among the reference's symbols: `lut` behind its kernarg list)
extern "C" __global__ __launch_bounds__(256) void attn_gate_quant_hadi8_lut_t256(
    const unsigned short *__restrict__ core, const unsigned short *__restrict__ gate, unsigned char *__restrict__ q,
    float *__restrict__ scale, int n, int hd, int gs, const float *__restrict__ had_t,
    const unsigned short *__restrict__ lut) {
  attn_gate_body<true>(core, gate, q, scale, n, hd, gs, had_t, lut);
}
// 16 waves a row, for few rows (no counterpart among the reference's symbols)
extern "C" __global__ __launch_bounds__(1024) void attn_gate_quant_hadi8_t1024(
    const unsigned short *__restrict__ core, const unsigned short *__restrict__ gate, unsigned char *__restrict__ q,
    float *__restrict__ scale, int n, int hd, int gs, const float *__restrict__ had_t) {
  if (n <= 8 * 1024) attn_gate_body<false, 1024, 1>(core, gate, q, scale, n, hd, gs, had_t, nullptr);
  else attn_gate_body<false, 1024>(core, gate, q, scale, n, hd, gs, had_t, nullptr);
}
extern "C" __global__ __launch_bounds__(1024) void attn_gate_quant_hadi8_lut_t1024(
    const unsigned short *__restrict__ core, const unsigned short *__restrict__ gate, unsigned char *__restrict__ q,
    float *__restrict__ scale, int n, int hd, int gs, const float *__restrict__ had_t,
    const unsigned short *__restrict__ lut) {
  if (n <= 8 * 1024) attn_gate_body<true, 1024, 1>(core, gate, q, scale, n, hd, gs, had_t, lut);
  else attn_gate_body<true, 1024>(core, gate, q, scale, n, hd, gs, had_t, lut);
}
// bf16(sigmoid) of all 65,536 bf16 inputs (bf16 bits [65536]): the table of attn_gate_quant_hadi8_lut_t256.
// grid 256, block 256.
extern "C" __global__ __launch_bounds__(256) void attn_gate_sigmoid_bf16_table(unsigned short *__restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  out[i] = (unsigned short)iu8_bf16_bits(glue_sigmoid_bf16(iu8_bf16_f32((unsigned short)i)));
}
