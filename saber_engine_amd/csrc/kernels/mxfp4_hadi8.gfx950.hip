// The Hadamard-basis int8 producers for gfx950: the code object `mxfp4_hadi8`, standing in for the
// reference's object of the same name (crates/saber-kernels/hip/mxfp4_hadi8.hip, symbols
// crates/saber-kernels/src/macaq_iu8.rs:864-875) with the same kernel symbols and kernarg layouts
// (`had_t` last). A producer's final bf16-rounded values v become u = v * t, x = H32 u per 32-block
// along K, x = x * (1/sqrt(32)) (crates/saber-kernels/hip/macaq_had.h:1-19), and the per-token int8
// law runs on x (iu8_common.h); codes are stored in the gfx950 A fragment order.
//
//   add_rms_quant_hadi8_t{256,512}_tiled1   v = bf16((f32(y) + f32(res)) * inv * (f32(w) + 1)), res_out = bf16(y + res)
//   silu_mul_quant_hadi8_t{256,512}_tiled1  v = bf16(bf16(silu(gate)) * up)
//   silu_mul_quant_hadi8_lut_t{256,512}     the same with bf16(silu(gate)) read from a table (LDS)
//   quant_hadi8_t{256,512}_tiled1           v = x (no counterpart among the reference's symbols: the
//                                           transform in front of the plain producer)
//   gdn_norm_quant_hadi8_t256_tiled1        v = bf16(((x * inv_head) * w) * silu_f32(z)), per 128-element head
//
// The sums of squares keep the reference's order: add_rms per-thread fma over its groups, then
// shfl_down 16..1 inside each 32 lanes, then over the T/32 partials; gdn_norm per group
// (x1*x1, fma x0, fma x2..x7), then the xor butterfly 8, 4, 2, 1 over the head's 16 lanes. Their
// `rsqrtf` is the one thing not taken over: the device's approximate reciprocal square root cannot be
// restated on a host, so inv = 1 / sqrt(x) here uses the IEEE square root and divide (`__builtin_sqrtf`, which
// this toolchain expands to the correctly rounded sequence; its `__fsqrt_rn` is the native approximation, an
// ulp off now and then, which showed as a bf16 value of a row flipped once in a few million elements). gdn_norm's
// gate silu_f32(z) = z / (1 + expf(-z)) stays in f32 and so carries the device's expf: a function of
// a bf16 input, it is tabled by a tap kernel of the test-only object `iu8_taps` (had_silu_f32 lives
// in iu8_had.h for both) for a test to hold against a host's.
#include "iu8_had.h"

template <int T>
static __device__ __forceinline__ void had_quant_body(const unsigned short *__restrict__ x, iu8_u8 *__restrict__ q,
                                                      float *__restrict__ scale, int K,
                                                      const float *__restrict__ had_t) {
  const int row = had_row(), tid = threadIdx.x, NV = K >> 3;
  x += (size_t)row * K;
  float sv[HAD_MAXG][8];
#pragma unroll
  for (int i = 0; i < HAD_MAXG; ++i) {
    const int g = tid + i * T;
    if (g >= NV) continue;
    had_load8(x + g * 8, sv[i]);
    had32(sv[i], had_t + 8 * g, tid);
  }
  had_tail<T>(sv, NV, q, scale, row, K);
}

// Bound by the VALU (transform, codes, activation) and by a row's latency for few rows: the activation is the hardware's exp2
// and reciprocal where they give the law's bf16 (iu8_silu_mul4), and the row's pieces leave in one batch of loads instead of
// one a group. us before / now: rows of 17,408 at 1 / 45 / 200 rows (t1024) 8.70 / 9.41 / 10.85 -> 6.62 / 7.37 / 9.26, at 777 /
// 2,048 / 6,144 (t512) 27.6 / 57.2 / 154.0 -> 23.6 / 44.1 / 118.9; 2,048 rows of 5,120 (t256) 19.7 -> 16.5, of 2,048 9.9 -> 8.2.
template <int T>
static __device__ __forceinline__ void had_silu_body(const unsigned short *__restrict__ gu, iu8_u8 *__restrict__ q,
                                                     float *__restrict__ scale, int N,
                                                     const float *__restrict__ had_t) {
#pragma clang fp contract(off)
  const int row = had_row(), tid = threadIdx.x, NV = N >> 3;
  gu += (size_t)row * 2 * N;
  // all of the row's pieces are requested before the first is used
  iu8_v4u rg[HAD_MAXG], ru[HAD_MAXG];
#pragma unroll
  for (int i = 0; i < HAD_MAXG; ++i) {
    const int g = tid + i * T;
    rg[i] = ru[i] = iu8_v4u{0u, 0u, 0u, 0u};
    if (g < NV) rg[i] = *(const iu8_v4u *)(gu + (unsigned)(g * 8)), ru[i] = *(const iu8_v4u *)(gu + N + (unsigned)(g * 8));
  }
  float sv[HAD_MAXG][8];
#pragma unroll
  for (int i = 0; i < HAD_MAXG; ++i) {
    const int g = tid + i * T;
    if (g >= NV) continue;
    unsigned p[4];
    iu8_silu_mul4(rg[i][0], rg[i][1], ru[i][0], ru[i][1], p[0], p[1]);
    iu8_silu_mul4(rg[i][2], rg[i][3], ru[i][2], ru[i][3], p[2], p[3]);
#pragma unroll
    for (int w = 0; w < 4; ++w) sv[i][2 * w] = __uint_as_float(p[w] << 16), sv[i][2 * w + 1] = __uint_as_float(p[w] & 0xFFFF0000u);
    had32(sv[i], had_t + 8 * g, tid);
  }
  had_tail<T>(sv, NV, q, scale, row, N);
}

template <int T>
static __device__ __forceinline__ void had_add_rms_body(const unsigned short *__restrict__ y,
                                                        const unsigned short *__restrict__ res,
                                                        const unsigned short *__restrict__ w, iu8_u8 *__restrict__ q,
                                                        float *__restrict__ scale, unsigned short *__restrict__ res_out,
                                                        int K, float eps, const float *__restrict__ had_t) {
#pragma clang fp contract(off)
  __shared__ float s_sum[T / 32];
  const int row = had_row(), tid = threadIdx.x, NV = K >> 3;
  y += (size_t)row * K, res += (size_t)row * K, res_out += (size_t)row * K;
  float sv[HAD_MAXG][8];
  float ssq = 0.f;
#pragma unroll
  for (int i = 0; i < HAD_MAXG; ++i) {
    const int g = tid + i * T;
    if (g >= NV) continue;
    float vy[8], vr[8];
    had_load8(y + g * 8, vy);
    had_load8(res + g * 8, vr);
    unsigned o[4];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float v = vy[j] + vr[j];
      sv[i][j] = v;
      ssq = __builtin_fmaf(v, v, ssq);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = iu8_bf16_pack(sv[i][2 * j], sv[i][2 * j + 1]);
    *(iu8_v4u *)(res_out + g * 8) = iu8_v4u{o[0], o[1], o[2], o[3]};
  }
  // the reference's trees (32 lanes, then the T/32 partials), so the sum's bits are its own
#pragma unroll
  for (int o = 16; o; o >>= 1) ssq = ssq + __shfl_down(ssq, o, 32);
  if ((tid & 31) == 0) s_sum[tid >> 5] = ssq;
  __syncthreads();
  if (tid < T / 32) {
    float v = s_sum[tid];
#pragma unroll
    for (int o = T / 64; o; o >>= 1) v = v + __shfl_down(v, o, 32);
    if (tid == 0) s_sum[0] = v;
  }
  __syncthreads();
  const float inv = __fdiv_rn(1.f, __builtin_sqrtf(__fdiv_rn(s_sum[0], (float)K) + eps));
#pragma unroll
  for (int i = 0; i < HAD_MAXG; ++i) {
    const int g = tid + i * T;
    if (g >= NV) continue;
    float vw[8];
    had_load8(w + g * 8, vw);
#pragma unroll
    for (int j = 0; j < 8; ++j) sv[i][j] = (sv[i][j] * inv) * (vw[j] + 1.f);
    had_bf16_round(sv[i]);
    had32(sv[i], had_t + 8 * g, tid);
  }
  had_tail<T>(sv, NV, q, scale, row, K);
}

// add_rms for few rows of up to 8,192 elements, 16 waves a row, with the sum of squares in the 256-thread form's order
// (which is part of its law: thread t of 256 runs one fma chain over its groups t, t + 256, t + 512, t + 768 in turn, then
// the 32-lane and 8-partial trees). Here thread tid owns group tid and puts y + res in LDS, from where the first 256 threads
// run the chains; everything else (the loads, y + res and its store, the weights, the transform, the codes) runs on four
// times the threads. Same bits as add_rms_quant_hadi8_t256_tiled1. (The chain was handed from slice to slice of 256 threads in
// four turns, six barriers in all: 5,120 wide at 1 / 16 / 200 rows 4.56 / 4.92 / 5.87 us, here 3.96 / 4.28 / 5.19; the t256 form,
// which has the one-addition lane stages and the paired roundings as well, at 777 / 2,048 rows 10.9 / 21.0 -> 9.8 / 19.1.)
static __device__ __forceinline__ void had_add_rms_v256_body(const unsigned short *__restrict__ y,
                                                             const unsigned short *__restrict__ res,
                                                             const unsigned short *__restrict__ w, iu8_u8 *__restrict__ q,
                                                             float *__restrict__ scale, unsigned short *__restrict__ res_out,
                                                             int K, float eps, const float *__restrict__ had_t) {
#pragma clang fp contract(off)
  constexpr int T = 1024, V = 256;
  __shared__ __attribute__((aligned(16))) float s_v[T * 8];
  __shared__ float s_sum[V / 32];
  const int row = had_row(), tid = threadIdx.x, NV = K >> 3, g = tid;
  const bool live = g < NV;
  y += (size_t)row * K, res += (size_t)row * K, res_out += (size_t)row * K;
  float sv[1][8], vw[8];
  iu8_v4f t_lo = {0.f, 0.f, 0.f, 0.f}, t_hi = t_lo;
  if (live) {  // everything the row needs is requested before the first of it is used
    float vy[8], vr[8];
    const iu8_v4u ry = *(const iu8_v4u *)(y + g * 8), rr = *(const iu8_v4u *)(res + g * 8);
    had_load8(w + g * 8, vw);
    t_lo = *(const iu8_v4f *)(had_t + 8 * g), t_hi = *(const iu8_v4f *)(had_t + 8 * g + 4);
    had_unpack8(ry, vy), had_unpack8(rr, vr);
    unsigned o[4];
#pragma unroll
    for (int j = 0; j < 8; ++j) sv[0][j] = vy[j] + vr[j];
    // element-pair-major: a wave's 8-byte pieces lie side by side
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      *(iu8_v2f *)&s_v[(j * T + g) * 2] = iu8_v2f{sv[0][2 * j], sv[0][2 * j + 1]};
      o[j] = iu8_bf16_pack(sv[0][2 * j], sv[0][2 * j + 1]);
    }
    *(iu8_v4u *)(res_out + g * 8) = iu8_v4u{o[0], o[1], o[2], o[3]};
  }
  __syncthreads();
  if (tid < V) {  // thread t's chain over the groups t, t + 256, t + 512, t + 768
    float ssq = 0.f;
#pragma unroll
    for (int i = 0; i < T / V; ++i)
      if (tid + i * V < NV) {
        iu8_v2f p[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) p[j] = *(const iu8_v2f *)&s_v[(j * T + tid + i * V) * 2];
#pragma unroll
        for (int j = 0; j < 4; ++j) ssq = __builtin_fmaf(p[j].x, p[j].x, ssq), ssq = __builtin_fmaf(p[j].y, p[j].y, ssq);
      }
    ssq = had_sum32(ssq);
    if ((tid & 31) == 0) s_sum[tid >> 5] = ssq;
  }
  __syncthreads();
  // the tree over the 8 partials (4, 2, 1 apart), by every thread
  const float ms = ((s_sum[0] + s_sum[4]) + (s_sum[2] + s_sum[6])) + ((s_sum[1] + s_sum[5]) + (s_sum[3] + s_sum[7]));
  const float inv = __fdiv_rn(1.f, __builtin_sqrtf(__fdiv_rn(ms, (float)K) + eps));
  if (live) {
#pragma unroll
    for (int j = 0; j < 8; ++j) sv[0][j] = (sv[0][j] * inv) * (vw[j] + 1.f);
    had_bf16_round(sv[0]);
    had32(sv[0], t_lo, t_hi, tid);
  }
  had_tail<T, 1>(sv, NV, q, scale, row, K);
}
extern "C" __global__ __launch_bounds__(1024) void add_rms_quant_hadi8_t1024(
    const unsigned short *__restrict__ y, const unsigned short *__restrict__ res, const unsigned short *__restrict__ w,
    unsigned char *__restrict__ q, float *__restrict__ scale, unsigned short *__restrict__ res_out, int K, float eps,
    const float *__restrict__ had_t) {
  had_add_rms_v256_body(y, res, w, q, scale, res_out, K, eps, had_t);
}

#define HAD_ARQ(name, T)                                                                                          \
  extern "C" __global__ __launch_bounds__(T) void name(                                                          \
      const unsigned short *__restrict__ y, const unsigned short *__restrict__ res,                              \
      const unsigned short *__restrict__ w, unsigned char *__restrict__ q, float *__restrict__ scale,            \
      unsigned short *__restrict__ res_out, int K, float eps, const float *__restrict__ had_t) {                 \
    had_add_rms_body<T>(y, res, w, q, scale, res_out, K, eps, had_t);                                            \
  }
HAD_ARQ(add_rms_quant_hadi8_t256_tiled1, 256)
HAD_ARQ(add_rms_quant_hadi8_t512_tiled1, 512)
#undef HAD_ARQ

#define HAD_SMQ(name, T)                                                                                          \
  extern "C" __global__ __launch_bounds__(T) void name(const unsigned short *__restrict__ gu,                    \
                                                       unsigned char *__restrict__ q, float *__restrict__ scale, \
                                                       int N, const float *__restrict__ had_t) {                 \
    had_silu_body<T>(gu, q, scale, N, had_t);                                                                    \
  }
HAD_SMQ(silu_mul_quant_hadi8_t256_tiled1, 256)
HAD_SMQ(silu_mul_quant_hadi8_t512_tiled1, 512)
HAD_SMQ(silu_mul_quant_hadi8_t1024, 1024)  // 16 waves a row: few long rows (no counterpart among the reference's symbols)
#undef HAD_SMQ

// silu_mul_quant with the bf16 silu read from a table: `lut` holds bf16(silu(x)) of every bf16 bit pattern x as
// macaq_silu_bf16_table (code object `macaq_i8q`) wrote it, i.e. this file's own expression
// vg / (1 + expf(-vg)) rounded to bf16, so the bytes are those of the computed form. Rows of 17,408, us on the computed
// form / here: 1 / 200 rows 6.51 / 9.12, 6.09 / 9.00; 777 / 2,048 rows 23.8 / 41.9, 22.5 / 41.3 (a branch and an address an element: 23.3 / 43.1); rows of
// 5,120 within 6 % either way; rows of 2,048 up to 512 rows 0.35-0.5 us in favour of the computed form. A workgroup copies the
// table's middle -- magnitudes from 2^-17 up to 2^15, both signs: 2 x 4,096 entries, 16 KiB -- into LDS beside
// its row's loads; a gate outside (one in some hundred thousand of unit-scale rows) is computed as before.
// The kernel is the computed form otherwise (a workgroup a row, the same lane map). No counterpart among
// the reference's symbols (`lut` behind its kernarg list).
template <int T>
static __device__ __forceinline__ void had_silu_lut_body(const unsigned short *__restrict__ gu, iu8_u8 *__restrict__ q,
                                                         float *__restrict__ scale, int N,
                                                         const float *__restrict__ had_t,
                                                         const unsigned short *__restrict__ lut) {
#pragma clang fp contract(off)
  __shared__ __attribute__((aligned(16))) unsigned short s_lut[2 * HAD_LUT_N];
  const int row = had_row(), tid = threadIdx.x, NV = N >> 3;
  gu += (size_t)row * 2 * N;
  // the row's pieces and the table are requested together, nothing is used before the last request has left
  iu8_v4u rg[HAD_MAXG], ru[HAD_MAXG];
  had_lut_copy<unsigned short, T> tb;
#pragma unroll
  for (int i = 0; i < HAD_MAXG; ++i) {
    const int g = tid + i * T;
    rg[i] = ru[i] = iu8_v4u{0u, 0u, 0u, 0u};
    if (g < NV) rg[i] = *(const iu8_v4u *)(gu + (unsigned)(g * 8)), ru[i] = *(const iu8_v4u *)(gu + N + (unsigned)(g * 8));
  }
  tb.request(lut, tid);
  tb.commit(s_lut, tid);
  __syncthreads();
  float sv[HAD_MAXG][8];
#pragma unroll
  for (int i = 0; i < HAD_MAXG; ++i) {
    const int g = tid + i * T;
    if (g >= NV) continue;
    unsigned t[4];
    bool far;
    had_lut8(s_lut, rg[i], t, far);
    if (__builtin_expect(far, 0)) {
      asm volatile("");  // stays a branch (iu8_code4_rcp has the reason)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        if (!had_lut_inside(rg[i][w])) t[w] = (t[w] & 0xFFFF0000u) | (__float_as_uint(iu8_silu_bf16(__uint_as_float(rg[i][w] << 16))) >> 16);
        if (!had_lut_inside(rg[i][w] >> 16)) t[w] = (t[w] & 0xFFFFu) | __float_as_uint(iu8_silu_bf16(__uint_as_float(rg[i][w] & 0xFFFF0000u)));
      }
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) {  // two products a v_cvt_pk_bf16_f32
      const unsigned p2 = iu8_bf16_pack(__uint_as_float(t[w] << 16) * __uint_as_float(ru[i][w] << 16),
                                        __uint_as_float(t[w] & 0xFFFF0000u) * __uint_as_float(ru[i][w] & 0xFFFF0000u));
      sv[i][2 * w] = __uint_as_float(p2 << 16);
      sv[i][2 * w + 1] = __uint_as_float(p2 & 0xFFFF0000u);
    }
    had32(sv[i], had_t + 8 * g, tid);
  }
  had_tail<T>(sv, NV, q, scale, row, N);
}
#define HAD_SMQ_LUT(name, T)                                                                                      \
  extern "C" __global__ __launch_bounds__(T) void name(                                                          \
      const unsigned short *__restrict__ gu, unsigned char *__restrict__ q, float *__restrict__ scale, int N,    \
      const float *__restrict__ had_t, const unsigned short *__restrict__ lut) {                                 \
    had_silu_lut_body<T>(gu, q, scale, N, had_t, lut);                                                           \
  }
HAD_SMQ_LUT(silu_mul_quant_hadi8_lut_t256, 256)
HAD_SMQ_LUT(silu_mul_quant_hadi8_lut_t512, 512)
HAD_SMQ_LUT(silu_mul_quant_hadi8_lut_t1024, 1024)
#undef HAD_SMQ_LUT

#define HAD_Q(name, T)                                                                                            \
  extern "C" __global__ __launch_bounds__(T) void name(const unsigned short *__restrict__ x,                     \
                                                       unsigned char *__restrict__ q, float *__restrict__ scale, \
                                                       int k, const float *__restrict__ had_t) {                 \
    had_quant_body<T>(x, q, scale, k, had_t);                                                                    \
  }
HAD_Q(quant_hadi8_t256_tiled1, 256)
HAD_Q(quant_hadi8_t512_tiled1, 512)
HAD_Q(quant_hadi8_t1024, 1024)
#undef HAD_Q

// One workgroup a row of N = heads * 128 elements; z rows `zs` elements apart; w the head's 128 weights.
template <int T>
static __device__ __forceinline__ void had_gdn_norm_body(const unsigned short *__restrict__ x,
                                                         const unsigned short *__restrict__ z, long zs,
                                                         const unsigned short *__restrict__ w, iu8_u8 *__restrict__ q,
                                                         float *__restrict__ scale, int N, float eps,
                                                         const float *__restrict__ had_t) {
#pragma clang fp contract(off)
  const int row = had_row(), tid = threadIdx.x, NV = N >> 3;
  x += (size_t)row * N, z += (size_t)row * zs;
  float sv[HAD_MAXG][8];
#pragma unroll
  for (int i = 0; i < HAD_MAXG; ++i) {
    // whole heads (16 lanes) are live or not together: NV is a multiple of 16, T a multiple of 16
    if (i * T >= NV) continue;
    const int g = tid + i * T;
    const bool on = g < NV;
    const int gl = on ? g : 0;
    float vz[8], vw[8];
    had_load8(x + gl * 8, sv[i]);
    float ssq = sv[i][1] * sv[i][1];
    ssq = __builtin_fmaf(sv[i][0], sv[i][0], ssq);
#pragma unroll
    for (int j = 2; j < 8; ++j) ssq = __builtin_fmaf(sv[i][j], sv[i][j], ssq);
    ssq = had_head_sum(ssq);
    if (!on) continue;
    const float inv = __fdiv_rn(1.f, __builtin_sqrtf(ssq * (1.f / 128.f) + eps));
    had_load8(z + g * 8, vz);
    had_load8(w + (g & 15) * 8, vw);
#pragma unroll
    for (int j = 0; j < 8; ++j) sv[i][j] = ((sv[i][j] * inv) * vw[j]) * had_silu_f32(vz[j]);
    had_bf16_round(sv[i]);
    had32(sv[i], had_t + 8 * g, tid);
  }
  had_tail<T>(sv, NV, q, scale, row, N);
}

// The same for rows of at most 8 T elements: one group a thread, everything requested before the first of it is used.
// Few rows are bound by one CU's arithmetic (a quarter of it the gate's exponential and
// divide) and the row's latencies: 6,144 wide at 1 / 16 / 45 / 200 rows 5.54 / 5.86 / 6.02 / 6.77 us in the loop of five groups, here
// 4.24 / 4.53 / 4.69 / 5.66; the loop, which now stops at the row's end, at 777 / 2,048 rows 14.0 / 25.4 -> 13.1 / 24.6.
template <int T>
static __device__ __forceinline__ void had_gdn_norm_one(const unsigned short *__restrict__ x, const unsigned short *__restrict__ z,
                                                        long zs, const unsigned short *__restrict__ w, iu8_u8 *__restrict__ q,
                                                        float *__restrict__ scale, int N, float eps, const float *__restrict__ had_t) {
#pragma clang fp contract(off)
  const int row = had_row(), tid = threadIdx.x, NV = N >> 3, g = min(tid, NV - 1);  // whole heads past the row's end repeat its last group
  const iu8_v4u rx = *(const iu8_v4u *)(x + (size_t)row * N + g * 8), rz = *(const iu8_v4u *)(z + (size_t)row * zs + g * 8);
  const iu8_v4u rw = *(const iu8_v4u *)(w + (g & 15) * 8);
  const iu8_v4f t_lo = *(const iu8_v4f *)(had_t + 8 * g), t_hi = *(const iu8_v4f *)(had_t + 8 * g + 4);
  float sv[1][8], vz[8], vw[8];
  had_unpack8(rx, sv[0]), had_unpack8(rz, vz), had_unpack8(rw, vw);
  float ssq = sv[0][1] * sv[0][1];
  ssq = __builtin_fmaf(sv[0][0], sv[0][0], ssq);
#pragma unroll
  for (int j = 2; j < 8; ++j) ssq = __builtin_fmaf(sv[0][j], sv[0][j], ssq);
  ssq = had_head_sum(ssq);
  if (tid < NV) {
    const float inv = __fdiv_rn(1.f, __builtin_sqrtf(ssq * (1.f / 128.f) + eps));
#pragma unroll
    for (int j = 0; j < 8; ++j) sv[0][j] = ((sv[0][j] * inv) * vw[j]) * had_silu_f32(vz[j]);
    had_bf16_round(sv[0]);
    had32(sv[0], t_lo, t_hi, tid);
  }
  had_tail<T, 1>(sv, NV, q, scale, row, N);
}

extern "C" __global__ __launch_bounds__(256) void gdn_norm_quant_hadi8_t256_tiled1(
    const unsigned short *__restrict__ x, const unsigned short *__restrict__ z, long zs,
    const unsigned short *__restrict__ w, unsigned char *__restrict__ q, float *__restrict__ scale, int N, float eps,
    const float *__restrict__ had_t) {
  had_gdn_norm_body<256>(x, z, zs, w, q, scale, N, eps, had_t);
}
// 16 waves a row: few rows (a head's sum is the 16 lanes' whatever the workgroup's size, so the bits are the same)
extern "C" __global__ __launch_bounds__(1024) void gdn_norm_quant_hadi8_t1024(
    const unsigned short *__restrict__ x, const unsigned short *__restrict__ z, long zs,
    const unsigned short *__restrict__ w, unsigned char *__restrict__ q, float *__restrict__ scale, int N, float eps,
    const float *__restrict__ had_t) {
  if (N <= 8 * 1024) had_gdn_norm_one<1024>(x, z, zs, w, q, scale, N, eps, had_t);
  else had_gdn_norm_body<1024>(x, z, zs, w, q, scale, N, eps, had_t);
}
