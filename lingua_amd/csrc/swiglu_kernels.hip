// SwiGLU gate fused with the row-wise fp8 cast, forward and backward.
//
// The MLP of lingua/transformer.py:430-471 computes w2(silu(w1(x)) * w3(x)).
// Between the GEMMs sit bf16 elementwise passes (silu, mul; in backward two
// muls and silu_backward) and, with the float8 recipe, the casts of the w2
// input and of the two gate gradients (lingua/float8.py:86-87, :43-47).  Each
// of those passes streams a [tokens, ffn] tensor through HBM.  The kernels
// below do the elementwise arithmetic while the row is in registers for its
// amax and cast anyway:
//
//   forward : h  = bf16(bf16(silu(h1)) * h3)          -> q(h), scale, [h], [col amax]
//   backward: g3 = bf16(dh * bf16(silu(h1)))
//             g1 = bf16(bf16(dh * h3) * sig * (1 + h1 * (1 - sig)))
//                                                      -> g1, g3, q(g1), q(g3), scales, [col amaxes]
//
// Every intermediate is rounded to bf16 where the unfused PyTorch chain
// materialises a bf16 tensor, so the results agree with that chain up to the
// last bits of the fp32 sigmoid: at most two bf16 ulps apart, identical for
// more than 99.5 % of the elements (the bound the tests state); amax, scale
// and e4m3 bytes are then exact functions of the bf16 values produced here.
// One workgroup per row (wave w of W owns the 512-column chunks w, w+W, ...),
// the layout of the long-row kernel of cast_kernels.hip; the amax -> scale ->
// cast stage is shared with it.
//
// Where every weight learns, neither h nor g1 and g3 is written: the weight gradients'
// transposed operands are made from dh, h1 and h3 by a kernel of their own (below).
//
// Bound by memory: 5 (+ 2 with h) bytes per element forward, 8 (+ 4 with g1 and g3) backward.  What
// reaches its rate is loads in flight, so a lane holds few chunks and a long row
// takes more waves rather than more registers per lane: four up to 4096 columns,
// eight up to 16384 forward (2 to 4 chunks) and up to 12288 backward (2 or 3),
// sixteen with 2 chunks beyond.  With more than four the column maxima live in
// LDS.  us inside a forward + backward, four waves / this: [16384,8192] forward
// 162.5 / 156.7 (6.0 TB/s), backward 292 / 262 (6.1 TB/s); [4093,14336] forward
// 82.6 / 76.9, backward (a two-pass kernel before) 149.7 / 124.7 (5.6 TB/s).
// Alone, with the folds of the column maxima: backward [16384,5632] 235 / 205,
// [16384,8704] 354 / 309, [16384,11008] 430 / 424, [16384,16384] 710 / 601.
// Without the bf16 results, alone, written / not: [16384,8192] forward 149 / 124 (5.4 TB/s),
// backward 248 / 198 (5.4); [4093,14336] 76 / 61 and 123 / 99; [8192,4096] 46 / 42 and 77 / 67.
#include "l8_common.h"

namespace l8 {

constexpr int kGateBlock = 256;
constexpr int kGateWaves = kGateBlock / 64;

// 1 / (1 + exp(-x)) with the hardware exp2 and reciprocal (about 1 ulp of fp32
// each).  The library exp and the IEEE division cost ~5x the instructions and
// made these kernels VALU-bound (302 us forward / 550 us backward on
// [16384, 11008] against ~230 / ~400 us of memory time); every result is
// rounded to bf16 right away, where an fp32 ulp decides one rounding in ~10^4.
L8_DEV float sigmoid_f32(float x) {
  const float e = __builtin_amdgcn_exp2f(x * -1.4426950408889634f);
  return __builtin_amdgcn_rcpf(1.0f + e);
}
// silu(x) = x / (1 + exp(-x)), fp32
L8_DEV float silu_f32(float x) { return x * sigmoid_f32(x); }

// The gate works on pairs, two elements of a dword: one conversion rounds both and leaves them packed (these kernels are
// within a third of being bound by the vector unit; element by element the gate took 19 issue slots per element forward
// and 31 backward, this takes 16 and 23).
struct Pair {
  float lo, hi;
};
L8_DEV Pair unpack2(uint32_t v) { return {__uint_as_float(v << 16), __uint_as_float(v & 0xffff0000u)}; }
L8_DEV uint32_t pack2(float lo, float hi) {  // (left to itself the compiler converts the halves of what is unpacked again one by one)
  uint32_t r;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(lo), "v"(hi));
  return r;
}

// two packed bf16 of h1 and h3 -> two packed bf16 of h
L8_DEV uint32_t gate_fwd2(uint32_t a, uint32_t b) {
  const Pair x = unpack2(a), y = unpack2(b);
  const Pair s = unpack2(pack2(silu_f32(x.lo), silu_f32(x.hi)));  // a bf16 tensor in the unfused chain
  return pack2(s.lo * y.lo, s.hi * y.hi);
}

// The backward gate, d = dh, a = h1, b = h3; h is gate_fwd2(a, b), for who wants it.  The derivative of silu, sig * (1 + a *
// (1 - sig)), as sig + (a * sig) * (1 - sig) with one fused multiply-add: a rounding less.
L8_DEV void gate_bwd2(uint32_t d, uint32_t a, uint32_t b, uint32_t &g1, uint32_t &g3, uint32_t &h) {
  const Pair x = unpack2(a), y = unpack2(b), z = unpack2(d);
  const Pair sig = {sigmoid_f32(x.lo), sigmoid_f32(x.hi)};
  const Pair xs = {x.lo * sig.lo, x.hi * sig.hi};
  const Pair s = unpack2(pack2(xs.lo, xs.hi));                    // what forward saved: bf16 silu(h1)
  const Pair gs = unpack2(pack2(z.lo * y.lo, z.hi * y.hi));       // gradient of the silu output, a bf16 tensor in the unfused chain
  g3 = pack2(z.lo * s.lo, z.hi * s.hi);
  g1 = pack2(gs.lo * __builtin_fmaf(xs.lo, 1.0f - sig.lo, sig.lo), gs.hi * __builtin_fmaf(xs.hi, 1.0f - sig.hi, sig.hi));
  h = pack2(s.lo * y.lo, s.hi * y.hi);
}
L8_DEV void gate_bwd2(uint32_t d, uint32_t a, uint32_t b, uint32_t &g1, uint32_t &g3) {
  uint32_t h;
  gate_bwd2(d, a, b, g1, g3, h);
}

template <int NCHW, bool COLMAX, int WAVES = kGateWaves>
__global__ __launch_bounds__(WAVES * 64, WAVES == kGateWaves ? 2 : 4) void swiglu_cast_rowwise_kernel(
    const uint16_t *__restrict__ h1, const uint16_t *__restrict__ h3, int64_t R, int C, int64_t ld1, int64_t ld3,
    uint16_t *__restrict__ hout, int64_t ldh, uint8_t *__restrict__ q, int64_t ldq, float *__restrict__ scale,
    uint16_t *__restrict__ amax_out, uint16_t *__restrict__ col_partials, int scale_rule) {
  __shared__ uint32_t red[2][WAVES];
  extern __shared__ __attribute__((aligned(16))) uint8_t dyn_lds[];
  constexpr bool CLDS = COLMAX && WAVES > kGateWaves;  // column maxima in LDS instead of registers
  v4i *lds_cm = (v4i *)dyn_lds;  // [C / 8]
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  auto col_of = [&](int j) { return (j * WAVES + wave) * 512 + lane * 8; };
  uint32_t cmax[(COLMAX && !CLDS) ? NCHW * 4 : 1];
  if (COLMAX) {
#pragma unroll
    for (int j = 0; j < NCHW; ++j) {
      if (CLDS) {
        if (col_of(j) < C) lds_cm[col_of(j) / 8] = v4i{0, 0, 0, 0};
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) cmax[j * 4 + k] = 0;
      }
    }
  }
  int it = 0;
  for (int64_t r = blockIdx.x; r < R; r += gridDim.x, ++it) {
    v4i a[NCHW], b[NCHW], h[NCHW];
#pragma unroll
    for (int j = 0; j < NCHW; ++j) {
      const int c = col_of(j);
      if (c < C) {
        a[j] = __builtin_nontemporal_load((const v4i *)(h1 + r * ld1 + c));
        b[j] = __builtin_nontemporal_load((const v4i *)(h3 + r * ld3 + c));
      } else {
        a[j] = v4i{0, 0, 0, 0};
        b[j] = v4i{0, 0, 0, 0};
      }
    }
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < NCHW; ++j) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        h[j][k] = (int)gate_fwd2((uint32_t)a[j][k], (uint32_t)b[j][k]);
        m = pk_absmax_u16(m, (uint32_t)h[j][k]);
        if (COLMAX && !CLDS) cmax[j * 4 + k] = pk_absmax_u16(cmax[j * 4 + k], (uint32_t)h[j][k]);
      }
      const int c = col_of(j);
      if (CLDS && c < C) {
        v4i old = lds_cm[c / 8];
#pragma unroll
        for (int k = 0; k < 4; ++k) old[k] = (int)pk_absmax_u16((uint32_t)old[k], (uint32_t)h[j][k]);
        lds_cm[c / 8] = old;
      }
      if (hout && c < C) __builtin_nontemporal_store(h[j], (v4i *)(hout + r * ldh + c));
    }
    m = wave_max_u32(max(m & 0xffffu, m >> 16));
    if (lane == 0) red[it & 1][wave] = m;
    __syncthreads();
    uint32_t amax_bits = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) amax_bits = max(amax_bits, red[it & 1][w]);
    const RowScale rs = row_scale(amax_bits, scale_rule);
    if (threadIdx.x == 0) {
      if (scale) scale[r] = rs.s;
      if (amax_out) amax_out[r] = (uint16_t)amax_bits;
    }
    if (q) {
      uint8_t *qrow = q + r * ldq;
#pragma unroll
      for (int j = 0; j < NCHW; ++j) {
        const int c = col_of(j);
        if (c < C) {
          if (rs.finite) __builtin_nontemporal_store(cvt8(h[j], rs.recip), (v2i *)(qrow + c));
          else *(v2i *)(qrow + c) = cvt8_slow(h[j], rs.recip);
        }
      }
    }
  }
  if (COLMAX) {
#pragma unroll
    for (int j = 0; j < NCHW; ++j) {
      const int c = col_of(j);
      if (c < C)
        *(v4i *)(col_partials + (int64_t)blockIdx.x * C + c) =
            CLDS ? lds_cm[c / 8] : v4i{(int)cmax[j * 4], (int)cmax[j * 4 + 1], (int)cmax[j * 4 + 2], (int)cmax[j * 4 + 3]};
    }
  }
}

template <int NCHW, bool COLMAX, int WAVES = kGateWaves>
__global__ __launch_bounds__(WAVES * 64, WAVES == kGateWaves ? 2 : 4) void swiglu_bwd_cast_rowwise_kernel(
    const uint16_t *__restrict__ dh, const uint16_t *__restrict__ h1, const uint16_t *__restrict__ h3, int64_t R, int C,
    int64_t lddh, int64_t ld1, int64_t ld3, uint16_t *__restrict__ g1out, uint16_t *__restrict__ g3out, int64_t ldg,
    uint8_t *__restrict__ q1, uint8_t *__restrict__ q3, int64_t ldq, float *__restrict__ scale1,
    float *__restrict__ scale3, uint16_t *__restrict__ col_partials1, uint16_t *__restrict__ col_partials3, int scale_rule) {
  __shared__ uint32_t red[2][2][WAVES];
  extern __shared__ __attribute__((aligned(16))) uint8_t dyn_lds[];
  constexpr bool CLDS = COLMAX && WAVES > kGateWaves;  // column maxima in LDS instead of registers
  v4i *lds_cm1 = (v4i *)dyn_lds, *lds_cm3 = lds_cm1 + C / 8;  // [C / 8] each
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  auto col_of = [&](int j) { return (j * WAVES + wave) * 512 + lane * 8; };
  uint32_t cmax1[(COLMAX && !CLDS) ? NCHW * 4 : 1], cmax3[(COLMAX && !CLDS) ? NCHW * 4 : 1];
  if (COLMAX) {
#pragma unroll
    for (int j = 0; j < NCHW; ++j) {
      if (CLDS) {
        if (col_of(j) < C) lds_cm1[col_of(j) / 8] = lds_cm3[col_of(j) / 8] = v4i{0, 0, 0, 0};
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) cmax1[j * 4 + k] = cmax3[j * 4 + k] = 0;
      }
    }
  }
  int it = 0;
  for (int64_t r = blockIdx.x; r < R; r += gridDim.x, ++it) {
    v4i g1[NCHW], g3[NCHW];
    uint32_t m1 = 0, m3 = 0;
#pragma unroll
    for (int j = 0; j < NCHW; ++j) {
      const int c = col_of(j);
      v4i d = {0, 0, 0, 0}, a = {0, 0, 0, 0}, b = {0, 0, 0, 0};
      if (c < C) {
        d = __builtin_nontemporal_load((const v4i *)(dh + r * lddh + c));
        a = __builtin_nontemporal_load((const v4i *)(h1 + r * ld1 + c));
        b = __builtin_nontemporal_load((const v4i *)(h3 + r * ld3 + c));
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        uint32_t x1, x3;
        gate_bwd2((uint32_t)d[k], (uint32_t)a[k], (uint32_t)b[k], x1, x3);
        g1[j][k] = (int)x1;
        g3[j][k] = (int)x3;
        m1 = pk_absmax_u16(m1, x1);
        m3 = pk_absmax_u16(m3, x3);
        if (COLMAX && !CLDS) {
          cmax1[j * 4 + k] = pk_absmax_u16(cmax1[j * 4 + k], x1);
          cmax3[j * 4 + k] = pk_absmax_u16(cmax3[j * 4 + k], x3);
        }
      }
      if (CLDS && c < C) {
        v4i o1 = lds_cm1[c / 8], o3 = lds_cm3[c / 8];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          o1[k] = (int)pk_absmax_u16((uint32_t)o1[k], (uint32_t)g1[j][k]);
          o3[k] = (int)pk_absmax_u16((uint32_t)o3[k], (uint32_t)g3[j][k]);
        }
        lds_cm1[c / 8] = o1;
        lds_cm3[c / 8] = o3;
      }
      if (g1out && c < C) {
        __builtin_nontemporal_store(g1[j], (v4i *)(g1out + r * ldg + c));
        __builtin_nontemporal_store(g3[j], (v4i *)(g3out + r * ldg + c));
      }
    }
    m1 = wave_max_u32(max(m1 & 0xffffu, m1 >> 16));
    m3 = wave_max_u32(max(m3 & 0xffffu, m3 >> 16));
    if (lane == 0) {
      red[it & 1][0][wave] = m1;
      red[it & 1][1][wave] = m3;
    }
    __syncthreads();
    uint32_t bits1 = 0, bits3 = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      bits1 = max(bits1, red[it & 1][0][w]);
      bits3 = max(bits3, red[it & 1][1][w]);
    }
    const RowScale rs1 = row_scale(bits1, scale_rule), rs3 = row_scale(bits3, scale_rule);
    if (threadIdx.x == 0) {
      scale1[r] = rs1.s;
      scale3[r] = rs3.s;
    }
    uint8_t *q1row = q1 + r * ldq, *q3row = q3 + r * ldq;
#pragma unroll
    for (int j = 0; j < NCHW; ++j) {
      const int c = col_of(j);
      if (c < C) {
        if (rs1.finite) __builtin_nontemporal_store(cvt8(g1[j], rs1.recip), (v2i *)(q1row + c));
        else *(v2i *)(q1row + c) = cvt8_slow(g1[j], rs1.recip);
        if (rs3.finite) __builtin_nontemporal_store(cvt8(g3[j], rs3.recip), (v2i *)(q3row + c));
        else *(v2i *)(q3row + c) = cvt8_slow(g3[j], rs3.recip);
      }
    }
  }
  if (COLMAX) {
#pragma unroll
    for (int j = 0; j < NCHW; ++j) {
      const int c = col_of(j);
      if (c < C) {
        *(v4i *)(col_partials1 + (int64_t)blockIdx.x * C + c) =
            CLDS ? lds_cm1[c / 8] : v4i{(int)cmax1[j * 4], (int)cmax1[j * 4 + 1], (int)cmax1[j * 4 + 2], (int)cmax1[j * 4 + 3]};
        *(v4i *)(col_partials3 + (int64_t)blockIdx.x * C + c) =
            CLDS ? lds_cm3[c / 8] : v4i{(int)cmax3[j * 4], (int)cmax3[j * 4 + 1], (int)cmax3[j * 4 + 2], (int)cmax3[j * 4 + 3]};
      }
    }
  }
}

// Wide rows (beyond 16384 columns, more than a workgroup holds in registers): 1024 threads per row, two passes.  Pass 1
// computes the gate, stores the bf16 result and reduces the row amax; pass 2
// reads the thread's own bf16 values back (they are still in L2) and casts.
// Column maxima live in LDS (one bf16 per column and tensor, each owned by one
// thread).  Any C that is a multiple of 8.
constexpr int kWideBlock = 1024;
constexpr int kWideWaves = kWideBlock / 64;

template <bool COLMAX>
__global__ __launch_bounds__(kWideBlock) void swiglu_cast_rowwise_wide_kernel(
    const uint16_t *__restrict__ h1, const uint16_t *__restrict__ h3, int64_t R, int C, int64_t ld1, int64_t ld3,
    uint16_t *__restrict__ hout, int64_t ldh, uint8_t *__restrict__ q, int64_t ldq, float *__restrict__ scale,
    uint16_t *__restrict__ amax_out, uint16_t *__restrict__ col_partials, int scale_rule) {
  __shared__ uint32_t red[2][kWideWaves];
  extern __shared__ __attribute__((aligned(16))) uint8_t dyn_lds[];
  v4i *lds_cm = (v4i *)dyn_lds;  // [C / 8]
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  if (COLMAX)
    for (int c = threadIdx.x * 8; c < C; c += kWideBlock * 8) lds_cm[c / 8] = v4i{0, 0, 0, 0};
  int it = 0;
  for (int64_t r = blockIdx.x; r < R; r += gridDim.x, ++it) {
    uint32_t m = 0;
    for (int c = threadIdx.x * 8; c < C; c += kWideBlock * 8) {
      const v4i a = __builtin_nontemporal_load((const v4i *)(h1 + r * ld1 + c));
      const v4i b = __builtin_nontemporal_load((const v4i *)(h3 + r * ld3 + c));
      v4i h;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        h[k] = (int)gate_fwd2((uint32_t)a[k], (uint32_t)b[k]);
        m = pk_absmax_u16(m, (uint32_t)h[k]);
      }
      if (COLMAX) {
        v4i old = lds_cm[c / 8];
#pragma unroll
        for (int k = 0; k < 4; ++k) old[k] = (int)pk_absmax_u16((uint32_t)old[k], (uint32_t)h[k]);
        lds_cm[c / 8] = old;
      }
      if (hout) *(v4i *)(hout + r * ldh + c) = h;
    }
    m = wave_max_u32(max(m & 0xffffu, m >> 16));
    if (lane == 0) red[it & 1][wave] = m;
    __syncthreads();
    uint32_t amax_bits = 0;
#pragma unroll
    for (int w = 0; w < kWideWaves; ++w) amax_bits = max(amax_bits, red[it & 1][w]);
    const RowScale rs = row_scale(amax_bits, scale_rule);
    if (threadIdx.x == 0) {
      if (scale) scale[r] = rs.s;
      if (amax_out) amax_out[r] = (uint16_t)amax_bits;
    }
    if (q) {
      uint8_t *qrow = q + r * ldq;
      for (int c = threadIdx.x * 8; c < C; c += kWideBlock * 8) {
        v4i h;
        if (hout) {
          h = *(const v4i *)(hout + r * ldh + c);  // this thread's own store of pass 1
        } else {
          const v4i a = *(const v4i *)(h1 + r * ld1 + c);
          const v4i b = *(const v4i *)(h3 + r * ld3 + c);
#pragma unroll
          for (int k = 0; k < 4; ++k) h[k] = (int)gate_fwd2((uint32_t)a[k], (uint32_t)b[k]);
        }
        if (rs.finite) __builtin_nontemporal_store(cvt8(h, rs.recip), (v2i *)(qrow + c));
        else *(v2i *)(qrow + c) = cvt8_slow(h, rs.recip);
      }
    }
  }
  if (COLMAX)
    for (int c = threadIdx.x * 8; c < C; c += kWideBlock * 8)
      *(v4i *)(col_partials + (int64_t)blockIdx.x * C + c) = lds_cm[c / 8];
}

template <bool COLMAX>
__global__ __launch_bounds__(kWideBlock) void swiglu_bwd_cast_rowwise_wide_kernel(
    const uint16_t *__restrict__ dh, const uint16_t *__restrict__ h1, const uint16_t *__restrict__ h3, int64_t R, int C,
    int64_t lddh, int64_t ld1, int64_t ld3, uint16_t *__restrict__ g1out, uint16_t *__restrict__ g3out, int64_t ldg,
    uint8_t *__restrict__ q1, uint8_t *__restrict__ q3, int64_t ldq, float *__restrict__ scale1,
    float *__restrict__ scale3, uint16_t *__restrict__ col_partials1, uint16_t *__restrict__ col_partials3, int scale_rule) {
  __shared__ uint32_t red[2][2][kWideWaves];
  extern __shared__ __attribute__((aligned(16))) uint8_t dyn_lds[];
  v4i *lds_cm1 = (v4i *)dyn_lds, *lds_cm3 = lds_cm1 + C / 8;  // [C / 8] each
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  if (COLMAX)
    for (int c = threadIdx.x * 8; c < C; c += kWideBlock * 8) lds_cm1[c / 8] = lds_cm3[c / 8] = v4i{0, 0, 0, 0};
  int it = 0;
  for (int64_t r = blockIdx.x; r < R; r += gridDim.x, ++it) {
    uint32_t m1 = 0, m3 = 0;
    for (int c = threadIdx.x * 8; c < C; c += kWideBlock * 8) {
      const v4i d = __builtin_nontemporal_load((const v4i *)(dh + r * lddh + c));
      const v4i a = __builtin_nontemporal_load((const v4i *)(h1 + r * ld1 + c));
      const v4i b = __builtin_nontemporal_load((const v4i *)(h3 + r * ld3 + c));
      v4i g1, g3;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        uint32_t x1, x3;
        gate_bwd2((uint32_t)d[k], (uint32_t)a[k], (uint32_t)b[k], x1, x3);
        g1[k] = (int)x1;
        g3[k] = (int)x3;
        m1 = pk_absmax_u16(m1, x1);
        m3 = pk_absmax_u16(m3, x3);
      }
      if (COLMAX) {
        v4i o1 = lds_cm1[c / 8], o3 = lds_cm3[c / 8];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          o1[k] = (int)pk_absmax_u16((uint32_t)o1[k], (uint32_t)g1[k]);
          o3[k] = (int)pk_absmax_u16((uint32_t)o3[k], (uint32_t)g3[k]);
        }
        lds_cm1[c / 8] = o1;
        lds_cm3[c / 8] = o3;
      }
      *(v4i *)(g1out + r * ldg + c) = g1;
      *(v4i *)(g3out + r * ldg + c) = g3;
    }
    m1 = wave_max_u32(max(m1 & 0xffffu, m1 >> 16));
    m3 = wave_max_u32(max(m3 & 0xffffu, m3 >> 16));
    if (lane == 0) {
      red[it & 1][0][wave] = m1;
      red[it & 1][1][wave] = m3;
    }
    __syncthreads();
    uint32_t bits1 = 0, bits3 = 0;
#pragma unroll
    for (int w = 0; w < kWideWaves; ++w) {
      bits1 = max(bits1, red[it & 1][0][w]);
      bits3 = max(bits3, red[it & 1][1][w]);
    }
    const RowScale rs1 = row_scale(bits1, scale_rule), rs3 = row_scale(bits3, scale_rule);
    if (threadIdx.x == 0) {
      scale1[r] = rs1.s;
      scale3[r] = rs3.s;
    }
    uint8_t *q1row = q1 + r * ldq, *q3row = q3 + r * ldq;
    for (int c = threadIdx.x * 8; c < C; c += kWideBlock * 8) {
      const v4i g1 = *(const v4i *)(g1out + r * ldg + c);  // this thread's own stores of pass 1
      const v4i g3 = *(const v4i *)(g3out + r * ldg + c);
      if (rs1.finite) __builtin_nontemporal_store(cvt8(g1, rs1.recip), (v2i *)(q1row + c));
      else *(v2i *)(q1row + c) = cvt8_slow(g1, rs1.recip);
      if (rs3.finite) __builtin_nontemporal_store(cvt8(g3, rs3.recip), (v2i *)(q3row + c));
      else *(v2i *)(q3row + c) = cvt8_slow(g3, rs3.recip);
    }
  }
  if (COLMAX)
    for (int c = threadIdx.x * 8; c < C; c += kWideBlock * 8) {
      *(v4i *)(col_partials1 + (int64_t)blockIdx.x * C + c) = lds_cm1[c / 8];
      *(v4i *)(col_partials3 + (int64_t)blockIdx.x * C + c) = lds_cm3[c / 8];
    }
}

// The three operands of the weight gradients that come out of the gate -- its two gradients (for dW1 and dW3) and its
// output (for dW2) -- quantised per column and written transposed, from what the gate reads: dh, h1 and h3.  Bound by
// memory at 9 bytes per element (6 read, 3 written).  Casting them from stored copies reads as much and writes as
// much, but the copies have to be written first: 6 bytes per element that the row-wise kernels then need not write.
// The gate is computed a second time for that, by the same functions: the same bf16 values, hence the bounds that the
// column amaxes give hold and the bytes are those of the casts of the copies.  us, the gate's three row-wise and transposed
// passes with stored copies / without: [16384,8192] 224 + 379 / 124 + 198 + 249, the whole forward + backward with 2048 wide
// ends 2458 / 2410; [4093,14336] with 4096 wide ends 2021 / 1995.  What this kernel reaches, 4.7 to 5.3 TB/s, is a matter of
// its addresses: without the gate's arithmetic it takes as long to 2 %, without the writes to LDS as well.
//
// TC columns x (256 / (TC / 8)) * 4 * TU rows per workgroup: 64 x 128.  Workgroups walk down the rows, each row of tiles a
// column block further on, which keeps power-of-two strides from piling onto a few memory channels on either side.  us alone,
// [16384,8192] | [4093,14336] | [5000,6000]: 64 x 128 so 249 | 93 | 66, across the columns 257 | 111 | 75, 128 x 128 243 | 96 |
// 59, 64 x 256 294 | 108 | -, 128 x 64 309 | 106 | 68; inside the step 64 x 128 is ahead of 128 x 128 by 0.3 %, and streaming
// stores (222 | 100 | 66 alone) cost the step 0.5 %: the products read what they leave in the caches.  A thread turns 4 rows x 8 columns of a unit into one dword per column; the
// dwords meet in three tiles in LDS, whose 16-byte pieces stand at position (piece ^ column chunk) of their row: both
// sides then spread over the banks (a padded row stride, being a multiple of 16 bytes, leaves the writes of a wave on 8
// of 64).
struct GateTransposed {
  const uint16_t *dh, *h1, *h3;
  int64_t R, lddh, ld1, ld3;
  const float *amax[3];  // column amaxes of g1, g3 and h
  uint8_t *q[3];         // [C, Rp] each
  int64_t ldq, Rp;
  float *scale[3];
  int C, vec_store, scale_rule;
};
template <int TC, int TU>
__global__ __launch_bounds__(256) void swiglu_bwd_cast_transposed_kernel(const GateTransposed p) {
#if defined(__HIP_DEVICE_COMPILE__)  // buffer descriptors exist in the device pass only
  constexpr int kCCH = TC / 8, kRG = 256 / kCCH, kTR = kRG * 4 * TU;
  constexpr int SEGS = kTR / 16;  // 16-byte pieces per row of a tile
  static_assert((SEGS & (SEGS - 1)) == 0 && kRG % 4 == 0, "pieces are swizzled by exclusive or");
  __shared__ __attribute__((aligned(16))) uint8_t tile[3][TC * kTR];
  __shared__ __attribute__((aligned(16))) float recips[3][TC];
  const int t = threadIdx.x;
  const int C = p.C;
  const int64_t R = p.R;
  const int nct = (C + TC - 1) / TC;
  const int nrt = (int)((p.Rp + kTR - 1) / kTR);
  const int rt = (int)(blockIdx.x % (unsigned)nrt);
  const int cb = (int)((blockIdx.x / (unsigned)nrt + (unsigned)rt) % (unsigned)nct);
  const int64_t r0 = (int64_t)rt * kTR;
  const int c0 = cb * TC;
  const int cc = t % kCCH, rg = t / kCCH;  // which 8 columns; which 4 rows of a unit
  const int c = c0 + cc * 8;
  const bool live = c < C;

  // The amaxes first, the tile right behind them: loads retire in order, so the divisions run under the tile's loads.
  uint32_t bits[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.amax[k], (uint32_t)C * 4u);
    bits[k] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, (c0 + t % TC) * 4, 0, 0);  // zero beyond column C
  }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  const int64_t rows_left = R - r0;
  const int rows = rows_left <= 0 ? 0 : rows_left < kTR ? (int)rows_left : kTR;
  v4i in[3][TU][4];
  // Descriptors over the tile's rows that exist: a row at or beyond R starts beyond them, a chunk at or beyond column C is
  // sent there.  The host keeps a tile's rows below 2^30 bytes.
  auto load = [&](v4i (&dst)[TU][4], const uint16_t *x, int64_t ld) {
    const uint32_t row_bytes = (uint32_t)ld * 2u;
    const uint32_t bytes = rows ? (uint32_t)(rows - 1) * row_bytes + (uint32_t)C * 2u : 0u;
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(x + r0 * ld, bytes);
    const uint32_t voff = (live ? (uint32_t)c * 2u : bytes) + (uint32_t)(rg * 4) * row_bytes;
#pragma unroll
    for (int u = 0; u < TU; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[u][i] = load16_nt(rs, voff, (uint32_t)(u * kRG * 4 + i) * row_bytes);
  };
  load(in[0], p.dh, p.lddh);
  load(in[1], p.h1, p.ld1);
  load(in[2], p.h3, p.ld3);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float amax = __uint_as_float(bits[k]);
    const bool finite = bits[k] < 0x7f800000u;
    const float s = finite ? scale_from_amax(amax, p.scale_rule) : __uint_as_float(bits[k] == 0x7f800000u ? 0x7f800000u : 0x7fc00000u);
    const float rc = finite ? recip_exact(s) : __uint_as_float(0x7fc00000u);  // NaN: this column is redone below
    if (t < TC) {
      if (rt == 0 && c0 + t < C) p.scale[k][c0 + t] = s;
      recips[k][t] = rc;
    }
  }
  __syncthreads();
  float rcp[3][8];
  bool all_fast = true;
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      rcp[k][j] = recips[k][cc * 8 + j];
      all_fast &= rcp[k][j] == rcp[k][j];
    }
  auto at = [&](int k, int u, int j) {  // the dword of rows (u * kRG + rg) * 4 .. + 3 of column j
    const int unit = u * kRG + rg;
    return (uint32_t *)(tile[k] + (cc * 8 + j) * kTR + (((unit >> 2) ^ (cc & (SEGS - 1))) * 16) + (unit & 3) * 4);
  };
#pragma unroll
  for (int u = 0; u < TU; ++u)
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      uint32_t g[3][4];  // two columns of four rows
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t d = (uint32_t)in[0][u][i][w], a = (uint32_t)in[1][u][i][w], b = (uint32_t)in[2][u][i][w];
        gate_bwd2(d, a, b, g[0][i], g[1][i], g[2][i]);
      }
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int hi = 0; hi < 2; ++hi) {
          const int j = 2 * w + hi;
          float v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(hi ? (g[k][i] & 0xffff0000u) : (g[k][i] << 16)) * rcp[k][j];
          int packed = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false);
          packed = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], packed, true);
          *at(k, u, j) = (uint32_t)packed;
        }
    }
  if (!all_fast) {
    // A column whose amax is not finite: redone from memory with the true reciprocal (0 or NaN) and the integer conversion.
#pragma unroll 1
    for (int k = 0; k < 3; ++k)
#pragma unroll 1
      for (int uj = 0; uj < TU * 8; ++uj) {
        const int u = uj >> 3, j = uj & 7;
        const float kept = recips[k][cc * 8 + j];
        if (kept == kept || c + j >= C) continue;
        const uint32_t b = __float_as_uint(p.amax[k][c + j]);
        const float rc = recip_exact(__uint_as_float(b == 0x7f800000u ? 0x7f800000u : 0x7fc00000u));
        uint32_t packed = 0;
        for (int i = 0; i < 4; ++i) {
          const int64_t r = r0 + (u * kRG + rg) * 4 + i;
          if (r >= R) continue;
          uint32_t g[3];
          gate_bwd2(p.dh[r * p.lddh + c + j], p.h1[r * p.ld1 + c + j], p.h3[r * p.ld3 + c + j], g[0], g[1], g[2]);
          const uint32_t x = k == 0 ? g[0] : k == 1 ? g[1] : g[2];
          packed |= e4m3fn_from_f32_slow(bf16_bits_to_f32(x) * rc) << (8 * i);
        }
        *at(k, u, j) = packed;
      }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int i = 0; i < TC * SEGS / 256; ++i) {
      const int idx = i * 256 + t;
      const int oc = idx / SEGS, seg = idx % SEGS;
      const int64_t r = r0 + seg * 16;
      if (c0 + oc < C && r < p.Rp) {
        const uint8_t *src = tile[k] + oc * kTR + ((seg ^ ((oc >> 3) & (SEGS - 1))) * 16);
        uint8_t *dst = p.q[k] + (int64_t)(c0 + oc) * p.ldq + r;
        if (p.vec_store && r + 16 <= p.Rp) {
          *(v4i *)dst = *(const v4i *)src;
        } else {
          for (int b = 0; b < 16 && r + b < p.Rp; ++b) dst[b] = src[b];
        }
      }
    }
#endif
}

// workgroups (= rows of a partial-maxima array) for R rows
static int64_t gate_blocks(int64_t R) {
  const int64_t cap = (int64_t)num_cus() * 2;
  return R < cap ? R : cap;
}

// the column maxima of the wide kernels must fit LDS: 2 B (forward) or 4 B (backward) per column
constexpr int64_t kGateMaxC = 65536;
constexpr int64_t kGateBwdMaxC = 32768;
constexpr int64_t kGateBwdOnePassC = 16384;  // beyond, the second pass reads the bf16 gradients back

// dynamic LDS above the default limit needs the attribute once per device
template <typename K>
static int allow_lds(K kernel, size_t bytes, bool (&done)[kMaxDev]) {
  if (bytes <= 48 * 1024) return L8_OK;
  const int slot = device_slot();
  if (slot >= 0 && done[slot]) return L8_OK;
  L8_HIP(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 159 * 1024));
  if (slot >= 0) done[slot] = true;
  return L8_OK;
}

static int launch_fwd_wide(const void *h1, const void *h3, int64_t R, int64_t C, int64_t ld1, int64_t ld3, void *h,
                           int64_t ldh, void *q, int64_t ldq, float *scale, void *amax, float *col_amax, void *ws,
                           hipStream_t st) {
  const int64_t blocks = gate_blocks(R);
  if (col_amax) {
    static bool done[kMaxDev] = {};
    const size_t lds = (size_t)C * 2;
    const int rc = allow_lds(swiglu_cast_rowwise_wide_kernel<true>, lds, done);
    if (rc != L8_OK) return rc;
    hipLaunchKernelGGL((swiglu_cast_rowwise_wide_kernel<true>), dim3((unsigned)blocks), dim3(kWideBlock), lds, st,
                       (const uint16_t *)h1, (const uint16_t *)h3, R, (int)C, ld1, ld3, (uint16_t *)h, ldh, (uint8_t *)q, ldq,
                       scale, (uint16_t *)amax, (uint16_t *)ws, l8::scale_rule());
    L8_HIP(hipGetLastError());
    return fold_colmax(ws, blocks, C, col_amax, st);
  }
  hipLaunchKernelGGL((swiglu_cast_rowwise_wide_kernel<false>), dim3((unsigned)blocks), dim3(kWideBlock), 0, st,
                     (const uint16_t *)h1, (const uint16_t *)h3, R, (int)C, ld1, ld3, (uint16_t *)h, ldh, (uint8_t *)q, ldq,
                     scale, (uint16_t *)amax, (uint16_t *)nullptr, l8::scale_rule());
  L8_HIP(hipGetLastError());
  return L8_OK;
}

static int launch_bwd_wide(const void *dh, const void *h1, const void *h3, int64_t R, int64_t C, int64_t lddh, int64_t ld1,
                           int64_t ld3, void *g1, void *g3, int64_t ldg, void *q1, void *q3, int64_t ldq, float *s1,
                           float *s3, float *ca1, float *ca3, void *ws, hipStream_t st) {
  const int64_t blocks = gate_blocks(R);
  if (ca1) {
    static bool done[kMaxDev] = {};
    uint16_t *w1 = (uint16_t *)ws, *w3 = w1 + blocks * C;
    const size_t lds = (size_t)C * 4;
    const int rc = allow_lds(swiglu_bwd_cast_rowwise_wide_kernel<true>, lds, done);
    if (rc != L8_OK) return rc;
    hipLaunchKernelGGL((swiglu_bwd_cast_rowwise_wide_kernel<true>), dim3((unsigned)blocks), dim3(kWideBlock), lds, st,
                       (const uint16_t *)dh, (const uint16_t *)h1, (const uint16_t *)h3, R, (int)C, lddh, ld1, ld3,
                       (uint16_t *)g1, (uint16_t *)g3, ldg, (uint8_t *)q1, (uint8_t *)q3, ldq, s1, s3, w1, w3, l8::scale_rule());
    L8_HIP(hipGetLastError());
    const FoldOperand both[2] = {{w1, ca1, blocks, C}, {w3, ca3, blocks, C}};
    return fold_colmax_many(both, 2, st);
  }
  hipLaunchKernelGGL((swiglu_bwd_cast_rowwise_wide_kernel<false>), dim3((unsigned)blocks), dim3(kWideBlock), 0, st,
                     (const uint16_t *)dh, (const uint16_t *)h1, (const uint16_t *)h3, R, (int)C, lddh, ld1, ld3,
                     (uint16_t *)g1, (uint16_t *)g3, ldg, (uint8_t *)q1, (uint8_t *)q3, ldq, s1, s3, (uint16_t *)nullptr,
                     (uint16_t *)nullptr, l8::scale_rule());
  L8_HIP(hipGetLastError());
  return L8_OK;
}

template <int NCHW, int WAVES = kGateWaves>
static int launch_fwd(const void *h1, const void *h3, int64_t R, int64_t C, int64_t ld1, int64_t ld3, void *h, int64_t ldh,
                      void *q, int64_t ldq, float *scale, void *amax, float *col_amax, void *ws, hipStream_t st) {
  const int64_t blocks = gate_blocks(R);
  if (col_amax) {
    const size_t lds = (WAVES > kGateWaves) ? (size_t)C * 2 : 0;
    hipLaunchKernelGGL((swiglu_cast_rowwise_kernel<NCHW, true, WAVES>), dim3((unsigned)blocks), dim3(WAVES * 64), lds, st,
                       (const uint16_t *)h1, (const uint16_t *)h3, R, (int)C, ld1, ld3, (uint16_t *)h, ldh, (uint8_t *)q, ldq,
                       scale, (uint16_t *)amax, (uint16_t *)ws, l8::scale_rule());
    L8_HIP(hipGetLastError());
    return fold_colmax(ws, blocks, C, col_amax, st);
  }
  hipLaunchKernelGGL((swiglu_cast_rowwise_kernel<NCHW, false, WAVES>), dim3((unsigned)blocks), dim3(WAVES * 64), 0, st,
                     (const uint16_t *)h1, (const uint16_t *)h3, R, (int)C, ld1, ld3, (uint16_t *)h, ldh, (uint8_t *)q, ldq,
                     scale, (uint16_t *)amax, (uint16_t *)nullptr, l8::scale_rule());
  L8_HIP(hipGetLastError());
  return L8_OK;
}

template <int NCHW, int WAVES = kGateWaves>
static int launch_bwd(const void *dh, const void *h1, const void *h3, int64_t R, int64_t C, int64_t lddh, int64_t ld1,
                      int64_t ld3, void *g1, void *g3, int64_t ldg, void *q1, void *q3, int64_t ldq, float *s1, float *s3,
                      float *ca1, float *ca3, void *ws, hipStream_t st) {
  const int64_t blocks = gate_blocks(R);
  if (ca1) {
    uint16_t *w1 = (uint16_t *)ws, *w3 = w1 + blocks * C;
    const size_t lds = (WAVES > kGateWaves) ? (size_t)C * 4 : 0;
    if (lds > 48 * 1024) {  // above the default limit for dynamic LDS; idempotent
      static bool raised[kMaxDev] = {};
      const int slot = device_slot();
      if (slot < 0 || !raised[slot])
        L8_HIP(hipFuncSetAttribute((const void *)swiglu_bwd_cast_rowwise_kernel<NCHW, true, WAVES>, hipFuncAttributeMaxDynamicSharedMemorySize, 64 * 1024));
      if (slot >= 0) raised[slot] = true;
    }
    hipLaunchKernelGGL((swiglu_bwd_cast_rowwise_kernel<NCHW, true, WAVES>), dim3((unsigned)blocks), dim3(WAVES * 64), lds, st,
                       (const uint16_t *)dh, (const uint16_t *)h1, (const uint16_t *)h3, R, (int)C, lddh, ld1, ld3,
                       (uint16_t *)g1, (uint16_t *)g3, ldg, (uint8_t *)q1, (uint8_t *)q3, ldq, s1, s3, w1, w3, l8::scale_rule());
    L8_HIP(hipGetLastError());
    const FoldOperand both[2] = {{w1, ca1, blocks, C}, {w3, ca3, blocks, C}};
    return fold_colmax_many(both, 2, st);
  }
  hipLaunchKernelGGL((swiglu_bwd_cast_rowwise_kernel<NCHW, false, WAVES>), dim3((unsigned)blocks), dim3(WAVES * 64), 0, st,
                     (const uint16_t *)dh, (const uint16_t *)h1, (const uint16_t *)h3, R, (int)C, lddh, ld1, ld3,
                     (uint16_t *)g1, (uint16_t *)g3, ldg, (uint8_t *)q1, (uint8_t *)q3, ldq, s1, s3, (uint16_t *)nullptr,
                     (uint16_t *)nullptr, l8::scale_rule());
  L8_HIP(hipGetLastError());
  return L8_OK;
}

static bool aligned16(const void *p) { return ((uintptr_t)p % 16) == 0; }

}  // namespace l8

using namespace l8;

extern "C" int64_t l8_swiglu_workspace(int64_t R, int64_t C) {
  if (R <= 0 || C <= 0) return 0;
  return 2 * gate_blocks(R) * C * (int64_t)sizeof(uint16_t);
}

extern "C" int l8_swiglu_cast_rowwise(const void *h1, const void *h3, int64_t R, int64_t C, int64_t ld1, int64_t ld3, void *h,
                                      int64_t ldh, void *q, int64_t ldq, float *scale, void *amax, float *col_amax,
                                      void *workspace, int64_t workspace_bytes, void *stream) {
  L8_REQUIRE(R >= 0 && C >= 0, "l8_swiglu_cast_rowwise: negative shape R=%lld C=%lld", (long long)R, (long long)C);
  if (R == 0 || C == 0) return empty_col_amax(col_amax, C, (hipStream_t)stream);
  L8_REQUIRE(h1 && h3 && q && scale, "l8_swiglu_cast_rowwise: null pointer");
  L8_REQUIRE(C % 8 == 0 && ld1 % 8 == 0 && ld3 % 8 == 0 && ld1 >= C && ld3 >= C,
             "l8_swiglu_cast_rowwise: C=%lld, ld1=%lld, ld3=%lld must be multiples of 8 and ld >= C", (long long)C,
             (long long)ld1, (long long)ld3);
  L8_REQUIRE(ldq % 8 == 0 && ldq >= C, "l8_swiglu_cast_rowwise: ldq=%lld must be a multiple of 8 and >= C", (long long)ldq);
  L8_REQUIRE(!h || (ldh % 8 == 0 && ldh >= C), "l8_swiglu_cast_rowwise: ldh=%lld must be a multiple of 8 and >= C", (long long)ldh);
  L8_REQUIRE(aligned16(h1) && aligned16(h3) && (!h || aligned16(h)) && ((uintptr_t)q % 8) == 0,
             "l8_swiglu_cast_rowwise: h1, h3, h must be 16-byte aligned and q 8-byte aligned");
  L8_REQUIRE(C <= kGateMaxC, "l8_swiglu_cast_rowwise: C=%lld exceeds %lld", (long long)C, (long long)kGateMaxC);
  if (col_amax) {
    const int64_t need = l8_swiglu_workspace(R, C) / 2;
    L8_REQUIRE(workspace && workspace_bytes >= need && aligned16(workspace),
               "l8_swiglu_cast_rowwise: col_amax needs a 16-byte aligned workspace of %lld bytes", (long long)need);
  }
  hipStream_t st = (hipStream_t)stream;
  const int64_t nchw = ((C + 511) / 512 + kGateWaves - 1) / kGateWaves;
#define L8_FWD(...) return launch_fwd<__VA_ARGS__>(h1, h3, R, C, ld1, ld3, h, ldh, q, ldq, scale, amax, col_amax, workspace, st)
  if (nchw <= 1) L8_FWD(1);
  if (nchw <= 2) L8_FWD(2);
  if (nchw <= 4) L8_FWD(2, 8);
  if (nchw <= 6) L8_FWD(3, 8);
  if (nchw <= 8) L8_FWD(4, 8);
#undef L8_FWD
  return launch_fwd_wide(h1, h3, R, C, ld1, ld3, h, ldh, q, ldq, scale, amax, col_amax, workspace, st);
}

// g1 and g3 are null for a caller that does not want them (`quantised_only`).
static int swiglu_bwd(const void *dh, const void *h1, const void *h3, int64_t R, int64_t C, int64_t lddh, int64_t ld1, int64_t ld3,
                      void *g1, void *g3, int64_t ldg, void *q1, void *q3, int64_t ldq, float *scale1, float *scale3, float *col_amax1,
                      float *col_amax3, void *workspace, int64_t workspace_bytes, void *stream, bool quantised_only) {
  L8_REQUIRE(R >= 0 && C >= 0, "l8_swiglu_bwd_cast_rowwise: negative shape R=%lld C=%lld", (long long)R, (long long)C);
  if (R == 0 || C == 0) {
    const int rc = empty_col_amax(col_amax1, C, (hipStream_t)stream);
    return rc == L8_OK ? empty_col_amax(col_amax3, C, (hipStream_t)stream) : rc;
  }
  L8_REQUIRE(dh && h1 && h3 && (quantised_only || (g1 && g3)) && q1 && q3 && scale1 && scale3, "l8_swiglu_bwd_cast_rowwise: null pointer");
  L8_REQUIRE((col_amax1 == nullptr) == (col_amax3 == nullptr), "l8_swiglu_bwd_cast_rowwise: pass both column amaxes or neither");
  L8_REQUIRE(C % 8 == 0 && lddh % 8 == 0 && ld1 % 8 == 0 && ld3 % 8 == 0 && ldg % 8 == 0 && ldq % 8 == 0,
             "l8_swiglu_bwd_cast_rowwise: C and every leading dimension must be multiples of 8");
  L8_REQUIRE(lddh >= C && ld1 >= C && ld3 >= C && (quantised_only || ldg >= C) && ldq >= C, "l8_swiglu_bwd_cast_rowwise: leading dimension < C");
  L8_REQUIRE(aligned16(dh) && aligned16(h1) && aligned16(h3) && aligned16(g1) && aligned16(g3) && ((uintptr_t)q1 % 8) == 0 &&
                 ((uintptr_t)q3 % 8) == 0,
             "l8_swiglu_bwd_cast_rowwise: bf16 operands must be 16-byte aligned and q1, q3 8-byte aligned");
  const int64_t max_c = quantised_only ? kGateBwdOnePassC : kGateBwdMaxC;
  L8_REQUIRE(C <= max_c, "l8_swiglu_bwd_cast_rowwise: C=%lld exceeds %lld", (long long)C, (long long)max_c);
  if (col_amax1) {
    const int64_t need = l8_swiglu_workspace(R, C);
    L8_REQUIRE(workspace && workspace_bytes >= need && aligned16(workspace),
               "l8_swiglu_bwd_cast_rowwise: column amaxes need a 16-byte aligned workspace of %lld bytes", (long long)need);
  }
  hipStream_t st = (hipStream_t)stream;
  const int64_t nchw = ((C + 511) / 512 + kGateWaves - 1) / kGateWaves;
#define L8_BWD(...)                                                                                                      \
  return launch_bwd<__VA_ARGS__>(dh, h1, h3, R, C, lddh, ld1, ld3, g1, g3, ldg, q1, q3, ldq, scale1, scale3, col_amax1, \
                                 col_amax3, workspace, st)
  if (nchw <= 1) L8_BWD(1);
  if (nchw <= 2) L8_BWD(2);
  if (nchw <= 4) L8_BWD(2, 8);
  if (nchw <= 6) L8_BWD(3, 8);
  if (nchw <= 8) L8_BWD(2, 16);
#undef L8_BWD
  return launch_bwd_wide(dh, h1, h3, R, C, lddh, ld1, ld3, g1, g3, ldg, q1, q3, ldq, scale1, scale3, col_amax1, col_amax3,
                         workspace, st);
}

extern "C" int l8_swiglu_bwd_cast_rowwise(const void *dh, const void *h1, const void *h3, int64_t R, int64_t C, int64_t lddh,
                                          int64_t ld1, int64_t ld3, void *g1, void *g3, int64_t ldg, void *q1, void *q3,
                                          int64_t ldq, float *scale1, float *scale3, float *col_amax1, float *col_amax3,
                                          void *workspace, int64_t workspace_bytes, void *stream) {
  return swiglu_bwd(dh, h1, h3, R, C, lddh, ld1, ld3, g1, g3, ldg, q1, q3, ldq, scale1, scale3, col_amax1, col_amax3, workspace,
                    workspace_bytes, stream, false);
}

extern "C" int l8_swiglu_bwd_cast_rowwise_q(const void *dh, const void *h1, const void *h3, int64_t R, int64_t C, int64_t lddh,
                                            int64_t ld1, int64_t ld3, void *q1, void *q3, int64_t ldq, float *scale1, float *scale3,
                                            float *col_amax1, float *col_amax3, void *workspace, int64_t workspace_bytes,
                                            void *stream) {
  return swiglu_bwd(dh, h1, h3, R, C, lddh, ld1, ld3, nullptr, nullptr, 0, q1, q3, ldq, scale1, scale3, col_amax1, col_amax3,
                    workspace, workspace_bytes, stream, true);
}

extern "C" int l8_swiglu_bwd_cast_transposed(const void *dh, const void *h1, const void *h3, int64_t R, int64_t C, int64_t lddh,
                                             int64_t ld1, int64_t ld3, const float *col_amax1, const float *col_amax3,
                                             const float *col_amaxh, void *q1, void *q3, void *qh, int64_t ldq, int64_t Rp,
                                             float *scale1, float *scale3, float *scaleh, void *stream) {
  L8_REQUIRE(R >= 0 && C >= 0 && Rp >= R, "l8_swiglu_bwd_cast_transposed: bad shape R=%lld C=%lld Rp=%lld", (long long)R, (long long)C, (long long)Rp);
  if (Rp == 0 || C == 0) return L8_OK;
  L8_REQUIRE(dh && h1 && h3 && col_amax1 && col_amax3 && col_amaxh && q1 && q3 && qh && scale1 && scale3 && scaleh,
             "l8_swiglu_bwd_cast_transposed: null pointer");
  const int64_t ld_max = lddh > ld1 ? (lddh > ld3 ? lddh : ld3) : (ld1 > ld3 ? ld1 : ld3);
  L8_REQUIRE(C % 8 == 0 && lddh % 8 == 0 && ld1 % 8 == 0 && ld3 % 8 == 0 && lddh >= C && ld1 >= C && ld3 >= C && ld_max < (1LL << 21),
             "l8_swiglu_bwd_cast_transposed: C and the row strides must be multiples of 8, the strides >= C and < 2 Mi");
  L8_REQUIRE(ldq >= Rp, "l8_swiglu_bwd_cast_transposed: ldq=%lld < Rp=%lld", (long long)ldq, (long long)Rp);
  L8_REQUIRE(aligned16(dh) && aligned16(h1) && aligned16(h3), "l8_swiglu_bwd_cast_transposed: dh, h1 and h3 must be 16-byte aligned");
  GateTransposed p{(const uint16_t *)dh, (const uint16_t *)h1, (const uint16_t *)h3, R, lddh, ld1, ld3, {col_amax1, col_amax3, col_amaxh},
                   {(uint8_t *)q1, (uint8_t *)q3, (uint8_t *)qh}, ldq, Rp, {scale1, scale3, scaleh}, (int)C,
                   ldq % 16 == 0 && aligned16(q1) && aligned16(q3) && aligned16(qh), l8::scale_rule()};
  constexpr int TC = 64, TU = 1, TR = 256 / (TC / 8) * 4 * TU;
  const int64_t blocks = (C + TC - 1) / TC * ((Rp + TR - 1) / TR);
  L8_REQUIRE(C < (1LL << 30) && blocks < (1LL << 31), "l8_swiglu_bwd_cast_transposed: too large");
  hipLaunchKernelGGL((swiglu_bwd_cast_transposed_kernel<TC, TU>), dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, p);
  L8_HIP(hipGetLastError());
  return L8_OK;
}
