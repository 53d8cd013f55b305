// RMSNorm fused with the row-wise fp8 cast of its output.
//
// The blocks of the model normalise the residual stream and hand the result to
// wq / wk / wv or w1 / w3 (lingua/transformer.py:283-289 for the norm,
// :357-359 and :469-471 for the consumers).  Eagerly that is seven elementwise
// / reduction kernels with fp32 temporaries for the norm, then one pass of the
// row-wise cast per consuming linear (lingua/float8.py:86-87, :43-47).  Here the
// row is read once, normalised, written as bf16 (autograd and the wgrad casts
// need it) and quantised from registers:
//
//   r  = rsqrt(mean(f32(x)^2) + eps)
//   y  = bf16( (f32(x) * r) * f32(w) )            (the reference's op order)
//   q, scale = row-wise cast of y, [rstd = r], [column amaxes of y]
//
// Everything after r is exact elementwise arithmetic; r itself depends on the
// order of the fp32 sum of squares, which differs from ATen's reduction, so y
// can differ from the eager result in the last bf16 bit of an element now and
// then (the tests bound it: at most one bf16 ulp, > 99.5 % identical).
// Two layouts, as in the row-wise casts: a wavefront per row for short rows, a
// 256-thread workgroup per row for the longer ones; both add a row up in the same
// order, so a row's result does not hang on the layout.
#include "l8_common.h"

namespace l8 {

constexpr int kNormBlock = 256;
constexpr int kNormWaves = kNormBlock / 64;

// sum over the 64 lanes of a wave, result uniform
L8_DEV float wave_sum_f32(float v) {
  auto step = [&](int moved) { v += __int_as_float(moved); };
  step(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));   // quad_perm [1,0,3,2]
  step(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true));   // quad_perm [2,3,0,1]
  step(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xF, 0xF, true));  // row_ror:4
  step(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, true));  // row_ror:8
  const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
  const float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
  const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
  const float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
  return (a + b) + (c + d);
}

// The weights of a lane's columns, kept in registers for all rows it sees: packed pairs as they are in memory (bf16),
// or one register each (fp32).  Zero beyond column C.
template <int N, bool W_F32>
struct NormWeights {
  uint32_t reg[N * (W_F32 ? 8 : 4)];
  template <typename ColOf>
  L8_DEV void load(const void *w, int C, ColOf col_of) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int c = col_of(j);
#pragma unroll
      for (int e = 0; e < (W_F32 ? 8 : 4); ++e) {
        uint32_t v = 0;
        // a bf16 weight may start at any even address: the copy states two-byte alignment
        if (c < C) {
          if (W_F32) v = ((const uint32_t *)w)[c + e];
          else __builtin_memcpy(&v, (const uint16_t *)w + c + 2 * e, 4);
        }
        reg[j * (W_F32 ? 8 : 4) + e] = v;
      }
    }
  }
  L8_DEV float get(int j, int e) const {
    if (W_F32) return __uint_as_float(reg[j * 8 + e]);
    const uint32_t p = reg[j * 4 + (e >> 1)];
    return __uint_as_float((e & 1) ? (p & 0xffff0000u) : (p << 16));
  }
};

#if defined(__HIP_DEVICE_COMPILE__)
// row r of x; zeros beyond column C and for a row at or beyond R (no branch around a load)
template <int N, typename ColOf>
L8_DEV void load_norm_row(v4i (&buf)[N], const uint16_t *x, int64_t r, int64_t R, int64_t ldx, int C, ColOf col_of) {
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(x + (r < R ? r : 0) * ldx, r < R ? (uint32_t)C * 2u : 0u);
#pragma unroll
  for (int j = 0; j < N; ++j) buf[j] = load16_nt(rs, (uint32_t)col_of(j) * 2u, 0);
}
L8_DEV void store16_nt(__amdgpu_buffer_rsrc_t rs, uint32_t voff, v4i data) {
  __builtin_amdgcn_raw_buffer_store_b128(data, rs, (int)voff, 0, 2 /* non-temporal */);
}
L8_DEV void store8_nt(__amdgpu_buffer_rsrc_t rs, uint32_t voff, v2i data) {
  __builtin_amdgcn_raw_buffer_store_b64(data, rs, (int)voff, 0, 2 /* non-temporal */);
}
#endif

// Short rows (C <= NCH * 512): one wavefront owns a row, so neither the sum of squares nor the row amax crosses waves
// and there is no barrier; the next row is requested before the current one is touched (loads through descriptors
// without branches, as in the row-wise cast).  HBM-bound: 5 bytes per element.
template <int NCH, bool COLMAX, bool W_F32>
__global__ __launch_bounds__(kNormBlock, 2) void rmsnorm_cast_rowwise_wave_kernel(
    const uint16_t *__restrict__ x, const void *__restrict__ w, int64_t R, int C, int64_t ldx, float eps,
    uint16_t *__restrict__ y, int64_t ldy, uint8_t *__restrict__ q, int64_t ldq, float *__restrict__ scale,
    float *__restrict__ rstd, uint16_t *__restrict__ col_partials, int scale_rule) {
#if defined(__HIP_DEVICE_COMPILE__)  // buffer descriptors exist in the device pass only
  extern __shared__ __attribute__((aligned(16))) uint8_t dyn_lds[];  // [C] bf16 when COLMAX
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto col_of = [&](int j) { return j * 512 + lane * 8; };
  uint32_t cmax[COLMAX ? NCH * 4 : 1];
  if (COLMAX) {
#pragma unroll
    for (int i = 0; i < NCH * 4; ++i) cmax[i] = 0;
  }
  NormWeights<NCH, W_F32> wt;
  wt.load(w, C, [&](int j) { return col_of(j); });
  const float inv_c = 1.0f / (float)C;
  const int64_t stride = (int64_t)gridDim.x * kNormWaves;
  int64_t r = (int64_t)blockIdx.x * kNormWaves + wave;
  v4i cur[NCH], nxt[NCH];
  load_norm_row<NCH>(cur, x, r, R, ldx, C, [&](int j) { return col_of(j); });
  while (r < R) {
    const int64_t rn = r + stride;
    load_norm_row<NCH>(nxt, x, rn, R, ldx, C, [&](int j) { return col_of(j); });
    // each chunk of 512 columns is summed for itself and the chunks are added in order, as the waves of a workgroup that
    // shares a row add theirs: one order of summation, hence one result, in both layouts
    float tot = 0.0f;
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
      float ss = 0.0f;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float lo = __uint_as_float((uint32_t)cur[j][k] << 16), hi = __uint_as_float((uint32_t)cur[j][k] & 0xffff0000u);
        ss += lo * lo;
        ss += hi * hi;
      }
      tot += wave_sum_f32(ss);
    }
    const float rinv = 1.0f / sqrtf(tot * inv_c + eps);
    const __amdgpu_buffer_rsrc_t rsY = make_rsrc(y + r * ldy, (uint32_t)C * 2u);
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
      v4i yv;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float lo = __uint_as_float((uint32_t)cur[j][k] << 16), hi = __uint_as_float((uint32_t)cur[j][k] & 0xffff0000u);
        const uint32_t ylo = bf16_rne_bits((lo * rinv) * wt.get(j, 2 * k));
        const uint32_t yhi = bf16_rne_bits((hi * rinv) * wt.get(j, 2 * k + 1));
        yv[k] = (int)(ylo | (yhi << 16));
        m = pk_absmax_u16(m, (uint32_t)yv[k]);
        if (COLMAX) cmax[j * 4 + k] = pk_absmax_u16(cmax[j * 4 + k], (uint32_t)yv[k]);
      }
      store16_nt(rsY, (uint32_t)col_of(j) * 2u, yv);
      cur[j] = yv;  // the row of y replaces the row of x in registers
    }
    const uint32_t amax_bits = wave_max_u32(max(m & 0xffffu, m >> 16));
    const RowScale rs = row_scale(amax_bits, scale_rule);
    if (lane == 0) {
      if (rstd) rstd[r] = rinv;
      if (scale) scale[r] = rs.s;
    }
    const __amdgpu_buffer_rsrc_t rsQ = make_rsrc(q ? q + r * ldq : nullptr, q ? (uint32_t)C : 0u);
#pragma unroll
    for (int j = 0; j < NCH; ++j) store8_nt(rsQ, (uint32_t)col_of(j), cvt8(cur[j], rs.recip));
    if (q && !rs.finite) {  // a non-finite amax: the bytes are redone from this lane's own y with the integer conversion
      asm volatile("" ::: "memory");
#pragma unroll 1
      for (int c = lane * 8; c < C; c += 512) *(v2i *)(q + r * ldq + c) = cvt8_slow(*(const v4i *)(y + r * ldy + c), rs.recip);
    }
#pragma unroll
    for (int j = 0; j < NCH; ++j) cur[j] = nxt[j];
    r = rn;
  }
  if (COLMAX) {  // the waves' column maxima meet in LDS, one wave after the other, and leave as this workgroup's row
    v4i *lds4 = (v4i *)dyn_lds;
    for (int wv = 0; wv < kNormWaves; ++wv) {
      if (wave == wv) {
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
          const int c = col_of(j);
          if (c < C) {
            v4i mine = {(int)cmax[j * 4], (int)cmax[j * 4 + 1], (int)cmax[j * 4 + 2], (int)cmax[j * 4 + 3]};
            if (wv > 0) {
              const v4i old = lds4[c / 8];
#pragma unroll
              for (int k = 0; k < 4; ++k) mine[k] = (int)pk_absmax_u16((uint32_t)old[k], (uint32_t)mine[k]);
            }
            if (wv == kNormWaves - 1) *(v4i *)(col_partials + (int64_t)blockIdx.x * C + c) = mine;
            else lds4[c / 8] = mine;
          }
        }
      }
      __syncthreads();
    }
  }
#endif
}

// Longer rows: one workgroup per row (a wave-per-row kernel would need more than 256 registers), the next row requested
// ahead of the two barriers of the current one.
template <int NCHW, bool COLMAX, bool W_F32>
__global__ __launch_bounds__(kNormBlock, 2) void rmsnorm_cast_rowwise_kernel(
    const uint16_t *__restrict__ x, const void *__restrict__ w, int64_t R, int C, int64_t ldx, float eps,
    uint16_t *__restrict__ y, int64_t ldy, uint8_t *__restrict__ q, int64_t ldq, float *__restrict__ scale,
    float *__restrict__ rstd, uint16_t *__restrict__ col_partials, int scale_rule) {
#if defined(__HIP_DEVICE_COMPILE__)  // buffer descriptors exist in the device pass only
  __shared__ float red_ss[2][kNormWaves];
  __shared__ uint32_t red_mx[2][kNormWaves];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  auto col_of = [&](int j) { return (j * kNormWaves + wave) * 512 + lane * 8; };
  uint32_t cmax[COLMAX ? NCHW * 4 : 1];
  if (COLMAX) {
#pragma unroll
    for (int i = 0; i < NCHW * 4; ++i) cmax[i] = 0;
  }
  NormWeights<NCHW, W_F32> wt;  // of this thread's columns, in registers for all its rows
  wt.load(w, C, [&](int j) { return col_of(j); });
  const float inv_c = 1.0f / (float)C;
  v4i cur[NCHW], nxt[NCHW];
  load_norm_row<NCHW>(cur, x, blockIdx.x, R, ldx, C, [&](int j) { return col_of(j); });
  int it = 0;
  for (int64_t r = blockIdx.x; r < R; r += gridDim.x, ++it) {
    load_norm_row<NCHW>(nxt, x, r + gridDim.x, R, ldx, C, [&](int j) { return col_of(j); });
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < NCHW; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float lo = __uint_as_float((uint32_t)cur[j][k] << 16), hi = __uint_as_float((uint32_t)cur[j][k] & 0xffff0000u);
        ss += lo * lo;
        ss += hi * hi;
      }
    ss = wave_sum_f32(ss);
    if (lane == 0) red_ss[it & 1][wave] = ss;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int wv = 0; wv < kNormWaves; ++wv) tot += red_ss[it & 1][wv];
    const float rinv = 1.0f / sqrtf(tot * inv_c + eps);
    if (threadIdx.x == 0 && rstd) rstd[r] = rinv;

    const __amdgpu_buffer_rsrc_t rsY = make_rsrc(y + r * ldy, (uint32_t)C * 2u);
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < NCHW; ++j) {
      v4i yv;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float lo = __uint_as_float((uint32_t)cur[j][k] << 16), hi = __uint_as_float((uint32_t)cur[j][k] & 0xffff0000u);
        const uint32_t ylo = bf16_rne_bits((lo * rinv) * wt.get(j, 2 * k));
        const uint32_t yhi = bf16_rne_bits((hi * rinv) * wt.get(j, 2 * k + 1));
        yv[k] = (int)(ylo | (yhi << 16));
        m = pk_absmax_u16(m, (uint32_t)yv[k]);
        if (COLMAX) cmax[j * 4 + k] = pk_absmax_u16(cmax[j * 4 + k], (uint32_t)yv[k]);
      }
      store16_nt(rsY, (uint32_t)col_of(j) * 2u, yv);
      cur[j] = yv;  // the row of y replaces the row of x in registers
    }
    m = wave_max_u32(max(m & 0xffffu, m >> 16));
    if (lane == 0) red_mx[it & 1][wave] = m;
    __syncthreads();
    uint32_t amax_bits = 0;
#pragma unroll
    for (int wv = 0; wv < kNormWaves; ++wv) amax_bits = max(amax_bits, red_mx[it & 1][wv]);
    const RowScale rs = row_scale(amax_bits, scale_rule);
    if (threadIdx.x == 0 && scale) scale[r] = rs.s;
    const __amdgpu_buffer_rsrc_t rsQ = make_rsrc(q ? q + r * ldq : nullptr, q ? (uint32_t)C : 0u);
#pragma unroll
    for (int j = 0; j < NCHW; ++j) store8_nt(rsQ, (uint32_t)col_of(j), cvt8(cur[j], rs.recip));
    if (q && !rs.finite) {  // as in the kernel above: redone from this thread's own y
      asm volatile("" ::: "memory");
#pragma unroll 1
      for (int c = threadIdx.x * 8; c < C; c += kNormBlock * 8)
        *(v2i *)(q + r * ldq + c) = cvt8_slow(*(const v4i *)(y + r * ldy + c), rs.recip);
    }
#pragma unroll
    for (int j = 0; j < NCHW; ++j) cur[j] = nxt[j];
  }
  if (COLMAX) {
#pragma unroll
    for (int j = 0; j < NCHW; ++j) {
      const int c = col_of(j);
      if (c < C)
        *(v4i *)(col_partials + (int64_t)blockIdx.x * C + c) =
            v4i{(int)cmax[j * 4], (int)cmax[j * 4 + 1], (int)cmax[j * 4 + 2], (int)cmax[j * 4 + 3]};
    }
  }
#endif
}

// Backward of the norm: with xhat = x * r and gh = gy * w,
//   gx = (gh - xhat * mean(gh * xhat)) * r        (bf16)
//   gw = sum over rows of gy * xhat               (fp32)
// One workgroup per row, also for short rows; the row products for gw are
// accumulated in registers over all rows a workgroup sees and leave as one row
// of fp32 partial sums per workgroup, which rmsnorm_gw_fold_kernel adds up column
// by column.  Which rows meet in a partial sum, and the order of every sum, hang
// on the number of rows alone (no atomics: the result does not depend on timing).
// Rows are requested AHEAD - 1 rows before they are used: a row of one chunk per
// lane (up to 2048 columns) is too few bytes in flight for one row ahead.
template <int NCHW, int AHEAD, bool W_F32>
__global__ __launch_bounds__(kNormBlock, 2) void rmsnorm_bwd_kernel(
    const uint16_t *__restrict__ gy, const uint16_t *__restrict__ x, const void *__restrict__ w,
    const float *__restrict__ rstd, int64_t R, int C, int64_t ldg, int64_t ldx, uint16_t *__restrict__ gx, int64_t ldgx,
    float *__restrict__ gw_partials) {
#if defined(__HIP_DEVICE_COMPILE__)
  static_assert(AHEAD % 2 == 0, "a buffer meets the same half of `red` every time");
  __shared__ float red[2][kNormWaves];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  auto col_of = [&](int j) { return (j * kNormWaves + wave) * 512 + lane * 8; };
  NormWeights<NCHW, W_F32> wt;
  wt.load(w, C, [&](int j) { return col_of(j); });
  float gwacc[NCHW][8];
#pragma unroll
  for (int j = 0; j < NCHW; ++j)
#pragma unroll
    for (int e = 0; e < 8; ++e) gwacc[j][e] = 0.0f;
  const float inv_c = 1.0f / (float)C;
  v4i xb[AHEAD][NCHW], gb[AHEAD][NCHW];
  float rb[AHEAD];
  auto request = [&](int a, int64_t r) {  // a row beyond R: zeros, nothing is read
    rb[a] = rstd[r < R ? r : 0];
    load_norm_row<NCHW>(xb[a], x, r, R, ldx, C, [&](int j) { return col_of(j); });
    load_norm_row<NCHW>(gb[a], gy, r, R, ldg, C, [&](int j) { return col_of(j); });
  };
#pragma unroll
  for (int a = 0; a < AHEAD - 1; ++a) request(a, blockIdx.x + a * (int64_t)gridDim.x);
  for (int64_t r0 = blockIdx.x; r0 < R; r0 += (int64_t)AHEAD * gridDim.x) {
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) {
      const int64_t r = r0 + a * (int64_t)gridDim.x;
      if (r >= R) break;  // the same for the whole workgroup
      request((a + AHEAD - 1) % AHEAD, r + (AHEAD - 1) * (int64_t)gridDim.x);
      const v4i(&xc)[NCHW] = xb[a], (&gc)[NCHW] = gb[a];
      const float rinv = rb[a];
      auto xhat = [&](int j, int e) {
        const uint32_t p = (uint32_t)xc[j][e >> 1];
        return __uint_as_float((e & 1) ? (p & 0xffff0000u) : (p << 16)) * rinv;
      };
      auto grad = [&](int j, int e) {
        const uint32_t p = (uint32_t)gc[j][e >> 1];
        return __uint_as_float((e & 1) ? (p & 0xffff0000u) : (p << 16));
      };
      float dot = 0.0f;
#pragma unroll
      for (int j = 0; j < NCHW; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float ge = grad(j, e), xh = xhat(j, e);
          gwacc[j][e] += ge * xh;
          dot += (ge * wt.get(j, e)) * xh;
        }
      dot = wave_sum_f32(dot);
      if (lane == 0) red[a & 1][wave] = dot;
      __syncthreads();
      float tot = 0.0f;
#pragma unroll
      for (int wv = 0; wv < kNormWaves; ++wv) tot += red[a & 1][wv];
      const float c1 = tot * inv_c;
      const __amdgpu_buffer_rsrc_t rsG = make_rsrc(gx + r * ldgx, (uint32_t)C * 2u);
#pragma unroll
      for (int j = 0; j < NCHW; ++j) {
        v4i out;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint32_t lo = bf16_rne_bits((grad(j, 2 * k) * wt.get(j, 2 * k) - xhat(j, 2 * k) * c1) * rinv);
          const uint32_t hi = bf16_rne_bits((grad(j, 2 * k + 1) * wt.get(j, 2 * k + 1) - xhat(j, 2 * k + 1) * c1) * rinv);
          out[k] = (int)(lo | (hi << 16));
        }
        store16_nt(rsG, (uint32_t)col_of(j) * 2u, out);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NCHW; ++j) {
    const int c = col_of(j);
    if (c < C) {
      float *dst = gw_partials + (int64_t)blockIdx.x * C + c;
      *(v4f *)dst = v4f{gwacc[j][0], gwacc[j][1], gwacc[j][2], gwacc[j][3]};
      *(v4f *)(dst + 4) = v4f{gwacc[j][4], gwacc[j][5], gwacc[j][6], gwacc[j][7]};
    }
  }
#endif
}

// gw[c] = sum over the partial rows: eight sums of every eighth row, each in the order of the rows, added in order.
// A workgroup owns 32 columns -- one 128-byte line of every partial row -- and passes them through LDS, 256 rows at a
// time: 16 bytes per thread and load, the next 256 rows in flight under the additions, which come one after the other
// but read LDS.  (With each addition waiting for its row from memory the fold of 512 rows of 2048 columns took 20 us.)
// gw leaves as fp32 or, for a bf16 weight, rounded: a conversion of its own was a launch of 4 to 5 us for a few KiB.
constexpr int kGwCols = 32, kGwThreads = 1024, kGwRows = 256, kGwSums = 8;
__global__ __launch_bounds__(kGwThreads) void rmsnorm_gw_fold_kernel(const float *__restrict__ partials, int n_slots, int C,
                                                                     void *__restrict__ gw, int gw_f32) {
  constexpr int QUADS = kGwCols / 4, STEP = kGwThreads / QUADS, LOADS = kGwRows / STEP;  // threads to a row, rows to a load
  __shared__ v4f rows[kGwRows][QUADS];
  __shared__ float sums[kGwSums][kGwCols];
  const int quad = threadIdx.x % QUADS, row = threadIdx.x / QUADS;
  const int tx = threadIdx.x % kGwCols, ty = threadIdx.x / kGwCols;
  const int col = blockIdx.x * kGwCols + quad * 4;
  v4f part[LOADS];
  auto request = [&](int s0) {  // without a branch around a load: a row beyond the last is the last again
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int sl = s0 + i * STEP + row;
      part[i] = *(const v4f *)(partials + (int64_t)(sl < n_slots ? sl : n_slots - 1) * C + (col < C ? col : 0));
    }
  };
  if (n_slots > 0) request(0);
  float s = 0.0f;
  for (int s0 = 0; s0 < n_slots; s0 += kGwRows) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) rows[i * STEP + row][quad] = part[i];
    __syncthreads();
    if (s0 + kGwRows < n_slots) request(s0 + kGwRows);
    if (ty < kGwSums) {
      const int n = n_slots - s0 < kGwRows ? n_slots - s0 : kGwRows;
#pragma unroll 8
      for (int sl = ty; sl < n; sl += kGwSums) s += reinterpret_cast<const float *>(&rows[sl][0])[tx];
    }
    __syncthreads();
  }
  if (ty < kGwSums) sums[ty][tx] = s;
  __syncthreads();
  const int c = blockIdx.x * kGwCols + tx;
  if (ty == 0 && c < C) {
    float t = sums[0][tx];
#pragma unroll
    for (int k = 1; k < kGwSums; ++k) t += sums[k][tx];
    if (gw_f32) ((float *)gw)[c] = t;
    else ((uint16_t *)gw)[c] = (uint16_t)bf16_rne_bits(t);
  }
}

static int64_t norm_blocks(int64_t R) {
  const int64_t cap = (int64_t)num_cus() * 2;
  return R < cap ? R : cap;
}

constexpr int64_t kNormMaxC = 4 * kNormWaves * 512;  // 8192: the weights of a thread's columns live in registers

// Which layout, forward: a wavefront per row up to 2048 columns, a workgroup per row beyond (up to 8192), where a wave's
// row, the row requested ahead, the weights and the column maxima no longer fit 256 registers.  Inside a 1B-sized step,
// [16384,2048], us: 59 (a workgroup per row, each row requested when its turn comes) -> 49 (next row requested ahead) ->
// 34 (a wavefront per row: 168 MB at 4.9 TB/s); [4093,4096], workgroup per row with the next row ahead: 25.5 -> 20.5.
// With no more rows than two per compute unit every row has a workgroup of its own, whose four waves share it: [1,2048]
// 2.8 -> 2.5, [64,2048] 3.5 -> 3.0, [512,2048] 3.8 -> 3.5, but [768,2048] 4.1 / 4.3 and [2048,2048] 5.5 / 7.5; with
// column maxima and their fold, of as many partial rows, 6.1 -> 4.7, 6.6 -> 5.2, 7.3 -> 7.1, 7.8 / 7.9, 9.9 / 11.3.
// Backward: a workgroup per row, whose share of gw is a sum over rows 2 x (compute units) apart, on its own, back to
// back, us: [16384,2048] 46.2 (no row ahead) -> 35.5 (three ahead: 201 MB at 5.7 TB/s; a wavefront per row the same),
// [8192,1024] 20.3 -> 15.8, [64,2048] 4.3 -> 3.8, [4093,4096] 23.7 -> 21.8 (one ahead); the fold of gw 17 to 22 -> 4.
// Four workgroups per compute unit instead of two: forward +-4 %, backward 7 % slower.
// workgroups of the wavefront-per-row kernel (never more than norm_blocks(R), which the workspaces are sized for)
static int64_t norm_wave_blocks(int64_t R) { return norm_blocks((R + kNormWaves - 1) / kNormWaves); }

// N = chunks of 512 columns per wave (WAVE) or of 2048 per workgroup
template <bool WAVE, int N, bool W_F32>
static int launch_norm(const void *x, const void *w, int64_t R, int64_t C, int64_t ldx, float eps, void *y, int64_t ldy,
                       void *q, int64_t ldq, float *scale, float *rstd, float *col_amax, void *ws, hipStream_t st) {
  const int64_t blocks = WAVE ? norm_wave_blocks(R) : norm_blocks(R);
  auto go = [&](auto kernel, size_t lds) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kNormBlock), lds, st, (const uint16_t *)x, w, R, (int)C, ldx, eps,
                       (uint16_t *)y, ldy, (uint8_t *)q, ldq, scale, rstd, (uint16_t *)ws, l8::scale_rule());
  };
  if constexpr (WAVE) {
    if (col_amax) go(rmsnorm_cast_rowwise_wave_kernel<N, true, W_F32>, (size_t)C * 2);
    else go(rmsnorm_cast_rowwise_wave_kernel<N, false, W_F32>, 0);
  } else {
    if (col_amax) go(rmsnorm_cast_rowwise_kernel<N, true, W_F32>, 0);
    else go(rmsnorm_cast_rowwise_kernel<N, false, W_F32>, 0);
  }
  L8_HIP(hipGetLastError());
  return col_amax ? fold_colmax(ws, blocks, C, col_amax, st) : L8_OK;
}

template <int N, bool W_F32>
static int launch_norm_bwd(const void *gy, const void *x, const void *w, const float *rstd, int64_t R, int64_t C,
                           int64_t ldg, int64_t ldx, void *gx, int64_t ldgx, void *gw, int gw_f32, void *ws, hipStream_t st) {
  const int64_t blocks = norm_blocks(R);
  hipLaunchKernelGGL((rmsnorm_bwd_kernel<N, N == 1 ? 4 : 2, W_F32>), dim3((unsigned)blocks), dim3(kNormBlock), 0, st, (const uint16_t *)gy,
                     (const uint16_t *)x, w, rstd, R, (int)C, ldg, ldx, (uint16_t *)gx, ldgx, (float *)ws);
  L8_HIP(hipGetLastError());
  hipLaunchKernelGGL(rmsnorm_gw_fold_kernel, dim3((unsigned)((C + kGwCols - 1) / kGwCols)), dim3(kGwThreads), 0, st,
                     (const float *)ws, (int)blocks, (int)C, gw, gw_f32);
  L8_HIP(hipGetLastError());
  return L8_OK;
}

}  // namespace l8

using namespace l8;

extern "C" int64_t l8_rmsnorm_bwd_workspace(int64_t R, int64_t C) {
  if (R <= 0 || C <= 0) return 0;
  return norm_blocks(R) * C * (int64_t)sizeof(float);
}

extern "C" int l8_rmsnorm_bwd(const void *gy, const void *x, const void *w, int w_is_f32, const float *rstd, int64_t R,
                              int64_t C, int64_t ldg, int64_t ldx, void *gx, int64_t ldgx, float *gw, void *workspace,
                              int64_t workspace_bytes, void *stream) {
  return l8_rmsnorm_bwd_as(gy, x, w, w_is_f32, rstd, R, C, ldg, ldx, gx, ldgx, gw, 1, workspace, workspace_bytes, stream);
}

extern "C" int l8_rmsnorm_bwd_as(const void *gy, const void *x, const void *w, int w_is_f32, const float *rstd, int64_t R,
                                 int64_t C, int64_t ldg, int64_t ldx, void *gx, int64_t ldgx, void *gw, int gw_is_f32, void *workspace,
                                 int64_t workspace_bytes, void *stream) {
  L8_REQUIRE(R >= 0 && C >= 0, "l8_rmsnorm_bwd: negative shape R=%lld C=%lld", (long long)R, (long long)C);
  if (C == 0) return L8_OK;
  L8_REQUIRE(gw, "l8_rmsnorm_bwd: null pointer");
  if (R == 0) {  // no rows: gw = 0, written by the fold kernel over zero partial rows
    hipLaunchKernelGGL(rmsnorm_gw_fold_kernel, dim3((unsigned)((C + kGwCols - 1) / kGwCols)), dim3(kGwThreads), 0, (hipStream_t)stream,
                       (const float *)nullptr, 0, (int)C, gw, gw_is_f32);
    L8_HIP(hipGetLastError());
    return L8_OK;
  }
  L8_REQUIRE(gy && x && w && rstd && gx, "l8_rmsnorm_bwd: null pointer");
  L8_REQUIRE(C % 8 == 0 && ldg % 8 == 0 && ldx % 8 == 0 && ldgx % 8 == 0 && ldg >= C && ldx >= C && ldgx >= C,
             "l8_rmsnorm_bwd: C=%lld and the leading dimensions must be multiples of 8 with ld >= C", (long long)C);
  L8_REQUIRE(((uintptr_t)gy % 16) == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)gx % 16) == 0,
             "l8_rmsnorm_bwd: gy, x and gx must be 16-byte aligned");
  L8_REQUIRE(C <= kNormMaxC, "l8_rmsnorm_bwd: C=%lld exceeds %lld", (long long)C, (long long)kNormMaxC);
  const int64_t need = l8_rmsnorm_bwd_workspace(R, C);
  L8_REQUIRE(workspace && workspace_bytes >= need && ((uintptr_t)workspace % 16) == 0,
             "l8_rmsnorm_bwd: needs a 16-byte aligned workspace of %lld bytes", (long long)need);
  hipStream_t st = (hipStream_t)stream;
#define L8_NORM_BWD(N)                                                                                               \
  return w_is_f32 ? launch_norm_bwd<N, true>(gy, x, w, rstd, R, C, ldg, ldx, gx, ldgx, gw, gw_is_f32, workspace, st)  \
                  : launch_norm_bwd<N, false>(gy, x, w, rstd, R, C, ldg, ldx, gx, ldgx, gw, gw_is_f32, workspace, st)
  const int64_t nchw = ((C + 511) / 512 + kNormWaves - 1) / kNormWaves;
  if (nchw <= 1) L8_NORM_BWD(1);
  if (nchw <= 2) L8_NORM_BWD(2);
  L8_NORM_BWD(4);
#undef L8_NORM_BWD
}

extern "C" int64_t l8_rmsnorm_workspace(int64_t R, int64_t C) {
  if (R <= 0 || C <= 0) return 0;
  return norm_blocks(R) * C * (int64_t)sizeof(uint16_t);
}

extern "C" int l8_rmsnorm_cast_rowwise(const void *x, const void *w, int w_is_f32, int64_t R, int64_t C, int64_t ldx, float eps,
                                       void *y, int64_t ldy, void *q, int64_t ldq, float *scale, float *rstd,
                                       float *col_amax, void *workspace, int64_t workspace_bytes, void *stream) {
  L8_REQUIRE(R >= 0 && C >= 0, "l8_rmsnorm_cast_rowwise: negative shape R=%lld C=%lld", (long long)R, (long long)C);
  if (R == 0 || C == 0) return empty_col_amax(col_amax, C, (hipStream_t)stream);
  L8_REQUIRE(x && w && y, "l8_rmsnorm_cast_rowwise: null pointer");
  L8_REQUIRE((q == nullptr) == (scale == nullptr), "l8_rmsnorm_cast_rowwise: pass q and scale together");
  L8_REQUIRE(C % 8 == 0 && ldx % 8 == 0 && ldy % 8 == 0 && ldx >= C && ldy >= C && (!q || (ldq % 8 == 0 && ldq >= C)),
             "l8_rmsnorm_cast_rowwise: C=%lld and the leading dimensions must be multiples of 8 with ld >= C", (long long)C);
  L8_REQUIRE(((uintptr_t)x % 16) == 0 && ((uintptr_t)y % 16) == 0 && ((uintptr_t)q % 8) == 0,
             "l8_rmsnorm_cast_rowwise: x and y must be 16-byte aligned and q 8-byte aligned");
  L8_REQUIRE(C <= kNormMaxC, "l8_rmsnorm_cast_rowwise: C=%lld exceeds %lld", (long long)C, (long long)kNormMaxC);
  L8_REQUIRE(!col_amax || q, "l8_rmsnorm_cast_rowwise: column amaxes come with the cast");
  if (col_amax) {
    const int64_t need = l8_rmsnorm_workspace(R, C);
    L8_REQUIRE(workspace && workspace_bytes >= need && ((uintptr_t)workspace % 16) == 0,
               "l8_rmsnorm_cast_rowwise: col_amax needs a 16-byte aligned workspace of %lld bytes", (long long)need);
  }
  hipStream_t st = (hipStream_t)stream;
#define L8_NORM(WAVE, N)                                                                                                        \
  return w_is_f32 ? launch_norm<WAVE, N, true>(x, w, R, C, ldx, eps, y, ldy, q, ldq, scale, rstd, col_amax, workspace, st)      \
                  : launch_norm<WAVE, N, false>(x, w, R, C, ldx, eps, y, ldy, q, ldq, scale, rstd, col_amax, workspace, st)
  const int64_t nch = (C + 511) / 512, nchw = (nch + kNormWaves - 1) / kNormWaves;
  if (nch <= 4 && R > norm_blocks(R)) L8_NORM(true, 4);
  if (nchw <= 1) L8_NORM(false, 1);
  if (nchw <= 2) L8_NORM(false, 2);
  L8_NORM(false, 4);
#undef L8_NORM
}
