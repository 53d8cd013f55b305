// Fused amax -> fp32 scale -> e4m3fn cast kernels for gfx950 (HBM-bound).
//
// Replaces the eager ATen chain of lingua/float8.py:43-47 (scale()), the row
// amax reductions at :86-87 / :112-114, the tensor amax at :115-118 and the
// weight transpose copy at :111.  Compulsory traffic per element is 2 bytes
// read + 1 byte written; every kernel here reads each input byte from HBM once.
#include <atomic>
#include <mutex>
#include <type_traits>

#include "l8_common.h"

namespace l8 {

// ---------------------------------------------------------------------------
// Row-wise: one wavefront owns one row at a time and keeps it in registers
// between the amax reduction and the cast.  Lane l of chunk j holds columns
// [j*512 + l*8, +8) (one 16-byte load, 1 KiB per wave instruction).
// A workgroup is 4 waves; waves stride over rows so that the optional
// column-amax by-product is accumulated in registers over many rows, merged
// once per workgroup in LDS and written as one row of a partial-maxima array
// that a small second kernel folds into the caller's column amaxes (overwriting them).
// ---------------------------------------------------------------------------
constexpr int kRowBlock = 256;
constexpr int kRowWaves = kRowBlock / 64;

// Row r of x into NCH register quadruples per lane, through a descriptor over the row: a chunk at or beyond column C
// returns zeros, and so does every chunk of a row at or beyond R (a descriptor of no bytes), so there is no branch
// around a load and the compiler's count of outstanding loads stays exact -- which is what lets a wave wait for the
// current row while the next one is still in flight.
#if defined(__HIP_DEVICE_COMPILE__)
template <int NCH>
L8_DEV void load_row(v4i (&buf)[NCH], const uint16_t *x, int64_t r, int64_t R, int64_t ldx, int C, int lane) {
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(x + (r < R ? r : 0) * ldx, r < R ? (uint32_t)C * 2u : 0u);
#pragma unroll
  for (int j = 0; j < NCH; ++j) buf[j] = load16_nt(rs, (uint32_t)(j * 512 + lane * 8) * 2u, 0);
}
#endif

// Several operands of one width as one list of rows: row r of the launch is row r - first of the operand that holds it.
// What a linear quantises together (activation and weight, the weights of projections that share an input) takes one
// launch, whose rows are in flight together, instead of one per operand that each fill and drain the chip.  us, one by one /
// together: [4096,2048] and [2048,2048] 6.6 + 6.2 / 10.9, [333,2048] and [8192,2048] 3.5 + 13.8 / 13.4, three [2048,2048]
// weights 5.2 + 4.9 + 4.9 / 9.0.
constexpr int kMaxRowOperands = 3;
constexpr int64_t kMaxRowwiseManyColumns = 8 * 4 * 512;  // eight chunks per lane of a workgroup
struct RowOperand {
  const uint16_t *x;
  int64_t first, ldx;  // first row in the list; the operands are in order
  uint8_t *q;
  int64_t ldq;
  float *scale;
  uint16_t *amax;
};
struct RowOperands {
  RowOperand op[kMaxRowOperands];  // unused ones start beyond the last row
};
#if defined(__HIP_DEVICE_COMPILE__)
L8_DEV RowOperand operand_of(const RowOperands &list, int64_t r) {
  RowOperand o = list.op[0];
#pragma unroll
  for (int i = 1; i < kMaxRowOperands; ++i) {  // member by member: a copy of the whole would live in scratch memory
    const RowOperand &t = list.op[i];
    const bool here = r >= t.first;
    o.x = here ? t.x : o.x;
    o.first = here ? t.first : o.first;
    o.ldx = here ? t.ldx : o.ldx;
    o.q = here ? t.q : o.q;
    o.ldq = here ? t.ldq : o.ldq;
    o.scale = here ? t.scale : o.scale;
    o.amax = here ? t.amax : o.amax;
  }
  return o;
}
#endif

// With column maxima a workgroup collects them of one operand, so each operand has workgroups of its own, in proportion to
// its rows: what one launch leaves in partial rows is then shared out, where each of several launches leaves as many.  us,
// one by one / together, with the folds (one each / one): three [16384,2048] 69.3 / 54.5 (5.5 TB/s), [16384,4096] 114 / 101,
// [4096,4096] 48.8 / 31.4, [1021,2048] 19.3 / 8.8, two [300,2048] 11.8 / 6.5; an activation and a weight without column maxima
// [1021,2048] and [2048,2048] 15.9 / 13.8, [4096,2048] and [2048,2048] 21.0 / 17.7, [16384,4096] and [11008,4096] 59.4 / 56.7.
struct RowGroup {
  const uint16_t *x;
  int64_t R, ldx;
  uint8_t *q;
  int64_t ldq;
  float *scale;
  uint16_t *amax, *partials;  // either may be null
  int first, blocks;          // its workgroups; the operands are in order, unused ones start beyond the last
};
struct RowGroups {
  RowGroup op[kMaxRowOperands];
};

// MANY without column maxima: the operands come from `list`, R counts the rows of all of them and x .. amax_out are not used.
// With them: everything but C comes from `list`.
template <bool COLMAX, bool MANY>
using RowList = std::conditional_t<MANY, std::conditional_t<COLMAX, RowGroups, RowOperands>, int>;
template <int NCH, bool COLMAX, bool MANY_OPERANDS = false>
__global__ __launch_bounds__(kRowBlock, 2) void cast_rowwise_kernel(
    const uint16_t *__restrict__ x, int64_t R, int C, int64_t ldx, uint8_t *__restrict__ q, int64_t ldq,
    float *__restrict__ scale, uint16_t *__restrict__ amax_out, uint16_t *__restrict__ col_partials, int scale_rule,
    const RowList<COLMAX, MANY_OPERANDS> list) {
#if defined(__HIP_DEVICE_COMPILE__)  // buffer descriptors exist in the device pass only
  constexpr bool GROUPS = MANY_OPERANDS && COLMAX, MANY = MANY_OPERANDS && !COLMAX;
  int block = blockIdx.x, blocks = gridDim.x;
  if constexpr (GROUPS) {
    int which = 0;
#pragma unroll
    for (int i = 1; i < kMaxRowOperands; ++i) which += block >= list.op[i].first ? 1 : 0;
    const RowGroup &op = list.op[which];
    x = op.x, R = op.R, ldx = op.ldx, q = op.q, ldq = op.ldq, scale = op.scale, amax_out = op.amax, col_partials = op.partials;
    block -= op.first, blocks = op.blocks;
  }
  extern __shared__ uint32_t lds_colmax[];  // [C/2] packed bf16 pairs when COLMAX
  // the next row is prefetched into a second register set unless that would
  // push the wave beyond 256 VGPRs (two waves per SIMD are worth more)
  constexpr bool PREFETCH = COLMAX ? (NCH <= 8) : (NCH <= 24);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // in a scalar register: the row descriptors hang on it
  const int64_t wave_stride = (int64_t)blocks * kRowWaves;
  int64_t r = (int64_t)block * kRowWaves + wave;
  auto load = [&](auto &buf, int64_t row) {
    constexpr int N = sizeof(buf) / sizeof(buf[0]);
    if constexpr (MANY) {
      const RowOperand op = operand_of(list, row);
      load_row<N>(buf, op.x - op.first * op.ldx, row, R, op.ldx, C, lane);
    } else {
      load_row<N>(buf, x, row, R, ldx, C, lane);
    }
  };

  uint32_t cmax[COLMAX ? NCH * 4 : 1];
  if (COLMAX) {
#pragma unroll
    for (int i = 0; i < NCH * 4; ++i) cmax[i] = 0;
  }

  v4i cur[NCH];
  load(cur, r);
  while (r < R) {
    const int64_t rn = r + wave_stride;
    v4i nxt[PREFETCH ? NCH : 1];
    if (PREFETCH) load(nxt, rn);

    // row amax on packed pairs
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < NCH; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        m = pk_absmax_u16(m, (uint32_t)cur[j][k]);
        if (COLMAX) cmax[j * 4 + k] = pk_absmax_u16(cmax[j * 4 + k], (uint32_t)cur[j][k]);
      }
    m = max(m & 0xffffu, m >> 16);
    const uint32_t amax_bits = wave_max_u32(m);  // bf16 bits, uniform
    const bool finite = amax_bits < 0x7f80u;
    float s;
    if (finite) {
      s = scale_from_amax(bf16_bits_to_f32(amax_bits), scale_rule);
    } else if (amax_bits == 0x7f80u) {
      s = __uint_as_float(0x7f800000u);  // inf / 448
    } else {
      s = __uint_as_float(0x7fc00000u);  // NaN amax -> NaN scale
    }
    const float recip = recip_exact(s);
    const uint16_t *xrow = x + r * ldx;
    uint8_t *qrow = q ? q + r * ldq : nullptr;
    if constexpr (MANY) {
      const RowOperand cur_op = operand_of(list, r);
      const int64_t ro = r - cur_op.first;
      xrow = cur_op.x + ro * cur_op.ldx;
      qrow = cur_op.q + ro * cur_op.ldq;
      if (lane == 0) {
        cur_op.scale[ro] = s;
        if (cur_op.amax) cur_op.amax[ro] = (uint16_t)amax_bits;
      }
    } else if (lane == 0) {
      if (scale) scale[r] = s;
      if (amax_out) amax_out[r] = (uint16_t)amax_bits;
    }
    const __amdgpu_buffer_rsrc_t rsQ = make_rsrc(qrow, MANY || q ? (uint32_t)C : 0u);  // stores beyond column C, or without q, are dropped
#pragma unroll
    for (int j = 0; j < NCH; ++j) store8(rsQ, (uint32_t)(j * 512 + lane * 8), cvt8(cur[j], recip));
    if ((MANY || q) && !finite) {
      // a row with a non-finite amax: redone from memory with the integer conversion, replacing the bytes above (one
      // small loop beside the common path instead of NCH unrolled copies of that conversion inside it)
#pragma unroll 1
      for (int c = lane * 8; c < C; c += 512) *(v2i *)(qrow + c) = cvt8_slow(*(const v4i *)(xrow + c), recip);
    }
    if (PREFETCH) {
#pragma unroll
      for (int j = 0; j < NCH; ++j) cur[j] = nxt[PREFETCH ? j : 0];
    } else {
      __builtin_amdgcn_sched_barrier(0);  // the row registers are reused: do not start the loads early
      load(cur, rn);
    }
    r = rn;
  }

  if (COLMAX && (!GROUPS || col_partials)) {
    // merge the four waves' column maxima through LDS, one wave after the other
    // (packed pairs, plain reads and writes), then write this workgroup's row of
    // the partial-maxima array; a second small kernel folds the rows.  (Global
    // atomics from every workgroup cost more than the cast itself.)
    v4i *lds4 = (v4i *)lds_colmax;
    for (int w = 0; w < kRowWaves; ++w) {
      if (wave == w) {
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
          const int c = j * 512 + lane * 8;
          if (c < C) {
            v4i mine = {(int)cmax[j * 4], (int)cmax[j * 4 + 1], (int)cmax[j * 4 + 2], (int)cmax[j * 4 + 3]};
            if (w > 0) {
              const v4i old = lds4[c / 8];
#pragma unroll
              for (int k = 0; k < 4; ++k) mine[k] = (int)pk_absmax_u16((uint32_t)old[k], (uint32_t)mine[k]);
            }
            if (w == kRowWaves - 1) *(v4i *)(col_partials + (int64_t)block * C + c) = mine;
            else lds4[c / 8] = mine;
          }
        }
      }
      __syncthreads();
    }
  }
#endif
}

// Long rows: the four waves of a workgroup share one row (wave w owns chunks
// w, w+4, w+8, ... of 512 columns), so a lane holds at most NCHW chunks and
// many workgroups fit a CU.  The row amax crosses waves through LDS with one
// barrier per row (double-buffered).  Column maxima of different waves cover
// disjoint columns and are merged into the global array directly.
template <int NCHW, bool COLMAX, bool MANY = false>
__global__ __launch_bounds__(kRowBlock, (NCHW <= 4 ? 4 : (NCHW <= 8 ? 2 : 1))) void cast_rowwise_wg_kernel(
    const uint16_t *__restrict__ x, int64_t R, int C, int64_t ldx, uint8_t *__restrict__ q, int64_t ldq,
    float *__restrict__ scale, uint16_t *__restrict__ amax_out, uint16_t *__restrict__ col_partials, int scale_rule,
    const std::conditional_t<MANY, RowOperands, int> list) {
#if defined(__HIP_DEVICE_COMPILE__)  // buffer descriptors exist in the device pass only
  __shared__ uint32_t red[2][kRowWaves];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  auto col_of = [&](int j) { return (j * kRowWaves + wave) * 512 + lane * 8; };
  auto load = [&](v4i (&buf)[NCHW], int64_t r) {  // zeros beyond column C and for a row beyond R, as in load_row
    const uint16_t *row = x + (r < R ? r : 0) * ldx;
    if constexpr (MANY) {
      const RowOperand op = operand_of(list, r);
      row = op.x + (r < R ? r - op.first : 0) * op.ldx;
    }
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(row, r < R ? (uint32_t)C * 2u : 0u);
#pragma unroll
    for (int j = 0; j < NCHW; ++j) buf[j] = load16_nt(rs, (uint32_t)col_of(j) * 2u, 0);
  };
  uint32_t cmax[COLMAX ? NCHW * 4 : 1];
  if (COLMAX) {
#pragma unroll
    for (int i = 0; i < NCHW * 4; ++i) cmax[i] = 0;
  }
  int64_t r = blockIdx.x;
  v4i cur[NCHW], nxt[NCHW];
  load(cur, r);
  for (int it = 0; r < R; ++it) {
    const int64_t rn = r + gridDim.x;
    load(nxt, rn);
    // Both rows are waited for here, the next one too.  Letting the next row's loads run on under the arithmetic and
    // the stores (the compiler's own wait would be vmcnt(NCHW)) measured 5 % slower on [16384,11008] when the input
    // had just been written by the kernel before (95.3 against 90.6 us), and no faster on a cold one.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < NCHW; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        m = pk_absmax_u16(m, (uint32_t)cur[j][k]);
        if (COLMAX) cmax[j * 4 + k] = pk_absmax_u16(cmax[j * 4 + k], (uint32_t)cur[j][k]);
      }
    m = wave_max_u32(max(m & 0xffffu, m >> 16));
    if (lane == 0) red[it & 1][wave] = m;
    __syncthreads();
    uint32_t amax_bits = 0;
#pragma unroll
    for (int w = 0; w < kRowWaves; ++w) amax_bits = max(amax_bits, red[it & 1][w]);
    const bool finite = amax_bits < 0x7f80u;
    float s;
    if (finite) s = scale_from_amax(bf16_bits_to_f32(amax_bits), scale_rule);
    else s = __uint_as_float(amax_bits == 0x7f80u ? 0x7f800000u : 0x7fc00000u);
    const float recip = recip_exact(s);
    const uint16_t *xrow = x + r * ldx;
    uint8_t *qrow = q ? q + r * ldq : nullptr;
    if constexpr (MANY) {
      const RowOperand cur_op = operand_of(list, r);
      const int64_t ro = r - cur_op.first;
      xrow = cur_op.x + ro * cur_op.ldx;
      qrow = cur_op.q + ro * cur_op.ldq;
      if (threadIdx.x == 0) {
        cur_op.scale[ro] = s;
        if (cur_op.amax) cur_op.amax[ro] = (uint16_t)amax_bits;
      }
    } else if (threadIdx.x == 0) {
      if (scale) scale[r] = s;
      if (amax_out) amax_out[r] = (uint16_t)amax_bits;
    }
    const __amdgpu_buffer_rsrc_t rsQ = make_rsrc(qrow, MANY || q ? (uint32_t)C : 0u);  // stores beyond column C, or without q, are dropped
#pragma unroll
    for (int j = 0; j < NCHW; ++j) store8(rsQ, (uint32_t)col_of(j), cvt8(cur[j], recip));
    if ((MANY || q) && !finite) {  // non-finite amax: redone from memory with the integer conversion, as in cast_rowwise_kernel
#pragma unroll 1
      for (int c = threadIdx.x * 8; c < C; c += kRowBlock * 8)
        *(v2i *)(qrow + c) = cvt8_slow(*(const v4i *)(xrow + c), recip);
    }
#pragma unroll
    for (int j = 0; j < NCHW; ++j) cur[j] = nxt[j];
    r = rn;
  }
  if (COLMAX) {
    // the four waves own disjoint columns: together they write this workgroup's
    // row of the partial-maxima array
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

// Folds the partial column maxima [n_slots, C] (bf16, one row per workgroup of a row-wise kernel) into
// col_amax[C] (fp32 bit patterns), which is overwritten.  A workgroup owns 64 columns -- one 128-byte line of
// every partial row -- and its 1024 threads read 16 bytes each from 128 rows at a time, so that a fold of a few
// hundred rows is two to four loads per thread, all in flight at once (the kernel is pure latency: a few MB
// read by a launch that lasts microseconds); the 128 row groups then meet in LDS.  One launch, no atomics,
// nothing to zero beforehand.
constexpr int kFoldCols = 64, kFoldThreads = 1024, kFoldRowGroups = kFoldThreads / 8;
// Tensors that are folded together (row y of the grid is one) share the launch: the fold of one is microseconds of latency
// on a few workgroups.  us, casts with their folds, one by one / together: four [16384,2048] 92.2 / 85.0, four [3290,1392]
// 42.7 / 34.2, [493,4832] and two [493,6784] 33.1 / 25.3.
struct FoldOperands {
  FoldOperand op[kMaxFolds];
};
__global__ __launch_bounds__(kFoldThreads) void colmax_fold_kernel(const FoldOperands list) {
  const FoldOperand &o = list.op[blockIdx.y];
  const uint16_t *__restrict__ partials = (const uint16_t *)o.partials;
  uint32_t *__restrict__ col_amax = (uint32_t *)o.col_amax;
  const int n_slots = (int)o.slots, C = (int)o.C;
  if ((int)blockIdx.x * kFoldCols >= C) return;
  __shared__ v4i red[kFoldRowGroups][8];
  __shared__ uint32_t red2[8][32];
  const int cc = threadIdx.x & 7;   // which 8 columns (16 bytes) of the 64
  const int sg = threadIdx.x >> 3;  // row group
  const int col = blockIdx.x * kFoldCols + cc * 8;
  v4i m = {0, 0, 0, 0};
  if (col < C) {
#pragma unroll 4
    for (int sl = sg; sl < n_slots; sl += kFoldRowGroups) {
      const v4i v = __builtin_nontemporal_load((const v4i *)(partials + (int64_t)sl * C + col));
#pragma unroll
      for (int k = 0; k < 4; ++k) m[k] = (int)pk_absmax_u16((uint32_t)m[k], (uint32_t)v[k]);
    }
  }
  red[sg][cc] = m;
  __syncthreads();
  if (threadIdx.x < 256) {
    const int pair = threadIdx.x & 31, part = threadIdx.x >> 5;  // 32 column pairs x 8 parts of 16 row groups
    uint32_t mm = 0;
#pragma unroll
    for (int g = 0; g < kFoldRowGroups / 8; ++g)
      mm = pk_absmax_u16(mm, reinterpret_cast<const uint32_t *>(&red[part * (kFoldRowGroups / 8) + g][0])[pair]);
    red2[part][pair] = mm;
  }
  __syncthreads();
  if (threadIdx.x < 32) {
    uint32_t mm = 0;
#pragma unroll
    for (int part = 0; part < 8; ++part) mm = pk_absmax_u16(mm, red2[part][threadIdx.x]);
    const int c = blockIdx.x * kFoldCols + threadIdx.x * 2;
    if (c < C) {
      col_amax[c] = (mm & 0xffffu) << 16;  // bf16 -> fp32 bit patterns
      col_amax[c + 1] = mm & 0xffff0000u;
    }
  }
}

// Zero fill for the two kernels that merge into col_amax with atomics (a kernel, not a memset, so that
// a caller may capture the sequence in a graph).
__global__ __launch_bounds__(256) void zero_u32_kernel(uint32_t *__restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0;
}

// Fallback for rows too long to keep in registers: two passes over the row by
// one workgroup (the second pass hits L2).
__global__ __launch_bounds__(kRowBlock) void cast_rowwise_long_kernel(
    const uint16_t *__restrict__ x, int64_t R, int C, int64_t ldx, uint8_t *__restrict__ q, int64_t ldq,
    float *__restrict__ scale, uint16_t *__restrict__ amax_out, uint32_t *__restrict__ col_amax, int scale_rule) {
  __shared__ uint32_t red[kRowWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int64_t r = blockIdx.x; r < R; r += gridDim.x) {
    const uint16_t *row = x + r * ldx;
    uint32_t m = 0;
    for (int c = threadIdx.x * 8; c < C; c += kRowBlock * 8) {
      const v4i v = *(const v4i *)(row + c);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        m = pk_absmax_u16(m, (uint32_t)v[k]);
        if (col_amax) {
          const uint32_t a = (uint32_t)v[k] & 0x7fff7fffu;
          if (a & 0xffffu) atomicMax(&col_amax[c + 2 * k], (a & 0xffffu) << 16);
          if (a >> 16) atomicMax(&col_amax[c + 2 * k + 1], a & 0xffff0000u);
        }
      }
    }
    m = wave_max_u32(max(m & 0xffffu, m >> 16));
    __syncthreads();
    if (lane == 0) red[wave] = m;
    __syncthreads();
    uint32_t amax_bits = 0;
#pragma unroll
    for (int w = 0; w < kRowWaves; ++w) amax_bits = max(amax_bits, red[w]);
    float s;
    if (amax_bits < 0x7f80u) s = scale_from_amax(bf16_bits_to_f32(amax_bits), scale_rule);
    else s = __uint_as_float(amax_bits == 0x7f80u ? 0x7f800000u : 0x7fc00000u);
    const float recip = recip_exact(s);
    if (threadIdx.x == 0) {
      if (scale) scale[r] = s;
      if (amax_out) amax_out[r] = (uint16_t)amax_bits;
    }
    if (q) {
      uint8_t *qrow = q + r * ldq;
      const bool finite = amax_bits < 0x7f80u;
      for (int c = threadIdx.x * 8; c < C; c += kRowBlock * 8) {
        const v4i v = *(const v4i *)(row + c);
        *(v2i *)(qrow + c) = finite ? cvt8(v, recip) : cvt8_slow(v, recip);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Column amax alone: each lane owns 8 columns and walks down a slab of rows.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void col_amax_kernel(const uint16_t *__restrict__ x, int64_t R, int C,
                                                       int64_t ldx, int rows_per_block,
                                                       uint32_t *__restrict__ col_amax) {
  const int c = (blockIdx.x * 256 + threadIdx.x) * 8;
  if (c >= C) return;
  const int64_t r0 = (int64_t)blockIdx.y * rows_per_block;
  const int64_t r1 = (r0 + rows_per_block < R) ? r0 + rows_per_block : R;
  uint32_t m[4] = {0, 0, 0, 0};
  for (int64_t r = r0; r < r1; ++r) {
    const v4i v = __builtin_nontemporal_load((const v4i *)(x + r * ldx + c));
#pragma unroll
    for (int k = 0; k < 4; ++k) m[k] = pk_absmax_u16(m[k], (uint32_t)v[k]);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (m[k] & 0xffffu) atomicMax(&col_amax[c + 2 * k], (m[k] & 0xffffu) << 16);
    if (m[k] >> 16) atomicMax(&col_amax[c + 2 * k + 1], m[k] & 0xffff0000u);
  }
}

// ---------------------------------------------------------------------------
// Column sums of bf16 x (the bias gradient, lingua/float8.py:127), in fp32, rounded to bf16 once.  Bound by memory from a few
// thousand rows on, by latency below: a workgroup owns 128 columns -- two lines of every row, which 64 columns read at the same
// rate up to 4096 columns and 10 % slower beyond, and 256 half as fast at [16384,2048] -- and a slab of rows, read 16 at a time
// with eight loads in flight per thread.  Slabs until there are four workgroups per unit, one per 128 rows begun at most and of
// equal heights; several slabs leave fp32 partial sums that the second kernel adds in their order.  The order of every sum
// hangs on the shape and the number of compute units.  us, PyTorch's sum / this, back to back: [4096,4096] 19.8 / 9.4,
// [5580,12176] 369 / 33, [16384,2048] 28 / 16, [16384,11008] 69 / 68 (a copy's rate: 64).
//
// Up to 2048 rows one launch whose workgroups own 32 columns and every row: a unit takes in some 40 bytes per clock, so what
// counts is how many of them read.  us, from HBM, slabs (of 1024 rows, then; one launch up to there) / 128 columns per workgroup
// of 1024 threads / 64 / 32: [400,4096] 4.7 / 4.6 / 3.6 / 3.3, [1021,2048] 7.7 / 7.0 / 6.0 / 4.1, [1021,4096] 11.1 / 10.8 / 9.1 /
// 6.2, [1801,2048] 10.3 / 12.3 / 9.1 / 8.1, [1801,11040] 13.3 / 15.4 / 11.6 / 12.1; [3000,4096] 12.1 / 20.6 / 15.0 / 13.2.
// ---------------------------------------------------------------------------
constexpr int kSumCols = 128, kSumThreads = 256, kWholeCols = 32;
constexpr int64_t kSumWhole = 2048;
__global__ __launch_bounds__(kSumThreads) void col_sum_kernel(const uint16_t *__restrict__ x, int64_t R, int C, int64_t ldx,
                                                          int64_t slab, float *__restrict__ partials, uint16_t *__restrict__ out) {
  constexpr int kSumRows = kSumThreads / (kSumCols / 8);
  __shared__ float sums[kSumRows][kSumCols + 1];
  const int cc = threadIdx.x % (kSumCols / 8), rg = threadIdx.x / (kSumCols / 8);
  const int col = blockIdx.x * kSumCols + cc * 8;
  const int64_t r1 = ((int64_t)blockIdx.y + 1) * slab < R ? ((int64_t)blockIdx.y + 1) * slab : R;
  float s[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  if (col < C) {
    const uint16_t *at = x + col;
#pragma unroll 8
    for (int64_t r = (int64_t)blockIdx.y * slab + rg; r < r1; r += kSumRows) {
      const v4i v = *(const v4i *)(at + r * ldx);
#pragma unroll
      for (int e = 0; e < 8; ++e) s[e] += __uint_as_float((e & 1) ? ((uint32_t)v[e >> 1] & 0xffff0000u) : ((uint32_t)v[e >> 1] << 16));
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) sums[rg][cc * 8 + e] = s[e];
  __syncthreads();
  if (threadIdx.x >= kSumCols) return;
  float t = sums[0][threadIdx.x];
#pragma unroll
  for (int k = 1; k < kSumRows; ++k) t += sums[k][threadIdx.x];
  const int c = blockIdx.x * kSumCols + threadIdx.x;
  if (c >= C) return;
  if (out) out[c] = (uint16_t)bf16_rne_bits(t);
  else partials[(int64_t)blockIdx.y * C + c] = t;
}
__global__ __launch_bounds__(256) void col_sum_fold_kernel(const float *__restrict__ partials, int slabs, int C, uint16_t *__restrict__ out) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= C) return;
  float t = 0.0f;
#pragma unroll 8
  for (int s = 0; s < slabs; ++s) t += partials[(int64_t)s * C + c];
  out[c] = (uint16_t)bf16_rne_bits(t);
}

// Sums of all rows of COLS columns by one workgroup, the same bits for every number of threads and columns: row r belongs to group
// r % 256, eight groups to a part.  Workgroup `block` of n; those of one XCD take neighbouring columns (64 bytes of a row are
// half a line).
constexpr int kWholeGroups = 256, kWholeParts = kWholeGroups / 8;
template <int THREADS, int COLS>
struct WholeSums {
  float groups[THREADS / (COLS / 8)][COLS + 1];
  float parts[kWholeParts][COLS];
};
template <int THREADS, int COLS>
L8_DEV void sum_columns(const uint16_t *__restrict__ x, int64_t R, int C, int64_t ldx, uint16_t *__restrict__ out, int block, int n, WholeSums<THREADS, COLS> &lds) {
  constexpr int kLanes = COLS / 8, kHeld = THREADS / kLanes, kPasses = kWholeGroups / kHeld;  // groups of rows that the threads hold at once
  const int t = threadIdx.x, xcd = block & 7, loc = block >> 3;
  const int c0 = ((n >> 3) * xcd + (xcd < (n & 7) ? xcd : n & 7) + loc) * COLS;
  const int cc = t % kLanes, col = c0 + cc * 8;
  float s[kPasses][8] = {};
  if (kPasses == 1 && col < C) {
#pragma unroll 8
    for (int64_t r = t / kLanes; r < R; r += kWholeGroups) {
      const v4i v = *(const v4i *)(x + r * ldx + col);
#pragma unroll
      for (int e = 0; e < 8; ++e) s[0][e] += __uint_as_float((e & 1) ? ((uint32_t)v[e >> 1] & 0xffff0000u) : ((uint32_t)v[e >> 1] << 16));
    }
  } else if (col < C) {
    // eight rows are requested together, without branches; beyond the last one they are that one again, and count as zeros
    constexpr int kBatch = 8 / kPasses;
    for (int64_t r0 = t / kLanes; r0 - t / kLanes < R; r0 += kBatch * kWholeGroups) {
      v4i v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int64_t r = r0 + (i / kPasses) * kWholeGroups + (i % kPasses) * kHeld;
        v[i] = *(const v4i *)(x + (r < R ? r : R - 1) * ldx + col);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const bool in = r0 + (i / kPasses) * kWholeGroups + (i % kPasses) * kHeld < R;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t w = in ? (uint32_t)v[i][e >> 1] : 0u;
          s[i % kPasses][e] += __uint_as_float((e & 1) ? w & 0xffff0000u : w << 16);
        }
      }
    }
  }
  const int c = t % COLS, part = t / COLS;
  float sum = 0.0f;
#pragma unroll
  for (int j = 0; j < kPasses; ++j) {
    if (j) __syncthreads();
#pragma unroll
    for (int e = 0; e < 8; ++e) lds.groups[t / kLanes][cc * 8 + e] = s[j][e];
    __syncthreads();
    float u = lds.groups[part * 8][c];
#pragma unroll
    for (int k = 1; k < 8; ++k) u += lds.groups[part * 8 + k][c];
    lds.parts[j * (THREADS / COLS) + part][c] = u;
    if (j == 0) sum = u;
  }
  __syncthreads();
  if (part > 0 || c0 + c >= C) return;
#pragma unroll
  for (int k = 1; k < kWholeParts; ++k) sum += lds.parts[k][c];
  out[c0 + c] = (uint16_t)bf16_rne_bits(sum);
}
__global__ __launch_bounds__(1024) void col_sum_whole_kernel(const uint16_t *__restrict__ x, int64_t R, int C, int64_t ldx, uint16_t *__restrict__ out) {
  __shared__ WholeSums<1024, kWholeCols> lds;
  sum_columns<1024, kWholeCols>(x, R, C, ldx, out, blockIdx.x, gridDim.x, lds);
}

// bf16 amax[n] -> bf16 amax_out[1]; one workgroup of 1024 threads.
// Bound by latencies: sixteen bytes per lane and load where the list is aligned, one round trip up to 32768 values.  us, two
// bytes per load / sixteen: 4691 values 2.1 / 2.05, 16384 3.0 / 2.0, 28465 4.2 / 2.25.
__global__ __launch_bounds__(1024) void amax_reduce_kernel(const uint16_t *__restrict__ amax, int64_t n,
                                                           uint16_t *__restrict__ out) {
  __shared__ uint32_t red[16];
  uint32_t m = 0;
  int64_t done = 0;
  if (((uintptr_t)amax & 15) == 0) {
    done = n / 8 * 8;
    uint32_t pk = 0;
#pragma unroll 4
    for (int64_t i = threadIdx.x; i < n / 8; i += 1024) {
      const v4i v = ((const v4i *)amax)[i];
#pragma unroll
      for (int k = 0; k < 4; ++k) pk = pk_absmax_u16(pk, (uint32_t)v[k]);
    }
    m = max(pk & 0xffffu, pk >> 16);
  }
  for (int64_t i = done + threadIdx.x; i < n; i += 1024) m = max(m, (uint32_t)(amax[i] & 0x7fffu));
  m = wave_max_u32(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x < 64) {
    m = wave_max_u32(threadIdx.x < 16 ? red[threadIdx.x] : 0u);
    if (threadIdx.x == 0) out[0] = (uint16_t)m;
  }
}

// ---------------------------------------------------------------------------
// Tensor-wise, same layout out as in: pure streaming.
// ---------------------------------------------------------------------------
L8_DEV float scale_from_amax_bits16(uint32_t amax_bits, int scale_rule) {
  if (amax_bits < 0x7f80u) return scale_from_amax(bf16_bits_to_f32(amax_bits), scale_rule);
  return __uint_as_float(amax_bits == 0x7f80u ? 0x7f800000u : 0x7fc00000u);
}
L8_DEV float scale_from_amax_bits32(uint32_t amax_bits, int scale_rule) {  // fp32 bit pattern of a non-negative amax
  if (amax_bits < 0x7f800000u) return scale_from_amax(__uint_as_float(amax_bits), scale_rule);
  return __uint_as_float(amax_bits == 0x7f800000u ? 0x7f800000u : 0x7fc00000u);
}

// A device-resident amax scalar, bf16 or fp32 (sign ignored): its scale, and whether it is finite.
L8_DEV float scale_from_amax_scalar(const void *amax, int amax_f32, bool &finite, int scale_rule) {
  if (amax_f32) {
    const uint32_t bits = *(const uint32_t *)amax & 0x7fffffffu;
    finite = bits < 0x7f800000u;
    return scale_from_amax_bits32(bits, scale_rule);
  }
  const uint32_t bits = *(const uint16_t *)amax & 0x7fffu;
  finite = bits < 0x7f80u;
  return scale_from_amax_bits16(bits, scale_rule);
}

__global__ __launch_bounds__(256) void cast_tensorwise_kernel(const uint16_t *__restrict__ x, int64_t R, int C,
                                                              int64_t ldx, const void *__restrict__ amax, int amax_f32,
                                                              uint8_t *__restrict__ q, int64_t ldq,
                                                              float *__restrict__ scale, int scale_rule) {
  bool finite;
  const float s = scale_from_amax_scalar(amax, amax_f32, finite, scale_rule);
  const float recip = recip_exact(s);
  if (blockIdx.x == 0 && threadIdx.x == 0) scale[0] = s;
  const int cpr = C / 8;  // 16-byte chunks per row
  const int64_t total = R * cpr;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / cpr;
    const int c = (int)(i - r * cpr) * 8;
    const v4i v = __builtin_nontemporal_load((const v4i *)(x + r * ldx + c));
    // the amax is handed in and must bound |x|: then every product is within
    // the finite e4m3 range and the hardware converter agrees with the ATen cast
    *(v2i *)(q + r * ldq + c) = finite ? cvt8(v, recip) : cvt8_slow(v, recip);
  }
}

// Row-wise cast with the row amaxes handed in, as lingua/float8.py:43-47 is called: the amax is an
// argument there, not a by-product.  It need not be the true amax of the row (a repeated tensor amax, a
// stale amax of delayed scaling), so a product may leave the finite e4m3 range: chunks whose largest
// product exceeds 448 take the integer conversion, which reproduces the ATen cast there (<= 464 rounds
// to 448, above gives the NaN code).
__global__ __launch_bounds__(256) void cast_rowwise_given_amax_kernel(const uint16_t *__restrict__ x, int64_t R, int C,
                                                                      int64_t ldx, const void *__restrict__ amax, int amax_f32,
                                                                      uint8_t *__restrict__ q, int64_t ldq,
                                                                      float *__restrict__ scale, int scale_rule) {
  const int cpr = C / 8;  // 16-byte chunks per row
  const int64_t total = R * cpr;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / cpr;
    const int c = (int)(i - r * cpr) * 8;
    // clamp(min=EPS) also lifts a negative amax
    const float s = scale_from_amax(amax_f32 ? ((const float *)amax)[r] : bf16_bits_to_f32(((const uint16_t *)amax)[r]), scale_rule);
    const float recip = recip_exact(s);
    if (c == 0) scale[r] = s;
    const v4i v = __builtin_nontemporal_load((const v4i *)(x + r * ldx + c));
    uint32_t m = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) m = pk_absmax_u16(m, (uint32_t)v[k]);
    m = max(m & 0xffffu, m >> 16);
    // !(p <= 448) also catches a NaN product (NaN element, NaN or infinite scale)
    const float p = bf16_bits_to_f32(m) * recip;
    *(v2i *)(q + r * ldq + c) = (p <= kE4M3Max) ? cvt8(v, recip) : cvt8_slow(v, recip);
  }
}

// ---------------------------------------------------------------------------
// Transposed casts (tensor-wise for the dgrad weight, column-wise for wgrad):
// a [256 rows x 64 cols] tile of x becomes a [64 x 256] tile of q.
// Thread t loads 8 columns (one 16-byte load) from each of 4 consecutive rows,
// packs, for each of its 8 columns, the 4 row-consecutive e4m3 bytes into one
// dword and writes it to the transposed tile in LDS; the tile is then read
// back as 16-byte row segments and stored as 256-byte runs of the output rows.
// ---------------------------------------------------------------------------
// Tile shapes: TC columns x (256 / (TC / 8)) * 4 * TU rows.  128 x 128 (TC 128, TU 2) is the one used; 64 x 128 (TC 64,
// TU 1) for tensors with too few 128 x 128 tiles to fill the chip.  Inside the MLP step, against the 64 x 256 tile this
// kernel had before: [16384,4096] 39.1 -> 37.3 us, [16384,11008] 110.1 -> 107.9, weights 28.0 -> 28.0; Llama-1B shapes:
// [16384,8192] 80.1 -> 73.8, [16384,2048] 21.0 -> 21.1, [8192,2048] 12.4 -> 11.8, [2048,2048] 5.2 -> 4.9 (64 x 128).
// 128 x 256 was another 1-5 % ahead on the two widest activations and 4 % behind on every weight.
// Tensors of at least 16384 rows and 8192 columns take 128 x 256 (TU 4): over 26 activation shapes, each timed right
// behind the kernel that produces it, 128 x 128 and 128 x 256 are within 1-3 % of each other there except at 11008
// columns (the 7B ffn width), where 128 x 128 alone falls off -- [16384,11008] 100 against 90 us, [32768,11008] 206
// against 187 -- while 10880, 11136, 11264 and 11520 columns show nothing of the kind.
// The loads are non-temporal, the stores are not: a workgroup writes 128-byte pieces of 128 output rows, the pieces
// next to them come from other workgroups a little later, and ordinary stores leave it to the L2 to write neighbours
// back together.  Inside the MLP step, ordinary against non-temporal stores: [16384,11008] 99.4 against 108.4 us,
// [16384,4096] 35.5 against 37.2, weights 26.2 against 27.7; ordinary loads instead cost 2-4 %.
template <int TC, int TU>
struct TransposeTile {
  static constexpr int kTC = TC;                  // columns of x per tile
  static constexpr int kCCH = TC / 8;             // 8-column chunks per tile row
  static constexpr int kRG = 256 / kCCH;          // 4-row groups covered by the 256 threads in one pass
  static constexpr int kTU = TU;                  // passes (4-row units per thread)
  static constexpr int kTR = kRG * 4 * TU;        // rows of x per tile
  static constexpr int kTStride = kTR + 16;       // LDS row stride in bytes
};
constexpr int kMaxTileRows = 256;                 // no tile is taller (bounds the row stride the host accepts)

// Where the scale comes from: one amax, a column amax each -- or the partial maxima that the row-wise cast's workgroups left
// of them, while these are few --, or one amax that every workgroup finds among the row amaxes
// (a few kilobytes from the L2 under the tile's loads, where a reduction of its own is a launch).  Weights inside a forward
// + backward, us, reduction + cast / this: [2048,2048] 4.7 + 4.7 / 5.2, [4096,14336] 4.8 + 33.6 / 34.7, [14336,4096]
// 7.5 + 34.0 / 36.8.
enum class AmaxFrom { kScalar, kColumns, kRows, kPartials };
constexpr int64_t kMaxAmaxRows = 16384;           // longest list that every workgroup reads

// Columns R .. Rp - 1 of q are zeros: what a reduction over the tokens pads them to.  The rows are whole 16-byte pieces
// then, also for an odd number of tokens: [4093,14336] 36.1 -> 33.9 us, [4093,4096] 13.6 -> 12.4, and no fill in front (5).
//
// Several tensors go through one launch as one list of tiles (the output gradients of linears on one activation and that
// activation; their weights): each alone fills and drains the chip in a few microseconds.  us, one by one / together:
// four [16384,2048] 79.6 / 68.0, [4093,4096] and two [4093,14336] 79.4 / 69.2, two [1021,2048] 5.8 / 3.9, four [3290,1392] 22.7 /
// 15.2, [16384,2048] and two [16384,8192] 173.9 / 165.3; weights: three [2048,2048] 11.8 / 7.5, two [14336,4096] 69.6 / 64.4.
struct TransposedOperand {
  const uint16_t *x;
  int64_t R, ldx;
  const void *amax;             // scalar, column amaxes or row amaxes, as FROM says
  uint8_t *q;
  int64_t ldq, Rp;
  float *scale;
  int C, n_amax, vec_store;     // n_amax: length of the list of row amaxes, rows of partial maxima, or 1 for an fp32 scalar
  int first;                    // first workgroup of the launch; the operands are in order, unused ones start beyond the last
  AmaxFrom from;                // read by the kernel for operands of several kinds
};
constexpr int kMaxTransposed = 4;
struct TransposedOperands {
  TransposedOperand op[kMaxTransposed];
};
// LDS of a workgroup
template <int TC, int TU>
struct TransposeShared {
  __attribute__((aligned(16))) uint8_t tile[TransposeTile<TC, TU>::kTC * TransposeTile<TC, TU>::kTStride];
  float recips[TC];
  uint32_t wave_amax[4], amaxes[TC];
};
#if defined(__HIP_DEVICE_COMPILE__)  // the buffer-resource type exists in the device pass only
template <AmaxFrom FROM, int TC, int TU>
L8_DEV void transpose_tile(const TransposedOperand &op, unsigned block, int scale_rule, TransposeShared<TC, TU> &lds) {
  const uint16_t *const __restrict__ x = op.x;
  const int64_t R = op.R, ldx = op.ldx, ldq = op.ldq, Rp = op.Rp;
  const int C = op.C, n_amax = op.n_amax, vec_store = op.vec_store, amax_f32 = FROM == AmaxFrom::kScalar ? n_amax : 0;
  const uint32_t *const __restrict__ col_amax = (const uint32_t *)op.amax;
  const uint16_t *const __restrict__ amax_rows = (const uint16_t *)op.amax;
  const void *const __restrict__ amax_scalar = op.amax;
  uint8_t *const __restrict__ q = op.q;
  float *const __restrict__ scale = op.scale;
  using T = TransposeTile<TC, TU>;
  constexpr bool ROWS = FROM == AmaxFrom::kRows, PARTIALS = FROM == AmaxFrom::kPartials, PER_COL = FROM == AmaxFrom::kColumns || PARTIALS;
  constexpr int kTC = T::kTC, kCCH = T::kCCH, kRG = T::kRG, kTU = T::kTU, kTR = T::kTR, kTStride = T::kTStride;
  uint8_t *const tile = lds.tile;
  float *const recips = lds.recips;
  uint32_t *const wave_amax = lds.wave_amax;
  const int t = threadIdx.x;
  // Workgroup w takes column block w % nct and row tile (w / nct + w % nct) % nrt:
  // a diagonal walk.  The workgroups resident at one time then touch addresses
  // that differ in their low bits on both sides, which keeps power-of-two row
  // strides (input stride C, output stride R) from piling onto a few memory
  // channels, while each column block still advances through consecutive row
  // tiles (long runs in the output rows) and each row tile through consecutive
  // column blocks (wide bands of the input rows).
  const int nct = (C + kTC - 1) / kTC;
  const int64_t nrt = (Rp + kTR - 1) / kTR;
  const int cb = (int)(block % nct);
  const int64_t rt = (block / nct + cb) % nrt;
  const int64_t r0 = rt * kTR;
  const int c0 = cb * kTC;
  const int cc = t % kCCH;  // which 8-column chunk of the tile
  const int rg = t / kCCH;  // which 4-row group of a pass
  const int c = c0 + cc * 8;

  // Loads without branches, through buffer descriptors whose range check returns zeros: the amax behind the
  // scale(s) first, the tile right behind it.  The counter of outstanding loads retires in order, so the wait for
  // the amax leaves the tile's loads in flight, and the division and the reciprocal run under them.  (With a branch
  // around each load the compiler waited for all of them after the fifth and again before the division.)
  uint32_t amax_lo = 0, amax_hi = 0;
  v4i listed[ROWS ? 4 : 1];
  [[maybe_unused]] v4i parts[PARTIALS ? 8 : 1], part_max = {0, 0, 0, 0};
  if constexpr (ROWS) {
    const __amdgpu_buffer_rsrc_t rsList = make_rsrc(amax_rows, (uint32_t)n_amax * 2u);  // zeros beyond the list
    for (int i0 = t * 8;; i0 += 4 * 256 * 8) {
#pragma unroll
      for (int k = 0; k < 4; ++k) listed[k] = __builtin_amdgcn_raw_buffer_load_b128(rsList, (i0 + k * 256 * 8) * 2, 0, 0);
      if (i0 - t * 8 + 4 * 256 * 8 >= n_amax) break;  // the last four stay in flight under the tile's loads
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int w = 0; w < 4; ++w) amax_lo = pk_absmax_u16(amax_lo, (uint32_t)listed[k][w]);
    }
  } else if constexpr (PARTIALS) {
    // this thread's 8 columns in every kRG-th partial row
    const __amdgpu_buffer_rsrc_t rsPart = make_rsrc(op.amax, (uint32_t)n_amax * (uint32_t)C * 2u);  // zeros beyond the last row
    const uint32_t at = c < C ? (uint32_t)c * 2u : 0x80000000u;
    for (int i0 = rg;; i0 += 8 * kRG) {
#pragma unroll
      for (int k = 0; k < 8; ++k) parts[k] = __builtin_amdgcn_raw_buffer_load_b128(rsPart, (int)(at + (uint32_t)(i0 + k * kRG) * (uint32_t)C * 2u), 0, 0);
      if (i0 - rg + 8 * kRG >= n_amax) break;  // the last eight stay in flight under the tile's loads
#pragma unroll
      for (int k = 0; k < 8; ++k)
#pragma unroll
        for (int w = 0; w < 4; ++w) part_max[w] = (int)pk_absmax_u16((uint32_t)part_max[w], (uint32_t)parts[k][w]);
    }
  } else if (PER_COL) {
    const __amdgpu_buffer_rsrc_t rsAmax = make_rsrc(col_amax, (uint32_t)C * 4u);
    amax_lo = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rsAmax, (c0 + t % kTC) * 4, 0, 0);  // zero beyond column C
  } else {
    // two or four bytes (bf16 or fp32) as two halves: the upper half of a bf16 amax lies beyond the descriptor
    const __amdgpu_buffer_rsrc_t rsAmax = make_rsrc(amax_scalar, amax_f32 ? 4u : 2u);
    amax_lo = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rsAmax, 0, 0, 0);
    amax_hi = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rsAmax, 2, 0, 0);
  }
  // keep the amax's load(s) here, ahead of the tile's: neither sunk to their first use nor rescheduled
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  // kTU units of 4 rows x 8 columns per thread.  The descriptor covers the tile's rows that exist, up to the last
  // column of the last one: a row at or beyond R starts beyond it, and a chunk at or beyond column C (which would
  // otherwise read the next row) is sent there (the range check covers the sum of the lane's and the scalar offset, dword by
  // dword).  The host keeps kTR * ldx * 2 below 2^30.
  const int64_t rows_left = R - r0;
  const uint32_t row_bytes = (uint32_t)ldx * 2u;
  const uint32_t tile_bytes = rows_left <= 0 ? 0u : (uint32_t)((rows_left < kTR ? (int)rows_left : kTR) - 1) * row_bytes + (uint32_t)C * 2u;
  const __amdgpu_buffer_rsrc_t rsX = make_rsrc(x + r0 * ldx, tile_bytes);
  const uint32_t voff = (c < C ? (uint32_t)c * 2u : tile_bytes) + (uint32_t)(rg * 4) * row_bytes;
  v4i in[kTU][4];
#pragma unroll
  for (int u = 0; u < kTU; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      in[u][i] = load16_nt(rsX, voff, (u * kRG * 4 + i) * row_bytes);

  if constexpr (PARTIALS) {
    // the columns' maxima over the kRG groups of partial rows meet in the tile's memory
    static_assert(kRG % 8 == 0 && kRG * kTC * 2 + 8 * kTC * 2 <= kTC * kTStride, "the maxima fit the tile's memory");
    uint32_t *const groups = (uint32_t *)tile, *const eighths = groups + kRG * (kTC / 2);  // [kRG][kTC / 2], [8][kTC / 2] pairs of columns
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
      for (int w = 0; w < 4; ++w) part_max[w] = (int)pk_absmax_u16((uint32_t)part_max[w], (uint32_t)parts[k][w]);
    *(v4i *)(groups + rg * (kTC / 2) + cc * 4) = part_max;
    __syncthreads();
    for (int i = t; i < 8 * (kTC / 2); i += 256) {
      const int pair = i % (kTC / 2), part = i / (kTC / 2);
      uint32_t m = 0;
#pragma unroll
      for (int g = 0; g < kRG / 8; ++g) m = pk_absmax_u16(m, groups[(part * (kRG / 8) + g) * (kTC / 2) + pair]);
      eighths[part * (kTC / 2) + pair] = m;
    }
    __syncthreads();
    uint32_t m = 0;
#pragma unroll
    for (int part = 0; part < 8; ++part) m = pk_absmax_u16(m, eighths[part * (kTC / 2) + (t % kTC) / 2]);
    amax_lo = (t & 1) ? m & 0xffff0000u : m << 16;  // bf16 -> fp32 bit patterns
    if (t < kTC) lds.amaxes[t] = amax_lo;
  }
  if (PER_COL) {
    // every wave computes the 64 scales (a branch around the division would pull the amax's load into it, behind
    // the tile's loads); the first one keeps them
    const float s = scale_from_amax_bits32(amax_lo, scale_rule);
    float rc = recip_exact(s);
    if (amax_lo >= 0x7f800000u) rc = __uint_as_float(0x7fc00000u);  // flag: slow path for this column
    if (t < kTC) {
      if (rt == 0 && c0 + t < C) scale[c0 + t] = s;
      recips[t] = rc;
    }
    __syncthreads();
  }
  if constexpr (ROWS) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int w = 0; w < 4; ++w) amax_lo = pk_absmax_u16(amax_lo, (uint32_t)listed[k][w]);
    const uint32_t m = wave_max_u32(max(amax_lo & 0xffffu, amax_lo >> 16));
    if ((t & 63) == 0) wave_amax[t >> 6] = m;
    __syncthreads();
    amax_lo = max(max(wave_amax[0], wave_amax[1]), max(wave_amax[2], wave_amax[3]));
  }
  float rcp[8];
  bool finite = true;
  if (PER_COL) {
#pragma unroll
    for (int j = 0; j < 8; ++j) rcp[j] = recips[cc * 8 + j];
  } else {
    const uint32_t amax_bits = (amax_lo | (amax_hi << 16)) & (amax_f32 ? 0x7fffffffu : 0x7fffu);  // the sign is ignored
    finite = amax_bits < (amax_f32 ? 0x7f800000u : 0x7f80u);
    const float s = amax_f32 ? scale_from_amax_bits32(amax_bits, scale_rule) : scale_from_amax_bits16(amax_bits, scale_rule);
    const float rc = recip_exact(s);
#pragma unroll
    for (int j = 0; j < 8; ++j) rcp[j] = rc;
    if (block == 0 && t == 0) scale[0] = s;
  }

  // convert and transpose inside the thread: column j <- rows 0..3 of each unit
  bool all_fast = finite;
#pragma unroll
  for (int u = 0; u < kTU; ++u)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int w = j >> 1;
      const bool hi = j & 1;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t p = (uint32_t)in[u][i][w];
        v[i] = __uint_as_float(hi ? (p & 0xffff0000u) : (p << 16)) * rcp[j];
      }
      if (PER_COL && u == 0) all_fast &= rcp[j] == rcp[j];
      int packed = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false);
      packed = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], packed, true);
      *(int *)(tile + (cc * 8 + j) * kTStride + (u * kRG + rg) * 4) = packed;
    }
  if (!all_fast) {
    // A column whose amax is not finite: its bytes are redone from memory with the true reciprocal (0 for an
    // infinite amax, NaN for a NaN) and the integer conversion, and replace what the line above wrote.
#pragma unroll 1
    for (int uj = 0; uj < kTU * 8; ++uj) {
      const int u = uj >> 3, j = uj & 7;
      float rc;
      if (PER_COL) {
        if (recips[cc * 8 + j] == recips[cc * 8 + j]) continue;
        const uint32_t bits = PARTIALS ? lds.amaxes[cc * 8 + j] : col_amax[c + j < C ? c + j : 0];
        rc = recip_exact(scale_from_amax_bits32(bits, scale_rule));
      } else {
        rc = rcp[0];
      }
      uint32_t packed = 0;
      for (int i = 0; i < 4; ++i) {
        const int64_t r = r0 + (u * kRG + rg) * 4 + i;
        if (r < R && c + j < C) packed |= e4m3fn_from_f32_slow(bf16_bits_to_f32(x[r * ldx + c + j]) * rc) << (8 * i);
      }
      *(uint32_t *)(tile + (cc * 8 + j) * kTStride + (u * kRG + rg) * 4) = packed;
    }
  }
  __syncthreads();
  // write out: 64 output rows (columns of x) x kTR bytes, 16 bytes per thread and step
  constexpr int SEGS = kTR / 16;  // 16-byte segments per output row
#pragma unroll
  for (int i = 0; i < kTC * SEGS / 256; ++i) {
    const int idx = i * 256 + t;
    const int oc = idx / SEGS;   // output row within the tile
    const int seg = idx % SEGS;
    const int col = c0 + oc;
    const int64_t r = r0 + seg * 16;
    if (col < C && r < Rp) {
      const v4i v = *(const v4i *)(tile + oc * kTStride + seg * 16);
      uint8_t *dst = q + (int64_t)col * ldq + r;
      if (vec_store && r + 16 <= Rp) {
        *(v4i *)dst = v;  // not a streaming store: see the note on the tile shapes
      } else {
        const uint8_t *src = tile + oc * kTStride + seg * 16;
        for (int b = 0; b < 16 && r + b < Rp; ++b) dst[b] = src[b];
      }
    }
  }
}
#endif

// MANY: the operands come from a list, all of one kind.
template <AmaxFrom FROM, int TC, int TU, bool MANY = false>
__global__ __launch_bounds__(256) void cast_transposed_kernel(const std::conditional_t<MANY, TransposedOperands, TransposedOperand> list, int scale_rule) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ TransposeShared<TC, TU> lds;
  if constexpr (MANY) {
    int which = 0;
#pragma unroll
    for (int i = 1; i < kMaxTransposed; ++i) which += (int)blockIdx.x >= list.op[i].first ? 1 : 0;
    const TransposedOperand &op = list.op[which];
    transpose_tile<FROM, TC, TU>(op, blockIdx.x - (unsigned)op.first, scale_rule, lds);
  } else {
    transpose_tile<FROM, TC, TU>(list, blockIdx.x, scale_rule, lds);
  }
#endif
}

// Operands of several kinds: the weight (row amaxes), the output gradient (partial maxima, or column amaxes) and the
// activation (column amaxes) of a linear's backward pass while each is small.  Bound by what a launch costs: us, all casts of
// the pass, five launches / two: M = 1021 N = K = 2048 14.4 / 10.6, 256 1024 1024 10.8 / 6.9, 1000 3008 2000 19.6 / 17.7,
// 256 8192 1024 17.3 / 14.3; and as many calls less for the host, which such a pass waits for: forward + backward of the first,
// with a bias, 140 -> 126 (with the sums in one launch and the products' early scales; an empty autograd function takes 66 .. 72
// of it, and where the host is at the faster of its two levels the whole pass takes 70 .. 77).
// The first workgroups make the bias gradient, if there is one, 16 columns each (32 on 64 workgroups were the last to finish).
// us at M = 1021 N = K = 2048: 7.5 and a launch of 5.9 for the sums / 10.0 together.
constexpr int kMixedCols = 16;
struct MixedOperands {
  TransposedOperands list;
  const uint16_t *sum_x;
  int64_t sum_rows, sum_ld;
  uint16_t *sums;
  int sum_cols, sum_blocks;
};
template <int TC, int TU>
__global__ __launch_bounds__(256) void cast_transposed_mixed_kernel(const MixedOperands p, int scale_rule) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ union {
    TransposeShared<TC, TU> cast;
    WholeSums<256, kMixedCols> sum;
  } shared;
  if ((int)blockIdx.x < p.sum_blocks) {
    sum_columns<256, kMixedCols>(p.sum_x, p.sum_rows, p.sum_cols, p.sum_ld, p.sums, blockIdx.x, p.sum_blocks, shared.sum);
    return;
  }
  TransposeShared<TC, TU> &lds = shared.cast;
  const int at = (int)blockIdx.x - p.sum_blocks;
  int which = 0;
#pragma unroll
  for (int i = 1; i < kMaxTransposed; ++i) which += at >= p.list.op[i].first ? 1 : 0;
  const TransposedOperand &op = p.list.op[which];
  const unsigned block = (unsigned)(at - op.first);
  if (op.from == AmaxFrom::kRows) transpose_tile<AmaxFrom::kRows, TC, TU>(op, block, scale_rule, lds);
  else if (op.from == AmaxFrom::kPartials) transpose_tile<AmaxFrom::kPartials, TC, TU>(op, block, scale_rule, lds);
  else transpose_tile<AmaxFrom::kColumns, TC, TU>(op, block, scale_rule, lds);
#endif
}

// ---------------------------------------------------------------------------
// host entry points
// ---------------------------------------------------------------------------
static bool aligned(const void *p, size_t a) { return ((uintptr_t)p % a) == 0; }

// Number of workgroups (= rows of the partial-maxima workspace) of the two
// register-resident row-wise kernels; 0 when the shape uses the two-pass kernel.
static int64_t rowwise_blocks(int64_t R, int64_t C, bool colmax) {
  const int64_t nch = (C + 511) / 512;
  const int64_t cus = num_cus();
  if (nch <= 8) {
    const int64_t blocks = (R + kRowWaves - 1) / kRowWaves, cap = cus * (colmax ? 2 : 8);
    return blocks < cap ? blocks : cap;
  }
  if ((nch + kRowWaves - 1) / kRowWaves <= 16) {
    // Workgroups per unit, each with a row in registers and a row requested ahead: enough rows in flight to cover the
    // memory's latency, no more than it wants (and, with column maxima, few partial rows to write and fold).  us, row
    // amaxes alone / cast / with column maxima: [16384,4608] 2 per unit 48.7 / 54.2 / 58.0, 4: 31.9 / 40.3 / 45.7,
    // 6: 28.5 / 41.2, 8: 32.5 / 44.0, with column maxima 3: 48.6; [32768,8192] 2: 102 / 127 / 133, 4: 85 / 130 / 143,
    // 8: 92 / 137, with column maxima 3: 138; behind its producer the cast of [32768,8192] takes 124 / 123 / 130 with 2 / 4 / 8.
    const bool short_row = nch <= 3 * kRowWaves;
    const int64_t cap = cus * (colmax ? (short_row ? 3 : 2) : (short_row ? 6 : 4));
    return R < cap ? R : cap;
  }
  return 0;
}

int fold_colmax_many(const FoldOperand *ops, int n, hipStream_t st) {
  FoldOperands list{};
  int64_t widest = 0;
  for (int i = 0; i < n; ++i) {
    list.op[i] = ops[i];
    if (ops[i].C > widest) widest = ops[i].C;
  }
  hipLaunchKernelGGL(colmax_fold_kernel, dim3((unsigned)((widest + kFoldCols - 1) / kFoldCols), (unsigned)n), dim3(kFoldThreads), 0, st, list);
  L8_HIP(hipGetLastError());
  return L8_OK;
}

int fold_colmax(const void *partials, int64_t slots, int64_t C, float *col_amax, hipStream_t st) {
  const FoldOperand one{partials, col_amax, slots, C};
  return fold_colmax_many(&one, 1, st);
}

static int zero_u32(void *p, int64_t n, hipStream_t st) {
  hipLaunchKernelGGL(zero_u32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, (uint32_t *)p, n);
  L8_HIP(hipGetLastError());
  return L8_OK;
}

int empty_col_amax(float *col_amax, int64_t C, hipStream_t st) { return col_amax && C > 0 ? zero_u32(col_amax, C, st) : L8_OK; }

template <int NCH>
static int launch_rowwise(const void *x, int64_t R, int64_t C, int64_t ldx, void *q, int64_t ldq, float *scale,
                          void *amax, float *col_amax, void *ws, hipStream_t st) {
  const int64_t blocks = rowwise_blocks(R, C, col_amax != nullptr);
  if (col_amax) {
    const size_t lds = (size_t)C * sizeof(uint16_t);
    hipLaunchKernelGGL((cast_rowwise_kernel<NCH, true>), dim3((unsigned)blocks), dim3(kRowBlock), lds, st,
                       (const uint16_t *)x, R, (int)C, ldx, (uint8_t *)q, ldq, scale, (uint16_t *)amax, (uint16_t *)ws, l8::scale_rule(), 0);
    L8_HIP(hipGetLastError());
    return L8_OK;  // the caller folds
  }
  hipLaunchKernelGGL((cast_rowwise_kernel<NCH, false>), dim3((unsigned)blocks), dim3(kRowBlock), 0, st,
                     (const uint16_t *)x, R, (int)C, ldx, (uint8_t *)q, ldq, scale, (uint16_t *)amax, (uint16_t *)nullptr, l8::scale_rule(), 0);
  L8_HIP(hipGetLastError());
  return L8_OK;
}

template <int NCHW>
static int launch_rowwise_wg(const void *x, int64_t R, int64_t C, int64_t ldx, void *q, int64_t ldq, float *scale,
                             void *amax, float *col_amax, void *ws, hipStream_t st) {
  const int64_t blocks = rowwise_blocks(R, C, col_amax != nullptr);
  if (col_amax) {
    hipLaunchKernelGGL((cast_rowwise_wg_kernel<NCHW, true>), dim3((unsigned)blocks), dim3(kRowBlock), 0, st,
                       (const uint16_t *)x, R, (int)C, ldx, (uint8_t *)q, ldq, scale, (uint16_t *)amax, (uint16_t *)ws, l8::scale_rule(), 0);
    L8_HIP(hipGetLastError());
    return L8_OK;  // the caller folds
  }
  hipLaunchKernelGGL((cast_rowwise_wg_kernel<NCHW, false>), dim3((unsigned)blocks), dim3(kRowBlock), 0, st,
                     (const uint16_t *)x, R, (int)C, ldx, (uint8_t *)q, ldq, scale, (uint16_t *)amax, (uint16_t *)nullptr, l8::scale_rule(), 0);
  L8_HIP(hipGetLastError());
  return L8_OK;
}

// Operands of one width in one launch, those with partials collecting column maxima; their folds (operand i's slots in
// slots[i], at most rowwise_blocks of it) are left to the caller.
static int cast_rowwise_groups(const l8_cast_rowwise_cols_item *items, int n, int64_t C, int64_t *slots, hipStream_t st) {
  RowGroups list{};
  int64_t rows = 0, first = 0;
  for (int i = 0; i < n; ++i) rows += items[i].R;
  const int64_t all = rowwise_blocks(rows, C, true);
  for (int i = 0; i < kMaxRowOperands; ++i) {
    if (i >= n) {
      list.op[i].first = INT32_MAX;
      continue;
    }
    const l8_cast_rowwise_cols_item &t = items[i];
    const int64_t most = rowwise_blocks(t.R, C, true), share = all * t.R / rows;
    slots[i] = share < 1 ? 1 : share < most ? share : most;
    list.op[i] = {(const uint16_t *)t.x, t.R, t.ldx, (uint8_t *)t.q, t.ldq, t.scale, (uint16_t *)t.amax,
                  t.col_amax ? (uint16_t *)t.workspace : nullptr, (int)first, (int)slots[i]};
    first += slots[i];
  }
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)first), dim3(kRowBlock), (size_t)C * sizeof(uint16_t), st, nullptr, 0, (int)C, 0, nullptr, 0,
                       nullptr, nullptr, nullptr, l8::scale_rule(), list);
  };
  if (C <= 4 * 512) go(cast_rowwise_kernel<4, true, true>);
  else go(cast_rowwise_kernel<8, true, true>);
  L8_HIP(hipGetLastError());
  return L8_OK;
}
constexpr int64_t kMaxGroupColumns = 8 * 512;  // a wavefront per row

static int cast_rowwise_many(const l8_cast_rowwise_item *items, int n, int64_t C, hipStream_t st) {
  RowOperands list{};
  int64_t rows = 0;
  for (int i = 0; i < kMaxRowOperands; ++i) {
    if (i < n) {
      const l8_cast_rowwise_item &t = items[i];
      list.op[i] = {(const uint16_t *)t.x, rows, t.ldx, (uint8_t *)t.q, t.ldq, t.scale, (uint16_t *)t.amax};
      rows += t.R;
    } else {
      list.op[i].first = INT64_MAX;
    }
  }
  const unsigned blocks = (unsigned)rowwise_blocks(rows, C, false);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kRowBlock), 0, st, nullptr, rows, (int)C, 0, nullptr, 0, nullptr, nullptr, nullptr,
                       l8::scale_rule(), list);
  };
  const int64_t nch = (C + 511) / 512, nchw = (nch + kRowWaves - 1) / kRowWaves;
  if (nch <= 4) go(cast_rowwise_kernel<4, false, true>);
  else if (nch <= 8) go(cast_rowwise_kernel<8, false, true>);
  else if (nchw <= 3) go(cast_rowwise_wg_kernel<3, false, true>);
  else if (nchw <= 4) go(cast_rowwise_wg_kernel<4, false, true>);
  else if (nchw <= 6) go(cast_rowwise_wg_kernel<6, false, true>);
  else go(cast_rowwise_wg_kernel<8, false, true>);
  L8_HIP(hipGetLastError());
  return L8_OK;
}

}  // namespace l8

using namespace l8;

// Can an operand with these pointers and strides be one of several (the checks of cast_rowwise_impl, as an answer)?
static bool many_serves(const l8_cast_rowwise_item &t, int64_t C) {
  return t.R > 0 && t.x && t.q && t.scale && t.ldx % 8 == 0 && t.ldx >= C && aligned(t.x, 16) && t.ldq % 8 == 0 && t.ldq >= C && aligned(t.q, 8);
}

extern "C" int l8_cast_rowwise_many(const l8_cast_rowwise_item *items, int64_t n, int64_t C, void *stream) {
  L8_REQUIRE(items && n >= 0 && C >= 0, "l8_cast_rowwise_many: null items, or a negative count");
  bool together = n > 1 && n <= kMaxRowOperands && C > 0 && C % 8 == 0 && C <= kMaxRowwiseManyColumns;
  for (int64_t i = 0; i < n && together; ++i) together = many_serves(items[i], C);
  if (together) return cast_rowwise_many(items, (int)n, C, (hipStream_t)stream);
  for (int64_t i = 0; i < n; ++i) {
    const l8_cast_rowwise_item &t = items[i];
    const int rc = l8_cast_rowwise(t.x, t.R, C, t.ldx, t.q, t.ldq, t.scale, t.amax, nullptr, nullptr, 0, stream);
    if (rc != L8_OK) return rc;
  }
  return L8_OK;
}

extern "C" int64_t l8_cast_rowwise_workspace(int64_t R, int64_t C) {
  if (R <= 0 || C <= 0) return 0;
  return rowwise_blocks(R, C, true) * C * (int64_t)sizeof(uint16_t);
}

// Up to this many rows of 513 to 4096 columns without column amaxes: a workgroup per row, one or two loads per lane, instead of a
// wave per row with up to eight.  us: [32,2048] 2.39 -> 2.28, [32,4096] 2.69 -> 2.38, [256,4096] 3.44 -> 2.87, [256,1536] 2.68 ->
// 2.56, [512,4096] 3.73 -> 3.48, [512,1024] 2.70 -> 2.62.
constexpr int64_t kFewRows = 512;

// Argument checks and dispatch shared by l8_cast_rowwise and l8_cast_rowwise_noalloc; `what` names the
// entry point in error messages.  `workspace` holds at least l8_cast_rowwise_workspace(R, C) bytes when
// col_amax is given (checked by the callers).  The partial column maxima are left to be folded where `fold` is given (and
// there are any: else its width is 0), and folded otherwise.
static int launch_rowwise_any(const char *what, const void *x, int64_t R, int64_t C, int64_t ldx, void *q, int64_t ldq,
                              float *scale, void *amax, float *col_amax, void *workspace, hipStream_t st);
static int cast_rowwise_impl(const char *what, const void *x, int64_t R, int64_t C, int64_t ldx, void *q, int64_t ldq,
                             float *scale, void *amax, float *col_amax, void *workspace, hipStream_t st, FoldOperand *fold = nullptr) {
  const int rc = launch_rowwise_any(what, x, R, C, ldx, q, ldq, scale, amax, col_amax, workspace, st);
  const int64_t slots = rc == L8_OK && col_amax ? rowwise_blocks(R, C, true) : 0;
  if (fold) *fold = {workspace, col_amax, slots, slots ? C : 0};
  else if (slots) return fold_colmax(workspace, slots, C, col_amax, st);
  return rc;
}

static int launch_rowwise_any(const char *what, const void *x, int64_t R, int64_t C, int64_t ldx, void *q, int64_t ldq,
                              float *scale, void *amax, float *col_amax, void *workspace, hipStream_t st) {
  L8_REQUIRE(x != nullptr, "%s: x is null", what);
  L8_REQUIRE((q == nullptr) || (scale != nullptr), "%s: q given without scale", what);
  L8_REQUIRE(C % 8 == 0 && ldx % 8 == 0 && ldx >= C, "%s: C=%lld and ldx=%lld must be multiples of 8, ldx >= C", what,
             (long long)C, (long long)ldx);
  L8_REQUIRE(aligned(x, 16), "%s: x must be 16-byte aligned", what);
  if (q) L8_REQUIRE(ldq % 8 == 0 && ldq >= C && aligned(q, 8), "%s: q must be 8-byte aligned with ldq %% 8 == 0, ldq >= C", what);
  L8_REQUIRE(C < (1LL << 31), "%s: C too large", what);
  void *ws = workspace;
  const int64_t nch = (C + 511) / 512;
  if (!col_amax && nch > 1 && nch <= 8 && R <= kFewRows) {
    auto few = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)R), dim3(kRowBlock), 0, st, (const uint16_t *)x, R, (int)C, ldx, (uint8_t *)q, ldq, scale, (uint16_t *)amax,
                         (uint16_t *)nullptr, l8::scale_rule(), 0);
    };
    if (nch <= 4) few(cast_rowwise_wg_kernel<1, false>);
    else few(cast_rowwise_wg_kernel<2, false>);
    L8_HIP(hipGetLastError());
    return L8_OK;
  }
  if (nch <= 4) return launch_rowwise<4>(x, R, C, ldx, q, ldq, scale, amax, col_amax, ws, st);
  if (nch <= 8) return launch_rowwise<8>(x, R, C, ldx, q, ldq, scale, amax, col_amax, ws, st);
  // longer rows: one workgroup per row, nchw = chunks per lane
  const int64_t nchw = (nch + kRowWaves - 1) / kRowWaves;
  if (nchw <= 3) return launch_rowwise_wg<3>(x, R, C, ldx, q, ldq, scale, amax, col_amax, ws, st);
  if (nchw <= 4) return launch_rowwise_wg<4>(x, R, C, ldx, q, ldq, scale, amax, col_amax, ws, st);
  if (nchw <= 6) return launch_rowwise_wg<6>(x, R, C, ldx, q, ldq, scale, amax, col_amax, ws, st);
  if (nchw <= 8) return launch_rowwise_wg<8>(x, R, C, ldx, q, ldq, scale, amax, col_amax, ws, st);
  if (nchw <= 16) return launch_rowwise_wg<16>(x, R, C, ldx, q, ldq, scale, amax, col_amax, ws, st);
  int64_t blocks = R < (int64_t)num_cus() * 8 ? R : (int64_t)num_cus() * 8;
  if (col_amax) {
    const int rc = zero_u32(col_amax, C, st);
    if (rc != L8_OK) return rc;
  }
  hipLaunchKernelGGL(cast_rowwise_long_kernel, dim3((unsigned)blocks), dim3(kRowBlock), 0, st, (const uint16_t *)x, R,
                     (int)C, ldx, (uint8_t *)q, ldq, scale, (uint16_t *)amax, (uint32_t *)col_amax, l8::scale_rule());
  L8_HIP(hipGetLastError());
  return L8_OK;
}

extern "C" int l8_cast_rowwise(const void *x, int64_t R, int64_t C, int64_t ldx, void *q, int64_t ldq, float *scale,
                               void *amax, float *col_amax, void *workspace, int64_t workspace_bytes, void *stream) {
  L8_REQUIRE(R >= 0 && C >= 0, "l8_cast_rowwise: negative shape R=%lld C=%lld", (long long)R, (long long)C);
  if (R == 0 || C == 0) return empty_col_amax(col_amax, C, (hipStream_t)stream);
  if (col_amax) {
    const int64_t need = l8_cast_rowwise_workspace(R, C);
    L8_REQUIRE(need == 0 || (workspace != nullptr && workspace_bytes >= need && aligned(workspace, 16)),
               "l8_cast_rowwise: col_amax needs a 16-byte aligned workspace of %lld bytes (l8_cast_rowwise_workspace)",
               (long long)need);
  }
  return cast_rowwise_impl("l8_cast_rowwise", x, R, C, ldx, q, ldq, scale, amax, col_amax, workspace, (hipStream_t)stream);
}

// slabs of rows, and rows of a slab
static int64_t col_sum_slabs(int64_t R, int64_t C, int64_t *slab) {
  const int64_t cols = (C + kSumCols - 1) / kSumCols;
  int64_t n = (4 * (int64_t)num_cus() + cols - 1) / cols;
  if (n > (R + 127) / 128) n = (R + 127) / 128;
  if (n < 1 || R <= kSumWhole) n = 1;
  *slab = (R + n - 1) / n;
  return *slab > 0 ? (R + *slab - 1) / *slab : 1;
}

extern "C" int64_t l8_col_sum_workspace(int64_t R, int64_t C) {
  if (R <= 0 || C <= 0) return 0;
  int64_t slab;
  const int64_t n = col_sum_slabs(R, C, &slab);
  return n > 1 ? n * C * (int64_t)sizeof(float) : 0;
}

extern "C" int l8_col_sum(const void *x, int64_t R, int64_t C, int64_t ldx, void *out, void *workspace, int64_t workspace_bytes, void *stream) {
  L8_REQUIRE(R >= 0 && C >= 0, "l8_col_sum: negative shape");
  if (C == 0) return L8_OK;
  L8_REQUIRE(out && (R == 0 || x), "l8_col_sum: null pointer");
  L8_REQUIRE(C % 8 == 0 && ldx % 8 == 0 && ldx >= C && aligned(x, 16) && C < (1LL << 31), "l8_col_sum: C, ldx multiples of 8 and x 16-byte aligned required");
  const int64_t need = l8_col_sum_workspace(R, C);
  L8_REQUIRE(need == 0 || (workspace && workspace_bytes >= need && aligned(workspace, 4)), "l8_col_sum: needs a workspace of %lld bytes (l8_col_sum_workspace)", (long long)need);
  int64_t slab;
  const int64_t n = col_sum_slabs(R, C, &slab);
  hipStream_t st = (hipStream_t)stream;
  if (R <= kSumWhole) {
    hipLaunchKernelGGL(col_sum_whole_kernel, dim3((unsigned)((C + kWholeCols - 1) / kWholeCols)), dim3(1024), 0, st, (const uint16_t *)x, R, (int)C, ldx, (uint16_t *)out);
    L8_HIP(hipGetLastError());
    return L8_OK;
  }
  hipLaunchKernelGGL(col_sum_kernel, dim3((unsigned)((C + kSumCols - 1) / kSumCols), (unsigned)n), dim3(kSumThreads), 0, st, (const uint16_t *)x, R, (int)C, ldx,
                     slab, (float *)workspace, n == 1 ? (uint16_t *)out : nullptr);
  L8_HIP(hipGetLastError());
  if (n == 1) return L8_OK;
  hipLaunchKernelGGL(col_sum_fold_kernel, dim3((unsigned)((C + 255) / 256)), dim3(256), 0, st, (const float *)workspace, (int)n, (int)C, (uint16_t *)out);
  L8_HIP(hipGetLastError());
  return L8_OK;
}

// (C % 8: a chunk across column C would reach the next workgroup's partial row)
static bool group_serves(const l8_cast_rowwise_cols_item &t, int64_t C) {
  return t.C == C && C % 8 == 0 && many_serves(l8_cast_rowwise_item{t.x, t.R, t.ldx, t.q, t.ldq, t.scale, t.amax}, C);
}

int l8::cast_rowwise_pair(const l8_cast_rowwise_cols_item *two, hipStream_t st, bool *served) {
  const int64_t C = two[0].C;
  *served = C > 0 && C <= kMaxGroupColumns && group_serves(two[0], C) && group_serves(two[1], C);
  if (!*served) return L8_OK;
  int64_t slots[kMaxRowOperands];
  const int rc = cast_rowwise_groups(two, 2, C, slots, st);
  return rc == L8_OK ? fold_colmax(two[0].workspace, slots[0], C, two[0].col_amax, st) : rc;
}

extern "C" int l8_cast_rowwise_cols_many(const l8_cast_rowwise_cols_item *items, int64_t n, void *stream) {
  L8_REQUIRE(n >= 0 && (n == 0 || items), "l8_cast_rowwise_cols_many: null items, or a negative count");
  for (int64_t i = 0; i < n; ++i) {
    const l8_cast_rowwise_cols_item &t = items[i];
    L8_REQUIRE(t.R >= 0 && t.C >= 0 && t.col_amax, "l8_cast_rowwise_cols_many: negative shape, or no column amaxes asked for");
    const int64_t need = l8_cast_rowwise_workspace(t.R, t.C);
    L8_REQUIRE(need == 0 || (t.workspace != nullptr && t.workspace_bytes >= need && aligned(t.workspace, 16)),
               "l8_cast_rowwise_cols_many: needs a 16-byte aligned workspace of %lld bytes (l8_cast_rowwise_workspace) per operand", (long long)need);
  }
  FoldOperand folds[kMaxFolds];
  int pending = 0;
  auto flush = [&]() {
    const int rc = pending ? fold_colmax_many(folds, pending, (hipStream_t)stream) : L8_OK;
    pending = 0;
    return rc;
  };
  for (int64_t i = 0; i < n;) {
    const l8_cast_rowwise_cols_item &t = items[i];
    if (t.R == 0 || t.C == 0) {
      const int rc = empty_col_amax(t.col_amax, t.C, (hipStream_t)stream);
      if (rc != L8_OK) return rc;
      ++i;
      continue;
    }
    int run = 0;  // neighbours of one width that one launch can serve
    while (i + run < n && run < kMaxRowOperands && t.C <= kMaxGroupColumns && group_serves(items[i + run], t.C)) ++run;
    if (run > 1) {
      if (pending + run > kMaxFolds) {
        const int rc = flush();
        if (rc != L8_OK) return rc;
      }
      int64_t slots[kMaxRowOperands];
      const int rc = cast_rowwise_groups(items + i, run, t.C, slots, (hipStream_t)stream);
      if (rc != L8_OK) return rc;
      for (int k = 0; k < run; ++k) folds[pending++] = {items[i + k].workspace, items[i + k].col_amax, slots[k], t.C};
      i += run;
    } else {
      int rc = cast_rowwise_impl("l8_cast_rowwise_cols_many", t.x, t.R, t.C, t.ldx, t.q, t.ldq, t.scale, t.amax, t.col_amax, t.workspace,
                                 (hipStream_t)stream, &folds[pending]);
      if (rc != L8_OK) return rc;
      if (folds[pending].C > 0) ++pending;
      ++i;
    }
    if (pending == kMaxFolds) {
      const int rc = flush();
      if (rc != L8_OK) return rc;
    }
  }
  return flush();
}

// ---------------------------------------------------------------------------
// l8_cast_rowwise for callers that cannot allocate: the partial column maxima go to a static device
// array instead of a caller-supplied workspace.  Each GPU holds its own copy of the array at its own
// address; the address is looked up once per device (with that device current) and kept.
// ---------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[L8_NOALLOC_SCRATCH_BYTES];
static std::atomic<void *> g_scratch_ptr[l8::kMaxDev];  // device address of `scratch`, per device
static std::mutex g_scratch_mutex;

// Device address of `scratch` on the current device (looked up on first use).
static int scratch_of_current_device(void **out) {
  int dev = -1;
  L8_HIP(hipGetDevice(&dev));
  L8_REQUIRE(dev >= 0 && dev < kMaxDev, "device ordinal %d beyond the %d this library keeps state for", dev, kMaxDev);
  void *ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!ptr) {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    ptr = g_scratch_ptr[dev].load(std::memory_order_relaxed);
    if (!ptr) {
      L8_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
      L8_REQUIRE(ptr != nullptr, "hipGetSymbolAddress returned a null address for the scratch array");
      g_scratch_ptr[dev].store(ptr, std::memory_order_release);
    }
  }
  *out = ptr;
  return L8_OK;
}

// Called by l8_device_check with `device` current, so that the look-up (which may load the code object)
// happens at set-up and not inside a caller's capture or serving loop.
int l8::noalloc_setup_current_device() {
  void *ptr = nullptr;
  return scratch_of_current_device(&ptr);
}

extern "C" int l8_cast_rowwise_noalloc(const void *x, int64_t R, int64_t C, int64_t ldx, void *q, int64_t ldq,
                                       float *scale, void *amax, float *col_amax, void *stream) {
  L8_REQUIRE(R >= 0 && C >= 0, "l8_cast_rowwise_noalloc: negative shape R=%lld C=%lld", (long long)R, (long long)C);
  if (R == 0 || C == 0) return empty_col_amax(col_amax, C, (hipStream_t)stream);
  void *ws = nullptr;
  if (col_amax) {
    const int64_t need = l8_cast_rowwise_workspace(R, C);
    L8_REQUIRE(need <= (int64_t)L8_NOALLOC_SCRATCH_BYTES,
               "l8_cast_rowwise_noalloc: [%lld,%lld] with column amaxes needs %lld bytes of scratch, the static array "
               "holds %lld (use l8_cast_rowwise with a workspace)",
               (long long)R, (long long)C, (long long)need, (long long)L8_NOALLOC_SCRATCH_BYTES);
    const int rc = scratch_of_current_device(&ws);
    if (rc != L8_OK) return rc;
  }
  return cast_rowwise_impl("l8_cast_rowwise_noalloc", x, R, C, ldx, q, ldq, scale, amax, col_amax, ws, (hipStream_t)stream);
}

extern "C" int l8_cast_rowwise_given_amax(const void *x, int64_t R, int64_t C, int64_t ldx, const void *amax,
                                          int amax_dtype, void *q, int64_t ldq, float *scale, void *stream) {
  L8_REQUIRE(R >= 0 && C >= 0, "l8_cast_rowwise_given_amax: negative shape");
  if (R == 0 || C == 0) return L8_OK;
  L8_REQUIRE(x && amax && q && scale, "l8_cast_rowwise_given_amax: null pointer");
  L8_REQUIRE(amax_dtype == L8_AMAX_BF16 || amax_dtype == L8_AMAX_F32, "l8_cast_rowwise_given_amax: bad amax_dtype %d", amax_dtype);
  L8_REQUIRE(aligned(amax, amax_dtype == L8_AMAX_F32 ? 4 : 2), "l8_cast_rowwise_given_amax: misaligned amax");
  L8_REQUIRE(C % 8 == 0 && ldx % 8 == 0 && ldx >= C && aligned(x, 16),
             "l8_cast_rowwise_given_amax: C, ldx multiples of 8 and x 16-byte aligned required");
  L8_REQUIRE(ldq >= C && ldq % 8 == 0 && aligned(q, 8),
             "l8_cast_rowwise_given_amax: q must be 8-byte aligned with ldq %% 8 == 0, ldq >= C");
  L8_REQUIRE(C < (1LL << 31), "l8_cast_rowwise_given_amax: C too large");
  const int64_t total = R * (C / 8);
  int64_t blocks = (total + 255) / 256;
  const int64_t cap = (int64_t)num_cus() * 16;
  if (blocks > cap) blocks = cap;
  hipLaunchKernelGGL(cast_rowwise_given_amax_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                     (const uint16_t *)x, R, (int)C, ldx, amax, amax_dtype, (uint8_t *)q, ldq, scale, l8::scale_rule());
  L8_HIP(hipGetLastError());
  return L8_OK;
}

extern "C" int l8_col_amax(const void *x, int64_t R, int64_t C, int64_t ldx, float *col_amax, void *stream) {
  L8_REQUIRE(R >= 0 && C >= 0, "l8_col_amax: negative shape");
  if (R == 0 || C == 0) return empty_col_amax(col_amax, C, (hipStream_t)stream);
  L8_REQUIRE(x && col_amax, "l8_col_amax: null pointer");
  L8_REQUIRE(C % 8 == 0 && ldx % 8 == 0 && ldx >= C && aligned(x, 16), "l8_col_amax: C, ldx multiples of 8 and x 16-byte aligned required");
  L8_REQUIRE(C < (1LL << 31), "l8_col_amax: C too large");
  const int gx = (int)((C / 8 + 255) / 256);
  // enough row slabs to fill the chip, at least 64 rows each
  int64_t slabs = (int64_t)num_cus() * 8 / gx;
  if (slabs < 1) slabs = 1;
  int64_t rows_per = (R + slabs - 1) / slabs;
  if (rows_per < 64) rows_per = 64;
  slabs = (R + rows_per - 1) / rows_per;
  L8_REQUIRE(slabs <= 65535, "l8_col_amax: too many row slabs");
  const int rc = zero_u32(col_amax, C, (hipStream_t)stream);
  if (rc != L8_OK) return rc;
  hipLaunchKernelGGL(col_amax_kernel, dim3(gx, (unsigned)slabs), dim3(256), 0, (hipStream_t)stream,
                     (const uint16_t *)x, R, (int)C, ldx, (int)rows_per, (uint32_t *)col_amax);
  L8_HIP(hipGetLastError());
  return L8_OK;
}

extern "C" int l8_amax_reduce(const void *amax, int64_t n, void *amax_out, void *stream) {
  L8_REQUIRE(n >= 1 && amax && amax_out, "l8_amax_reduce: need n >= 1 and non-null pointers");
  hipLaunchKernelGGL(amax_reduce_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, (const uint16_t *)amax, n,
                     (uint16_t *)amax_out);
  L8_HIP(hipGetLastError());
  return L8_OK;
}

// What a transposed cast is asked for: one of amax (bf16 or fp32 scalar), col_amax and amax_rows is set.
struct TransposedCast {
  const void *x;
  int64_t R, C, ldx;
  const void *amax;
  int amax_f32;
  const float *col_amax;
  const void *amax_rows;
  int64_t n_amax;
  void *q;
  int64_t ldq, Rp;
  float *scale;
};

// `n` casts of one kind (all from column amaxes, all from row amaxes, or one from a scalar) as one list of tiles; with
// `partials` (one per cast; those with slots stand in for column amaxes) of any kinds but the scalar.
template <int TC, int TU>
static int launch_transposed_tile(const TransposedCast *a, int n, hipStream_t st, const FoldOperand *partials = nullptr, void *sums = nullptr) {
  using T = TransposeTile<TC, TU>;
  static_assert(T::kTR <= kMaxTileRows, "the row-stride limit assumes no taller tile");
  TransposedOperands list{};
  int64_t gx = 0;
  for (int i = 0; i < kMaxTransposed; ++i) {
    if (i >= n) {
      list.op[i].first = INT32_MAX;
      continue;
    }
    const TransposedCast &t = a[i];
    const void *amax = t.col_amax ? (const void *)t.col_amax : t.amax_rows ? t.amax_rows : t.amax;
    list.op[i] = {(const uint16_t *)t.x, t.R, t.ldx, amax, (uint8_t *)t.q, t.ldq, t.Rp, t.scale, (int)t.C,
                  t.amax_rows ? (int)t.n_amax : t.amax_f32, (t.ldq % 16 == 0 && aligned(t.q, 16)) ? 1 : 0, (int)gx,
                  t.col_amax ? AmaxFrom::kColumns : t.amax_rows ? AmaxFrom::kRows : AmaxFrom::kScalar};
    if (partials && partials[i].slots) {
      list.op[i].amax = partials[i].partials;
      list.op[i].n_amax = (int)partials[i].slots;
      list.op[i].from = AmaxFrom::kPartials;
    }
    gx += ((t.C + T::kTC - 1) / T::kTC) * ((t.Rp + T::kTR - 1) / T::kTR);
    L8_REQUIRE(gx < INT32_MAX, "transposed cast: shape too large (%lld x %lld)", (long long)t.R, (long long)t.C);
  }
  auto go = [&](auto kernel, const auto &what) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)gx), dim3(256), 0, st, what, l8::scale_rule());
  };
  if constexpr (TC == 64) {
    if (partials) {
      MixedOperands mixed{list, (const uint16_t *)a[0].x, a[0].R, a[0].ldx, (uint16_t *)sums, (int)a[0].C, 0};
      if (sums) mixed.sum_blocks = (int)((a[0].C + kMixedCols - 1) / kMixedCols);
      gx += mixed.sum_blocks;
      go(cast_transposed_mixed_kernel<TC, TU>, mixed);
      L8_HIP(hipGetLastError());
      return L8_OK;
    }
  }
  if (n > 1) {
    if (a[0].col_amax) go(cast_transposed_kernel<AmaxFrom::kColumns, TC, TU, true>, list);
    else go(cast_transposed_kernel<AmaxFrom::kRows, TC, TU, true>, list);
  } else if (a[0].col_amax) {
    go(cast_transposed_kernel<AmaxFrom::kColumns, TC, TU>, list.op[0]);
  } else if (a[0].amax_rows) {
    go(cast_transposed_kernel<AmaxFrom::kRows, TC, TU>, list.op[0]);
  } else {
    go(cast_transposed_kernel<AmaxFrom::kScalar, TC, TU>, list.op[0]);
  }
  L8_HIP(hipGetLastError());
  return L8_OK;
}

static int launch_transposed(const TransposedCast *a, int n, hipStream_t st) {
  int64_t tiles128 = 0;
  bool large = true;
  for (int i = 0; i < n; ++i) {
    // a tile's rows within 1 GiB: then no sum of a lane's offset (up to twice the tile) and a row's scalar offset wraps
    L8_REQUIRE((int64_t)kMaxTileRows * a[i].ldx * 2 < (1LL << 30), "transposed cast: row stride too large (%lld elements)", (long long)a[i].ldx);
    tiles128 += ((a[i].C + 127) / 128) * ((a[i].R + 127) / 128);
    large = large && a[i].R >= 16384 && a[i].C >= 8192;
  }
  if (tiles128 < 4 * (int64_t)num_cus())  // too few 128 x 128 tiles for four workgroups per compute unit
    return launch_transposed_tile<64, 1>(a, n, st);
  if (large)  // the large activations: see the note on the tile shapes
    return launch_transposed_tile<128, 4>(a, n, st);
  return launch_transposed_tile<128, 2>(a, n, st);
}

// Up to this many partial rows a transposed cast's workgroup reads them itself (32 KB of its 64 columns from the L2, beside
// 16 KB of its own operand) instead of waiting for a launch that folds them: what 1024 rows leave, or 256 beyond 4096 columns
// (rowwise_blocks).
constexpr int64_t kMaxReadPartials = 256;

static bool bwd_casts_together(int64_t M, int64_t N, int64_t K) {
  auto tiles = [](int64_t rows, int64_t cols) { return ((cols + 127) / 128) * ((rows + 127) / 128); };
  const int64_t slots = rowwise_blocks(M, N, true);
  // (in launch_transposed's terms: 64-column tiles)
  return M > 0 && N > 0 && K > 0 && N % 8 == 0 && N <= kMaxAmaxRows && slots > 0 && slots <= kMaxReadPartials &&
         tiles(M, N) + tiles(N, K) + tiles(M, K) < 4 * (int64_t)num_cus();
}

static int check_transposed(const char *what, const TransposedCast &a) {
  L8_REQUIRE(a.x && a.q, "%s: null pointer", what);
  L8_REQUIRE(a.C % 8 == 0 && a.ldx % 8 == 0 && a.ldx >= a.C && aligned(a.x, 16), "%s: C, ldx multiples of 8 and x 16-byte aligned required", what);
  L8_REQUIRE(a.C < (1LL << 31), "%s: C too large", what);
  L8_REQUIRE(a.Rp >= a.R && a.ldq >= a.Rp, "%s: transposed output needs ldq >= R and its padding", what);
  return L8_OK;
}

extern "C" int l8_cast_tensorwise(const void *x, int64_t R, int64_t C, int64_t ldx, const void *amax, int amax_dtype,
                                  int transpose, void *q, int64_t ldq, float *scale, void *stream) {
  L8_REQUIRE(R >= 0 && C >= 0, "l8_cast_tensorwise: negative shape");
  L8_REQUIRE(amax && scale, "l8_cast_tensorwise: amax and scale must be non-null");
  L8_REQUIRE(amax_dtype == L8_AMAX_BF16 || amax_dtype == L8_AMAX_F32, "l8_cast_tensorwise: bad amax_dtype %d", amax_dtype);
  L8_REQUIRE(aligned(amax, amax_dtype == L8_AMAX_F32 ? 4 : 2), "l8_cast_tensorwise: misaligned amax");
  if (R == 0 || C == 0) return L8_OK;
  L8_REQUIRE(x && q, "l8_cast_tensorwise: null pointer");
  L8_REQUIRE(C % 8 == 0 && ldx % 8 == 0 && ldx >= C && aligned(x, 16), "l8_cast_tensorwise: C, ldx multiples of 8 and x 16-byte aligned required");
  L8_REQUIRE(C < (1LL << 31), "l8_cast_tensorwise: C too large");
  hipStream_t st = (hipStream_t)stream;
  if (transpose) {
    L8_REQUIRE(ldq >= R, "l8_cast_tensorwise: transposed output needs ldq >= R");
    const TransposedCast a{x, R, C, ldx, amax, amax_dtype == L8_AMAX_F32, nullptr, nullptr, 0, q, ldq, R, scale};
    return launch_transposed(&a, 1, st);
  }
  L8_REQUIRE(ldq >= C && ldq % 8 == 0 && aligned(q, 8), "l8_cast_tensorwise: q must be 8-byte aligned with ldq %% 8 == 0, ldq >= C");
  const int64_t total = R * (C / 8);
  int64_t blocks = (total + 255) / 256;
  const int64_t cap = (int64_t)num_cus() * 16;
  if (blocks > cap) blocks = cap;
  hipLaunchKernelGGL(cast_tensorwise_kernel, dim3((unsigned)blocks), dim3(256), 0, st, (const uint16_t *)x, R, (int)C,
                     ldx, amax, amax_dtype, (uint8_t *)q, ldq, scale, l8::scale_rule());
  L8_HIP(hipGetLastError());
  return L8_OK;
}

// The weight of dgrad with the row amaxes that forward left: bf16 amax_rows[n], as l8_amax_reduce and l8_cast_tensorwise
// would take it.
extern "C" int l8_cast_tensorwise_t_rows(const void *x, int64_t R, int64_t C, int64_t ldx, const void *amax_rows, int64_t n, void *q,
                                         int64_t ldq, float *scale, void *stream) {
  L8_REQUIRE(R >= 0 && C >= 0, "l8_cast_tensorwise_t_rows: negative shape");
  L8_REQUIRE(amax_rows && scale && n >= 8 && n <= kMaxAmaxRows && n % 8 == 0 && aligned(amax_rows, 16),
             "l8_cast_tensorwise_t_rows: 16-byte aligned amaxes, a multiple of 8 of them and at most %lld, required", (long long)kMaxAmaxRows);
  if (R == 0 || C == 0) return L8_OK;
  const TransposedCast a{x, R, C, ldx, nullptr, 0, nullptr, amax_rows, n, q, ldq, R, scale};
  const int rc = check_transposed("l8_cast_tensorwise_t_rows", a);
  return rc == L8_OK ? launch_transposed(&a, 1, (hipStream_t)stream) : rc;
}

static int cast_colwise(const char *what, const void *x, int64_t R, int64_t C, int64_t ldx, const float *col_amax, void *q,
                        int64_t ldq, int64_t Rp, float *scale, void *stream) {
  L8_REQUIRE(R >= 0 && C >= 0, "%s: negative shape", what);
  if (C == 0) return L8_OK;
  L8_REQUIRE(col_amax && scale, "%s: col_amax and scale must be non-null", what);
  L8_REQUIRE(R > 0, "%s: R must be positive when C > 0", what);
  const TransposedCast a{x, R, C, ldx, nullptr, 0, col_amax, nullptr, 0, q, ldq, Rp, scale};
  const int rc = check_transposed(what, a);
  return rc == L8_OK ? launch_transposed(&a, 1, (hipStream_t)stream) : rc;
}

extern "C" int l8_cast_colwise_transposed(const void *x, int64_t R, int64_t C, int64_t ldx, const float *col_amax,
                                          void *q, int64_t ldq, float *scale, void *stream) {
  return cast_colwise("l8_cast_colwise_transposed", x, R, C, ldx, col_amax, q, ldq, R, scale, stream);
}

extern "C" int l8_cast_colwise_transposed_pad(const void *x, int64_t R, int64_t C, int64_t ldx, const float *col_amax,
                                              void *q, int64_t ldq, int64_t Rp, float *scale, void *stream) {
  return cast_colwise("l8_cast_colwise_transposed_pad", x, R, C, ldx, col_amax, q, ldq, Rp, scale, stream);
}

extern "C" int l8_linear_bwd_casts(const l8_linear_bwd_casts_args *p) { return l8_linear_bwd_casts_bias(p, nullptr); }

extern "C" int l8_linear_bwd_casts_bias(const l8_linear_bwd_casts_args *p, void *bias_grad) {
  L8_REQUIRE(p && bwd_casts_together(p->M, p->N, p->K), "l8_linear_bwd_casts: null arguments, or a shape that l8_linear_bwd_casts_pays does not name");
  const l8_linear_bwd_casts_args &a = *p;
  hipStream_t st = (hipStream_t)a.stream;
  L8_REQUIRE(a.g && a.qg && a.sg && a.qgt && a.sgt && (a.qwt == nullptr || (a.w && a.amax_w && a.swt && aligned(a.amax_w, 16))) &&
                 (a.qat == nullptr || (a.a && a.a_col && a.sat)), "l8_linear_bwd_casts: null or misaligned pointer");
  const int64_t need = l8_cast_rowwise_workspace(a.M, a.N);
  L8_REQUIRE(a.workspace && a.workspace_bytes >= need && aligned(a.workspace, 16), "l8_linear_bwd_casts: needs a 16-byte aligned workspace of %lld bytes", (long long)need);
  TransposedCast casts[3];
  FoldOperand partials[3] = {};
  int n = 0;
  casts[n] = {a.g, a.M, a.N, a.ldg, nullptr, 0, nullptr, nullptr, 0, a.qgt, a.ldqgt, a.Mp, a.sgt};
  partials[n++] = {a.workspace, nullptr, rowwise_blocks(a.M, a.N, true), a.N};
  if (a.qat) casts[n++] = {a.a, a.M, a.K, a.lda, nullptr, 0, a.a_col, nullptr, 0, a.qat, a.ldqat, a.Mp, a.sat};
  if (a.qwt) casts[n++] = {a.w, a.N, a.K, a.ldw, nullptr, 0, nullptr, a.amax_w, a.N, a.qwt, a.ldqwt, a.N, a.swt};
  for (int i = 0; i < n; ++i) {
    const int rc = check_transposed("l8_linear_bwd_casts", casts[i]);
    if (rc != L8_OK) return rc;
    L8_REQUIRE((int64_t)kMaxTileRows * casts[i].ldx * 2 < (1LL << 30), "l8_linear_bwd_casts: row stride too large (%lld elements)", (long long)casts[i].ldx);
  }
  // (the column amaxes' place is not written: the partial maxima stay in the workspace for the casts behind)
  const int rc = launch_rowwise_any("l8_linear_bwd_casts", a.g, a.M, a.N, a.ldg, a.qg, a.ldqg, a.sg, nullptr, (float *)a.workspace, a.workspace, st);
  return rc == L8_OK ? launch_transposed_tile<64, 1>(casts, n, st, partials, bias_grad) : rc;
}

extern "C" int l8_linear_bwd_casts_pays(int64_t M, int64_t N, int64_t K) { return bwd_casts_together(M, N, K) ? 1 : 0; }

extern "C" int l8_cast_transposed_many(const l8_cast_transposed_item *items, int64_t n, void *stream) {
  L8_REQUIRE(n >= 0 && (n == 0 || items), "l8_cast_transposed_many: null items, or a negative count");
  TransposedCast casts[kMaxTransposed];
  for (int64_t i = 0; i < n; ++i) {  // all are checked before any of them is enqueued
    const l8_cast_transposed_item &t = items[i];
    L8_REQUIRE(t.R > 0 && t.C > 0 && t.scale && (t.col_amax != nullptr) != (t.amax_rows != nullptr),
               "l8_cast_transposed_many: operands with rows, a scale and either column amaxes or row amaxes required");
    L8_REQUIRE(!t.amax_rows || (t.n_amax >= 8 && t.n_amax <= kMaxAmaxRows && t.n_amax % 8 == 0 && aligned(t.amax_rows, 16)),
               "l8_cast_transposed_many: 16-byte aligned row amaxes, a multiple of 8 of them and at most %lld, required", (long long)kMaxAmaxRows);
    const int rc = check_transposed("l8_cast_transposed_many", TransposedCast{t.x, t.R, t.C, t.ldx, nullptr, 0, t.col_amax, t.amax_rows, t.n_amax, t.q, t.ldq, t.Rp, t.scale});
    if (rc != L8_OK) return rc;
    L8_REQUIRE((int64_t)kMaxTileRows * t.ldx * 2 < (1LL << 30), "l8_cast_transposed_many: row stride too large (%lld elements)", (long long)t.ldx);
  }
  for (int64_t i = 0; i < n;) {  // runs of one kind
    int run = 0;
    for (; i < n && run < kMaxTransposed; ++i, ++run) {
      const l8_cast_transposed_item &t = items[i];
      if (run && (t.col_amax != nullptr) != (casts[0].col_amax != nullptr)) break;
      casts[run] = TransposedCast{t.x, t.R, t.C, t.ldx, nullptr, 0, t.col_amax, t.amax_rows, t.n_amax, t.q, t.ldq, t.Rp, t.scale};
    }
    const int rc = launch_transposed(casts, run, (hipStream_t)stream);
    if (rc != L8_OK) return rc;
  }
  return L8_OK;
}
