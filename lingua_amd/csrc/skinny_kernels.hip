// Products of a few tokens with a whole weight: y[M,N] = x[M,K] . w[N,K]^T, M <= 64.
//
// What generation and short prompts call (lingua/float8.py:85-96 with M in the tens): every weight byte is used for a
// handful of tokens, so the weight's bytes per second are all that counts, and a 128 x 128 tile leaves most of the chip
// without work ([32,4096] . [11008,4096]^T has 86 of them).  Here a workgroup owns 16 weight rows (or 32) and ALL tokens:
//
//   * its eight waves split K between them (step s of 128 elements goes to wave s % 8), so that even a [2048,2048] weight
//     puts a thousand waves to work, each with all of its few loads in flight, and no wave waits for another;
//   * memory is read in whole 128-byte lines, eight lanes to a row.  (Read in the layout that the matrix instruction
//     wants -- neighbouring lanes hold neighbouring ROWS -- the four lanes that are served together hit four lines, and
//     a compute unit took in 14 bytes per clock.)  Each wave turns its tiles round in 2 KiB of LDS of its own: LDS
//     operations of one wave are served in order, so that takes no barrier;
//   * the eight partial tiles meet in LDS and are added in the order of the waves: the result depends on K alone, not on
//     the grid, the number of rows or of tokens.
//
// SW > 0 takes the weight in bf16 and quantises it in registers between its only read and the product (2 bytes of traffic
// per element instead of the cast's 3 and the product's 1): same row amax, scale and bytes as the row-wise cast
// (lingua/float8.py:43-47, :87), hence the same y.  SX > 0 does the same to a handful of tokens.
#include "l8_common.h"
#include "skinny.h"

namespace l8 {

constexpr int kSkWaves = 8;
constexpr int kSkBlock = kSkWaves * 64;
constexpr int kSkStep = 128;            // elements of K per matrix instruction
static_assert(kSkinnyMaxQuantK == kSkinnyMaxQuantSteps * kSkStep * kSkWaves, "a wave keeps its share of a row in registers");
constexpr int kSkTile = 16 * kSkStep;   // bytes of a tile of 16 rows of one step

#if defined(__HIP_DEVICE_COMPILE__)
L8_DEV uint32_t absmax4(uint32_t m, v4i v) {
#pragma unroll
  for (int k = 0; k < 4; ++k) m = pk_absmax_u16(m, (uint32_t)v[k]);
  return m;
}
// maximum over the 16 lanes of a DPP row, in every lane of it
L8_DEV uint32_t dpp_row_max(uint32_t v) {
  int x = (int)v;
  auto step = [&](int moved) { x = (int)max((uint32_t)x, (uint32_t)moved); };
  step(__builtin_amdgcn_update_dpp(0, x, 0xB1, 0xF, 0xF, true));   // quad_perm [1,0,3,2]
  step(__builtin_amdgcn_update_dpp(0, x, 0x4E, 0xF, 0xF, true));   // quad_perm [2,3,0,1]
  step(__builtin_amdgcn_update_dpp(0, x, 0x124, 0xF, 0xF, true));  // row_ror:4
  step(__builtin_amdgcn_update_dpp(0, x, 0x128, 0xF, 0xF, true));  // row_ror:8
  return (uint32_t)x;
}
// 16-byte chunk c (of 8) of row r of a tile lives at chunk position c ^ f(r): the fragment reads of 16 rows then cover
// all 64 banks once (as in the GEMM)
L8_DEV int tile_pos(int r, int c) { return r * kSkStep + ((c ^ (r & 7) ^ ((r >> 3) & 1)) * 16); }
#endif

// MT tiles of 16 tokens, NT of 16 weight rows, U steps of a wave requested together.
// SW > 0: the weight comes in bf16, at most SW steps per wave are held in registers.
// SX > 0: x comes in bf16 (one tile of tokens), at most SX steps per wave are held in registers.
template <int MT, int NT, int U, int SW, int SX>
__global__ __launch_bounds__(kSkBlock, (SW > 4 || (SW && (MT > 2 || SX > 0)) || SX > 4 ? 2 : 4)) void linear_skinny_kernel(const SkinnyArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr bool QW = SW > 0, QX = SX > 0;
  static_assert(NT == 1 || (!QW && !QX), "one tile of weight rows is quantised");
  static_assert(!QX || (MT == 1 && (QW ? SW == SX : U == SX)), "x is quantised for one tile of tokens");
  constexpr int kBuf = 2 * kSkTile;  // a wave's two tile buffers: weight rows, tokens
  constexpr int kRed = MT * NT * 64 * 16;
  __shared__ __attribute__((aligned(16))) uint8_t lds[kSkWaves * (kBuf > kRed ? kBuf : kRed)];
  __shared__ uint32_t amax_w[kSkWaves][16], amax_x[kSkWaves][16];
  __shared__ float scale_w[16], scale_x[16];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * (16 * NT);
  const int KT = (p.K + kSkStep - 1) / kSkStep;
  constexpr uint32_t kBeyond = 0x80000000u;  // an offset no descriptor covers: the load returns zeros
  constexpr int EW = QW ? 2 : 1, EX = QX ? 2 : 1;  // bytes per element of the weight and of x

  const int64_t w_left = ((int64_t)(p.N - n0 - 1) * p.ldw + p.K) * EW;
  const __amdgpu_buffer_rsrc_t rsW = make_rsrc((const uint8_t *)p.w + (int64_t)n0 * p.ldw * EW, w_left < 0x7fffffff ? (uint32_t)w_left : 0x7fffffffu);
  const __amdgpu_buffer_rsrc_t rsX = make_rsrc(p.x, (uint32_t)(((int64_t)(p.M - 1) * p.ldx + p.K) * EX));
  uint8_t *const wbuf = lds + wave * kBuf, *const xbuf = wbuf + kSkTile;
  // fp8 tile of 16 rows x 128 bytes: two loads of eight rows each
  const int lrow = lane >> 3, lchunk = lane & 7;
  const int put0 = tile_pos(lrow, lchunk), put1 = tile_pos(lrow + 8, lchunk);
  // bf16 tile of 16 rows x 256 bytes: four loads of four rows each, 16 lanes to a row
  const int qrow = lane >> 4, qchunk = lane & 15, qput = (qchunk & 1) * 8;
  // fragment: lane l holds row l % 16, chunks 2 (l / 16) and 2 (l / 16) + 1 of the step
  const int frow = lane & 15, fpiece = lane >> 4;
  const int get0 = tile_pos(frow, 2 * fpiece), get1 = tile_pos(frow, 2 * fpiece + 1);
  auto mask = [&](int k) { return k < p.K ? 0u : kBeyond; };
  auto fragment = [&](uint8_t *buf) {
    __builtin_amdgcn_wave_barrier();
    const v4i f0 = *(const v4i *)(buf + get0), f1 = *(const v4i *)(buf + get1);
    __builtin_amdgcn_wave_barrier();
    return v8i{f0[0], f0[1], f0[2], f0[3], f1[0], f1[1], f1[2], f1[3]};
  };
  auto turn = [&](uint8_t *buf, v4i a, v4i b) {
    *(v4i *)(buf + put0) = a;
    *(v4i *)(buf + put1) = b;
    return fragment(buf);
  };
  auto load_x = [&](int s, int mt, v4i &a, v4i &b) {
    const int k = s * kSkStep + lchunk * 16;
    const uint32_t off = (uint32_t)((mt * 16 + lrow) * (int)p.ldx + k) | mask(k);
    a = __builtin_amdgcn_raw_buffer_load_b128(rsX, (int)off, 0, 0);
    b = __builtin_amdgcn_raw_buffer_load_b128(rsX, (int)off, 8 * (int)p.ldx, 0);
  };
  auto load_w = [&](int s, int nt, v4i &a, v4i &b) {
    const int k = s * kSkStep + lchunk * 16;
    const uint32_t off = (uint32_t)((nt * 16 + lrow) * (int)p.ldw + k) | mask(k);
    a = load16_nt(rsW, off, 0);
    b = load16_nt(rsW, off, (uint32_t)(8 * (int)p.ldw));
  };

  v4f acc[NT * MT];
#pragma unroll
  for (int t = 0; t < NT * MT; ++t) acc[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  auto mma = [&](v8i wf, v8i xf, v4f c) { return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf, xf, c, 0, 0, 0, 0, 0, 0); };

  // Row j * 4 + qrow of a tile held as raw[..][j]: its maximum over this wave's share of K, and 1 / scale from all waves'.
  auto row_maxima = [&](auto &raw, uint32_t (&out)[kSkWaves][16], int rows) {
    constexpr int S = sizeof(raw) / sizeof(raw[0]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j * 4 >= rows) break;
      uint32_t m = 0;
#pragma unroll
      for (int i = 0; i < S; ++i) m = absmax4(m, raw[i][j]);
      m = dpp_row_max(max(m & 0xffffu, m >> 16));
      if (qchunk == 0) out[wave][j * 4 + qrow] = m;
    }
  };
  auto row_scales = [&](const uint32_t (&amax)[kSkWaves][16], float (&scale)[16], float (&recip)[4], int rows) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j * 4 >= rows) break;
      uint32_t bits = 0;
#pragma unroll
      for (int v = 0; v < kSkWaves; ++v) bits = max(bits, amax[v][j * 4 + qrow]);
      // Of a row whose amax is not finite every product is zero or NaN and its scale infinite or NaN: all its results
      // are NaN whichever way its bytes are made, so there is no integer conversion here.
      const RowScale rs = row_scale(bits, p.scale_rule);
      recip[j] = rs.recip;
      if (wave == 0 && qchunk == 0) scale[j * 4 + qrow] = rs.s;
    }
  };
  // the same tile as bytes, in the layout of the matrix instruction
  auto quantised = [&](uint8_t *buf, const v4i (&raw)[4], const float (&recip)[4], int rows) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j * 4 >= rows) break;
      *(v2i *)(buf + tile_pos(j * 4 + qrow, qchunk >> 1) + qput) = cvt8(raw[j], recip[j]);
    }
    return fragment(buf);
  };

  [[maybe_unused]] v4i xraw[QX ? SX : 1][4];
  [[maybe_unused]] float xrecip[4], wrecip[4];
  if constexpr (QX) {
#pragma unroll
    for (int i = 0; i < SX; ++i) {
      const int k = (wave + i * kSkWaves) * kSkStep + qchunk * 8;
      const uint32_t off = (uint32_t)((qrow * (int)p.ldx + k) * 2) | mask(k);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        xraw[i][j] = j * 4 < p.M ? __builtin_amdgcn_raw_buffer_load_b128(rsX, (int)off, j * 4 * (int)p.ldx * 2, 0) : v4i{0, 0, 0, 0};
    }
  }
  if constexpr (QW) {
    v4i raw[SW][4];
#pragma unroll
    for (int i = 0; i < SW; ++i) {
      const int k = (wave + i * kSkWaves) * kSkStep + qchunk * 8;
      const uint32_t off = (uint32_t)((qrow * (int)p.ldw + k) * 2) | mask(k);
#pragma unroll
      for (int j = 0; j < 4; ++j) raw[i][j] = load16_nt(rsW, off, (uint32_t)(j * 4 * (int)p.ldw * 2));
    }
    if constexpr (QX) row_maxima(xraw, amax_x, p.M);
    row_maxima(raw, amax_w, 16);
    __syncthreads();
    if constexpr (QX) row_scales(amax_x, scale_x, xrecip, p.M);
    row_scales(amax_w, scale_w, wrecip, 16);
#pragma unroll
    for (int i = 0; i < SW; ++i) {
      if constexpr (QX) {
        const v8i wf = quantised(wbuf, raw[i], wrecip, 16);
        acc[0] = mma(wf, quantised(xbuf, xraw[i], xrecip, p.M), acc[0]);
      } else {
        v4i a[MT], b[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) load_x(wave + i * kSkWaves, mt, a[mt], b[mt]);
        const v8i wf = quantised(wbuf, raw[i], wrecip, 16);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt] = mma(wf, turn(xbuf, a[mt], b[mt]), acc[mt]);
      }
    }
  } else if constexpr (QX) {
    v4i wa[U], wb[U];
#pragma unroll
    for (int u = 0; u < U; ++u) load_w(wave + u * kSkWaves, 0, wa[u], wb[u]);
    row_maxima(xraw, amax_x, p.M);
    __syncthreads();
    row_scales(amax_x, scale_x, xrecip, p.M);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const v8i xf = quantised(xbuf, xraw[u], xrecip, p.M);
      acc[0] = mma(turn(wbuf, wa[u], wb[u]), xf, acc[0]);
    }
  } else {
    for (int s0 = wave; s0 < KT; s0 += kSkWaves * U) {
      v4i wa[U][NT], wb[U][NT], xa[U][MT], xb[U][MT];
#pragma unroll
      for (int u = 0; u < U; ++u)  // the weight first: its bytes come from HBM, the tokens' from the L2
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) load_w(s0 + u * kSkWaves, nt, wa[u][nt], wb[u][nt]);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) load_x(s0 + u * kSkWaves, mt, xa[u][mt], xb[u][mt]);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        v8i wf[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) wf[nt] = turn(wbuf, wa[u][nt], wb[u][nt]);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const v8i xf = turn(xbuf, xa[u][mt], xb[u][mt]);
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) acc[nt * MT + mt] = mma(wf[nt], xf, acc[nt * MT + mt]);
        }
      }
    }
  }

  // ---- the waves' partial tiles, added in the order of the waves ----
  __syncthreads();  // the tile buffers become the array of partial tiles
  static_assert(NT * MT <= kSkWaves, "a wave adds up one tile");
  v4f(*red)[NT * MT][64] = reinterpret_cast<v4f(*)[NT * MT][64]>(lds);
#pragma unroll
  for (int t = 0; t < NT * MT; ++t) red[wave][t][lane] = acc[t];
  __syncthreads();
  if (wave >= NT * MT) return;
  v4f sum = red[0][wave][lane];
#pragma unroll
  for (int v = 1; v < kSkWaves; ++v) sum += red[v][wave][lane];
  // lane: token (lane & 15) of token tile wave % MT, rows 4 * (lane >> 4) .. + 3 of weight tile wave / MT
  const int m = wave % MT * 16 + frow, nl = wave / MT * 16 + fpiece * 4, n = n0 + nl;
  if (m >= p.M || n >= p.N) return;
  const float sa = QX ? scale_x[frow] : p.sx_row ? p.sx[m] : p.sx[0];
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int ne = n + e < p.N ? n + e : p.N - 1;
    const float sb = QW ? scale_w[nl + e] : (p.sw_row ? p.sw[ne] : p.sw[0]);
    v[e] = sum[e] * sa * sb;
    if (p.bias) v[e] += bf16_bits_to_f32(p.bias[ne]);
  }
  uint16_t *dst = p.y + (int64_t)m * p.ldy + n;
  if (p.add) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < p.N) v[e] = bf16_round(v[e]) + bf16_bits_to_f32(dst[e]);
  }
  if (n + 4 <= p.N && (((uintptr_t)dst) & 7) == 0) {
    *(v2i *)dst = v2i{(int)(bf16_rne_bits(v[0]) | (bf16_rne_bits(v[1]) << 16)), (int)(bf16_rne_bits(v[2]) | (bf16_rne_bits(v[3]) << 16))};
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < p.N) dst[e] = (uint16_t)bf16_rne_bits(v[e]);
  }
#endif
}

template <int MT, int NT, int U, int SW, int SX>
static int skinny_go(const SkinnyArgs &p, hipStream_t st) {
  hipLaunchKernelGGL((linear_skinny_kernel<MT, NT, U, SW, SX>), dim3((unsigned)((p.N + 16 * NT - 1) / (16 * NT))), dim3(kSkBlock), 0, st, p);
  L8_HIP(hipGetLastError());
  return L8_OK;
}

bool skinny_serves(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int w_bytes) {
  // offsets inside a workgroup's 16 weight rows and inside x are 31-bit
  return M >= 1 && M <= kSkinnyMaxM && N >= 1 && N < (1LL << 31) - 16 && K + kSkStep * kSkWaves * 4 < (1LL << 30) &&
         (16 * ldw + K) * w_bytes < (1LL << 31) && 64 * ldx + K < (1LL << 31) &&
         (w_bytes == 1 || K <= (int64_t)kSkinnyMaxQuantK);
}

// A handful of tokens is quantised by every workgroup for itself, from registers: its cast is a launch of a few
// microseconds for a few kilobytes.  The rows are read by every workgroup as bf16 (twice the bytes), and what a wave
// holds of them costs the quantised weight its second workgroup on a unit.  us, weights cold, product alone / with x
// quantised in it (the cast on its own: 2 to 4, and a launch): [1,2048].[2048,2048] 3.6 / 3.6, [8,4096].[4096,4096]
// 5.5 / 6.6, [8,4096].[11008,4096] 10.0 / 12.8, but [16,4096].[4096,4096] 5.8 / 9.0.  Weight quantised too:
// [8,2048].[8192,2048] 12.2 / 11.6, [8,4096].[4096,4096] 10.3 / 11.8, but [1,4096].[11008,4096], where a unit has two
// workgroups, 20.8 / 28.0.
bool skinny_quantises_x(int64_t M, int64_t N, int64_t K, int64_t ldx, int w_bytes) {
  return M >= 1 && M <= 8 && K <= 4 * kSkStep * kSkWaves && (16 * ldx + K) * 2 < (1LL << 31) &&
         (w_bytes == 1 || K <= 2 * kSkStep * kSkWaves || (N + 15) / 16 <= num_cus());
}

// How many steps a wave requests together (U): all of them where it has two, else four while the registers last, one with
// more tokens.  us, weights cold: [1,2048].[2048,2048] U = 2 / 4 3.4 / 3.9; [7,4096].[4096,4096] 5.8 / 5.4; [1,4096].
// [11008,4096] 10.6 / 9.3 (4.8 TB/s; 19.4 with 128 x 128 tiles); two token tiles U = 1 / 2 / 4: [32,11008].[4096,11008]
// 14.0 / 14.8 / 14.9 (43.9 with tiles), [32,4096].[4096,4096] 7.1 / 7.2 / 6.7, [17,2048].[8192,2048] 6.1 / 5.8 / 7.4; four
// token tiles U = 1 / 2: [64,4096].[11008,4096] 19.8 / 20.7 (19.6), [64,14336].[4096,14336] 23.6 / 24.3 (57.4).
//
// Two tiles of weight rows per workgroup (NT): a compute unit takes in some 25 bytes per clock, weight and tokens together, and
// every workgroup reads all tokens; so what counts is rounds of one workgroup per unit, times the rows that each reads.  Twice the
// rows need half the rounds of tokens, and above 16 rows per unit 257 tiles are no longer two rounds for little more than one's
// work.  Sums, their order and the results are the same.  us, weights cold, one tile / two: [1,8960].[5120,8960] 12.9 / 10.9,
// [1,5120].[12800,5120] 16.1 / 13.6, [16,4096].[14336,4096] 13.4 / 12.0, [32,8960].[5120,8960] 19.8 / 14.5, [32,4096].[8192,4096]
// 11.8 / 9.8, [64,6752].[6000,6752] 21.0 / 15.8; where the rule says one: [1,8192].[2560,8192] 6.6 / 8.8, [64,8192].[2560,8192]
// 12.5 / 14.9, [8,3648].[10496,3648] 8.4 / 9.4.  Beyond four rounds 16 tokens or fewer keep HBM busy either way and gain nothing:
// [16,4096].[20480,4096] 16.9 / 18.1, [1,4096].[24576,4096] 18.0 / 19.3, but [32,4096].[32000,4096] 35.3 / 27.8.  U there, 2 / 4: three or four steps [16,4096].[8192,4096] 9.2 / 8.1, else
// [1,2048].[6400,2048] 4.8 / 5.6, [16,8960].[5120,8960] 12.9 / 13.8; two token tiles 1 / 2: [32,6752].[6000,6752] 11.8 / 13.2.
int skinny_linear(const SkinnyArgs &p, bool w_is_bf16, bool x_is_bf16, hipStream_t st) {
  const int mt = (p.M + 15) / 16;
  const int steps = (p.K + kSkStep * kSkWaves - 1) / (kSkStep * kSkWaves);  // of a wave
  if (x_is_bf16) {
    if (w_is_bf16) return steps <= 2 ? skinny_go<1, 1, 1, 2, 2>(p, st) : skinny_go<1, 1, 1, 4, 4>(p, st);
    return steps <= 2 ? skinny_go<1, 1, 2, 0, 2>(p, st) : skinny_go<1, 1, 4, 0, 4>(p, st);
  }
  if (w_is_bf16) {
#define L8_SKINNY_Q(MT)                                 \
  if (steps <= 4) return skinny_go<MT, 1, 1, 4, 0>(p, st); \
  if (steps <= 8) return skinny_go<MT, 1, 1, 8, 0>(p, st); \
  return skinny_go<MT, 1, 1, kSkinnyMaxQuantSteps, 0>(p, st)
    if (mt == 1) { L8_SKINNY_Q(1); }
    if (mt == 2) { L8_SKINNY_Q(2); }
    L8_SKINNY_Q(4);
#undef L8_SKINNY_Q
  }
  const int64_t cus = num_cus(), t16 = ((int64_t)p.N + 15) / 16, t32 = ((int64_t)p.N + 31) / 32;
  if ((p.M > 16 || t16 <= 4 * cus) && (t32 + cus - 1) / cus * (32 + p.M) < (t16 + cus - 1) / cus * (16 + p.M) && 32 * p.ldw + p.K < (1LL << 31)) {
    if (mt == 1) return steps == 3 || steps == 4 ? skinny_go<1, 2, 4, 0, 0>(p, st) : skinny_go<1, 2, 2, 0, 0>(p, st);
    if (mt == 2) return skinny_go<2, 2, 1, 0, 0>(p, st);
    if (mt == 3) return skinny_go<3, 2, 1, 0, 0>(p, st);
    return skinny_go<4, 2, 1, 0, 0>(p, st);
  }
  if (mt == 1) return steps <= 2 ? skinny_go<1, 1, 2, 0, 0>(p, st) : skinny_go<1, 1, 4, 0, 0>(p, st);
  if (mt == 2) return steps <= 2 ? skinny_go<2, 1, 2, 0, 0>(p, st) : skinny_go<2, 1, 1, 0, 0>(p, st);
  if (mt == 3) return skinny_go<3, 1, 1, 0, 0>(p, st);
  return skinny_go<4, 1, 1, 0, 0>(p, st);
}

}  // namespace l8
