// fp8 (e4m3fn) x fp8 -> bf16 "NT" GEMM on the gfx950 matrix cores.
//
//   C[m,n] = bf16( (sum_k A[m,k] * B[n,k]) * sa[m|0] * sb[n|0] + bias[n] )
//
// Stands in for torch._scaled_mm and the manual post-scaling around it at
// lingua/float8.py:65-77 (forward: row x row scales, bias fused; dgrad: row x
// scalar scales) and serves the fp8 wgrad (row x row scales, reduction over
// tokens).
//
// Structure
//   * workgroup tile BM x BN, K consumed in tiles of 128 bytes (two
//     v_mfma_f32_32x32x64_f8f6f4 steps), WM x WN wavefronts, each owning
//     TM x TN accumulator tiles of 32x32;
//   * global -> LDS by `buffer_load_dwordx4 ... lds` (no staging registers).
//     Each row segment is a full 128-byte line: 64-byte segments halve the
//     L2 request rate that can be sustained (measured).  LDS is a ring of R
//     slots, each holding the A or the B panel of one K tile; units are
//     issued in the order A(0), B(0), A(1), ...  With R = 5 the ring holds the
//     K tile being read, the K tile being published and one more unit, so
//     loads stay in flight across every barrier; waits are partial
//     (`s_waitcnt vmcnt(n)`), one barrier per K tile;
//   * fragments are software-pipelined through two register sets: each half
//     of a trip runs the MFMAs of one 64-byte step while the next step is
//     read from LDS.  A wave issues in order, so the instruction stream is
//     laid out by hand as groups of one MFMA + its share of the LDS reads +
//     its share of the panel loads, with scheduling fences between groups:
//     one unit is requested during each half of a trip.  (Requesting both
//     units in a burst after the barrier left the waves queueing at the
//     vector-memory port with idle matrix cores: 2830 -> 2310 shader clocks
//     per trip, the matrix cores alone need 2048.);
//   * LDS rows are 128 bytes (8 chunks of 16 B); chunk c of row r lives at
//     position c ^ f(r), f(r) = (r & 7) ^ ((r >> 3) & 1): the 16-byte
//     fragment reads of any 16 consecutive rows then cover all 64 banks once
//     (SQ_LDS_BANK_CONFLICT = 0; f(r) = r & 7 alone measured 50 % conflict
//     cycles).  The permutation is applied on the global address side because
//     the LDS side of a direct load is lane-linear;
//   * the matrix cores compute the tile transposed (D[n][m]) so that each lane
//     ends up with 4 consecutive n per accumulator quad; a v_permlane32_swap
//     pairs lanes l / l+32 into 16 consecutive n.  The scaled, bf16-rounded
//     C tile is staged through the (by then idle) LDS ring and leaves as
//     whole rows, 1 KiB of consecutive bytes per wave store;
//   * workgroup -> tile mapping is XCD-aware: the 8 XCDs each get a contiguous
//     range of a grouped (GROUP_M tall) tile order so that the workgroups
//     resident on one XCD share A and B panels in that XCD's L2.
//
// L8_GEMM_DIAG (compile-time, never set in the shipped build) removes one side
// of the main loop to attribute stalls: 1 = no global loads after the prologue,
// 2 = no LDS reads / matrix-core work, 3 = no stores of C, 4 = as 2 with every workgroup loading the same tile (all
// L2 hits).  Results are wrong by construction.
#include <atomic>
#include <type_traits>

#include "l8_common.h"
#include "skinny.h"

namespace l8 {

struct GemmArgs {
  const uint8_t *A, *B;
  int M, N, K;
  int64_t lda, ldb, ldc;
  const float *sa, *sb;
  int sa_row, sb_row;
  const uint16_t *bias;
  uint16_t *C;
  int add;  // C = bf16(bf16(product) + C) instead of C = bf16(product): a sum of gradients without a pass of its own
  int tiles_m, tiles_n;
  uint64_t *dbg;  // L8_GEMM_PROF builds only
  // persistent kernels, optional (null = every tile is computed by one workgroup): workspace for tiles whose
  // K range is shared out over several workgroups -- one flag and one fp32 tile of partial sums per workgroup
  uint32_t *sk_flags;
  float *sk_partials;
  uint32_t sk_epoch;  // value that marks a flag as set in THIS launch (never 0; flags are never cleared)
  int sk_wait_limit;  // polls of a flag before the waiting workgroup gives up and poisons its tile
  // MULTI kernels: products with the same B, one below the other.  A, sa, C and M above are the first one's; a further one
  // starts at row `first` of the launch, a multiple of the tiles' BM, an unused one beyond the last.
  struct Part {
    const uint8_t *A;
    const float *sa;
    uint16_t *C;
    int first, M;
  } part[2];
  // SUM kernels: further products whose sum with the first one is C.  A, B, K, lda, ldb, sa (one per row) and sb (one) above
  // are the first one's.
  struct Term {
    const uint8_t *A, *B;
    const float *sa, *sb;
    int64_t lda, ldb;
    int K;
  } term[2];
  int terms;  // how many of them
};

typedef __attribute__((address_space(3))) void *lds_ptr_t;

// The buffer-resource type and the matrix-core builtins exist only in the
// device pass; the host pass sees empty kernel bodies (it needs the symbols only).

// 16-byte-per-lane buffer store with a scalar-register offset, followed by two wait states.  A vector-ALU write to
// one of the store's data registers right behind it can reach the register before the store has read it: with two
// waves per SIMD a form of the persistent kernel with eight waves stored, now and then, the next row pair's values in
// 4 of 64 lanes (found by the exact-integer tests; two wait states cure it, which is what the compiler's hazard recognizer inserts behind
// stores of more than 8 bytes -- except behind buffer stores whose soffset is a register, like these, which an old
// rule exempts).  Every such store in this file goes through here.
#if defined(__HIP_DEVICE_COMPILE__)
template <int AUX>
L8_DEV void store16_aux(v4i data, __amdgpu_buffer_rsrc_t rs, uint32_t voff, int soff) {
  __builtin_amdgcn_raw_buffer_store_b128(data, rs, voff, soff, AUX);
  asm volatile("s_nop 1" : : "v"(data));  // the operand keeps every later write to these registers behind the wait
}
#endif
#define store16(data, rs, voff, soff, aux) store16_aux<aux>(data, rs, voff, soff)

[[maybe_unused]] constexpr uint32_t kOOB = 0x80000000u;
// cache policy of a buffer access that must be coherent over the whole device (sc0 | sc1)
[[maybe_unused]] constexpr int kCoherent = 1 | 16;
// Sharing out the K range of the last, partly filled round of tiles: what a partial tile costs its writer and its
// reader, in K tiles' time (256 KiB leave a compute unit at ~16 bytes per clock), and the least number of K tiles
// the split must take off the owners of the tail tiles to be used at all.
[[maybe_unused]] constexpr int kSkWriteCost = 8, kSkFixCost = 4, kSkMinSaved = 16;
// Workspace layout: kSkMaxGrid flag words (one per tail-tile slot), then 64 words of which the first counts the
// tiles whose owner gave up waiting for a helper (and stored NaNs), then the fp32 tiles of partial sums.
[[maybe_unused]] constexpr int kSkMaxGridWords = 1024, kSkGaveUpWord = kSkMaxGridWords;

#ifndef L8_GEMM_DIAG
#define L8_GEMM_DIAG 0
#endif
#ifndef L8_STRADDLE
#define L8_STRADDLE 2
#endif
// groups (of one MFMA each) of the two halves of a trip over which the persistent kernel issues the half's LDS reads
#ifndef L8_READ_GROUPS1
#define L8_READ_GROUPS1 24
#endif
#ifndef L8_READ_GROUPS2
#define L8_READ_GROUPS2 30
#endif
// ... and the number of a half tile's 32 MFMAs in front of the barrier of a trip
#ifndef L8_HALF_TILE_BARRIER
#define L8_HALF_TILE_BARRIER 10
#endif
// L8_GEMM_PROF (compile-time, never set in the shipped build): the persistent kernel takes the `bias` pointer for
// a buffer of 16 x uint64 per workgroup and records wall-clock ticks (100 MHz) at its start, after the prologue
// and at its end, and shader-clock cycles spent in the K loops and in the C-tile stores.
#ifndef L8_GEMM_PROF
#define L8_GEMM_PROF 0
#endif

#if defined(__HIP_DEVICE_COMPILE__)
// Eight bf16 plus eight bf16, each sum rounded to nearest even: what PyTorch's add makes of two bf16 tensors.
L8_DEV v4i add_bf16x8(v4i a, v4i b) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  v4i r;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float lo = __uint_as_float((uint32_t)a[k] << 16) + __uint_as_float((uint32_t)b[k] << 16);
    const float hi = __uint_as_float((uint32_t)a[k] & 0xffff0000u) + __uint_as_float((uint32_t)b[k] & 0xffff0000u);
    const bf2 p = {(__bf16)lo, (__bf16)hi};
    r[k] = __builtin_bit_cast(int, p);
  }
  return r;
}
#endif

// s_waitcnt for vmcnt <= n and lgkmcnt == 0 (expcnt untouched)
#define L8_WAIT_VM_LGKM0(n) \
  __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (0x7 << 4) | (0x0 << 8) | ((((n) >> 4) & 0x3) << 14))

// R > 5, the small tiles: the deep form of the main loop.  The fragments of a whole K tile are in registers before its trip
// begins, read during the trip before; a slot is given away one trip later than above, when the MFMAs that used it have been
// issued, so that no wave waits for LDS at the barrier; and the ring holds as many whole K tiles as fit.  us, before (nine
// slots of one panel) / now: [2048,16384].[2048,16384] 65.3 / 60.2, [700,11008].[4096,11008] 40.7 / 37.7, [512,4096].[4096,4096]
// 15.0 / 13.9, [493,6784].[4832,6784] 26.8 / 24.8, [1021,2048].[2048,2048] 9.8 / 9.4, [333,2048].[8192,2048] 12.0 / 11.5.  What
// bounds them now is the way from the L2 to LDS: 33 to 38 bytes per clock and unit with every one of these tiles (and with
// the half tiles below), whatever the depth; touching the L2 two to ten K tiles ahead cost a tenth and gained nothing.
//
// s_waitcnt for vmcnt <= n alone
#define L8_WAIT_VM(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (0x7 << 4) | (0xF << 8) | ((((n) >> 4) & 0x3) << 14))

// Whole K tiles of a BM x BN problem that the LDS holds for each of KS groups of waves (six are enough).
constexpr int deep_slots(int bm, int bn, int ks) {
  const int n = 160 * 1024 / (ks * (bm + bn) * 128);
  return n < 6 ? n : 6;
}
constexpr int plain_lds(int bm, int bn, int r, int ks) { return ks * (r > 5 ? deep_slots(bm, bn, ks) * (bm + bn) : r * (bm > bn ? bm : bn)) * 128; }

// KS > 1: KS groups of WM x WN waves, each with a ring of its own, take K tiles in turn (group g the tiles g, g + KS, ..)
// and add their accumulators at the end, in the order of the groups.
template <int WM, int WN, int TM, int TN, int R, int GROUP_M, int PF, int KS = 1>
__global__ __launch_bounds__(WM *WN *KS * 64) void gemm_nt_kernel(const GemmArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int BM = WM * TM * 32, BN = WN * TN * 32, BK = 128;
  constexpr int NW = WM * WN;
  constexpr int A_BYTES = BM * BK, B_BYTES = BN * BK;
  constexpr int UNIT = A_BYTES > B_BYTES ? A_BYTES : B_BYTES;  // one ring slot holds an A or a B panel of one K tile
  constexpr bool DEEP = R > 5;
  constexpr int NS = deep_slots(BM, BN, KS), RING = DEEP ? NS * (A_BYTES + B_BYTES) : R * UNIT;  // of one group of waves
  static_assert((BM / 8) % NW == 0 && (BN / 8) % NW == 0, "tile rows must split evenly over waves");
  constexpr int NA = BM / 8 / NW, NB = BN / 8 / NW;  // 1 KiB wave loads (8 rows x 128 B) per panel per wave
  // L2 touches (PF > 0): one lane per panel row, every wave covers 64 rows per instruction
  constexpr int PFA = PF > 0 ? (BM + NW * 64 - 1) / (NW * 64) : 0, PFB = PF > 0 ? (BN + NW * 64 - 1) / (NW * 64) : 0;
  constexpr int IA = NA + PFA, IB = NB + PFB;  // vector-memory instructions per unit per wave
  // loads of the units that may still be in flight when a K tile is published:
  // the ring holds the tile being read (2 slots), the tile being published (2
  // slots) and R-4 younger units, the first of which is an A panel
  constexpr int PEND = ((R - 4 + 1) / 2) * IA + ((R - 4) / 2) * IB;
  constexpr int PEND0 = ((R - 3 + 1) / 2) * IA + ((R - 3) / 2) * IB;  // same for the prologue (R-3 younger units)
  static_assert(R >= 4 && PEND0 <= 63, "vmcnt is a 6-bit counter");
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];

  const int lane = threadIdx.x & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = KS > 1 ? wave_all / NW : 0, wave = KS > 1 ? wave_all % NW : wave_all;
  const int wm = wave / WN, wn = wave % WN;

  // ---- XCD-aware, grouped workgroup -> tile mapping ----
  int tile_m, tile_n, row_in_group;
  {
    const int nb = p.tiles_m * p.tiles_n;
    const int pid = blockIdx.x;
    const int q = nb >> 3, rem = nb & 7;
    const int xcd = pid & 7, loc = pid >> 3;
    const int lin = (xcd < rem) ? xcd * (q + 1) + loc : rem * (q + 1) + (xcd - rem) * q + loc;
    const int per_group = GROUP_M * p.tiles_n;
    const int grp = lin / per_group;
    const int first_m = grp * GROUP_M;
    const int gsz = (p.tiles_m - first_m < GROUP_M) ? p.tiles_m - first_m : GROUP_M;
    const int in_grp = lin - grp * per_group;
    row_in_group = in_grp % gsz;
    tile_m = first_m + row_in_group;
    tile_n = in_grp / gsz;
  }
  if (L8_GEMM_DIAG == 4) { tile_m = 0; tile_n = 0; }
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  // ---- global -> LDS load plan ----
  // lane l of a wave load fills LDS row l/8, position l%8 of an 8-row group;
  // position p of row r holds chunk p ^ f(r), f(r) = (r & 7) ^ ((r >> 3) & 1)
  const int lrow = lane >> 3, lpos = lane & 7;
  const uint8_t *Ablk = p.A + (int64_t)m0 * p.lda;
  const uint8_t *Bblk = p.B + (int64_t)n0 * p.ldb;
  const int64_t a_left = (int64_t)(p.M - m0 - 1) * p.lda + p.K;
  const int64_t b_left = (int64_t)(p.N - n0 - 1) * p.ldb + p.K;
  const __amdgpu_buffer_rsrc_t rsA = make_rsrc(Ablk, a_left < 0x7fffffff ? (uint32_t)a_left : 0x7fffffffu);
  const __amdgpu_buffer_rsrc_t rsB = make_rsrc(Bblk, b_left < 0x7fffffff ? (uint32_t)b_left : 0x7fffffffu);

  // Wave load j of a panel covers the 8 rows of group g = wave * N + j.  The
  // per-lane part of the address depends on the parity of g only (N is even, so
  // on the parity of j); the rest is scalar.  Rows beyond M / N need no test:
  // their offsets lie beyond the resource's range.
  static_assert(NA % 2 == 0 && NB % 2 == 0, "wave loads per panel must be even");
  const uint32_t a_voff[2] = {(uint32_t)(lrow * (int)p.lda + (lpos ^ lrow) * 16), (uint32_t)(lrow * (int)p.lda + (lpos ^ lrow ^ 1) * 16)};
  const uint32_t b_voff[2] = {(uint32_t)(lrow * (int)p.ldb + (lpos ^ lrow) * 16), (uint32_t)(lrow * (int)p.ldb + (lpos ^ lrow ^ 1) * 16)};
  const int a_lda8 = 8 * (int)p.lda, b_ldb8 = 8 * (int)p.ldb;
  const int a_srow = wave * NA * a_lda8, b_srow = wave * NB * b_ldb8;
  // L2 touches.  The 32 workgroups resident on an XCD form a GROUP_M x (32 / GROUP_M)
  // block of tiles: 32 / GROUP_M of them stream the same A panel and GROUP_M the
  // same B panel.  Each workgroup touches (one dword per 128-byte line) only its
  // share of the rows of the K tile PF trips ahead, so that the line is in the
  // XCD's L2 when the panel loads of all the sharers ask for it.
  uint32_t pfa_voff[PFA > 0 ? PFA : 1], pfb_voff[PFB > 0 ? PFB : 1];
  if constexpr (PF > 0) {
    constexpr int SA = 32 / GROUP_M >= 1 ? 32 / GROUP_M : 1, SB = GROUP_M;
    const int slice_a = tile_n % SA, slice_b = row_in_group % SB;
#pragma unroll
    for (int i = 0; i < PFA; ++i) {
      const int row = (i * NW + wave) * 64 + lane;
      pfa_voff[i] = (row < BM && row % SA == slice_a && m0 + row < p.M) ? (uint32_t)(row * (int)p.lda) : kOOB;
    }
#pragma unroll
    for (int i = 0; i < PFB; ++i) {
      const int row = (i * NW + wave) * 64 + lane;
      pfb_voff[i] = (row < BN && row % SB == slice_b && n0 + row < p.N) ? (uint32_t)(row * (int)p.ldb) : kOOB;
    }
  }
  const int chunk_even = (lpos ^ lrow) * 16, chunk_odd = (lpos ^ lrow ^ 1) * 16;  // byte offset in the row, by parity of g

  // ---- scales and bias ----
  // The small tiles request them in front of their panels: loads retire in order, so they are there when the K loop starts,
  // and the partial waits below count as before.  Requested behind the loop, with a branch around each load, a product of a
  // few microseconds ended in the latency of loads that wait for one another.  us, operands cold, before / now: [1021,2048].
  // [2048,2048] with a bias 12.4 / 9.6, without 9.8 / 9.3; [32,4096].[11008,4096] 16.1 / 14.1 and 14.6 / 14.1; [128,1024].
  // [1024,1024] without 5.8 / 5.3.  Two 128 x 128 workgroups on a unit cover for each other: there the registers are worth more
  // (requested early [64,4096].[36864,4096] 46.4 -> 46.9).
  constexpr bool EARLY = DEEP;
  const int l31 = lane & 31, h = lane >> 5;
  float sav[TM], sb_all;
  float sbv[TN][4][4];  // of the 16 n per 32-column tile that this lane holds before the half-wave swap
  v2i biasv[TN][4];
  const bool bias_vec = p.bias && ((uintptr_t)p.bias & 7) == 0 && p.N % 2 == 0;  // whole dwords up to column N
  auto scales = [&]() __attribute__((always_inline)) {
    const int m_left = p.M - m0 < BM ? p.M - m0 : BM, n_left = p.N - n0 < BN ? p.N - n0 : BN;
    const __amdgpu_buffer_rsrc_t rsSa = make_rsrc(p.sa + (p.sa_row ? m0 : 0), p.sa_row ? m_left * 4 : 4);
    const __amdgpu_buffer_rsrc_t rsSb = make_rsrc(p.sb + (p.sb_row ? n0 : 0), p.sb_row ? n_left * 4 : 4);
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
      sav[tm] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsSa, p.sa_row ? ((wm * TM + tm) * 32 + l31) * 4 : 0, 0, 0));
    sb_all = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsSb, 0, 0, 0));  // the one scale, if it is one
#pragma unroll
    for (int i = 0; i < TN * 4; ++i) {
      const v4i t = __builtin_amdgcn_raw_buffer_load_b128(rsSb, ((wn * TN + i / 4) * 32 + 8 * (i % 4) + 4 * h) * 4, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) sbv[i / 4][i % 4][e] = __uint_as_float((uint32_t)t[e]);
    }
    if (bias_vec) {
      const __amdgpu_buffer_rsrc_t rsBias = make_rsrc(p.bias + n0, n_left * 2);
#pragma unroll
      for (int i = 0; i < TN * 4; ++i)
        biasv[i / 4][i % 4] = __builtin_amdgcn_raw_buffer_load_b64(rsBias, ((wn * TN + i / 4) * 32 + 8 * (i % 4) + 4 * h) * 2, 0, 0);
    }
  };
  if constexpr (EARLY) {
    if (group == 0) scales();
    asm volatile("" ::: "memory");
  }

  const int KT = (p.K + BK * KS - 1) / (BK * KS);  // trips
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)smem + group * RING;
  auto wrap = [](int slot) { return slot >= R ? slot - R : slot; };  // slot in [0, 2R)
  // Units are issued in the order A(0), B(0), A(1), B(1), ...; unit u lives in
  // ring slot u % R (the callers keep the slot numbers as running scalars).
  // Every unit issues its full count of loads so that the vmcnt arithmetic is
  // uniform; K tiles at or beyond the end, rows beyond M / N and chunks beyond
  // K use an out-of-range offset, which the buffer unit turns into zeros in LDS.
  // load_one: i-th vector-memory instruction (of IA or IB) of the unit of K
  // tile kt (A or B panel) to LDS offset `at`: first the L2 touches, then
  // the 1 KiB panel loads.
  auto load_one = [&](bool is_b, int kt, int at, int i) {
    const int k0 = (kt * KS + group) * BK;
    const uint32_t m_even = (k0 + chunk_even < p.K) ? 0u : kOOB, m_odd = (k0 + chunk_odd < p.K) ? 0u : kOOB;
    if (!is_b) {
      const uint32_t dst = lds0 + at + wave * (NA * 1024);
      // a touched dword lands in this wave's own part of the slot and is
      // overwritten by the panel loads that follow (a wave's loads return in order)
      if (i < PFA)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsA, reinterpret_cast<lds_ptr_t>(dst), 4,
                                                 pfa_voff[i < PFA ? i : 0] | ((k0 + PF * KS * BK < p.K) ? 0u : kOOB), k0 + PF * KS * BK, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsA, reinterpret_cast<lds_ptr_t>(dst + (i - PFA) * 1024), 16,
                                                 a_voff[(i - PFA) & 1] | (((i - PFA) & 1) ? m_odd : m_even),
                                                 k0 + a_srow + (i - PFA) * a_lda8, 0, 0);
    } else {
      const uint32_t dst = lds0 + at + wave * (NB * 1024);
      if (i < PFB)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsB, reinterpret_cast<lds_ptr_t>(dst), 4,
                                                 pfb_voff[i < PFB ? i : 0] | ((k0 + PF * KS * BK < p.K) ? 0u : kOOB), k0 + PF * KS * BK, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsB, reinterpret_cast<lds_ptr_t>(dst + (i - PFB) * 1024), 16,
                                                 b_voff[(i - PFB) & 1] | (((i - PFB) & 1) ? m_odd : m_even),
                                                 k0 + b_srow + (i - PFB) * b_ldb8, 0, 0);
    }
  };

  // ---- LDS -> register fragment plan ----
  const int fr = (l31 & 7) ^ ((l31 >> 3) & 1);
  uint32_t foff[2][2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int j = 0; j < 2; ++j) foff[s][j] = l31 * BK + (((s * 4 + h * 2 + j) ^ fr) * 16);
  const int a_base = wm * (TM * 32 * BK);
  const int b_base = wn * (TN * 32 * BK);

  // LDS addresses of the two 16-byte pieces a lane reads of its row, for step s
  // of the K tile whose panels sit at LDS offsets at_a / at_b.  The additions are
  // opaque to the compiler on purpose: it would otherwise keep a register per
  // (slot, piece) combination alive across the loop.
  typedef const __attribute__((address_space(3))) v4i *lds_v4i_ptr;
  auto frag_addrs = [&](int at_a, int at_b, int s, uint32_t (&ad)[4]) {
    const uint32_t sa = lds0 + at_a + a_base, sb = lds0 + at_b + b_base;
    asm volatile("v_add_u32 %0, %1, %2" : "=v"(ad[0]) : "s"(sa), "v"(foff[s][0]));
    asm volatile("v_add_u32 %0, %1, %2" : "=v"(ad[1]) : "s"(sa), "v"(foff[s][1]));
    asm volatile("v_add_u32 %0, %1, %2" : "=v"(ad[2]) : "s"(sb), "v"(foff[s][0]));
    asm volatile("v_add_u32 %0, %1, %2" : "=v"(ad[3]) : "s"(sb), "v"(foff[s][1]));
  };
  // fragment f, in the order the MFMAs need them: B0, A0 .. A(TM-1), B1 ..
  auto read_one = [&](const uint32_t (&ad)[4], v8i (&af)[TM], v8i (&bf)[TN], int f) {
    const bool is_b = f == 0 || f > TM;
    const int t = f == 0 ? 0 : (f > TM ? f - TM : f - 1);
    const v4i lo = *reinterpret_cast<lds_v4i_ptr>(ad[is_b ? 2 : 0] + t * (32 * BK));
    const v4i hi = *reinterpret_cast<lds_v4i_ptr>(ad[is_b ? 3 : 1] + t * (32 * BK));
    const v8i v = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    if (is_b) bf[t] = v;
    else af[t] = v;
  };

  v16f acc[TN][TM];
#pragma unroll
  for (int tn = 0; tn < TN; ++tn)
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[tn][tm][v] = 0.0f;

  // MFMA number idx (of TM*TN) of one 64-byte step
  auto mma_one = [&](v8i (&af)[TM], v8i (&bf)[TN], int idx) {
    const int tn = idx / TM, tm = idx % TM;
    // D[i = n][j = m]: B rows feed the "A" port, A rows the "B" port
    acc[tn][tm] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bf[tn], af[tm], acc[tn][tm], 0, 0, 0, 0, 0, 0);
  };

  // The loads of one trip are two units.  The first is spread over the MFMAs of
  // the first half, the second over those of the second half: a burst of all
  // of them after the barrier would keep the waves queueing at the
  // vector-memory port instead of issuing MFMAs.
  //   prologue: units 0 .. R-2 in flight, K tile 0 published, its first half read
  if constexpr (DEEP) {
    // Trip kt: K tile kt + 1 has landed for every wave behind the barrier (a partial wait for its own loads in front of it);
    // MFMAs on K tile kt, whose fragments were requested in the trip before, beside the reads of kt + 1 and the loads of
    // kt + NS - 1, which go where kt - 1 was: every wave has issued the MFMAs of kt - 1, so its reads are done.
    constexpr int KTILE = A_BYTES + B_BYTES, LOADS = IA + IB, N_MMA = 2 * TM * TN, N_RD = 4 * (TM + TN);
    constexpr int PEND_D = (NS - 3) * LOADS;
    static_assert(NS >= 4 && (NS - 2) * LOADS <= 63, "vmcnt is a 6-bit counter");
    struct Frags { v8i a[2][TM], b[2][TN]; };
    auto slot_after = [](int slot, int n) { return slot + n >= NS ? slot + n - NS : slot + n; };
    auto load_tile_part = [&](int kt, int slot, int j) {
      if (j < IA) load_one(false, kt, slot * KTILE, j);
      else load_one(true, kt, slot * KTILE + A_BYTES, j - IA);
    };
    // piece r of a K tile's fragments: step by step, in the order the MFMAs need them
    auto read_part = [&](const uint32_t (&ad)[2][4], Frags &f, int r) __attribute__((always_inline)) {
      const int step = r / (2 * (TM + TN)), q = (r % (2 * (TM + TN))) >> 1, h = r & 1;
      const bool is_b = q == 0 || q > TM;
      const int t = q == 0 ? 0 : (q > TM ? q - TM : q - 1);
      const v4i v = *reinterpret_cast<lds_v4i_ptr>(ad[step][(is_b ? 2 : 0) + h] + t * (32 * BK));
      v8i &d = is_b ? f.b[step][t] : f.a[step][t];
#pragma unroll
      for (int k = 0; k < 4; ++k) d[h * 4 + k] = v[k];
    };
    Frags f0, f1;
    uint32_t ad[2][4];
#pragma unroll
    for (int u = 0; u < NS - 1; ++u)
#pragma unroll
      for (int j = 0; j < LOADS; ++j) load_tile_part(u, u, j);
    L8_WAIT_VM((NS - 2) * LOADS);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    frag_addrs(0, A_BYTES, 0, ad[0]);
    frag_addrs(0, A_BYTES, 1, ad[1]);
#pragma unroll
    for (int r = 0; r < N_RD; ++r) read_part(ad, f0, r);
    int slot = 0;  // of K tile kt
    auto trip = [&](int kt, Frags &cur, Frags &nxt) __attribute__((always_inline)) {
      L8_WAIT_VM(PEND_D);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const int next = slot_after(slot, 1), free = slot_after(slot, NS - 1);
      frag_addrs(next * KTILE, next * KTILE + A_BYTES, 0, ad[0]);
      frag_addrs(next * KTILE, next * KTILE + A_BYTES, 1, ad[1]);
#pragma unroll
      for (int i = 0; i < N_MMA; ++i) {
        mma_one(cur.a[i / (TM * TN)], cur.b[i / (TM * TN)], i % (TM * TN));
#pragma unroll
        for (int r = (N_RD * i) / N_MMA; r < (N_RD * (i + 1)) / N_MMA; ++r) read_part(ad, nxt, r);
#pragma unroll
        for (int j = (LOADS * i) / N_MMA; j < (LOADS * (i + 1)) / N_MMA; ++j) load_tile_part(kt + NS - 1, free, j);
        __builtin_amdgcn_sched_barrier(0);
      }
      slot = next;
    };
    int kt = 0;
#pragma unroll 1
    for (; kt + 2 <= KT; kt += 2) {
      trip(kt, f0, f1);
      trip(kt + 1, f1, f0);
    }
    if (kt < KT) trip(kt, f0, f1);
  } else {
#pragma unroll
  for (int u = 0; u < R - 1; ++u) {
#pragma unroll
    for (int i = 0; i < ((u & 1) ? IB : IA); ++i) load_one(u & 1, u >> 1, u * UNIT, i);
  }
  v8i af0[TM], bf0[TN], af1[TM], bf1[TN];
  uint32_t ad[4];
  L8_WAIT_VM_LGKM0(PEND0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  frag_addrs(0, UNIT, 0, ad);
#pragma unroll
  for (int f = 0; f < TM + TN; ++f) read_one(ad, af0, bf0, f);

  // One trip = one K tile of 128 = two matrix-core steps of 64.
  //   first half : MFMAs on (kt, step 0) while (kt, step 1) is read from LDS and
  //                unit 2kt+R-1 is requested (its slot, of K tile kt-1, was
  //                released at the previous barrier);
  //   barrier    : every wave has now read all of K tile kt (lgkmcnt 0), and
  //                K tile kt+1 has landed for every wave (partial vmcnt wait);
  //   second half: MFMAs on (kt, step 1) while (kt+1, step 0) is read and unit
  //                2kt+R is requested into the slot K tile kt just released.
  // Each group below is one MFMA plus its share of the LDS reads and of the
  // loads; the scheduling fences keep the groups in this order.
  constexpr int N_MMA = TM * TN, NF = TM + TN;
  constexpr int STRADDLE = L8_STRADDLE < N_MMA - 2 ? L8_STRADDLE : 0;
  constexpr int S1 = N_MMA - STRADDLE;  // MFMA groups before the barrier
  constexpr int S2 = N_MMA + STRADDLE;  // and after it
  constexpr int SR = N_MMA > 2 ? N_MMA - 2 : N_MMA;  // the last two groups of a trip are left without reads
  constexpr bool U1_IS_B = ((R - 1) & 1) != 0, U2_IS_B = (R & 1) != 0;  // panel kind of units 2kt+R-1 and 2kt+R
  constexpr int I1 = U1_IS_B ? IB : IA, I2 = U2_IS_B ? IB : IA;
  int s0 = 0;  // ring slot of unit 2kt
  for (int kt = 0; kt < KT; ++kt) {
    const int slot_u1 = wrap(s0 + R - 1);  // unit 2kt+R-1 reuses the slot of unit 2kt-1
    frag_addrs(s0 * UNIT, wrap(s0 + 1) * UNIT, 1, ad);
#pragma unroll
    for (int i = 0; i < S1; ++i) {
      if (L8_GEMM_DIAG != 2 && L8_GEMM_DIAG != 4) {
        mma_one(af0, bf0, i);
#pragma unroll
        for (int f = (NF * i) / S1; f < (NF * (i + 1)) / S1; ++f) read_one(ad, af1, bf1, f);
      }
      if (L8_GEMM_DIAG != 1) {
#pragma unroll
        for (int j = (I1 * i) / S1; j < (I1 * (i + 1)) / S1; ++j) load_one(U1_IS_B, kt + (R - 1) / 2, slot_u1 * UNIT, j);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    L8_WAIT_VM_LGKM0(PEND);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // the last MFMAs of the first half are issued after the barrier: they need
    // registers only and keep the matrix cores busy while the waves regroup
    frag_addrs(wrap(s0 + 2) * UNIT, wrap(s0 + 3) * UNIT, 0, ad);
#pragma unroll
    for (int i = 0; i < S2; ++i) {
      if (L8_GEMM_DIAG != 2 && L8_GEMM_DIAG != 4) {
        if (i < STRADDLE) mma_one(af0, bf0, S1 + i);
        else mma_one(af1, bf1, i - STRADDLE);
        if (i >= STRADDLE) {  // (kt+1, step 0) replaces the fragments the straddling MFMAs have just consumed
#pragma unroll
          for (int f = (NF * (i - STRADDLE)) / SR; f < (NF * (i - STRADDLE + 1)) / SR && f < NF; ++f) read_one(ad, af0, bf0, f);
        }
      }
      if (L8_GEMM_DIAG != 1) {
#pragma unroll
        for (int j = (I2 * i) / S2; j < (I2 * (i + 1)) / S2; ++j) load_one(U2_IS_B, kt + R / 2, s0 * UNIT, j);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    s0 = wrap(s0 + 2);
  }
  }
  // ---- epilogue ----
  if constexpr (!EARLY) scales();  // one memory latency, under the wait that drains the ring
  if (!p.sb_row) {
#pragma unroll
    for (int i = 0; i < TN * 16; ++i) sbv[i / 16][i / 4 % 4][i % 4] = sb_all;
  }
  if (p.bias && !bias_vec) {  // element by element
    const __amdgpu_buffer_rsrc_t rsBias = make_rsrc(p.bias + n0, (p.N - n0 < BN ? p.N - n0 : BN) * 2);
#pragma unroll
    for (int i = 0; i < TN * 4; ++i) {
      uint32_t b[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        b[e] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rsBias, ((wn * TN + i / 4) * 32 + 8 * (i % 4) + 4 * h + e) * 2, 0, 0);
      biasv[i / 4][i % 4] = v2i{(int)(b[0] | b[1] << 16), (int)(b[2] | b[3] << 16)};
    }
  }
  // every wave's tail loads (out of range, zero-filling) and LDS reads are done
  // before the ring is reused as the staging area of the C tile
  L8_WAIT_VM_LGKM0(0);
  __builtin_amdgcn_s_barrier();
  if constexpr (KS > 1) {
    // every group's ring is idle: the others leave their sums in theirs, the first group adds them to its own
    static_assert(BM * BN * 4 <= RING, "a group's sums must fit in its ring");
    typedef __attribute__((address_space(3))) v4f *lds_v4f_ptr;
    constexpr int PIECE = NW * 64 * 16;
    const uint32_t mine = lds0 + (wave * 64 + lane) * 16;
    if (group > 0) {
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
          for (int qd = 0; qd < 4; ++qd)
            *reinterpret_cast<lds_v4f_ptr>(mine + ((tn * TM + tm) * 4 + qd) * PIECE) =
                v4f{acc[tn][tm][qd * 4], acc[tn][tm][qd * 4 + 1], acc[tn][tm][qd * 4 + 2], acc[tn][tm][qd * 4 + 3]};
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (group == 0) {
#pragma unroll
      for (int g = 1; g < KS; ++g)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
#pragma unroll
          for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
              const v4f t = *reinterpret_cast<lds_v4f_ptr>(mine + g * RING + ((tn * TM + tm) * 4 + qd) * PIECE);
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[tn][tm][qd * 4 + e] += t[e];
            }
    }
  }

  // lane (l31, h) of tile (tn, tm) holds m = l31 and, in accumulator quad qd,
  // n = 8*qd + 4*h + {0..3}.  After the half-wave swap, lanes with h == 0 hold
  // n = 0..15 and lanes with h == 1 hold n = 16..31 of row m: 32 bytes of bf16.
  // Stored from there, every store instruction would scatter 16-byte pieces
  // over 32 rows.  The tile goes through LDS instead (rows padded by 16 bytes
  // so that the 16 lanes of a write phase hit 16 different bank groups) and
  // leaves as whole rows: one store instruction covers 1 KiB of consecutive
  // bytes of C per row pair.
  constexpr int C_ROW = BN * 2 + 16;  // staged row pitch in bytes
  static_assert(BM * C_ROW <= KS * RING, "the C tile must fit in the ring");
  typedef __attribute__((address_space(3))) v4i *lds_v4i_wptr;
  auto convert_and_stage = [&](auto has_bias) {
    constexpr bool HAS_BIAS = decltype(has_bias)::value;
#pragma unroll
  for (int tn = 0; tn < TN; ++tn) {
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      const float sa = sav[tm];
      uint32_t pk[8];  // quad qd -> pk[2qd], pk[2qd+1]
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = acc[tn][tm][qd * 4 + e] * sa * sbv[tn][qd][e];
          if constexpr (HAS_BIAS) v[e] += bf16_bits_to_f32(((uint32_t)biasv[tn][qd][e >> 1] >> (16 * (e & 1))) & 0xffffu);
        }
        typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
        bf2 lo = {(__bf16)v[0], (__bf16)v[1]}, hi = {(__bf16)v[2], (__bf16)v[3]};
        pk[2 * qd] = __builtin_bit_cast(uint32_t, lo);
        pk[2 * qd + 1] = __builtin_bit_cast(uint32_t, hi);
      }
      // swap: (quad0 of upper lanes) <-> (quad2 of lower lanes); (quad1 upper) <-> (quad3 lower)
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        auto r0 = __builtin_amdgcn_permlane32_swap(pk[0 + d], pk[4 + d], false, false);
        pk[0 + d] = r0[0];
        pk[4 + d] = r0[1];
        auto r1 = __builtin_amdgcn_permlane32_swap(pk[2 + d], pk[6 + d], false, false);
        pk[2 + d] = r1[0];
        pk[6 + d] = r1[1];
      }
      // lower lanes: pk[0,1]=n0..3 pk[4,5]=n4..7 pk[2,3]=n8..11 pk[6,7]=n12..15
      // upper lanes: pk[0,1]=n16..19 pk[4,5]=n20..23 pk[2,3]=n24..27 pk[6,7]=n28..31
      const uint32_t at = lds0 + ((wm * TM + tm) * 32 + l31) * C_ROW + ((wn * TN + tn) * 32 + 16 * h) * 2;
      *reinterpret_cast<lds_v4i_wptr>(at) = v4i{(int)pk[0], (int)pk[1], (int)pk[4], (int)pk[5]};
      *reinterpret_cast<lds_v4i_wptr>(at + 16) = v4i{(int)pk[2], (int)pk[3], (int)pk[6], (int)pk[7]};
    }
  }
  };
  if (group == 0) {
    if (p.bias) convert_and_stage(std::true_type{});
    else convert_and_stage(std::false_type{});
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's part of the tile is in LDS
  __builtin_amdgcn_s_barrier();
  if (group > 0) return;
  // 16-byte chunk c of the tile: row c / CPR, columns 8 * (c % CPR) .. +7
  constexpr int CPR = BN / 8, CHUNKS = BM * CPR;
  static_assert(CHUNKS % (NW * 64) == 0, "whole wave stores");
  const bool c_vec = (p.ldc % 8 == 0) && (((uintptr_t)p.C & 15) == 0);
  constexpr int ITERS = CHUNKS / (NW * 64), ROWS_PER_IT = NW * 64 / CPR;
  static_assert((NW * 64) % CPR == 0, "a wave store covers whole rows");
  const int row0 = (wave * 64 + lane) / CPR, col = ((wave * 64 + lane) % CPR) * 8;
  if (c_vec && m0 + BM <= p.M && n0 + BN <= p.N && L8_GEMM_DIAG != 3) {
    // interior tile: no masks, one pointer and one LDS address stepped by constants; streaming stores, so
    // that the C tile on its way out does not push the operand panels out of the L2
    uint16_t *dst = p.C + (int64_t)(m0 + row0) * p.ldc + n0 + col;
    const uint32_t at = lds0 + row0 * C_ROW + col * 2;
    if (p.add) {
#pragma unroll 8
      for (int it = 0; it < ITERS; ++it) {
        v4i *at_c = (v4i *)(dst + (int64_t)it * ROWS_PER_IT * p.ldc);
        __builtin_nontemporal_store(add_bf16x8(*reinterpret_cast<lds_v4i_ptr>(at + it * (ROWS_PER_IT * C_ROW)), __builtin_nontemporal_load(at_c)), at_c);
      }
      return;
    }
#pragma unroll
    for (int it = 0; it < ITERS; ++it)
      __builtin_nontemporal_store(*reinterpret_cast<lds_v4i_ptr>(at + it * (ROWS_PER_IT * C_ROW)),
                                  (v4i *)(dst + (int64_t)it * ROWS_PER_IT * p.ldc));
  } else if (L8_GEMM_DIAG != 3) {
#pragma unroll 4
    for (int it = 0; it < ITERS; ++it) {
      const int row = row0 + it * ROWS_PER_IT;
      const v4i v = *reinterpret_cast<lds_v4i_ptr>(lds0 + row * C_ROW + col * 2);
      const int m = m0 + row, n = n0 + col;
      if (m < p.M && n < p.N) {
        uint16_t *dst = p.C + (int64_t)m * p.ldc + n;
        if (c_vec && n + 8 <= p.N) {
          __builtin_nontemporal_store(p.add ? add_bf16x8(v, *(const v4i *)dst) : v, (v4i *)dst);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (n + e < p.N) {
              const uint32_t h = ((uint32_t)v[e >> 1] >> (16 * (e & 1))) & 0xffffu;
              dst[e] = p.add ? (uint16_t)bf16_rne_bits(bf16_bits_to_f32(h) + bf16_bits_to_f32(dst[e])) : (uint16_t)h;
            }
        }
      }
    }
  }
#else
  (void)p;
#endif
}

// ---------------------------------------------------------------------------
// Persistent variant for large problems: one workgroup per compute unit walks a
// list of 256x256 tiles, and the panel stream (global -> LDS ring) runs on
// from the last K tile of one output tile into the first K tiles of the next,
// so that only the very first tile of a workgroup pays a prologue.
//
// The C tile leaves straight from the accumulators, with no staging in LDS
// (the ring stays in use by the panel stream) and no barrier:
//   * the matrix cores compute D[i = m][j = n'] (A rows on the first port) in
//     tiles of 16x16;
//   * LDS row tn*16 + j of a wave's 128-row span of the B panel holds the
//     global B row 8*j + tn of that span (the permutation is applied on the
//     global-address side of the direct-to-LDS loads, which is free), so that
//     lane j owns, at the same accumulator index of its eight tn tiles, the
//     eight CONSECUTIVE output columns 8*j .. 8*j+7: 16 bytes of a C row, and
//     one 16-byte store per lane covers 256 contiguous bytes of a row per 16
//     lanes (four rows per wave instruction, whole 128-byte lines).
//
// The instruction is v_mfma_f32_16x16x128_f8f6f4, not 32x32x64: the same flop
// per cycle for less power, and power is what sets this kernel's clock.  Matrix
// instructions back to back on random operands, no memory traffic: 4.27 PFLOP/s
// at 2.16 GHz against 3.98 at 1.97 (both 4.96 at 2.40 on zeros).  A K tile of
// 128 bytes is then ONE step of 64 instructions, row by row of the wave's 8 x 8
// tiles: the eight B fragments stay for the whole step, an A fragment for the
// eight instructions of its row.
// us, one launch behind the other on one box, 32x32x64 / this: [16384,11008] K =
// 4096 502 / 490, [16384,4096] K = 11008 476 / 463, [11008,4096] K = 16384 500 /
// 480, [16384,2048] K = 8192 187 / 180, [32768,8192] K = 2048 398 / 386.  A K tile
// takes 2260 to 2310 cycles of the 2048 that its instructions need (2120 to 2190
// before: a 32-cycle instruction hides less of what stands between two of them),
// a C tile 5800 to 6300 (6700 before: no exchange of column groups between
// lanes), at 1.6 to 1.85 GHz.  Cycles are not what bounds it: variants of the
// loop's layout from 2260 to 2380 cycles took the same time, one of 3500 cycles
// 20 % more.  Without the panel loads it runs at 2.2 GHz: they are the largest
// consumer beside the matrix cores.
//
// BM x BN = 256 x 128 and 128 x 256 are half tiles for problems that whole ones
// would spread over few units or an unlucky number of rounds.  A trip is 32
// instructions per wave and wants 48 KiB through the L2 where a whole tile's 64
// instructions want 64: it takes 1270 to 1360 cycles of the 1024 of its
// instructions, 1075 without the panel loads.  The ring holds three whole K tiles,
// and the barrier stands after the tenth instruction so that the 24 LDS reads of
// a trip spread evenly (after the sixteenth: 1300 to 1385 cycles).
// Work split: the tiles are dealt to the 8 XCDs in contiguous ranges of the
// grouped order (as in the kernel above); inside an XCD, workgroup `loc`
// takes tiles loc, loc + W, loc + 2W, ... of the range (W workgroups per XCD),
// so the workgroups resident on an XCD always work on W consecutive tiles of
// the grouped order and share their panels in that XCD's L2.
// ---------------------------------------------------------------------------
// ADD: the bf16 tile is added to what C holds (two gradients of one activation) in the epilogue.  The C values are
// requested C_AHEAD row groups before they are used: the counter retires in order, so the wait for them is also one for the
// stores issued before they were requested, and those have had that long.
//
// MULTI: up to three products with one B (the weight gradients of linears on one activation) as one list of tiles.  On its
// own [2048,16384].[2048,16384]^T has 64 tiles of 256 x 256, too few for this kernel, and [11008,4096] leaves a third of the
// units without work in its last round; together they fill the rounds.
//
// SUM: C = A0.B0^T + A1.B1^T (+ A2.B2^T), each with row scales for A and one scale for B (the gradient of an activation that
// several linears read), as one K loop over all of them: the stream of panels runs on from the last K tile of one product
// into the first of the next.  The accumulators hold multiples of the present product's scale, so at a change of products
// they are multiplied by the quotient of the old one and the new, row by row, under the matrix instructions of the new
// product's first K tile (768 vector instructions beside its 64: 2.5 us per change of two rounds of tiles).  C is rounded and
// written once, where ADD reads it back and rounds it per product.
//
// A sum of products is below 2^33 units and no finer than 2^-18, so units within 2^90 of one another keep what the
// accumulators hold between 2^-108 and 2^125, however often they are rescaled.  A row whose units lie further apart (or beyond
// fp32's normal numbers) would overflow on the way or lose a product that is alone in its column: such rows are computed
// again behind the loop, product by product, each rounded and added as l8_gemm_nt_add does: there no accumulators are live
// (a second conversion of the tile beside the first spills 250 registers).  Looking at the units costs a launch 0.3 .. 0.5 us:
// 2 x [16384,2048] K = 512 38.1 -> 38.6, 3 x [16384,2048] K = 2048 140.8 -> 141.4.  (Rows with a scale that is infinite or NaN
// stay: the casts give such a scale to rows whose every product is NaN.)
#if defined(__HIP_DEVICE_COMPILE__)
L8_DEV bool units_apart(float a, float b, float c) {
  const float least = fminf(fminf(fabsf(a), fabsf(b)), fabsf(c)), largest = fmaxf(fmaxf(fabsf(a), fabsf(b)), fabsf(c));
  return !(least >= 0x1p-126f && largest < INFINITY && largest <= least * 0x1p90f);
}

// 16 rows from m on, 128 columns from n on, of a sum of products, the rows with units far apart alone: one wave, operands
// straight from memory.  The instruction and the order of K are those of the kernel below.
L8_DEV void sum_rows_one_by_one(const GemmArgs &p, int m, int n) {
  int lane = threadIdx.x & 63;
  const int l15 = lane & 15, quad = lane >> 4;
  const float sb[3] = {p.sb[0], p.term[0].sb[0], p.terms > 1 ? p.term[1].sb[0] : p.sb[0]};  // (two products at least)
  float sa[4][3];
  bool redo[4], any = false;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = m + 4 * quad + e;
    const int at = row < p.M ? row : p.M - 1;
    redo[e] = row < p.M;
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      sa[e][t] = t == 0 ? p.sa[at] : t <= p.terms ? p.term[t ? t - 1 : 0].sa[at] : sa[e][0];
      redo[e] = redo[e] && fabsf(sa[e][t]) < INFINITY && fabsf(sb[t]) < INFINITY;
    }
    redo[e] = redo[e] && units_apart(sa[e][0] * sb[0], sa[e][1] * sb[1], sa[e][2] * sb[2]);
    any |= redo[e];
  }
  if (__ballot(any) == 0) return;
#pragma unroll 1
  for (int c = n; c < n + 128 && c < p.N; c += 16) {
    v4f sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
    for (int t = 0; t <= p.terms; ++t) {
      const uint8_t *A = t == 0 ? p.A : p.term[t - 1].A, *B = t == 0 ? p.B : p.term[t - 1].B;
      const int64_t lda = t == 0 ? p.lda : p.term[t - 1].lda, ldb = t == 0 ? p.ldb : p.term[t - 1].ldb;
      const int K = t == 0 ? p.K : p.term[t - 1].K;
      // rows at or beyond M (N) start beyond the descriptor's end and read as zeros
      const int64_t a_left = (int64_t)(p.M - m - 1) * lda + K, b_left = (int64_t)(p.N - c - 1) * ldb + K;
      const __amdgpu_buffer_rsrc_t rsA = make_rsrc(A + (int64_t)m * lda, a_left < 0x7fffffff ? (uint32_t)a_left : 0x7fffffffu);
      const __amdgpu_buffer_rsrc_t rsB = make_rsrc(B + (int64_t)c * ldb, b_left < 0x7fffffff ? (uint32_t)b_left : 0x7fffffffu);
      v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
      for (int k0 = 0; k0 < K; k0 += 128) {
        v8i a, b;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k = k0 + quad * 32 + h * 16;  // K is a multiple of 16
          const v4i va = __builtin_amdgcn_raw_buffer_load_b128(rsA, k < K ? l15 * (int)lda + k : (int)kOOB, 0, 0);
          const v4i vb = __builtin_amdgcn_raw_buffer_load_b128(rsB, k < K ? l15 * (int)ldb + k : (int)kOOB, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) a[h * 4 + i] = va[i], b[h * 4 + i] = vb[i];
        }
        acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, acc, 0, 0, 0, 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = t == 0 ? sa[e][0] : t == 1 ? sa[e][1] : sa[e][2], b = t == 0 ? sb[0] : t == 1 ? sb[1] : sb[2];
        const float part = (float)(__bf16)(acc[e] * (a * b));
        sum[e] = t == 0 ? part : (float)(__bf16)(sum[e] + part);
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (redo[e] && c + l15 < p.N) ((__bf16 *)p.C)[(int64_t)(m + 4 * quad + e) * p.ldc + c + l15] = (__bf16)sum[e];
  }
}
#endif

template <int GROUP_M, bool HAS_BIAS, bool SK = false, bool ADD = false, bool MULTI = false, int BM = 256, int BN = 256, bool SUM = false>
__global__ __launch_bounds__(256) void gemm_nt_stream_kernel(const GemmArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)
  // one wave per SIMD, 128x128 per wave (the least LDS traffic per flop) or, in a half tile, 64x128
  static_assert(((BM == 256 || BM == 192) && BN == 256) || (BM == 256 && BN == 128) || (BM == 128 && BN == 256), "whole, three-quarter or half tiles");
  constexpr bool HALF_TILE = BM * BN == 32768;
  static_assert(!SK || (BM == 256 && !HALF_TILE), "the shared-K exchange is written for whole tiles");
  static_assert(!(SUM || MULTI) || !HALF_TILE, "lists and sums of products are made of whole or three-quarter tiles");
  static_assert(!SUM || !(HAS_BIAS || SK || ADD || MULTI), "a sum of products is a kernel of its own");
  constexpr int BK = 128, NW = 4, TM = HALF_TILE ? 4 : BM / 32, TN = 8, WN = BN / 128;
  constexpr int WROWS = TM * 16;  // rows of the tile per wave
  constexpr int A_BYTES = BM * BK, B_BYTES = BN * BK;                // the panels of one K tile
  constexpr int NLA = BM / 8 / NW, NLB = BN / 8 / NW;                // 1 KiB wave loads (8 rows x 128 B) per panel per wave
  // The LDS ring.  Whole tiles: five slots of one panel, 2.5 K tiles; panels are requested four ahead.  Half tiles: three
  // slots of one K tile; five ahead.  A trip requests one panel before its barrier (into the slot that the barrier before
  // released) and one behind it (into the slot that this K tile's A panel just left).
  constexpr int R = HALF_TILE ? 3 : 5, UNIT = HALF_TILE ? A_BYTES + B_BYTES : B_BYTES;  // (A_BYTES <= B_BYTES)
  constexpr int AHEAD = HALF_TILE ? 5 : 4;
  constexpr bool U1_IS_B = AHEAD % 2 != 0;                           // the panel requested before the barrier
  constexpr int NL1 = U1_IS_B ? NLB : NLA, NL2 = U1_IS_B ? NLA : NLB;
  constexpr int PEND = HALF_TILE ? NLA + NLB : NLA;    // in flight at the barrier of a trip: what lies beyond the next K tile
  constexpr int PEND0 = HALF_TILE ? 2 * NLA + NLB : NLA + NLB;  // prologue: K tile 1 and more may be in flight when K tile 0 is published
  constexpr int N_STORES = TM * 4;  // store instructions per wave and C tile
  static_assert(N_STORES + PEND <= 63, "vmcnt is a 6-bit counter");
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;

  // ---- this workgroup's tiles ----
  const int nb = p.tiles_m * p.tiles_n;
  const int xcd = blockIdx.x & 7, loc = blockIdx.x >> 3, W = gridDim.x >> 3;
  const int q = nb >> 3, rem = nb & 7;
  const int first = (xcd < rem) ? xcd * (q + 1) : rem * (q + 1) + (xcd - rem) * q;
  const int cnt = q + (xcd < rem ? 1 : 0);
  const int KT = (p.K + BK - 1) / BK;
  // SK instantiation -- tail of the XCD's range: the r = cnt % W tiles left after the full rounds would keep r
  // workgroups busy for a whole K loop and H = W - r idle.  When the idle ones can take enough off the others to
  // pay for an exchange of partial sums, each tail tile's K range is cut in two at the same place: the last r
  // workgroups take the first k_split K tiles of one tail tile each, in step with each other like a normal round
  // (workgroups that are at the same K tile at the same time share their panels in the XCD's L2; a split that
  // staggers them costs more in panel traffic than it saves), and own the tile; the first H workgroups (helpers)
  // multiply the remaining K tiles of tail tiles loc, loc + H, ... one after the other, again in step with each
  // other, and leave fp32 partial sums, which the owners add to their own before they store the tile.  Owners
  // wait only for workgroups with lower numbers (dispatched earlier), which never wait for anybody.
  // With m = ceil(r / H) pieces per helper, L K tiles per piece, a partial tile costing a helper about
  // kSkWriteCost K tiles' time to write and an owner kSkFixCost to add, both finish together when
  // m * (L + kSkWriteCost) = KT - L + kSkFixCost.
  const int n_rounds = cnt / W, r_tail = cnt - n_rounds * W, n_help = W - r_tail;
  const int m_help = (r_tail + n_help - 1) / n_help;
  const int l_help = (KT + kSkFixCost - m_help * kSkWriteCost) / (m_help + 1);
  const bool sk = SK && p.sk_partials != nullptr && n_rounds > 0 && r_tail > 0 && l_help >= kSkMinSaved;
  const int k_split = KT - l_help;
  const bool helper = loc < n_help;
  const int n_tail = !sk ? 0 : (helper ? (loc < r_tail ? (r_tail - loc + n_help - 1) / n_help : 0) : 1);  // pieces of this workgroup
  const int n_seg = sk ? n_rounds : (loc < cnt ? (cnt - loc + W - 1) / W : 0);                              // whole tiles
  if (n_seg + n_tail == 0) return;
  [[maybe_unused]] uint64_t prof[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (L8_GEMM_PROF) {
    prof[0] = __builtin_amdgcn_s_memrealtime();
    prof[5] = __builtin_readcyclecounter();
  }
  auto tile_at = [&](int lin, int &m0, int &n0) {
    const int per_group = GROUP_M * p.tiles_n;
    const int grp = lin / per_group;
    const int first_m = grp * GROUP_M;
    const int gsz = (p.tiles_m - first_m < GROUP_M) ? p.tiles_m - first_m : GROUP_M;
    const int in_grp = lin - grp * per_group;
    m0 = (first_m + in_grp % gsz) * BM;
    n0 = (in_grp / gsz) * BN;
  };
  // The whole tiles of a workgroup are first + loc, + W, + 2 W, ...: two cursors walk that sequence, one for the loader
  // (two K tiles ahead) and one for the multiply / store side, each holding (group, index in the group) so that a
  // tile's origin costs a shift and a mask.  (tile_at's divisions, a hundred dependent instructions each between the
  // scalar and the vector unit, took a thousand cycles per tile with idle matrix cores, on either side.)
  static_assert((GROUP_M & (GROUP_M - 1)) == 0, "GROUP_M is a power of two");
  struct TileCursor { int grp, in_grp; };
  const int per_group_c = GROUP_M * p.tiles_n;
  TileCursor cur_mul, cur_ld;
  {
    const int lin0 = first + loc;
    cur_mul.grp = lin0 / per_group_c;
    cur_mul.in_grp = lin0 - cur_mul.grp * per_group_c;
    cur_ld = cur_mul;
  }
  auto cursor_origin = [&](const TileCursor &c, int &m0, int &n0) {
    const int first_m = c.grp * GROUP_M;
    const int left = p.tiles_m - first_m;
    if (left >= GROUP_M) {
      m0 = (first_m + (c.in_grp & (GROUP_M - 1))) * BM;
      n0 = (c.in_grp / GROUP_M) * BN;
    } else {  // the last, shorter group of tile rows
      m0 = (first_m + c.in_grp % left) * BM;
      n0 = (c.in_grp / left) * BN;
    }
  };
  auto cursor_step = [&](TileCursor &c) {
    c.in_grp += W;
    while (c.in_grp >= per_group_c) {
      c.in_grp -= per_group_c;
      ++c.grp;
    }
  };
  // piece pc of the tail (highest tile first): tile origin, K-tile range [kb, ke); returns the tail tile's number
  // piece pc of this workgroup's tail: the tail tile's number (tile origin in m0, n0); every piece of a workgroup
  // covers the same K tiles [piece_kb, piece_ke)
  const int piece_kb = helper ? k_split : 0, piece_ke = helper ? KT : k_split;
  auto piece_of = [&](int pc, int &m0, int &n0) -> int {
    const int tt = helper ? loc + pc * n_help : loc - n_help;
    tile_at(first + n_rounds * W + tt, m0, n0);
    return tt;
  };

  // ---- global -> LDS load plan ----
  // lane l of a wave load fills LDS row l/8, position l%8 of an 8-row group; position p of LDS row r holds
  // chunk p ^ f(r), f(r) = (r & 7) ^ ((r >> 3) & 1).  Wave load i (of NL) of a panel fills the LDS rows of group
  // g = wave * NL + i.  For the A panel LDS row = tile row.  For the B panel LDS row r = span*128 + tn*16 + j
  // holds tile row span*128 + 8*j + tn: within a group (8 consecutive j) the rows are 8 apart, and the group's
  // first row is span*128 + 64*(g & 1) + (g%16)/2.
  // The per-lane constants of the K loop (eight registers) are formed from an opaque copy of the lane number.  In the
  // instantiation that shares K ranges out they are formed afresh in front of every tile's K loop: there, values that
  // lived across the conversion of the C tile (the point of highest register pressure) were the ones the allocator
  // chose to spill, and it reloaded them inside the K loop.  The others have the registers to keep them (two hundred
  // cycles per tile with idle matrix cores otherwise).
  uint32_t a_voff[2], b_voff[2], foff[2];
  int chunk_even, chunk_odd;
  int ld_K = p.K;  // the loader's reduction length (SUM: the present product's)
  auto row_offsets = [&](int lrow, int lda, int ldb) {
    a_voff[0] = (uint32_t)(lrow * lda + chunk_even);
    a_voff[1] = (uint32_t)(lrow * lda + chunk_odd);
    b_voff[0] = (uint32_t)(lrow * 8 * ldb + chunk_even);
    b_voff[1] = (uint32_t)(lrow * 8 * ldb + chunk_odd);
  };
  auto lane_consts = [&]() {
    int l = lane;
    asm volatile("" : "+v"(l));
    const int lrow = l >> 3, lpos = l & 7;
    chunk_even = (lpos ^ lrow) * 16;
    chunk_odd = (lpos ^ lrow ^ 1) * 16;
    row_offsets(lrow, (int)p.lda, (int)p.ldb);
    const int l15 = l & 15, piece = l >> 4;  // fragment: lane l holds row l % 16, 16-byte chunks 2 (l / 16) and 2 (l / 16) + 1
    const int fr = (l15 & 7) ^ (l15 >> 3);
#pragma unroll
    for (int j = 0; j < 2; ++j) foff[j] = l15 * BK + (((piece * 2 + j) ^ fr) * 16);
  };
  lane_consts();
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
  auto wrap = [](int slot) { return slot >= R ? slot - R : slot; };

  // the product that the tile row at m0 belongs to (m0 becomes its row inside that product)
  auto part_of = [&](int &m0) {
    GemmArgs::Part t = {p.A, p.sa, p.C, 0, p.M};
    if constexpr (MULTI) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const bool here = m0 >= p.part[i].first;
        t.A = here ? p.part[i].A : t.A;
        t.sa = here ? p.part[i].sa : t.sa;
        t.C = here ? p.part[i].C : t.C;
        t.first = here ? p.part[i].first : t.first;
        t.M = here ? p.part[i].M : t.M;
      }
      m0 -= t.first;
    }
    return t;
  };

  // loader cursor: the K tile whose panels are requested next (two K tiles ahead of the one being multiplied)
  int ld_seg = 0, ld_kt = 0;
  [[maybe_unused]] int ld_ke = KT;  // SK: the loader's piece ends here; SUM: its product
  [[maybe_unused]] int ld_term = 0, ld_m0 = 0, ld_n0 = 0;  // SUM: its product and tile
  // SUM: row and K offset of the load before; row offsets of this wave's first A and B row group, and the steps from group to group
  [[maybe_unused]] int ld_off = 0, ld_a0 = 0, ld_step_a = 0, ld_b0 = 0, ld_step_b = 0, ld_back_b = 0;
  __amdgpu_buffer_rsrc_t ld_rsA, ld_rsB;
  auto ld_open = [&](int seg) {
    if (SUM && seg < n_seg) {
      if (ld_term == 0) {
        cursor_origin(cur_ld, ld_m0, ld_n0);
        cursor_step(cur_ld);
      }
      GemmArgs::Term t = {p.A, p.B, p.sa, p.sb, p.lda, p.ldb, p.K};
#pragma unroll
      for (int i = 0; i < 2; ++i) {  // member by member: a copy of the whole would live in scratch memory
        const bool here = ld_term == i + 1;
        t.A = here ? p.term[i].A : t.A;
        t.B = here ? p.term[i].B : t.B;
        t.lda = here ? p.term[i].lda : t.lda;
        t.ldb = here ? p.term[i].ldb : t.ldb;
        t.K = here ? p.term[i].K : t.K;
      }
      ld_K = t.K;
      ld_ke = (t.K + BK - 1) / BK;
      int l = lane;
      asm volatile("" : "+v"(l));
      row_offsets(l >> 3, (int)t.lda, (int)t.ldb);
      // (opaque: kept in registers, not formed again in every trip)
      const int gb = wave * NLB;
      ld_step_a = 8 * (int)t.lda;
      ld_a0 = wave * NLA * ld_step_a;
      ld_step_b = 64 * (int)t.ldb;
      ld_back_b = -63 * (int)t.ldb;
      ld_b0 = ((gb >> 4) * 128 + 64 * (gb & 1) + ((gb & 15) >> 1)) * (int)t.ldb;
      asm volatile("" : "+s"(ld_step_a), "+s"(ld_a0), "+s"(ld_step_b), "+s"(ld_back_b), "+s"(ld_b0));
      const int64_t a_left = (int64_t)(p.M - ld_m0 - 1) * t.lda + t.K;
      const int64_t b_left = (int64_t)(p.N - ld_n0 - 1) * t.ldb + t.K;
      ld_rsA = make_rsrc(t.A + (int64_t)ld_m0 * t.lda, a_left < 0x7fffffff ? (uint32_t)a_left : 0x7fffffffu);
      ld_rsB = make_rsrc(t.B + (int64_t)ld_n0 * t.ldb, b_left < 0x7fffffff ? (uint32_t)b_left : 0x7fffffffu);
    } else if (seg < n_seg + n_tail) {
      int m0, n0;
      if (!SK || seg < n_seg) {
        cursor_origin(cur_ld, m0, n0);  // ld_open is called for seg = 0, 1, 2, ... in turn
        cursor_step(cur_ld);
        if (SK) ld_ke = KT;
      } else {
        piece_of(seg - n_seg, m0, n0);
        ld_kt = piece_kb;
        ld_ke = piece_ke;
      }
      const GemmArgs::Part t = part_of(m0);
      const int64_t a_left = (int64_t)(t.M - m0 - 1) * p.lda + p.K;
      const int64_t b_left = (int64_t)(p.N - n0 - 1) * p.ldb + p.K;
      ld_rsA = make_rsrc(t.A + (int64_t)m0 * p.lda, a_left < 0x7fffffff ? (uint32_t)a_left : 0x7fffffffu);
      ld_rsB = make_rsrc(p.B + (int64_t)n0 * p.ldb, b_left < 0x7fffffff ? (uint32_t)b_left : 0x7fffffffu);
    } else {  // past the last tile: every load is out of range and fills its LDS bytes with zeros
      ld_rsA = make_rsrc(p.A, 0);
      ld_rsB = make_rsrc(p.B, 0);
      if (SK || SUM) ld_ke = 0x7fffffff;
    }
  };
  auto ld_advance = [&]() {
    if (++ld_kt == (SK || SUM ? ld_ke : KT)) {
      ld_kt = 0;
      if (SUM) {
        if (++ld_term > p.terms) {
          ld_term = 0;
          ++ld_seg;
        }
        ld_open(ld_seg);
      } else {
        ld_open(++ld_seg);
      }
    }
  };
  // i-th wave load of the A or B panel of the loader's K tile into the panel at LDS offset `at`
  auto load_one = [&](bool is_b, int at, int i) {
    const int k0 = ld_kt * BK;
    const uint32_t m_even = (k0 + chunk_even < ld_K) ? 0u : kOOB, m_odd = (k0 + chunk_odd < ld_K) ? 0u : kOOB;
    const int g = wave * (is_b ? NLB : NLA) + i;  // 8-row group of the panel's LDS image
    const uint32_t dst = lds0 + at + g * 1024;
    // SUM: row offsets change with the product, so a load's is formed from the one before (one addition, as many as K's
    // offset takes otherwise), not kept in scalar registers
    if (!is_b) {
      int at_row = k0 + g * 8 * (int)p.lda;
      if constexpr (SUM) at_row = ld_off = i == 0 ? k0 + ld_a0 : ld_off + ld_step_a;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ld_rsA, reinterpret_cast<lds_ptr_t>(dst), 16, a_voff[i & 1] | ((i & 1) ? m_odd : m_even), at_row, 0, 0);
    } else {
      const int row = (g >> 4) * 128 + 64 * (g & 1) + ((g & 15) >> 1);
      int at_row = k0 + row * (int)p.ldb;
      if constexpr (SUM) at_row = ld_off = i == 0 ? k0 + ld_b0 : ld_off + ((i & 1) ? ld_step_b : ld_back_b);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ld_rsB, reinterpret_cast<lds_ptr_t>(dst), 16, b_voff[i & 1] | ((i & 1) ? m_odd : m_even), at_row, 0, 0);
    }
  };
  // LDS offset of the panel of the K tile `ahead` beyond the one whose slot is s0 (whole tiles: a slot per panel)
  auto panel_at = [&](int s0, int ahead, bool is_b) {
    if constexpr (HALF_TILE) return wrap(s0 + ahead) * UNIT + (is_b ? A_BYTES : 0);
    else return wrap(s0 + 2 * ahead + (is_b ? 1 : 0)) * UNIT;
  };

  // ---- LDS -> register fragment plan ----
  const int a_base = wm * (WROWS * BK);
  const int b_base = wn * (128 * BK);
  typedef const __attribute__((address_space(3))) v4i *lds_v4i_ptr;
  // LDS addresses of the two 16-byte pieces a lane reads of its A row (ad[0], ad[1]) and B row (ad[2], ad[3]); opaque
  // additions, as in the kernel above
  auto frag_addrs = [&](int panel_a, int panel_b, uint32_t (&ad)[4]) {
    const uint32_t sa = lds0 + panel_a + a_base, sb = lds0 + panel_b + b_base;
    asm volatile("v_add_u32 %0, %1, %2" : "=v"(ad[0]) : "s"(sa), "v"(foff[0]));
    asm volatile("v_add_u32 %0, %1, %2" : "=v"(ad[1]) : "s"(sa), "v"(foff[1]));
    asm volatile("v_add_u32 %0, %1, %2" : "=v"(ad[2]) : "s"(sb), "v"(foff[0]));
    asm volatile("v_add_u32 %0, %1, %2" : "=v"(ad[3]) : "s"(sb), "v"(foff[1]));
  };
  // piece h of the fragment of tile t (16 rows) at the addresses of its lower and upper piece
  auto read_piece = [&](const uint32_t *ad, v8i &f, int t, int h) {
    const v4i v = *reinterpret_cast<lds_v4i_ptr>(ad[h] + t * (16 * BK));
#pragma unroll
    for (int k = 0; k < 4; ++k) f[h * 4 + k] = v[k];
  };

  v4f acc[TM][TN];

  // One accumulator element, fetched where it is used.  Written as assembly with an accumulator-register operand:
  // given plain reads, the register allocator moves the whole accumulator set into ordinary vector registers in
  // front of the conversion of the C tile and pays for it with spills inside the K loop.
  auto acc_read = [&](int tm, int tn, int i) -> float {
    float x;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(acc[tm][tn][i]));
    return x;
  };
  // ---- C tile straight from the accumulators ----
  // acc[tm][tn][e] of lane l is C[m][n] with m = wm*WROWS + tm*16 + 4*(l / 16) + e and n = wn*128 + 8*(l % 16) + tn
  // (tile coordinates).  The host launches this kernel only when every lane's eight columns are in or out as a whole
  // and its 16-byte store is aligned: N % 8 == 0, ldc % 8 == 0, C 16-byte aligned, row scales 16-byte and bias
  // 8-byte aligned.
  // The scales (and the bias) of a tile are requested before its K loop, a handful of registers per lane: lane l
  // holds the A scales of tile rows wm*WROWS + l and + 64 + l (handed to the lanes that need them by lane permutes at
  // the end) and the B scales / bias of its own eight columns.  Requested among the stores of the
  // tile they would make their consumer wait for every store ahead of them (the counter retires in order).
  int seg_sa[2] = {0, 0};
  v4i seg_sb[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
  [[maybe_unused]] v4i seg_bias = {0, 0, 0, 0};
  // The descriptors cover the whole scale (bias) vectors and live as long as the kernel: a tile's requests then cost a
  // few address instructions (with a descriptor per tile, sixty scalar instructions at one per five cycles stood
  // between two tiles).  Rows past M and columns past N fall outside the range and read as zero; M, N < 2^29 here
  // (the host checks) so the byte offsets fit.
  const __amdgpu_buffer_rsrc_t rsSa = make_rsrc(p.sa, p.sa_row ? (uint32_t)p.M * 4u : 4u);
  const __amdgpu_buffer_rsrc_t rsSb = make_rsrc(p.sb, p.sb_row ? (uint32_t)p.N * 4u : 4u);
  [[maybe_unused]] const __amdgpu_buffer_rsrc_t rsBias = make_rsrc(HAS_BIAS ? (const void *)p.bias : (const void *)p.sb, (uint32_t)p.N * 2u);
  // a scale that is one number for the whole operand is read once (read per tile, between the stores of one tile
  // and the K loop of the next, it was a vector load whose result was copied at once: a wait for every store)
  const int sa_one = MULTI || p.sa_row ? 0 : __builtin_amdgcn_readfirstlane(__float_as_int(p.sa[0]));
  const int sb_one = p.sb_row ? 0 : __builtin_amdgcn_readfirstlane(__float_as_int(p.sb[0]));
  [[maybe_unused]] int sb_term[2] = {0, 0};
  if constexpr (SUM) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
      if (t < p.terms) sb_term[t] = __builtin_amdgcn_readfirstlane(__float_as_int(p.term[t].sb[0]));
  }
  auto load_scales = [&](int m0, int n0) {
    // lane-derived values are formed afresh from an opaque copy of the lane number wherever a tile's prologue or
    // epilogue needs them, so that none of them lives across a K loop
    int l = lane;
    asm volatile("" : "+v"(l));
    const int col = wn * 128 + 8 * (l & 15);  // this lane's eight output columns
    if (MULTI || p.sa_row) {
      __amdgpu_buffer_rsrc_t rs = rsSa;
      if constexpr (MULTI) {
        const GemmArgs::Part t = part_of(m0);
        rs = make_rsrc(t.sa, (uint32_t)t.M * 4u);
      }
      seg_sa[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, (wm * WROWS + l) * 4, m0 * 4, 0);
      if constexpr (TM > 4) seg_sa[1] = __builtin_amdgcn_raw_buffer_load_b32(rs, (wm * WROWS + 64 + l) * 4, m0 * 4, 0);
    } else {
      seg_sa[0] = seg_sa[1] = sa_one;
    }
    if (p.sb_row) {
      seg_sb[0] = __builtin_amdgcn_raw_buffer_load_b128(rsSb, col * 4, n0 * 4, 0);
      seg_sb[1] = __builtin_amdgcn_raw_buffer_load_b128(rsSb, col * 4 + 16, n0 * 4, 0);
    } else {
      seg_sb[0] = seg_sb[1] = v4i{sb_one, sb_one, sb_one, sb_one};
    }
    if constexpr (HAS_BIAS) seg_bias = __builtin_amdgcn_raw_buffer_load_b128(rsBias, col * 2, n0 * 2, 0);
  };
  // (A compute unit drains its stores at about 16 bytes per clock: the 128 KiB of a C tile keep it busy for some
  // 8000 cycles, of which the conversion below hides about half.)
  // PARTS (a tile whose last K tiles were multiplied by another workgroup): rs_p is the partial sum over those K
  // tiles, added to the workgroup's own.
  // Byte offset of piece i (of 64) of this wave in a slot.  The slots are 256 KiB apart and the workgroups of a
  // launch write theirs in step: the pieces are rotated by the slot number so that stores issued at the same time
  // do not all fall on the same memory channels.
  [[maybe_unused]] auto piece_off = [&](int slot, int i) { return (wave * (TM * TN) + ((i + slot * 5) & (TM * TN - 1))) * 1024; };
  [[maybe_unused]] __amdgpu_buffer_rsrc_t rs_p;
  [[maybe_unused]] int p_slot = 0;
  auto store_tile_as = [&](int m0, int n0, auto parts_tag, auto sbrow_tag) {
    constexpr bool PARTS = decltype(parts_tag)::value;
    // SB_ROW false: one scale for all columns; it is folded into the row scales (two multiplications per lane and
    // tile instead of one per element)
    constexpr bool SB_ROW = decltype(sbrow_tag)::value;
    // Opaque copies: everything below would otherwise be hoisted out of the K loop as loop-invariant (row
    // offsets in scalar registers, per-lane addresses in vector registers) and held across it.
    int ldc2 = (int)p.ldc * 2;
    asm volatile("" : "+s"(ldc2));
    int l = lane;
    asm volatile("" : "+v"(l));
    const int quad = l >> 4;                // this lane's four rows of a tile of sixteen
    int lane_col = wn * 128 + 8 * (l & 15);  // first of the eight columns this lane stores
    asm volatile("" : "+v"(lane_col));
    const GemmArgs::Part t = part_of(m0);
    const int64_t c_left = ((int64_t)(t.M - m0 - 1) * p.ldc + (p.N - n0)) * 2;
    const __amdgpu_buffer_rsrc_t rsC = make_rsrc(t.C + (int64_t)m0 * p.ldc + n0, c_left < 0x7fffffff ? (uint32_t)c_left : 0x7fffffffu);
    float sbv[TN];
    [[maybe_unused]] float bv[TN];
#pragma unroll
    for (int e = 0; e < TN; ++e) sbv[e] = __int_as_float(seg_sb[e >> 2][e & 3]);
    if constexpr (HAS_BIAS) {
#pragma unroll
      for (int e = 0; e < TN; ++e) bv[e] = __uint_as_float(e & 1 ? (uint32_t)seg_bias[e >> 1] & 0xffff0000u : (uint32_t)seg_bias[e >> 1] << 16);
    }
    // Row scale of tile row wm*WROWS + r: lane r % 64 of seg_sa[r / 64]; a lane needs r = tm*16 + 4*quad + e.
    // The lane permutes of the next tm are in flight while the current one is converted.  They are
    // written as assembly for the immediate offset (as plain address arithmetic their addresses were
    // precomputed into a register each and spilled) and are waited for by hand: LDS operations return in order, so
    // "at most 4 outstanding" means that everything but the group requested last has arrived.
    const int sa_addr = 16 * quad;  // byte address of lane 4*quad
    const int sa_regs[2] = {SB_ROW ? seg_sa[0] : __float_as_int(__int_as_float(seg_sa[0]) * sbv[0]),
                            SB_ROW ? seg_sa[1] : __float_as_int(__int_as_float(seg_sa[1]) * sbv[0])};
    float sa_grp[2][4];
    auto request_row_scales = [&](int tm, float (&dst)[4]) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        asm volatile("ds_bpermute_b32 %0, %1, %2 offset:%3"
                     : "=v"(dst[e])
                     : "v"(sa_addr), "v"(sa_regs[tm >> 2]), "n"(4 * ((tm & 3) * 16 + e)));
    };
    request_row_scales(0, sa_grp[0]);
    // partial sums of the tile row tm: one 16-byte piece per lane and accumulator, laid out as write_partial
    // stores them; requested one tile row ahead
    [[maybe_unused]] v4f pbuf[2][TN];
    [[maybe_unused]] const int p_voff = lane * 16;
    [[maybe_unused]] auto request_parts = [&](int tm, v4f (&dst)[TN]) {
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
        dst[tn] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs_p, p_voff, piece_off(p_slot, tm * TN + tn), kCoherent));
    };
    if constexpr (PARTS) request_parts(0, pbuf[0]);
    // (the values of C that an ADD tile is added to, 16 bytes per lane and row)
    constexpr int C_AHEAD = 8;
    [[maybe_unused]] v4i cbuf[C_AHEAD + 1];
    // Lanes whose columns lie beyond N store nothing (N % 8 == 0 here: a lane is in or out as a whole).
    const uint32_t c_voff = (n0 + lane_col < p.N) ? (uint32_t)(4 * quad * ldc2 + lane_col * 2) : kOOB;
    [[maybe_unused]] auto request_c = [&](int i, v4i &dst) {  // i = tm * 4 + e
      dst = __builtin_amdgcn_raw_buffer_load_b128(rsC, c_voff, (wm * WROWS + (i >> 2) * 16 + (i & 3)) * ldc2, 2 /* streaming */);
    };
    if constexpr (ADD) {
#pragma unroll
      for (int i = 0; i < C_AHEAD; ++i) request_c(i, cbuf[i]);
    }
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      float(&sa_cur)[4] = sa_grp[tm & 1];
      if constexpr (PARTS) {
        if (tm + 1 < TM) request_parts(tm + 1, pbuf[(tm + 1) & 1]);
      }
      if (tm + 1 < TM) {
        request_row_scales(tm + 1, sa_grp[(tm + 1) & 1]);
        asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(sa_cur[0]), "+v"(sa_cur[1]), "+v"(sa_cur[2]), "+v"(sa_cur[3]));
      } else {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(sa_cur[0]), "+v"(sa_cur[1]), "+v"(sa_cur[2]), "+v"(sa_cur[3]));
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = tm * 4 + e;
        if constexpr (ADD) {
          if (i + C_AHEAD < TM * 4) request_c(i + C_AHEAD, cbuf[(i + C_AHEAD) % (C_AHEAD + 1)]);
        }
        const float sa = sa_cur[e];
        v4i out;
#pragma unroll
        for (int pair = 0; pair < TN / 2; ++pair) {
          float v[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const int tn = pair * 2 + k;
            float a = acc_read(tm, tn, e);
            if constexpr (PARTS) a = a + pbuf[tm & 1][tn][e];  // ascending K
            v[k] = SB_ROW ? a * sa * sbv[tn] : a * sa;
            if constexpr (HAS_BIAS) v[k] += bv[tn];
          }
          typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
          const bf2 b = {(__bf16)v[0], (__bf16)v[1]};
          out[pair] = __builtin_bit_cast(int, b);
        }
        if constexpr (ADD) out = add_bf16x8(out, cbuf[i % (C_AHEAD + 1)]);
        if (L8_GEMM_DIAG != 3)  // experiment: no stores
          store16(out, rsC, c_voff, (wm * WROWS + tm * 16 + e) * ldc2, 2 /* streaming */);
        // one row at a time: left free, the scheduler reads a hundred accumulator registers ahead and the register
        // pressure of this conversion makes the allocator spill values the K loop uses in every trip
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  auto store_tile = [&](int m0, int n0, auto parts_tag) {
    // The tile's scales (and bias) are used here, on every path, so that the compiler's bookkeeping of outstanding
    // loads knows them landed whichever conversion follows.  Without it the path "requested as a row of scales,
    // converted with a scalar scale" (which no launch takes) left their registers marked as awaited, and the first
    // write to one of them between two tiles got an s_waitcnt vmcnt(0) -- a wait for every store of the tile just
    // written, some 600 cycles with idle matrix cores.
    if constexpr (HAS_BIAS) asm volatile("" : : "v"(seg_sa[0]), "v"(seg_sa[1]), "v"(seg_sb[0]), "v"(seg_sb[1]), "v"(seg_bias));
    else asm volatile("" : : "v"(seg_sa[0]), "v"(seg_sa[1]), "v"(seg_sb[0]), "v"(seg_sb[1]));
    if constexpr (SUM) {
      store_tile_as(m0, n0, parts_tag, std::false_type{});
    } else {
      if (p.sb_row) store_tile_as(m0, n0, parts_tag, std::true_type{});
      else store_tile_as(m0, n0, parts_tag, std::false_type{});
    }
  };

  // ---- SK: exchange of partial sums for tiles whose K range is shared out ----
  // Tail tile tt of XCD x has flag sk_flags[tt * 8 + x] and the fp32 tile sk_partials[(tt * 8 + x) * 65536 ...],
  // laid out the way the accumulators are held (one 16-byte piece per lane, wave, accumulator and quad: whole KiB per wave store).
  // Partial sums and flags are written and read with device-coherent accesses (they bypass the caches that are
  // not shared by all compute units), so no cache needs flushing or invalidating: a wave waits until its own
  // stores are acknowledged, the workgroup meets at a barrier, and one lane then raises the flag.
  [[maybe_unused]] auto partial_rsrc = [&](int slot) {
    return make_rsrc(p.sk_partials + (int64_t)slot * (BM * BN), BM * BN * 4);
  };
  [[maybe_unused]] auto write_partial = [&](int slot) {
    const __amdgpu_buffer_rsrc_t rs = partial_rsrc(slot);
    const int voff = lane * 16;
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) {
        const v4f v = {acc_read(tm, tn, 0), acc_read(tm, tn, 1), acc_read(tm, tn, 2), acc_read(tm, tn, 3)};
        store16(__builtin_bit_cast(v4i, v), rs, voff, piece_off(slot, tm * TN + tn), kCoherent);
        if (tn & 1) __builtin_amdgcn_sched_barrier(0);
      }
    L8_WAIT_VM_LGKM0(0);  // this wave's part of the tile has reached the point of coherence
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (threadIdx.x == 0) __hip_atomic_store(p.sk_flags + slot, p.sk_epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  // Wait until the partial sums in `slot` have been published in this launch.  Their maker has a lower number
  // than the caller (dispatched earlier) and never waits for anybody.  The wait is bounded all the same: a flag
  // that never comes poisons the tile with a NaN instead of hanging the GPU.
  [[maybe_unused]] auto wait_partial = [&](int slot) -> bool {
#pragma unroll 1
    for (int spin = 0; spin < p.sk_wait_limit; ++spin) {
      const uint32_t f = __hip_atomic_load(p.sk_flags + slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if ((uint32_t)__builtin_amdgcn_readfirstlane((int)f) == p.sk_epoch) return true;
      __builtin_amdgcn_s_sleep(32);
    }
    return false;
  };

  // ---- prologue: the first AHEAD panels of the workgroup's stream requested, K tile 0 published, its first fragments read ----
  ld_open(0);
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) {
#pragma unroll
    for (int i = 0; i < (u & 1 ? NLB : NLA); ++i) load_one(u & 1, panel_at(0, u >> 1, u & 1), i);
    if (u & 1) ld_advance();
  }
  L8_WAIT_VM_LGKM0(PEND0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  // One trip = one K tile = TM x TN MFMAs, row by row of the wave's tiles.
  //   before the barrier: the first BAR of them, while the A fragments that are not there yet are read and a panel is
  //                requested;
  //   barrier    : every wave has now read all of this K tile (lgkmcnt 0), and the next one has landed for every
  //                wave (partial vmcnt wait);
  //   behind it  : the others, while the next K tile's eight B fragments and first two A fragments are read and
  //                another panel is requested.
  // A fragment lives for its row, the B fragments for the whole trip: two sets of them, in turn.  A wave issues in
  // order and the matrix cores want an MFMA every 32 cycles, half a dozen issue slots, so a group is one MFMA with at
  // most one LDS read (half tiles, which are bound by LDS: now and then two) and one panel load, and the scheduling fences
  // keep the groups as they are laid out here.
  constexpr int N_MMA = TM * TN, BAR = HALF_TILE ? L8_HALF_TILE_BARRIER : N_MMA / 2, REST = N_MMA - BAR;
  constexpr int A_EARLY = 2;                       // A fragments read in the trip before
  constexpr int N_RD1 = 2 * (TM - A_EARLY), N_RD2 = 2 * (TN + A_EARLY);
  // groups over which the reads before and behind the barrier are spread
  constexpr int RD1_GROUPS = HALF_TILE ? BAR - 4 : L8_READ_GROUPS1 * TM / 8, RD2_GROUPS = HALF_TILE ? REST - 2 : L8_READ_GROUPS2 * TM / 8;
  static_assert(RD1_GROUPS <= BAR - 4 && RD2_GROUPS <= REST, "reads before the barrier land before it");
  v8i af[TM], bf0[TN], bf1[TN];
  uint32_t ad[4];
  // read number r behind the barrier: B0, A0, B1, .. B7, A1, .. (the order of their use), two pieces each
  auto read_next = [&](v8i (&bn)[TN], int r) {
    const int f = r >> 1;
    if (f == 0) read_piece(ad + 2, bn[0], 0, r & 1);
    else if (f == 1) read_piece(ad, af[0], 0, r & 1);
    else if (f <= TN) read_piece(ad + 2, bn[f - 1], f - 1, r & 1);
    else read_piece(ad, af[f - TN], f - TN, r & 1);
  };
  frag_addrs(panel_at(0, 0, false), panel_at(0, 0, true), ad);
#pragma unroll
  for (int r = 0; r < N_RD2; ++r) read_next(bf0, r);
  int s0 = 0;  // ring slot of the K tile being multiplied (whole tiles: of its A panel)
  // FIRST: the first K tile of an output tile (the accumulators start from zero); `stores`: the stores of a C tile have
  // been issued since the panels that the trip's barrier waits for were requested.  They are younger than the panels and
  // the counter retires in order, so the count allows for them (waiting for the stores themselves would stall the start
  // of every tile).
  // RESCALE (SUM): the first K tile of a further product.  ratio holds what the accumulators' rows are multiplied by, a value
  // per accumulator index; tile i + 1 is rescaled under the instruction of tile i.
  [[maybe_unused]] float ratio[SUM ? TM * 4 : 1];
  [[maybe_unused]] auto rescale = [&](int i) __attribute__((always_inline)) {
    const int tm = i / TN, tn = i % TN;
    v4f n;
#pragma unroll
    for (int e = 0; e < 4; ++e) n[e] = acc_read(tm, tn, e) * ratio[SUM ? tm * 4 + e : 0];
    acc[tm][tn] = n;
  };
  auto trip = [&](auto first_tag, bool stores, v8i (&bc)[TN], v8i (&bn)[TN], auto rescale_tag) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first_tag)::value, RESCALE = decltype(rescale_tag)::value;
    if constexpr (RESCALE) rescale(0);
    const int at1 = panel_at(s0, AHEAD / 2, U1_IS_B), at2 = panel_at(s0, 0, false);
    auto mma_one = [&](int i) __attribute__((always_inline)) {
      const int tm = i / TN, tn = i % TN;
      acc[tm][tn] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(af[tm], bc[tn], FIRST ? v4f{0.0f, 0.0f, 0.0f, 0.0f} : acc[tm][tn], 0, 0, 0, 0, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < BAR; ++i) {
      mma_one(i);
      if constexpr (RESCALE) rescale(i + 1);
      if (i < RD1_GROUPS) {
#pragma unroll
        for (int r = (N_RD1 * i) / RD1_GROUPS; r < (N_RD1 * (i + 1)) / RD1_GROUPS; ++r) read_piece(ad, af[A_EARLY + r / 2], A_EARLY + r / 2, r & 1);
      }
#pragma unroll
      for (int j = (NL1 * i) / BAR; j < (NL1 * (i + 1)) / BAR; ++j) load_one(U1_IS_B, at1, j);
      if (i == RD1_GROUPS) {
        int slot = s0;
        if constexpr (SUM) asm volatile("" : "+s"(slot));  // (else these addresses are formed in front of the second instruction)
        frag_addrs(panel_at(slot, 1, false), panel_at(slot, 1, true), ad);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (U1_IS_B) ld_advance();
    if (FIRST && stores) L8_WAIT_VM_LGKM0(N_STORES + PEND);
    else L8_WAIT_VM_LGKM0(PEND);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < REST; ++i) {
      mma_one(BAR + i);
      if constexpr (RESCALE) {
        if (i + 1 < REST) rescale(BAR + i + 1);
      }
      if (i < RD2_GROUPS) {
#pragma unroll
        for (int r = (N_RD2 * i) / RD2_GROUPS; r < (N_RD2 * (i + 1)) / RD2_GROUPS; ++r) read_next(bn, r);
      }
#pragma unroll
      for (int j = (NL2 * i) / REST; j < (NL2 * (i + 1)) / REST; ++j) load_one(!U1_IS_B, at2, j);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!U1_IS_B) ld_advance();
    s0 = wrap(s0 + (HALF_TILE ? 1 : 2));
  };
  // n K tiles of one output tile.  Its first one finds its B fragments in bf0.
  auto k_loop = [&](int n, bool stores, bool further = false) __attribute__((always_inline)) {
    constexpr std::false_type no{};
    if (SUM && further) trip(no, false, bf0, bf1, std::integral_constant<bool, SUM>{});
    else trip(std::true_type{}, stores, bf0, bf1, no);
#pragma unroll 1
    for (n -= 1; n >= 2; n -= 2) {
      trip(no, false, bf1, bf0, no);
      trip(no, false, bf0, bf1, no);
    }
    if (n) {
      trip(no, false, bf1, bf0, no);
    } else {  // an odd number of K tiles: the next tile's fragments are in the other set
#pragma unroll
      for (int t = 0; t < TN; ++t) bf0[t] = bf1[t];
    }
  };
  [[maybe_unused]] int again = 0;  // SUM: this lane has seen a row with units far apart
#pragma unroll 1
  for (int seg = 0; seg < n_seg; ++seg) {
    [[maybe_unused]] uint64_t t_loop = 0;
    if (L8_GEMM_PROF) {
      if (seg == 0) prof[1] = __builtin_amdgcn_s_memrealtime();
      t_loop = __builtin_readcyclecounter();
    }
    int m0, n0;
    cursor_origin(cur_mul, m0, n0);
    cursor_step(cur_mul);
    if (SK && seg > 0) lane_consts();
    if constexpr (SUM) {
      // A product's unit is the scale of its row times that of its B; all row scales of the tile are requested here, lane l
      // holding those of rows wm*WROWS + l and + 64 + l.
      int l = lane;
      asm volatile("" : "+v"(l));
      int bits[3][2];
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(t == 0 ? p.sa : p.term[t ? t - 1 : 0].sa, t <= p.terms ? (uint32_t)p.M * 4u : 0u);
        bits[t][0] = __builtin_amdgcn_raw_buffer_load_b32(rs, (wm * WROWS + l) * 4, m0 * 4, 0);
        bits[t][1] = TM > 4 ? __builtin_amdgcn_raw_buffer_load_b32(rs, (wm * WROWS + 64 + l) * 4, m0 * 4, 0) : 0;
      }
      k_loop(KT, seg > 0);
      float unit[2] = {__int_as_float(bits[0][0]) * __int_as_float(sb_one), __int_as_float(bits[0][1]) * __int_as_float(sb_one)};
      const int rows = (p.M - m0 < BM ? p.M - m0 : BM) - wm * WROWS;  // of this wave, and maybe of the one below
#pragma unroll
      for (int h = 0; h < (TM > 4 ? 2 : 1); ++h) {
        int row = lane;
        asm volatile("" : "+v"(row));
        const float next = __int_as_float(bits[1][h]) * __int_as_float(sb_term[0]), last = __int_as_float(bits[2][h]) * __int_as_float(sb_term[1]);
        again |= row + 64 * h < rows && units_apart(unit[h], next, p.terms > 1 ? last : next);
      }
      auto go_on = [&](int t) __attribute__((always_inline)) {
        int quot[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float next = __int_as_float(bits[1][h]) * __int_as_float(t == 1 ? sb_term[0] : sb_term[1]);
          quot[h] = __float_as_int(unit[h] / next);
          unit[h] = next;
        }
        int at = lane;
        asm volatile("" : "+v"(at));
        const int from = 16 * (at >> 4);
#pragma unroll
        for (int i = 0; i < TM * 4; ++i)
          ratio[i] = __int_as_float(__builtin_amdgcn_ds_bpermute(from + 4 * (((i >> 2) & 3) * 16 + (i & 3)), quot[i >> 4]));
        k_loop((p.term[t - 1].K + BK - 1) / BK, false, true);
      };
#pragma unroll 1
      for (int t = 1; t <= p.terms; ++t) {
        if (t == 2) {
          bits[1][0] = bits[2][0];
          bits[1][1] = bits[2][1];
        }
        go_on(t);
      }
      seg_sa[0] = __float_as_int(unit[0]);
      seg_sa[1] = __float_as_int(unit[1]);
      seg_sb[0][0] = __float_as_int(1.0f);
    } else {
      load_scales(m0, n0);
      k_loop(KT, seg > 0);
    }
    if (L8_GEMM_PROF) {
      const uint64_t t = __builtin_readcyclecounter();
      prof[3] += t - t_loop;
      t_loop = t;
    }
    store_tile(m0, n0, std::false_type{});
    if (L8_GEMM_PROF) prof[4] += __builtin_readcyclecounter() - t_loop;
  }
  if constexpr (SK) {
    // ---- the workgroup's share of the tail ----
    bool after_store = true;  // the segment before ended with the N_STORES stores of a C tile (n_seg > 0 here)
#pragma unroll 1
    for (int pc = 0; pc < n_tail; ++pc) {
      int m0, n0;
      const int tt = piece_of(pc, m0, n0);
      const bool owns = !helper;  // the tile's first K tiles: this workgroup adds the helper's sums and stores the tile
      const int slot = tt * 8 + xcd;
      lane_consts();
      if (owns) load_scales(m0, n0);
      k_loop(piece_ke - piece_kb, after_store);  // write_partial waited for everything in flight
      if (!owns) {
        write_partial(slot);
        after_store = false;
      } else {
        if (!wait_partial(slot)) {
          seg_sa[0] = seg_sa[1] = 0x7fc00000;  // every row scale a NaN
          // and the host can find out: one more tile poisoned, counted in the workspace (never reset by the library)
          if (threadIdx.x == 0) atomicAdd(p.sk_flags + kSkGaveUpWord, 1u);
        }
        rs_p = partial_rsrc(slot);
        p_slot = slot;
        store_tile(m0, n0, std::true_type{});
        after_store = true;
      }
    }
  }
  // the tail requests (out of range, zero filling) must have landed before the workgroup's LDS is released
  L8_WAIT_VM_LGKM0(0);
  if constexpr (SUM) {
    if (__ballot(again != 0) != 0) {
#pragma unroll 1
      for (int seg = 0; seg < n_seg; ++seg) {
        int m0, n0;
        tile_at(first + loc + seg * W, m0, n0);
#pragma unroll 1
        for (int tm = 0; tm < TM; ++tm)
          if (m0 + wm * WROWS + tm * 16 < p.M) sum_rows_one_by_one(p, m0 + wm * WROWS + tm * 16, n0 + wn * 128);
      }
    }
  }
  if (L8_GEMM_PROF) {
    prof[2] = __builtin_amdgcn_s_memrealtime();
    prof[5] = __builtin_readcyclecounter() - prof[5];
    prof[6] = n_seg;
    prof[7] = ((uint64_t)__builtin_amdgcn_s_getreg(63508) << 32) | (uint32_t)__builtin_amdgcn_s_getreg(63492);  // XCC_ID, HW_ID
    if (threadIdx.x == 0 && p.dbg) {
      uint64_t *d = p.dbg + (int64_t)blockIdx.x * 8;
      for (int i = 0; i < 8; ++i) d[i] = prof[i];
    }
  }
#else
  (void)p;
#endif
}

// ---------------------------------------------------------------------------
// tile configurations ("algos")
// ---------------------------------------------------------------------------
typedef void (*gemm_fn)(const GemmArgs);
struct Algo {
  const char *name;
  gemm_fn fn;
  int bm, bn, threads, lds;
  bool persistent;   // one workgroup per compute unit walks a list of tiles
  gemm_fn fn_bias;   // persistent kernels: the instantiation that adds a bias (the plain kernels branch inside)
  gemm_fn fn_add;    // persistent kernels: the instantiation that adds to C (bias-free), or null (the plain kernels branch inside)
  gemm_fn fn_sk;     // persistent kernels: the instantiation that can share a tile's K range out (bias-free), or null
};

// X(WM, WN, TM, TN, R, GROUP_M, PF) -- 1-based position in this list is the `algo` number
#define L8_ALGO_LIST(X)                                                          \
  X(2, 2, 4, 4, 5, 4, 0)  /* 1: 256x256, 4 waves (128x128 each), ring of 5    */ \
  X(2, 2, 2, 2, 5, 4, 0)  /* 2: 128x128, 4 waves (small problems)             */ \
  X(2, 4, 4, 2, 5, 4, 0)  /* 3: 256x256, 8 waves (128x64 each)                */ \
  X(4, 2, 2, 4, 5, 4, 0)  /* 4: 256x256, 8 waves (64x128 each)                */ \
  X(2, 2, 4, 4, 5, 8, 0)  /* 5: algo 1 with taller groups                     */ \
  X(2, 2, 4, 4, 5, 2, 0)  /* 6: algo 1 with shorter groups                    */ \
  X(2, 2, 4, 4, 5, 4, 4)  /* 7: algo 1 with L2 touches 4 K tiles ahead        */ \
  X(2, 4, 4, 2, 5, 4, 4)  /* 8: algo 3 with L2 touches 4 K tiles ahead        */ \
  X(2, 2, 4, 4, 5, 16, 0) /* 9: algo 1 with groups of 16                      */ \
  X(2, 4, 4, 2, 5, 8, 0)  /* 10: algo 3 with taller groups                    */

// (R, and the _r of a name: 5 is the ring of five panels; beyond that it only says that the loop is the deep one, whose
// ring holds as many whole K tiles as the LDS does -- deep_slots.  The t of a name counts 32x32 pieces of a wave's tile,
// also in the persistent kernels, whose instruction is 16x16.)
// 18 .. 20: small problems, one workgroup per compute unit or fewer: the deep loop (five K tiles in the ring for 128x128, six
// for the smaller ones; a second workgroup has no use for the LDS) and smaller tiles where 128 x 128 ones would be too few
#define L8_SMALL_ALGO_LIST(X)                         \
  X(2, 2, 2, 2, 9, 4, 0) /* 18: 128x128            */ \
  X(2, 2, 1, 2, 9, 4, 0) /* 19: 64x128             */ \
  X(2, 2, 2, 1, 9, 4, 0) /* 20: 128x64             */

// X(WM, WN, TM, TN, R, GROUP_M, KS): the smallest tiles, K tiles dealt to two groups of waves with a ring each.  A trip
// costs them 310 ns whatever they load (wait, barrier, LDS reads, one or two matrix instructions in a row; a deeper ring
// changed nothing), so two trips run side by side.  us, before the deep loop, weight just written, one group / two / four:
// [333,8192].[2048,8192] 19.5 / 14.6 / 16.7, [100,11008].[4096,11008] 24.9 / 18.7 / 22.2, [200,4096].[4096,4096] 11.2 / 8.9 /
// 9.3.  Larger tiles gain nothing: 128x128 [700,11008].[4096,11008] 39.2 / 39.7, 64x128 [1021,2048].[2048,2048] cold 9.3 / 9.9.
#define L8_SPLIT_ALGO_LIST(X)                         \
  X(2, 2, 1, 1, 9, 4, 2) /* 21: 64x64              */ \
  X(1, 2, 1, 1, 9, 4, 2) /* 22: 32x64              */

#define L8_INSTANTIATE(WM, WN, TM, TN, R, GM, PF) \
  template __global__ void gemm_nt_kernel<WM, WN, TM, TN, R, GM, PF>(const GemmArgs);
L8_ALGO_LIST(L8_INSTANTIATE)
L8_SMALL_ALGO_LIST(L8_INSTANTIATE)
#define L8_SPLIT_INSTANTIATE(WM, WN, TM, TN, R, GM, KS) \
  template __global__ void gemm_nt_kernel<WM, WN, TM, TN, R, GM, 0, KS>(const GemmArgs);
L8_SPLIT_ALGO_LIST(L8_SPLIT_INSTANTIATE)

#define L8_ALGO_ROW(WM, WN, TM, TN, R, GM, PF)                                                                \
  {"mt" #WM "x" #WN "w_" #TM "x" #TN "t_r" #R "_g" #GM "_pf" #PF, gemm_nt_kernel<WM, WN, TM, TN, R, GM, PF>, \
   WM * TM * 32, WN * TN * 32, WM * WN * 64, plain_lds(WM * TM * 32, WN * TN * 32, R, 1), false, nullptr, nullptr, nullptr},

#define L8_SPLIT_ALGO_ROW(WM, WN, TM, TN, R, GM, KS)                                                               \
  {"mt" #WM "x" #WN "w_" #TM "x" #TN "t_r" #R "_g" #GM "_ks" #KS, gemm_nt_kernel<WM, WN, TM, TN, R, GM, 0, KS>, \
   WM * TM * 32, WN * TN * 32, WM * WN * KS * 64, plain_lds(WM * TM * 32, WN * TN * 32, R, KS), false, nullptr, nullptr, nullptr},

template __global__ void gemm_nt_stream_kernel<8, false>(const GemmArgs);
template __global__ void gemm_nt_stream_kernel<8, true>(const GemmArgs);
template __global__ void gemm_nt_stream_kernel<4, false>(const GemmArgs);
template __global__ void gemm_nt_stream_kernel<4, true>(const GemmArgs);
template __global__ void gemm_nt_stream_kernel<4, false, true>(const GemmArgs);
template __global__ void gemm_nt_stream_kernel<4, false, false, true>(const GemmArgs);
template __global__ void gemm_nt_stream_kernel<4, false, false, false, true>(const GemmArgs);
template __global__ void gemm_nt_stream_kernel<4, false, false, false, false, 256, 256, true>(const GemmArgs);
template __global__ void gemm_nt_stream_kernel<4, false, false, false, true, 192, 256>(const GemmArgs);
template __global__ void gemm_nt_stream_kernel<4, false, false, false, false, 192, 256, true>(const GemmArgs);
template __global__ void gemm_nt_stream_kernel<2, false>(const GemmArgs);
template __global__ void gemm_nt_stream_kernel<2, true>(const GemmArgs);
template __global__ void gemm_nt_stream_kernel<16, false>(const GemmArgs);
template __global__ void gemm_nt_stream_kernel<16, true>(const GemmArgs);

static_assert(kSkinnyAlgo == 17, "position in the list below");
static const Algo kAlgos[] = {
    L8_ALGO_LIST(L8_ALGO_ROW)
    /* 11, 12: persistent 256x256 tiles, 4 waves, one panel stream across tiles, C stored from the accumulators */
    {"stream_mt2x2w_4x4t_r5_g8", gemm_nt_stream_kernel<8, false>, 256, 256, 256, 5 * 256 * 128, true, gemm_nt_stream_kernel<8, true>, gemm_nt_stream_kernel<4, false, false, true>, nullptr},
    {"stream_mt2x2w_4x4t_r5_g4", gemm_nt_stream_kernel<4, false>, 256, 256, 256, 5 * 256 * 128, true, gemm_nt_stream_kernel<4, true>,
     gemm_nt_stream_kernel<4, false, false, true>, nullptr},
    /* 13, 14: other shapes of the block of tiles resident on an XCD (2 x 16 and 16 x 2 instead of 4 x 8: 18 panels
       shared by 32 tiles instead of 12), kept for the traffic comparison */
    {"stream_mt2x2w_4x4t_r5_g2", gemm_nt_stream_kernel<2, false>, 256, 256, 256, 5 * 256 * 128, true, gemm_nt_stream_kernel<2, true>, gemm_nt_stream_kernel<4, false, false, true>, nullptr},
    {"stream_mt2x2w_4x4t_r5_g16", gemm_nt_stream_kernel<16, false>, 256, 256, 256, 5 * 256 * 128, true, gemm_nt_stream_kernel<16, true>, gemm_nt_stream_kernel<4, false, false, true>, nullptr},
    /* 15: algo 12 that may share the K range of the last round's tiles out between workgroups (l8_gemm_nt_ws with
       a workspace; without one it is algo 12).  Measured neutral on the shapes it applies to: the part is
       power-limited, and the compute units that the plain split leaves idle in the last round let the busy ones
       clock higher, which recovers most of what the idle ones lose. */
    {"stream_mt2x2w_4x4t_r5_g4_sk", gemm_nt_stream_kernel<4, false>, 256, 256, 256, 5 * 256 * 128, true, gemm_nt_stream_kernel<4, true>,
     gemm_nt_stream_kernel<4, false, false, true>, gemm_nt_stream_kernel<4, false, true>},
    /* 16: was algo 12 with eight waves (two per SIMD), behind it since the fragments of a K tile take 192 registers;
       the number stands for algo 12 */
    {"stream_mt2x2w_4x4t_r5_g4", gemm_nt_stream_kernel<4, false>, 256, 256, 256, 5 * 256 * 128, true, gemm_nt_stream_kernel<4, true>,
     gemm_nt_stream_kernel<4, false, false, true>, nullptr},
    /* 17: at most 64 tokens: 16 rows of B and all of A per workgroup, K split over its waves (skinny_kernels.hip) */
    {"skinny_8w_16n", nullptr, 64, 16, 512, 0, false, nullptr, nullptr, nullptr},
    L8_SMALL_ALGO_LIST(L8_ALGO_ROW)
    L8_SPLIT_ALGO_LIST(L8_SPLIT_ALGO_ROW)
    /* 23, 24: algo 12 on half tiles, for problems that whole ones would spread over too few compute units or rounds */
    {"stream_mt4x1w_2x4t_r3_g4", gemm_nt_stream_kernel<4, false, false, false, false, 256, 128>, 256, 128, 256, 3 * 384 * 128, true,
     gemm_nt_stream_kernel<4, true, false, false, false, 256, 128>, gemm_nt_stream_kernel<4, false, false, true, false, 256, 128>, nullptr},
    {"stream_mt2x2w_2x4t_r3_g8", gemm_nt_stream_kernel<8, false, false, false, false, 128, 256>, 128, 256, 256, 3 * 384 * 128, true,
     gemm_nt_stream_kernel<8, true, false, false, false, 128, 256>, gemm_nt_stream_kernel<8, false, false, true, false, 128, 256>, nullptr},
    /* 25: algo 12 on three quarters of a tile, for problems that leave whole ones' last round nearly empty */
    {"stream_mt2x2w_3x4t_r5_g4", gemm_nt_stream_kernel<4, false, false, false, false, 192, 256>, 192, 256, 256, 5 * 256 * 128, true,
     gemm_nt_stream_kernel<4, true, false, false, false, 192, 256>, gemm_nt_stream_kernel<4, false, false, true, false, 192, 256>, nullptr},
};
constexpr int kNumAlgos = sizeof(kAlgos) / sizeof(kAlgos[0]);

}  // namespace l8

using namespace l8;

extern "C" int l8_gemm_algo_count(void) { return kNumAlgos; }
extern "C" const char *l8_gemm_algo_name(int algo) {
  return (algo >= 1 && algo <= kNumAlgos) ? kAlgos[algo - 1].name : nullptr;
}

// plain kernel for a problem with at least one 256x256 tile per compute unit: four waves with 128x128 wave
// tiles (least LDS traffic per flop) unless K is so short (measured: below 4096) that the conversion of the C
// tile, which eight waves share out over twice as many wave slots, weighs more than the K loop
static int pick_plain_big(int64_t K) { return K >= 4096 ? 5 : 3; }

// 9/16 of the units have a 256 x 256 tile
static bool fills_with_big_tiles(int64_t M, int64_t N) { return ((M + 255) / 256) * ((N + 255) / 256) * 16 >= (int64_t)num_cus() * 9; }

static int pick_algo(int64_t M, int64_t N, int64_t K, bool three_quarters = true) {
  if (M <= 8) return kSkinnyAlgo;  // whatever the chip: the smallest calls do not pay for asking
  const int64_t cus = num_cus();
  auto tiles = [&](int64_t bm, int64_t bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  const bool big = fills_with_big_tiles(M, N);
  // A few tokens: the weight's bytes are what counts (skinny_kernels.hip).  us, against the best tile: [20,2048].
  // [2048,2048] 4.2 / 7.5, [64,11008].[4096,11008] 18.9 / 28.8, [32,4096].[11008,4096] 14.6 / 13.5; from 48 tokens on
  // the 64 x 64 tiles win where there are enough of them ([48,4096].[11008,4096] 17.6 / 14.0, [40,4096].[8192,4096]
  // 12.2 / 12.1, [64,8192].[8192,8192] 25.3 / 23.5).
  // With 9/16 of the units at work on 32 x 64 tiles, more than one tile of 16 tokens or rows beyond 4096 make the skinny
  // kernels the slower ones (every workgroup reads all of x): [32,4096].[11008,4096] 14.4 / 13.0, [32,5120].[14336,5120]
  // 24.6 / 17.1, [16,5120].[9216,5120] 15.8 / 13.7, but [16,4096].[11008,4096] 10.9 / 12.5, [32,4096].[8192,4096] 10.6 / 11.8.
  const int64_t wide = tiles(32, 64);
  if (M <= 32 && (M > 16 || K > 4096) && wide * 16 >= cus * 9 && wide <= cus) return 22;
  // A weight so wide that one row of big tiles would fill the chip gains nothing from them (they compute 256 rows): up to
  // 16 tokens stay here, more go to the 128 x 128 tiles.  us, weight cold, skinny / 128 x 128 / 256 x 256: [1,4096].
  // [36864,4096] 26 / 39 / 49, [16,4096].[36864,4096] 28 / 39 / 50, [32,4096].[36864,4096] 40 / 40 / 50, [64,4096].
  // [36864,4096] 54 / 42 / 50, [1,4096].[128256,4096] 79 / 108 / 113, [16,4096].[128256,4096] 99 / 110 / 115,
  // [32,4096].[128256,4096] 129 / 111 / 115, [64,4096].[128256,4096] 179 / 113 / 116.
  if (M <= 16 || (M <= 32 && !big) || (M <= kSkinnyMaxM && tiles(64, 64) * 16 < cus * 7)) return kSkinnyAlgo;
  // Otherwise the smallest tile that gives no compute unit a second workgroup: these kernels are bound by their LDS
  // traffic and by what a K tile costs whatever its size, so more units at work are worth more than the larger tile's
  // economy.  us, operands of several problems in turn, 128 x 128 with two workgroups per unit (configuration 2) / 128 x 128 /
  // 64 x 128 / 128 x 64 / 64 x 64: [200,4096].[4096,4096] 18.9 / 15.0 / 11.8 / 12.1 / 9.8, [333,8192].[2048,8192] 32.6 / 25.6 /
  // 19.8 / 20.7 / 15.4, [1021,2048].[2048,2048] 12.4 / 11.1 / 9.8 / 10.0 / 12.9, [512,4096].[4096,4096] 19.3 / 16.0 / 13.7 / 13.8 /
  // 18.6, [1392,3280].[1392,3280] 17.1 / 14.7 / 12.4 / 12.5 / 16.8, [333,2048].[8192,2048] 12.5 / 10.9 / 16.2 / 15.7 / 18.5,
  // [700,11008].[4096,11008] 65.9 / 50.8 / 71.4 / 64.7 / 69.7, [2048,16384].[2048,16384] 87.6 / 75.0 / 99.9 / 98.5 / 128.3.
  if (tiles(64, 64) <= cus) return 21;
  if (tiles(64, 128) <= cus) return 19;
  if (tiles(128, 64) <= cus) return 20;
  if (tiles(128, 128) <= cus) return 18;
  // Barely more than that with a short reduction, or few rows: two 128 x 128 workgroups share a unit.  us, these / the half
  // tiles below: [64,4096].[36864,4096] 42 / 44, [1500,1440].[3008,1440] 14.5 / 13.5 with rows on lines and 16.3 / 17 without;
  // longer reductions [1884,4544].[2384,4544] 28.3 / 26.5, [3973,3488].[1072,3488] 25.0 / 21.9.
  if (M <= kSkinnyMaxM || (!big && K <= 2048 && tiles(128, 128) * 8 <= cus * 9)) return 2;
  // Beyond: the persistent kernel, on whole tiles or on half ones (of the two forms the one with fewer rounds).  It is
  // bound by its rounds of one tile per unit, and a round of half tiles takes 0.59 of a round of whole ones (1300 against
  // 2280 cycles per K tile: 1.5 times the bytes per flop through the L2, which then is what a trip waits for; with short
  // reductions less, the C tile weighs more).  So half tiles where their rounds are at most 3/2 of the others', 5/3 up to
  // K = 4096, 7/4 up to 2048.  us, 128 x 128 / half / whole: [4096,2048].[2048,2048] 19.9 / 18.4 / 26.0,
  // [1645,9776].[4272,9776] 63.5 / 53.3 / 82.2, [502,11312].[9568,11312] 94.4 / 68.4 / 100.5, [3115,2336].[2752,2336] 31.5
  // / 30.1 / 25.8 (286 half tiles are two rounds, 143 whole ones are one), [1566,1136].[9904,1136] 28.3 / 22.1 / 31.8,
  // [1294,7392].[13664,7392] 142 / 126 / 138, [14991,4032].[2224,4032] 127 / 118 / 123 and [2710,8832].[14064,8832] 322 /
  // 278 / 263 (5 against 3), [11181,1328].[3424,1328] 60.3 / 49.9 / 55.6, [5561,1664].[9104,1664] 92.8 / 81.0 / 88.4 (7
  // rounds against 4), but [4093,4096]. [14336,4096] 204 / 169 / 163 (also 7 against 4), [6191,3568].[4016,3568] 88 / 83 /
  // 73 (4 against 2).
  auto rounds = [&](int64_t t) { return (t + cus - 1) / cus; };
  const int64_t whole = rounds(tiles(256, 256)), tall = rounds(tiles(256, 128)), wide2 = rounds(tiles(128, 256));
  const int64_t half = wide2 < tall ? wide2 : tall;
  // Three quarters of a tile (192 x 256) where whole ones would leave more than that of their rounds idle: where they need no
  // more rounds, each of 0.87 .. 0.93 of the time (a K tile is 1536 cycles of matrix instructions instead of 2048, its loads
  // and the C tile's conversion shrink less), and half tiles not so few that they are ahead.  A round more is never made up
  // for.  us, whole / half / three quarters: [3000,3600] K = 512 13.7 / - / 11.9, 4096 42.0 / 46.9 / 36.8, 11008 106 / - / 100,
  // [2800,5120].[3072,5120] 46.5 / - / 40.6, [180,2048].[65536,2048] 36.9 / - / 32.4, [520,1024].[16384,1024] 15.7 / - / 12.9,
  // [1801,2912].[11040,2912] 65.4 / 67.8 / 56.8, [1676,4128].[9360,4128] 91 / 97 / 82, [4800,9216].[4864,9216] 172 / 173 / 161,
  // [12288,1024].[2048,1024] 30.3 / 28.5 / 27.2, [5000,4096].[6656,4096] - / 121 / 107; but [3290,1392].[3904,1392] (two rounds
  // against one) 21.2 / - / 30.3, [4093,4096].[14336,4096] (five against four) 168 / 184 / 176, [300,4096].[36864,4096] (two
  // rounds of half tiles) - / 59.6 / 76.6, [3115,2752].[2336,2752] (one) 30.4 / 23.3 / 24.8.
  const int64_t quarters = rounds(tiles(192, 256));
  if (three_quarters && big && quarters <= whole && half * 5 > quarters * 7) return 25;
  if (half * 2 <= whole * 3 || (K <= 4096 && half * 3 <= whole * 5) || (K <= 2048 && half * 4 <= whole * 7)) return wide2 < tall ? 24 : 23;
  return 12;
}

// Host arithmetic only: the tile configuration `algo = 0` resolves to for this problem on the current device when
// the operands allow every kernel (aligned, N % 8 == 0): what a caller that reports per-kernel figures names.
extern "C" int l8_gemm_pick(int64_t M, int64_t N, int64_t K) {
  L8_REQUIRE(M > 0 && N > 0 && K > 0, "l8_gemm_pick: empty problem");
  return pick_algo(M, N, K);
}

// flags (one 4-byte word per workgroup, first 4 KiB) + one fp32 256x256 tile per workgroup of a persistent launch
constexpr int64_t kSkMaxGrid = kSkMaxGridWords, kSkFlagBytes = (kSkMaxGrid + 64) * 4, kSkTileBytes = 256 * 256 * 4;
static std::atomic<uint32_t> g_sk_epoch{0};
// polls (about a microsecond each) an owner spends on a helper's flag before it gives up: a third of a second
static std::atomic<int> g_sk_wait_limit{1 << 18};

extern "C" int l8_gemm_set_wait_limit(int polls) {
  L8_REQUIRE(polls >= 0, "l8_gemm_set_wait_limit: negative limit");
  g_sk_wait_limit = polls;
  return L8_OK;
}

extern "C" int64_t l8_gemm_workspace_gave_up_offset(void) { return (int64_t)kSkGaveUpWord * 4; }

extern "C" int64_t l8_gemm_workspace(void) {
  const int64_t cus8 = (num_cus() / 8) * 8;
  return kSkFlagBytes + (cus8 < 8 ? 8 : cus8) * kSkTileBytes;
}

// Does sharing out the K range of the last round's tiles pay for an XCD with `cnt` tiles, W workgroups and KT K
// tiles per tile?  (Same test as in the kernel.)
static bool sk_pays(int64_t cnt, int64_t W, int64_t KT) {
  const int64_t n_rounds = cnt / W, r = cnt % W, n_help = W - r;
  const int64_t m_help = (r + n_help - 1) / n_help;
  const int64_t l_help = (KT + kSkFixCost - m_help * kSkWriteCost) / (m_help + 1);
  return n_rounds > 0 && r > 0 && l_help >= kSkMinSaved;
}

// Host arithmetic only (no GPU needed): on a part with `compute_units` compute units, how many of the 8 XCDs would
// share out the K range of their last round's tiles under tile configuration 15 for this problem.
extern "C" int l8_gemm_shares_k(int64_t M, int64_t N, int64_t K, int compute_units) {
  L8_REQUIRE(M >= 0 && N >= 0 && K >= 0 && compute_units >= 8, "l8_gemm_shares_k: bad argument");
  const int64_t nblocks = ((M + 255) / 256) * ((N + 255) / 256), KT = (K + 127) / 128;
  const int64_t cus8 = (compute_units / 8) * 8, want = (nblocks + 7) / 8 * 8;
  int64_t grid = want < cus8 ? want : cus8;
  if (grid < 8) grid = 8;
  const int64_t W = grid / 8, q = nblocks / 8, rem = nblocks % 8;
  return (int)((sk_pays(q + 1, W, KT) ? rem : 0) + (sk_pays(q, W, KT) ? 8 - rem : 0));
}

// one workgroup per compute unit, a multiple of 8 of them (the hardware deals workgroups to the 8 XCDs in turn)
static int64_t persistent_grid(int64_t nblocks) {
  const int64_t cus8 = (num_cus() / 8) * 8, want = (nblocks + 7) / 8 * 8;
  const int64_t grid = want < cus8 ? want : cus8;
  return grid < 8 ? 8 : grid;
}

static int gemm_nt_impl(const void *A, const void *B, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                        const float *sa, int sa_mode, const float *sb, int sb_mode, const void *bias, void *C,
                        int64_t ldc, int add, int algo, void *workspace, int64_t workspace_bytes, void *stream) {
  L8_REQUIRE(M >= 0 && N >= 0 && K >= 0, "l8_gemm_nt: negative shape");
  if (M == 0 || N == 0) return L8_OK;
  L8_REQUIRE(A && B && C && sa && sb, "l8_gemm_nt: null pointer");
  L8_REQUIRE(K > 0, "l8_gemm_nt: K must be positive");
  L8_REQUIRE(K % 16 == 0, "l8_gemm_nt: K=%lld must be a multiple of 16", (long long)K);
  L8_REQUIRE(lda % 16 == 0 && ldb % 16 == 0 && lda >= K && ldb >= K, "l8_gemm_nt: lda=%lld, ldb=%lld must be multiples of 16 and >= K",
             (long long)lda, (long long)ldb);
  L8_REQUIRE(((uintptr_t)A % 16) == 0 && ((uintptr_t)B % 16) == 0, "l8_gemm_nt: A and B must be 16-byte aligned");
  L8_REQUIRE(ldc >= N, "l8_gemm_nt: ldc=%lld < N=%lld", (long long)ldc, (long long)N);
  L8_REQUIRE((sa_mode == L8_SCALE_SCALAR || sa_mode == L8_SCALE_ROW) && (sb_mode == L8_SCALE_SCALAR || sb_mode == L8_SCALE_ROW),
             "l8_gemm_nt: bad scale mode");
  L8_REQUIRE(M < (1LL << 31) && N < (1LL << 31) && K < (1LL << 31), "l8_gemm_nt: dimension too large");
  L8_REQUIRE(algo >= 0 && algo <= kNumAlgos, "l8_gemm_nt: algo %d out of range 0..%d", algo, kNumAlgos);
  const bool chosen = algo == 0;
  if (chosen) algo = pick_algo(M, N, K);
  // (rows so far apart that whole tiles are refused below are refused, not served by the shorter ones)
  if (chosen && algo == 25 && 256 * lda + K >= (1LL << 31)) algo = pick_algo(M, N, K, false);
  // Rows so far apart that 256 of them pass the 32-bit offsets below: a problem of middling size, which taller tiles would
  // only serve faster, takes 128 x 128 ones and is refused where 128 rows are too many.
  if (chosen && kAlgos[algo - 1].persistent && !fills_with_big_tiles(M, N) && (256 * lda + K >= (1LL << 31) || 256 * ldb + K >= (1LL << 31)))
    algo = 2;
  if (kAlgos[algo - 1].persistent) {
    // the persistent kernel stores 16 aligned bytes (eight columns) per lane and reads the row scales 16 bytes
    // at a time; operands that do not allow that go to the plain kernel with the same tile shape
    // (and addresses its scale vectors with 32-bit byte offsets)
    const bool ok = N % 8 == 0 && ldc % 8 == 0 && ((uintptr_t)C % 16) == 0 && ldc < (1LL << 22) &&
                    M < (1LL << 29) && N < (1LL << 29) &&
                    (sa_mode != L8_SCALE_ROW || ((uintptr_t)sa % 16) == 0) &&
                    (sb_mode != L8_SCALE_ROW || ((uintptr_t)sb % 16) == 0) &&
                    (bias == nullptr || (((uintptr_t)bias % 8) == 0 && kAlgos[algo - 1].fn_bias != nullptr)) &&
                    (!add || kAlgos[algo - 1].fn_add != nullptr);
    if (!ok) {
      if (algo == 25) algo = chosen ? pick_algo(M, N, K, false) : 12;
      algo = kAlgos[algo - 1].bm * kAlgos[algo - 1].bn < 256 * 256 ? 2 : pick_plain_big(K);
    }
  }
  if (algo == kSkinnyAlgo) {
    if (skinny_serves(M, N, K, lda, ldb, 1))
      return skinny_linear(SkinnyArgs{A, B, (int)M, (int)N, (int)K, lda, ldb, sa, sb, sa_mode == L8_SCALE_ROW, sb_mode == L8_SCALE_ROW,
                                      (const uint16_t *)bias, (uint16_t *)C, ldc, 0, add}, false, false, (hipStream_t)stream);
    algo = 2;
  }
  const Algo &al = kAlgos[algo - 1];
  // 32-bit in-tile byte offsets: (tile rows) * ld + K must stay below 2^31
  L8_REQUIRE((int64_t)al.bm * lda + K < (1LL << 31) && (int64_t)al.bn * ldb + K < (1LL << 31),
             "l8_gemm_nt: leading dimension too large for 32-bit tile offsets");
  GemmArgs p;
  p.A = (const uint8_t *)A;
  p.B = (const uint8_t *)B;
  p.M = (int)M;
  p.N = (int)N;
  p.K = (int)K;
  p.lda = lda;
  p.ldb = ldb;
  p.ldc = ldc;
  p.sa = sa;
  p.sb = sb;
  p.sa_row = sa_mode == L8_SCALE_ROW;
  p.sb_row = sb_mode == L8_SCALE_ROW;
  p.bias = (const uint16_t *)bias;
  p.add = add;
  p.sk_flags = nullptr;
  p.sk_partials = nullptr;
  p.sk_epoch = 0;
  p.sk_wait_limit = 0;
  p.dbg = nullptr;
  if (L8_GEMM_PROF && al.persistent) {
    p.dbg = (uint64_t *)bias;
    p.bias = nullptr;
  }
  p.C = (uint16_t *)C;
  p.tiles_m = (int)((M + al.bm - 1) / al.bm);
  p.tiles_n = (int)((N + al.bn - 1) / al.bn);
  const int64_t nblocks = (int64_t)p.tiles_m * p.tiles_n;
  L8_REQUIRE(nblocks < (1LL << 31), "l8_gemm_nt: too many tiles");
  static bool attr_done[kMaxDev][kNumAlgos] = {};  // idempotent; a race only repeats the call
  const int slot = device_slot();
  if (slot < 0 || !attr_done[slot][algo - 1]) {
    L8_HIP(hipFuncSetAttribute((const void *)al.fn, hipFuncAttributeMaxDynamicSharedMemorySize, al.lds));
    if (al.fn_bias) L8_HIP(hipFuncSetAttribute((const void *)al.fn_bias, hipFuncAttributeMaxDynamicSharedMemorySize, al.lds));
    if (al.fn_add) L8_HIP(hipFuncSetAttribute((const void *)al.fn_add, hipFuncAttributeMaxDynamicSharedMemorySize, al.lds));
    if (al.fn_sk) L8_HIP(hipFuncSetAttribute((const void *)al.fn_sk, hipFuncAttributeMaxDynamicSharedMemorySize, al.lds));
    if (slot >= 0) attr_done[slot][algo - 1] = true;
  }
  const int64_t grid = al.persistent ? persistent_grid(nblocks) : nblocks;
  gemm_fn fn = (al.fn_add && add) ? al.fn_add : (al.fn_bias && p.bias) ? al.fn_bias : al.fn;
  if (al.fn_sk && !p.bias && !add && workspace != nullptr && grid <= kSkMaxGrid && workspace_bytes >= kSkFlagBytes + grid * kSkTileBytes) {
    // the kernel decides per XCD (their tile counts differ by at most one) with the same test
    const int64_t W = grid / 8, KT = (K + 127) / 128, q = nblocks / 8;
    bool use = sk_pays(q, W, KT) || (nblocks % 8 != 0 && sk_pays(q + 1, W, KT));
    if (use) {
      // Not inside a stream capture: the launch number is a kernel argument, and a replayed launch would find
      // the flags of the replay before already at its number.
      hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
      if (hipStreamIsCapturing((hipStream_t)stream, &cs) != hipSuccess) {
        (void)hipGetLastError();
        use = false;
      } else if (cs != hipStreamCaptureStatusNone) {
        use = false;
      }
    }
    if (use) {
      fn = al.fn_sk;
      p.sk_flags = (uint32_t *)workspace;
      p.sk_partials = (float *)((uint8_t *)workspace + kSkFlagBytes);
      uint32_t e = ++g_sk_epoch;
      if (e == 0) e = ++g_sk_epoch;  // 0 is what an untouched flag holds
      p.sk_epoch = e;
      p.sk_wait_limit = g_sk_wait_limit;
    }
  }
  hipLaunchKernelGGL(fn, dim3((unsigned)grid), dim3(al.threads), al.lds, (hipStream_t)stream, p);
  L8_HIP(hipGetLastError());
  return L8_OK;
}

extern "C" int l8_gemm_nt(const void *A, const void *B, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                          const float *sa, int sa_mode, const float *sb, int sb_mode, const void *bias, void *C,
                          int64_t ldc, int algo, void *stream) {
  return gemm_nt_impl(A, B, M, N, K, lda, ldb, sa, sa_mode, sb, sb_mode, bias, C, ldc, 0, algo, nullptr, 0, stream);
}

extern "C" int l8_gemm_nt_add(const void *A, const void *B, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                              const float *sa, int sa_mode, const float *sb, int sb_mode, void *C, int64_t ldc, int algo,
                              void *stream) {
  return gemm_nt_impl(A, B, M, N, K, lda, ldb, sa, sa_mode, sb, sb_mode, nullptr, C, ldc, 1, algo, nullptr, 0, stream);
}

extern "C" int l8_gemm_nt_ws(const void *A, const void *B, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                             const float *sa, int sa_mode, const float *sb, int sb_mode, const void *bias, void *C,
                             int64_t ldc, int algo, void *workspace, int64_t workspace_bytes, void *stream) {
  L8_REQUIRE(workspace == nullptr || ((uintptr_t)workspace % 16) == 0, "l8_gemm_nt_ws: workspace must be 16-byte aligned");
  return gemm_nt_impl(A, B, M, N, K, lda, ldb, sa, sa_mode, sb, sb_mode, bias, C, ldc, 0, algo, workspace, workspace_bytes, stream);
}

// Do products of M[i] rows with one B of N rows run faster as one launch of the persistent kernel?  Bound by the matrix cores
// of the units that have a tile: apart, each product leaves units without one (in its last round, or in all of it on the
// smaller tiles); together they do so once.  us, apart / together, 256 units:
//   3 x [2048,K].[2048,K]^T, 192 tiles: K = 256 18.6 / 10.9, 1024 25.4 / 18.1, 4096 57.8 / 42.3, 16384 192.5 / 145.7 (2.83 PFLOP/s)
//   [2048 + 512 + 512], 96 tiles: 256 14.9 / 9.6, 1024 19.6 / 15.6, 4096 40.1 / 38.5, but 16384 119.0 / 122.5
//   3 x [1408,..], 108 tiles: 4096 43.1 / 38.2, 16384 142.0 / 124.3;  3 x [1280,..], 75: 131.3 / 121.9;  3 x [1024,..], 48: 80.7 / 120.9
//   2 x [2816,..].[1024,..], 88 tiles: 1024 16.3 / 15.0, 4096 36.3 / 37.1;  2 x [2048,..], 64 tiles: 29.4 / 36.2
//   whole rounds: 3 x [4096,4096].[4096,4096] 152.5 / 142.4, 2 x [14336,4096].[4096,4096] 353 / 328, 2 x [11008,4096].[4096,4096] 272 / 267
// so from 3/8 of a tile per unit on, a little more where the reduction is long.
extern "C" int l8_gemm_multi_pays(const l8_gemm_part *parts, int64_t n, int64_t N, int64_t K) {
  int64_t tiles = 0;
  for (int64_t i = 0; i < n; ++i) tiles += ((parts[i].M + 255) / 256) * ((N + 255) / 256);
  return tiles * 32 >= (int64_t)num_cus() * (K > 4096 ? 13 : 12);
}

// Three quarters of a whole tile by the rule of single products (pick_algo).
extern "C" int l8_gemm_multi_tile_rows(const l8_gemm_part *parts, int64_t n, int64_t N) {
  const int64_t cus = num_cus();
  int64_t whole = 0, quarters = 0;
  for (int64_t i = 0; i < n; ++i) {
    whole += (parts[i].M + 255) / 256 * ((N + 255) / 256);
    quarters += (parts[i].M + 191) / 192 * ((N + 255) / 256);
  }
  return whole * 16 >= cus * 9 && (quarters + cus - 1) / cus <= (whole + cus - 1) / cus ? 192 : 256;
}

extern "C" int l8_gemm_nt_multi(const l8_gemm_part *parts, int64_t n, const void *B, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                                const float *sb, int sb_mode, int64_t ldc, int algo, void *stream) {
  L8_REQUIRE(n >= 0 && (n == 0 || parts), "l8_gemm_nt_multi: null list or negative count");
  bool one = algo == 0 && n >= 2 && n <= 3 && B && sb && N > 0 && N < (1LL << 29) && K > 0 && K % 16 == 0 && K < (1LL << 31) && N % 8 == 0 &&
             ldc % 8 == 0 && ldc >= N && ldc < (1LL << 22) && lda % 16 == 0 && ldb % 16 == 0 && lda >= K && ldb >= K &&
             256 * lda + K < (1LL << 31) && 256 * ldb + K < (1LL << 31) && ((uintptr_t)B % 16) == 0 &&
             (sb_mode == L8_SCALE_SCALAR || (sb_mode == L8_SCALE_ROW && ((uintptr_t)sb % 16) == 0));
  int64_t tile_rows = 0;
  for (int64_t i = 0; one && i < n; ++i) {
    const l8_gemm_part &t = parts[i];
    one = t.A && t.C && t.sa && t.M > 0 && t.M < (1LL << 28) && ((uintptr_t)t.A % 16) == 0 && ((uintptr_t)t.C % 16) == 0 && ((uintptr_t)t.sa % 16) == 0;
    tile_rows += (t.M + 255) / 256;
  }
  one = one && tile_rows * ((N + 255) / 256) < (1LL << 31) && l8_gemm_multi_pays(parts, n, N, K);
  if (!one) {
    for (int64_t i = 0; i < n; ++i) {
      const l8_gemm_part &t = parts[i];
      const int rc = gemm_nt_impl(t.A, B, t.M, N, K, lda, ldb, t.sa, L8_SCALE_ROW, sb, sb_mode, nullptr, t.C, ldc, 0, algo, nullptr, 0, stream);
      if (rc != L8_OK) return rc;
    }
    return L8_OK;
  }
  constexpr int kLds = 5 * 256 * 128;
  const int64_t bm = l8_gemm_multi_tile_rows(parts, n, N);
  const gemm_fn fn = bm == 256 ? gemm_nt_stream_kernel<4, false, false, false, true> : gemm_nt_stream_kernel<4, false, false, false, true, 192, 256>;
  tile_rows = 0;
  for (int64_t i = 0; i < n; ++i) tile_rows += (parts[i].M + bm - 1) / bm;
  GemmArgs p{};
  p.A = (const uint8_t *)parts[0].A;
  p.B = (const uint8_t *)B;
  p.M = (int)parts[0].M;
  p.N = (int)N;
  p.K = (int)K;
  p.lda = lda;
  p.ldb = ldb;
  p.ldc = ldc;
  p.sa = parts[0].sa;
  p.sb = sb;
  p.sa_row = 1;
  p.sb_row = sb_mode == L8_SCALE_ROW;
  p.C = (uint16_t *)parts[0].C;
  p.tiles_m = (int)tile_rows;
  p.tiles_n = (int)((N + 255) / 256);
  int64_t first = 0;
  for (int i = 0; i < 2; ++i) {
    first += (parts[i].M + bm - 1) / bm * bm;
    if (i + 1 < n) p.part[i] = {(const uint8_t *)parts[i + 1].A, parts[i + 1].sa, (uint16_t *)parts[i + 1].C, (int)first, (int)parts[i + 1].M};
    else p.part[i] = {p.A, p.sa, p.C, 0x7fffffff, p.M};
  }
  static std::atomic<bool> attr_done[2][kMaxDev] = {};  // idempotent; a race only repeats the call
  const int slot = device_slot();
  if (slot < 0 || !attr_done[bm == 256][slot]) {
    L8_HIP(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, kLds));
    if (slot >= 0) attr_done[bm == 256][slot] = true;
  }
  hipLaunchKernelGGL(fn, dim3((unsigned)persistent_grid((int64_t)p.tiles_m * p.tiles_n)), dim3(256), kLds, (hipStream_t)stream, p);
  L8_HIP(hipGetLastError());
  return L8_OK;
}

// The sum of products as one K loop, or as one product that the others are added to?  As one it saves, per product after the
// first, the conversion of a C tile and its way to memory and back, and pays 2000 cycles per tile for the change of scales.
// Bound by the matrix cores' power either way: beyond K = 8192 per product what is saved no longer shows.  us, one by one /
// as one: 3 x [16384,2048] K = 2048 194.8 / 157.4, K = 2048 + 512 + 512 125.9 / 84.2, 2 x K = 512 58.4 / 39.6, K = 4096 197.7 / 176.6,
// K = 5632 254 / 234, K = 8192 355.5 / 352.5 and, on another machine, 382.9 / 387.5; 2 x [16384,4096] K = 4096 384.6 / 349.4,
// K = 6144 540.8 / 511.9, K = 11008 924 / 922; 2 x [8192,5120] K = 7168 431 / 399; 2 x [4093,4096] K = 14336 298 / 290 and,
// on another machine, 311 / 323.  Against 64 bits the sum is 1.7e-3 off (one rounding to bf16), before 2.4e-3 with two products
// and 2.9e-3 with three.
static bool sum_in_one(const l8_gemm_term *terms, int64_t n, int64_t M, int64_t N, const void *C, int64_t ldc) {
  if (n < 2 || n > 3 || M <= 0 || N <= 0 || M >= (1LL << 29) || N >= (1LL << 29) || N % 8 || ldc % 8 || ldc < N || ldc >= (1LL << 22) || ((uintptr_t)C % 16)) return false;
  int64_t K = 0;
  for (int64_t i = 0; i < n; ++i) {
    const l8_gemm_term &t = terms[i];
    if (!t.A || !t.B || !t.sa || !t.sb || t.K < 512 || t.K % 16 || t.lda % 16 || t.ldb % 16 || t.lda < t.K || t.ldb < t.K ||
        256 * t.lda + t.K >= (1LL << 31) || 256 * t.ldb + t.K >= (1LL << 31) || ((uintptr_t)t.A % 16) || ((uintptr_t)t.B % 16))
      return false;
    K += t.K;
  }
  return K < n * 8192 && ((M + 255) / 256) * ((N + 255) / 256) < (1LL << 31) && pick_algo(M, N, K, false) == 12;
}

extern "C" int l8_gemm_nt_sum(const l8_gemm_term *terms, int64_t n, int64_t M, int64_t N, void *C, int64_t ldc, int algo, void *stream) {
  L8_REQUIRE(n >= 1 && terms, "l8_gemm_nt_sum: no terms");
  if (algo != 0 || !sum_in_one(terms, n, M, N, C, ldc)) {
    for (int64_t i = 0; i < n; ++i) {
      const l8_gemm_term &t = terms[i];
      const int rc = gemm_nt_impl(t.A, t.B, M, N, t.K, t.lda, t.ldb, t.sa, L8_SCALE_ROW, t.sb, L8_SCALE_SCALAR, nullptr, C, ldc, i > 0, algo, nullptr, 0, stream);
      if (rc != L8_OK) return rc;
    }
    return L8_OK;
  }
  constexpr int kLds = 5 * 256 * 128;
  int64_t K = 0;
  for (int64_t i = 0; i < n; ++i) K += terms[i].K;
  const int64_t bm = pick_algo(M, N, K) == 25 ? 192 : 256;
  const gemm_fn fn = bm == 256 ? gemm_nt_stream_kernel<4, false, false, false, false, 256, 256, true> : gemm_nt_stream_kernel<4, false, false, false, false, 192, 256, true>;
  GemmArgs p{};
  p.A = (const uint8_t *)terms[0].A;
  p.B = (const uint8_t *)terms[0].B;
  p.M = (int)M;
  p.N = (int)N;
  p.K = (int)terms[0].K;
  p.lda = terms[0].lda;
  p.ldb = terms[0].ldb;
  p.ldc = ldc;
  p.sa = terms[0].sa;
  p.sb = terms[0].sb;
  p.sa_row = 1;
  p.C = (uint16_t *)C;
  p.tiles_m = (int)((M + bm - 1) / bm);
  p.tiles_n = (int)((N + 255) / 256);
  p.terms = (int)n - 1;
  for (int i = 0; i < 2; ++i) {
    const l8_gemm_term &t = terms[i + 1 < n ? i + 1 : 0];
    p.term[i] = {(const uint8_t *)t.A, (const uint8_t *)t.B, t.sa, t.sb, t.lda, t.ldb, (int)t.K};
  }
  static std::atomic<bool> attr_done[2][kMaxDev] = {};  // idempotent; a race only repeats the call
  const int slot = device_slot();
  if (slot < 0 || !attr_done[bm == 256][slot]) {
    L8_HIP(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, kLds));
    if (slot >= 0) attr_done[bm == 256][slot] = true;
  }
  hipLaunchKernelGGL(fn, dim3((unsigned)persistent_grid((int64_t)p.tiles_m * p.tiles_n)), dim3(256), kLds, (hipStream_t)stream, p);
  L8_HIP(hipGetLastError());
  return L8_OK;
}
