// One call per pass of a linear: the casts and the product of lingua/float8.py:85-96 enqueued by one entry, their
// temporaries in one workspace.  A caller in an interpreted language pays for one crossing and one allocation where it
// paid for one per kernel; with a few tokens that was most of the time.  Same results as the entries called one by one.
#include "l8_common.h"
#include "skinny.h"

namespace l8 {

// Row stride of a quantised operand that this library lays out itself: whole 128-byte lines.  The products read their
// operands in segments of 128 bytes of a row; with rows that start in the middle of a line every segment is two lines, and
// the L2's request rate is what bounds the products of middling size.  us, rows K bytes apart / on lines: [1676,9360].[4128,
// 9360] 95.6 / 64.0, [1216,9936].[3904,9936] 89.6 / 57.0, [2976,16240].[3424,16240] 171.9 / 147.7, [3290,1392].[1392,1392]
// 17.4 / 13.1, [493,4832].[6784,4832] 25.2 / 20.2, [16225,2976].[3424,2976] 140.9 / 131.6; a line more changed nothing.
static int64_t fp8_row_stride(int64_t K) { return (K + 127) / 128 * 128; }

// Hands out 256-byte aligned pieces of a workspace; with a null base it only adds sizes up.
struct Pieces {
  uint8_t *base;
  int64_t used = 0;
  void *take(int64_t bytes) {
    uint8_t *p = base ? base + used : nullptr;
    used += (bytes + 255) / 256 * 256;
    return p;
  }
};

struct LinearFwd {
  void *qx, *qw, *col_ws;
  float *sx, *sw;
  int64_t ldqx, ldqw;
  int64_t col_ws_bytes;
  bool w_on_the_way, x_on_the_way;  // quantised inside the product
};

// `ldqx`, `ldqw`: row strides of the quantised operands that the caller hands in.
static LinearFwd plan(const l8_linear_fwd_args &a, int64_t ldqx, int64_t ldqw, Pieces &ws) {
  LinearFwd t{};
  // A few tokens and nobody who wants the weight's bytes or amaxes: one pass over the weight instead of three (read,
  // written, read).  us, weights cold, cast + product / one kernel: [1,4096].[11008,4096] 44 / 20.8, [7,4096].[4096,4096]
  // 25 / 10.4, [8,2048].[8192,2048] 20 / 12.  Only where the product of the quantised operands is that kernel too: every
  // kernel adds up K in an order of its own, and a linear's result shall not hang on who wants its gradient or keeps its
  // weight quantised.  Where that product runs on tiles, one kernel would save at most a third: [17,4096].[11008,4096]
  // 35 / 27, [32,4096].[16384,4096] 50 / 36, but [32,5120].[14336,5120] 54 / 54, [64,4096].[11008,4096] 36 / 36.
  auto skinny = [&] { return a.algo == 0 && a.M > 0 && a.N > 0 && a.K > 0 && l8_gemm_pick(a.M, a.N, a.K) == kSkinnyAlgo; };
  t.w_on_the_way = !a.qw && !a.amax_w && skinny_serves(a.M, a.N, a.K, a.K, a.ldw, 2) && skinny();
  const int w_bytes = t.w_on_the_way ? 2 : 1;
  t.x_on_the_way = !a.qx && !a.col_amax_x && skinny_quantises_x(a.M, a.N, a.K, a.ldx, w_bytes) &&
                   (t.w_on_the_way || (skinny_serves(a.M, a.N, a.K, a.ldx, a.qw ? ldqw : fp8_row_stride(a.K), 1) && skinny()));
  if (!t.x_on_the_way) {
    t.ldqx = a.qx ? ldqx : fp8_row_stride(a.K);
    t.qx = a.qx ? a.qx : ws.take(a.M * t.ldqx);
    t.sx = a.qx ? a.sx : (float *)ws.take(a.M * 4);
  }
  if (!t.w_on_the_way) {
    t.ldqw = a.qw ? ldqw : fp8_row_stride(a.K);
    t.qw = a.qw ? a.qw : ws.take(a.N * t.ldqw);
    t.sw = a.qw ? a.sw : (float *)ws.take(a.N * 4);
  }
  t.col_ws_bytes = a.col_amax_x ? l8_cast_rowwise_workspace(a.M, a.K) : 0;
  t.col_ws = t.col_ws_bytes ? ws.take(t.col_ws_bytes) : nullptr;
  return t;
}

}  // namespace l8

using namespace l8;

static int check_fwd(const l8_linear_fwd_args *a) {
  L8_REQUIRE(a != nullptr, "l8_linear_fwd: null arguments");
  L8_REQUIRE(a->M >= 0 && a->N >= 0 && a->K >= 0, "l8_linear_fwd: negative shape");
  L8_REQUIRE((a->qx != nullptr) == (a->sx != nullptr) && (a->qw != nullptr) == (a->sw != nullptr),
             "l8_linear_fwd: a quantised operand comes with its scales");
  L8_REQUIRE(!a->x_ready || (a->qx && !a->col_amax_x), "l8_linear_fwd: x_ready without qx, or with col_amax_x");
  L8_REQUIRE(!a->w_ready || (a->qw && !a->amax_w), "l8_linear_fwd: w_ready without qw, or with amax_w");
  return L8_OK;
}

// All that the casts and the product ask of their operands, so that a call is refused before any of them is enqueued.
static int check_operands(const l8_linear_fwd_args &a, int64_t ldqx, int64_t ldqw) {
  auto aligned = [](const void *p, uintptr_t n) { return (uintptr_t)p % n == 0; };
  auto source = [&](const void *p, int64_t ld) { return p && a.K % 8 == 0 && ld % 8 == 0 && ld >= a.K && aligned(p, 16); };
  if (!a.x_ready && a.M > 0 && a.K > 0)
    L8_REQUIRE(source(a.x, a.ldx), "l8_linear_fwd: x must be 16-byte aligned, K=%lld and ldx=%lld multiples of 8, ldx >= K",
               (long long)a.K, (long long)a.ldx);
  if (!a.w_ready && a.N > 0 && a.K > 0)
    L8_REQUIRE(source(a.w, a.ldw), "l8_linear_fwd: w must be 16-byte aligned, K=%lld and ldw=%lld multiples of 8, ldw >= K",
               (long long)a.K, (long long)a.ldw);
  if (a.M == 0 || a.N == 0) return L8_OK;
  L8_REQUIRE(a.K > 0 && a.K % 16 == 0, "l8_linear_fwd: K=%lld must be positive and a multiple of 16", (long long)a.K);
  L8_REQUIRE(a.M < (1LL << 31) && a.N < (1LL << 31) && a.K < (1LL << 31), "l8_linear_fwd: dimension too large");
  L8_REQUIRE(aligned(a.qx, 16) && aligned(a.qw, 16), "l8_linear_fwd: qx and qw must be 16-byte aligned");
  auto rows = [&](const void *q, int64_t ld) { return !q || (ld >= a.K && ld % 16 == 0); };
  L8_REQUIRE(rows(a.qx, ldqx) && rows(a.qw, ldqw), "l8_linear_fwd: ldqx=%lld and ldqw=%lld must be multiples of 16, >= K",
             (long long)ldqx, (long long)ldqw);
  L8_REQUIRE(a.y && a.ldy >= a.N, "l8_linear_fwd: y is null, or ldy=%lld < N=%lld", (long long)a.ldy, (long long)a.N);
  L8_REQUIRE(a.algo >= 0 && a.algo <= l8_gemm_algo_count(), "l8_linear_fwd: algo %lld out of range", (long long)a.algo);
  return L8_OK;
}

extern "C" int64_t l8_linear_fwd_rows_workspace(const l8_linear_fwd_args *a, int64_t ldqx, int64_t ldqw) {
  if (check_fwd(a) != L8_OK) return L8_EINVAL;
  Pieces ws{nullptr};
  plan(*a, ldqx, ldqw, ws);
  return ws.used;
}

extern "C" int64_t l8_linear_fwd_workspace(const l8_linear_fwd_args *a) { return l8_linear_fwd_rows_workspace(a, a ? a->K : 0, a ? a->K : 0); }

extern "C" int l8_linear_fwd(const l8_linear_fwd_args *a) { return l8_linear_fwd_rows(a, a ? a->K : 0, a ? a->K : 0); }

extern "C" int l8_linear_fwd_rows(const l8_linear_fwd_args *a, int64_t ldqx, int64_t ldqw) {
  int rc = check_fwd(a);
  if (rc == L8_OK) rc = check_operands(*a, ldqx, ldqw);
  if (rc != L8_OK) return rc;
  Pieces ws{(uint8_t *)a->workspace};
  const LinearFwd t = plan(*a, ldqx, ldqw, ws);
  L8_REQUIRE(ws.used <= a->workspace_bytes && ((uintptr_t)a->workspace % 256) == 0,
             "l8_linear_fwd: needs a 256-byte aligned workspace of %lld bytes", (long long)ws.used);
  const bool cast_x = !a->x_ready && !t.x_on_the_way, cast_w = !t.w_on_the_way && !a->w_ready;
  bool together = cast_x && cast_w && !a->col_amax_x;
  if (cast_x && cast_w && a->col_amax_x) {
    const l8_cast_rowwise_cols_item two[2] = {{a->x, a->M, a->K, a->ldx, t.qx, t.ldqx, t.sx, nullptr, a->col_amax_x, t.col_ws, t.col_ws_bytes},
                                              {a->w, a->N, a->K, a->ldw, t.qw, t.ldqw, t.sw, a->amax_w, nullptr, nullptr, 0}};
    rc = cast_rowwise_pair(two, (hipStream_t)a->stream, &together);
    if (rc != L8_OK) return rc;
  } else if (together) {
    const l8_cast_rowwise_item items[2] = {{a->x, a->M, a->ldx, t.qx, t.ldqx, t.sx, nullptr}, {a->w, a->N, a->ldw, t.qw, t.ldqw, t.sw, a->amax_w}};
    rc = l8_cast_rowwise_many(items, 2, a->K, a->stream);
    if (rc != L8_OK) return rc;
  }
  if (cast_x && !together) {
    rc = l8_cast_rowwise(a->x, a->M, a->K, a->ldx, t.qx, t.ldqx, t.sx, nullptr, a->col_amax_x, t.col_ws, t.col_ws_bytes, a->stream);
    if (rc != L8_OK) return rc;
  }
  if (cast_w && !together) {
    rc = l8_cast_rowwise(a->w, a->N, a->K, a->ldw, t.qw, t.ldqw, t.sw, a->amax_w, nullptr, nullptr, 0, a->stream);
    if (rc != L8_OK) return rc;
  }
  if (t.x_on_the_way || t.w_on_the_way)
    return skinny_linear(SkinnyArgs{t.x_on_the_way ? a->x : t.qx, t.w_on_the_way ? a->w : t.qw, (int)a->M, (int)a->N, (int)a->K,
                                    t.x_on_the_way ? a->ldx : t.ldqx, t.w_on_the_way ? a->ldw : t.ldqw, t.sx, t.sw, 1, 1,
                                    (const uint16_t *)a->bias, (uint16_t *)a->y, a->ldy, scale_rule(), 0},
                         t.w_on_the_way, t.x_on_the_way, (hipStream_t)a->stream);
  return l8_gemm_nt(t.qx, t.qw, a->M, a->N, a->K, t.ldqx, t.ldqw, t.sx, L8_SCALE_ROW, t.sw, L8_SCALE_ROW, a->bias, a->y, a->ldy,
                    (int)a->algo, a->stream);
}
