// extern "C" entry points of libflashmuon_hip.so: argument validation, workspace carving and the
// Newton-Schulz composition.  No torch types, no allocation, no synchronisation.
#include "../../include/flashmuon.h"
#include "fm_internal.h"
#include "fm_routes.h"
#include <atomic>

using namespace fm;

namespace {

inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

struct Range { uintptr_t lo, hi; };
// byte range of a rows x cols matrix with row stride ld and element size esz
inline Range mat_range(const void* p, int64_t rows, int64_t cols, int64_t ld, int esz) {
  Range r;
  r.lo = reinterpret_cast<uintptr_t>(p);
  r.hi = (rows <= 0 || cols <= 0) ? r.lo : r.lo + (uintptr_t)(((rows - 1) * ld + cols) * esz);
  return r;
}
inline bool overlaps(Range a, Range b) { return a.lo < b.hi && b.lo < a.hi; }
inline bool misaligned(const void* p, int esz) { return (reinterpret_cast<uintptr_t>(p) % esz) != 0; }
inline int dtype_size(int dt) { return dt == FM_F32 ? 4 : 2; }
inline bool bad_dtype(int dt) { return dt != FM_BF16 && dt != FM_F16 && dt != FM_F32; }
inline int hip_status(int rc) { return rc == 0 ? FM_OK : (rc == kErrWorkspace ? FM_ERR_WORKSPACE : FM_ERR_LAUNCH); }
// a workspace is only used when it is 256-byte aligned; otherwise the call runs without one
inline void* usable_ws(void* ws) { return (reinterpret_cast<uintptr_t>(ws) % 256 == 0) ? ws : nullptr; }

// workspace of fm_newtonschulz_batched_bf16, carved in this order; per-matrix arrays are
// batch-major with the strides below
struct NsLayout {
  size_t partials, pdiag, x[2], xt[2], a, p, gemm, total;
  size_t pdiag_stride;   // floats between the fp32 diagonals of consecutive matrices
  int M, K;              // the sizes the iteration runs on: those of the matrix, or padded (below)
  bool padded;
  int edge_s, edge_x;    // tiles of the one-launch iteration
  bool flow;             // one launch for all products: x[0], a and p hold kFlowSteps (+ 1) iterates and squares
  size_t counters;
};
// 64x64 tiles for X' as long as every CU gets at most one, and for the symmetric products as long as they are
// about one round (a longer K makes the 64-tiles of A = X X^T pay a little further): 512^2 104 us on 64x64
// tiles, 115 with X' on 128x128, 144 all on 128x128; 8 of 384 x 768 152, 111 and 133; 24 of 768^2 520, 423 and 360.
void ns_flow_edges(int batch, int m, int k, int* es, int* ex) {
  const int64_t t = (m + 63) / 64, sym = t * (t + 1) / 2 * batch, rect = t * ((k + 63) / 64) * batch;
  *ex = rect <= 256 ? 64 : 128;
  *es = rect <= 256 || sym <= 256 || (sym <= 440 && k >= 2 * m) ? 64 : 128;
}
// A matrix whose sides are not whole 128-tiles would take the general GEMM path in every stage
// (0.5-0.8 times the vendor GEMMs).  Its iterates live in the workspace anyway, so they are kept
// zero-padded to whole tiles instead: zero rows and columns stay zero through every step, and the
// tiled paths run.  Whole 256x256 tiles pay for up to 128 more rows and columns, also where the
// sides are whole multiples of 128 already, once the 256x256 path has enough of them: for a single
// matrix from a short side of 2176 on, of a square one of 2816 (five steps at 3200^2 0.86 ms, padded to 3328^2 0.79; 3200 x
// 8000 1.66 and 1.55; 2176 x 4400 0.58 and 0.55; but 2176^2 0.407 and 0.422, 2688^2 0.509 and 0.539), for a batch as
// soon as its 256x256 tiles fill the GPU (32 of 1664^2 4.6 ms, of 1792^2 4.2; 2688 x 7168 36 and
// 2816 x 7168 26).  The long side alone goes to a multiple of 256 where the short one is one already
// (32 of 2048 x 5504 15.4 ms, of 2048 x 5632 11.9; one matrix 0.72 and 0.59; below 1536 rows a single
// matrix gains nothing).
// `flow`: one launch where that is the faster one (ns_flow_chosen).
NsLayout ns_layout(int batch, int rows, int cols, bool flow) {
  const int m = rows < cols ? rows : cols, k = rows < cols ? cols : rows;
  const size_t B = (size_t)batch;
  NsLayout l = {};
  if (flow && !any_knob_set() && ns_flow_chosen(batch, m, k)) {
    l.flow = true;
    ns_flow_edges(batch, m, k, &l.edge_s, &l.edge_x);
    l.M = (m + l.edge_x - 1) / l.edge_x * l.edge_x;
    l.K = (k + l.edge_x - 1) / l.edge_x * l.edge_x;
    l.padded = l.M != m || l.K != k;
    size_t off = 0;
    auto take = [&](size_t bytes) { size_t o = off; off += align_up(bytes, 256); return o; };
    const size_t M = (size_t)l.M, K = (size_t)l.K;
    l.partials = take(B * kSumsqBlocks * sizeof(float));
    l.pdiag_stride = M;
    l.pdiag = take(B * M * kFlowSteps * sizeof(float));
    l.x[0] = take(B * M * K * 2 * (kFlowSteps + 1));
    l.a = take(B * M * M * 2 * kFlowSteps);
    l.p = take(B * M * M * 2 * kFlowSteps);
    l.counters = take((size_t)flow_counter_words(batch, kFlowSteps) * sizeof(unsigned));
    l.gemm = off;
    l.total = off;
    return l;
  }
  l.M = (m + 127) / 128 * 128;
  l.K = (k + 127) / 128 * 128;
  {
    const int64_t t = (l.M + 255) / 256;
    const bool near_square = k < m + m / 5;
    const bool both = l.M >= (batch == 1 && near_square ? 2816 : 2176) || (l.M >= 1152 && (int64_t)batch * t * (t + 1) / 2 >= 120);
    if (both) l.M = (int)t * 256;
    if (l.M % 256 == 0 && (both || l.M >= 1536 || (batch >= 4 && l.M >= 768))) l.K = (k + 255) / 256 * 256;
  }
  l.padded = l.M != m || l.K != k;
  const size_t M = (size_t)l.M, K = (size_t)l.K;
  size_t off = 0;
  auto take = [&](size_t bytes) { size_t o = off; off += align_up(bytes, 256); return o; };
  l.partials = take(B * kSumsqBlocks * sizeof(float));
  l.pdiag_stride = align_up(M, 64);
  l.pdiag = take(B * l.pdiag_stride * sizeof(float));
  for (int i = 0; i < 2; ++i) { l.x[i] = take(B * M * K * 2); l.xt[i] = take(B * M * K * 2); }
  l.a = take(B * M * M * 2);
  l.p = take(B * M * M * 2);
  // partial tiles of the three products of a step: two M x M (symmetric) and one M x K, `batch` each
  const size_t g1 = gemm_fast_workspace_bytes(l.M, l.M, batch), g2 = gemm_fast_workspace_bytes(l.M, l.K, batch);
  l.gemm = take(g1 > g2 ? g1 : g2);
  l.total = off;
  return l;
}

// ---- scratch of fm_syrk_bf16_static -------------------------------------------------------------
// 256 partial tiles of 256 KiB: what the 256x256 schedule needs at most when it cuts only the items
// of its last round (more than that only buys a deeper k split of outputs with few tiles, which
// this entry point then does without).  Every GPU the library runs on holds its own copy of the
// array, at its own address, until the process ends.
constexpr size_t kStaticScratchBytes = (size_t)256 * 256 * 256 * sizeof(float);   // 64 MiB
static __device__ __align__(256) unsigned char fm_static_scratch[kStaticScratchBytes];

// device address of the array on the current device, looked up once per device (in host code the
// array's name is only a handle for this lookup, never an address a kernel could use)
int static_scratch(void** out) {
  constexpr int kMaxDev = 64;
  static std::atomic<void*> per_device[kMaxDev];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDev) return FM_ERR_LAUNCH;
  void* p = per_device[dev].load(std::memory_order_acquire);
  if (!p) {
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(fm_static_scratch)) != hipSuccess || !p) return FM_ERR_LAUNCH;
    per_device[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return FM_OK;
}

}  // namespace

extern "C" {

const char* fm_status_string(int status) {
  switch (status) {
    case FM_OK: return "ok";
    case FM_ERR_NULL: return "a required pointer is NULL";
    case FM_ERR_SHAPE: return "invalid or inconsistent dimensions";
    case FM_ERR_STRIDE: return "leading dimension smaller than the row length";
    case FM_ERR_DTYPE: return "unsupported dtype code";
    case FM_ERR_ALIAS: return "an output overlaps an input";
    case FM_ERR_WORKSPACE: return "workspace missing or too small";
    case FM_ERR_LAUNCH: return "kernel launch failed";
    case FM_ERR_ALIGN: return "pointer not aligned to its element size";
    default: return "unknown status";
  }
}

const char* fm_version(void) { return "0.1.0"; }

size_t fm_gemm_workspace_bytes(int rows_out, int cols_out) {
  if (rows_out <= 0 || cols_out <= 0) return 0;
  return gemm_fast_workspace_bytes(rows_out, cols_out, 1);
}

int fm_set_knob(int which, long long value) { return set_knob(which, value) == 0 ? FM_OK : FM_ERR_SHAPE; }

// X * X^T in 16 bits of sides that the 256-tiles of launch_gemm_nt do not fit: in place (fm_gemm_ragged.hip), or behind
// a copy of X with rows of whole stages, where 16-byte copies cannot take the rows or too many of them would cross a line.
//   Sides that are no whole 128-tiles, from 65536 elements of X on (below that the general path's single launch wins).
// us, zero-padded copies of both X and Y around the tiled paths before, now: 600^2 17.3 -> 10.7, 1000^2 16.7 -> 11.0, 2000^2 32 ->
// 23, 3000 x 1000 33 -> 24, 3000 x 5000 79 -> 70, 3900 x 8000 140 -> 104, 600 x 8000 32 -> 22, 6500^2 356 -> 294.
//   Odd numbers of whole 128-tiles with rows on 128-byte lines, by syrk_whole_in_place.
struct SyrkRagged { int Kp; size_t slots, x, total; };
constexpr int64_t kSyrkRaggedMinElems = 256 * 256;
static bool whole_tiles(int M, int K) { return M % 128 == 0 && K % 64 == 0; }
static bool syrk_ragged_layout(int M, int K, SyrkRagged* p) {
  if (M <= 0 || K <= 0 || (int64_t)M * K < kSyrkRaggedMinElems || K >= (1 << 22)) return false;
  if (whole_tiles(M, K) && (M % 256 == 0 || any_knob_set() || syrk_whole_slim(M, K) || !syrk_whole_in_place(M, K, cu_count()))) return false;
  p->Kp = (K + 63) / 64 * 64;
  p->slots = syrk_ragged_workspace_bytes(M, K);
  p->x = align_up(p->slots, 256);   // (a copy has as many stages, and so the same pieces)
  // the last 256 bytes of a workspace are left alone: the tickets of the 256-tiles' last rounds are counted there
  p->total = p->x + (whole_tiles(M, K) ? 0 : align_up((size_t)M * p->Kp * 2, 256)) + 256;
  return true;
}
// Both X and Y as copies padded to whole 256-tiles, where that is estimated to be faster (syrk_padded_pays), or, with a knob set,
// to the 128- or 256-tiles of the schedules that it speaks of.
struct SyrkPad { int Mp, Kp; size_t x, y, gemm, total; };
static SyrkPad syrk_pad_layout(int M, int K) {
  SyrkPad p;
  const int edge = any_knob_set() && M <= 2816 ? 128 : 256;
  p.Mp = (M + edge - 1) / edge * edge;
  p.Kp = (K + 63) / 64 * 64;
  p.x = 0;
  p.y = align_up((size_t)p.Mp * p.Kp * 2, 256);
  p.gemm = p.y + align_up((size_t)p.Mp * p.Mp * 2, 256);
  p.total = p.gemm + gemm_fast_workspace_bytes(p.Mp, p.Mp, 1);
  return p;
}

size_t fm_syrk_workspace_bytes(int M, int K) {
  if (M <= 0) return 0;
  size_t need = gemm_fast_workspace_bytes(M, M, 1);
  SyrkRagged r;
  if (!syrk_ragged_layout(M, K, &r)) return need;
  if (r.total > need) need = r.total;
  // (rows may lie on lines or not, and Y's rows allow 16-byte stores or not)
  if ((any_knob_set() && !whole_tiles(M, K)) || (K % 64 == 0 && syrk_padded_pays(M, K, kRowsLines, true)) ||
      ((!whole_tiles(M, K) || M > 15 * 256) && syrk_padded_pays(M, K, kRowsAny, true))) {
    const SyrkPad p = syrk_pad_layout(M, K);
    if (p.total > need) need = p.total;
  }
  if (!whole_tiles(M, K)) {   // what the interface promises room for, whichever way is taken: X and Y padded to 128-tiles
    const size_t Mp = (size_t)(M + 127) / 128 * 128, both = Mp * (r.Kp + Mp) * 2;
    if (both > need) need = both;
  }
  return need;
}

size_t fm_syrk_f32_workspace_bytes(int M, int K) { return M <= 0 || K <= 0 ? 0 : syrk_f32_workspace_bytes(M, K); }

static int syrk_impl(const void* X, int64_t ldx, void* Y, int64_t ldy_row, int64_t ldy_col, int M, int K,
                     void* ws, size_t ws_bytes, fm_stream_t stream, int elem, bool may_copy = true) {
  if (M < 0 || K < 0) return FM_ERR_SHAPE;
  if (M == 0) return FM_OK;
  if (!X && K > 0) return FM_ERR_NULL;
  if (!Y) return FM_ERR_NULL;
  if (ldx < K) return FM_ERR_STRIDE;
  if (ldy_row == 0 || ldy_col == 0) return FM_ERR_STRIDE;
  if (M > 1) {
    // distinct (i, j) must not share an address: the larger stride has to step over a whole line
    // of the smaller one (true of every dense or padded row- or column-major layout)
    const int64_t ar = ldy_row < 0 ? -ldy_row : ldy_row, ac = ldy_col < 0 ? -ldy_col : ldy_col;
    const int64_t lo = ar < ac ? ar : ac, hi = ar < ac ? ac : ar;
    if (hi < (int64_t)M * lo) return FM_ERR_STRIDE;
  }
  const int es = elem == kElemF32 ? 4 : 2;
  if (misaligned(X, es) || misaligned(Y, es)) return FM_ERR_ALIGN;
  {   // Y must not overlap X: every tile of Y is written while other tiles still read X
    const int64_t ar = ldy_row < 0 ? -ldy_row : ldy_row, ac = ldy_col < 0 ? -ldy_col : ldy_col;
    const int64_t back = (ldy_row < 0 ? (M - 1) * ar : 0) + (ldy_col < 0 ? (M - 1) * ac : 0);
    Range y;
    y.lo = reinterpret_cast<uintptr_t>(Y) - (uintptr_t)(back * es);
    y.hi = y.lo + (uintptr_t)(((M - 1) * (ar + ac) + 1) * es);
    if (K > 0 && overlaps(mat_range(X, M, K, ldx, es), y)) return FM_ERR_ALIAS;
  }
  hipStream_t hs = static_cast<hipStream_t>(stream);
  if (elem == kElemF32)
    return hip_status(launch_syrk_f32(static_cast<const float*>(X), ldx, static_cast<float*>(Y), ldy_row, ldy_col, M, K,
                                      usable_ws(ws), ws_bytes, hs));
  GemmArgs a = {};
  a.E = nullptr; a.lde = 0;
  a.alpha = 0.0f; a.beta = 1.0f; a.symmetric = 1; a.elem = elem;
  // Y is symmetric, so a unit stride in either direction makes its lines rows for the write-out
  const int64_t ldy = ldy_col == 1 ? ldy_row : ldy_row == 1 ? ldy_col : 0;
  const uintptr_t w0 = reinterpret_cast<uintptr_t>(ws);
  auto room = [&](size_t need) {   // a workspace of that size which is nobody's operand
    const Range w = {w0, w0 + need};
    return need == 0 || (usable_ws(ws) && ws_bytes >= need && !overlaps(mat_range(X, M, K, ldx, es), w) && !overlaps(mat_range(Y, M, M, ldy, es), w));
  };
  SyrkRagged r;
  if (ldy >= M && syrk_ragged_layout(M, K, &r)) {
    const bf16_t* const x = static_cast<const bf16_t*>(X);
    bf16_t* const y = static_cast<bf16_t*>(Y);
    const int how = syrk_ragged_reads(x, ldx, K);
    const SyrkPad p = syrk_pad_layout(M, K);
    const bool aligned = ldy % 8 == 0 && (reinterpret_cast<uintptr_t>(Y) & 15) == 0;
    const int rows = how == kReadsLines ? kRowsLines : ldx % 32 == 0 ? kRowsHalfLines : kRowsAny;
    // (an odd number of whole tiles off the lines is left to launch_gemm_nt)
    const bool in_place = how == kReadsLines || (how == kReadsRows && !whole_tiles(M, K));
    const bool slots = room(r.slots ? r.slots + 256 : 0), forced = any_knob_set();   // (a knob has left whole tiles to launch_gemm_nt)
    // (whole tiles off the lines, padded or by the pairs of workgroups of launch_gemm_nt: 10112 x 8192 686 us / 1082; few of them stay there)
    if (may_copy && (how == kReadsLines || !whole_tiles(M, K) || M > 15 * 256) && (forced || syrk_padded_pays(M, K, rows, aligned)) && room(p.total)) {
      unsigned char* w = static_cast<unsigned char*>(ws);
      bf16_t* Xp = reinterpret_cast<bf16_t*>(w + p.x);
      bf16_t* Yp = reinterpret_cast<bf16_t*>(w + p.y);
      if (launch_copy2d_batched(x, ldx, 0, &Xp, p.Kp, 1, M, K, p.Mp, p.Kp, hs)) return FM_ERR_LAUNCH;
      a.A = a.B = Xp; a.lda = a.ldb = p.Kp;
      a.C = a.C2 = Yp; a.c_rs = a.c2_rs = p.Mp; a.c_cs = a.c2_cs = 1;
      a.Ma = a.Nb = p.Mp; a.Kc = p.Kp;
      if (launch_gemm_nt(a, w + p.gemm, ws_bytes - p.gemm, hs)) return FM_ERR_LAUNCH;
      return hip_status(launch_copy2d_batched(Yp, p.Mp, 0, &y, ldy, 1, M, M, M, M, hs));
    }
    const bool copy_wanted = how == kReadsNot || (how == kReadsRows && syrk_copy_pays(M, K, rows == kRowsHalfLines));
    if (!forced && in_place && slots && !copy_wanted)
      return hip_status(launch_syrk_ragged(x, ldx, y, ldy, M, K, elem == kElemF16, ws, r.slots, hs));
    if (!forced && may_copy && !whole_tiles(M, K) && room(r.total)) {
      bf16_t* copy = reinterpret_cast<bf16_t*>(static_cast<unsigned char*>(ws) + r.x);
      if (launch_copy2d_batched(x, ldx, 0, &copy, r.Kp, 1, M, K, M, r.Kp, hs)) return FM_ERR_LAUNCH;
      return hip_status(launch_syrk_ragged(copy, r.Kp, y, ldy, M, r.Kp, elem == kElemF16, ws, r.slots, hs));
    }
    // no room for a copy, or none allowed: in place where the rows can be read, with whole tiles if there is no room for parts either
    // (3000 x 5000 75 us, the general schedule 99)
    if (!forced && in_place && !whole_tiles(M, K))
      return hip_status(launch_syrk_ragged(x, ldx, y, ldy, M, K, elem == kElemF16, slots ? ws : nullptr, slots ? r.slots : 0, hs));
  }
  a.A = a.B = static_cast<const bf16_t*>(X); a.lda = a.ldb = ldx;
  a.C = a.C2 = static_cast<bf16_t*>(Y);
  a.c_rs = a.c2_rs = ldy_row; a.c_cs = a.c2_cs = ldy_col;
  a.Ma = a.Nb = M; a.Kc = K;
  return hip_status(launch_gemm_nt(a, usable_ws(ws), ws_bytes, hs));
}

int fm_syrk_bf16(const void* X, int64_t ldx, void* Y, int64_t ldy_row, int64_t ldy_col, int M, int K,
                 void* ws, size_t ws_bytes, fm_stream_t stream) {
  return syrk_impl(X, ldx, Y, ldy_row, ldy_col, M, K, ws, ws_bytes, stream, kElemBf16);
}

int fm_syrk_bf16_static(const void* X, int64_t ldx, void* Y, int64_t ldy_row, int64_t ldy_col, int M, int K,
                        fm_stream_t stream) {
  if (M > FM_STATIC_MAX_M || K > FM_STATIC_MAX_K) return FM_ERR_SHAPE;
  void* scratch = nullptr;
  const int rc = static_scratch(&scratch);
  if (rc != FM_OK) return rc;
  // the schedules, and the bits, of fm_syrk_bf16 given a workspace of these 64 MiB (no padded copies)
  return syrk_impl(X, ldx, Y, ldy_row, ldy_col, M, K, scratch, kStaticScratchBytes, stream, kElemBf16, false);
}

int fm_syrk_f16(const void* X, int64_t ldx, void* Y, int64_t ldy_row, int64_t ldy_col, int M, int K,
                void* ws, size_t ws_bytes, fm_stream_t stream) {
  return syrk_impl(X, ldx, Y, ldy_row, ldy_col, M, K, ws, ws_bytes, stream, kElemF16);
}

int fm_syrk_f32(const void* X, int64_t ldx, void* Y, int64_t ldy_row, int64_t ldy_col, int M, int K,
                void* ws, size_t ws_bytes, fm_stream_t stream) {
  return syrk_impl(X, ldx, Y, ldy_row, ldy_col, M, K, ws, ws_bytes, stream, kElemF32);
}

int fm_syrk_poly_bf16(const void* A, int64_t lda, void* P, int64_t ldp, int M, float b, float c,
                      float* diag_out, void* ws, size_t ws_bytes, fm_stream_t stream) {
  if (M < 0) return FM_ERR_SHAPE;
  if (M == 0) return FM_OK;
  if (!A || !P) return FM_ERR_NULL;
  if (lda < M || ldp < M) return FM_ERR_STRIDE;
  if (misaligned(A, 2) || misaligned(P, 2) || misaligned(diag_out, 4)) return FM_ERR_ALIGN;
  if (overlaps(mat_range(A, M, M, lda, 2), mat_range(P, M, M, ldp, 2))) return FM_ERR_ALIAS;
  if (diag_out && (overlaps(mat_range(diag_out, 1, M, M, 4), mat_range(A, M, M, lda, 2)) ||
                   overlaps(mat_range(diag_out, 1, M, M, 4), mat_range(P, M, M, ldp, 2))))
    return FM_ERR_ALIAS;
  GemmArgs a = {};
  a.A = a.B = a.E = a.ET = static_cast<const bf16_t*>(A); a.lda = a.ldb = a.lde = a.ldet = lda;   // A is symmetric
  a.C = a.C2 = static_cast<bf16_t*>(P);
  a.c_rs = a.c2_rs = ldp; a.c_cs = a.c2_cs = 1;
  a.Ma = a.Nb = a.Kc = M;
  a.alpha = b; a.beta = c; a.symmetric = 1;
  a.diag_out = diag_out;
  return hip_status(launch_gemm_nt(a, usable_ws(ws), ws_bytes, static_cast<hipStream_t>(stream)));
}

int fm_gemm_axpby_bf16(const void* P, int64_t ldp, const void* XT, int64_t ldxt, const void* X,
                       int64_t ldx, void* Xout, int64_t ldo, void* XoutT, int64_t ldot, int M, int K,
                       float alpha, const float* row_alpha, void* ws, size_t ws_bytes,
                       fm_stream_t stream) {
  if (M < 0 || K < 0) return FM_ERR_SHAPE;
  if (M == 0 || K == 0) return FM_OK;
  if (!P || !XT || !X) return FM_ERR_NULL;
  if (!Xout && !XoutT) return FM_ERR_NULL;
  if (ldp < M || ldxt < M || ldx < K) return FM_ERR_STRIDE;
  if ((Xout && ldo < K) || (XoutT && ldot < M)) return FM_ERR_STRIDE;
  if (misaligned(P, 2) || misaligned(XT, 2) || misaligned(X, 2) || misaligned(Xout, 2) ||
      misaligned(XoutT, 2) || misaligned(row_alpha, 4))
    return FM_ERR_ALIGN;
  const Range in[3] = {mat_range(P, M, M, ldp, 2), mat_range(XT, K, M, ldxt, 2),
                       mat_range(X, M, K, ldx, 2)};
  const Range o1 = mat_range(Xout, M, K, ldo, 2), o2 = mat_range(XoutT, K, M, ldot, 2);
  for (int i = 0; i < 3; ++i) {
    if (Xout && overlaps(in[i], o1)) return FM_ERR_ALIAS;
    if (XoutT && overlaps(in[i], o2)) return FM_ERR_ALIAS;
  }
  if (Xout && XoutT && overlaps(o1, o2)) return FM_ERR_ALIAS;
  GemmArgs a = {};
  a.A = static_cast<const bf16_t*>(P); a.lda = ldp;
  a.B = static_cast<const bf16_t*>(XT); a.ldb = ldxt;
  a.E = static_cast<const bf16_t*>(X); a.lde = ldx;
  a.ET = a.B; a.ldet = ldxt;
  a.C = static_cast<bf16_t*>(Xout); a.c_rs = ldo; a.c_cs = 1;
  a.C2 = static_cast<bf16_t*>(XoutT); a.c2_rs = ldot; a.c2_cs = 1;
  a.Ma = M; a.Nb = K; a.Kc = M;
  a.alpha = alpha; a.beta = 1.0f; a.symmetric = 0;
  a.row_alpha = row_alpha;
  return hip_status(launch_gemm_nt(a, usable_ws(ws), ws_bytes, static_cast<hipStream_t>(stream)));
}

size_t fm_sumsq_workspace_bytes(void) { return kSumsqBlocks * sizeof(float); }

int fm_sumsq(const void* G, int dtype, int rows, int cols, int64_t ldg, float* out, void* ws,
             size_t ws_bytes, fm_stream_t stream) {
  if (bad_dtype(dtype)) return FM_ERR_DTYPE;
  if (rows < 0 || cols < 0) return FM_ERR_SHAPE;
  if (!out) return FM_ERR_NULL;
  if (!G && (int64_t)rows * cols > 0) return FM_ERR_NULL;
  if (ldg < cols) return FM_ERR_STRIDE;
  if (!ws || ws_bytes < fm_sumsq_workspace_bytes()) return FM_ERR_WORKSPACE;
  if (misaligned(G, dtype_size(dtype)) || misaligned(out, 4) || misaligned(ws, 4)) return FM_ERR_ALIGN;
  return hip_status(launch_sumsq(G, dtype, rows, cols, ldg, out, static_cast<float*>(ws),
                                 static_cast<hipStream_t>(stream)));
}

int fm_scale_cast_bf16(const void* G, int dtype, int rows, int cols, int64_t ldg, const float* sumsq,
                       float eps, void* D, int64_t ldd, void* T, int64_t ldt, fm_stream_t stream) {
  if (bad_dtype(dtype)) return FM_ERR_DTYPE;
  if (rows < 0 || cols < 0) return FM_ERR_SHAPE;
  if (rows == 0 || cols == 0) return FM_OK;
  if (!G || !sumsq) return FM_ERR_NULL;
  if (!D && !T) return FM_ERR_NULL;
  if (ldg < cols || (D && ldd < cols) || (T && ldt < rows)) return FM_ERR_STRIDE;
  if (misaligned(G, dtype_size(dtype)) || misaligned(D, 2) || misaligned(T, 2) || misaligned(sumsq, 4))
    return FM_ERR_ALIGN;
  const Range g = mat_range(G, rows, cols, ldg, dtype_size(dtype));
  if (D && overlaps(g, mat_range(D, rows, cols, ldd, 2))) return FM_ERR_ALIAS;
  if (T && overlaps(g, mat_range(T, cols, rows, ldt, 2))) return FM_ERR_ALIAS;
  return hip_status(launch_scale_cast(G, dtype, rows, cols, ldg, sumsq, eps, static_cast<bf16_t*>(D),
                                      ldd, static_cast<bf16_t*>(T), ldt,
                                      static_cast<hipStream_t>(stream)));
}

size_t fm_newtonschulz_batched_workspace_bytes(int batch, int rows, int cols) {
  if (batch <= 0 || rows <= 0 || cols <= 0) return 0;
  return ns_layout(batch, rows, cols, true).total;
}

size_t fm_newtonschulz_batched_min_workspace_bytes(int batch, int rows, int cols) {
  if (batch <= 0 || rows <= 0 || cols <= 0) return 0;
  const size_t best = ns_layout(batch, rows, cols, true).total, launches = ns_layout(batch, rows, cols, false).total;
  return best < launches ? best : launches;
}

size_t fm_newtonschulz_workspace_bytes(int rows, int cols) {
  return fm_newtonschulz_batched_workspace_bytes(1, rows, cols);
}

// the momentum update that comes before: of g and buf, one of which is G
struct NsMomentum { void* const* g; void* const* buf; float w_buf, w_nes; int nesterov; };

static int ns_impl(const void* const* G, int dtype, int batch, int rows, int cols, int64_t ldg, void* const* out, int64_t ldout, int steps,
                   float a, float b, float c, float eps, void* ws, size_t ws_bytes, fm_stream_t stream, const NsMomentum* mom) {
  if (bad_dtype(dtype)) return FM_ERR_DTYPE;
  if (rows < 0 || cols < 0 || steps < 0 || batch < 0 || batch > kMaxBatch) return FM_ERR_SHAPE;
  if (rows == 0 || cols == 0 || batch == 0) return FM_OK;
  if (!G || !out) return FM_ERR_NULL;
  if (ldg < cols || ldout < cols) return FM_ERR_STRIDE;
  for (int i = 0; i < batch; ++i) {
    if (!G[i] || !out[i]) return FM_ERR_NULL;
    if (misaligned(G[i], dtype_size(dtype)) || misaligned(out[i], 2)) return FM_ERR_ALIGN;
    const Range oi = mat_range(out[i], rows, cols, ldout, 2);
    for (int j = 0; j < batch; ++j) {
      if (overlaps(mat_range(G[j], rows, cols, ldg, dtype_size(dtype)), oi)) return FM_ERR_ALIAS;
      if (j != i && overlaps(mat_range(out[j], rows, cols, ldout, 2), oi)) return FM_ERR_ALIAS;
    }
  }
  NsLayout l = ns_layout(batch, rows, cols, true);
  if (l.flow && ws_bytes < l.total) l = ns_layout(batch, rows, cols, false);   // which keeps two iterates, not one for every step
  if (!ws || ws_bytes < l.total) return FM_ERR_WORKSPACE;
  if (reinterpret_cast<uintptr_t>(ws) % 256 != 0) return FM_ERR_ALIGN;
  {
    Range w;
    w.lo = reinterpret_cast<uintptr_t>(ws);
    w.hi = w.lo + l.total;
    for (int i = 0; i < batch; ++i)
      if (overlaps(mat_range(G[i], rows, cols, ldg, dtype_size(dtype)), w) ||
          overlaps(mat_range(out[i], rows, cols, ldout, 2), w))
        return FM_ERR_ALIAS;
  }

  // sums of squares of G, behind its momentum update or with it
  auto squares = [&](float* partials, unsigned* zero, int n_zero) -> int {
    hipStream_t hs = static_cast<hipStream_t>(stream);
    const int64_t n = (int64_t)rows * cols;
    int rc = 0;
    if (mom) {
      if (launch_momentum_sumsq_batched(mom->g, mom->buf, batch, dtype, n, mom->w_buf, mom->w_nes, mom->nesterov, partials, hs, zero, n_zero, &rc))
        return rc;
      rc = launch_momentum_nesterov_batched(mom->g, mom->buf, batch, dtype, n, mom->w_buf, mom->w_nes, mom->nesterov, hs);
      if (rc) return rc;
    }
    return launch_sumsq_parts_batched(G, batch, dtype, rows, cols, ldg, partials, hs, zero, n_zero);
  };
  unsigned char* w = static_cast<unsigned char*>(ws);
  if (l.flow && steps > 0) {
    hipStream_t hs = static_cast<hipStream_t>(stream);
    const bool tall = rows > cols;
    float* sumsq = reinterpret_cast<float*>(w + l.partials);
    const int parts = sumsq_parts((int64_t)rows * cols);
    unsigned* counters = reinterpret_cast<unsigned*>(w + l.counters);
    const int n_counters = flow_counter_words(batch, steps < kFlowSteps ? steps : kFlowSteps);
    const int64_t mk = (int64_t)l.M * l.K;
    bf16_t* X = reinterpret_cast<bf16_t*>(w + l.x[0]);
    if (squares(sumsq, counters, n_counters)) return FM_ERR_LAUNCH;
    bf16_t* x[kMaxBatch];
    for (int i = 0; i < batch; ++i) x[i] = X + i * mk;
    if (launch_scale_cast_batched(G, batch, dtype, rows, cols, ldg, sumsq, parts, eps, tall ? nullptr : x, l.K, tall ? x : nullptr, l.K,
                                  hs, tall ? l.K : l.M, tall ? l.M : l.K))
      return FM_ERR_LAUNCH;
    FlowProblem f = {};
    f.A = reinterpret_cast<bf16_t*>(w + l.a); f.P = reinterpret_cast<bf16_t*>(w + l.p); f.a_step = (int64_t)batch * l.M * l.M;
    f.pdiag = reinterpret_cast<float*>(w + l.pdiag); f.d_step = (int64_t)batch * l.pdiag_stride; f.d_mat = (int64_t)l.pdiag_stride;
    f.M = l.M; f.K = l.K; f.batch = batch; f.edge_s = l.edge_s; f.edge_x = l.edge_x;
    f.a = a; f.b = b; f.c = c;
    f.counters = counters;
    const int64_t bmk = batch * mk;
    for (int i = 0; i * kFlowSteps < steps; ++i) {
      const NsFlowLaunch n = ns_flow_launch(steps, i);
      f.steps = n.steps;
      f.X = X + n.from * bmk; f.x_step = n.turn * bmk;
      const bool last = n.first + n.steps == steps;
      // what is not the last launch leaves its result in the slot behind its own, from where the next one
      // goes the other way
      void* o[kMaxBatch];
      for (int j = 0; j < batch; ++j) o[j] = last ? out[j] : (void*)(f.X + n.steps * f.x_step + j * mk);
      f.out = o;
      f.ldout = last ? ldout : l.K;
      f.rows = last ? rows : l.M; f.cols = last ? cols : l.K; f.tall = last && tall;
      if (i > 0 && launch_zero_words(counters, n_counters, hs)) return FM_ERR_LAUNCH;
      if (launch_ns_flow(f, hs)) return FM_ERR_LAUNCH;
    }
    return FM_OK;
  }
  void* gws = w + l.gemm;
  const size_t gws_bytes = l.total - l.gemm;
  hipStream_t hs = static_cast<hipStream_t>(stream);
  const bool tall = rows > cols;
  const bool padded = l.padded && steps > 0;
  const int M = padded ? l.M : (tall ? cols : rows), K = padded ? l.K : (tall ? rows : cols);
  const int64_t mk = (int64_t)M * K, mm = (int64_t)M * M;

  // The iteration runs on X (M x K) with M <= K.  G is X when it is wide and X^T when it is
  // tall, so the scaled cast of G is X in one case and X^T in the other.
  bf16_t* X = reinterpret_cast<bf16_t*>(w + l.x[0]);
  bf16_t* XT = reinterpret_cast<bf16_t*>(w + l.xt[0]);
  {
    // Frobenius norms (partial sums), then the scaled bf16 cast in both orientations: one launch each for the
    // batch.  The last 256 bytes of the GEMM scratch hold the ticket word of the sub-tile rounds: whatever
    // the caller's memory held there could pass for a launch number no launch ever reaches (the products
    // would still be right, on the fixed assignment of sub-tiles), so it starts from zero.
    float* sumsq = reinterpret_cast<float*>(w + l.partials);
    const int parts = sumsq_parts((int64_t)rows * cols);
    const bool word = steps > 0 && gws_bytes >= 256;
    if (squares(sumsq, word ? reinterpret_cast<unsigned*>(w + l.total - 256) : nullptr, word ? 64 : 0)) return FM_ERR_LAUNCH;
    bf16_t* d[kMaxBatch];
    bf16_t* t[kMaxBatch];
    for (int i = 0; i < batch; ++i) {
      if (steps == 0) { d[i] = static_cast<bf16_t*>(out[i]); t[i] = nullptr; }
      else if (!tall) { d[i] = X + i * mk; t[i] = XT + i * mk; }
      else            { d[i] = XT + i * mk; t[i] = X + i * mk; }
    }
    const int64_t ldd = steps == 0 ? ldout : (!tall ? K : M), ldt = !tall ? M : K;
    // with padding: G's orientation is (tall ? K x M : M x K) there, and what lies beyond G is zeroed
    if (launch_scale_cast_batched(G, batch, dtype, rows, cols, ldg, sumsq, parts, eps, d, ldd,
                                  steps == 0 ? nullptr : t, ldt, hs, padded ? (tall ? K : M) : rows,
                                  padded ? (tall ? M : K) : cols))
      return FM_ERR_LAUNCH;
  }
  if (steps == 0) return FM_OK;

  bf16_t* A = reinterpret_cast<bf16_t*>(w + l.a);
  bf16_t* P = reinterpret_cast<bf16_t*>(w + l.p);
  float* pdiag = reinterpret_cast<float*>(w + l.pdiag);   // diagonal of P, kept in fp32
  // Sides of whole 128-tiles, padded to 256: the last product writes what exists of its result itself (24 of 5504 x 2048: 167 us
  // for the copy out of the padded one).
  bool cut_out = padded && rows % 128 == 0 && cols % 128 == 0 && ldout % 8 == 0 && ldout < (1 << 21);
  for (int i = 0; i < batch; ++i) cut_out = cut_out && (reinterpret_cast<uintptr_t>(out[i]) & 15) == 0;
  for (int s = 0; s < steps; ++s) {
    const bool last = s + 1 == steps;
    bf16_t* Xn = reinterpret_cast<bf16_t*>(w + l.x[(s + 1) & 1]);
    bf16_t* XTn = reinterpret_cast<bf16_t*>(w + l.xt[(s + 1) & 1]);
    GemmArgs g = {};
    // A = X X^T
    g.A = g.B = X; g.lda = g.ldb = K; g.bs_a = g.bs_b = mk;
    g.C = g.C2 = A; g.c_rs = g.c2_rs = M; g.c_cs = g.c2_cs = 1; g.bs_c = g.bs_c2 = mm;
    g.Ma = g.Nb = M; g.Kc = K; g.beta = 1.0f; g.symmetric = 1; g.batch = batch;
    if (launch_gemm_nt(g, gws, gws_bytes, hs)) return FM_ERR_LAUNCH;
    // P = b A + c A A, diagonal in fp32
    g = GemmArgs{};
    g.A = g.B = g.E = g.ET = A; g.lda = g.ldb = g.lde = g.ldet = M;
    g.bs_a = g.bs_b = g.bs_e = g.bs_et = mm;
    g.C = g.C2 = P; g.c_rs = g.c2_rs = M; g.c_cs = g.c2_cs = 1; g.bs_c = g.bs_c2 = mm;
    g.Ma = g.Nb = g.Kc = M; g.alpha = b; g.beta = c; g.symmetric = 1; g.batch = batch;
    g.diag_out = pdiag; g.bs_do = (int64_t)l.pdiag_stride;
    if (launch_gemm_nt(g, gws, gws_bytes, hs)) return FM_ERR_LAUNCH;
    // X' = (a + diag) X + P X, and its transpose; the last step writes the caller's orientation only
    g = GemmArgs{};
    g.A = P; g.lda = M; g.bs_a = mm;
    g.B = XT; g.ldb = M; g.bs_b = mk;
    g.E = X; g.lde = K; g.bs_e = mk;
    g.ET = XT; g.ldet = M; g.bs_et = mk;
    g.Ma = M; g.Nb = K; g.Kc = M; g.alpha = a; g.beta = 1.0f; g.symmetric = 0; g.batch = batch;
    g.row_alpha = pdiag; g.bs_ra = (int64_t)l.pdiag_stride;
    g.c_cs = g.c2_cs = 1;
    if (!last) {
      g.C = Xn; g.c_rs = K; g.bs_c = mk;
      g.C2 = XTn; g.c2_rs = M; g.bs_c2 = mk;
    } else if (padded && !cut_out) {  // the orientation the caller wants, into the workspace, and from there out
      if (!tall) { g.C = Xn; g.c_rs = K; g.bs_c = mk; }
      else { g.C2 = XTn; g.c2_rs = M; g.bs_c2 = mk; }
    } else if (!tall) {   // the result has G's shape: X itself
      g.C = static_cast<bf16_t*>(out[0]); g.c_rs = ldout; g.use_c_list = 1;
      for (int i = 0; i < batch; ++i) g.c_list[i] = static_cast<bf16_t*>(out[i]);
    } else {              // or its transpose
      g.C2 = static_cast<bf16_t*>(out[0]); g.c2_rs = ldout; g.use_c2_list = 1;
      for (int i = 0; i < batch; ++i) g.c2_list[i] = static_cast<bf16_t*>(out[i]);
    }
    if (last && cut_out) { g.rows_v = tall ? cols : rows; g.cols_v = tall ? rows : cols; }
    if (launch_gemm_nt(g, gws, gws_bytes, hs)) return FM_ERR_LAUNCH;
    X = Xn; XT = XTn;
  }
  if (padded && !cut_out) {
    bf16_t* o[kMaxBatch];
    for (int i = 0; i < batch; ++i) o[i] = static_cast<bf16_t*>(out[i]);
    if (launch_copy2d_batched(tall ? XT : X, tall ? M : K, mk, o, ldout, batch, rows, cols, rows, cols, hs))
      return FM_ERR_LAUNCH;
  }
  return FM_OK;
}

int fm_newtonschulz_batched_bf16(const void* const* G, int dtype, int batch, int rows, int cols,
                                 int64_t ldg, void* const* out, int64_t ldout, int steps, float a,
                                 float b, float c, float eps, void* ws, size_t ws_bytes,
                                 fm_stream_t stream) {
  return ns_impl(G, dtype, batch, rows, cols, ldg, out, ldout, steps, a, b, c, eps, ws, ws_bytes, stream, nullptr);
}

int fm_newtonschulz_bf16(const void* G, int dtype, int rows, int cols, int64_t ldg, void* out,
                         int64_t ldout, int steps, float a, float b, float c, float eps, void* ws,
                         size_t ws_bytes, fm_stream_t stream) {
  const void* gs[1] = {G};
  void* os[1] = {out};
  if (rows > 0 && cols > 0 && (!G || !out)) return FM_ERR_NULL;
  return fm_newtonschulz_batched_bf16(gs, dtype, 1, rows, cols, ldg, os, ldout, steps, a, b, c, eps,
                                      ws, ws_bytes, stream);
}

int fm_momentum_nesterov(void* g, void* buf, int dtype, int64_t n, float w_buf, float w_nes,
                         int nesterov, fm_stream_t stream) {
  if (bad_dtype(dtype)) return FM_ERR_DTYPE;
  if (n < 0) return FM_ERR_SHAPE;
  if (n == 0) return FM_OK;
  if (!g || !buf) return FM_ERR_NULL;
  const int esz = dtype_size(dtype);
  if (misaligned(g, esz) || misaligned(buf, esz)) return FM_ERR_ALIGN;
  if (overlaps(mat_range(g, 1, n, n, esz), mat_range(buf, 1, n, n, esz))) return FM_ERR_ALIAS;
  return hip_status(launch_momentum_nesterov(g, buf, dtype, n, w_buf, w_nes, nesterov,
                                             static_cast<hipStream_t>(stream)));
}

static int momentum_checks(void* const* g, void* const* buf, int batch, int dtype, int64_t n) {
  if (!g || !buf) return FM_ERR_NULL;
  const int esz = dtype_size(dtype);
  for (int i = 0; i < batch; ++i) {
    if (!g[i] || !buf[i]) return FM_ERR_NULL;
    if (misaligned(g[i], esz) || misaligned(buf[i], esz)) return FM_ERR_ALIGN;
    for (int j = 0; j < batch; ++j) {
      if (overlaps(mat_range(g[i], 1, n, n, esz), mat_range(buf[j], 1, n, n, esz))) return FM_ERR_ALIAS;
      if (j != i && (overlaps(mat_range(g[i], 1, n, n, esz), mat_range(g[j], 1, n, n, esz)) ||
                     overlaps(mat_range(buf[i], 1, n, n, esz), mat_range(buf[j], 1, n, n, esz))))
        return FM_ERR_ALIAS;
    }
  }
  return FM_OK;
}

int fm_momentum_nesterov_batched(void* const* g, void* const* buf, int batch, int dtype, int64_t n,
                                 float w_buf, float w_nes, int nesterov, fm_stream_t stream) {
  if (bad_dtype(dtype)) return FM_ERR_DTYPE;
  if (n < 0 || batch < 0 || batch > kMaxBatch) return FM_ERR_SHAPE;
  if (n == 0 || batch == 0) return FM_OK;
  const int rc = momentum_checks(g, buf, batch, dtype, n);
  if (rc != FM_OK) return rc;
  return hip_status(launch_momentum_nesterov_batched(g, buf, batch, dtype, n, w_buf, w_nes, nesterov,
                                                     static_cast<hipStream_t>(stream)));
}

int fm_momentum_newtonschulz_batched(void* const* g, void* const* buf, int dtype, int batch, int rows, int cols, float w_buf,
                                     float w_nes, int nesterov, void* const* out, int64_t ldout, int steps, float a, float b,
                                     float c, float eps, void* ws, size_t ws_bytes, fm_stream_t stream) {
  if (bad_dtype(dtype)) return FM_ERR_DTYPE;
  if (rows < 0 || cols < 0 || batch < 0 || batch > kMaxBatch) return FM_ERR_SHAPE;
  if (rows == 0 || cols == 0 || batch == 0) return FM_OK;
  const int64_t n = (int64_t)rows * cols;
  const int rc = momentum_checks(g, buf, batch, dtype, n);
  if (rc != FM_OK) return rc;
  if (!out) return FM_ERR_NULL;
  // what is not orthogonalised is written too: neither outputs nor scratch may lie on it
  void* const* const other = nesterov ? buf : g;
  const Range w = {reinterpret_cast<uintptr_t>(ws), reinterpret_cast<uintptr_t>(ws) + ws_bytes};
  for (int i = 0; i < batch; ++i) {
    const Range r = mat_range(other[i], rows, cols, cols, dtype_size(dtype));
    if (overlaps(r, w)) return FM_ERR_ALIAS;
    for (int j = 0; j < batch; ++j)
      if (overlaps(r, mat_range(out[j], rows, cols, ldout, 2))) return FM_ERR_ALIAS;
  }
  const NsMomentum mom = {g, buf, w_buf, w_nes, nesterov};
  return ns_impl(nesterov ? g : buf, dtype, batch, rows, cols, cols, out, ldout, steps, a, b, c, eps, ws, ws_bytes, stream, &mom);
}

int fm_weight_update_batched(void* const* p, int p_dtype, const void* const* u_bf16, int batch, int64_t n,
                             float decay_mul, float alpha, fm_stream_t stream) {
  if (bad_dtype(p_dtype)) return FM_ERR_DTYPE;
  if (n < 0 || batch < 0 || batch > kMaxBatch) return FM_ERR_SHAPE;
  if (n == 0 || batch == 0) return FM_OK;
  if (!p || !u_bf16) return FM_ERR_NULL;
  const int esz = dtype_size(p_dtype);
  for (int i = 0; i < batch; ++i) {
    if (!p[i] || !u_bf16[i]) return FM_ERR_NULL;
    if (misaligned(p[i], esz) || misaligned(u_bf16[i], 2)) return FM_ERR_ALIGN;
    for (int j = 0; j < batch; ++j) {
      if (overlaps(mat_range(p[i], 1, n, n, esz), mat_range(u_bf16[j], 1, n, n, 2))) return FM_ERR_ALIAS;
      if (j != i && overlaps(mat_range(p[i], 1, n, n, esz), mat_range(p[j], 1, n, n, esz))) return FM_ERR_ALIAS;
    }
  }
  return hip_status(launch_weight_update_batched(p, reinterpret_cast<const bf16_t* const*>(u_bf16), batch,
                                                 p_dtype, n, decay_mul, alpha,
                                                 static_cast<hipStream_t>(stream)));
}

int fm_weight_update(void* p, int p_dtype, const void* u_bf16, int64_t n, float decay_mul,
                     float alpha, fm_stream_t stream) {
  if (bad_dtype(p_dtype)) return FM_ERR_DTYPE;
  if (n < 0) return FM_ERR_SHAPE;
  if (n == 0) return FM_OK;
  if (!p || !u_bf16) return FM_ERR_NULL;
  const int esz = dtype_size(p_dtype);
  if (misaligned(p, esz) || misaligned(u_bf16, 2)) return FM_ERR_ALIGN;
  if (overlaps(mat_range(p, 1, n, n, esz), mat_range(u_bf16, 1, n, n, 2))) return FM_ERR_ALIAS;
  return hip_status(launch_weight_update(p, p_dtype, static_cast<const bf16_t*>(u_bf16), n,
                                         decay_mul, alpha, static_cast<hipStream_t>(stream)));
}

}  // extern "C"
