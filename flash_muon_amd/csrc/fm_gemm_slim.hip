// 64x128 tiles of the NT contraction, one workgroup of four waves per CU, for products whose 128x128 tiles are at most
// half as many as CUs: twice the workgroups on three quarters of the operand bytes each.
//
// Bound by the rate at which a CU copies into its LDS (some 90 KB/us, whatever the others do): 24 KiB per 64-wide k stage, 0.27 us,
// where a 128x128 tile takes 0.36 for its 32; the waves' 32x64 blocks read 48 KiB of fragments a stage beside that, and their 16
// MFMAs a stage are a quarter of the time.  So the ring is as deep as the LDS allows, six stages with five on their way.
// us, 128x128 tiles / this: X X^T 1536 x 2048 17.1 / 13.7, 1792 x 4096 27.9 / 22.5, 2048^2 17.8 / 15.1, 2048 x 4096 28.4 / 24.3; five Newton-Schulz steps
// on 6400 x 1600 518 / 506, 1536^2 254 / 231, 2048^2 317 / 290, 2 of 1024 x 4096 335 / 297, 4 of 768 x 3072 327 / 295.
#include "fm_routes.h"
#include "fm_tile128.h"

namespace fm {

namespace {

using t128::copy16;
using t128::mfma16;
using t128::pack2;
using t128::perm_a;
using t128::perm_b;

constexpr int TM = 64, TN = 128, BK = 64, ROW = BK * 2;
constexpr int A_BYTES = TM * ROW, B_BYTES = TN * ROW, STAGE = A_BYTES + B_BYTES, DEPTH = 6;   // 24 KiB, 144 KiB
constexpr int COPIES = 6;   // per wave and stage: 2 of operand A, 4 of B

// 16-byte chunk c of LDS row r sits at c ^ swz(r): any 16 consecutive rows cover all 64 banks, and so do the rows that a diagonal
// item gathers, which come in pairs 16 apart
__device__ __forceinline__ int swz(int row) { return ((row >> 1) & 7) ^ ((row >> 4) & 1); }

struct Frag { bf16x8_t a[2], b[4]; };
struct Lane {
  uint32_t fa[2][2], fb[2][2];   // fragments 0 and 1 (and 2 and 3, 4 KiB further on) of k32 substep kk in slot 0
  uint32_t ldsw;                 // where this wave's copies land inside a slot
  uint32_t voA[2], voB[4];
};

template <int SLOT, int KK>
__device__ __forceinline__ void read_frag(Frag& f, const unsigned char* smem, const Lane& L, int t) {   // read t of 6: a0 b0 .. b3 a1
  if (t == 0 || t == 5) f.a[t == 0 ? 0 : 1] = *reinterpret_cast<const bf16x8_t*>(smem + L.fa[KK][t == 0 ? 0 : 1] + SLOT * STAGE);
  else f.b[t - 1] = *reinterpret_cast<const bf16x8_t*>(smem + L.fb[KK][(t - 1) & 1] + SLOT * STAGE + ((t - 1) >> 1) * 4096);
}

// The stage in SLOT, whose first fragments f0 holds.  Behind the barrier in its middle, before which every wave has read the
// stage and waited for its copies of the next one, the copies of the stage six ahead go into its slot.
template <bool F16, int SLOT>
__device__ __forceinline__ void stage(f32x4_t (&acc)[2][4], Frag& f0, Frag& f1, const unsigned char* smem, const Lane& L, const bf16_t* nA,
                                      const bf16_t* nB) {
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the fragments of the first half
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    if (q < 6) read_frag<SLOT, 1>(f1, smem, L, q);
    acc[q >> 2][q & 3] = mfma16<F16>(f0.a[q >> 2], f0.b[q & 3], acc[q >> 2][q & 3]);
    __builtin_amdgcn_sched_barrier(0);
  }
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((DEPTH - 2) * COPIES) : "memory");
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    if (q < 6) read_frag<(SLOT + 1) % DEPTH, 0>(f0, smem, L, q);
    if (q < 2) copy16(L.voA[q], nA, L.ldsw, SLOT * STAGE + q * 4096);
    else if (q < 6) copy16(L.voB[q - 2], nB, L.ldsw, SLOT * STAGE + A_BYTES + (q - 2) * 4096);
    acc[q >> 2][q & 3] = mfma16<F16>(f1.a[q >> 2], f1.b[q & 3], acc[q >> 2][q & 3]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// ---- a diagonal 128x128 tile of X X^T as one item ------------------------------------------------
// Its panel is operand B's, 16 KiB a stage, and serves as operand A too: the fragments of its rows are gathered from where
// operand B's order keeps them.  Waves 0 and 1 take the lower triangles of the 64x64 squares on the diagonal, three 32x32 blocks each (all four
// of them make these items the last ones to end: 2048^2 16.9 us), waves 2 and 3 a 32x64 half each of the square below them.  T tile rows make T^2 items: 256 of a 2048^2 product, one a CU, where halves of the diagonal tiles would make 272.
struct DLane {
  uint32_t fa[2][4], fb[2][2];   // A fragment i, B fragments 0 and 1 of k32 substep kk in slot 0
  uint32_t ldsw, vo[4];
};
template <int NA> struct DFrag { bf16x8_t a[NA], b[4]; };
// where operand B's order keeps the row that fragment row l of operand A holds
__device__ __forceinline__ int gather_row(int l) { const int r = perm_a(l); return (r & ~31) + ((r & 31) >> 1) + 16 * (r & 1); }

template <int NA, int SLOT, int KK>
__device__ __forceinline__ void read_dfrag(DFrag<NA>& f, const unsigned char* smem, const DLane& L, int t) {
  if (t < NA) f.a[t] = *reinterpret_cast<const bf16x8_t*>(smem + L.fa[KK][t] + SLOT * STAGE);
  else f.b[t - NA] = *reinterpret_cast<const bf16x8_t*>(smem + L.fb[KK][(t - NA) & 1] + SLOT * STAGE + ((t - NA) >> 1) * 4096);
}
// MFMA q of a wave: with four A fragments tiles (0..1, 0..1), (2..3, 0..1) and (2..3, 2..3)
__host__ __device__ constexpr int d_mfmas(int na) { return na == 4 ? 12 : 8; }
__host__ __device__ constexpr int d_i(int na, int q) { return na == 2 ? q >> 2 : q < 4 ? q >> 1 : 2 + ((q >> 1) & 1); }
__host__ __device__ constexpr int d_j(int na, int q) { return na == 2 ? q & 3 : (q & 1) + (q < 8 ? 0 : 2); }
template <bool F16, int NA, int SLOT>
__device__ __forceinline__ void dstage(f32x4_t (&acc)[4][4], DFrag<NA>& f0, DFrag<NA>& f1, const unsigned char* smem, const DLane& L, const bf16_t* nP) {
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
#pragma unroll
  for (int q = 0; q < d_mfmas(NA); ++q) {
    if (q < NA + 4) read_dfrag<NA, SLOT, 1>(f1, smem, L, q);
    f32x4_t& c = acc[d_i(NA, q)][d_j(NA, q)];
    c = mfma16<F16>(f0.a[d_i(NA, q)], f0.b[d_j(NA, q)], c);
    __builtin_amdgcn_sched_barrier(0);
  }
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((DEPTH - 2) * 4) : "memory");
#pragma unroll
  for (int q = 0; q < d_mfmas(NA); ++q) {
    if (q < NA + 4) read_dfrag<NA, (SLOT + 1) % DEPTH, 0>(f0, smem, L, q);
    if (q < 4) copy16(L.vo[q], nP, L.ldsw, SLOT * STAGE + A_BYTES + q * 4096);
    f32x4_t& c = acc[d_i(NA, q)][d_j(NA, q)];
    c = mfma16<F16>(f1.a[d_i(NA, q)], f1.b[d_j(NA, q)], c);
    __builtin_amdgcn_sched_barrier(0);
  }
}
// the first DEPTH stages of the panel are on their way, the first one has landed everywhere
template <bool F16, int NA>
__device__ __forceinline__ void diag_loop(f32x4_t (&acc)[4][4], int nk, const unsigned char* smem, const DLane& L, const bf16_t* gP) {
  const int last = nk - 1;
#pragma unroll
  for (int i = 0; i < NA; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  DFrag<NA> f0, f1;
#pragma unroll
  for (int t = 0; t < NA + 4; ++t) read_dfrag<NA, 0, 0>(f0, smem, L, t);
#define FM_SLIM_DSTAGE(SLOT, S)                                          \
  {                                                                      \
    const int kn = (S) + DEPTH < last ? (S) + DEPTH : last;              \
    dstage<F16, NA, SLOT>(acc, f0, f1, smem, L, gP + kn * BK);           \
    if ((S) + 1 >= nk) break;                                            \
  }
  for (int s = 0;; s += 6) {
    FM_SLIM_DSTAGE(0, s)
    FM_SLIM_DSTAGE(1, s + 1)
    FM_SLIM_DSTAGE(2, s + 2)
    FM_SLIM_DSTAGE(3, s + 3)
    FM_SLIM_DSTAGE(4, s + 4)
    FM_SLIM_DSTAGE(5, s + 5)
  }
#undef FM_SLIM_DSTAGE
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// position -> tile, halves of 128x128 tiles next to each other, in 8x8 blocks of those (upper triangle of a symmetric product)
__device__ __forceinline__ void item_at(const GemmArgs& g, int diag_items, int pos, int& b, int& ti, int& tj, int& h) {
  if (diag_items) {   // those of the tiles off the diagonal, then the diagonal tiles
    const int T = g.tiles_m, off = T * (T - 1);
    b = pos / (T * T);
    pos -= b * T * T;
    h = pos & 1;
    ti = tj = pos - off;
    if (pos < off) {
      band_tri_decode(pos >> 1, T - 1, ti, tj);
      ++tj;
    }
    return;
  }
  h = pos & 1;
  pos >>= 1;
  const int per = g.num_tiles / g.batch;
  b = pos / per;
  pos -= b * per;
  if (g.symmetric) {
    band_tri_decode(pos, g.tiles_m, ti, tj);
  } else {
    const int band = pos / (8 * g.tiles_n), r = pos - band * 8 * g.tiles_n;
    const int rows = g.tiles_m - band * 8 < 8 ? g.tiles_m - band * 8 : 8;
    tj = r / rows;
    ti = band * 8 + (r - tj * rows);
  }
}

constexpr int MIRROR_PITCH = 80;   // bytes per staged column of the mirrored copy: 32 rows and 16 more, for the banks
constexpr int STAGING = 32 * 128 + 64 * MIRROR_PITCH;   // a wave's 32x64 block, by rows and by columns

// the operand E of a block, in the layout of the sums, and what it is multiplied with
struct Pre { uint4 e[2][2]; float al[8]; };
__device__ __forceinline__ void load_e(Pre& pre, const GemmArgs& g, int row0, int col0, int lane) {
  const int n = lane & 15, grp = lane >> 4;
  const bf16_t* const e = g.ET + (int64_t)(col0 + 2 * n) * g.ldet + row0 + 8 * grp;
#pragma unroll
  for (int J = 0; J < 2; ++J)
#pragma unroll
    for (int b = 0; b < 2; ++b) pre.e[J][b] = *reinterpret_cast<const uint4*>(e + (32 * J + b) * g.ldet);
#pragma unroll
  for (int k = 0; k < 8; ++k) pre.al[k] = g.alpha + (g.row_alpha ? g.row_alpha[row0 + 8 * grp + k] : 0.0f);
}

// A wave's 32x64 block at (row0, col0), as in fm_tile128.h: a lane holds rows 8 grp .. + 7 of columns 32 J + 2 n, + 1; both copies go
// through wave-private LDS and out 16 bytes per lane.  `diag`: in a diagonal tile of a symmetric product.  KIND 1 and 2: the upper and lower
// half of a 64x64 square on the diagonal, of which the wave holds columns 0 .. 31 above, whose other columns are written as the
// mirror image of columns 0 .. 31 below.
template <bool F16, int KIND = 0>
__device__ __forceinline__ void write_block(const GemmArgs& g, bool use_e, const Pre& pre, const f32x4_t (&a0)[4], const f32x4_t (&a1)[4],
                                            bool direct, bool mirror, bool diag, int row0, int col0, unsigned char* T, int lane) {
  const int n = lane & 15, grp = lane >> 4;
  const bool dout = diag && g.diag_out != nullptr;
  unsigned char* const T2 = T + 32 * 128;
#pragma unroll
  for (int J = 0; J < (KIND == 1 ? 1 : 2); ++J) {
    float v[2][8];   // [b][8 rows]
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int k = 0; k < 8; ++k) v[b][k] = (k < 4 ? a0 : a1)[2 * J + b][k & 3];
    if (use_e) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const uint32_t e[4] = {pre.e[J][b].x, pre.e[J][b].y, pre.e[J][b].z, pre.e[J][b].w};
#pragma unroll
        for (int k = 0; k < 8; ++k)
          v[b][k] = __builtin_fmaf(pre.al[k], elem_to_f32<F16>((unsigned short)((k & 1) ? (e[k >> 1] >> 16) : (e[k >> 1] & 0xffffu))), g.beta * v[b][k]);
      }
    }
    if (dout && row0 - col0 == 32 * J) {   // this 32x32 sub-block lies on the diagonal: the lanes with n / 4 == grp hold rows 2 n and 2 n + 1 of it
      float dv[2] = {0.0f, 0.0f};
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const bool on = 2 * n + b == 8 * grp + k;
          dv[b] = on ? v[b][k] : dv[b];
          v[b][k] = on ? 0.0f : v[b][k];
        }
      if ((n >> 2) == grp) {
        g.diag_out[row0 + 2 * n] = dv[0];
        g.diag_out[row0 + 2 * n + 1] = dv[1];
      }
    }
    if (direct) {   // row R of the block in LDS row R ^ (R / 16 % 2), its 64-byte halves swapped where R / 8 is odd
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int R = 8 * grp + k;
        *reinterpret_cast<uint32_t*>(T + ((R ^ (grp >> 1)) * 128) + ((J ^ (grp & 1)) * 64) + 4 * n) = pack2<F16>(v[0][k], v[1][k]);
      }
    }
    if (mirror && (KIND != 2 || J == 0)) {
#pragma unroll
      for (int b = 0; b < 2; ++b)
        *reinterpret_cast<uint4*>(T2 + (32 * J + 2 * n + b) * MIRROR_PITCH + 16 * grp) =
            uint4{pack2<F16>(v[b][0], v[b][1]), pack2<F16>(v[b][2], v[b][3]), pack2<F16>(v[b][4], v[b][5]), pack2<F16>(v[b][6], v[b][7])};
    }
  }
  if (direct) {
    const int lr = lane >> 3, ch = lane & 7;
    bf16_t* const dst = g.C + (int64_t)(row0 + lr) * g.c_rs + col0 + 8 * ch;
    uint4 d[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int R = 8 * it + lr;
      d[it] = *reinterpret_cast<const uint4*>(T + ((R ^ (it >> 1)) * 128) + (((ch >> 2) ^ (it & 1)) * 64) + (ch & 3) * 16);
    }
#pragma unroll
    for (int it = 0; it < 4; ++it)
      if (KIND != 1 || ch < 4) *reinterpret_cast<uint4*>(dst + (int64_t)(8 * it) * g.c_rs) = d[it];
  }
  if (mirror) {
    const int lc = lane >> 2, ch = lane & 3;
    bf16_t* const dst = g.C2 + (int64_t)(col0 + lc) * g.c2_rs + row0 + 8 * ch;
    uint4 d[4];
#pragma unroll
    for (int it = 0; it < (KIND == 2 ? 2 : 4); ++it) d[it] = *reinterpret_cast<const uint4*>(T2 + (16 * it + lc) * MIRROR_PITCH + 16 * ch);
#pragma unroll
    for (int it = 0; it < (KIND == 2 ? 2 : 4); ++it) *reinterpret_cast<uint4*>(dst + (int64_t)(16 * it) * g.c2_rs) = d[it];
  }
}

template <bool F16>
__global__ __launch_bounds__(256) void gemm_nt_slim_kernel(GemmArgs gb, int diag_items) {
  __shared__ __align__(1024) unsigned char smem[DEPTH * STAGE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave >> 1, wn = wave & 1;
  // workgroups are dealt round-robin to the 8 XCDs: give each XCD a contiguous run of tiles
  int w = (int)blockIdx.x;
  {
    const int chunk = (int)gridDim.x >> 3;
    if (w < chunk * 8) w = (w & 7) * chunk + (w >> 3);
  }
  int bi, ti, tj, h;
  item_at(gb, diag_items, w, bi, ti, tj, h);
  const GemmArgs g = batch_view(gb, bi);
  const int m0 = ti * 128 + h * TM, n0 = tj * TN;
  const bool use_e = !F16 && g.E != nullptr;   // (fp16 problems carry no operand E)
  if (use_e && !block_written(g, ti * 128, n0)) return;

  Lane L;
  {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int ra = wm * 32 + 16 * i + (lane & 15), rb = wn * 64 + 16 * i + (lane & 15);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        L.fa[kk][i] = (uint32_t)(ra * ROW + (((4 * kk + (lane >> 4)) ^ swz(ra)) << 4));
        L.fb[kk][i] = (uint32_t)(A_BYTES + rb * ROW + (((4 * kk + (lane >> 4)) ^ swz(rb)) << 4));
      }
    }
    L.ldsw = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem + wave * 1024;
#pragma unroll
    for (int q = 0; q < 4; ++q) {   // copy q of a wave fills LDS rows (4 q + wave) 8 .. + 7 of an operand
      const int row = (q * 4 + wave) * 8 + (lane >> 3), chunk = (lane & 7) ^ swz(row);
      if (q < 2) L.voA[q] = (uint32_t)(perm_a(row) * (int)g.lda + chunk * 8) * 2u;
      L.voB[q] = (uint32_t)(perm_b(row) * (int)g.ldb + chunk * 8) * 2u;
    }
  }
  const bf16_t* const gA = g.A + (int64_t)m0 * g.lda;
  const bf16_t* const gB = g.B + (int64_t)n0 * g.ldb;
  const int nk = g.Kc / BK, last = nk - 1;

  if (diag_items && ti == tj) {
    DLane D;
    D.ldsw = L.ldsw;
#pragma unroll
    for (int q = 0; q < 4; ++q) D.vo[q] = L.voB[q];
    const int dr = wave < 2 ? 64 * wave : 32 * wave, dc = wave < 2 ? 64 * wave : 0;   // (waves 2 and 3: rows 64 and 96)
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int rb = dc + 16 * i + (lane & 15);
        D.fb[kk][i] = (uint32_t)(A_BYTES + rb * ROW + (((4 * kk + (lane >> 4)) ^ swz(rb)) << 4));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = gather_row((dr & ~31) + 16 * i + (lane & 15)) & (TN - 1);   // (fragments 2 and 3 of waves 2 and 3 are not read)
        D.fa[kk][i] = (uint32_t)(A_BYTES + r * ROW + (((4 * kk + (lane >> 4)) ^ swz(r)) << 4));
      }
    }
#pragma unroll
    for (int s = 0; s < DEPTH; ++s) {
      const int k = s < last ? s : last;
#pragma unroll
      for (int q = 0; q < 4; ++q) copy16(D.vo[q], gB + k * BK, D.ldsw, s * STAGE + A_BYTES + q * 4096);
    }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"((DEPTH - 1) * 4) : "memory");
    f32x4_t acc[4][4];
    if (wave < 2) diag_loop<F16, 4>(acc, nk, smem, D, gB);
    else diag_loop<F16, 2>(acc, nk, smem, D, gB);
    unsigned char* const T = smem + wave * STAGING;
    Pre pre;
    if (wave < 2) {
      if (use_e) load_e(pre, g, n0 + dr, n0 + dc, lane);
      write_block<F16, 1>(g, use_e, pre, acc[0], acc[1], true, false, true, n0 + dr, n0 + dc, T, lane);
      if (use_e) load_e(pre, g, n0 + dr + 32, n0 + dc, lane);
      write_block<F16, 2>(g, use_e, pre, acc[2], acc[3], true, true, true, n0 + dr + 32, n0 + dc, T, lane);
    } else {
      if (use_e) load_e(pre, g, n0 + dr, n0 + dc, lane);
      write_block<F16>(g, use_e, pre, acc[0], acc[1], true, true, false, n0 + dr, n0 + dc, T, lane);
    }
    return;
  }

  const int row0 = m0 + wm * 32, col0 = n0 + wn * 64;
  Pre pre;   // the operand E first: it is long there when needed
  if (use_e) load_e(pre, g, row0, col0, lane);

  // stages past the end are the last stage again (into slots nobody reads), so that the number of copies in flight is
  // the same at every wait
#pragma unroll
  for (int s = 0; s < DEPTH; ++s) {
    const int k = s < last ? s : last;
#pragma unroll
    for (int q = 0; q < 2; ++q) copy16(L.voA[q], gA + k * BK, L.ldsw, s * STAGE + q * 4096);
#pragma unroll
    for (int q = 0; q < 4; ++q) copy16(L.voB[q], gB + k * BK, L.ldsw, s * STAGE + A_BYTES + q * 4096);
  }
  f32x4_t acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"((DEPTH - 1) * COPIES) : "memory");
  Frag f0, f1;
#pragma unroll
  for (int t = 0; t < 6; ++t) read_frag<0, 0>(f0, smem, L, t);
#define FM_SLIM_STAGE(SLOT, S)                                                    \
  {                                                                               \
    const int kn = (S) + DEPTH < last ? (S) + DEPTH : last;                       \
    stage<F16, SLOT>(acc, f0, f1, smem, L, gA + kn * BK, gB + kn * BK);           \
    if ((S) + 1 >= nk) break;                                                     \
  }
  for (int s = 0;; s += 6) {
    FM_SLIM_STAGE(0, s)
    FM_SLIM_STAGE(1, s + 1)
    FM_SLIM_STAGE(2, s + 2)
    FM_SLIM_STAGE(3, s + 3)
    FM_SLIM_STAGE(4, s + 4)
    FM_SLIM_STAGE(5, s + 5)
  }
#undef FM_SLIM_STAGE
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  const bool tdiag = g.symmetric && ti == tj;   // both halves of such a tile hold their own mirror images
  write_block<F16>(g, use_e, pre, acc[0], acc[1], g.C != nullptr, g.C2 != nullptr && !tdiag, tdiag, row0, col0, smem + wave * STAGING, lane);
}

}  // namespace

bool gemm_slim_fits(const GemmArgs& a, int cus) {
  const long long tm = a.Ma / 128, tn = a.Nb / 128, nb = a.batch < 1 ? 1 : a.batch;
  return (a.symmetric ? tm * tm : 2 * tm * tn) * nb <= cus;
}

int launch_gemm_slim(const GemmArgs& a, hipStream_t stream) {   // tiles_m, tiles_n and num_tiles are those of 128x128 tiles
  // diagonal tiles as one item where they may be and their halves would be too many
  const int diag_items = 2 * a.num_tiles > cu_count();
  const dim3 grid((unsigned)(diag_items ? a.tiles_m * a.tiles_m * a.batch : 2 * a.num_tiles)), block(256);
  if (a.elem == kElemF16) hipLaunchKernelGGL(gemm_nt_slim_kernel<true>, grid, block, 0, stream, a, diag_items);
  else hipLaunchKernelGGL(gemm_nt_slim_kernel<false>, grid, block, 0, stream, a, diag_items);
  return (int)hipGetLastError();
}

}  // namespace fm
