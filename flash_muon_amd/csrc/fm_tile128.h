// A 128x128 tile of the NT contraction on 16x16x32 MFMAs for workgroups of four waves (64x64 each) that
// share a CU in pairs: 80 KiB of LDS each, so that one workgroup's start, write-out and waits lie under
// the other's multiplications.
//
// Bound by the LDS: a 64-wide k stage of a tile takes 512 cycles of MFMA issue, 64 KiB of fragment reads
// and 32 KiB of incoming copies at 128 bytes per clock, 750 cycles.
#pragma once
#include "fm_internal.h"

namespace fm {
namespace t128 {

constexpr int EDGE = 128;
constexpr int BK = 64;                     // k per stage
constexpr int ROW = BK * 2;                // bytes per LDS row
constexpr int OPER = EDGE * ROW;           // one operand of a stage: 16 KiB
// the ring: three stages of operand A, two of operand B; stage s of A in slot s % 3, of B in slot s % 2
constexpr int B_OFF = 3 * OPER;
constexpr int SMEM = 5 * OPER;             // 81920

// 16-byte chunk c of LDS row r sits at c ^ swz16(r).  LDS row l of a stage holds row perm_a(l) of operand
// A's panel and perm_b(l) of operand B's, so that a lane's sums of a 32x32 sub-block are 8 consecutive
// rows of 2 adjacent columns: register r of tile (2 I + a, 2 J + b) of lane (n = lane % 16, g = lane / 16)
// is row 32 I + 8 g + 4 a + r, column 32 J + 2 n + b of the wave's block.
__device__ __forceinline__ int swz16(int row) { return (row >> 1) & 7; }
__host__ __device__ constexpr int perm_a(int l) { return (l & ~31) + 8 * ((l >> 2) & 3) + 4 * ((l >> 4) & 1) + (l & 3); }
__host__ __device__ constexpr int perm_b(int l) { return (l & ~31) + 2 * (l & 15) + ((l >> 4) & 1); }

template <bool F16>
__device__ __forceinline__ f32x4_t mfma16(bf16x8_t a, bf16x8_t b, f32x4_t c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// One wave-wide global -> LDS copy of 16 bytes per lane to lds + off + 16 lane.  The compiler does not see
// the LDS write: every use is ordered by hand with s_waitcnt vmcnt and a barrier.
__device__ __forceinline__ void copy16(uint32_t voff, const void* sbase, uint32_t lds, int off) {
  asm volatile("s_add_i32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(voff), "s"(sbase), "s"(lds), "n"(off) : "memory", "scc", "m0");
}

struct Frag { bf16x8_t a[4], b[4]; };

// what a lane keeps for a tile: LDS byte addresses of fragment 0 per k32 substep, copy offsets
struct Lane {
  uint32_t fa[2], fb[2];   // operand A in slot 0, operand B in slot 0
  uint32_t ldsw;           // where this wave's copies land inside a slot
};

__device__ __forceinline__ Lane lane_setup(unsigned char* smem, int lane, int wave) {
  Lane L;
  const int ra = (wave >> 1) * 64 + (lane & 15), rb = (wave & 1) * 64 + (lane & 15);
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    L.fa[kk] = (uint32_t)(ra * ROW + (((4 * kk + (lane >> 4)) ^ swz16(ra)) << 4));
    L.fb[kk] = (uint32_t)(B_OFF + rb * ROW + (((4 * kk + (lane >> 4)) ^ swz16(rb)) << 4));
  }
  L.ldsw = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem + wave * 1024;
  return L;
}

// The 16 MFMAs of k32 substep KK of the stage in (AS, BS); the 8 fragment reads of the next substep ride on
// every second of them, and on the others the 4 copies of operand A of the stage two ahead (KK 0, into the
// slot that the stage before has left) or of operand B (KK 1, behind the barrier, into this stage's slot).
template <bool F16, int AS, int BS, int KK>
__device__ __forceinline__ void substep(f32x4_t (&acc)[4][4], const Frag& cur, Frag& nxt, const unsigned char* smem,
                                        const Lane& L, const uint32_t (&vo)[4], const bf16_t* g) {
  constexpr int AFREE = (AS + 2) % 3, AN = KK == 0 ? AS : (AS + 1) % 3, BN = KK == 0 ? BS : BS ^ 1, KN = KK ^ 1;
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    if ((q & 1) == 0) {
      const int t = q >> 1;   // a0 b0 b1 b2 b3 a1 a2 a3
      if (t == 0 || t > 4) {
        const int i = t == 0 ? 0 : t - 4;
        nxt.a[i] = *reinterpret_cast<const bf16x8_t*>(smem + L.fa[KN] + AN * OPER + i * 2048);
      } else {
        nxt.b[t - 1] = *reinterpret_cast<const bf16x8_t*>(smem + L.fb[KN] + BN * OPER + (t - 1) * 2048);
      }
    } else if ((q & 3) == 3) {
      if constexpr (KK == 0) copy16(vo[q >> 2], g, L.ldsw, AFREE * OPER + (q >> 2) * 4096);
      else copy16(vo[q >> 2], g, L.ldsw, B_OFF + BS * OPER + (q >> 2) * 4096);
    }
    acc[q >> 2][q & 3] = mfma16<F16>(cur.a[q >> 2], cur.b[q & 3], acc[q >> 2][q & 3]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <bool F16, int AS, int BS>
__device__ __forceinline__ void stage(f32x4_t (&acc)[4][4], Frag& f0, Frag& f1, const unsigned char* smem, const Lane& L,
                                      const uint32_t (&voA)[4], const uint32_t (&voB)[4], const bf16_t* nA, const bf16_t* nB) {
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the fragments of this substep
  substep<F16, AS, BS, 0>(acc, f0, f1, smem, L, voA, nA);
  // my copies of the next stage have landed (all but the 4 newest, operand A of the stage after), and
  // behind the barrier everybody's; nobody reads this stage's slot of B any more
  __builtin_amdgcn_s_waitcnt(0x0074);   // vmcnt(4) lgkmcnt(0)
  asm volatile("s_barrier" ::: "memory");
  substep<F16, AS, BS, 1>(acc, f1, f0, smem, L, voB, nB);
}

// n k stages (n >= 1).  `first` issues the 8 copies of stage 0 and `landed` is called when this wave's have landed, in
// front of the barrier that says so for everybody; stage s >= 1 is at (gA, gB) + s BK, as stage 0 is if `lo` is 0.
// voA, voB: byte offsets of this lane's four copies per operand.  `count`, where a thread has one, is counted up once
// the first stage has landed everywhere: by then the stores that every wave issued before this call have completed
// too (one counter tracks both, in order).  On return no copy is in flight and nobody reads the ring.
template <bool F16, class First, class Landed>
__device__ __forceinline__ void main_loop_from(f32x4_t (&acc)[4][4], int n, const unsigned char* smem, const Lane& L,
                                               const uint32_t (&voA)[4], const uint32_t (&voB)[4], const bf16_t* gA, const bf16_t* gB,
                                               unsigned* count, int lo, const First& first, const Landed& landed) {
  // stages past the end are the last stage again, or stage `lo` (into slots nobody reads), so that the number of
  // copies in flight is the same at every wait
  const int last = n - 1, fill = last < lo ? lo : last, k1 = last < 1 ? fill : 1;
  first();
#pragma unroll
  for (int q = 0; q < 4; ++q) copy16(voA[q], gA + k1 * BK, L.ldsw, OPER + q * 4096);
#pragma unroll
  for (int q = 0; q < 4; ++q) copy16(voB[q], gB + k1 * BK, L.ldsw, B_OFF + OPER + q * 4096);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  landed();
  asm volatile("s_barrier" ::: "memory");
  if (count) __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  Frag f0, f1;
#pragma unroll
  for (int i = 0; i < 4; ++i) f0.a[i] = *reinterpret_cast<const bf16x8_t*>(smem + L.fa[0] + i * 2048);
#pragma unroll
  for (int i = 0; i < 4; ++i) f0.b[i] = *reinterpret_cast<const bf16x8_t*>(smem + L.fb[0] + i * 2048);
#define FM_T128_STAGE(AS, BS, S)                                                                  \
  {                                                                                               \
    const int kn = (S) + 2 < last ? (S) + 2 : fill;                                               \
    stage<F16, AS, BS>(acc, f0, f1, smem, L, voA, voB, gA + kn * BK, gB + kn * BK);               \
    if ((S) + 1 >= n) break;                                                                      \
  }
  for (int s = 0;; s += 6) {   // the slots come round every 6 stages
    FM_T128_STAGE(0, 0, s)
    FM_T128_STAGE(1, 1, s + 1)
    FM_T128_STAGE(2, 0, s + 2)
    FM_T128_STAGE(0, 1, s + 3)
    FM_T128_STAGE(1, 0, s + 4)
    FM_T128_STAGE(2, 1, s + 5)
  }
#undef FM_T128_STAGE
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// ... all of them from (gA, gB) on
template <bool F16>
__device__ __forceinline__ void main_loop(f32x4_t (&acc)[4][4], int n, const unsigned char* smem, const Lane& L,
                                          const uint32_t (&voA)[4], const uint32_t (&voB)[4], const bf16_t* gA, const bf16_t* gB,
                                          unsigned* count) {
  main_loop_from<F16>(acc, n, smem, L, voA, voB, gA, gB, count, 0, [&]() {
#pragma unroll
    for (int q = 0; q < 4; ++q) copy16(voA[q], gA, L.ldsw, q * 4096);
#pragma unroll
    for (int q = 0; q < 4; ++q) copy16(voB[q], gB, L.ldsw, B_OFF + q * 4096);
  }, []() {});
}

// ---- the same with both operands k-major --------------------------------------------------------
// A stage is 32 rows (k) of 128 columns of each operand, 256 bytes a row, as a symmetric matrix and the X of
// X' = P X lie in memory: no transposed copy of X is needed.  Fragments come out of the transposing LDS
// read (16 lanes read 4 k of 16 columns and get one column's 4 k each); 32-byte chunk c of row k sits at
// c ^ ((k & 3) | (k / 8 % 2) 4), which puts the 8 rows that half a wave reads on different banks.  Fragment i
// is columns 16 i .. + 15 of the wave's 64: register r of tile (i, j) of lane (n, g) is row 16 i + 4 g + r,
// column 16 j + n of the block.  Stages half as long and freed whole let five of them fill the same LDS with
// four on their way.
constexpr int KK_BK = 32, KK_OPER = KK_BK * 256, KK_STAGE = 2 * KK_OPER, KK_RING = 5;

struct LaneT {
  uint32_t fa[4], fb[4];   // fragment i, first half of its 8 k, slot 0
  uint32_t ldsw;
};

__device__ __forceinline__ LaneT lane_setup_t(unsigned char* smem, int lane, int wave) {
  LaneT L;
  const int t = lane & 15, g = lane >> 4, f = (t >> 2) | ((g & 1) << 2);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    L.fa[i] = (uint32_t)((8 * g + (t >> 2)) * 256 + (((4 * (wave >> 1) + i) ^ f) << 5) + (t & 3) * 8);
    L.fb[i] = (uint32_t)(KK_OPER + (8 * g + (t >> 2)) * 256 + (((4 * (wave & 1) + i) ^ f) << 5) + (t & 3) * 8);
  }
  L.ldsw = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem + wave * 1024;
  return L;
}

typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4_t;
__device__ __forceinline__ bf16x4_t read_tr(const unsigned char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4_t*)p);
}
__device__ __forceinline__ bf16x8_t join(bf16x4_t lo, bf16x4_t hi) { return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7); }

struct FragT { bf16x4_t a[4][2], b[4][2]; };

template <int SLOT>
__device__ __forceinline__ void read_t(FragT& f, const unsigned char* smem, const LaneT& L, int t) {   // read t of 16: a0 a0 b0 b0 .. b3 b3 a1 a1 ..
  const int h = t & 1, x = t >> 1;
  if (x >= 1 && x < 5) f.b[x - 1][h] = read_tr(smem + L.fb[x - 1] + SLOT * KK_STAGE + h * 1024);
  else f.a[x == 0 ? 0 : x - 4][h] = read_tr(smem + L.fa[x == 0 ? 0 : x - 4] + SLOT * KK_STAGE + h * 1024);
}

// stage in SLOT: `cur` holds its fragments; those of the next stage are read, and behind the barrier, which
// says that everybody has this stage's, the copies of the stage five ahead go into its slot
template <int SLOT>
__device__ __forceinline__ void stage_t(f32x4_t (&acc)[4][4], const FragT& cur, FragT& nxt, const unsigned char* smem, const LaneT& L,
                                        const uint32_t (&voA)[2], const uint32_t (&voB)[2], const bf16_t* nA, const bf16_t* nB) {
  // my copies of the next stage have landed (those of the three after it may be on their way)
  __builtin_amdgcn_s_waitcnt(0x007C);   // vmcnt(12) lgkmcnt(0)
  asm volatile("s_barrier" ::: "memory");
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    read_t<(SLOT + 1) % KK_RING>(nxt, smem, L, q);
    if ((q & 3) == 3) {
      if (q < 8) copy16(voA[q >> 2], nA, L.ldsw, SLOT * KK_STAGE + (q >> 2) * 4096);
      else copy16(voB[(q >> 2) - 2], nB, L.ldsw, SLOT * KK_STAGE + KK_OPER + ((q >> 2) - 2) * 4096);
    }
    acc[q >> 2][q & 3] = mfma16<false>(join(cur.a[q >> 2][0], cur.a[q >> 2][1]), join(cur.b[q & 3][0], cur.b[q & 3][1]), acc[q >> 2][q & 3]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// n stages (n >= 1) of 32 rows from (gA, gB) on; a stage of an operand is step_a, step_b elements further on
__device__ __forceinline__ void main_loop_t(f32x4_t (&acc)[4][4], int n, const unsigned char* smem, const LaneT& L,
                                            const uint32_t (&voA)[2], const uint32_t (&voB)[2], const bf16_t* gA, int step_a,
                                            const bf16_t* gB, int step_b, unsigned* count) {
  // stages past the end are the last stage again (into slots nobody reads)
  const int last = n - 1;
#pragma unroll
  for (int s = 0; s < KK_RING; ++s) {
    const int k = s < last ? s : last;
#pragma unroll
    for (int q = 0; q < 2; ++q) copy16(voA[q], gA + k * step_a, L.ldsw, s * KK_STAGE + q * 4096);
#pragma unroll
    for (int q = 0; q < 2; ++q) copy16(voB[q], gB + k * step_b, L.ldsw, s * KK_STAGE + KK_OPER + q * 4096);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  asm volatile("s_waitcnt vmcnt(16)\n\ts_barrier" ::: "memory");
  if (count) __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  FragT f0, f1;
#pragma unroll
  for (int t = 0; t < 16; ++t) read_t<0>(f0, smem, L, t);
  // (running pointers, so that a stage's addresses are two scalar additions)
  const bf16_t* pA = gA + (KK_RING - 1 < last ? KK_RING - 1 : last) * step_a;
  const bf16_t* pB = gB + (KK_RING - 1 < last ? KK_RING - 1 : last) * step_b;
#define FM_KK_STAGE(SLOT, S, CUR, NXT)                                                            \
  {                                                                                               \
    const bool more = (S) + KK_RING <= last;                                                      \
    pA += more ? step_a : 0;                                                                      \
    pB += more ? step_b : 0;                                                                      \
    stage_t<SLOT>(acc, CUR, NXT, smem, L, voA, voB, pA, pB);                                      \
    if ((S) + 1 >= n) break;                                                                      \
  }
  for (int s = 0;; s += 10) {   // slots and fragment sets come round every 10 stages
    FM_KK_STAGE(0, s, f0, f1)
    FM_KK_STAGE(1, s + 1, f1, f0)
    FM_KK_STAGE(2, s + 2, f0, f1)
    FM_KK_STAGE(3, s + 3, f1, f0)
    FM_KK_STAGE(4, s + 4, f0, f1)
    FM_KK_STAGE(0, s + 5, f1, f0)
    FM_KK_STAGE(1, s + 6, f0, f1)
    FM_KK_STAGE(2, s + 7, f1, f0)
    FM_KK_STAGE(3, s + 8, f0, f1)
    FM_KK_STAGE(4, s + 9, f1, f0)
  }
#undef FM_KK_STAGE
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// copy q of a wave fills rows (4 q + wave) 4 .. + 3 of an operand's stage
__device__ __forceinline__ void copy_offsets_t(uint32_t (&vo)[2], int ld, int lane, int wave) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int k = (q * 4 + wave) * 4 + (lane >> 4), f = (k & 3) | (((k >> 3) & 1) << 2);
    vo[q] = (uint32_t)(k * ld + ((((lane & 15) >> 1) ^ f) * 2 + (lane & 1)) * 8) * 2u;
  }
}

// byte offsets of a lane's copies: copy q of a wave fills LDS rows (4 q + wave) 8 .. + 7 of an operand
__device__ __forceinline__ void copy_offsets(uint32_t (&voA)[4], uint32_t (&voB)[4], int lda, int ldb, int lane, int wave) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int row = (q * 4 + wave) * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ swz16(row);
    voA[q] = (uint32_t)(perm_a(row) * lda + chunk * 8) * 2u;
    voB[q] = (uint32_t)(perm_b(row) * ldb + chunk * 8) * 2u;
  }
}

// ---- write-out ----------------------------------------------------------------------------------
// A wave's 64x64 block at (row0, col0): v = (alpha + row_alpha[i]) E + beta acc (or acc), rounded once;
// the direct copy to C by rows and the mirrored or transposed one to C2 by columns, both through 8 KiB of
// wave-private LDS each and out as whole 128-byte lines, 8 lanes a line.  E is read transposed (ET), 8
// consecutive rows of a column per 16-byte load, which is what a lane holds of that column.
struct Out {
  const bf16_t* ET; int ldet;     // nullptr: no operand E
  bf16_t* C; int64_t c_rs;        // nullptr: no such output
  bf16_t* C2; int64_t c2_rs;
  float alpha, beta;
  const float* row_alpha;
  float* diag_out;                // fp32 diagonal split off (blocks on the diagonal of a symmetric product)
  int limit;                      // EDGE: rows and columns of the output that exist
};

typedef int v4i __attribute__((ext_vector_type(4)));

template <bool F16>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  const f2 v = {lo, hi};
  if constexpr (F16) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, h2));
  } else {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, b2));
  }
}

// One lane's 16 bytes of a row of a square output of `limit` rows: columns c .. c + 7 of row r, at any alignment of the
// element type
__device__ __forceinline__ void store_edge(bf16_t* C, int64_t ld, int r, int c, int limit, uint4 d) {
  if (r >= limit) return;
  bf16_t* const dst = C + r * ld + c;
  if (c + 8 <= limit) {
    __builtin_memcpy(dst, &d, 16);
  } else {
    union { uint4 v; unsigned short h[8]; } u;
    u.v = d;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (c + e < limit) reinterpret_cast<unsigned short*>(dst)[e] = u.h[e];
  }
}

// AUX: cache policy of the stores (0, or 16: written through to memory, for readers on other XCDs).  EDGE: blocks may
// reach beyond the output, whose rows may start at any element.
template <bool F16, int AUX, bool EDGE = false>
__device__ __forceinline__ void write_block(const Out& o, bool diag, const f32x4_t (&acc)[4][4], unsigned char* T, int row0,
                                            int col0, int lane) {
  asm volatile("" : "+v"(lane));   // offsets derived anew for every tile, not kept across the main loop
  const int n = lane & 15, g = lane >> 4;
  const bool use_e = !F16 && o.ET != nullptr, direct = o.C != nullptr, mirror = o.C2 != nullptr && !diag;
  const bool dout = diag && row0 == col0 && o.diag_out != nullptr;
  unsigned char* const T2 = T + 8192;
  uint4 ev[2][2][2];
  float al[2][8];
  if (use_e) {
    const bf16_t* e = o.ET + (int64_t)(col0 + 2 * n) * o.ldet + row0 + 8 * g;
#pragma unroll
    for (int I = 0; I < 2; ++I)
#pragma unroll
      for (int J = 0; J < 2; ++J)
#pragma unroll
        for (int b = 0; b < 2; ++b) ev[I][J][b] = *reinterpret_cast<const uint4*>(e + (32 * J + b) * o.ldet + 32 * I);
#pragma unroll
    for (int I = 0; I < 2; ++I)
#pragma unroll
      for (int k = 0; k < 8; k += 4) {
        f32x4_t ra = {0.0f, 0.0f, 0.0f, 0.0f};
        if (o.row_alpha) ra = *reinterpret_cast<const f32x4_t*>(o.row_alpha + row0 + 32 * I + 8 * g + k);
#pragma unroll
        for (int r = 0; r < 4; ++r) al[I][k + r] = o.alpha + ra[r];
      }
  }
#pragma unroll
  for (int I = 0; I < 2; ++I)
#pragma unroll
    for (int J = 0; J < 2; ++J) {
      float v[2][8];   // [b][8 rows]
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int k = 0; k < 8; ++k) v[b][k] = acc[2 * I + (k >> 2)][2 * J + b][k & 3];
      if (use_e) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const uint32_t w[4] = {ev[I][J][b].x, ev[I][J][b].y, ev[I][J][b].z, ev[I][J][b].w};
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const float e = elem_to_f32<F16>((unsigned short)((k & 1) ? (w[k >> 1] >> 16) : (w[k >> 1] & 0xffffu)));
            v[b][k] = __builtin_fmaf(al[I][k], e, o.beta * v[b][k]);
          }
        }
      }
      if (dout && I == J) {   // the lanes with n / 4 == g hold rows 2 n and 2 n + 1 of the sub-block's diagonal
        float dv[2] = {0.0f, 0.0f};
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const bool on = 2 * n + b == 8 * g + k;
            dv[b] = on ? v[b][k] : dv[b];
            v[b][k] = on ? 0.0f : v[b][k];
          }
        if ((n >> 2) == g) {
          float* d = o.diag_out + row0 + 32 * I + 2 * n;
          if constexpr (AUX != 0) {
            __hip_atomic_store(d, dv[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(d + 1, dv[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          } else {
            d[0] = dv[0];
            d[1] = dv[1];
          }
        }
      }
      if (direct) {
        // row R of the block in LDS row R ^ (R / 16 % 2), its 64-byte halves swapped where R / 8 is odd: the four
        // row groups of a wave's store then cover all 64 banks
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int R = 32 * I + 8 * g + k;
          *reinterpret_cast<uint32_t*>(T + ((R ^ (g >> 1)) * 128) + ((J ^ (g & 1)) * 64) + 4 * n) = pack2<F16>(v[0][k], v[1][k]);
        }
      }
      if (mirror) {
        // column c in LDS row c ^ (c / 16 % 2), its 16-byte chunk p at p ^ (c / 2 % 8)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const int c = 32 * J + 2 * n + b;
          *reinterpret_cast<uint4*>(T2 + ((c ^ (n >> 3)) * 128) + (((4 * I + g) ^ (n & 7)) << 4)) =
              uint4{pack2<F16>(v[b][0], v[b][1]), pack2<F16>(v[b][2], v[b][3]), pack2<F16>(v[b][4], v[b][5]), pack2<F16>(v[b][6], v[b][7])};
        }
      }
    }
  const int lr = lane >> 3, ch = lane & 7;
  if (direct) {
    const __amdgpu_buffer_rsrc_t buf = __builtin_amdgcn_make_buffer_rsrc(o.C + (int64_t)row0 * o.c_rs + col0, 0, 0xffffffff, 0x00020000);
    const uint32_t vo = (uint32_t)(lr * (int)o.c_rs + ch * 8) * 2u;
    uint4 d[8];
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int R = 8 * it + lr, gg = it & 3;   // R / 8 % 4
      d[it] = *reinterpret_cast<const uint4*>(T + ((R ^ (gg >> 1)) * 128) + (((ch >> 2) ^ (gg & 1)) * 64) + (ch & 3) * 16);
    }
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      if constexpr (EDGE) store_edge(o.C, o.c_rs, row0 + 8 * it + lr, col0 + 8 * ch, o.limit, d[it]);
      else __builtin_amdgcn_raw_buffer_store_b128(v4i{(int)d[it].x, (int)d[it].y, (int)d[it].z, (int)d[it].w}, buf, (int)vo, it * 16 * (int)o.c_rs, AUX);
    }
  }
  if (mirror) {
    const __amdgpu_buffer_rsrc_t buf = __builtin_amdgcn_make_buffer_rsrc(o.C2 + (int64_t)col0 * o.c2_rs + row0, 0, 0xffffffff, 0x00020000);
    const uint32_t vo = (uint32_t)(lr * (int)o.c2_rs + ch * 8) * 2u;
    uint4 d[8];
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int c = 8 * it + lr;
      d[it] = *reinterpret_cast<const uint4*>(T2 + ((c ^ ((c >> 4) & 1)) * 128) + ((ch ^ ((c >> 1) & 7)) << 4));
    }
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      if constexpr (EDGE) store_edge(o.C2, o.c2_rs, col0 + 8 * it + lr, row0 + 8 * ch, o.limit, d[it]);
      else __builtin_amdgcn_raw_buffer_store_b128(v4i{(int)d[it].x, (int)d[it].y, (int)d[it].z, (int)d[it].w}, buf, (int)vo, it * 16 * (int)o.c2_rs, AUX);
    }
  }
}

// Write-out behind main_loop_t: acc is rows j (columns of X) by columns i (rows of X) of a wave's 64x64 block
// at (j0, i0): X'[i][j] = (alpha + row_alpha[i]) X[i][j] + acc.  The block of X, loaded before the main loop,
// goes into 8 KiB of wave-private LDS (row i: 128 bytes, 16-byte chunk p at p ^ (i / 2 % 8)) and is replaced
// there by the result, which leaves by rows of X' (tall false), or is staged by rows of X'^T beside it.
// Rows and columns of the output beyond rows_v and cols_v do not exist; `vec`: 16-byte stores are allowed.
struct OutT {
  bf16_t* C; int64_t c_rs;
  float alpha;
  int rows_v, cols_v;
  bool tall, vec;
};
struct PreT { v4i e[8]; float ra[4]; };

__device__ __forceinline__ void load_block_t(PreT& pre, const bf16_t* X, int ldx, const float* row_alpha, int j0, int i0, int lane) {
  const bf16_t* const src = X + (int64_t)(i0 + (lane >> 3)) * ldx + j0 + (lane & 7) * 8;
#pragma unroll
  for (int it = 0; it < 8; ++it) pre.e[it] = *reinterpret_cast<const v4i*>(src + (int64_t)(8 * it) * ldx);
#pragma unroll
  for (int j = 0; j < 4; ++j) pre.ra[j] = row_alpha[i0 + 16 * j + (lane & 15)];
}

template <int AUX>
__device__ __forceinline__ void write_block_t(const OutT& o, const PreT& pre, const f32x4_t (&acc)[4][4], unsigned char* T, int j0,
                                              int i0, int lane) {
  asm volatile("" : "+v"(lane));
  const int n = lane & 15, g = lane >> 4, lr = lane >> 3, ch = lane & 7;
  unsigned char* const T2 = T + 8192;
#pragma unroll
  for (int it = 0; it < 8; ++it) {
    const int R = 8 * it + lr;
    *reinterpret_cast<v4i*>(T + R * 128 + ((ch ^ ((R >> 1) & 7)) << 4)) = pre.e[it];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float al = o.alpha + pre.ra[j];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      uint2* const at = reinterpret_cast<uint2*>(T + (16 * j + n) * 128 + (((2 * a + (g >> 1)) ^ ((n >> 1) & 7)) << 4) + (g & 1) * 8);
      const uint2 e = *at;
      float v[4];
      v[0] = __builtin_fmaf(al, elem_to_f32<false>((unsigned short)(e.x & 0xffffu)), acc[a][j][0]);
      v[1] = __builtin_fmaf(al, elem_to_f32<false>((unsigned short)(e.x >> 16)), acc[a][j][1]);
      v[2] = __builtin_fmaf(al, elem_to_f32<false>((unsigned short)(e.y & 0xffffu)), acc[a][j][2]);
      v[3] = __builtin_fmaf(al, elem_to_f32<false>((unsigned short)(e.y >> 16)), acc[a][j][3]);
      if (!o.tall) {
        *at = uint2{pack2<false>(v[0], v[1]), pack2<false>(v[2], v[3])};
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {   // row R: 128 bytes, 16-byte chunk p at p ^ (R / 2 % 8)
          const int R = 16 * a + 4 * g + r;
          *reinterpret_cast<unsigned short*>(T2 + R * 128 + (((2 * j + (n >> 3)) ^ ((R >> 1) & 7)) << 4) + (n & 7) * 2) = f32_to_elem<false>(v[r]);
        }
      }
    }
  }
  const int r0 = o.tall ? j0 : i0, c0 = o.tall ? i0 : j0;
  const unsigned char* const S = o.tall ? T2 : T;
  uint4 d[8];
#pragma unroll
  for (int it = 0; it < 8; ++it) {
    const int R = 8 * it + lr;
    d[it] = *reinterpret_cast<const uint4*>(S + R * 128 + ((ch ^ ((R >> 1) & 7)) << 4));
  }
  if (o.vec && r0 + 64 <= o.rows_v && c0 + 64 <= o.cols_v) {
    const __amdgpu_buffer_rsrc_t buf = __builtin_amdgcn_make_buffer_rsrc(o.C + r0 * o.c_rs + c0, 0, 0xffffffff, 0x00020000);
    const uint32_t vo = (uint32_t)(lr * (int)o.c_rs + ch * 8) * 2u;
#pragma unroll
    for (int it = 0; it < 8; ++it)
      __builtin_amdgcn_raw_buffer_store_b128(v4i{(int)d[it].x, (int)d[it].y, (int)d[it].z, (int)d[it].w}, buf, (int)vo, it * 16 * (int)o.c_rs, AUX);
  } else {
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int R = r0 + 8 * it + lr, c = c0 + ch * 8;
      if (R >= o.rows_v) continue;
      unsigned short* const dst = reinterpret_cast<unsigned short*>(o.C) + R * o.c_rs + c;
      union { uint4 v; unsigned short h[8]; } u;
      u.v = d[it];
      if (o.vec && c + 8 <= o.cols_v) {
        *reinterpret_cast<uint4*>(dst) = u.v;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (c + e < o.cols_v) dst[e] = u.h[e];
      }
    }
  }
}

}  // namespace t128
}  // namespace fm
