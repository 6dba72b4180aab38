// A 64x64 tile of the NT contraction for products of few tiles, where what counts is how soon a tile is done:
// four waves of 32x32 on 16x16x32 MFMAs, five stages of 64 k (16 KiB) in 80 KiB of LDS, four of them on their
// way, so that a memory round trip is shared by four stages.  A stage moves as many operand bytes as it has
// LDS time for (32 KiB of fragment reads, 16 KiB of copies: 375 cycles) for 128 cycles of MFMA issue, which
// is why larger products run on larger tiles.
#pragma once
#include "fm_tile128.h"

namespace fm {
namespace t64 {

constexpr int EDGE = 64;
constexpr int BK = 64;
constexpr int OPER = 64 * 128;          // one operand of a stage, k-contiguous (64 rows of 64 k) or k-major (64 k of 64 columns)
constexpr int STAGE = 2 * OPER;
constexpr int RING = 5;
constexpr int SMEM = RING * STAGE;      // 81920
static_assert(SMEM == t128::SMEM, "both tile sizes share one LDS layout");

// KMAJOR: both operands as they lie in memory when the contraction runs over rows (see the k-major loop of
// fm_tile128.h); 32-byte chunk c of row k sits at c ^ ((k / 2 % 2) | (k / 8 % 2) 2).  Otherwise rows of 64 k,
// 16-byte chunk c of row r at c ^ swz16(r).
struct Lane {
  uint32_t fa[2], fb[2];   // fragment 0 per k32 substep (k-contiguous), or fragment i (k-major)
  uint32_t ldsw;
};
// [substep][fragment], k-major: in the two halves they are read in
template <bool KMAJOR> struct Frag { bf16x8_t a[2][2], b[2][2]; };
template <> struct Frag<true> { t128::bf16x4_t a[2][2][2], b[2][2][2]; };
__device__ __forceinline__ bf16x8_t whole(bf16x8_t v) { return v; }
__device__ __forceinline__ bf16x8_t whole(const t128::bf16x4_t (&v)[2]) { return t128::join(v[0], v[1]); }

template <bool KMAJOR>
__device__ __forceinline__ Lane lane_setup(unsigned char* smem, int lane, int wave) {
  Lane L;
  const int t = lane & 15, g = lane >> 4, wm = wave >> 1, wn = wave & 1;
  if constexpr (KMAJOR) {
    const int f = ((t >> 3) & 1) | ((g & 1) << 1);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      L.fa[i] = (uint32_t)((8 * g + (t >> 2)) * 128 + (((2 * wm + i) ^ f) << 5) + (t & 3) * 8);
      L.fb[i] = (uint32_t)(OPER + (8 * g + (t >> 2)) * 128 + (((2 * wn + i) ^ f) << 5) + (t & 3) * 8);
    }
  } else {
    const int ra = wm * 32 + t, rb = wn * 32 + t;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      L.fa[kk] = (uint32_t)(ra * 128 + (((4 * kk + g) ^ t128::swz16(ra)) << 4));
      L.fb[kk] = (uint32_t)(OPER + rb * 128 + (((4 * kk + g) ^ t128::swz16(rb)) << 4));
    }
  }
  L.ldsw = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem + wave * 1024;
  return L;
}

// copy q of a wave fills rows (4 q + wave) 8 .. + 7 of an operand's stage
template <bool KMAJOR>
__device__ __forceinline__ void copy_offsets(uint32_t (&vo)[2], int ld, int lane, int wave) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int row = (q * 4 + wave) * 8 + (lane >> 3), p = lane & 7;
    const int chunk = KMAJOR ? ((p >> 1) ^ (((row >> 1) & 1) | (((row >> 3) & 1) << 1))) * 2 + (p & 1) : p ^ t128::swz16(row);
    vo[q] = (uint32_t)(row * ld + chunk * 8) * 2u;
  }
}

// the reads of substep KK of the stage at byte offset `at` of the ring: 8 (k-major: two per fragment) or 4
template <bool KMAJOR, int KK>
__device__ __forceinline__ void read_frag(Frag<KMAJOR>& f, const unsigned char* at, const Lane& L, int t) {   // t of 4: a0 b0 b1 a1
  const int i = t == 0 ? 0 : t == 3 ? 1 : t - 1;
  const bool is_a = t == 0 || t == 3;
  if constexpr (KMAJOR) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned char* p = at + (is_a ? L.fa[i] : L.fb[i]) + KK * 4096 + h * 512;
      if (is_a) f.a[KK][i][h] = t128::read_tr(p);
      else f.b[KK][i][h] = t128::read_tr(p);
    }
  } else {
    const bf16x8_t v = *reinterpret_cast<const bf16x8_t*>(at + (is_a ? L.fa[KK] : L.fb[KK]) + i * 2048);
    if (is_a) f.a[KK][i] = v;
    else f.b[KK][i] = v;
  }
}

// `slot`, `next`: byte offsets of this stage and the next one in the ring
template <bool KMAJOR>
__device__ __forceinline__ void stage(f32x4_t (&acc)[2][2], const Frag<KMAJOR>& cur, Frag<KMAJOR>& nxt, const unsigned char* smem,
                                      const Lane& L, int slot, int next, const uint32_t (&voA)[2], const uint32_t (&voB)[2],
                                      const bf16_t* nA, const bf16_t* nB) {
  // this stage's fragments are here; my copies of the next stage have landed (those of the three after it
  // may be on their way), and behind the barrier everybody's, and this stage's slot is free
  __builtin_amdgcn_s_waitcnt(0x007C);   // vmcnt(12) lgkmcnt(0)
  asm volatile("s_barrier" ::: "memory");
  const uint32_t lds = L.ldsw + slot;
  const unsigned char* const at = smem + next;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    if (q < 2) t128::copy16(voA[q], nA, lds, q * 4096);
    else if (q < 4) t128::copy16(voB[q - 2], nB, lds, OPER + (q - 2) * 4096);
    if (q < 4) read_frag<KMAJOR, 0>(nxt, at, L, q);
    else read_frag<KMAJOR, 1>(nxt, at, L, q - 4);
    const int kk = q >> 2, i = (q >> 1) & 1, j = q & 1;
    acc[i][j] = t128::mfma16<false>(whole(cur.a[kk][i]), whole(cur.b[kk][j]), acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// n k stages (n >= 1) from (gA, gB) on, a stage step_a, step_b elements further on; `count` as in t128::main_loop
template <bool KMAJOR>
__device__ __forceinline__ void main_loop(f32x4_t (&acc)[2][2], int n, const unsigned char* smem, const Lane& L,
                                          const uint32_t (&voA)[2], const uint32_t (&voB)[2], const bf16_t* gA, int step_a,
                                          const bf16_t* gB, int step_b, unsigned* count) {
  const int last = n - 1;
#pragma unroll
  for (int s = 0; s < RING; ++s) {
    const int64_t k = s < last ? s : last;
#pragma unroll
    for (int q = 0; q < 2; ++q) t128::copy16(voA[q], gA + k * step_a, L.ldsw, s * STAGE + q * 4096);
#pragma unroll
    for (int q = 0; q < 2; ++q) t128::copy16(voB[q], gB + k * step_b, L.ldsw, s * STAGE + OPER + q * 4096);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  asm volatile("s_waitcnt vmcnt(16)\n\ts_barrier" ::: "memory");
  if (count) __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  Frag<KMAJOR> f0, f1;
#pragma unroll
  for (int t = 0; t < 4; ++t) read_frag<KMAJOR, 0>(f0, smem, L, t);
#pragma unroll
  for (int t = 0; t < 4; ++t) read_frag<KMAJOR, 1>(f0, smem, L, t);
  const bf16_t* pA = gA + (int64_t)(RING - 1 < last ? RING - 1 : last) * step_a;
  const bf16_t* pB = gB + (int64_t)(RING - 1 < last ? RING - 1 : last) * step_b;
  int slot = 0, next = STAGE;
  auto one = [&](int s, const Frag<KMAJOR>& cur, Frag<KMAJOR>& nxt) {
    const bool more = s + RING <= last;
    pA += more ? step_a : 0;
    pB += more ? step_b : 0;
    stage<KMAJOR>(acc, cur, nxt, smem, L, slot, next, voA, voB, pA, pB);
    slot = next;
    next = next == (RING - 1) * STAGE ? 0 : next + STAGE;
  };
  for (int s = 0;; s += 2) {
    one(s, f0, f1);
    if (s + 1 >= n) break;
    one(s + 1, f1, f0);
    if (s + 2 >= n) break;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// ---- write-out ----------------------------------------------------------------------------------
// The tile's rows r (operand A) and columns c (operand B): v = al[c] E[c][r] + beta acc, or acc.  The block of
// E, loaded before the main loop, goes into LDS by its rows c (128 bytes of r each, 16-byte chunk p at
// p ^ (c / 2 % 8)) and is replaced there by the result, which leaves by rows c (`by_c`); rows r are staged beside
// it, element by element, where they are wanted (`by_r`).  Rows and columns of an output beyond what
// exists of it are not stored.
struct Out {
  bf16_t* C; int64_t ld;        // by_r: C[(r0 + r) ld + c0 + c], by_c: C[(c0 + c) ld + r0 + r]
  bool by_r, by_c, vec;
  int rows_v, cols_v;           // of C
  float beta;
  float* diag_out;              // fp32 diagonal split off (a diagonal tile), or nullptr
};
struct Pre { t128::v4i e[2]; float al[2]; };

// E: rows c0 .. of pitch ld, columns r0 ..
__device__ __forceinline__ void load_block(Pre& pre, const bf16_t* E, int64_t ld, int tid) {
#pragma unroll
  for (int q = 0; q < 2; ++q) pre.e[q] = *reinterpret_cast<const t128::v4i*>(E + (int64_t)(q * 32 + (tid >> 3)) * ld + (tid & 7) * 8);
}

template <int AUX>
__device__ __forceinline__ void store_rows(const Out& o, const unsigned char* S, int row0, int col0, int tid) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int R = q * 32 + (tid >> 3), ch = tid & 7;
    const t128::v4i d = *reinterpret_cast<const t128::v4i*>(S + R * 128 + ((ch ^ ((R >> 1) & 7)) << 4));
    const int row = row0 + R, col = col0 + ch * 8;
    bf16_t* const dst = o.C + row * o.ld + col;
    if (o.vec && row0 + 64 <= o.rows_v && col0 + 64 <= o.cols_v) {
      const __amdgpu_buffer_rsrc_t buf = __builtin_amdgcn_make_buffer_rsrc(o.C + row0 * o.ld + col0, 0, 0xffffffff, 0x00020000);
      __builtin_amdgcn_raw_buffer_store_b128(d, buf, (R * (int)o.ld + ch * 8) * 2, 0, AUX);
    } else if (row < o.rows_v) {
      union { t128::v4i v; unsigned short h[8]; } u;
      u.v = d;
      if (o.vec && col + 8 <= o.cols_v) {
        *reinterpret_cast<t128::v4i*>(dst) = d;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (col + e < o.cols_v) reinterpret_cast<unsigned short*>(dst)[e] = u.h[e];
      }
    }
  }
}

template <bool HAS_E, int AUX>
__device__ __forceinline__ void write_tile(const Out& o, const Pre& pre, const f32x4_t (&acc)[2][2], unsigned char* smem, int r0, int c0,
                                           int lane, int wave) {
  asm volatile("" : "+v"(lane));
  const int n = lane & 15, g = lane >> 4, wm = wave >> 1, wn = wave & 1, tid = wave * 64 + lane;
  unsigned char* const TC = smem;          // by rows c
  unsigned char* const TR = smem + 8192;   // by rows r
  if constexpr (HAS_E) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int c = q * 32 + (tid >> 3);
      *reinterpret_cast<t128::v4i*>(TC + c * 128 + (((tid & 7) ^ ((c >> 1) & 7)) << 4)) = pre.e[q];
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = wn * 32 + 16 * j + n, r = wm * 32 + 16 * i + 4 * g;
      uint2* const at = reinterpret_cast<uint2*>(TC + c * 128 + (((r >> 3) ^ ((c >> 1) & 7)) << 4) + (g & 1) * 8);
      float v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = acc[i][j][k];
      if constexpr (HAS_E) {
        const uint2 e = *at;
        v[0] = __builtin_fmaf(pre.al[j], elem_to_f32<false>((unsigned short)(e.x & 0xffffu)), o.beta * v[0]);
        v[1] = __builtin_fmaf(pre.al[j], elem_to_f32<false>((unsigned short)(e.x >> 16)), o.beta * v[1]);
        v[2] = __builtin_fmaf(pre.al[j], elem_to_f32<false>((unsigned short)(e.y & 0xffffu)), o.beta * v[2]);
        v[3] = __builtin_fmaf(pre.al[j], elem_to_f32<false>((unsigned short)(e.y >> 16)), o.beta * v[3]);
      }
      if (o.diag_out && wm == wn && i == j && (n >> 2) == g) {   // rows r .. + 3 meet column c at k = n % 4
        float dv = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const bool on = k == (n & 3);
          dv = on ? v[k] : dv;
          v[k] = on ? 0.0f : v[k];
        }
        if constexpr (AUX != 0) __hip_atomic_store(o.diag_out + r0 + c, dv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else o.diag_out[r0 + c] = dv;
      }
      if (o.by_c) *at = uint2{t128::pack2<false>(v[0], v[1]), t128::pack2<false>(v[2], v[3])};
      if (o.by_r) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          *reinterpret_cast<unsigned short*>(TR + (r + k) * 128 + (((c >> 3) ^ (((r + k) >> 1) & 7)) << 4) + (c & 7) * 2) = f32_to_elem<false>(v[k]);
      }
    }
  __syncthreads();
  if (o.by_c) store_rows<AUX>(o, TC, c0, r0, tid);
  if (o.by_r) store_rows<AUX>(o, TR, r0, c0, tid);
}

}  // namespace t64
}  // namespace fm
