// Y = X * X^T in fp32 for gfx950, on the fp32 matrix instruction (32x32x2: fp32 products, fp32 sums).
//
// Bound by the matrix units: 256 flop per clock and CU, a sixteenth of the bf16 rate, so that a 64x64
// tile already needs 16 bytes of operands per clock and CU (the L2s deliver 64) and 32 KiB of LDS reads
// per 1024 cycles.  What the time depends on is that every CU has the same number of k stages to do.
// So: 64x64 tiles (four waves of 32x32), two workgroups per CU that fill each other's waits, whole
// tiles in rounds of 512, and the tiles that are left over shared out as one run of k stages, an equal
// piece per workgroup; their sums go to memory as fp32 parts and a second kernel adds them in k order,
// so the bits do not depend on timing.
//
// Measured (N(0,1) input): 4096 x 4096 568 us, 123 TFLOP/s executed, the matrix units busy for 82 % of the
// cycles (77 % with the fragments of a stage read behind its barrier: 602 us; no change with three
// workgroups per CU, two chains of sums, four stages in the ring, or all operands out of one L2 panel);
// 2048 x 4096 157 us (whole 128x128 tiles, 136 of them on 256 CUs: 309), 1024 x 4096 55 us.
#include "fm_internal.h"

namespace fm {

namespace {

constexpr int T32 = 64;                         // tile edge
constexpr int BK32 = 32;                        // k per stage: 128-byte LDS rows
constexpr int OPER32 = T32 * 128;               // one operand of a stage: 8 KiB
constexpr int STAGE32 = 2 * OPER32;
constexpr int RING32 = 3;                       // stages: one multiplied, one landing, one on its way
constexpr int kF32Grid = 512;                   // workgroups: two per CU
constexpr int kPartFloats32 = T32 * T32;
constexpr int kMinPiece = 8;                    // stages a piece of a left-over tile has at least

struct F32Args {
  const float* X; int64_t ldx;
  float* Y; int64_t rs, cs;
  int M, K;
  int T, nk;            // tile rows, k stages per tile
  int rounds, rem;      // full rounds of gridDim.x tiles, tiles left over
  int piece;            // stages per workgroup of the left-over tiles' run, 0: whole tiles, one per workgroup
  float* parts;         // two slots per workgroup: a piece lies in at most two tiles
};

// sixteen bytes of zeros for the lanes of a copy that lie beyond the end of a row
__device__ const float fm_zeros_f32[4] = {0.0f, 0.0f, 0.0f, 0.0f};

// One wave-wide global -> LDS copy, VEC floats per lane: lane l lands at lds + 4 VEC l.  The compiler
// does not see the LDS write; every use is ordered by hand with s_waitcnt vmcnt and a barrier.
template <int VEC>
__device__ __forceinline__ void copy_f32(const float* src, uint32_t lds) {
  if constexpr (VEC == 4)
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(src), "s"(lds) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" :: "v"(src), "s"(lds) : "memory", "m0");
}

// One wave's 32x32 block at (row0, col0) of Y and its mirror image, from the accumulators: register
// 4 q + e of lane l is row 8 q + 4 (l / 32) + e, column l % 32.  Both copies come from the same register;
// on a diagonal tile only what lies on or above the diagonal counts.
__device__ __forceinline__ void f32_write_block(const F32Args& p, const f32x16_t& acc, bool diag, int row0, int col0, int lane) {
  const int col = col0 + (lane & 31), rbase = row0 + 4 * (lane >> 5);
  if (col >= p.M) return;
  const bool vec = !diag && p.cs == 1 && p.rs % 4 == 0 && (reinterpret_cast<uintptr_t>(p.Y) & 15) == 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int row = rbase + 8 * q;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (row + e < p.M && (!diag || col >= row + e)) p.Y[(int64_t)(row + e) * p.rs + (int64_t)col * p.cs] = acc[4 * q + e];
    if (vec && row + 4 <= p.M) {
      *reinterpret_cast<f32x4_t*>(p.Y + (int64_t)col * p.rs + row) = f32x4_t{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (row + e < p.M && (!diag || col > row + e)) p.Y[(int64_t)col * p.rs + (int64_t)(row + e) * p.cs] = acc[4 * q + e];
    }
  }
}

// VEC: floats per lane and copy: 4 where every row of X and K allow 16-byte accesses, else 1
template <int VEC>
__global__ __launch_bounds__(256) void syrk_f32_kernel(F32Args p) {
  __shared__ __align__(1024) unsigned char smem[RING32 * STAGE32];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int G = (int)gridDim.x;
  // of the two workgroups of a CU (ids 256 apart) one goes first: equal, they wait for their data together
  if (blockIdx.x & 256) __builtin_amdgcn_s_setprio(1);
  // workgroups are dealt round-robin to the 8 XCDs: give each XCD a contiguous run of positions
  int w = (int)blockIdx.x;
  {
    const int chunk = G >> 3;
    if (w < chunk * 8) w = (w & 7) * chunk + (w >> 3);
  }
  constexpr int N = 2 * (VEC == 4 ? 1 : 4);           // copies per wave, operand and stage
  constexpr int ROWS = VEC == 4 ? 8 : 2;              // LDS rows one copy fills
  // copy q of this wave fills rows 16 wave + ROWS q .. of an operand; 16-byte chunk c of row r sits at c ^ swz(r)
  int lrow[N], kofs[N];
#pragma unroll
  for (int q = 0; q < N; ++q) {
    lrow[q] = 16 * wave + ROWS * q + (VEC == 4 ? lane >> 3 : lane >> 5);
    const int pos = VEC == 4 ? lane & 7 : (lane >> 2) & 7;
    kofs[q] = ((pos ^ swz(lrow[q])) << 2) + (VEC == 4 ? 0 : lane & 3);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem;
  const uint32_t ldsw = lds0 + wave * 2048;
  const int ra = wm * 32 + (lane & 31), rb = wn * 32 + (lane & 31);
  const uint32_t ao = (uint32_t)(ra * 128 + (((lane >> 5) ^ swz(ra)) << 4));
  const uint32_t bo = (uint32_t)(OPER32 + rb * 128 + (((lane >> 5) ^ swz(rb)) << 4));

  // k stages [kb, ke) of tile (ti, tj) into acc
  auto run = [&](int ti, int tj, int kb, int ke, f32x16_t& acc) {
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    if (kb >= ke) return;
    const float* pa[N];
    const float* pb[N];
#pragma unroll
    for (int q = 0; q < N; ++q) {   // rows past the end repeat the last row; what they give is never stored
      int a = ti * T32 + lrow[q], b = tj * T32 + lrow[q];
      a = a < p.M ? a : p.M - 1;
      b = b < p.M ? b : p.M - 1;
      pa[q] = p.X + (int64_t)a * p.ldx + kofs[q];
      pb[q] = p.X + (int64_t)b * p.ldx + kofs[q];
    }
    auto issue = [&](int stage, int slot) {
      const uint32_t base = ldsw + slot * STAGE32;
      const int k0 = stage * BK32;
      if (k0 + BK32 <= p.K) {
#pragma unroll
        for (int q = 0; q < N; ++q) copy_f32<VEC>(pa[q] + k0, base + q * (ROWS * 128));
#pragma unroll
        for (int q = 0; q < N; ++q) copy_f32<VEC>(pb[q] + k0, base + OPER32 + q * (ROWS * 128));
      } else {   // the last stage of a K that is no multiple of 32: zeros beyond the end of the rows
#pragma unroll
        for (int q = 0; q < N; ++q) copy_f32<VEC>(k0 + kofs[q] < p.K ? pa[q] + k0 : fm_zeros_f32, base + q * (ROWS * 128));
#pragma unroll
        for (int q = 0; q < N; ++q) copy_f32<VEC>(k0 + kofs[q] < p.K ? pb[q] + k0 : fm_zeros_f32, base + OPER32 + q * (ROWS * 128));
      }
    };
    // stages past the end are the last stage again (into slots nobody reads), so that the number of
    // copies in flight is the same at every wait
    issue(kb, 0);
    issue(kb + 1 < ke ? kb + 1 : ke - 1, 1);
    // The fragments of a stage are read while the second half of the stage before is multiplied, behind a
    // barrier in its middle.
    int nxt = 2, rd = 1;
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(2 * N) : "memory");
    __syncthreads();
    f32x4_t f[2][2][4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      f[0][0][ks] = *reinterpret_cast<const f32x4_t*>(smem + (ao ^ (ks << 5)));
      f[0][1][ks] = *reinterpret_cast<const f32x4_t*>(smem + (bo ^ (ks << 5)));
    }
    auto stage = [&](int s, f32x4_t (&cur)[2][4], f32x4_t (&nx)[2][4]) {
      issue(s + 2 < ke ? s + 2 : ke - 1, nxt);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(cur[0][e >> 2][e & 3], cur[1][e >> 2][e & 3], acc, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt vmcnt(%0)" :: "n"(2 * N) : "memory");   // stage s + 1 has landed
      __builtin_amdgcn_s_waitcnt(0xC07F);
      asm volatile("s_barrier" ::: "memory");
      const unsigned char* st = smem + rd * STAGE32;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        nx[0][ks] = *reinterpret_cast<const f32x4_t*>(st + (ao ^ (ks << 5)));
        nx[1][ks] = *reinterpret_cast<const f32x4_t*>(st + (bo ^ (ks << 5)));
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 8; e < 16; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(cur[0][e >> 2][e & 3], cur[1][e >> 2][e & 3], acc, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      nxt = nxt == 2 ? 0 : nxt + 1;
      rd = rd == 2 ? 0 : rd + 1;
    };
    int s = kb;
    for (; s + 2 <= ke; s += 2) {
      stage(s, f[0], f[1]);
      stage(s + 1, f[1], f[0]);
    }
    if (s < ke) stage(s, f[0], f[1]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();   // no copy in flight and no wave still reading: the ring is free
  };

  f32x16_t acc;
  int ti, tj;
  for (int r = 0; r < p.rounds + (p.piece == 0 ? 1 : 0); ++r) {
    if (r == p.rounds && w >= p.rem) break;
    band_tri_decode(r * G + w, p.T, ti, tj);
    run(ti, tj, 0, p.nk, acc);
    f32_write_block(p, acc, ti == tj, ti * T32 + wm * 32, tj * T32 + wn * 32, lane);
  }
  if (p.piece == 0) return;
  int s = w * p.piece;
  const int end = s + p.piece < p.rem * p.nk ? s + p.piece : p.rem * p.nk;
  for (int slot = 0; s < end; ++slot) {   // at most two tiles: piece <= nk
    const int t = s / p.nk, kb = s - t * p.nk;
    const int ke = kb + (end - s) < p.nk ? kb + (end - s) : p.nk;
    band_tri_decode(p.rounds * G + t, p.T, ti, tj);
    run(ti, tj, kb, ke, acc);
    float* const dst = p.parts + (int64_t)(2 * w + slot) * kPartFloats32 + wave * 1024 + lane * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<f32x4_t*>(dst + q * 256) = f32x4_t{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    s += ke - kb;
  }
}

// One wave per 32x32 block of a left-over tile: adds the block's parts in k order and writes it out.
__global__ __launch_bounds__(64) void syrk_f32_reduce_kernel(F32Args p, int main_grid) {
  const int lane = threadIdx.x;
  const int t = (int)(blockIdx.x >> 2), blk = (int)(blockIdx.x & 3);
  int ti, tj;
  band_tri_decode(p.rounds * main_grid + t, p.T, ti, tj);
  const int s0 = t * p.nk, w0 = s0 / p.piece, w1 = (s0 + p.nk - 1) / p.piece;
  f32x16_t acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll 4
  for (int w = w0; w <= w1; ++w) {
    const int slot = 2 * w + (w * p.piece >= s0 ? 0 : 1);   // a piece that began in the tile before has this one second
    const float* src = p.parts + (int64_t)slot * kPartFloats32 + blk * 1024 + lane * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4_t v = *reinterpret_cast<const f32x4_t*>(src + q * 256);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[4 * q + e] += v[e];
    }
  }
  f32_write_block(p, acc, ti == tj, ti * T32 + (blk >> 1) * 32, tj * T32 + (blk & 1) * 32, lane);
}

// Rounds, left-over tiles and their pieces for an M x K operand.  In units of one k stage of one CU
// (1024 cycles, 0.45 us): left-over tiles kept whole cost nk for every 256 of them begun, cut into
// equal pieces rem nk / 256 and about 16 more for the parts' way through memory and the second launch.
void f32_schedule(int M, int K, F32Args& p) {
  p.T = (M + T32 - 1) / T32;
  p.nk = (K + BK32 - 1) / BK32;
  const int64_t tiles = (int64_t)p.T * (p.T + 1) / 2;
  p.rounds = (int)(tiles / kF32Grid);
  p.rem = (int)(tiles % kF32Grid);
  p.piece = 0;
  const int64_t left = (int64_t)p.rem * p.nk;
  if (p.rem > 0 && left < (1 << 30) && left / 256 + 16 < (int64_t)((p.rem + 255) / 256) * p.nk) {
    p.piece = (int)((left + kF32Grid - 1) / kF32Grid);
    if (p.piece < kMinPiece) p.piece = kMinPiece;
    if (p.piece > p.nk) p.piece = p.nk;
  }
}

}  // namespace

// (The last slot is never written - the last piece lies in the last tile alone, as piece <= nk - so that the ticket word that a workspace
// shared with 16-bit products holds in its last 256 bytes stays as it is.)
size_t syrk_f32_workspace_bytes(int M, int K) {
  F32Args p = {};
  f32_schedule(M, K, p);
  return p.piece ? (size_t)2 * kF32Grid * kPartFloats32 * sizeof(float) : 0;
}

int launch_syrk_f32(const float* X, int64_t ldx, float* Y, int64_t rs, int64_t cs, int M, int K, void* ws,
                    size_t ws_bytes, hipStream_t stream) {
  F32Args p = {};
  p.X = X; p.ldx = ldx; p.Y = Y; p.rs = rs; p.cs = cs; p.M = M; p.K = K;
  f32_schedule(M, K, p);
  p.parts = static_cast<float*>(ws);
  if (!ws || ws_bytes < (size_t)2 * kF32Grid * kPartFloats32 * sizeof(float)) p.piece = 0;
  const int64_t tiles = (int64_t)p.T * (p.T + 1) / 2;
  const unsigned grid = p.piece || p.rounds > 0 ? kF32Grid : (unsigned)tiles;
  if (!p.piece && p.rounds == 0) p.rem = (int)tiles;   // one tile per workgroup
  const bool vec = ldx % 4 == 0 && K % 4 == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0;
  if (vec) hipLaunchKernelGGL(syrk_f32_kernel<4>, dim3(grid), dim3(256), 0, stream, p);
  else hipLaunchKernelGGL(syrk_f32_kernel<1>, dim3(grid), dim3(256), 0, stream, p);
  if (p.piece) hipLaunchKernelGGL(syrk_f32_reduce_kernel, dim3((unsigned)p.rem * 4), dim3(64), 0, stream, p, (int)grid);
  return (int)hipGetLastError();
}

}  // namespace fm
