// Y = X * X^T of 16-bit matrices whose sides are no whole tiles, read and written in place.
//
// 128x128 tiles (fm_tile128.h), two workgroups per CU.  Rows of a tile beyond the last row of X repeat that row, and
// what they give is not stored.  The k that a stage of 64 does not divide comes first, as a stage whose copies end with the row: the
// lanes beyond it fetch the row's first 16 bytes of that stage once more and put zeros in their place before the
// barrier that hands the stage over.
//
// Schedule: whole tiles in rounds of 512, all workgroups in step so that those of an XCD find each other's panels in its L2
// (the tiles left over as one run of k stages, an equal piece per workgroup, which balances better but puts every
// workgroup at another k: 3000 x 5000 115 us, 8000^2 580 against 430).  Of the tiles left over, up to 256 stay whole, one per CU, and the
// rest are cut along k for the second workgroups; 256 or fewer are cut for as many workgroups where k is long.  The
// pieces' fp32 sums go to memory and a second kernel adds them in k order, so the bits do not depend on timing.
//
// Bound by the copies into the LDS: 0.43 us per 64-wide k stage, tile and CU with two workgroups (copies alone 0.36, 90 bytes
// per ns and CU), 0.53 with one.  Behind a copy of X 3000 x 5000 takes 53 us of 70, the copy 10.6, the second kernel 6.
#include "fm_routes.h"
#include "fm_tile128.h"

namespace fm {

namespace {

constexpr int kGrid = kRaggedGrid;
constexpr int kPartFloats = 128 * 128;

struct RaggedArgs {
  const bf16_t* X; int64_t ldx;
  bf16_t* Y; int64_t ldy;
  int M, tail, nk;      // elements of k beyond whole stages, stages per tile (the tail's among them)
  int T;                // tile rows
  int rounds;           // full rounds of gridDim.x tiles
  int whole, cut, parts;// of the tiles left over: kept whole, cut, pieces of each of these
  float* slots;         // the pieces' sums: all tiles' first pieces, then their second ones, ..
};

// k stages [kb, ke) of tile (ti, tj)
template <bool F16>
__device__ __forceinline__ void run_stages(const RaggedArgs& p, int ti, int tj, int kb, int ke, f32x4_t (&acc)[4][4], unsigned char* smem,
                                           const t128::Lane& L, int lane, int wave) {
  uint32_t voA[4], voB[4], hA[4], hB[4];
  int chunk[4];
  const int endA = p.M - 1 - ti * 128, endB = p.M - 1 - tj * 128;   // last row of X, from the tile's first
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int row = (q * 4 + wave) * 8 + (lane >> 3);
    chunk[q] = (lane & 7) ^ t128::swz16(row);
    const int a = t128::perm_a(row), b = t128::perm_b(row);
    const uint32_t ra = (uint32_t)(a < endA ? a : endA) * (uint32_t)p.ldx, rb = (uint32_t)(b < endB ? b : endB) * (uint32_t)p.ldx;
    const uint32_t c = chunk[q] * 8, h = (int)c < p.tail ? c : 0;
    voA[q] = (ra + c) * 2u;
    voB[q] = (rb + c) * 2u;
    hA[q] = (ra + h) * 2u;
    hB[q] = (rb + h) * 2u;
  }
  const bf16_t* const A = p.X + (int64_t)ti * 128 * p.ldx;
  const bf16_t* const B = p.X + (int64_t)tj * 128 * p.ldx;
  const bool head = p.tail != 0 && kb == 0;
  const int64_t k0 = (int64_t)(kb - (p.tail != 0 ? 1 : 0)) * t128::BK;
  const int64_t s0 = head ? (int64_t)(p.nk - 1) * t128::BK : k0;    // where stage kb is
  t128::main_loop_from<F16>(acc, ke - kb, smem, L, voA, voB, A + k0, B + k0, nullptr, head ? 1 : 0, [&]() {
#pragma unroll
    for (int q = 0; q < 4; ++q) t128::copy16(head ? hA[q] : voA[q], A + s0, L.ldsw, q * 4096);
#pragma unroll
    for (int q = 0; q < 4; ++q) t128::copy16(head ? hB[q] : voB[q], B + s0, L.ldsw, t128::B_OFF + q * 4096);
  }, [&]() {
    if (head) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (chunk[q] * 8 >= p.tail) {
          unsigned char* const at = smem + wave * 1024 + q * 4096 + lane * 16;
          *reinterpret_cast<uint4*>(at) = uint4{0, 0, 0, 0};
          *reinterpret_cast<uint4*>(at + t128::B_OFF) = uint4{0, 0, 0, 0};
        }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  });
}

template <bool F16>
__device__ __forceinline__ void write_out(const RaggedArgs& p, int ti, int tj, const f32x4_t (&acc)[4][4], unsigned char* T, int lane, int wave) {
  t128::Out o = {};
  o.C = o.C2 = p.Y;
  o.c_rs = o.c2_rs = p.ldy;
  o.limit = p.M;
  t128::write_block<F16, 0, true>(o, ti == tj, acc, T, ti * 128 + (wave >> 1) * 64, tj * 128 + (wave & 1) * 64, lane);
}

template <bool F16>
__global__ __launch_bounds__(256, 2) void syrk_ragged_kernel(RaggedArgs p) {
  __shared__ __align__(1024) unsigned char smem[t128::SMEM];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = (int)gridDim.x;
  // workgroups are dealt round-robin to the 8 XCDs: give each XCD a contiguous run of positions
  int w = (int)blockIdx.x;
  {
    const int chunk = G >> 3;
    if (w < chunk * 8) w = (w & 7) * chunk + (w >> 3);
  }
  const t128::Lane L = t128::lane_setup(smem, lane, wave);
  f32x4_t acc[4][4];
  int ti, tj;
  for (int r = 0; r < p.rounds; ++r) {
    band_tri_decode(r * G + w, p.T, ti, tj);
    run_stages<F16>(p, ti, tj, 0, p.nk, acc, smem, L, lane, wave);
    write_out<F16>(p, ti, tj, acc, smem + wave * 16384, lane, wave);
    __syncthreads();   // the staging is free for the next tile's copies
  }
  // Of the tiles left over the whole ones go to the first workgroup of every CU (ids below 256), the pieces to the
  // second or, without whole ones, to all.
  int at = w, whole = p.whole, cut = p.cut * p.parts;
  if (G == kGrid && whole > 0 && whole <= 256) {
    const int id = (int)blockIdx.x;
    at = (id & 7) * 32 + ((id >> 3) & 31);
    if (id < 256) cut = 0; else whole = 0;
  }
  if (at < whole) {
    band_tri_decode(p.rounds * G + at, p.T, ti, tj);
    run_stages<F16>(p, ti, tj, 0, p.nk, acc, smem, L, lane, wave);
    write_out<F16>(p, ti, tj, acc, smem + wave * 16384, lane, wave);
  } else if (at < cut) {
    const int part = at / p.cut;
    band_tri_decode(p.rounds * G + p.whole + at - part * p.cut, p.T, ti, tj);
    run_stages<F16>(p, ti, tj, p.nk * part / p.parts, p.nk * (part + 1) / p.parts, acc, smem, L, lane, wave);
    float* const dst = p.slots + (int64_t)at * kPartFloats + wave * 4096 + lane * 4;
#pragma unroll
    for (int i = 0; i < 16; ++i) *reinterpret_cast<f32x4_t*>(dst + i * 256) = acc[i >> 2][i & 3];
  }
}

// One wave per 64x64 block of a left-over tile: adds the block's parts in k order and writes it out.
template <bool F16>
__global__ __launch_bounds__(64) void syrk_ragged_reduce_kernel(RaggedArgs p, int main_grid) {
  __shared__ __align__(1024) unsigned char smem[16384];
  const int lane = threadIdx.x;
  const int t = (int)(blockIdx.x >> 2), blk = (int)(blockIdx.x & 3);
  int ti, tj;
  band_tri_decode(p.rounds * main_grid + p.whole + t, p.T, ti, tj);
  f32x4_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i >> 2][i & 3] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 2
  for (int k = 0; k < p.parts; ++k) {
    const float* src = p.slots + ((int64_t)k * p.cut + t) * kPartFloats + blk * 4096 + lane * 4;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i >> 2][i & 3] += *reinterpret_cast<const f32x4_t*>(src + i * 256);
  }
  write_out<F16>(p, ti, tj, acc, smem, lane, blk);
}

void set_schedule(int M, int K, RaggedArgs& p) {
  const RaggedSchedule s = ragged_schedule(M, K);
  p.M = M;
  p.tail = K % t128::BK;
  p.nk = s.nk; p.T = s.T;
  p.rounds = s.rounds; p.whole = s.whole; p.cut = s.cut; p.parts = s.parts;
}

}  // namespace

size_t syrk_ragged_workspace_bytes(int M, int K) {
  const RaggedSchedule s = ragged_schedule(M, K);
  return (size_t)s.cut * s.parts * kPartFloats * sizeof(float);
}

int syrk_ragged_reads(const bf16_t* X, int64_t ldx, int K) {
  if (K < t128::BK || K % 8 != 0 || ldx % 8 != 0 || ldx >= (1 << 23) || (reinterpret_cast<uintptr_t>(X) & 15) != 0) return kReadsNot;
  return ldx % 64 == 0 && (reinterpret_cast<uintptr_t>(X) & 127) == 0 ? kReadsLines : kReadsRows;
}

int launch_syrk_ragged(const bf16_t* X, int64_t ldx, bf16_t* Y, int64_t ldy, int M, int K, bool f16, void* ws, size_t ws_bytes, hipStream_t stream) {
  RaggedArgs p = {};
  set_schedule(M, K, p);
  p.X = X; p.ldx = ldx; p.Y = Y; p.ldy = ldy;
  p.slots = static_cast<float*>(ws);
  if (!ws || ws_bytes < (size_t)p.cut * p.parts * kPartFloats * sizeof(float)) { p.whole += p.cut; p.cut = 0; p.parts = 1; }
  const int groups = p.whole > 0 && p.cut > 0 ? kGrid : p.whole + p.cut * p.parts;
  const unsigned grid = p.rounds > 0 ? kGrid : (unsigned)groups;
  if (f16) hipLaunchKernelGGL(syrk_ragged_kernel<true>, dim3(grid), dim3(256), 0, stream, p);
  else hipLaunchKernelGGL(syrk_ragged_kernel<false>, dim3(grid), dim3(256), 0, stream, p);
  if (p.cut) {
    if (f16) hipLaunchKernelGGL(syrk_ragged_reduce_kernel<true>, dim3((unsigned)p.cut * 4), dim3(64), 0, stream, p, (int)grid);
    else hipLaunchKernelGGL(syrk_ragged_reduce_kernel<false>, dim3((unsigned)p.cut * 4), dim3(64), 0, stream, p, (int)grid);
  }
  return (int)hipGetLastError();
}

}  // namespace fm
