// The Newton-Schulz iteration of a batch of small or middling matrices as one launch.
//
// One step is three products, A = X X^T, P = b A + c A^2 and X' = a X + P X, and as launches of their own
// 15 of them follow each other, each with its start, its last tiles on a part of the chip and its gap.
// Here the 128x128 tiles of all products of all steps are items of eight queues, which two workgroups
// per CU draw from in order; an item waits until the tiles it reads from are counted as done.
//
// Queues.  The items of a product (all matrices of the batch, one after the other) are cut into eight
// contiguous runs, one per XCD, so that the workgroups of an XCD share operand panels in its L2; which
// XCD a workgroup is on is taken from its number and steers speed only.
//
// No deadlock, whatever part of the grid is resident: an item depends on items of the product before it
// only.  Of the items not yet done, take one of the earliest product.  What it depends on is done.  If it
// is drawn, the workgroup that drew it is running and holds no earlier one undone, so it gets to it; if
// not, it is at or behind the head of its queue, whose head is of the same product and ready, and every
// workgroup that waits looks at the heads of all queues and takes one that is ready and of an earlier product
// than its own.
//
// Coherence.  The L2s of the XCDs are not coherent for plain accesses.  Results that other workgroups
// read are stored through to memory (agent scope), and counted after the stores have been acknowledged;
// the iterate, A, P and its diagonal have memory of their own for every step, so that no address is read
// before it has been written and plain loads can find no stale line.
//
// What bounds it.  Few tiles: the chain of a product, 1.1 us from the first copy to the first stage, 0.2 us per
// 64-wide k stage of a 64x64 tile, 0.9 for the write-out and 2 to 4 from the last tile done to the next product's
// first copy (stores acknowledged, counted, seen): 512^2 6.5 us a product, 1024^2 8.5, where a launch takes 8
// and 10.  One counter per matrix instead of 16 words cost 5 to 9 us there (additions queue up).  Many tiles:
// the LDS, whose 750 cycles per stage and 128x128 tile are 0.38 us under load, and about 4 us of every tile that
// the CU's other workgroup does not cover.  24 of 768^2 360 us, in launches 393; 8 of 1024 x 2816 583 and 700;
// 16 of 512^2 137 and 185.
#include "fm_tile64.h"

namespace fm {

namespace {

constexpr int kQueues = 8;
constexpr int kLine = 32;             // words between counters: 128 bytes
constexpr int kMaxSubs = 16;          // words a count is spread over

struct FlowArgs {
  bf16_t* X; int64_t x_step;          // X of step s at X + s x_step, matrix m at + m M K
  bf16_t* A; bf16_t* P; int64_t a_step;
  float* pdiag; int64_t d_step, d_mat;
  int M, K, batch, steps;             // whole 128-tiles
  int ts, tm, tk;                     // symmetric tiles along M, X' tiles along M and K
  int sym_tiles, rect_tiles;          // of a symmetric product, of X'
  float a, b, c;
  unsigned* tickets;                  // [kQueues] of kLine words
  unsigned* done;                     // [3 steps][batch][subs] of kLine words
  int subs;
  PtrList out; int64_t ldout;
  int rows, cols;                     // of the output
  int tall, vec;
};

constexpr int kEnd = -1, kFlush = -2;   // messages that are no item
struct Item { int prod, m, tile; };   // product 3 step + {0: A, 1: P, 2: X'}

// items of queue q in a product of n tiles in all: [n q / 8, n (q + 1) / 8)
__device__ __forceinline__ int run_begin(int n, int q) { return (int)((unsigned)n * (unsigned)q >> 3); }

__device__ __forceinline__ int queue_total(const FlowArgs& p, int q) {
  const int ns = p.sym_tiles * p.batch, nr = p.rect_tiles * p.batch;
  return p.steps * (2 * (run_begin(ns, q + 1) - run_begin(ns, q)) + run_begin(nr, q + 1) - run_begin(nr, q));
}
__device__ __forceinline__ Item item_at(const FlowArgs& p, int q, int t) {
  const int ns = p.sym_tiles * p.batch, nr = p.rect_tiles * p.batch;
  const int s0 = run_begin(ns, q), r0 = run_begin(nr, q), cs = run_begin(ns, q + 1) - s0, cr = run_begin(nr, q + 1) - r0;
  const int per = 2 * cs + cr, step = t / per;
  t -= step * per;
  Item it;
  const int op = t < cs ? 0 : t < 2 * cs ? 1 : 2;
  const int i = op == 2 ? r0 + t - 2 * cs : s0 + t - op * cs, tiles = op == 2 ? p.rect_tiles : p.sym_tiles;
  it.prod = 3 * step + op;
  it.m = i / tiles;
  it.tile = i - it.m * tiles;
  return it;
}
__device__ __forceinline__ unsigned load_agent(const unsigned* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void count_up(unsigned* p) { __hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// The tiles done of matrix m in product `prod` are counted in `subs` words on lines of their own, tile t in
// word t % subs: additions to one word are taken one after the other, some 30 ns each.
__device__ __forceinline__ unsigned* counts(const FlowArgs& p, int prod, int m) {
  return p.done + (size_t)((prod * p.batch + m) * p.subs) * kLine;
}
// What an item waits for is looked at by a whole wave: lane i reads word i, `enough` adds them up.
__device__ __forceinline__ unsigned look_at(const FlowArgs& p, const Item& it, int lane) {
  return it.prod > 0 && lane < p.subs ? load_agent(counts(p, it.prod - 1, it.m) + lane * kLine) : 0u;
}
__device__ __forceinline__ bool enough(const FlowArgs& p, const Item& it, unsigned seen) {
  if (it.prod == 0) return true;
#pragma unroll
  for (int o = kMaxSubs / 2; o > 0; o >>= 1) seen += __shfl_xor(seen, o, 64);
  return __builtin_amdgcn_readfirstlane(seen) >= (unsigned)(it.prod % 3 == 0 ? p.rect_tiles : p.sym_tiles);   // of the product before
}
__device__ __forceinline__ unsigned draw(unsigned* head, int lane) {
  unsigned t = 0;
  if (lane == 0) t = __hip_atomic_fetch_add(head, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return t;   // lane 0's
}

// an item for a workgroup that waits for one of product `prod`: the head of some queue, if it is of an earlier
// product and ready
__device__ bool help(const FlowArgs& p, int prod, Item& it, int lane) {
  for (int q = 0; q < kQueues; ++q) {
    unsigned* const head = p.tickets + q * kLine;
    unsigned t = __builtin_amdgcn_readfirstlane(load_agent(head));
    if ((int)t >= queue_total(p, q)) continue;
    const Item c = item_at(p, q, (int)t);
    if (c.prod >= prod || !enough(p, c, look_at(p, c, lane))) continue;
    int got = 0;
    if (lane == 0) got = __hip_atomic_compare_exchange_strong(head, &t, t + 1, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(got)) {
      it = c;
      return true;
    }
  }
  return false;
}

// cache policy of stores that other XCDs read (sc1: written through to memory)
constexpr int kThrough = 16;

// Edges of the tiles, 128 or 64: ES of the symmetric products, EX of X'
template <int ES, int EX>
__global__ __launch_bounds__(256, 2) void ns_flow_kernel(FlowArgs p) {
  __shared__ __align__(1024) unsigned char smem[t128::SMEM];   // the ring of either tile size
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  typedef volatile __attribute__((address_space(3))) int lds_int;
  lds_int* const msg = (lds_int*)(smem);   // between items the ring is free

  // Wave 0, all lanes alike: the queue it draws from, how many it has found empty, the ticket drawn ahead and
  // the item it stands for, with what was seen of the counts that one waits for.
  int q = (int)blockIdx.x & (kQueues - 1), empty = 0;
  unsigned next = 0, seen = 0;
  bool drawn = false, holding = false, looked = false;
  Item mine = {}, ahead = {};
  // the count of the item before, if its stores have not been waited for yet (thread 0; `open`: all threads)
  unsigned* count = nullptr;
  bool open = false;

  for (;;) {
    if (wave == 0) {
      Item now = {kEnd, 0, 0};
      if (looked) {   // the item of the ticket drawn ahead
        mine = ahead;
        holding = true;
        drawn = false;
      }
      while (!holding && empty < kQueues) {
        if (!drawn) next = draw(p.tickets + q * kLine, lane);
        const int t = (int)__builtin_amdgcn_readfirstlane(next);
        drawn = false;
        if (t < queue_total(p, q)) {
          mine = item_at(p, q, t);
          holding = true;
        } else {
          q = (q + 1) & (kQueues - 1);
          ++empty;
        }
      }
      if (holding) {
        if (enough(p, mine, looked ? seen : look_at(p, mine, lane))) {
          now = mine;
          holding = false;
        } else if (open) {   // nothing to go on with: first say that the item before is done
          now.prod = kFlush;
        } else {
          for (int n = 1;; ++n) {
            if (enough(p, mine, look_at(p, mine, lane))) { now = mine; holding = false; break; }
            if ((n & 63) == 0 && help(p, mine.prod, now, lane)) break;
          }
        }
        looked = false;
      }
      if (lane == 0) {
        msg[0] = now.prod;
        msg[1] = now.m;
        msg[2] = now.tile;
      }
      // the next ticket of the same queue comes while this item is worked on
      if (now.prod >= 0 && !holding) {
        next = draw(p.tickets + q * kLine, lane);
        drawn = true;
      }
    }
    __syncthreads();
    const int prod = __builtin_amdgcn_readfirstlane(msg[0]), m = __builtin_amdgcn_readfirstlane(msg[1]),
              tile = __builtin_amdgcn_readfirstlane(msg[2]);
    __syncthreads();   // everybody has read the message before the copies overwrite it
    if (prod < 0) {
      if (open) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's results are in memory ...
        __syncthreads();                                   // ... and every wave's
        if (threadIdx.x == 0) count_up(count);
        open = false;
        count = nullptr;
      }
      if (prod == kEnd) break;
      continue;
    }
    const int step = prod / 3, op = prod - 3 * step;
    const int64_t mk = (int64_t)p.M * p.K, mm = (int64_t)p.M * p.M;
    const bf16_t* const X = p.X + step * p.x_step + m * mk;
    bf16_t* const A = p.A + step * p.a_step + m * mm;
    bf16_t* const P = p.P + step * p.a_step + m * mm;
    float* const pd = p.pdiag + step * p.d_step + m * p.d_mat;
    int l = lane;
    asm volatile("" : "+v"(l));   // per-lane addresses derived anew for every item
    // behind the main loop: what the next item is and waits for, answered while this one is written out
    auto look = [&]() {
      if (wave == 0 && drawn) {
        const int t = (int)__builtin_amdgcn_readfirstlane(next);
        if (t < queue_total(p, q)) {
          ahead = item_at(p, q, t);
          seen = look_at(p, ahead, lane);
          looked = true;
        }
      }
    };
    const bool last = step + 1 == p.steps;
    if (op < 2) {
      int ti, tj;
      band_tri_decode(tile, p.ts, ti, tj);
      if constexpr (ES == 128) {
        f32x4_t acc[4][4];
        uint32_t voA[4], voB[4];
        const bf16_t* const S = op == 0 ? X : A;
        const int lds_ = op == 0 ? p.K : p.M;
        const t128::Lane L = t128::lane_setup(smem, l, wave);
        t128::copy_offsets(voA, voB, lds_, lds_, l, wave);
        t128::main_loop<false>(acc, lds_ / t128::BK, smem, L, voA, voB, S + (int64_t)ti * 128 * lds_, S + (int64_t)tj * 128 * lds_, count);
        look();
        t128::Out o;
        o.C = o.C2 = op == 0 ? A : P;
        o.c_rs = o.c2_rs = p.M;
        o.ET = op == 0 ? nullptr : A;
        o.ldet = p.M;
        o.alpha = p.b;
        o.beta = p.c;
        o.row_alpha = nullptr;
        o.diag_out = op == 0 ? nullptr : pd;
        t128::write_block<false, kThrough>(o, ti == tj, acc, smem + wave * 16384, ti * 128 + (wave >> 1) * 64, tj * 128 + (wave & 1) * 64, l);
      } else {
        // rows of the tile belong to operand A (r), columns to operand B (c)
        const int r0 = ti * 64, c0 = tj * 64;
        f32x4_t acc[2][2];
        uint32_t vo[2];
        t64::Pre pre;
        t64::Out o;
        o.diag_out = nullptr;
        o.beta = 1.0f;
        o.C = op == 0 ? A : P;
        o.ld = p.M;
        o.by_c = true;
        o.by_r = ti != tj;   // a diagonal tile holds its own mirror image
        o.vec = true;
        o.rows_v = o.cols_v = p.M;
        if (op == 0) {
          const t64::Lane L = t64::lane_setup<false>(smem, l, wave);
          t64::copy_offsets<false>(vo, p.K, l, wave);
          t64::main_loop<false>(acc, p.K / t64::BK, smem, L, vo, vo, X + (int64_t)r0 * p.K, t64::BK, X + (int64_t)c0 * p.K, t64::BK, count);
          look();
          t64::write_tile<false, kThrough>(o, pre, acc, smem, r0, c0, l, wave);
        } else {   // A is symmetric: its columns are read as rows
          t64::load_block(pre, A + (int64_t)c0 * p.M + r0, p.M, wave * 64 + l);
          pre.al[0] = pre.al[1] = p.b;
          o.beta = p.c;
          if (ti == tj) o.diag_out = pd;
          const t64::Lane L = t64::lane_setup<true>(smem, l, wave);
          t64::copy_offsets<true>(vo, p.M, l, wave);
          t64::main_loop<true>(acc, p.M / t64::BK, smem, L, vo, vo, A + r0, t64::BK * p.M, A + c0, t64::BK * p.M, count);
          look();
          t64::write_tile<true, kThrough>(o, pre, acc, smem, r0, c0, l, wave);
        }
      }
    } else {
      // X' = (a + diag P) X + P X, computed as columns of X (rows of the tile) by rows of P
      const int band = tile / (8 * p.tk), r = tile - band * 8 * p.tk;
      const int brows = p.tm - band * 8 < 8 ? p.tm - band * 8 : 8;
      const int tj = r / brows, ti = band * 8 + (r - tj * brows);
      bf16_t* const Xn = last ? reinterpret_cast<bf16_t*>(p.out.p[m]) : p.X + (step + 1) * p.x_step + m * mk;
      const int64_t ld = last ? p.ldout : p.K;
      const int rows_v = last ? p.rows : p.M, cols_v = last ? p.cols : p.K;
      const bool tall = last && p.tall, vec = !last || p.vec;
      uint32_t voX[2], voP[2];
      if constexpr (EX == 128) {
        const int j0 = tj * 128 + (wave >> 1) * 64, i0 = ti * 128 + (wave & 1) * 64;
        f32x4_t acc[4][4];
        t128::PreT pre;
        t128::load_block_t(pre, X, p.K, pd, j0, i0, l);
        const t128::LaneT L = t128::lane_setup_t(smem, l, wave);
        t128::copy_offsets_t(voX, p.K, l, wave);
        t128::copy_offsets_t(voP, p.M, l, wave);
        t128::main_loop_t(acc, p.M / t128::KK_BK, smem, L, voX, voP, X + tj * 128, t128::KK_BK * p.K, P + ti * 128,
                          t128::KK_BK * p.M, count);
        look();
        const t128::OutT o = {Xn, ld, p.a, rows_v, cols_v, tall, vec};
        t128::write_block_t<kThrough>(o, pre, acc, smem + wave * 16384, j0, i0, l);
      } else {
        const int r0 = tj * 64, c0 = ti * 64;
        f32x4_t acc[2][2];
        t64::Pre pre;
        t64::load_block(pre, X + (int64_t)c0 * p.K + r0, p.K, wave * 64 + l);
#pragma unroll
        for (int j = 0; j < 2; ++j) pre.al[j] = p.a + pd[c0 + (wave & 1) * 32 + 16 * j + (l & 15)];
        const t64::Lane L = t64::lane_setup<true>(smem, l, wave);
        t64::copy_offsets<true>(voX, p.K, l, wave);
        t64::copy_offsets<true>(voP, p.M, l, wave);
        t64::main_loop<true>(acc, p.M / t64::BK, smem, L, voX, voP, X + r0, t64::BK * p.K, P + c0, t64::BK * p.M, count);
        look();
        const t64::Out o = {Xn, ld, tall, !tall, vec, rows_v, cols_v, 1.0f, nullptr};
        t64::write_tile<true, kThrough>(o, pre, acc, smem, r0, c0, l, wave);
      }
    }
    // its stores are waited for, and the item counted, when the next one's first stage has landed
    open = true;
    if (threadIdx.x == 0) count = counts(p, prod, m) + (tile & (p.subs - 1)) * kLine;
    __syncthreads();   // the staging is free for the next message
  }
}

}  // namespace

// words per count: about 64 for all matrices of a product
static int flow_subs(int batch) {
  int s = kMaxSubs;
  while (s > 1 && s * batch > 64) s >>= 1;
  return s;
}
int flow_counter_words(int batch, int steps) { return (kQueues + 3 * steps * batch * flow_subs(batch)) * kLine; }

int launch_ns_flow(const FlowProblem& f, hipStream_t stream) {
  FlowArgs p = {};
  p.X = f.X; p.x_step = f.x_step;
  p.A = f.A; p.P = f.P; p.a_step = f.a_step;
  p.pdiag = f.pdiag; p.d_step = f.d_step; p.d_mat = f.d_mat;
  p.M = f.M; p.K = f.K; p.batch = f.batch; p.steps = f.steps;
  p.ts = f.M / f.edge_s;
  p.tm = f.M / f.edge_x; p.tk = f.K / f.edge_x;
  p.sym_tiles = p.ts * (p.ts + 1) / 2;
  p.rect_tiles = p.tm * p.tk;
  p.a = f.a; p.b = f.b; p.c = f.c;
  p.tickets = f.counters;
  p.done = f.counters + kQueues * kLine;
  p.subs = flow_subs(f.batch);
  p.ldout = f.ldout; p.rows = f.rows; p.cols = f.cols; p.tall = f.tall;
  p.vec = f.ldout % 8 == 0 && f.ldout < (1 << 21);
  for (int i = 0; i < f.batch; ++i) {
    p.out.p[i] = f.out[i];
    if (reinterpret_cast<uintptr_t>(f.out[i]) & 15) p.vec = 0;
  }
  // as many workgroups as the largest product has items, in whole rounds of the queues
  const int64_t most = (int64_t)(p.rect_tiles > p.sym_tiles ? p.rect_tiles : p.sym_tiles) * f.batch;
  int grid = 2 * cu_count();
  if (grid > most) grid = (int)(most + kQueues - 1) / kQueues * kQueues;
#define FM_FLOW(ES, EX) hipLaunchKernelGGL((ns_flow_kernel<ES, EX>), dim3((unsigned)grid), dim3(256), 0, stream, p)
  if (f.edge_x == 64) FM_FLOW(64, 64);
  else if (f.edge_s == 64) FM_FLOW(64, 128);
  else FM_FLOW(128, 128);
#undef FM_FLOW
  return (int)hipGetLastError();
}

}  // namespace fm
