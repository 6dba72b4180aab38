// Which kernel or schedule a call takes, as plain arithmetic on its sizes: no device code and no HIP header, so that a
// host compiler can build it by itself and the rules can be checked without a GPU.
#pragma once
#include <stdint.h>

namespace fm {

// Blocks of 256 threads, four 8-element chunks per thread, for scale_cast_rows_kernel's walk over a rows_p x cols_p matrix
// (cols_p a multiple of 8), or 0 where it does not take it: the walk's index is an int, and every thread's last step goes
// up to one grid beyond the last chunk.  Larger matrices run on scale_cast_kernel, whose blocks are 64x64 tiles.
inline int64_t scale_cast_rows_blocks(int64_t rows_p, int64_t cols_p) {
  const int64_t chunks = rows_p * (cols_p / 8), blocks = (chunks + 1023) / 1024;
  return chunks + blocks * 256 <= INT32_MAX ? blocks : 0;
}

// D alone with a given sum of squares: on the kernel of 64x64 tiles where those are whole, up to 2^25 elements, rather than on the walk over rows.  us, tiles /
// rows: 1024^2 4.0 / 4.1, 1536^2 4.1 / 4.9, 2560^2 6.4 / 7.3, 2048 x 5504 9.2 / 10.2, 4096^2 12.4 / 12.8; but 4096 x 11008 30.7 / 28.1, 8192^2 41.7 / 41.0, and
// 3000^2 11.0 / 8.5, 3 x 1000000 9.0 / 5.3, 1000000 x 8 33 / 7.6.
inline bool scale_cast_d_on_tiles(int64_t rows, int64_t cols) { return rows % 64 == 0 && cols % 64 == 0 && rows * cols <= (1 << 25); }

// T alone, of whole 128-tiles and a given sum of squares, on the kernel of 128x128 tiles rather than that of 64x64: from about half as many of them as
// CUs on.  us, 64 / 128: 768^2 3.9 / 4.3, 1024^2 4.1 / 4.3 (64 tiles; fp32 4.1 / 4.6), 1536^2 4.8 / 4.8, 2048^2 6.4 / 5.4, 4096^2 15.9 / 13.0.
inline bool scale_cast_t_on_128(int64_t tiles) { return tiles >= 128; }

// Which matrices iterate in one launch (fm_flow.hip): M x K with M <= K, `batch` of them.
// Five steps in us, one launch / launches per product.  One or two matrices, whose products are chains of short launches:
// 256^2 91 / 109, 1024^2 137 / 158, 1408^2 185 / 233, 1024 x 4096 209 / 234, 1408 x 2816 225 / 302, 2 of 640 x 2560 156 / 245, 2 of 1408^2 249 /
// 285; but 1536^2 258 / 254, 1280 x 5120 383 / 304 (its first product is cut along k there), 2 of 768 x 3072 236 / 223.  More of
// them, with an odd number of 128-tiles (padded to 256-tiles, or on tiles of 128 in launches): 12 of 1152^2 532 / 817, 16
// of 1408^2 1009 / 1669, 6 of 1408 x 3872 976 / 1224, 12 of 1664^2 1253 / 1821; an even one, as long as the 256-tiles
// do not fill the GPU by themselves: 24 of 768^2 360 / 393, 16 of 768 x 3072 672 / 972, 16 of 1280^2 817 / 911, 6 of 1280 x 3520 774 / 844, 24 of
// 1536^2 2046 / 2102; but 6 of 768 x 3072 407 / 366, 6 of 1024 x 2048 424 / 377, 6 of 1280^2 451 / 423, 24 of 2048^2 4600 / 4200.
// So up to 768 rows of more than 1.5 : 1, and a few of 1280, only once X' would be more than about one round of 256-tiles (x, its 128-tiles, over 1000
// and 1050): 12 of 744 x 1992 433 / 571 and 8 of 768 x 3072 431 / 559, but 8 of 696 x 1864 344 / 321 (x = 720) and 10 of 768 x 1760 361 / 352; 4 of
// 1272 x 3416 586 / 678, but 4 of 1160 x 3112 550 / 517.  Three to seven of 1024 gain only where X' is about 256 or 512 tiles, one or two a CU (4 of
// 1024^2 199 / 234, 7 of 1024 x 1152 312 / 346, but 6 of 1024^2 280 / 274, 3 of 1024 x 1536 272 / 260, 6 of 960 x 1440 368 / 339), or long.  30 and more
// of 1280 fill the 256-tiles when long: 32 of 1280 x 3440 3693 / 3684, of 1216 x 4256 4466 / 4275.
// An odd number of 128-tiles, 11 and more: the larger it is, the less the padding costs, and the longer the matrices and the more of them, the
// better the 256-tiles are filled.  11: 16 of 1408 x 7744 4596 / 4974, but x 11264 6681 / 6581, 2 of 1408 x 2112 364 / 332, 3 of 1408 x 2816 520 / 440.
// 13: 12 of 1664 x 5488 3428 / 3757, 32 of 1608 x 3216 5870 / 6173, but 28 of 1608 x 6432 9348 / 8948, 5 of 1664^2 605 / 577.  15: 8 of 1920 x 3840
// 2152 / 2376, 24 of 1856 x 2784 5090 / 5280, but 12 of 1920 x 5160 4318 / 4216, 32 of 1920 x 7680 16558 / 14446.  Three of 9: 1088^2 212 / 235, but
// 1088 x 2176 339 / 307.
inline bool ns_flow_odd(int batch, int T, double r) {
  if (batch == 3) return T <= 7 ? r <= 2.75 : T == 9 && r <= 1.125;
  if (T <= 9) return true;
  if (T == 11) return r <= (batch <= 5 ? 12 : batch <= 8 ? 9 : 6);
  if (T == 13) return batch <= 5 ? r > 1.125 && r <= 6 : r <= (batch == 6 ? 4.5 : batch <= 8 ? 3.5 : batch <= 12 ? 4.1 : batch <= 16 ? 3.5 :
                                                                    batch < 28 ? 3 : 2.5);
  if (T == 15) return batch == 4 ? r > 1.125 && r <= 6 : r <= (batch == 5 ? 3 : batch <= 7 ? 2.25 : batch <= 10 ? 2.75 : batch <= 16 ? 2.1 :
                                                                    batch <= 24 ? 1.5 : 1.25);
  return false;
}
inline bool ns_flow_pays(int batch, int m, int k) {
  const double r = (double)k / m;
  if (m <= 512) return true;
  if (batch == 1) return m <= 1024 || (m <= 1408 && r <= 2.25);
  if (batch == 2) return m <= 640 || (m <= 1280 && r <= 2.75) || (m <= 1408 && r <= 1.125);
  const int T = (m + 127) / 128;
  const int64_t x = (int64_t)batch * T * (((int64_t)k + 127) / 128);
  if (T & 1) return ns_flow_odd(batch, T, r);
  if (m <= 768) return r <= 1.5 || (batch >= 8 && x > 1000);
  if (m <= 1024) return batch >= 8 || r > 3 || (x > 480 && x <= 512) || r <= (batch == 3 ? 1.4 : batch == 4 ? 1.125 : 0);
  if (m <= 1280) return r <= (batch < 30 ? 3.5 : 2.7) && (batch >= 12 || (batch >= 4 && r > 2.5 && x > 1050));
  return m <= 1536 && batch >= 16 && r <= 1.5;
}
// A long K: A = X X^T is whole tiles there, a chain of K / 64 stages (0.2 us each on a 64-tile), where a launch of its own is cut
// along k; and X' is 128-tiles, where a launch of its own has 256-tiles once there are enough of them.  With x the 128-tiles of X':
//   x about the CUs: up to K 8192.  512 x 8192 221 / 235 but x 10240 306 / 247, x 16384 398 / 275, x 65536 1268 / 629; 128 x 8192 166 / 179, x 16384
//   264 / 198; 1024 x 4096 212 / 242 but x 5120 (320 tiles) 314 / 277, x 16384 562 / 445; 2 of 512 x 4096 168 / 228 but x 8192 302 / 263; 4 of 256 x
//   8192 247 / 262;
//   an odd number of tile rows, which the 256-tiles do not fit, and enough matrices: up to 32768.  16 of 640 x 12288 1959 / 2383, 8 of 896 x 16384
//   2265 / 2464, 12 of 384 x 32768 2112 / 2281, but 4 of 576 x 131072 7547 / 6641;
//   eight matrices or more: up to 8192 below 1024 tiles, then 16384, 32768 for 24 of them (8 of 256 x 16384 509 / 531, 24 of 512 x 24576
//   4135 / 4206; but 8 of 128 x 16384 341 / 293, 8 of 512 x 24576 1682 / 1587, 16 of 256 x 24576 1353 / 1273), of more than 768 rows only while x <= 5000
//   (12 of 1024 x 6144 1568 / 1759 but 16 of it 2031 / 1978, 12 of 1024 x 12288 3081 / 2910);
//   fewer: one round of 256-tiles at most (x < 1024) up to K 4096 or 5120 (4 of 384 x 4096 206 / 245; but 2 of 512 x 5120 239 / 234, 3 of 512 x 6144
//   318 / 287, 6 of 256 x 8192 307 / 267; not above 768 rows: 4 of 960 x 3072 441 / 379), and beyond it where the 256-tiles' last round is a fifth
//   empty or more (4 of 1024 x 6144 679 / 822, 4 of 512 x 12288 481 / 631; but 4 of 1024 x 8192 921 / 817, 6 of 512 x 10240 633 / 585).
inline bool ns_flow_short_enough(int batch, int m, int k) {
  if (k <= 2048) return true;
  const int64_t T = (m + 127) / 128, x = batch * T * ((k + 127) / 128);
  if (x <= 280 || (m <= 256 && x <= 512)) return k <= 8192;
  if ((T & 1) && T > 1 && batch * T >= 18) return k <= 32768;
  if (batch >= 8) return k <= (x <= 1024 ? 8192 : batch < 24 ? 16384 : 32768) && (m <= 768 || k <= 4 * m || x <= 5000);
  if (x < 1024) return (m <= 768 || 4 * (int64_t)k <= 11 * (int64_t)m) && k <= (batch <= 4 ? 4096 : 5120);
  return k <= 12288 && x <= (x + 1023) / 1024 * 820;
}
inline bool ns_flow_chosen(int batch, int m, int k) { return ns_flow_pays(batch, m, k) && ns_flow_short_enough(batch, m, k); }
// The one-launch iteration has room for the iterates of kFlowSteps steps and the one they begin with, in slots 0 .. kFlowSteps.  More steps take
// further launches, which go back and forth over the slots: step i of a launch reads slot `from` + i `turn` and leaves the next iterate in
// the slot behind it (the very last step in the caller's output).  Every launch but the last has to take all kFlowSteps steps: one
// that went back by more slots than the one before it went forward would leave the workspace.
constexpr int kFlowSteps = 5;
struct NsFlowLaunch { int first, steps, from, turn; };   // first: of its steps
inline NsFlowLaunch ns_flow_launch(int steps, int i) {   // launch i of the (steps + kFlowSteps - 1) / kFlowSteps
  const int first = i * kFlowSteps, left = steps - first;
  return NsFlowLaunch{first, left < kFlowSteps ? left : kFlowSteps, i & 1 ? kFlowSteps : 0, i & 1 ? -1 : 1};
}

// ---- X X^T in 16 bits of sides that the 256-tiles do not fit -------------------------------------
// The in-place kernel's schedule (fm_gemm_ragged.hip): 128x128 tiles in full rounds of 512 workgroups; of those left over `whole` in one
// piece and `cut` in `parts` pieces along k each.
constexpr int kRaggedGrid = 512;                        // workgroups: two per CU
constexpr int kRaggedMinPiece = 8, kRaggedMaxParts = 16;   // stages a piece has at least, pieces of a tile
struct RaggedSchedule { int T, nk, rounds, whole, cut, parts; };
inline RaggedSchedule ragged_schedule(int M, int K) {
  RaggedSchedule s;
  s.nk = (K + 63) / 64;
  s.T = (M + 127) / 128;
  const int64_t tiles = (int64_t)s.T * (s.T + 1) / 2;
  s.rounds = (int)(tiles / kRaggedGrid);
  const int rem = (int)(tiles % kRaggedGrid);
  s.whole = rem; s.cut = 0; s.parts = 1;
  if (rem > 256) {
    int n = 256 / (rem - 256);
    if (n > kRaggedMaxParts) n = kRaggedMaxParts;
    if (n > s.nk / kRaggedMinPiece) n = s.nk / kRaggedMinPiece;
    if (n > 1 && s.nk - s.nk / n >= 40) { s.whole = 256; s.cut = rem - 256; s.parts = n; }
  } else if (rem > 0) {
    int n = 256 / rem;
    if (n > kRaggedMaxParts) n = kRaggedMaxParts;
    if (n > s.nk / kRaggedMinPiece) n = s.nk / kRaggedMinPiece;
    if (n > 1 && s.nk - s.nk / n >= (s.rounds > 0 ? 45 : 25)) { s.whole = 0; s.cut = rem; s.parts = n; }
  }
  return s;
}

// Its time in us, in place or (`lines` false) behind a copy of X, and that of both X and Y as copies padded to whole 256-tiles
// (a round of 256 of them, the rest cut along k; `aligned`: rows of Y that 16-byte stores can take).  Constants: least squares over 400 sizes
// of 2900 to 28000 rows and K of 200 to 16000, 4 % rms each.  A stage of a tile slows down once X and what is written beside it outgrow the 256 MB
// of the memory-side cache, on 128-tiles (twice the operand bytes per flop) from about 100 MB of X on.
inline double syrk_ragged_us(int M, int K, bool lines) {
  const RaggedSchedule s = ragged_schedule(M, K);
  const double mk = (double)M * K, mm = (double)M * M, mb = 2e-6 * mk;
  double t = s.rounds * (0.77 * s.nk - 4.8) + 6.8e-7 * mm;
  if (s.cut) t += s.whole ? 0.62 * s.nk - 3.6 : 0.37 * s.nk / s.parts + 11.2;
  else if (s.whole) t += s.whole <= 256 ? 0.37 * s.nk + 0.5 : 0.66 * s.nk - 0.6;
  double slow = 1.0 + (lines ? 0.0045 * (mb - 105.0) : 0.005 * (mb - 100.0));
  slow = slow < 1.0 ? 1.0 : slow > 1.5 ? 1.5 : slow;
  return t * slow + (lines ? 3.5 : 7.5 + 6.8e-7 * mk);
}
inline double syrk_padded_us(int M, int K, bool aligned) {
  const int64_t T = (M + 255) / 256, tiles = T * (T + 1) / 2, rounds = tiles / 256, rem = tiles % 256;
  const double nk = (K + 63) / 64, mk = (double)M * K, out = (aligned ? 7.1e-7 : 15.4e-7) * M * M;
  if (T == 16)   // 256 half tiles, one round
    return 12.4 + 6.8e-7 * mk + out + (mk < 7e7 ? 0.71 : 0.85) * nk;
  double t = 4.4 + 1.9e-6 * mk + out + rounds * (1.07 * nk + 19.6);
  const int64_t parts = rem ? 256 / rem : 1;
  if (rem && parts < 16) t += 0.753 * nk / parts + (parts == 1 ? 8.0 : 11.4);   // (up to 16 of them run as sub-tiles beside the rounds)
  return t;
}
// Whether rows that 16-byte copies can take but that do not lie on 128-byte lines (`half`: on halves of them) are copied first: a 128-byte piece of such a
// row makes two requests of one.  us, in place / behind a copy of X: 3000 x 5000 75 / 70, 7000 x 2000 129 / 110; but 2000^2 23 / 30, 4000 x 1000 33 / 37,
// where a launch and 8 bytes of traffic per element cost more than they save in 16384 stages of tiles or less; and with a tile on half of the CUs (on half
// lines four fifths), whose stages the requests do not hold up, 1000 x 65544 106 / 126, 1920 x 65544 349 / 385, half lines 1956 x 12000 94 / 104, 2468 x
// 12000 100 / 112 (but 2432 x 9304, 190 tiles, 92 / 88, 2768 x 9784, 253 tiles, 107 / 101).
inline bool syrk_copy_pays(int M, int K, bool half) {
  const RaggedSchedule s = ragged_schedule(M, K);
  const int64_t tiles = (int64_t)s.T * (s.T + 1) / 2;
  return tiles > (half ? 210 : 136) && tiles * s.nk >= 16384;
}
// Whether it is padded, for matrices that may be (the copies cost memory: not for a gain of under 4 % of the estimates).  us, in place
// or behind a copy of X / padded: 4000^2 86 / 78, 3936 x 4000 69 / 77, 5280 x 6000 183 / 167, 5536 x 4000 127 / 130, 7776 x 4000 242 / 248, 8096 x 8040 509 / 453,
// 8008 x 4000 246 / 263, 8008 x 16000 1102 / 821, 10000 x 8000 887 / 700, 16008 x 2000 544 / 646, x 4000 1159 / 974, x 8000 2576 / 1684, 24000 x 4000 3036 / 2152; of whole
// tiles 7552 x 4096 195 / 253, x 16384 898 / 781, 10112 x 8192 1007 / 711, 16256 x 8192 2783 / 1722.
// Below 16 tile rows of 256, where the padded product is cut along k over all CUs: of 8 to 10, whose 120 to 210 tiles of 128 leave CUs idle, by the time of
// a stage in place (rows on lines, on half lines, neither) against a linear fit of the padded way: 2043 x 7496 74 / 67, 1956 x 12000 94 / 93, 2468 x 12000 100 / 116,
// 2560 x 30416 289 / 223, x 24000 on lines 180 / 191, 2200 x 72576 on lines 581 / 416; of more only a matrix that does not fit the cache: 2980 x 24000 (143 MB) 220
// / 319, 3664 x 24072 off them (176 MB) 391 / 340, 3200 x 32768 on lines (210 MB) 317 / 406, 2980 x 60000 (358 MB) 768 / 531; of fewer (1000 x 262144 340 / 497) none.
constexpr int kRowsLines = 0, kRowsHalfLines = 1, kRowsAny = 2;
inline bool syrk_padded_pays(int M, int K, int rows, bool aligned) {
  if (K < 1500 || K > (1 << 21) - 128 || M <= 7 * 256) return false;   // (4056 x 1248 38 / 43; what the 256-tiles' byte offsets allow)
  const int T = (M + 255) / 256, nk = (K + 63) / 64;
  if (T <= 10) return 0.96 * (3.6 * T + (0.144 + 0.026 * T) * nk) < 2.0 + (rows == kRowsLines ? 0.47 : rows == kRowsHalfLines ? 0.51 : 0.60) * nk;
  if (T < 16) return 2e-6 * M * K > (rows == kRowsLines ? 260.0 : T >= 14 ? 130.0 : 200.0);
  return 0.96 * syrk_padded_us(M, K, aligned) < syrk_ragged_us(M, K, rows == kRowsLines);
}

// ---- 128x128 tiles of whole, aligned matrices, one per CU (launch_gemm_mid) ------------------------
// Parts per tile along k, by estimate in microseconds (measured: 0.36 per stage, 4.5 for a
// tile's start and write-out; cut, 11 for the fp32 round trip and the second launch and 0.035 per
// part for their traffic).  At most as many parts as fill the chip, of at least 8 stages each; the
// tiles stay whole unless the cut saves a tenth.
inline double mid_cut_us(long long tiles, int nk, int s) { return (double)((nk + s - 1) / s) * 0.36 + 11.0 + 0.035 * (double)(tiles * s); }
inline int mid_parts(long long tiles, int nk, int grid) {
  if (tiles * 2 > grid || nk < 16) return 1;
  int smax = (int)(grid / tiles);
  if (smax > nk / 8) smax = nk / 8;
  if (smax > 16) smax = 16;
  int best = 1;
  double t_best = 0.9 * (nk * 0.36 + 4.5);
  for (int s = 2; s <= smax; ++s) {
    const double t = mid_cut_us(tiles, nk, s);
    if (t < t_best) { t_best = t; best = s; }
  }
  return best;
}
// (a stage costs 0.36 us while about half the CUs work and 0.52 when all do; a write-out with an
// operand E costs 5 more)
inline double mid_us(long long tiles, int nk, int grid, int parts, bool with_e) {
  if (parts > 1) return mid_cut_us(tiles, nk, parts) + (with_e ? 5.0 : 0.0);
  const double occ = tiles >= grid ? 1.0 : (double)tiles / grid;
  const double stage = 0.36 + 0.36 * (occ > 0.55 ? occ - 0.55 : 0.0);
  return (double)((tiles + grid - 1) / grid) * (nk * stage + (with_e ? 11.0 : 6.0));
}

// The same as halves of the tiles, at most one a CU (fm_gemm_slim.hip): a stage of 24 KiB, no cut.  us, whole tiles / halves: X X^T 1536 x
// 1024 11.1 / 8.8, x 4096 27.8 / 22.1, 1792 x 2048 17.4 / 14.1, x 6144 39.7 / 33.0, 2048^2 17.8 / 15.1, x
// 8192 50.8 / 43.2.  (Beyond 72 stages all of these kernels take 3 to 4 us more than their stages before, and a
// stage of 2048 rows beyond 336 of them 0.30 to 0.32: x 20480 100, x 22528 122, x 24576 123, x 32768 164, where 256-tiles cut along k, whose estimate is
// as high, take 105 and 130 for the last two.)
inline double slim_us(long long tiles, int nk, int grid, bool with_e) {
  const double occ = 2.0 * tiles >= grid ? 1.0 : 2.0 * (double)tiles / grid;
  return 5.7 + nk * (0.223 + 0.037 * occ) * (nk > 336 ? 1.25 : 1.0) + (nk > 72 ? 3.0 : 0.0) + (with_e ? 2.0 : 0.0);
}
// Halves rather than whole tiles always, and than tiles cut into `parts` along a long k where they are estimated to be 5 % faster: they
// hardly ever are.  us, cut / halves: 1536 x 5120 27.5 / 29.8, x 6144 30.0 / 32.2, x 8192 33.7 / 38.0, 1664 x 7680 37.7 / 40.5, 1792 x 8128 42.1 / 43.8, x
// 16384 65.3 / 70.3, 512 x 8192 22.9 / 33.9, 1024 x 8192 24.9 / 35.5; near ties 1664 x 8192 38.5 / 39.6, 1792 x 8192 41.1 / 39.1.
inline bool slim_pays(long long tiles, int nk, int grid, int parts, bool with_e) {
  return parts == 1 || slim_us(tiles, nk, grid, with_e) < 0.95 * mid_us(tiles, nk, grid, parts, with_e);
}

// X X^T of an odd number of whole 128-tiles on halves of them rather than in place or on whole tiles (below).  us, otherwise / halves: 640 x 2048 13.4 / 12.1, 896 x
// 1024 9.3 / 8.7, 1152 x 2048 14.6 / 12.4, 1664 x 4096 25.5 / 22.7, 1920 x 4096 27.7 / 24.0; but 640 x 4096 15.4 / 18.9, 1152 x 8192 24.0 / 26.9.
inline bool syrk_whole_slim(int M, int K) { return M <= 1920 && K >= 1024 && K <= (M >= 1664 ? 4096 : 2048); }

// X X^T of an odd number of whole 128-tiles, rows on lines: in place on tiles that share a CU in pairs (fm_gemm_ragged.hip), or on the
// tiles above.  us, above / in place: more tiles than CUs 2944^2 46.7 / 38.2, 4224^2 96 / 78, 5504 x 2048 81 / 62, 8064 x 1024 114 / 70; 121 to
// 256 of them 2176^2 20.7 / 21.8, 2688^2 26.3 / 26.9.  Fewer: the deeper ring above starts later (4 us) and takes 0.36 us a stage where
// this one takes 0.53, which is why a long k, cut or not, is better off there: 1408 x 1024 11.5 / 9.5, x 2048 16.9 / 18.8, x 4096 27.4 / 21.5 (cut in
// place alone), x 8192 31.8 / 31.4, x 16384 48.1 / 51.3, x 32768 80 / 94; 1920 x 3072 23.3 / 26.9, x 6144 40.0 / 34.7, x 32768 125 / 144; 640 x 32768 31.3 / 28.1.
// (estimates within 10 % of these; a near tie stays in place)
inline bool syrk_whole_in_place(int M, int K, int cus) {
  const int64_t T = M / 128, tiles = T * (T + 1) / 2;
  if (tiles > 256) return true;
  if (tiles > 120) return false;
  const RaggedSchedule s = ragged_schedule(M, K);
  const double load = tiles < 66 ? tiles / 66.0 : 1.0, busy = tiles < 28 ? tiles / 28.0 : 1.0;
  const double t = s.cut ? 9.0 + 0.015 * s.cut * s.parts + (0.36 + 0.12 * busy * busy) * ((s.nk + s.parts - 1) / s.parts)
                         : 2.2 + (0.33 + 0.19 * load * load) * s.nk;
  return 0.97 * t <= mid_us(tiles, s.nk, cus, mid_parts(tiles, s.nk, cus), false);
}

// ---- 256-tiles left over after full rounds --------------------------------------------------------
// `rem` of them, 17 to half as many as CUs: a round of `split` parts of each along k, which go to memory as fp32, and a second kernel that adds them;
// or a launch of their halves behind the rounds.  What the halves gain, fitted to X X^T of 23 to 27 tile rows (us): 7 and 0.105 a tile for the
// parts' way through memory and the second kernel, and a stage of a part (1.3 / split) against one of a half (0.3 to 0.7, by the CUs they fill).
//   20 left (5888 rows) K 1024 63.3 / 54.7; 44 (6144) K 1024 65.4 / 56.3, 2048 91.5 / 86.4; 69 (6400) K 1024 69.5 / 57.2, 4096 155.8 / 148.5, but 6144 198 / 207, 7168
// 239 / 242; 95 (6656) K 1024 73.2 / 58.0, 4096 168 / 151, 8192 292 / 275; 122 (6912) K 256 54.6 / 35.3, 4096 173.5 / 156.5; five Newton-Schulz steps on 32 of 2048^2
// (128 left) 5600 / 5450, on 8 of 3072^2 (112) 4440 / 4270.
inline bool half_tail_pays(int rem, int split, int nk, int grid) {
  const double fill = 0.3 + 0.6 * 2.0 * rem / grid, half = fill < 0.7 ? fill : 0.7;
  return 7.0 + 0.105 * rem + nk * (1.3 / split - half) > 2.0;
}

}  // namespace fm
