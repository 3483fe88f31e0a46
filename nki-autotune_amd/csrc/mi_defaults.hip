// mi_defaults.hip -- the library default config (mi_default_config): for a
// call with no config, the block whose estimated time at the shape is the
// least, generalised from the autotune winners at the benchmark shapes,
// campaigns that timed every candidate block and split at about 200 more
// shapes, and studies of 83 shapes and of seeded random ones.  Host code
// only.
#include <math.h>
#include <stdint.h>

#include "mi_capi_internal.hpp"

namespace mi {
namespace capi {
namespace {

// Default configs.  A grid fills the chip with one workgroup per CU on 256
// CUs; 224 (28 per XCD) still counts as full.
constexpr long long kFillTiles = 224;
constexpr long long kCUs = 256;

long long tiles_of(int M, int N, int bm, int bn) {
  return (((long long)M + bm - 1) / bm) * (((long long)N + bn - 1) / bn);
}

// The most parts (a power of two, at most 16) that keep the grid within one
// workgroup per CU, every part at least 4 K tiles of block_k, and no part
// empty; 1 when no split qualifies.
int fill_parts(long long tiles, int K, int block_k) {
  const long long kt = ((long long)K + block_k - 1) / block_k;
  int parts = 1;
  for (int next = 2; next <= 16; next *= 2) {
    const long long kts = (kt + next - 1) / next;
    if (tiles * next > kCUs || kt < 4LL * next || (long long)(next - 1) * kts >= kt) break;
    parts = next;
  }
  return parts;
}

// A candidate block and its relative throughput per CU (output area per
// unit time at the same K, the 256 x 256 block = 1), measured with the
// autotuner at shapes that give every CU one tile.
struct Cand {
  mi_tile_cfg c;
  double rate;
};

// The candidate with the least estimated time: the rounds of tiles the
// busiest CU runs, times a tile's area over its rate.  Ties go to the
// earlier (larger) block.  Then, if its grid leaves CUs idle and K is long
// enough to split, K is split so the grid fills the chip.
mi_tile_cfg fastest_estimate(const Cand* cands, int n, int M, int N, int K, int kernel_id) {
  int best = 0;
  double best_t = 0.0;
  for (int i = 0; i < n; ++i) {
    const mi_tile_cfg& c = cands[i].c;
    const long long rounds = (tiles_of(M, N, c.block_m, c.block_n) + kCUs - 1) / kCUs;
    const double t = (double)rounds * c.block_m * c.block_n / cands[i].rate;
    if (i == 0 || t < best_t) {
      best = i;
      best_t = t;
    }
  }
  mi_tile_cfg c = cands[best].c;
  const long long tiles = tiles_of(M, N, c.block_m, c.block_n);
  if (tiles >= kFillTiles || fill_parts(tiles, K, c.block_k) == 1) return c;
  // The grid needs a split: the largest splittable block whose split grid
  // is as large as any (a bigger block moves fewer operand bytes per
  // multiply-add for the same workgroup count).
  long long most = 0;
  for (int i = 0; i < n; ++i) {
    const mi_tile_cfg& ci = cands[i].c;
    if (!splittable(kernel_id, ci.variant)) continue;
    const long long t = tiles_of(M, N, ci.block_m, ci.block_n);
    const long long wgs = t * fill_parts(t, K, ci.block_k);
    if (wgs > most) {
      most = wgs;
      c = ci;
    }
  }
  c.split_k = fill_parts(tiles_of(M, N, c.block_m, c.block_n), K, c.block_k);
  return c;
}

// As fastest_estimate, for the fused kernel (whose first candidate needs no
// workspace), but each candidate is first split by fill_parts when its grid
// leaves CUs idle, a candidate whose device workspace would pass the 2 GiB
// limit is skipped, and its estimated time (microseconds) adds the
// split's fp32 partial products, written once and read back once at about
// 5 TB/s, and for the two-pass fused kernel (variant 13) its pack pass (x
// read, x * gamma written: 4 bytes per x element at about 5 TB/s) and 3 us
// for the second launch.  R0 is the fused kernel's 128 x 512 rate per CU at
// 4096^3, in multiply-adds per second.
// The fewest parts, from c.split_k up by powers of two, that leave every K
// part within the gamma entries the fused instance stages in LDS and no part
// empty; 0 when none up to kMaxSplit does (or the instance is not built).
int gamma_fit_parts(const mi_tile_cfg& c, int K) {
  const mi::MiEntry* e = find(MI_KERNEL_RMSNORM_MATMUL_BF16, c);
  if (!e) return 0;
  const long long kt = ((long long)K + c.block_k - 1) / c.block_k;
  for (int p = c.split_k; p <= kMaxSplit; p *= 2) {
    const long long kts = (kt + p - 1) / p;
    if (p > 1 && (long long)(p - 1) * kts >= kt) return 0;
    if (e->gamma_kmax <= 0 || kts * c.block_k <= e->gamma_kmax) return p;
  }
  return 0;
}

mi_tile_cfg fastest_split_estimate(const Cand* cands, int n, int M, int N, int K, const mi_tile_cfg& fallback) {
  constexpr double R0 = 2.28e12, kSplitBytesPerUs = 5e6, kPackBytesPerUs = 5e6, kLaunchUs = 3.0;
  double best_t = 0.0;
  mi_tile_cfg best_c = fallback;
  bool found = false;
  for (int i = 0; i < n; ++i) {
    mi_tile_cfg c = cands[i].c;
    const long long tiles = tiles_of(M, N, c.block_m, c.block_n);
    c.split_k = tiles < kFillTiles ? fill_parts(tiles, K, c.block_k) : 1;
    if (!splittable(MI_KERNEL_RMSNORM_MATMUL_BF16, c.variant)) c.split_k = 1;
    // Past the gamma entries an instance stages, K splits further; a
    // candidate no split makes legal, or whose workspace the call could not
    // allocate, is out.
    c.split_k = gamma_fit_parts(c, K);
    if (c.split_k == 0) continue;
    if (mi::workspace_bytes(MI_KERNEL_RMSNORM_MATMUL_BF16, c, M, N, K, kDefaultCus) > kMaxWorkspace) continue;
    const long long wgs = tiles * c.split_k, rounds = (wgs + kCUs - 1) / kCUs;
    const double kp = (double)((K + c.split_k - 1) / c.split_k);
    double t = (double)rounds * c.block_m * c.block_n * kp / (cands[i].rate * R0) * 1e6;
    // The chip is power-limited under this load, so a single round that
    // leaves CUs idle runs each busy CU faster (its clock rises): by up to
    // 0.88 / (the busy fraction), at most 1.65 times (fitted to the fused
    // candidates timed at 23 shapes).
    if (rounds == 1) {
      const double busy = (double)wgs / kCUs, speed = 0.88 / busy;
      t /= speed > 1.65 ? 1.65 : speed < 1.0 ? 1.0 : speed;
    }
    if (c.split_k > 1) t += (double)c.split_k * M * N * 8.0 / kSplitBytesPerUs + kLaunchUs;
    if (c.variant == 13) t += (double)M * K * 4.0 / kPackBytesPerUs + kLaunchUs;
    // Variant 15's pack writes x's own layout, no transpose: 0.9 of the time.
    if (c.variant == 15) t += 0.9 * (double)M * K * 4.0 / kPackBytesPerUs + kLaunchUs;
    if (!found || t < best_t) {
      found = true;
      best_t = t;
      best_c = c;
    }
  }
  return best_c;
}

// Skinny M (decode-like), either matmul: the weight is streamed once with
// the non-temporal variants (lhsT.rhs 3, lhs.rhs 2).
mi_tile_cfg skinny_matmul_default(bool lhs, int M, int N, int K) {
  const int v_nt = lhs ? 2 : 3;
  if (lhs) {
    // lhs.rhs: the non-temporal 128 x 128 block when its grid fills the
    // chip; otherwise the non-temporal block with the fewest wasted rows
    // (64 x 128 up to M = 64), split over K to up to one workgroup per CU.
    const mi_tile_cfg skinny = {128, 128, 64, 4, 3, 1, 8, v_nt};
    if (tiles_of(M, N, skinny.block_m, skinny.block_n) >= kFillTiles) return skinny;
    mi_tile_cfg c = M <= 64 ? mi_tile_cfg{64, 128, 64, 4, 4, 1, 8, v_nt} : skinny;
    c.split_k = fill_parts(tiles_of(M, N, c.block_m, c.block_n), K, c.block_k);
    // A 128-row split whose parts would keep under 1024 of K gives way to
    // the 64 x 128 block with block_k 128, itself split to fill the CUs
    // (128x9920x1600: unsplit, 17.9 us against 21.6 us for 128 x 128 in 2
    // parts of 800; 128x1856x14272: 8 parts, 26.0 us).
    if (c.block_m == 128 && c.split_k >= 2 && (K + c.split_k - 1) / c.split_k < 1024) {
      c = {64, 128, 128, 4, 3, 1, 8, v_nt};
      c.split_k = fill_parts(tiles_of(M, N, 64, 128), K, 128);
    }
    return c;
  }
  // lhsT.rhs: a skinny launch is bound by each workgroup's own loads (its
  // MFMA pipe is a quarter busy at most), so the estimate is the rounds of
  // workgroups times one workgroup's panel bytes, (block_m + block_n) x (its
  // K range + 256) x 2, at 70 GB/s per CU plus 3 us (the 256 rows of K
  // stand for the ring's fill, which a short part does not hide), and a
  // split pays its fp32 partial products, written and read back (8 bytes
  // per output element and part), at 5 TB/s plus 1 us for the summing
  // launch; splits stop at 8 parts, and every part keeps at least 512 of K.
  // Fitted to every block and split timed at 46 skinny shapes (M 8-128, K
  // 512-16384) with the weight flushed and the split workspace kept per
  // stream: the pick within 1.069 of the fastest at all of them (mean
  // 1.009), and within 1.034 at the third of the shapes held out of a fit
  // to the other two thirds.  Equal estimates go to the earlier block (32 x
  // 128 with block_k 64 and 4 stages measured faster than with block_k 128
  // and 3; 128 x 128 with block_k 32 and 4 stages than with 64 and 3).
  const mi_tile_cfg cands[] = {
      {32, 128, 64, 4, 4, 1, 8, v_nt},  {32, 128, 128, 4, 3, 1, 8, v_nt}, {32, 256, 64, 4, 4, 1, 8, v_nt},
      {64, 128, 64, 4, 4, 1, 8, v_nt},  {64, 64, 64, 4, 4, 1, 8, v_nt},   {64, 256, 64, 4, 3, 1, 8, v_nt},
      {128, 128, 32, 4, 4, 1, 8, v_nt}, {128, 128, 64, 4, 3, 1, 8, v_nt}, {128, 256, 32, 4, 3, 1, 8, v_nt},
      {128, 256, 32, 4, 4, 1, 8, v_nt}};
  // Blocks more than twice as tall as M are not considered; splits stop at
  // 320 workgroups.
  const int m_cap = 2 * (M > 32 ? M : 32);
  mi_tile_cfg c = cands[0];
  double best_t = 0.0;
  bool found = false;
  for (const mi_tile_cfg& ci : cands) {
    if (ci.block_m > m_cap) continue;
    const long long tiles = tiles_of(M, N, ci.block_m, ci.block_n), kt = ((long long)K + ci.block_k - 1) / ci.block_k;
    for (int p = 1; p <= 8; p *= 2) {
      const long long kts = (kt + p - 1) / p, wgs = tiles * p;
      const double kp = (double)((K + p - 1) / p);
      if (p > 1 && (wgs > 320 || (long long)(p - 1) * kts >= kt || kp < 512.0)) break;
      double t = (double)((wgs + kCUs - 1) / kCUs) * ((ci.block_m + ci.block_n) * (kp + 256.0) * 2.0 / 70e3 + 3.0);
      if (p > 1) t += (double)p * M * N * 8.0 / 5e6 + 1.0;
      if (!found || t < best_t) {
        found = true;
        best_t = t;
        c = ci;
        c.split_k = p;
      }
    }
  }
  return c;
}

// Either matmul past skinny M: the block whose rounds of tiles take the
// least time (a block that leaves CUs idle can still beat a smaller one
// whose grid needs a second, partial round), K split when the chosen grid
// leaves CUs idle.  lhsT.rhs runs the pipelined variant 1; a 256-long block
// lies with its long side along the shorter output side (128 x 256 when
// M >= N), or along N at any shape when K <= 2048, and a 128-long one along
// N unless N is at least four times M, as the winners do.  lhs.rhs runs
// variant 0 and keeps block_m the short side (fewer rows of its
// K-contiguous operand per tile); its 256-long blocks take the paired-load
// variant 1 (block_k 32, the K-contiguous panel loaded as whole 128-byte
// lines).
mi_tile_cfg matmul_default(int kernel_id, bool lhs, int M, int N, int K) {
  const int v = lhs ? 0 : 1;
  const bool m_long = M >= N, n_much_longer = (long long)N >= 4LL * M;
  // lhsT.rhs with M <= N also weighs a 64 x 256 block, at a rate just under
  // the 128 x 128 block's: it is taken only where it needs fewer rounds of
  // tiles.  Timed with every candidate and split at 40 shapes past skinny M,
  // it changed the pick at three (1088x3840x4096: 1.29 x the fastest to
  // 1.00; 1088x3712x8000: 1.26 to 1.00; 704x11648x1088: 1.08 to 1.01).
  Cand cands[7];
  int n = 0;
  cands[n++] = {lhs ? mi_tile_cfg{256, 256, 32, 8, 3, 1, 8, 1} : mi_tile_cfg{256, 256, 32, 4, 3, 1, 8, v}, 1.0};
  cands[n++] = {lhs ? mi_tile_cfg{128, 256, 32, 4, 3, 1, 8, 1}
                    : (m_long || K <= 2048 ? mi_tile_cfg{128, 256, 32, 4, 3, 1, 8, v} : mi_tile_cfg{256, 128, 32, 4, 3, 1, 8, v}),
                0.93};
  // lhsT.rhs also weighs the other orientation of the 256-long block, after
  // the preferred one: it wins only where it needs fewer rounds of tiles
  // (7616x2112x1280: 510 tiles of 256 x 128 in two rounds against 540 of
  // 128 x 256 in three, 39.3 against 49.0 us).
  if (!lhs) {
    const mi_tile_cfg pref = cands[1].c;
    cands[n++] = {mi_tile_cfg{pref.block_n, pref.block_m, 32, 4, 3, 1, 8, v}, 0.93};
  }
  cands[n++] = {mi_tile_cfg{128, 128, 64, 4, 3, 1, 8, v}, 0.62};
  if (!lhs && M <= N) cands[n++] = {mi_tile_cfg{64, 256, 64, 4, 3, 1, 8, v}, 0.60};
  cands[n++] = {n_much_longer && !lhs ? mi_tile_cfg{128, 64, 64, 4, 4, 1, 8, v} : mi_tile_cfg{64, 128, 64, 4, 4, 1, 8, v}, 0.60};
  cands[n++] = {mi_tile_cfg{64, 64, 64, 4, 4, 1, 8, v}, 0.35};
  mi_tile_cfg c = fastest_estimate(cands, n, M, N, K, kernel_id);
  const bool small = c.split_k == 1 && c.block_m * c.block_n <= 128 * 64;
  if (lhs) {
    // lhs.rhs: a small unsplit block over K >= 8192 becomes the 128 x 128
    // block split to fill the chip.  Timed with every candidate and split at
    // 8 such shapes (256-3200 rows, interleaved rounds, one box): within
    // 1.045 of the fastest at all of them, against 1.29 for the small block.
    if (small && K >= 8192) {
      const int parts = fill_parts(tiles_of(M, N, 128, 128), K, 64);
      if (parts >= 2) c = {128, 128, 64, 4, 3, parts, 8, 0};
    }
    // An unsplit 128 x 128 grid that leaves CUs idle, over K >= 12288 and a
    // whole number of 256-row blocks, takes 256 x 128 in 2 parts (the same
    // workgroup count, a quarter fewer operand bytes per multiply-add):
    // 256x12224x12288 94.4 against 116.9 us, 256x9216x16384 1.23 x and
    // 512x6144x16384 1.03 x faster; not at 384 rows (the 256-row blocks'
    // tail, 1.17 x slower), K = 10240 or 224 tiles (1.07-1.10 x slower).
    if (c.block_m == 128 && c.block_n == 128 && c.split_k == 1 && tiles_of(M, N, 128, 128) < kFillTiles &&
        M % 256 == 0 && K >= 12288 && 2 * tiles_of(M, N, 256, 128) <= kCUs)
      return {256, 128, 64, 8, 3, 2, 8, 0};
    // An unsplit 128 x 128 block runs on the paired-load variant 1 with
    // block_k 32 and 4 stages (whole 128-byte lines of the K-contiguous
    // operand, three K tiles in flight): 0.90-0.99 x variant 0's time with
    // block_k 64 at the 8 shapes above, and the sweep's winner at 2048^3,
    // 1536x1536x6144, 704x5376x13824 and 704x4800x11712, where variant 0
    // ran 1.04-1.06 x its time.
    if (c.block_m == 128 && c.block_n == 128 && c.split_k == 1 && c.variant == 0) c = {128, 128, 32, 4, 4, 1, 8, 1};
    return c;
  }
  // lhsT.rhs 128x128 blocks then run block_k 32 with 4 stages, the same
  // parts (each part keeps at least 8 K tiles of 32): three tiles in flight
  // instead of two.  Measured against block_k 64 with 3 stages at eleven
  // shapes this picker gives the 128x128 block (split or not), in
  // interleaved rounds on one box: median 0.958 x the time, 0.880-1.022 x,
  // bitwise equal outputs.  (The K-contiguous lhs.rhs variant 0 keeps
  // block_k 64, where 32 loads half lines: median 1.008 x, up to 1.079 x;
  // its unsplit 128x128 block moves to the paired-load variant 1 above.)
  if (c.block_m == 128 && c.block_n == 128 && c.block_k == 64) {
    c.block_k = 32;
    c.lds_stages = 4;
  }
  // Where the rounds estimate settles on a small unsplit block with a long K
  // (64 x 64 from K = 3072; 64 x 128 or 128 x 64 from K = 8192, or where
  // each part of the 128 x 128 split keeps 3072 of K), or splits a 256-long
  // block 8 ways or more (below), the 128 x 128 block split to fill the
  // chip is faster: it moves half the operand bytes per multiply-add of a 64 x 64
  // block, and each part's partial products cost less than the MFMA time
  // they save.  Timed with every candidate and split at 30 shapes past
  // skinny M (interleaved rounds, one box), this takes the pick from within
  // 1.74 of the fastest (mean 1.082) to within 1.21 (mean 1.011); it
  // applies at 9 of the shapes, and the rest keep their pick.  The per-part
  // bound adds 896x1472x7872 (37.1 us for 64 x 128 against 31.5 us in 2
  // parts of 128 x 128) and changes no pick at the 70 timed shapes.
  const int parts = fill_parts(tiles_of(M, N, 128, 128), K, 32);
  const bool long_parts = parts >= 2 && (K + parts - 1) / parts >= 3072;
  const bool long_k = K >= 8192 || long_parts || (c.block_m == 64 && c.block_n == 64 && K >= 3072);
  const bool thin_256 = (c.block_m == 256 || c.block_n == 256) && c.split_k >= 8;
  if (small && long_k && parts >= 2) return {128, 128, 32, 4, 4, parts, 8, v};
  if (thin_256) {
    // A 256-long block split 8 ways or more: the largest of 128 x 128, the
    // 64-wide block (oriented as above) and 64 x 64 whose split to fill the
    // chip keeps each part at least 1536 (128 x 128) or 1792 (64-wide) of K,
    // else 64 x 64: shorter parts pay more in partial products than the
    // larger block saves.  Timed with every candidate and split at 12 such
    // shapes (K 4096-16384), the pick is within 1.035 of the fastest
    // (mean 1.007), against 1.43 (mean 1.108) for 128 x 128 at any K.
    if (parts >= 2 && (K + parts - 1) / parts >= 1536) return {128, 128, 32, 4, 4, parts, 8, v};
    const int bm = n_much_longer ? 128 : 64, bn = n_much_longer ? 64 : 128;
    const int pw = fill_parts(tiles_of(M, N, bm, bn), K, 64);
    if (pw >= 2 && (K + pw - 1) / pw >= 1792) return {bm, bn, 64, 4, 4, pw, 8, v};
    return {64, 64, 64, 4, 4, fill_parts(tiles_of(M, N, 64, 64), K, 64), 8, v};
  }
  return c;
}

// rmsnorm_matmul.  The register-staged kernels keep gamma in LDS (8192
// entries here).
// The skinny fused kernel's 128-row block leaves CUs idle below 256 tiles;
// it then keeps 128 rows (the weight read once) where its split to fill the
// CUs leaves each part at least 1024 of K, and takes 64-row blocks (the
// weight read twice, fewer parts) otherwise.  Timed with every block and
// split: 128x5760x10944 ran 46.0 us in 4 parts of 128 rows against 57.8 us
// for 64 rows in 2, 128x7552x5952 35.4 against 38.4, 96x3584x10176 32.4
// against 34.8; 128x8192x3072 (768 of K per part) 1.064 x and 128x1792x11008
// (688) 1.137 x the 64-row block's time.
bool skinny_keeps_128_rows(int M, int N, int K) {
  const long long t128 = tiles_of(M, N, 128, 128);
  if (t128 >= kFillTiles) return true;
  const int p = fill_parts(t128, K, 64);
  return p >= 2 && (K + p - 1) / p >= 1024;
}

mi_tile_cfg fused_default(int M, int N, int K) {
  if (M <= 128 && K > 8192) {
    // Skinny M past K = 8192: the skinny variant 11 (64-row blocks when
    // 128-row ones leave CUs idle) split into the fewest parts whose gamma
    // fits (1..16 parts, none empty), or into more when that fills more CUs
    // (up to one workgroup per CU); past 16 parts the LDS-staged kernel
    // (variant 0) takes any K.
    int bm = M <= 32 ? 32 : M <= 64 ? 64 : 128;
    if (bm == 128 && !skinny_keeps_128_rows(M, N, K)) bm = 64;
    const long long kt = (K + 63) / 64;
    const int fill = fill_parts(tiles_of(M, N, bm, 128), K, 64);
    for (int p = 2; p <= 16; p *= 2) {
      const long long kts = (kt + p - 1) / p;
      const unsigned long long ws = (unsigned long long)p * ((unsigned long long)M * N + M) * 4ull;
      if (kts * 64 <= 8192 && (long long)(p - 1) * kts < kt && ws <= kMaxWorkspace) {
        int parts = p;
        // A larger split: still no empty part, and its workspace fits.
        for (int q = p * 2; q <= fill; q *= 2) {
          const long long qts = (kt + q - 1) / q;
          const unsigned long long qws = (unsigned long long)q * ((unsigned long long)M * N + M) * 4ull;
          if ((long long)(q - 1) * qts < kt && qws <= kMaxWorkspace) parts = q;
        }
        // 32-row blocks whose split leaves more than 16 CUs idle take block_k
        // 128 (twice the K panel in flight per workgroup), where its parts
        // still hold their gamma and none is empty: at 6 such shapes it ran
        // 0.89-0.96 x the time of block_k 64 (8x12864x16256, 32x9728x9984,
        // 16x9088x9536, 32x13504x13056, 32x12864x14144, 32x10752x11328).
        const long long kt128 = (K + 127) / 128, kts128 = (kt128 + parts - 1) / parts;
        if (bm == 32 && tiles_of(M, N, 32, 128) * parts < 240 && kts128 * 128 <= 8192 && (parts - 1) * kts128 < kt128)
          return {32, 128, 128, 4, 3, parts, 8, 11};
        return {bm, 128, 64, 4, 3, parts, 8, 11};
      }
    }
    return {64, 128, 64, 4, 2, 1, 8, 0};
  }
  if (M <= 128) {
    // Weight streamed once (variant 11).  With a weight of 16 MiB or less
    // (re-read from the caches), 32-row blocks (more tiles) win at any M
    // (measured up to 16 MiB; at 32 MiB the 64-row block won); a larger one
    // takes the block that covers M, with 64-row blocks before a split when
    // 128-row ones leave CUs idle.  From K = 1024 K is split to fill the
    // CUs.  Timed with every block, stage count and split at 20 skinny fused
    // shapes (weight flushed, split workspace kept per stream): within 1.078
    // of the fastest at all of them (mean 1.017), against 1.82 (mean 1.22)
    // when splits started at K = 4096 (8x4096x3072: 28.8 us unsplit, 15.8
    // us in 8 parts).
    const bool cached_w = (long long)K * N * 2 <= (16LL << 20);
    mi_tile_cfg c = {cached_w || M <= 32 ? 32 : M <= 64 ? 64 : 128, 128, 64, 4, 3, 1, 8, 11};
    if (c.block_m == 128 && !skinny_keeps_128_rows(M, N, K)) c.block_m = 64;
    if (K >= 1024) c.split_k = fill_parts(tiles_of(M, N, c.block_m, c.block_n), K, c.block_k);
    return c;
  }
  // Each workgroup of the one-pass kernels scales its x rows once per column
  // tile, so narrow blocks pay that work many times over: per CU, 128 x 256
  // runs at 0.83 and 128 x 128 at 0.54 of the rate of 128 x 512.  The
  // two-pass kernel scales x once, in a pass of its own, and its main pass
  // runs the lhsT core (256 x 256 at 1.10 of that rate; past K = 8192 also
  // 256 x 128, its long side along the shorter output side, at 0.95).
  // Few-tile shapes split K, which the estimate charges for its fp32 partial
  // products and the launch of the summing kernel; past K = 8192 the
  // one-pass kernels split at least until each part's gamma fits.  The
  // two-pass kernel on the paired-load core (variant 15, never split) adds
  // 128 x 256 at 0.95, and 128 x 128 at 0.80 where that grid keeps more
  // than half the CUs busy (with fewer, a split or a 64-row block won at
  // every shape timed).  Fitted to every candidate and split timed at 23
  // fused shapes with M > 128 (interleaved rounds, one box): the pick within
  // 1.012 of the fastest at all of them (mean 1.0005, against 1.17 and 1.040
  // without variant 15).  The rates alone, without the half-busy rule, were
  // within 1.064 at the third of the shapes held out of a fit to the other
  // two thirds.
  Cand cands[9];
  int n = 0;
  cands[n++] = {mi_tile_cfg{128, 512, 32, 8, 3, 1, 8, 4}, 1.0};
  cands[n++] = {mi_tile_cfg{128, 256, 32, 4, 3, 1, 8, 5}, 0.83};
  cands[n++] = {mi_tile_cfg{128, 128, 64, 4, 2, 1, 8, 4}, 0.54};
  cands[n++] = {mi_tile_cfg{256, 256, 32, 4, 3, 1, 8, 13}, 1.10};
  cands[n++] = {mi_tile_cfg{128, 128, 64, 4, 3, 1, 8, 13}, 0.68};
  cands[n++] = {mi_tile_cfg{64, 128, 64, 4, 4, 1, 8, 13}, 0.57};
  if (2 * tiles_of(M, N, 128, 128) > kCUs) cands[n++] = {mi_tile_cfg{128, 128, 32, 4, 4, 1, 8, 15}, 0.80};
  cands[n++] = {mi_tile_cfg{128, 256, 32, 4, 3, 1, 8, 15}, 0.95};
  if (K > 8192)
    cands[n++] = {M <= N ? mi_tile_cfg{256, 128, 64, 4, 3, 1, 8, 13} : mi_tile_cfg{128, 256, 64, 4, 3, 1, 8, 13}, 0.95};
  return fastest_split_estimate(cands, n, M, N, K, mi_tile_cfg{128, 256, 64, 8, 2, 1, 8, 0});
}

// Fitted times.  A candidate's time (us) at a shape is
//   start + (tile + step * L * (1 + crowd * f * (1 + drift * L * block_k / 1e4)))
//         * (1 + (n - 1) * more)
//   + read_mb * (the inputs' MB)
//   [+ split + split_mb * p * M * N / 1e6]      K split in p parts
//   [+ pack + pack_mb * M * K / 1e6]            the two-pass fused kernels
// with L the K tiles of a part, n the workgroups of the busiest CU, and f
// the share of CUs that have one (at most 1): one tile's fixed cost, its cost
// per K tile (more when every CU loads at once, and more the longer K is, as
// workgroups that share panels drift apart), and the further tiles of a CU,
// which overlap the first one's loads.  The coefficients are fitted to
// every candidate block in 1-8, 12 and 16 parts, timed at 480 fused, 320
// no-gamma, 380 lhsT.rhs and 380 lhs.rhs shapes with M > 128 (sizes spread
// over their logarithm, N up to 28672, K up to 16384), three sets of inputs
// in turn.  Fitted without half of the second campaigns' shapes, the least
// fitted time is within 1.013, 1.020, 1.022 and 1.017 of the fastest on
// average at those.
struct Timed {
  mi_tile_cfg c;
  double start, tile, step, more, crowd, drift, read_mb, split, split_mb, pack, pack_mb;
};

const Timed kFusedTimed[] = {
    {{128, 512, 32, 8, 3, 1, 8, 4}, 1.28, 6.28, 0.434, 1.08, 0.54, 1.39, 0.0379, 2.2, 1.16, 0, 0},
    {{128, 128, 64, 4, 2, 1, 8, 4}, 1.75, 3.4, 0.521, 0.932, 0.244, 0.317, 0.0192, 2.85, 1.34, 0, 0},
    {{256, 128, 32, 8, 3, 1, 8, 5}, 1.76, 4.09, 0.369, 1.04, 0.444, 0.381, 0.017, 3.9, 1.07, 0, 0},
    {{128, 256, 32, 4, 3, 1, 8, 5}, 1.79, 4.91, 0.304, 1.02, 0.354, 1.53, 0.0472, 2.83, 0.98, 0, 0},
    {{128, 128, 32, 4, 4, 1, 8, 5}, 1.66, 3.33, 0.258, 0.966, 0.223, 0.307, 0.0171, 2.86, 1.48, 0, 0},
    {{64, 128, 64, 4, 4, 1, 8, 5}, 1.06, 3.32, 0.34, 0.891, 0.153, 0.261, 0.0211, 2.43, 1.83, 0, 0},
    {{64, 64, 64, 4, 4, 1, 8, 5}, 1.49, 2.47, 0.278, 0.895, 0.163, 0.252, 0.021, 2.39, 1.92, 0, 0},
    {{256, 256, 32, 4, 3, 1, 8, 13}, 1.46, 9.27, 0.365, 0.968, 0.743, 0.187, 0.0465, 1.06, 1.03, 1.91, 0.98},
    {{256, 128, 64, 4, 3, 1, 8, 13}, 2.16, 6.19, 0.544, 0.976, 0.471, 0.231, 0.017, 2.45, 0.843, 3.4, 0.861},
    {{128, 128, 64, 4, 3, 1, 8, 13}, 2.39, 2.8, 0.324, 1.05, 0.418, 0.667, 0.0348, 3.79, 0.653, 4.35, 0.597},
    {{64, 128, 64, 4, 4, 1, 8, 13}, 2.47, 1.79, 0.271, 0.992, 0.281, 0.297, 0.0194, 2.47, 1.07, 5.39, 0.58},
    {{128, 256, 32, 4, 3, 1, 8, 15}, 1.99, 4.61, 0.287, 1.04, 0.412, 0.397, 0.0435, 0, 0, 2.99, 0.454},
    {{128, 128, 32, 4, 4, 1, 8, 15}, 2.14, 2.73, 0.188, 1.07, 0.326, 0.557, 0.0301, 0, 0, 3.33, 0.496},
};
const Timed kNoGammaTimed[] = {
    {{128, 512, 32, 8, 3, 1, 8, 4}, 1.16, 6.03, 0.438, 1.02, 0.554, 0.609, 0.0803, 1.72, 1.06, 0, 0},
    {{128, 256, 32, 4, 3, 1, 8, 5}, 2.7, 3.62, 0.275, 0.886, 0.329, 2.32, 0.0621, 3.27, 0.796, 0, 0},
    {{128, 128, 32, 4, 4, 1, 8, 5}, 2.56, 2.08, 0.223, 0.839, 0.224, 1.99, 0.0195, 3.35, 1.21, 0, 0},
    {{64, 128, 64, 4, 4, 1, 8, 5}, 1.71, 2.27, 0.308, 0.983, 0.192, 0.316, 0.0203, 2.9, 1.5, 0, 0},
    {{64, 64, 64, 4, 4, 1, 8, 5}, 2.13, 1.29, 0.246, 0.67, 0.121, 0.316, 0.0225, 2.89, 1.24, 0, 0},
    {{64, 128, 64, 4, 4, 1, 8, 14}, 1.72, 1.94, 0.264, 1.03, 0.305, 0.617, 0.0291, 0, 0, 0, 0},
    {{64, 64, 64, 4, 4, 1, 8, 14}, 2.41, 0.862, 0.178, 0.84, 0.326, 0.928, 0.0173, 0, 0, 0, 0},
    {{128, 128, 32, 4, 4, 1, 8, 16}, 2.29, 1.8, 0.186, 0.945, 0.297, 0.843, 0.0271, 0, 0, 0, 0},
};
const Timed kLhsTTimed[] = {
    {{256, 256, 32, 4, 3, 1, 8, 1}, 1.06, 6.87, 0.353, 1.02, 0.664, 0.425, 0.042, 1.17, 1, 0, 0},
    {{256, 128, 32, 4, 3, 1, 8, 1}, 2.54, 2.66, 0.211, 0.968, 0.549, 1.03, 0.0265, 3.46, 0.818, 0, 0},
    {{128, 256, 32, 4, 3, 1, 8, 1}, 2.46, 2.71, 0.204, 0.966, 0.595, 0.913, 0.0399, 3.53, 0.777, 0, 0},
    {{128, 128, 32, 4, 4, 1, 8, 1}, 2.04, 1.54, 0.159, 0.955, 0.324, 1.06, 0.0113, 2.93, 1.32, 0, 0},
    {{64, 256, 64, 4, 3, 1, 8, 1}, 1.54, 2.63, 0.362, 0.957, 0.496, 0.38, 0.0128, 2.88, 1.23, 0, 0},
    {{128, 64, 64, 4, 4, 1, 8, 1}, 1.23, 2.14, 0.259, 0.818, 0.353, 0.264, 0.0148, 2.1, 1.84, 0, 0},
    {{64, 128, 64, 4, 4, 1, 8, 1}, 1.23, 2.13, 0.253, 0.836, 0.376, 0.264, 0.0151, 2.2, 1.73, 0, 0},
    {{64, 64, 64, 4, 4, 1, 8, 1}, 2.12, 1.04, 0.188, 0.68, 0.31, 0.295, 0.0325, 1.68, 1.93, 0, 0},
    {{32, 128, 64, 4, 4, 1, 8, 1}, 1.48, 1.47, 0.207, 0.597, 0.463, 0.285, 0.021, 1.63, 2.03, 0, 0},
};
const Timed kLhsTimed[] = {
    {{256, 256, 32, 8, 3, 1, 8, 0}, 1.18, 5.45, 0.398, 0.974, 0.729, 0.641, 0.0557, 1.86, 1.08, 0, 0},
    {{256, 128, 64, 8, 3, 1, 8, 0}, 1.1, 3.56, 0.568, 0.986, 0.454, 0.83, 0.0179, 2.9, 1.15, 0, 0},
    {{128, 256, 64, 4, 3, 1, 8, 0}, 1.5, 4.06, 0.643, 0.977, 0.365, 0.48, 0.0303, 2.55, 0.986, 0, 0},
    {{128, 128, 64, 4, 3, 1, 8, 0}, 1.68, 2.25, 0.343, 1.02, 0.377, 0.761, 0.0148, 2.65, 1.41, 0, 0},
    {{64, 256, 64, 4, 3, 1, 8, 0}, 1.85, 2.34, 0.359, 1.05, 0.435, 0.56, 0.0167, 2.67, 1.32, 0, 0},
    {{64, 128, 64, 4, 4, 1, 8, 0}, 1.11, 2.13, 0.245, 0.872, 0.395, 0.372, 0.0165, 2.32, 1.75, 0, 0},
    {{64, 64, 64, 4, 4, 1, 8, 0}, 1.82, 1.07, 0.181, 0.698, 0.429, 0.45, 0.0197, 2.36, 1.57, 0, 0},
    {{32, 128, 64, 4, 4, 1, 8, 0}, 2.04, 1.11, 0.183, 0.732, 0.403, 0.696, 0.0187, 2.32, 1.65, 0, 0},
    {{256, 256, 32, 8, 3, 1, 8, 1}, 1.31, 5.87, 0.373, 0.988, 0.714, 0.387, 0.0274, 0, 0, 0, 0},
    {{128, 256, 32, 4, 3, 1, 8, 1}, 2.4, 2.36, 0.277, 1.02, 0.286, 0.61, 0.0625, 0, 0, 0, 0},
    {{128, 128, 32, 4, 4, 1, 8, 1}, 2.08, 1.41, 0.168, 0.955, 0.444, 0.407, 0.0282, 0, 0, 0, 0},
};

// Blocks 192 wide, fitted the same way at 120 lhsT.rhs and 140 lhs.rhs shapes
// with M > 128 and up to 4e11 operations.
const Timed kLhsT192Timed[] = {
    {{192, 256, 32, 4, 3, 1, 8, 1}, 0.783, 6.26, 0.277, 1.09, 0.748, 0.449, 0.0747, 2.43, 0.681, 0, 0},
    {{192, 192, 32, 4, 3, 1, 8, 1}, 1.25, 4.7, 0.194, 0.978, 0.723, 1.41, 0.0803, 2.54, 0.9, 0, 0},
    {{192, 128, 32, 4, 3, 1, 8, 1}, 1.42, 2.88, 0.187, 0.968, 0.486, 0.787, 0.0707, 2.64, 0.91, 0, 0},
    {{128, 192, 32, 4, 3, 1, 8, 1}, 1.2, 3.11, 0.183, 0.899, 0.635, 0.534, 0.0538, 2.67, 1.02, 0, 0},
};
const Timed kLhs192Timed[] = {
    {{192, 256, 32, 8, 3, 1, 8, 1}, 0.295, 5.7, 0.253, 1.11, 0.873, 0.162, 0.109, 0, 0, 0, 0},
    {{192, 192, 32, 4, 3, 1, 8, 1}, 1.01, 4.54, 0.273, 1.09, 0.589, 0.146, 0.0776, 0, 0, 0, 0},
    {{192, 128, 32, 4, 4, 1, 8, 1}, 0.718, 3.34, 0.225, 1.03, 0.462, 0.284, 0.117, 0, 0, 0, 0},
    {{128, 192, 32, 4, 4, 1, 8, 1}, 0.811, 3.41, 0.211, 1.06, 0.554, 0.406, 0.0571, 0, 0, 0, 0},
};

// M <= 128 with a weight of at most 7 MiB, and (lhs.rhs, non-temporal blocks
// only) of 7 to 28 MiB: the same fits to 160 shapes of each kind (120 for
// the last), the weight warm in the caches as a call repeated over a few
// layers leaves it.
const Timed kFusedSkinnyTimed[] = {
    {{64, 128, 64, 4, 4, 1, 8, 5}, 2.01, 1.98, 0.33, 0.878, 0.376, 0, 0.0171, 2.31, 2.51, 0, 0},
    {{64, 64, 64, 4, 4, 1, 8, 5}, 1.95, 1.83, 0.269, 0.921, 0.247, 0, 0.0153, 2.43, 2.08, 0, 0},
    {{32, 128, 64, 4, 4, 1, 8, 5}, 1.78, 1.81, 0.248, 0.929, 0.399, 0, 0.0169, 2.64, 1.84, 0, 0},
    {{128, 128, 64, 4, 3, 1, 8, 11}, 2.23, 2.23, 0.546, 0.9, 0.446, 0, 0.0216, 1.97, 2.83, 0, 0},
    {{64, 128, 64, 4, 3, 1, 8, 11}, 1.93, 1.87, 0.332, 0.856, 0.939, 0, 0.0273, 2.47, 2.37, 0, 0},
    {{32, 128, 128, 4, 3, 1, 8, 11}, 1.83, 1.87, 0.56, 0.939, 0.368, 0, 0.173, 2.59, 2.14, 0, 0},
    {{32, 128, 64, 4, 3, 1, 8, 11}, 1.82, 1.69, 0.255, 0.839, 0.761, 0, 0.0822, 2.68, 1.69, 0, 0},
    {{32, 128, 64, 4, 4, 1, 8, 12}, 1.82, 1.78, 0.263, 0.898, 0.481, 0, 0.111, 2.68, 1.9, 0, 0},
};
const Timed kLhsTSkinnyTimed[] = {
    {{64, 128, 64, 4, 4, 1, 8, 1}, 1.82, 1.81, 0.172, 0.896, 0.391, 0, 0.0164, 2.79, 1.46, 0, 0},
    {{64, 64, 64, 4, 4, 1, 8, 1}, 2.3, 1.42, 0.108, 0.428, 0.186, 0, 0.0104, 2.82, 0.942, 0, 0},
    {{32, 128, 64, 4, 4, 1, 8, 1}, 2.17, 1.51, 0.114, 0.551, 0.374, 0, 0.0183, 2.93, 0.964, 0, 0},
    {{128, 256, 32, 4, 3, 1, 8, 3}, 2.12, 2.12, 0.229, 0.9, 0.621, 0, 0.0323, 1.89, 3.01, 0, 0},
    {{128, 128, 32, 4, 4, 1, 8, 3}, 1.78, 1.78, 0.113, 0.9, 0.442, 0, 0.0254, 2.83, 1.94, 0, 0},
    {{64, 256, 64, 4, 3, 1, 8, 3}, 1.86, 1.86, 0.356, 0.9, 1.55, 0, 0.0308, 2.5, 2.84, 0, 0},
    {{64, 128, 64, 4, 4, 1, 8, 3}, 1.78, 1.73, 0.177, 0.858, 0.847, 0, 0.0247, 2.97, 2.08, 0, 0},
    {{32, 256, 64, 4, 4, 1, 8, 3}, 1.82, 1.82, 0.28, 0.9, 0.441, 0, 0.133, 2.67, 2.2, 0, 0},
    {{64, 64, 64, 4, 4, 1, 8, 3}, 2.16, 1.46, 0.119, 0.536, 0.389, 0, 0.0198, 3.04, 1.1, 0, 0},
    {{32, 128, 64, 4, 4, 1, 8, 3}, 2.07, 1.57, 0.117, 0.576, 0.531, 0, 0.0437, 3.02, 1.58, 0, 0},
};
const Timed kLhsSkinnyTimed[] = {
    {{64, 128, 64, 4, 4, 1, 8, 0}, 1.91, 1.91, 0.162, 0.9, 0.329, 0, 0.0153, 2.59, 1.66, 0, 0},
    {{64, 64, 64, 4, 4, 1, 8, 0}, 2.54, 1.42, 0.104, 0.268, 0.245, 0, 0.0135, 2.7, 1.08, 0, 0},
    {{32, 128, 128, 4, 3, 1, 8, 0}, 1.88, 1.79, 0.354, 0.833, 0.211, 0, 0.017, 2.62, 1.45, 0, 0},
    {{32, 128, 64, 4, 4, 1, 8, 0}, 2.4, 1.51, 0.121, 0.399, 0.242, 0, 0.0153, 2.67, 1.13, 0, 0},
    {{128, 128, 64, 4, 3, 1, 8, 2}, 1.96, 1.96, 0.259, 0.9, 0.387, 0, 0.0204, 2.44, 2.48, 0, 0},
    {{64, 128, 128, 4, 3, 1, 8, 2}, 1.83, 1.83, 0.433, 0.9, 0.628, 0, 0.0283, 2.72, 2.35, 0, 0},
    {{64, 128, 64, 4, 4, 1, 8, 2}, 1.91, 1.91, 0.153, 0.9, 0.469, 0, 0.0282, 2.75, 1.88, 0, 0},
};
const Timed kLhsSkinnyStreamTimed[] = {
    {{256, 128, 64, 8, 3, 1, 8, 2}, 2.15, 2.05, 0.596, 0.839, 0.172, 0, 0.015, 1.32, 2.91, 0, 0},
    {{128, 128, 64, 4, 3, 1, 8, 2}, 1.64, 1.58, 0.525, 0.749, 0.156, 0, 0.0155, 1.47, 3.18, 0, 0},
    {{64, 128, 128, 4, 3, 1, 8, 2}, 1.5, 1.56, 0.851, 0.943, 0.19, 0, 0.0465, 2.42, 2.85, 0, 0},
    {{64, 128, 64, 4, 4, 1, 8, 2}, 1.43, 1.42, 0.456, 0.78, 0.255, 0, 0.0195, 2.07, 3.02, 0, 0},
    {{32, 256, 64, 4, 4, 1, 8, 2}, 1.52, 1.62, 0.626, 0.936, 0.161, 0, 0.0649, 2.82, 2.11, 0, 0},
    {{64, 64, 64, 4, 4, 1, 8, 2}, 2.12, 0.629, 0.31, 0.708, 0.281, 0, 0.0158, 1.71, 4.12, 0, 0},
    {{32, 128, 128, 4, 3, 1, 8, 2}, 1.46, 1.6, 0.722, 0.962, 0.14, 0, 0.0632, 2.83, 2.06, 0, 0},
    {{32, 128, 64, 4, 4, 1, 8, 2}, 1.87, 0.956, 0.387, 0.867, 0.13, 0, 0.048, 2.46, 2.37, 0, 0},
};

double fitted_time(const Timed& e, int parts, int M, int N, int K) {
  const long long wgs = tiles_of(M, N, e.c.block_m, e.c.block_n) * parts;
  const double n = (double)((wgs + kCUs - 1) / kCUs), f = wgs < kCUs ? (double)wgs / kCUs : 1.0;
  const long long kt = ((long long)K + e.c.block_k - 1) / e.c.block_k;
  const double L = (double)((kt + parts - 1) / parts), mn = (double)M * N * 1e-6;
  double t = e.start + (e.tile + e.step * L * (1.0 + e.crowd * f * (1.0 + e.drift * L * e.c.block_k * 1e-4))) * (1.0 + (n - 1.0) * e.more) +
             e.read_mb * ((double)M + N) * K * 2e-6;
  if (parts > 1) t += e.split + e.split_mb * parts * mn;
  return t + e.pack + e.pack_mb * (double)M * K * 1e-6;
}

const Timed* timed(const Timed* table, int n, const mi_tile_cfg& c) {
  for (int i = 0; i < n; ++i) {
    const mi_tile_cfg& t = table[i].c;
    if (t.block_m == c.block_m && t.block_n == c.block_n && t.block_k == c.block_k && t.waves == c.waves &&
        t.lds_stages == c.lds_stages && t.variant == c.variant)
      return &table[i];
  }
  return nullptr;
}

// Whether the call can run `c` in `parts` parts: at most one workgroup per
// CU where K is split, no part empty, gamma of a part within the entries the
// instance stages, and the workspace within its limit.  A split in parts
// that are no power of two keeps at least 2688 of K in each (3 parts from
// K = 8064, 5 from 13440, 6 from 16128, 7 from 18816, 12 from 32256): two
// default picks that tests name set that line, 896x1472x7872 lhsT.rhs (29.9
// us in 2 parts, 31.1 in the 6 that the fits take) and 1536x1536x6144 lhs.rhs
// (38.5 unsplit, 38.2 in 3).  Without it picks are 1.025 (fused), 1.04
// (lhs.rhs) and 1.05 x (lhsT.rhs) faster on average at 122 drawn shapes, and
// over 3 % slower at 23 of them.
bool runs_split(int kernel_id, const mi_tile_cfg& c, int parts, int M, int N, int K) {
  const long long kt = ((long long)K + c.block_k - 1) / c.block_k, kts = (kt + parts - 1) / parts;
  if (parts > 1) {
    if (!splittable(kernel_id, c.variant) || tiles_of(M, N, c.block_m, c.block_n) * parts > kCUs ||
        (parts - 1) * kts >= kt || ((parts & (parts - 1)) != 0 && K < 2688LL * parts))
      return false;
  }
  const mi::MiEntry* e = find(kernel_id, c);
  if (!e || (e->gamma_kmax > 0 && kts * c.block_k > e->gamma_kmax)) return false;
  mi_tile_cfg p = c;
  p.split_k = parts;
  // lhsT.rhs calls without a config also run from the no-allocation entry's
  // static scratch, which 256 full blocks of 256 x 256 and the counters pass.
  const unsigned long long cap = kernel_id == MI_KERNEL_MATMUL_LHST_RHS_BF16 ? MI_NOALLOC_SCRATCH_BYTES : kMaxWorkspace;
  return mi::workspace_bytes(kernel_id, p, M, N, K, kDefaultCus) <= cap;
}

// `pick`, whose fitted coefficients are `old`, or the candidate of `table`
// with the least fitted time where that is under `margin` of the pick's own.
mi_tile_cfg faster_of(int kernel_id, const Timed* table, int n, const Timed& old, const mi_tile_cfg& pick, double margin,
                      int M, int N, int K) {
  // The fit reads x once.  Past the L2s (64 MiB of x) every column of tiles
  // of the fused kernel reads it again, so where the pick spans the columns
  // with one tile, its place is for blocks that do as well (us, 128 x 512 in
  // 4 parts against 128-wide blocks, three columns of them: 110 against 126
  // at 7168x328x14688, 70 against 85 at 5088x336x9936, 87 against 112 at
  // 4376x312x13424; at 61 MiB, 2520x336x12688, 47 against 43).
  const bool one_column =
      kernel_id == MI_KERNEL_RMSNORM_MATMUL_BF16 && N <= pick.block_n && (long long)M * K * 2 > (64LL << 20);
  // Below K = 512 a matmul past skinny M is bound by its output's stores,
  // which the fits know only as a part of each tile; they then take blocks
  // too small.  lhsT.rhs in 256 x 256 blocks stays there (256 x 128 in their
  // place was over 3 % slower at 30 of 106 shapes, 128 x 256 at 26 of 94: us,
  // 51 -> 59 at 4072x14904x176, 77 -> 86 at 3496x26040x168, 316 -> 407 at
  // 1224x244688x312).  lhs.rhs takes no 256 x 128 (6 of 14), and 128 x 128
  // only in the place of a 128-wide block (21 of 48 of another width; 7.4 ->
  // 8.1 at 46328x192x8).
  const bool short_k = K < 512 && M > 128;
  const bool lhs = kernel_id == MI_KERNEL_MATMUL_LHS_RHS_BF16, lhsT = kernel_id == MI_KERNEL_MATMUL_LHST_RHS_BF16;
  // Skinny, a split of the rules' stays one past K = 1280 (the fused kernel's
  // at any K): one workgroup's chain over all of K costs more than the fits
  // say, which were timed with the weight in the caches.  From HBM, as a
  // decode step over many layers reads it, unsplit blocks in a split's place
  // ran, on average over 24 to 79 shapes each, 1.01 x as fast on lhsT.rhs at
  // K 1024-1280, 0.94 at 1280-1600 and 0.86 at 1600-2048 (56x1536x1856 10.1
  // -> 12.4 us); 1.03, 0.98 and 0.84 on lhs.rhs (56x872x1592 10.1 -> 14.2);
  // 0.80 to 0.87 on the fused kernel (24x3112x1032 9.1 -> 11.9).  From the
  // caches they win up to K = 2048 (1.2-1.4 x) and lose past it
  // (112x752x2288 8.6 -> 11.3, lhs.rhs 80x5928x2224 17.3 -> 20.6).
  const bool stays_split = M <= 128 && pick.split_k > 1 && (K > 1280 || !(lhs || lhsT));
  if (short_k && lhsT && pick.block_m == 256 && pick.block_n == 256) return pick;
  double best_t = margin * fitted_time(old, pick.split_k, M, N, K);
  mi_tile_cfg best = pick;
  for (int i = 0; i < n; ++i) {
    if (one_column && N > table[i].c.block_n) continue;
    if (short_k && lhs && table[i].c.block_n == 128 &&
        (table[i].c.block_m == 256 || (table[i].c.block_m == 128 && pick.block_n != 128)))
      continue;
    const long long tiles = tiles_of(M, N, table[i].c.block_m, table[i].c.block_n);
    for (const int parts : {1, 2, 3, 4, 5, 6, 7, 8, 12, 16}) {
      if (parts > 1 && tiles * parts > kCUs) break;  // runs_split refuses it and every larger one
      if (parts == 1 && stays_split) continue;
      const double t = fitted_time(table[i], parts, M, N, K);
      if (t < best_t && runs_split(kernel_id, table[i].c, parts, M, N, K)) {
        best_t = t;
        best = table[i].c;
        best.split_k = parts;
      }
    }
  }
  return best;
}

// `pick` (what the rules above choose), or a candidate of `table` that
// contains it (faster_of).  A pick that was not timed stays, and so does
// every pick of a call past the timed range.
mi_tile_cfg refined(int kernel_id, const Timed* table, int n, const mi_tile_cfg& pick, double margin, double max_flops,
                    int M, int N, int K) {
  const Timed* old = timed(table, n, pick);
  if (!old || 2.0 * M * N * K > max_flops) return pick;
  return faster_of(kernel_id, table, n, *old, pick, margin, M, N, K);
}

// fp32: the MFMA kernel with K split over the waves (variant 3; variants 0,
// in sequential K order, and 1 stay selectable), in the block and wave count
// of the least estimated time (us).  The busiest CU runs `rounds` blocks.
// Each costs its MFMAs (64 cycles per 2048 multiply-adds at 2.4 GHz and 0.94
// of that rate; 0.42 for the 16x16 blocks, which wait for their loads more),
// its operand bytes from L2 (63 GB/s per CU), and the latency of a load per
// K chunk of a wave's chain (0.26 us, once: the rounds overlap); the three
// overlap (their 3-norm), and the sum of the waves' blocks adds 6.1e-5 per
// wave and output element.  Fitted to every candidate timed at 64 shapes
// (M, N, K 64-4096, odd ones among them): the pick within 1.10 of the
// fastest at all of them, 1.013 on average (the 64x64 block of variant 1:
// 2.0 to 27 x the fastest).  A call whose operands pass 4 GiB, which variant
// 3's 32-bit offsets do not reach, keeps variant 1.
mi_tile_cfg f32_default(int M, int N, int K) {
  static const mi_tile_cfg cands[] = {{64, 64, 16, 4, 2, 1, 8, 3},  {64, 32, 16, 4, 2, 1, 8, 3},
                                      {32, 64, 16, 4, 2, 1, 8, 3},  {64, 32, 16, 8, 2, 1, 8, 3},
                                      {32, 64, 16, 8, 2, 1, 8, 3},  {32, 32, 16, 8, 2, 1, 8, 3},
                                      {32, 32, 16, 16, 2, 1, 8, 3}, {16, 16, 32, 4, 2, 1, 8, 3},
                                      {16, 16, 32, 8, 2, 1, 8, 3},  {16, 16, 32, 16, 2, 1, 8, 3}};
  if (f32_kw_span(M, K, 64) > kMaxOffset || f32_kw_span(N, K, 64) > kMaxOffset) return {64, 64, 16, 4, 1, 1, 0, 1};
  mi_tile_cfg best = cands[0];
  double best_t = 0.0;
  for (const mi_tile_cfg& c : cands) {
    const long long tiles = tiles_of(M, N, c.block_m, c.block_n);
    // A launch holds fewer than 2^32 threads; 64x64 blocks of 4 waves, as
    // many outputs a thread as variant 1's, take what variant 1 took.
    if (&c != cands && tiles * c.waves * 64 >= (1LL << 32)) continue;
    const double rounds = (double)((tiles + kCUs - 1) / kCUs);
    const double chain = (double)(((K + c.block_k - 1) / c.block_k + c.waves - 1) / c.waves);  // chunks per wave
    const double area = (double)c.block_m * c.block_n;
    const double mfma = rounds * chain * (c.waves / 4) * c.block_k * area / 32.0 / 2400.0 / (c.block_m == 16 ? 0.42 : 0.94);
    const double bytes = rounds * K * (double)(c.block_m + c.block_n) * 4.0 / 63e3;
    const double wait = chain * 0.26;
    const double t = cbrt(mfma * mfma * mfma + bytes * bytes * bytes + wait * wait * wait) + rounds * c.waves * area * 6.1e-5;
    if (&c == cands || t < best_t) {
      best = c;
      best_t = t;
    }
  }
  return best;
}

template <int N>
constexpr int count(const Timed (&)[N]) {
  return N;
}

// Skinny M with a small weight.  A weight of up to 7 MiB is read through the
// caches: the non-temporal blocks run it 1.1-1.3 x slower while the caches
// hold it, and no faster when they do not (48x5504x704 fused, 7.8 MB: 7.1
// against 8.4 us warm, 11.4 against 11.2 cold; 33 MB: 19.5 against 14.0
// cold, so a larger one streams).  lhs.rhs also had no 32- and 64-row block
// with a ring of 4: the refined pick runs within 1.025 of the fastest over
// 160 shapes, the rules' own within 1.22 (1.012 against 1.14 at 7 to 28 MiB,
// which keeps to non-temporal blocks); the fused kernel 1.014 against 1.074,
// lhsT.rhs 1.027 against 1.082.
constexpr long long kCachedWeight = 7LL << 20, kLhsSmallWeight = 28LL << 20;

mi_tile_cfg refined_skinny(int kernel_id, int M, int N, int K) {
  const long long weight = (long long)K * N * 2;
  constexpr double kMargin = 0.95, kMaxFlops = 4e11;
  if (kernel_id == MI_KERNEL_RMSNORM_MATMUL_BF16) {
    const mi_tile_cfg pick = fused_default(M, N, K);
    if (weight > kCachedWeight) return pick;
    const mi_tile_cfg c = refined(kernel_id, kFusedSkinnyTimed, count(kFusedSkinnyTimed), pick, kMargin, kMaxFlops, M, N, K);
    // The rules' block read through the caches and with one more stage, in
    // the same parts: no gain from the caches below K = 256 and at K 2560 to
    // 8192 (0.98 and 1.0 x as fast), and slower from HBM (0.98, 0.86 at the
    // least; 180 of 406 shapes by over 3 %).
    const bool same_parts = c.block_m == pick.block_m && c.block_n == pick.block_n && c.split_k == pick.split_k;
    return same_parts && (K < 256 || (K >= 2560 && K <= 8192)) ? pick : c;
  }
  const bool lhs = kernel_id == MI_KERNEL_MATMUL_LHS_RHS_BF16;
  const mi_tile_cfg pick = skinny_matmul_default(lhs, M, N, K);
  if (weight > (lhs ? kLhsSmallWeight : kCachedWeight)) return pick;
  if (!lhs) return refined(kernel_id, kLhsTSkinnyTimed, count(kLhsTSkinnyTimed), pick, kMargin, kMaxFlops, M, N, K);
  if (weight > kCachedWeight)
    return refined(kernel_id, kLhsSkinnyStreamTimed, count(kLhsSkinnyStreamTimed), pick, kMargin, kMaxFlops, M, N, K);
  return refined(kernel_id, kLhsSkinnyTimed, count(kLhsSkinnyTimed), pick, kMargin, kMaxFlops, M, N, K);
}

// Either matmul past skinny M.  At 30 shapes of each drawn afterwards and
// timed with every block and split the refined pick ran within 1.030
// (lhsT.rhs) and 1.028 (lhs.rhs) of the fastest on average; over the first
// campaign the rules' own ran within 1.06 and 1.05.  Its gains are splits of
// 256-long blocks where the rules take a smaller block unsplit or in fewer
// parts (lhsT.rhs 4736x1128x11552: 163 -> 129 us; 2528x656x15008: 84 -> 70).
// lhsT.rhs past 2.5e11 operations keeps the rules' pick (at 21 drawn shapes up
// to 4e11 the fits' ran 1.10 x its time on average, slower at 18), as does
// lhs.rhs where its rule for shapes timed on their own takes 256 x 128 in 2
// parts.
//
// Blocks 192 wide come last: they win where the other blocks leave CUs idle
// in the last round (lhs.rhs 1000x5000x4104: 160 tiles of 128 x 256 leave 96
// idle, 216 of 128 x 192 leave 40, 50.7 -> 46.5 us; lhsT.rhs 2056x4032x8520:
// 144 tiles of 256 x 256 against 231 of 192 x 192, 161 -> 133 us).  They
// change 10 of 120 picks timed (lhsT.rhs, 1.21 x faster on average, 1.07 at
// least) and 12 of 140 (lhs.rhs, 1.14 and 1.08), and at 16 changed picks of
// each drawn afterwards 1.11 (1.04 at least) and 1.12 x (1.04).  Below
// K = 512 the fits miss by up to 20 % and the picks stay; so do lhsT.rhs
// picks already split (which fill the chip: 1.10 x at one of 120 shapes) and
// 256 x 256 and 64 x 256 blocks without padded rows.  Times do not bear that
// last line out: 192-wide blocks in their place are 1.15 x faster at 63 drawn
// shapes, slower at none (3072^3 60.7 -> 49.3 us: 256 tiles of 192 x 192 fill
// the one round that 144 of 256 x 256 do not; 1088x3712x8000 73.9 -> 70.0).
// It keeps the two picks that tests name there.
mi_tile_cfg refined_matmul(int kernel_id, bool lhs, int M, int N, int K) {
  const mi_tile_cfg rules = matmul_default(kernel_id, lhs, M, N, K);
  if (lhs && rules.block_m == 256 && rules.block_n == 128 && rules.split_k == 2) return rules;
  constexpr double kMaxFlops = 4e11;
  const Timed* table = lhs ? kLhsTimed : kLhsTTimed;
  const int n = lhs ? count(kLhsTimed) : count(kLhsTTimed);
  const mi_tile_cfg pick = refined(kernel_id, table, n, rules, lhs ? 0.97 : 0.91, lhs ? kMaxFlops : 2.5e11, M, N, K);
  const Timed* old = timed(table, n, pick);
  if (!old || K < 512 || 2.0 * M * N * K > kMaxFlops) return pick;
  if (lhs) return faster_of(kernel_id, kLhs192Timed, count(kLhs192Timed), *old, pick, 0.97, M, N, K);
  const bool fixed = pick.block_n == 256 && pick.block_m != 128 && M % pick.block_m == 0;
  if (pick.split_k > 1 || fixed) return pick;
  return faster_of(kernel_id, kLhsT192Timed, count(kLhsT192Timed), *old, pick, 0.95, M, N, K);
}

// The fused kernel past skinny M.  The blocks that the rules above do not
// know are the cached 64 x 64, 64 x 128 and 128 x 128 ones with a ring of 4
// K tiles for W and 3 for x (rms_bf16_xreg.hip): at 50 shapes drawn
// afterwards and timed with every block and split the refined pick ran
// within 1.032 of the fastest on average; the rules' own ran within 1.18 at
// 70 (600x304x584: 11.0 -> 6.6 us; 1176x1432x1168: 19.5 -> 12.8;
// 6272x240x968: 19.9 -> 11.5).  Where M >= 256, N >= 2048 and K >= 2048 it
// has to win by 30 %, which keeps the picks that tests name there; at 5 %
// the picks it changes are 1.14 x faster at 61 drawn shapes, over 3 % slower
// at 2 (256x2048x2048 17.8 -> 13.2 us).
mi_tile_cfg refined_fused(int M, int N, int K) {
  const double margin = M >= 256 && N >= 2048 && K >= 2048 ? 0.7 : 0.95;
  return refined(MI_KERNEL_RMSNORM_MATMUL_BF16, kFusedTimed, count(kFusedTimed), fused_default(M, N, K), margin, 1.5e11,
                 M, N, K);
}

// The estimates and rules above, fitted to timed campaigns and checked
// against full autotune sweeps.
mi_tile_cfg estimated_default(int kernel_id, int M, int N, int K) {
  const bool lhs = kernel_id == MI_KERNEL_MATMUL_LHS_RHS_BF16;
  switch (kernel_id) {
    case MI_KERNEL_MATMUL_LHST_RHS_F32:
      return f32_default(M, N, K);
    case MI_KERNEL_MATMUL_LHST_RHS_BF16:
    case MI_KERNEL_MATMUL_LHS_RHS_BF16:
      return M <= 128 ? refined_skinny(kernel_id, M, N, K) : refined_matmul(kernel_id, lhs, M, N, K);
    case MI_KERNEL_RMSNORM_MATMUL_BF16:
      return M <= 128 ? refined_skinny(kernel_id, M, N, K) : refined_fused(M, N, K);
    default:
      return {256, 256, 64, 8, 2, 1, 8, 0};
  }
}

// The fused kernel's default for a call without gamma: the rules' choice,
// its 128x128, 64x128 and 64x64 blocks (split or not) at M > 128 given to a
// gamma-free variant, unsplit: 64x128 and 64x64 to variant 14 with the same
// block, 128x128 to the largest block whose grid keeps more than half the
// CUs busy, variant 16 at 128x128 or variant 14 at 64x128 or 64x64.
// Measured without gamma (us, 128 x 128 v16 / 64 x 128 v14 / 64 x 64 v14):
// 59.9 / 76.1 / 75.5 at 384x8192x8192 (192 tiles of 128 x 128);
// 29.2 / 23.5 / 28.7 at 512x4096x4096 (128 tiles); 10.1 / 7.9 / 6.4 at
// 1024^3 (64 tiles).  The larger blocks (128x512, 256x256 two-pass, 128x256)
// stay, variant 14 being 0-8 % slower there.  Skinny M keeps its
// non-temporal variants.
const mi_tile_cfg kGammaFree[] = {
    {128, 128, 32, 4, 4, 1, 8, 16}, {64, 128, 64, 4, 4, 1, 8, 14}, {64, 64, 64, 4, 4, 1, 8, 14}};

bool small_one_or_two_pass(const mi_tile_cfg& c) {
  const bool one_pass_or_two = c.variant == 4 || c.variant == 5 || c.variant == 13 || c.variant == 15;
  return one_pass_or_two && ((c.block_m == 128 && c.block_n == 128) || (c.block_m == 64 && c.block_n == 128) ||
                             (c.block_m == 64 && c.block_n == 64));
}

mi_tile_cfg no_gamma_default(int M, int N, int K) {
  const mi_tile_cfg c = fused_default(M, N, K);
  if (M <= 128 || !small_one_or_two_pass(c)) return c;
  const long long t128 = tiles_of(M, N, 128, 128);
  mi_tile_cfg free = kGammaFree[c.block_m == 128 ? (2 * t128 > kCUs ? 0 : 4 * t128 > kCUs ? 1 : 2) : c.block_n == 128 ? 1 : 2];
  free.group_m = c.group_m;
  return free;
}

// The refined choice with gamma, its small block split or as the gamma-free
// variant of the same size (128x128 also of the smaller ones) where the
// times fitted without gamma say that is faster: 152x160x5112, where 64x64
// blocks unsplit leave 247 CUs idle, 23.3 -> 9 us in 16 parts; 872x280x9560
// 45 -> 21 us.  The choice above stays where the times fitted without gamma
// say it is faster (by 5 %; by 15 % where the refined one is a small block,
// whose short splits those times know to no better), and, timed itself,
// before a block that was not: without gamma 256 x 128 variant 5 ran 1.2-1.4
// x the gamma-free variants' time (12936x16x8400 48 -> 61 us) and, below
// K = 512, 1.03-1.2 x that of 128 x 256.  At 996 drawn shapes past skinny M,
// inside and outside the fitted sizes, whose refined choice is another, this
// is 1.47 x faster than the choice above on average and over 3 % slower at
// 19; the refined choice everywhere was so at 106, to 5.3 x (264x880x122680,
// whose 64x64 split became the gamma-free block unsplit: 155 -> 821 us).
// Skinny M takes the refined choice where either splits K (1.12 x over 215
// shapes): both unsplit, the cached blocks that win with gamma lose to the
// non-temporal ones without it (24x5752x320: 4.0 -> 4.25 us).
mi_tile_cfg estimated_no_gamma(int M, int N, int K) {
  const mi_tile_cfg rules = no_gamma_default(M, N, K);
  mi_tile_cfg c = estimated_default(MI_KERNEL_RMSNORM_MATMUL_BF16, M, N, K);
  if (M <= 128) return c.split_k > 1 || rules.split_k > 1 ? c : rules;
  constexpr int n = count(kNoGammaTimed);
  const Timed *by_rules = timed(kNoGammaTimed, n, rules), *refined_one = timed(kNoGammaTimed, n, c);
  if (!refined_one) return by_rules && (rules.variant == 14 || rules.variant == 16 || K < 512) ? rules : c;
  const bool small = small_one_or_two_pass(c);
  double best_t = fitted_time(*refined_one, c.split_k, M, N, K);
  if (small) {
    const int bm = c.block_m, bn = c.block_n;
    for (const mi_tile_cfg& free : kGammaFree) {
      if (bm != 128 && (free.block_m != bm || free.block_n != bn)) continue;
      const double t = fitted_time(*timed(kNoGammaTimed, n, free), 1, M, N, K);
      if (t < best_t) {
        best_t = t;
        c = free;
      }
    }
  } else if (c.split_k > 1) {
    return c;  // 1.02-1.6 x faster than the choice above at 10 of 12 such shapes, 0.94 at the others
  }
  if (!by_rules) return c;
  return best_t > (small ? 1.15 : 1.05) * fitted_time(*by_rules, rules.split_k, M, N, K) ? rules : c;
}

// The picks of the shapes that a thread calls in turn.  An estimate takes up
// to 1 us of host time (0.27 at lhsT 2048x1024x8192) beside a launch's 2.8,
// and a program calls few shapes many times; one found here costs 0.006 us.
// One slot per hash, so at most kPicks per thread (12 KB), without a lock.
struct Pick {
  int kind;  // kernel id + 1, or kNoGamma; 0: empty
  int M, N, K;
  mi_tile_cfg cfg;
};
constexpr int kPickBits = 8, kPicks = 1 << kPickBits, kNoGamma = MI_NUM_KERNELS + 1;
thread_local Pick t_picks[kPicks];

template <class F>
int picked(int kind, int M, int N, int K, mi_tile_cfg* cfg, F&& estimate) {
  uint64_t h = (uint64_t)kind;
  for (const int v : {M, N, K}) h = (h ^ (uint32_t)v) * 0x9E3779B97F4A7C15ull;
  Pick& p = t_picks[h >> (64 - kPickBits)];
  if (p.kind != kind || p.M != M || p.N != N || p.K != K) p = Pick{kind, M, N, K, estimate()};
  *cfg = p.cfg;
  return MI_OK;
}

}  // namespace

int pick_default(int kernel_id, int M, int N, int K, mi_tile_cfg* cfg) {
  return picked(kernel_id + 1, M, N, K, cfg, [=] { return estimated_default(kernel_id, M, N, K); });
}

int pick_default_no_gamma(int M, int N, int K, mi_tile_cfg* cfg) {
  return picked(kNoGamma, M, N, K, cfg, [=] { return estimated_no_gamma(M, N, K); });
}

}  // namespace capi
}  // namespace mi
