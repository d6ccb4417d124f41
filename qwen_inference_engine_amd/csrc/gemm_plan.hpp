// gemm_plan.hpp — how the split GEMMs cut their work (host only but for the index that a kernel shares; no HIP).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>

#if defined(__HIPCC__)
#define QIE_PLAN_HD __host__ __device__
#else
#define QIE_PLAN_HD
#endif

namespace qie {

// ---------------------------------------------------------------- k_linear_f32.hip
namespace lf {
constexpr int BM = 64, BN = 64, BK = 32;
constexpr int LEVELS = 4;           // of the tree of K segments: 16 at most
constexpr int slab(int bm) { return 2 * bm * BN; }   // floats of a part: both K halves

struct Plan {
    int n_nt, n_mt;      // tiles of N; tiles of M per group (of the most rows a group may have)
    int log_segs;        // K segments, as a power of two: by K alone
    int log_parts;       // workgroups a tile
    int64_t row_tiles;   // indices row_tile() gives
};

// Index of the row tile from row m0 of group z (tile mt of the group) among those that exist.  Groups follow one another inside
// [0, M): a later group's rows lie further on and its z is larger, so m0 / bm + z is no other tile's, and below M / bm + groups.
QIE_PLAN_HD inline int64_t row_tile(bool grouped, int m0, int z, int mt, int n_mt, int bm = BM) {
    return grouped ? (int64_t)(m0 / bm) + z : (int64_t)z * n_mt + mt;
}

// Rows of a tile, the same bits: 32 where groups are small, whose last tiles are mostly padding (us, 64 | 32: eight experts of some 69 rows, 1,024 x
// 1,408 and 704 x 1,024, 42 | 32 and 21 | 20; of some 25 rows 26 | 20 and 19.5 | 14.5), or where few tiles of 64 would be cut into more parts (102 rows
// 1,024 x 1,024 12.5 | 10); else 64 (275 rows 1,024 x 3,072 45 | 53).
inline int tile_rows(int64_t M, int64_t N, int64_t batch, bool grouped) {
    if (grouped) return M < 128 * batch ? 32 : BM;
    return M <= 224 && (M + BM - 1) / BM * ((N + BN - 1) / BN) * batch <= 128 ? 32 : BM;
}

// Segments of 8 k-tiles or more: of 4, their meetings cost a wave 5 % beside its products (a pass of the fp32 replay 4.08 ms, of 8
// 4.04).  Workgroups a tile: until about 512 (two a CU) have work.  Grouped: rows spread over the groups.
// (At most 1,024 parts have slabs then: 32 MB on 256 CUs.)
inline Plan plan(int64_t M, int64_t N, int64_t K, int64_t batch, bool grouped, int64_t cus, int bm = BM) {
    Plan p{};
    p.n_nt = (int)((N + BN - 1) / BN);
    p.n_mt = (int)((M + bm - 1) / bm);
    p.row_tiles = grouped ? p.n_mt - 1 + batch : p.n_mt * batch;
    const int64_t busy = grouped ? std::max<int64_t>(batch, p.n_mt + batch / 2) : p.n_mt * batch;
    const int64_t want = 2 * cus / (busy * p.n_nt);
    while (p.log_segs < LEVELS && (K / BK / 8) >> (p.log_segs + 1)) p.log_segs++;
    while (p.log_parts < p.log_segs && want >> (p.log_parts + 1)) p.log_parts++;
    return p;
}
}  // namespace lf

// a / b of tile counts (below 2^22), uniform over a wave.  On the device by a float's reciprocal and one step of correction: an
// integer division is some forty instructions of a kernel's start, which cost short products 0.2 us
QIE_PLAN_HD inline int quotient(int a, int b) {
#if defined(__HIP_DEVICE_COMPILE__)
    int q = (int)((float)a * __builtin_amdgcn_rcpf((float)b));
    const int r = a - q * b;
    q += r >= b ? 1 : r < 0 ? -1 : 0;
    return __builtin_amdgcn_readfirstlane(q);
#else
    return a / b;
#endif
}

// ---------------------------------------------------------------- order of the tiles of the split GEMMs
// Workgroup numbers run down bands of `gm` row tiles, column tile by column tile: the workgroups that an XCD runs at a time (32 CUs,
// neighbours in number) cover about as many rows as columns, which is the least that its L2 has to fetch for them.  One band of all
// row tiles fetched A anew for every column tile.  Qwen2-7B at 8,192 rows, one band / bands: gate and up 1,800 / 1,690 us, down
// 950 / 885, QKV 263 / 256, O 234 / 228 (256x256 tiles); Qwen2-0.5B down at 6,000 rows 68 / 60.
QIE_PLAN_HD inline void banded(int wid, int n_mt, int n_nt, int gm, int* mt, int* nt) {
    const int band = gm * n_nt, b = quotient(wid, band), at = wid - b * band;
    const int h = n_mt - b * gm < gm ? n_mt - b * gm : gm, c = quotient(at, h);
    *mt = b * gm + at - c * h;
    *nt = c;
}

// height of even bands, up to about twice as tall as wide (`at_once` tiles of bm x bn outputs) and then as many as the row tiles hold whole, so
// up to twice that: fewer bands read the weights less often, and bands of 4 row tiles of 256 x 128 where 8 or 12 fit one band lost 4 %
inline int band_height(int n_mt, int bm, int bn, int at_once) {
    int h = 1;
    while ((h + 1) * (h + 1) * bm <= 2 * at_once * bn) h++;
    const int bands = std::max(1, n_mt / h);
    return (n_mt + bands - 1) / bands;
}

// ---------------------------------------------------------------- k_decode_fp8.hip, long rows
namespace d8s {
// Whole 16-row tiles a workgroup, one workgroup a CU (dec8s_kernel), or every tile split over `parts` of K.  Whole tiles read their weights
// 10 to 35 % faster but go by rounds of the chip: not where they keep less than three quarters of it busy, nor where a last round is mostly
// empty and K long, sooner with the 8 rows of X a chunk (M > 4) than with 4.  us, split / whole, M = 1 and 8: 17,408 x 4,608 (1.1 rounds)
// 20.1 / 20.3 and 21.4 / 25.0, x 5,120 (1.25) 21.6 / 20.8 and 23.1 / 25.6, x 6,400 (1.6) 27.9 / 22.3 and 28.8 / 28.1; 9,728 x 4,608 14.0 / 15.1 at 8
// rows; 5,120 x 5,120 9.9 / 8.6 and 10.6 / 10.3; 2,560 x 4,608 7.2 / 6.1 and 8.7 / 6.7.  The split form has at most 7 tiles a workgroup and two
// workgroups a CU: from 14 sums a CU on they no longer run at once and it takes a third longer.
inline bool whole_tiles(int64_t M, int64_t K, int64_t tiles, int64_t parts, int64_t cus) {
    if (tiles * 4 < cus * 3) return false;
    if (tiles <= cus || K <= 2560 || (K <= 5120 && tiles <= 2 * cus)) return true;
    const int64_t rounds = (tiles + cus - 1) / cus;
    const bool crowded = parts * tiles >= 14 * cus;
    if (M <= 4) return crowded || 10 * rounds * cus <= 16 * tiles;
    return 10 * rounds * cus <= (crowded || (K <= 10240 && tiles <= 2 * cus) ? 14 : tiles <= 2 * cus ? 13 : 12) * tiles;
}
}  // namespace d8s

// ---------------------------------------------------------------- k_gemm.hip, 256x256 kernel
namespace g8p {
// parts per tile: the fewest rounds of (tile, part) items over the CUs, in units of a tile
// (112 tiles: 2 parts = one round of half tiles; 144 tiles: 3 parts, two rounds of thirds)
// (short parts lose: QKV at 3 x 19 and O at 2 x 28 k-tiles measured 108 -> 112 and 71 -> 69 us,
// the last arriver's serial slab read and the per-part pipeline fill eat the gain; down at
// 2 x 148: 309 -> 247 us), so a part keeps >= 64 k-tiles (mink): split-K 2 for the O projection at 2,048 rows (112 tiles
// -> 224, K = 3,584) ran 94-98 vs 84 us for the 256x128 kernel; QKV at 3 parts 114 vs 89
inline int splitk(int64_t tiles, int64_t cus, int nk, int mink = 64) {
    int best = 1;
    double best_t = 1e30;
    for (int s = 1; s <= 4 && nk / s >= mink; s++) {
        const double t = (double)((tiles * s + cus - 1) / cus) / s;
        if (t < best_t - 1e-9) {
            best_t = t;
            best = s;
        }
    }
    return best;
}
// Parts per tile of a product of M rows and nk k-tiles of 64: 1 where the tiles fill the chip; 0: not its launch.  Unsplit, the tiles must
// cover half the chip: QKV at 144 tiles 101.7 -> 87.8 us, but O at 112 tiles 78 -> 103 us (its 256x128 kernel fills 224 CUs).
inline int parts(int64_t M, int64_t cols, int64_t K, int64_t cus, int mink = 64) {
    if (M < 256 || K % 64 != 0 || K < 256) return 0;
    const int64_t tiles = ((M + 255) / 256) * ((cols + 255) / 256);
    if (tiles >= cus) return 1;
    const int s = splitk(tiles, cus, (int)(K / 64), mink);
    return s == 1 && 2 * tiles < cus ? 0 : s;
}
// expected time, us, of `s` parts a tile: 1.45 a k-tile and 5 a round of the chip (fitted as k_gemm_mid.hip's tiles; over 20 projections at 256 to
// 8,192 rows the kernel now takes 2 % less on the average, 0.84 to 1.24 of this)
inline float us_in(int64_t M, int64_t cols, int64_t K, int64_t cus, int s) {
    const int64_t tiles = ((M + 255) / 256) * ((cols + 255) / 256), nk = K / 64;
    return (float)((tiles * s + cus - 1) / cus) * (nk / (float)s * 1.45f + 5.f) + 5.f + (s > 1 ? 8.f * s : 0.f);
}
inline float us(int64_t M, int64_t cols, int64_t K, int64_t cus) {
    const int s = parts(M, cols, K, cus);
    return s == 0 ? 1e30f : us_in(M, cols, K, cus, s);
}
}  // namespace g8p

// ---------------------------------------------------------------- k_gemm_mid.hip
namespace mid {
constexpr int BK = 64;

// Times of a tile, us, fitted to the projections of Qwen2-0.5B / 1.5B / 7B, Qwen3-14B and of 4,096 columns at 17 to 2,300 rows (474
// shapes, each measured on every tile with 1 to 8 segments; what the rule below picks is 1.6 % over the best of all of them on the
// average and 17 % at most, with the constants fitted to 168 shapes before the kernel's ring and tickets changed 2.3 %).  Of
// 80 other shapes that went to another tile: 0.95 of their time on the average, 1.01 at most: 1,536 -> 2 x 8,960 gate / up at 184 rows 28.8 -> 24.1 us,
// 3,584 -> 4,608 at 489 36.4 -> 31.1, 17,408 -> 5,120 at 133 61.3 -> 53.5.
// Up to one workgroup a CU a1 + s1 per k-tile, more a2 + (rounds of the chip) * (f2 + s2 per k-tile).  A k-tile costs what its
// lines take through one CU (about 50 GB/s where they come from HBM or another die, 120 GB/s from L2), not its matrix work,
// which is why the tall tiles win as soon as the rows fill them.  The constants are an MI355X's, whole (256 CUs): `cus` moves
// the rounds, but the slopes hold the bandwidth that 256 CUs share, so a part with fewer would still get a correct plan, not
// the fastest one.
struct Tile {
    int bm, bn, slots, per_cu;   // per_cu: workgroups that fit a CU's LDS
    float a1, s1, a2, f2, s2;
};
constexpr Tile TILES[] = {
    {64, 64, 5, 2, 3.16f, .285f, 4.93f, .68f, .487f}, {64, 128, 3, 2, 2.5f, .468f, 5.f, 1.05f, .71f},
    {128, 64, 3, 2, 3.16f, .423f, 4.06f, 1.75f, .677f}, {128, 128, 4, 1, 5.38f, .539f, 4.43f, 2.78f, .554f},
    {192, 128, 4, 1, 5.27f, .65f, 0.f, 6.45f, .693f}, {256, 128, 3, 1, 7.23f, .748f, 15.87f, .53f, .931f},
    {320, 64, 3, 1, 4.68f, .711f, 5.22f, 2.82f, .769f}, {320, 128, 2, 1, 8.f, 1.041f, 12.67f, .28f, 1.196f},
};
constexpr int N_TILES = sizeof(TILES) / sizeof(TILES[0]);
// Above the rows that were fitted the same tiles keep the times of an earlier fit: there the new ones took 0.98 on the average of 94 products but
// 1.05 to 1.09 of Qwen2-7B down's at 6,784 rows (789 us -> 857), Qwen3-14B down's at 4,864 and Qwen2-0.5B QKV's at 4,384.
constexpr int64_t FITTED_ROWS = 2304;
constexpr Tile TALL_TILES[] = {
    {64, 64, 5, 2, 3.2f, .285f, 5.f, .7f, .487f},   {64, 128, 3, 2, 2.6f, .475f, 5.4f, 1.1f, .74f},
    {128, 64, 3, 2, 3.3f, .43f, 4.7f, 1.8f, .70f},  {128, 128, 4, 1, 5.9f, .54f, 7.5f, 3.9f, .575f},
    {192, 128, 4, 1, 8.f, .65f, 5.f, 6.f, .72f},    {256, 128, 3, 1, 9.9f, .90f, 12.f, 2.5f, 1.037f},
    {320, 64, 3, 1, 6.9f, .70f, 6.5f, 3.f, .787f},  {320, 128, 2, 1, 9.4f, 1.11f, 14.f, 2.f, 1.2f},
};
static_assert(sizeof(TALL_TILES) == sizeof(TILES), "one tile, one number");
// Tiles of 160 columns, numbered on from TILES: where the columns of 128-column tiles start a round of the chip that they hardly fill
// (37,888 columns: 296 tiles, 237 of these), and so many rows of the workgroups' own (weights) that a tile of fewer columns loads more
// for the same outputs.  Whole only.
constexpr Tile WIDE[] = {
    {128, 160, 4, 1, 4.89f, .657f, 9.82f, .01f, .655f}, {192, 160, 3, 1, 6.33f, .776f, 3.01f, 4.56f, .829f},
    {256, 160, 3, 1, 4.85f, 1.139f, 0.f, 8.74f, .922f}, {320, 160, 2, 1, 6.26f, 1.498f, 0.f, 10.73f, 1.137f},
};
constexpr int N_WIDE = sizeof(WIDE) / sizeof(WIDE[0]);
constexpr Tile TALL_WIDE[] = {
    {128, 160, 4, 1, 3.f, 1.f, 11.7f, 0.f, .69f}, {192, 160, 3, 1, 6.6f, 1.1f, 7.1f, 6.3f, .825f},
    {256, 160, 3, 1, 8.8f, 1.29f, 0.f, 10.f, 1.f}, {320, 160, 2, 1, 9.6f, 1.56f, 0.f, 13.f, 1.17f},
};
static_assert(sizeof(TALL_WIDE) == sizeof(WIDE), "one tile, one number");
inline const Tile& shape(int tile) { return tile < N_TILES ? TILES[tile] : WIDE[tile - N_TILES]; }

// Row strides (elements of x, and of y in up to 4 bytes) whose offsets inside a tile of 320 rows fit the kernel's 32 bits: unsigned for x, signed for
// y, whose columns past the end lie at 2^31.
inline bool strides_fit(int64_t ldx, int64_t ldy) { return ldx <= 1 << 22 && ldy <= 1 << 20; }

struct Plan {
    int tile, whole, splitk, n_mt, n_nt;
    float us;
};

// the last round of a launch costs nearly a whole one
inline float rounds(float x) {
    const float f = (float)(int)x;
    return f + (x > f ? std::max(.8f, x - f + .3f) : 0.f);
}

// Tile and split: the tiles run whole round by round of the chip; the last, partial round's tiles may be cut into `splitk`
// K ranges (3 us a part for 128x128 outputs: slab out, slab in).
inline Plan plan(int64_t M, int64_t cols, int64_t K, int64_t cus) {
    Plan best{-1, 0, 1, 0, 0, 1e30f};
    const int nk = (int)(K / BK);
    const float floor_us = (float)cols * K * 2 / 5.3e6f + 4.f;   // the weights at the rate they stream here
    for (int c = 0; c < N_TILES; c++) {
        const Tile& t = (M > FITTED_ROWS ? TALL_TILES : TILES)[c];
        const int64_t n_mt = (M + t.bm - 1) / t.bm, n_nt = (cols + t.bn - 1) / t.bn, tiles = n_mt * n_nt;
        if (tiles > (1 << 22)) continue;   // (of 32-bit workgroup counts)
        const float room = (float)(cus * t.per_cu);
        for (int s = 1; s <= 12 && s <= nk; s++) {
            const int64_t whole = s == 1 ? tiles : tiles / (cus * t.per_cu) * (cus * t.per_cu), cut = (tiles - whole) * s;
            float us;
            if (s == 1) {
                us = tiles <= cus ? t.a1 + nk * t.s1 : t.a2 + rounds(tiles / room) * (t.f2 + nk * t.s2);
                // 64 x 64 on most CUs in one round, little of the last row tile filled: the rows that it lacks cost nothing, and the others' come the faster.
                // us, split 128 x 64 / this: 3,584 -> 3,584 at 193 rows 18.1 / 16.4, 220 18.5 / 17.5, 230 18.8 / 18.2, 245 (.83 filled) 19.2 / 19.7; 2,560 ->
                // 2,560 at 211 14.0 / 12.0; 5,120 -> 5,120 at 140 26.2 / 23.0, 166 27.6 / 27.3
                if (c == 0 && M <= FITTED_ROWS && tiles <= cus && 2 * tiles > cus && 10 * ((M - 1) % t.bm + 1) <= 6 * t.bm) us *= .95f;
            } else {
                if (cut == 0) break;
                const float len = (float)((nk + s - 1) / s);
                us = whole / room * (t.f2 + nk * t.s2) + (M > FITTED_ROWS ? 3.f * s * (t.bm * t.bn) / 16384.f + 1.f : 2.82f * s * (t.bm * t.bn) / 16384.f + .74f);
                us += cut <= cus ? t.a1 + len * t.s1 : t.a2 + rounds(cut / room) * (t.f2 + len * t.s2);
            }
            us = std::max(us, floor_us);
            if (us < best.us) best = {c, (int)whole, s, (int)n_mt, (int)n_nt, us};
        }
    }
    return best;
}

// The plan among tiles of 160 columns.  Which tiles it takes were measured against plan()'s and the 256x256 kernel on 20 projections (Qwen2-0.5B,
// 1.5B and 7B, Qwen3-14B, and 2,048, 4,096 wide ones) at 72 to 8,192 rows.  Up to two rounds of the chip (320 rows: one): 0.72 to
// 1.01 of their time, 0.88 on the average of the 73 shapes in 676 that it takes.  In more rounds each column tile's weights come as often as there
// are row tiles and the others win: Qwen2-0.5B gate / up at 1,600 rows 47.5 us | 59.4 (128 x 160, 3.1 rounds), Qwen2-7B gate / up at 640 rows 166.7 | 179.1
// (320 x 160, 1.9), Qwen3-14B down at 8,192 1,122 | 1,274 (256 x 160, 4), 5,120 718 | 792 (320 x 160, 2).  Except 320 rows x 160 over many row tiles
// (2,000 rows on) whose A stays in the Infinity Cache: Qwen2-7B QKV at 8,192 rows 249.0 | 240.3, O at 6,000 175.5 | 167.5, Qwen3-14B QKV at 7,000 448 | 435.
inline Plan plan_wide(int64_t M, int64_t cols, int64_t K, int64_t cus) {
    Plan best{-1, 0, 1, 0, 0, 1e30f};
    const int nk = (int)(K / BK);
    const float floor_us = (float)cols * K * 2 / 5.3e6f + 4.f;   // as in plan()
    for (int c = 0; c < N_WIDE; c++) {
        const Tile& t = (M > FITTED_ROWS ? TALL_WIDE : WIDE)[c];
        const int64_t n_mt = (M + t.bm - 1) / t.bm, n_nt = (cols + t.bn - 1) / t.bn, tiles = n_mt * n_nt;
        const int64_t most = t.bm < 320 ? 2 : M >= 2048 && M * K * 2 <= 80000000 ? 4 : 1;   // rounds
        if (tiles > most * cus) continue;
        const float us = std::max(floor_us, tiles <= cus ? t.a1 + nk * t.s1 : t.a2 + rounds(tiles / (float)cus) * (t.f2 + nk * t.s2));
        if (us < best.us) best = {N_TILES + c, (int)tiles, 1, (int)n_mt, (int)n_nt, us};
    }
    return best;
}

// The best of all tiles, the 256x256 kernel left aside
inline Plan best(int64_t M, int64_t cols, int64_t K, int64_t cus) {
    const Plan pl = plan(M, cols, K, cus), wide = plan_wide(M, cols, K, cus);
    // (split plans of gate / up's many columns take 10 to 30 % longer than the fit says)
    return M > 64 && wide.tile >= 0 && wide.us < (pl.splitk > 1 ? 1.1f : 1.f) * pl.us ? wide : pl;
}

// The tiles that take a product; tile -1: none, k_gemm.hip's kernels do.
inline Plan choose(int64_t M, int64_t cols, int64_t K, int64_t cus) {
    const Plan none{-1, 0, 1, 0, 0, 1e30f};
    if (K % BK != 0) return none;   // (rows of x and weights are on the 16-byte grid of LDS-DMA: qie_linear)
    const float other_us = g8p::us(M, cols, K, cus);
    const Plan pl = plan(M, cols, K, cus), wide = plan_wide(M, cols, K, cus);
    // (split plans of gate / up's many columns take 10 to 30 % longer than the fit says)
    if (M > 64 && wide.tile >= 0 && wide.us < (pl.splitk > 1 ? 1.1f : 1.f) * pl.us && wide.us < .97f * other_us) return wide;
    return pl.tile >= 0 && pl.us < .88f * other_us ? pl : none;   // 12 %: what the two fits are off by on long prompts
}
// Columns that the 256x256 kernel takes of a product, whole rounds of the chip, with the rest to the tiles above in a launch behind it; 0: one
// launch does all.  A last round of 256x256 tiles that fills little of the chip costs a whole one, and tiles of fewer columns fill it with what
// is left.  us, one launch / two: Qwen2-7B gate / up 400 rows 148 / 133, 900 rows 266 / 238, 1,500 360 / 344, down 6,000 793 / 677; Qwen3-14B gate / up
// 512 rows 209 / 164, 1,024 365 / 305, 2,048 610 / 571; Qwen2-0.5B gate / up 3,500 rows 96 / 79.
// f32: results in fp32.  The tiles sum the two halves of every k-tile apart, the 256x256 kernel in one chain: errors against 64 bits of 1.86e-7 and 2.69e-7
// at K = 2,048.  bf16 results round either away; fp32 ones stay with the tiles that would take the whole product.
inline int64_t columns_ahead(int64_t M, int64_t cols, int64_t K, int64_t cus, bool f32) {
    const int64_t n_mt = (M + 255) / 256, n_nt = (cols + 255) / 256;
    if (K % BK != 0 || K < 256 || M < 256 || n_mt * n_nt <= cus) return 0;   // (no launch of the 256x256 kernel)
    if (f32 && choose(M, cols, K, cus).tile >= 0) return 0;
    // (fitted rows: the tiles' times are 3 to 10 % short of the measured beside the 256x256 kernel's; without 1.06 of them Qwen3-14B gate / up at 2,048
    // rows would leave 10,240 columns, which takes 2 % longer than 2,048)
    const float more = M > FITTED_ROWS ? 1.f : 1.06f;
    const float whole = std::min(g8p::us(M, cols, K, cus), more * best(M, cols, K, cus).us);
    float least = .97f * whole;
    int64_t ahead = 0;
    const int64_t full = n_mt * n_nt / cus;
    for (int64_t r = full; r >= 1 && r >= full - 1; r--) {
        const int64_t c = r * cus / n_mt * 256;
        if (c <= 0 || c >= cols) continue;
        const Plan rest = best(M, cols - c, K, cus);
        // (320 x 128 tiles, whole, of long K: 1.2 to 1.35 a k-tile measured where the fit says 1.11.  Qwen3-14B down at 4,880 to 5,120 rows 748 in one launch,
        // 775 in two, with such a rest; 14,336 -> 4,096 at 6,144 rows 615, 618)
        const float slow = K > 8192 && rest.tile == 7 && rest.splitk == 1 ? 1.21f : 1.f;
        const float us = g8p::us_in(M, c, K, cus, 1) + more * slow * rest.us;   // (the first launch is never split)
        if (us < least) {
            least = us;
            ahead = c;
        }
    }
    return ahead;
}

}  // namespace mid

// ---------------------------------------------------------------- k_gemm_few.hip, and products in parts that the norm behind them adds up
namespace few {
// Times, us, fitted to 20 projections (Qwen2-0.5B / 1.5B / 7B, Qwen3-14B, 1,024 and 2,048 wide ones) at 17 to 1,300 rows, 4,900 launches: up to a workgroup
// a CU a1 + s1 per k-tile of 64, more a2 + (rounds of the chip) * (f2 + s2 per k-tile), and what the weights take from memory, as the root of their
// squares' sum; 6.3 % (rms) off.
struct Time {
    float a1, s1, a2, f2, s2;
};
struct Form {
    int fi, fj, slots;   // fragments of 16 rows, of 16 columns; chunks of a wave's ring
    Time t;
};
constexpr int WAVES = 4;
constexpr Form FORMS[] = {
    {2, 1, 4, {0.f, 0.0884f, 2.95f, 0.294f, 0.0711f}},
    {2, 2, 2, {0.f, 0.128f, 1.03f, 1.31f, 0.186f}},
    {2, 4, 2, {1.34f, 0.183f, 0.216f, 2.39f, 0.163f}},
    {4, 2, 2, {1.05f, 0.175f, 0.504f, 2.48f, 0.15f}},
    {4, 4, 2, {3.f, 0.226f, 1.47f, 3.15f, 0.212f}},
};
constexpr int N_FORMS = sizeof(FORMS) / sizeof(FORMS[0]);
constexpr std::size_t lds(const Form& f) {   // the rings; behind the loop the waves' sums
    const std::size_t ring = (std::size_t)WAVES * f.slots * 16 * (f.fi + f.fj) * 128, sums = (std::size_t)WAVES * f.fi * f.fj * 1024;
    return ring > sums ? ring : sums;
}

// A tile's rows as a buffer: its bytes, and where row r begins.  A load past its end gives zeros and reads nothing.  That check is documented for a
// lane's offset (the scalar offset beside it, says the compiler's manual, is left out; gfx950 was seen to count it), so the lane's offset alone has to
// hold rows that do not exist away: it has a row and a piece of 16 bytes, the scalar offset the k of a chunk, which lies in every row.
QIE_PLAN_HD inline uint32_t bytes_of(int rows, int64_t ld, int64_t K) { return (uint32_t)(((int64_t)(rows - 1) * ld + K) * 2); }
QIE_PLAN_HD inline uint32_t row_at(int r, int64_t ld) { return (uint32_t)r * (uint32_t)ld * 2; }

inline float us_of(const Time& t, int64_t workgroups, int per_cu, int64_t nk, bool one_row_tile, int64_t cols, int64_t K, int64_t cus) {
    const float work = workgroups <= cus ? t.a1 + nk * t.s1 : t.a2 + mid::rounds(workgroups / (float)(cus * per_cu)) * (t.f2 + nk * t.s2);
    const float weights = (float)cols * K * 2e-6f / (one_row_tile ? 6.42f : 5.92f) + 3.91f;
    return std::sqrt(work * work + weights * weights);
}
inline float us_in(const Form& f, int64_t M, int64_t cols, int64_t K, int64_t parts, int64_t cus) {
    const int64_t n_mt = (M + 16 * f.fi - 1) / (16 * f.fi), tiles = n_mt * ((cols + 16 * f.fj - 1) / (16 * f.fj));
    return us_of(f.t, tiles * parts, (int)(160 * 1024 / lds(f)), (K / 64 + parts - 1) / parts, n_mt == 1, cols, K, cus);
}
// what the other kernels are expected to take for a product
inline float others(int64_t M, int64_t cols, int64_t K, int64_t cus) { return std::min(mid::best(M, cols, K, cus).us, g8p::us(M, cols, K, cus)); }

struct Plan {
    int form;   // -1: not its shape
    float us;
};
// The form that takes a product.  Up to 512 rows, as fitted; gate and up up to 32 (beyond, x is read too often: Qwen2-7B at 64 rows 58.9 us | 60.7,
// 1,536 -> 2 x 8,960 at 40 rows 18.1 | 20.1).  `ragged`: weight segments that are no multiples of 64 rows, which tiles would cross.
inline Plan choose(int64_t M, int64_t cols, int64_t K, int64_t cus, bool gated, bool ragged) {
    Plan best{-1, 1e30f};
    if (K % 64 != 0 || ragged || M > (gated ? 32 : 512)) return best;
    if (gated) return {(cols + 63) / 64 <= cus ? 2 : 1, 0.f};
    for (int c = 0; c < N_FORMS; c++) {
        if (16 * FORMS[c].fi >= 2 * M && FORMS[c].fi > 2) continue;
        const float us = us_in(FORMS[c], M, cols, K, 1, cus);
        if (us < best.us) best = {c, us};
    }
    return best.us < .97f * others(M, cols, K, cus) ? best : Plan{-1, 1e30f};
}
}  // namespace few

// Products with a residual and a norm behind them (O and down of a prompt's layer) in parts of K whose sums the norm's launch adds up: its blocks read
// them on all CUs at once, where the last of a tile's workgroups reads the others' one after the other (3 us a part of 128 x 128 outputs).
namespace apart {
constexpr few::Time MID[] = {   // k_gemm_mid.hip's tiles, TILES and WIDE
    {2.09f, 0.252f, 4.09f, 0.f, 0.381f}, {2.9f, 0.416f, 5.39f, 0.f, 0.566f}, {3.33f, 0.398f, 5.73f, 0.f, 0.517f},
    {5.76f, 0.48f, 8.44f, 0.f, 0.497f}, {6.82f, 0.58f, 8.99f, 0.f, 0.613f}, {6.73f, 0.747f, 6.86f, 0.f, 0.781f},
    {6.35f, 0.651f, 7.39f, 0.f, 0.629f}, {4.36f, 1.1f, 5.f, 0.f, 1.07f}, {6.17f, 0.566f, 9.87f, 0.f, 0.575f},
    {5.87f, 0.701f, 8.14f, 0.f, 0.763f}, {4.97f, 0.944f, 7.55f, 0.f, 1.02f}, {3.12f, 1.28f, 3.59f, 2.23f, 1.29f},
};
static_assert(sizeof(MID) / sizeof(MID[0]) == mid::N_TILES + mid::N_WIDE, "one tile, one time");
constexpr int64_t FLOATS = 16 << 20;   // of all parts: what a stream has from the start
struct Plan {
    int form, tile, parts;   // k_gemm_few.hip's form, or k_gemm_mid.hip's tile; both -1: one launch each for product and norm
    float us;                // of both launches
};
// the norm's launch with `parts` to add; alone it takes 2.6 and 1.1 for a million values
inline float sum_us(int64_t M, int64_t N, int64_t parts) { return 2.59f + 1.55e-6f * (float)(parts * M * N); }

// us, apart | here: Qwen2-7B down at 113 rows 46.1 | 38.3, 301 rows 68.0 | 59.4, O at 301 rows 27.0 | 24.1; Qwen3-14B down at 113 rows 55.8 | 46.1;
// Qwen2-0.5B down at 113 rows 13.0 | 10.6, O at 33 rows 6.6 | 6.2.  From 700 rows on the parts' bytes take what they give, but where the tiles leave CUs
// idle (4,864 -> 896 at 800 rows 25.0 | 21.9).
// How much of the expected time of product and norm apart a plan may take: the fit is some percent off either way, by sizes.  Of weights of 8M and more, and of
// up to 64 rows, cut products take less than it says (5,120 x 17,408 at 113 rows 1.006 expected, 0.835 measured; 3,584 x 18,944 at 17 rows 0.994, 0.885).
// Of smaller weights at more rows they take more where rows are multiples of 512 (1,024 x 2,816 at 400 rows 0.989, 1.133; 2,048 x 2,048 at 640 rows
// 1.01, 1.081), else what it says or less (896 x 896 at 113 rows 1.006, 0.977).  Of 470 such plans, of 30 projections (256 to 5,120 wide) at 17 to 1,000
// rows, 374 are taken so, in 0.93 of the time on the average; 5 take 2.5 % longer or more, 1.063 at worst.  (All up to 1.03: 44, 1.133 at worst.)
inline float worth(int64_t M, int64_t N, int64_t K) {
    return M > 700 ? .9f : M <= 64 || N * K >= 8 << 20 ? 1.03f : N % 512 != 0 ? 1.015f : .97f;
}
inline Plan choose(int64_t M, int64_t N, int64_t K, int64_t cus) {
    Plan best{-1, -1, 1, 1e30f};
    if (K % 64 != 0 || N % 8 != 0 || M <= 16 || M > 1024) return best;
    for (int parts = 1; parts <= 16 && parts * M * N <= FLOATS; parts++) {
        const float sum = sum_us(M, N, parts);
        for (int c = 0; c < few::N_FORMS && M <= 640 && (parts == 1 || K / 64 >= 4 * parts); c++) {
            const few::Form& f = few::FORMS[c];
            if (f.fi > 2 && 16 * f.fi >= 2 * M) continue;
            const int64_t tiles = ((M + 16 * f.fi - 1) / (16 * f.fi)) * ((N + 16 * f.fj - 1) / (16 * f.fj));
            if (parts > 1 && tiles * parts > 3 * cus) continue;
            const float us = few::us_in(f, M, N, K, parts, cus) + sum;
            if (us < best.us) best = {c, -1, parts, us};
        }
        for (int c = 0; c < mid::N_TILES + mid::N_WIDE && parts > 1 && K / 64 >= 2 * parts; c++) {
            const mid::Tile& t = mid::shape(c);
            const int64_t n_mt = (M + t.bm - 1) / t.bm, tiles = n_mt * ((N + t.bn - 1) / t.bn);
            if (t.bm - M >= 64 || tiles * parts > 2 * cus) continue;
            const float us = few::us_of(MID[c], tiles * parts, t.per_cu, (K / 64 + parts - 1) / parts, n_mt == 1, N, K, cus) + sum;
            if (us < best.us) best = {-1, c, parts, us};
        }
    }
    const few::Plan whole = few::choose(M, N, K, cus, false, false);
    const float now = std::min(whole.us, few::others(M, N, K, cus)) + 2.6f + 1.1e-6f * (float)(M * N);
    return best.us < worth(M, N, K) * now ? best : Plan{-1, -1, 1, 1e30f};
}
}  // namespace apart

}  // namespace qie
