// gemm_plan.hpp — how the split GEMMs cut their work (host only but for the index that a kernel shares; no HIP).
#pragma once

#include <algorithm>
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
constexpr int SLAB = 2 * BM * BN;   // floats of a part: both K halves

struct Plan {
    int n_nt, n_mt;      // tiles of N; tiles of M per group (of the most rows a group may have)
    int log_segs;        // K segments, as a power of two: by K alone
    int log_parts;       // workgroups a tile
    int64_t row_tiles;   // indices row_tile() gives
};

// Index of the row tile from row m0 of group z (tile mt of the group) among those that exist.  Groups follow one another inside
// [0, M): a later group's rows lie further on and its z is larger, so m0 / 64 + z is no other tile's, and below M / 64 + groups.
QIE_PLAN_HD inline int64_t row_tile(bool grouped, int m0, int z, int mt, int n_mt) {
    return grouped ? (int64_t)(m0 / BM) + z : (int64_t)z * n_mt + mt;
}

// Workgroups a tile: until about 512 (two a CU) have work, each keeping 4 k-tiles.  Grouped: rows spread over the groups.
// (At most 1,024 parts have slabs then: 32 MB on 256 CUs.)
inline Plan plan(int64_t M, int64_t N, int64_t K, int64_t batch, bool grouped, int64_t cus) {
    Plan p{};
    p.n_nt = (int)((N + BN - 1) / BN);
    p.n_mt = (int)((M + BM - 1) / BM);
    p.row_tiles = grouped ? p.n_mt - 1 + batch : p.n_mt * batch;
    const int64_t busy = grouped ? std::max<int64_t>(batch, p.n_mt + batch / 2) : p.n_mt * batch;
    const int64_t want = std::min<int64_t>(2 * cus / (busy * p.n_nt), K / BK / 4);
    while (p.log_segs < LEVELS && (K / BK / 4) >> (p.log_segs + 1)) p.log_segs++;
    while (p.log_parts < p.log_segs && want >> (p.log_parts + 1)) p.log_parts++;
    return p;
}
}  // namespace lf

}  // namespace qie
