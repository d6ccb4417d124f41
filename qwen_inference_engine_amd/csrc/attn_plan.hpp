// attn_plan.hpp: which form of the prompts' attention kernel (k_attention.hip) a call takes (no HIP: host tests compile this file)
#pragma once

#include <cstdint>

namespace qie {

// Waves of a prefill attention workgroup, and row groups of a wave, for `npair` pairs of 16-row groups of each of `heads` (sequence, head)s.  The same bits.
// Pairs: 2 waves, and 4, while every workgroup has a CU of its own: a wave's chain of key tiles is what takes the time, and it runs faster the
// fewer waves share the CU (Qwen2-7B, 301 rows: 8 waves 16.7 us, 4 12.5); then 8.
// Where the pairs fill four fifths of the chip and no more than all of it, their even split is the faster form, us pairs | single groups: 28 heads of 128, 1,024 rows
// 27.4 | 28.5, 2,048 60.0 | 63.1, 2,300 67.7 | 71.3, 2 x 1,000 35.6 | 38.2, 3 x 700 29.2 | 29.3; 14 heads of 64, 1,024 rows 18.1 | 18.8, 2,048 32.0 | 34.5 (from three
// fifths in long prompts of head size 64: 1,500 rows 25.2 | 26.1; 2 x 330 9.4 | 8.7).  Elsewhere
// single groups: 28 heads of 128, 40 rows 7.2 | 5.4, 420 15.6 | 14.5, 1,200 39.7 | 34.0, 2,600 118 | 88, 6,000 431 | 362, 8 x 1,024 122 | 121; 40 heads, 800 rows
// 31.2 | 25.8, 2,048 99 | 76; 14 heads of 64, 113 rows 6.0 | 4.9, 2,600 51.2 | 44.1, 8,192 280 | 221, 3 x 2,500 97 | 72.  Their workgroups are of 4 waves; of 8 at head size 128 (32 KB of LDS for
// a tile of keys, so two workgroups a CU) where the pairs would take more than the chip: 2,600 rows 93 | 88, 6,000 427 | 362, but 1,400 38.6 | 44.9.
struct PrefillAttnPlan {
    int waves, groups;
};
inline PrefillAttnPlan prefill_attn_plan(int64_t npair, int64_t heads, int hd, int64_t cus) {
    auto wgs = [&](int nw) { return (npair + nw - 1) / nw * heads; };
    const int nw = wgs(2) <= cus ? 2 : wgs(4) <= cus ? 4 : 8;
    if (wgs(nw) <= cus && 5 * wgs(nw) > (hd == 64 && npair > 36 ? 3 : 4) * cus && (hd == 128 || nw < 8)) return {nw, 2};
    return {hd == 128 && wgs(8) > cus ? 8 : 4, 1};
}

// of `rows` rows a sequence; below 32 one form
inline PrefillAttnPlan prefill_attn_plan_of(int64_t rows, int64_t heads, int hd, int64_t cus) {
    return rows < 32 ? PrefillAttnPlan{2, 2} : prefill_attn_plan(((rows + 15) / 16 + 1) / 2, heads, hd, cus);
}

}  // namespace qie
