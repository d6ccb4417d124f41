// attn_decode.hpp — the fused MFMA decode attention body (k_attention.hip) and the helpers
// it shares with the prefill kernel, as a header so that the persistent decode kernel
// (k_persist.hip) runs the SAME body (same arithmetic, bit-identical outputs) as one of its
// roles.  Replaces selfattention (layers/src/self_attension.cu:10-149) for one query row.
#pragma once
#include <type_traits>

#include "qie_common.hpp"
#include "../../include/qie/qie_ops.h"

namespace qie {

constexpr int kMaxGroup = 8;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int kv16_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));

// 16 bytes per lane global -> LDS (LDS-DMA); `lds` is the wave-instruction's 1-KiB base,
// lane l lands at lds + 16 l
__device__ __forceinline__ void dma16(const uint16_t* src, uint16_t* lds) {
    __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void*)(src),
                                     (__attribute__((address_space(3))) void*)(lds), 16, 0, 0);
}


// ---------------------------------------------------------------------------
// Fused decode attention: q-projection post-processing (qk-norm + RoPE) in the
// prologue, KV append of the new token (qkv_post fused away), split-K over the context,
// and the split combine done by the last arriving wave of each (row, kv head, wave's heads):
// write-through (sc1) partials + ticket, sc1 loads in the combiner.
// Grid: (nsplit_max, nkv, B); row m has one query token at position pos[m].
struct DecodeAttnParams {
    const uint16_t* qkv;      // [B][(nq + 2 nkv) * HD] projection output (bias added)
    const int32_t* pos;
    const uint16_t* q_norm;
    const uint16_t* k_norm;
    const float* cs;
    const float* sn;
    uint16_t* kc;
    uint16_t* vc;
    KvMap km;
    int layer, nkv, nq, G, max_ctx, nsplit_max;   // G = nq / nkv
    int splits_target;        // ~splits per (row, kv head) at long context
    int dbg;                  // timing experiments only (QIE_DEC_DBG): 1 no combine, 64 exit at once
    int pre_roped;            // q and the new k arrive rotated by the QKV projection's epilogue
                              // (REF numerics, no qk-norm): the prologue only moves them
    float eps;
    int numerics;
    float* part_o;            // [B][nq][nsplit_max][HD]
    float* part_ml;           // [B][nq][nsplit_max][2]
    unsigned* counters;       // [B][nkv][waves][kDecMTicket], zero at rest
    uint16_t* out;            // [B][nq * HD]
    // engine-maintained RoPE row of each sequence's CURRENT position (finalize / set_state
    // write it, tagged with the position; [B][rope_cur_stride(HD)]): the prologue's RoPE
    // loads need no position, so they go out before it is known.  Null (operator API) or a stale tag: the table row at pos.
    const float* rc;
    int spec_ok;              // the speculative K loads may be issued (see fill_dec_params)
    // Arguments of 192 bytes, whole lines of the segment that the host writes, take it 0.5 us a launch longer than of 200 (4.8 -> 5.3 us a call of
    // qie_attention_decode; captured launches the same).  Behind what the kernel reads.
    int64_t unused = 0;
};
static_assert(sizeof(DecodeAttnParams) % 64 != 0, "arguments of the decode attention");

constexpr int kDecMaxSplits = 512;   // 64k keys per (row, kv head)

__device__ __forceinline__ void unpack_bf8(const uint4& r, float* f) {
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int j = 0; j < 4; j++) { f[2 * j] = bf_lo(w[j]); f[2 * j + 1] = bf_hi(w[j]); }
}
__device__ __forceinline__ uint4 sel4(bool c, const uint4& a, const uint4& b) {
    return make_uint4(c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z, c ? a.w : b.w);
}
// Opaque register pass-through: math on the value cannot be hoisted above this point,
// so the wait for its load lands here (after the K/V loads were issued), not before them.
__device__ __forceinline__ void pin4(uint4& v) {
    asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w));
}
__device__ __forceinline__ void pin4(float4& v) {
    asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w));
}

// Split fp32 probabilities into bf16 parts (hi, then the remainder's hi, ...) two lanes'
// values at a time: one v_cvt_pk_bf16_f32 per pair and packed fp32 subtractions.  A scalar
// (__bf16) cast per element compiled to one cvt_pk per element (half of it wasted) plus a
// shift and a subtraction each — 7 VALU per element for three parts, now 4.5.  Same RNE
// rounding, same exact remainders: bit-identical parts.
typedef float pf32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 pbf16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t cvt_pk_bf16(pf32x2_t v) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, pbf16x2_t));
}
__device__ __forceinline__ pf32x2_t unpk_bf16(uint32_t u) {
    return pf32x2_t{__uint_as_float(u << 16), __uint_as_float(u & 0xffff0000u)};
}
// e[0..7] -> NP bf16x8 parts (NP = 2: hi + lo; 3: hi + mid + lo)
template <int NP>
__device__ __forceinline__ void split_bf16x8(const float* e, uint4* parts) {
    uint32_t w[NP][4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        pf32x2_t r = pf32x2_t{e[2 * j], e[2 * j + 1]};
#pragma unroll
        for (int k = 0; k < NP; k++) {
            w[k][j] = cvt_pk_bf16(r);
            if (k + 1 < NP) r = r - unpk_bf16(w[k][j]);
        }
    }
#pragma unroll
    for (int k = 0; k < NP; k++) parts[k] = make_uint4(w[k][0], w[k][1], w[k][2], w[k][3]);
}

// ---------------------------------------------------------------------------
// Decode attention on MFMA.  The q heads of one kv head (G <= 8, padded to 16) play the role of the 16 "query rows" of the prefill
// kernel.  Workgroup = (split, kv head, row of the batch); a step covers 128 keys, 32 for each of four waves, and a wave goes through its
// own keys without a look at the others':
//   S^T = K . Q^T : A = K rows straight from memory into registers (lane: key l & 15, 8 contiguous d), B = Q^T from LDS (bf16 after
//                   norm + RoPE).  D: lane = head l & 15, keys 16 t + 4 (l >> 4) + r of tiles t = 0, 1;
//   O  += P . V   : those 8 probabilities of a lane are A's 8 k slots as they lie (k slot 8 g + 4 t + r is key 16 t + 4 g + r), in three
//                   bf16 parts (hi, mid, lo: the 24 bits of the fp32 value, so every product is the fp32 product); B = the V rows in that
//                   order, transposed by ds_read_b64_tr_b16 out of LDS that only this wave writes and reads.
// The waves' (max, sum, O) meet in LDS once per split, the splits in memory, by the last-arriving wave of a head's (tickets by wave).
// What it waits for is memory and instruction latency, at one wave a SIMD (Qwen2-7B, 2,049 keys: 4 MB of K / V in 68 workgroups), so the
// layout spares instructions and meetings.  With the scores of all 128 keys exponentiated and split by every wave, each for its slice of d,
// a step had two barriers and took 1.7 us behind its loads, now 0.9; with one ticket a kv head, its workgroup alone read all splits back:
// 2.7 us for 17, now 1.8 by four waves on CUs of their own.  V goes out behind the prologue while K is on its way: 3 to 10 % of a launch over waiting
// for K first (8 rows paged in 352 workgroups 2 % longer: some CUs have two, and one's V goes ahead of the other's K).  From launch to launch in a
// graph, the form with barriers / now, us: Qwen2-0.5B at 129 keys 6.2 / 4.1, 7 rows at 700 8.5 / 5.3, Qwen2-7B at 2,049 9.2 / 7.3, 4 rows at 1,500 11.2 /
// 7.6, 8 at 1,025 paged 11.9 / 9.2, Qwen3-14B at 6,001 14.3 / 10.0.
constexpr int kDecMStep = 128;      // keys per step
constexpr int kDecMWaves = 4;       // waves that have keys
constexpr int kDecMSplits = 32;     // default split target
constexpr int kDecMTicket = 32;     // a ticket's words: 128 bytes (16 tickets in one line took 2 us of the 17 splits' adds)
constexpr int kDecMOneSplit = 2;    // contexts of up to this many steps run as ONE split

__host__ __device__ __forceinline__ int decm_chunk(int ctx, int target) {
    // Short contexts: one block walks both steps instead of two one-step splits that pay
    // the publish + ticket + combine round trips (Qwen2-0.5B, ctx 129-256: 8.8 -> 7.4 us
    // per launch, 1,235 -> 1,271 tok/s).  Longer contexts want the CUs: a split's K/V comes
    // through one CU.
    if (ctx <= kDecMOneSplit * kDecMStep) return kDecMOneSplit * kDecMStep;
    const int per = kDecMStep * target;
    return ctx <= per ? kDecMStep : kDecMStep * ((ctx + per - 1) / per);
}
// splits of a context: chunks of one or two steps without a division
__host__ __device__ __forceinline__ int decm_splits(int ctx, int chunk) {
    if (chunk == kDecMStep) return (ctx + kDecMStep - 1) / kDecMStep;
    if (chunk == 2 * kDecMStep) return (ctx + 2 * kDecMStep - 1) / (2 * kDecMStep);
    return (ctx + chunk - 1) / chunk;
}

struct DecPro {
    uint4 raw, nraw;
    float4 c0, s0, c1, s1;
    bool is_q, is_k, is_v, pro, nrm, hf;
};

// this lane's RoPE coefficients from a table row (cos row cp, sin row sp)
template <int HD>
__device__ __forceinline__ void dec_rope_load(DecPro& d, int dl, const float* cp, const float* sp) {
    const int rb = d.hf ? (dl * 8) % (HD / 2) : dl * 4;
    const int rb2 = d.hf ? rb + 4 : rb;
    d.c0 = *reinterpret_cast<const float4*>(cp + rb);
    d.s0 = *reinterpret_cast<const float4*>(sp + rb);
    d.c1 = *reinterpret_cast<const float4*>(cp + rb2);
    d.s1 = *reinterpret_cast<const float4*>(sp + rb2);
}

template <int HD, bool PR>
__device__ __forceinline__ DecPro dec_pro_issue(const DecodeAttnParams& a, const uint16_t* row, int g, int G, int grp,
                                                int dl, const float* cp, const float* sp, bool has_new) {
    DecPro d;
    d.is_q = grp < G;
    d.is_k = grp == G;
    d.is_v = grp == G + 1;
    d.pro = d.is_q || ((d.is_k || d.is_v) && has_new);
    d.hf = a.numerics == QIE_NUMERICS_HF;
    const uint16_t* src = d.is_q ? row + (g * G + grp) * HD
                                 : (d.is_k ? row + a.nq * HD + g * HD : row + (a.nq + a.nkv) * HD + g * HD);
    if (!(d.is_q || d.is_k || d.is_v)) src = row;
    d.raw = *reinterpret_cast<const uint4*>(src + dl * 8);
    if constexpr (PR) {   // rotated upstream, no qk-norm: nothing else to load
        d.nrm = false;
        return d;
    }
    const uint16_t* nwp = d.is_q ? a.q_norm : a.k_norm;
    d.nrm = nwp != nullptr && !d.is_v;
    d.nraw = *reinterpret_cast<const uint4*>((nwp ? nwp : row) + dl * 8);
    dec_rope_load<HD>(d, dl, cp, sp);
    return d;
}

// qk-norm + RoPE of the q heads and the new k, then q -> LDS (bf16), new k/v -> cache
// and LDS.  Branch-free: loads unconditional, only the stores predicated.
template <int HD, bool PR>
__device__ __forceinline__ void dec_pro_finish(const DecodeAttnParams& a, DecPro& d, int dl, int grp, int64_t poff,
                                               uint16_t* kb, uint16_t* vb, uint16_t (*q_s)[HD],
                                               uint16_t (*kv_new)[HD]) {
#pragma clang fp contract(off)
    constexpr int LPT = HD / 8;
    if constexpr (PR) {   // q / new k already rotated: move them
        pin4(d.raw);
        if (d.is_q) {
            *reinterpret_cast<uint4*>(&q_s[grp][dl * 8]) = d.raw;
        } else if (d.pro) {
            *reinterpret_cast<uint4*>((d.is_k ? kb : vb) + poff + dl * 8) = d.raw;
            *reinterpret_cast<uint4*>(&kv_new[d.is_k ? 0 : 1][dl * 8]) = d.raw;
        }
        return;
    }
    pin4(d.raw); pin4(d.nraw); pin4(d.c0); pin4(d.s0); pin4(d.c1); pin4(d.s1);
    float x[8], wv[8];
    unpack_bf8(d.raw, x);
    unpack_bf8(d.nraw, wv);
    // qk-norm (Qwen3) and HF numerics are launch-uniform: branch around them instead of
    // computing both forms per element (Qwen2, REF: neither — 8 divisions and the HF RoPE
    // products per lane were dead work on the critical path)
    if (a.q_norm != nullptr || a.k_norm != nullptr) {   // per lane: d.nrm picks q_norm / k_norm
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < 8; j++) ss += x[j] * x[j];
        ss = group_sum<LPT>(ss);
        const float rms = sqrtf((ss / (float)HD) + a.eps);
        if (d.hf) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float xn = rbf(wv[j] * rbf(x[j] * (1.0f / rms)));
                x[j] = d.nrm ? xn : x[j];
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float xn = rbf((x[j] / rms) * wv[j]);
                x[j] = d.nrm ? xn : x[j];
            }
        }
    }
    const float cv[8] = {d.c0.x, d.c0.y, d.c0.z, d.c0.w, d.c1.x, d.c1.y, d.c1.z, d.c1.w};
    const float sv[8] = {d.s0.x, d.s0.y, d.s0.z, d.s0.w, d.s1.x, d.s1.y, d.s1.z, d.s1.w};
    float y[8];
    if (d.hf) {
        float o[8];
#pragma unroll
        for (int j = 0; j < 8; j++) o[j] = __shfl_xor(x[j], LPT / 2, 64);
        const float sg = dl < LPT / 2 ? -1.f : 1.f;   // rotate_half: first half takes -x[j + hd/2]
#pragma unroll
        for (int j = 0; j < 8; j++) y[j] = rbf(rbf(x[j] * cv[j]) + rbf((sg * o[j]) * sv[j]));
    } else {
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
            y[j] = rbf(x[j] * cv[j / 2] - x[j + 1] * sv[j / 2]);
            y[j + 1] = rbf(x[j + 1] * cv[j / 2] + x[j] * sv[j / 2]);
        }
    }
#pragma unroll
    for (int j = 0; j < 8; j++) x[j] = d.is_v ? x[j] : y[j];
    const uint4 packed = make_uint4(pack2(x[0], x[1]), pack2(x[2], x[3]), pack2(x[4], x[5]), pack2(x[6], x[7]));
    if (d.is_q) {
        *reinterpret_cast<uint4*>(&q_s[grp][dl * 8]) = packed;
    } else if (d.pro) {
        uint16_t* dst = (d.is_k ? kb : vb) + poff + dl * 8;
        *reinterpret_cast<uint4*>(dst) = packed;
        *reinterpret_cast<uint4*>(&kv_new[d.is_k ? 0 : 1][dl * 8]) = packed;
    }
}

// Body of the decode attention for split s of kv head g, batch row by.
// Hooks of the body (X): the stand-alone kernel runs it with AttnNoHook — q / k / v rows from
// a.qkv, outputs to a.out.  The persistent decode kernel (k_persist.hip) passes a hook whose
// gather() fills the q / k / v row image (a.qkv points at it) from the projection's hand-off
// granules AFTER this block's K / V loads are issued (they need no q), and whose out4
// takes the block's output values (to publish them as granules).  The arithmetic is the same.
struct AttnNoHook {
    static constexpr bool on = false;
    __device__ void gather() {}
    __device__ void out4(int64_t, unsigned long long) {}
};

template <int HD, bool PG, int NWA, bool PR, class X = AttnNoHook>
__device__ __forceinline__ void attn_decode_mfma2_body(const DecodeAttnParams& a, const int g, const int s, const int by,
                                                       X* hook = nullptr) {
#pragma clang fp contract(off)
    constexpr int KS = kDecMStep;
    constexpr int LPT = HD / 8;          // prologue: lanes per head row
    constexpr int KSTEPS = HD / 32;      // MFMA k-steps over d for S
    constexpr int CPR = HD / 8;          // 16-byte chunks per row
    constexpr int DT = HD / 16;          // output d tiles
    constexpr int VCH = 32 * CPR / 64;   // V chunks per lane per step
    constexpr int NT = 64 * NWA;         // threads
    static_assert(NWA >= kDecMWaves, "attn_decode: four waves have keys");
    __shared__ __attribute__((aligned(16))) uint16_t q_s[16][HD];
    __shared__ __attribute__((aligned(16))) uint16_t kv_new[2][HD];
    __shared__ __attribute__((aligned(16))) uint16_t v_s[kDecMWaves][32 * HD];   // V rows of a wave's keys; behind the steps its O
    __shared__ __attribute__((aligned(16))) float2 ml_s[kDecMWaves][16];

    const int64_t m = by;
    const int G = a.G;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, gq = lane >> 4;
    const int grp = tid / LPT, dl = tid % LPT;
    // (a constant where it is true of every wave: loads under a branch made the prologue wait for all of K, ahead of V)
    const bool keyed = NWA == kDecMWaves || wave < kDecMWaves;
    const int QKVD = (a.nq + 2 * a.nkv) * HD;
    const uint16_t* row = a.qkv + m * (int64_t)QKVD;
    const int64_t head_off = kv_run_off(a.km, (int64_t)a.layer * a.nkv + g, HD);
    uint16_t* kb = a.kc + head_off;
    uint16_t* vb = a.vc + head_off;
    // steps in flight; at head dim 128 one, in 250 registers: a second workgroup on the CU hides more than a second step (and the persistent
    // kernel has no registers for it)
    constexpr int SETS = X::on || HD == 128 ? 1 : 2;
    uint4 kf[SETS][2][KSTEPS], vr[SETS][VCH];   // [step % SETS]
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, SETS - 1> odd{};
    // loads of this wave's 32 of the `n` keys (128 at most count) that start at element `so` of a run; rows past them read as zeros
    // (a 128-key step never straddles a page: chunks and pages are multiples of 128)
    const int k_at = 32 * wave * HD * 2;
    auto load_k = [&](auto x, int64_t so, int n) {
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(kb + so, (short)0, n * HD * 2, 0x00020000);
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ks++)
                kf[x][t][ks] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, k_at + (16 * t + fr) * HD * 2 + 16 * gq + 64 * ks, 0, 0));
    };
    auto load_v = [&](auto x, int64_t so, int n) {
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(vb + so, (short)0, n * HD * 2, 0x00020000);
#pragma unroll
        for (int i = 0; i < VCH; i++)
            vr[x][i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, k_at + lane * 16 + i * 1024, 0, 0));
    };
    // Speculative step (contiguous cache): the split of every context of 257 ..
    // 128 * splits keys is keys [128 s, 128 s + 128) (decm_chunk's one-step rule), so its
    // K loads go out with the position load instead of one HBM round trip behind it.
    // The rotated q / k / v row goes out first (position-independent): vmcnt retires in
    // order, and the prologue that waits for it must not wait behind the whole step.
    // Without the pre-rotation the same holds when the engine keeps the current position's
    // RoPE row (a.rc, tagged with the position): the prologue's loads then need no position
    // either, and a stale tag (a position set some other way) reloads the table row.
    // (Paged: the pages of a one-step and of a two-step split, 0.3 us of a launch each one after the other, come with the position; the K / V loads themselves, issued
    // ahead by them, made eight users slower: 3,563 tok/s against 3,624.)
    const bool ahead = PR || a.rc != nullptr;   // uniform: the prologue's loads need no position
    const bool spec = !PG && ahead && a.spec_ok;
    const int p = a.pos[m];
    int page1 = 0, page2 = 0, page3 = 0;
    if constexpr (PG) {
        const int32_t* tb = a.km.table + m * a.km.max_pages;
        page1 = tb[min((KS * s) >> a.km.shift, a.km.max_pages - 1)];
        page2 = tb[min((2 * KS * s) >> a.km.shift, a.km.max_pages - 1)];
        page3 = tb[min((2 * KS * s + KS) >> a.km.shift, a.km.max_pages - 1)];
    }
    const float* rcm = a.rc ? a.rc + m * rope_cur_stride(HD) : a.cs;
    const int rtag = a.rc ? __float_as_int(rcm[0]) : -1;
    DecPro pr;
    if (spec) {
        if constexpr (X::on) {   // the row is gathered after the K / V step is in flight
            if (keyed) load_k(even, kv_tok<false>(a.km, m, KS * s, HD), min(KS, a.max_ctx - KS * s));
            __builtin_amdgcn_sched_barrier(0);
            hook->gather();
            pr = dec_pro_issue<HD, PR>(a, row, g, G, grp, dl, rcm + 8, rcm + 8 + HD / 2, false);
        } else {
            pr = dec_pro_issue<HD, PR>(a, row, g, G, grp, dl, rcm + 8, rcm + 8 + HD / 2, false);
            __builtin_amdgcn_sched_barrier(0);
            if (keyed) load_k(even, kv_tok<false>(a.km, m, KS * s, HD), min(KS, a.max_ctx - KS * s));
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
        if constexpr (X::on) hook->gather();
        if (ahead) pr = dec_pro_issue<HD, PR>(a, row, g, G, grp, dl, rcm + 8, rcm + 8 + HD / 2, false);
    }
    const int ctx = p + 1;
    const int chunk = decm_chunk(ctx, a.splits_target);
    const int nsplit = decm_splits(ctx, chunk);
    if (s >= nsplit || QIE_DBG(a.dbg & 64)) return;
    const int t0 = s * chunk, t1 = min(ctx, t0 + chunk);
    const int nstep = (t1 - t0 + KS - 1) / KS;
    const bool has_new = (t1 == ctx);
    auto run_of = [&](int tok) -> int64_t {   // kv_tok of the first key of a step
        if constexpr (PG) {
            int page = page1;
            if (tok != KS * s) page = tok == 2 * KS * s ? page2 : tok == 2 * KS * s + KS ? page3 : a.km.table[m * a.km.max_pages + (tok >> a.km.shift)];
            return (int64_t)page * a.km.stride + (int64_t)(tok & ((1 << a.km.shift) - 1)) * HD;
        } else {
            return kv_tok<false>(a.km, m, tok, HD);
        }
    };
    auto keys_of = [&](int st) { return min(KS, t1 - t0 - st * KS); };
    auto load_step = [&](auto x, int st) {
        const int64_t so = run_of(t0 + st * KS);
        load_k(x, so, keys_of(st));
        load_v(x, so, keys_of(st));
    };

    // ---------------- loads: prologue operands, then the first step's K, and its V behind the prologue: a CU has some 40 KB of loads in
    // flight, and a wave that has more to send waits
    if (ahead) {
        pr.pro = pr.is_q || ((pr.is_k || pr.is_v) && has_new);
        if (!PR && rtag != p)   // uniform: the kept row is not this position's
            dec_rope_load<HD>(pr, dl, a.cs + (int64_t)p * (HD / 2), a.sn + (int64_t)p * (HD / 2));
    } else {
        pr = dec_pro_issue<HD, PR>(a, row, g, G, grp, dl, a.cs + (int64_t)p * (HD / 2), a.sn + (int64_t)p * (HD / 2),
                                   has_new);
    }
    __builtin_amdgcn_sched_barrier(0);
    // (uniform) the speculative step is this split's first step iff the split starts at key
    // KS s: one-step splits, and split 0 of every context (the one-split contexts of <= 2
    // steps, Qwen2-0.5B's ctx 129-256, re-issued the same loads behind the position: +1.2 us)
    // (rows past the context hold whatever the cache has there: their scores are masked to -inf)
    const int64_t so0 = run_of(t0);
    const int64_t new_at = has_new ? run_of(p & ~(KS - 1)) + (p & (KS - 1)) * HD : 0;   // the new token's place (a step's keys are in one page)
    if (keyed && (!spec || t0 != KS * s)) load_k(even, so0, keys_of(0));
    dec_pro_finish<HD, PR>(a, pr, dl, grp, new_at, kb, vb, q_s, kv_new);
    if (keyed) load_v(even, so0, keys_of(0));
    if (SETS > 1 && keyed && nstep > 1) load_step(odd, 1);
    for (int idx = tid; idx < (16 - G) * CPR; idx += NT)   // padded q rows
        *reinterpret_cast<uint4*>(&q_s[G + idx / CPR][(idx % CPR) * 8]) = make_uint4(0, 0, 0, 0);
    __syncthreads();

    const float scale = sqrtf((float)HD);
    // dot / scale as q = dot * (1 / scale) plus one FMA residual step (Markstein): the
    // correctly rounded quotient for every dot above 2^-100 in magnitude (k_decode_fp8.hip
    // d8_rms_pair), three VALU ops instead of the IEEE division sequence's ~10 with its
    // serial latency
    const float inv_scale = 1.0f / scale;
    auto qdiv = [&](float d) {
        const float q = d * inv_scale;
        if constexpr (HD == 64) return q;   // sqrt(hd) a power of two: exact
        else return fmaf(fmaf(-q, scale, d), inv_scale, q);
    };
    const int nq = a.nq;
    uint16_t* vw = &v_s[wave < kDecMWaves ? wave : 0][0];
    if (keyed) {
        bf16x8_t qb[KSTEPS];
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ks++) qb[ks] = *reinterpret_cast<const bf16x8_t*>(&q_s[fr][32 * ks + 8 * gq]);
        float m_run = -INFINITY, l_run = 0.f;
        f32x4_t oacc[DT];
#pragma unroll
        for (int d = 0; d < DT; d++) oacc[d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        // element of row r, column c (a multiple of 4) of the V rows: 32-byte chunks of a row in turn, so that the 16 rows of a
        // transposing read lie in different banks
        auto v_at = [&](int r, int c) { return r * HD + (((c >> 4) ^ (HD == 128 ? r & 7 : (r >> 1) & 3)) << 4) + (c & 15); };
        const int q4 = fr >> 2, p4 = fr & 3;
        auto process = [&](auto x, int st) {
            const int kb0 = t0 + st * KS, k0 = kb0 + 32 * wave;
            // the new token's K / V rows from LDS (uniform: the wave that has it)
            if (p >= k0 && p < k0 + 32) {
#pragma unroll
                for (int ks = 0; ks < KSTEPS; ks++) {
                    const uint4 kn = *reinterpret_cast<const uint4*>(&kv_new[0][32 * ks + 8 * gq]);
#pragma unroll
                    for (int t = 0; t < 2; t++) kf[x][t][ks] = sel4(k0 + 16 * t + fr == p, kn, kf[x][t][ks]);
                }
                const uint4 vn = *reinterpret_cast<const uint4*>(&kv_new[1][(lane % CPR) * 8]);   // (64 is a multiple of CPR)
#pragma unroll
                for (int i = 0; i < VCH; i++) vr[x][i] = sel4(k0 + (lane + 64 * i) / CPR == p, vn, vr[x][i]);
            }
            // ---- S^T of this wave's 32 keys: lane = head fr, keys 16 t + 4 gq + r
            f32x4_t sacc[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ks++)
#pragma unroll
                for (int t = 0; t < 2; t++)
                    sacc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kf[x][t][ks]), qb[ks], sacc[t], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < VCH; i++) {
                const int c = lane + 64 * i;
                *reinterpret_cast<uint4*>(vw + v_at(c / CPR, (c % CPR) * 8)) = vr[x][i];
            }
            wave_lds_fence();   // (here: the reads below may go ahead of the exponentials)
            if (st + SETS < nstep) load_step(x, st + SETS);
            // scores s = dot / sqrt(hd) (self_attension.cu); those past the split's end are no keys (uniform)
            float e[8];
#pragma unroll
            for (int j = 0; j < 8; j++) e[j] = qdiv(sacc[j / 4][j % 4]);
            if (k0 + 32 > t1) {
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (k0 + 16 * (j / 4) + 4 * gq + j % 4 >= t1) e[j] = -INFINITY;
            }
            float mt = fmaxf(fmaxf(fmaxf(e[0], e[1]), fmaxf(e[2], e[3])), fmaxf(fmaxf(e[4], e[5]), fmaxf(e[6], e[7])));
            mt = xor32_max(xor16_max(mt));
            const float m_new = fmaxf(m_run, mt);
            const float m_use = m_new == -INFINITY ? 0.f : m_new;
            // __expf (v_exp_f32 on x * log2 e, ~2 ulp): the reference build itself
            // compiles with -use_fast_math, i.e. the same approximation
            const float alpha = __expf(m_run - m_use);
#pragma unroll
            for (int j = 0; j < 8; j++) e[j] = __expf(e[j] - m_use);
            const float ls = xor32_sum(xor16_sum(((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]))));
            l_run = l_run * alpha + ls;
            m_run = m_new;
            // bit-identical skip, as in the prefill kernel: step 0's O is zero, and alpha == 1
            // exactly where no row's max grew (wave-uniform ballot)
            if (st > 0 && __builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
                float ar[4];
#pragma unroll
                for (int r = 0; r < 4; r++) ar[r] = __shfl(alpha, gq * 4 + r, 64);
#pragma unroll
                for (int d = 0; d < DT; d++)
#pragma unroll
                    for (int r = 0; r < 4; r++) oacc[d][r] *= ar[r];
            }
            uint4 pp[3];
            split_bf16x8<3>(e, pp);
            const bf16x8_t ph = __builtin_bit_cast(bf16x8_t, pp[0]), pm = __builtin_bit_cast(bf16x8_t, pp[1]),
                           pl = __builtin_bit_cast(bf16x8_t, pp[2]);
            constexpr int DG = 4;   // tiles of d at a time
#pragma unroll
            for (int d0 = 0; d0 < DT; d0 += DG) {
            bf16x8_t vt[DG];
#pragma unroll
            for (int dd = 0; dd < DG; dd++) {
                const int d = d0 + dd;
                const i16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) i16x4_t*)(vw + v_at(4 * gq + q4, 16 * d + 4 * p4)));
                const i16x4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) i16x4_t*)(vw + v_at(16 + 4 * gq + q4, 16 * d + 4 * p4)));
                vt[dd] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
            }
#pragma unroll
            for (int dd = 0; dd < DG; dd++) oacc[d0 + dd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ph, vt[dd], oacc[d0 + dd], 0, 0, 0);
#pragma unroll
            for (int dd = 0; dd < DG; dd++) oacc[d0 + dd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pm, vt[dd], oacc[d0 + dd], 0, 0, 0);
#pragma unroll
            for (int dd = 0; dd < DG; dd++) oacc[d0 + dd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl, vt[dd], oacc[d0 + dd], 0, 0, 0);
            }
            wave_lds_fence();   // the next step's V, and O behind the last, go where these rows were
        };
        for (int st = 0; st < nstep; st += 2) {
            process(even, st);
            if (st + 1 < nstep) process(odd, st + 1);
        }
        // ---------------- the waves' results to LDS (O where this wave's V rows were: its own reads of them are done)
        if (gq == 0) ml_s[wave][fr] = make_float2(m_run, l_run);
        float* ow = reinterpret_cast<float*>(vw);   // [8 heads][HD]
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int h = 4 * gq + r;
            if (h < G) {
#pragma unroll
                for (int d = 0; d < DT; d++) ow[h * HD + 16 * d + fr] = oacc[d][r];
            }
        }
    }
    __syncthreads();
    // ---------------- thread (head gi, 4 dims from 4 d4): the split's maximum, sum and O.  From here on every wave goes by itself: its
    // heads have a ticket of their own, so that the last arrivers of a kv head's waves are spread over its splits' CUs
    const int items = G * (HD / 4);
    if (64 * wave >= items) return;   // uniform
    const bool has_item = tid < items;
    const int gi = has_item ? tid / (HD / 4) : 0, d4 = tid % (HD / 4);
    float2 wml[kDecMWaves];
#pragma unroll
    for (int w = 0; w < kDecMWaves; w++) wml[w] = ml_s[w][gi];
    const float m_spl = fmaxf(fmaxf(wml[0].x, wml[1].x), fmaxf(wml[2].x, wml[3].x));
    const float m_at = m_spl == -INFINITY ? 0.f : m_spl;   // (all keys of the split at -inf: its sum is 0, not NaN)
    float l_spl = 0.f;
    float4 o_spl = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < kDecMWaves; w++) {
        const float c = __expf(wml[w].x - m_at);   // 0 for a wave without keys
        const float4 o = reinterpret_cast<const float4*>(&v_s[w][0])[gi * (HD / 4) + d4];
        l_spl = fmaf(wml[w].y, c, l_spl);
        o_spl.x = fmaf(c, o.x, o_spl.x);
        o_spl.y = fmaf(c, o.y, o_spl.y);
        o_spl.z = fmaf(c, o.z, o_spl.z);
        o_spl.w = fmaf(c, o.w, o_spl.w);
    }
    // divided (not multiplied by 1/l): the softmax normalisation's one rounding
    auto result = [&](const float4& o, float l) {
        return (unsigned long long)pack2(o.x / l, o.y / l) | ((unsigned long long)pack2(o.z / l, o.w / l) << 32);
    };
    const int64_t out_at = m * (int64_t)nq * HD + (int64_t)(g * G + gi) * HD + d4 * 4;
    if (nsplit == 1) {
        if (has_item) {
            const unsigned long long pk = result(o_spl, l_spl);
            if constexpr (X::on) hook->out4(out_at, pk);
            else *reinterpret_cast<unsigned long long*>(a.out + out_at) = pk;
        }
        return;
    }
    // write-through (sc1) stores: published by the drain + ticket below, no release fence
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc((void*)a.part_o, 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc((void*)a.part_ml, 0, 0x7fffffff, 0x00020000);
    const int hbase = (int)((m * nq + g * G + gi) * (int64_t)a.nsplit_max);
    if (has_item) {
        __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{__float_as_uint(o_spl.x), __float_as_uint(o_spl.y), __float_as_uint(o_spl.z), __float_as_uint(o_spl.w)},
                                               ro, ((hbase + s) * (HD / 4) + d4) * 16, 0, 16);
        if (d4 == 0) __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{__float_as_uint(m_spl), __float_as_uint(l_spl)}, rm, (hbase + s) * 8, 0, 16);
    }
    // ---------------- publish this split; the last arriver combines
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // stored
    if (QIE_DBG(a.dbg & 1)) return;
    unsigned* cnt = a.counters + ((m * a.nkv + g) * kDecMWaves + wave) * kDecMTicket;
    unsigned old = 0;
    if (lane == 0) old = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    old = __builtin_amdgcn_readfirstlane(old);
    if (old != (unsigned)nsplit - 1) return;   // uniform
    asm volatile("" ::: "memory");
    // The splits of the head by 16-B sc1 buffer loads (L2 / memory side, never a stale L1 line) on a uniform resource: every partial
    // was stored sc1 by a wave that drained (vmcnt 0) before its ticket add, and this wave's add came last.  (With an acquire fence instead 9.79 against 9.56 us per launch; 8-B agent-scope atomic loads 11.4 against 10.7.)
    // A thread loads the (m, l) of EVERY split of its head together with its 16 bytes of their O, groups of four that exist in flight
    // together (up to JB splits: one round trip), then merges them itself.
    constexpr int JB = 24;
    float mx = -INFINITY, ls = 0.f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int j0 = 0; j0 < nsplit; j0 += JB) {
        float4 v[JB];
        float2 w[JB];
#pragma unroll
        for (int b = 0; b < JB; b += 4) {
            if (j0 + b >= nsplit) break;   // uniform
#pragma unroll
            for (int jj = b; jj < b + 4; jj++) {
                const u32x2_t q2 = __builtin_amdgcn_raw_buffer_load_b64(rm, (hbase + min(j0 + jj, nsplit - 1)) * 8, 0, 16);
                w[jj] = make_float2(__uint_as_float(q2.x), __uint_as_float(q2.y));
            }
        }
#pragma unroll
        for (int b = 0; b < JB; b += 4) {
            if (j0 + b >= nsplit) break;
#pragma unroll
            for (int jj = b; jj < b + 4; jj++) {
                const u32x4_t q4 = __builtin_amdgcn_raw_buffer_load_b128(ro, ((hbase + min(j0 + jj, nsplit - 1)) * (HD / 4) + d4) * 16, 0, 16);
                v[jj] = make_float4(__uint_as_float(q4.x), __uint_as_float(q4.y), __uint_as_float(q4.z), __uint_as_float(q4.w));
            }
        }
        float mb = mx;
#pragma unroll
        for (int b = 0; b < JB; b += 4) {
            if (j0 + b >= nsplit) break;
#pragma unroll
            for (int jj = b; jj < b + 4; jj++) mb = fmaxf(mb, j0 + jj < nsplit ? w[jj].x : -INFINITY);
        }
        const float mu = mb == -INFINITY ? 0.f : mb;
        const float sc = __expf(mx - mu);   // 0 on the first batch (mx = -inf)
        ls *= sc;
        acc.x *= sc; acc.y *= sc; acc.z *= sc; acc.w *= sc;
#pragma unroll
        for (int b = 0; b < JB; b += 4) {
            if (j0 + b >= nsplit) break;
#pragma unroll
            for (int jj = b; jj < b + 4; jj++) {
                const float c = j0 + jj < nsplit ? __expf(w[jj].x - mu) : 0.f;
                ls = fmaf(w[jj].y, c, ls);
                acc.x = fmaf(c, v[jj].x, acc.x);
                acc.y = fmaf(c, v[jj].y, acc.y);
                acc.z = fmaf(c, v[jj].z, acc.z);
                acc.w = fmaf(c, v[jj].w, acc.w);
            }
        }
        mx = mb;
    }
    if (lane == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // (persistent kernel: who sees the output may take the next layer's ticket)
    if constexpr (X::on) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (has_item) {
        const unsigned long long pk = result(acc, ls);
        if constexpr (X::on) hook->out4(out_at, pk);
        else *reinterpret_cast<unsigned long long*>(a.out + out_at) = pk;
    }
}

}  // namespace qie
