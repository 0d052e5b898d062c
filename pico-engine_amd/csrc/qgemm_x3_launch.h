// Launch side of qgemm_x3.h: sizes of the x3 form, the kernels' tile rule, and the per-format
// launchers (instantiated in qgemm_x3_<format>.hip).
#pragma once

#include "qgemm_x3.h"

namespace pe {

inline int64_t x3_plane_bytes(int64_t m, int64_t k) { return ((m + 31) / 32) * (k / 32) * kX3Block; }
// The block sums follow the planes.
inline float* x3_sums(void* x3, int64_t m, int64_t k) { return (float*)((uint8_t*)x3 + x3_plane_bytes(m, k)); }

inline int x3_weight_ok(int type, int64_t n, int64_t k) {
    if (type != PE_TYPE_Q5_0 && type != PE_TYPE_Q8_0 && type != PE_TYPE_Q4_K && type != PE_TYPE_Q6_K)
        return PE_ERR_TYPE;
    // whole steps of two blocks (Q5_0, Q8_0), whole super-blocks; rows as long as pe_qgemm takes;
    // a row tile's column tiles in one grid
    if (n <= 0 || n > 1 << 28 || k <= 0 || k % (block_elems(type) == 256 ? 256 : 64) || k > 32768) return PE_ERR_SHAPE;
    return PE_OK;
}
// attn_v may differ from attn_q / attn_k within the 32-block or the super-block formats.
inline bool x3_qkv_pair(int t, int tv) { return t == tv || block_elems(t) == block_elems(tv); }

template <int T, int T1, int NT, int WM, int WK, int EPI>
int x3_launch(X3Args p, hipStream_t s) {
    constexpr int R = WM;
    if constexpr (EPI == kX3Plain) p.n_tiles = (int)((p.seg[0].n + 32 * NT - 1) / (32 * NT));
    if constexpr (EPI == kX3Silu) p.n_tiles = (int)((p.out_kb + NT / 2 - 1) / (NT / 2));
    if constexpr (EPI == kX3Qkv) p.n_tiles = (int)((p.seg[0].n + p.seg[1].n + p.seg[2].n) / (32 * NT));
    p.seg[1].tile0 = EPI == kX3Qkv ? (int)(p.seg[0].n / (32 * NT)) : p.n_tiles;
    p.seg[2].tile0 = EPI == kX3Qkv ? (int)((p.seg[0].n + p.seg[1].n) / (32 * NT)) : p.n_tiles;
    const int mt = (p.m + 32 * R - 1) / (32 * R);
    const int64_t blocks = 8LL * ((p.n_tiles + 7) / 8) * mt;
    if (blocks * (64 * WM * WK) > 0xFFFFFFFFLL) return PE_ERR_SHAPE;  // more than one grid holds
    hipLaunchKernelGGL((k_x3<T, T1, NT, WM, WK, EPI>), dim3((unsigned)blocks), dim3(64 * WM * WK), 0, s, p, mt);
    return launch_status();
}

// Tile rules, from sweeps over m 13..511 on the 0.5B and 7B shapes (us per launch, MI355X).
// A launch's 32 x 32 tiles against the 256 CUs decide: few tiles want the K loop split over many
// waves, many tiles want a weight operand decoded once for several row tiles.
//   plain: one tile per workgroup, 8 K shares (896 x 896, m 13: 5.4 against 8.4 for two column
//     tiles); two column tiles once the tiles exceed two per CU, or one per CU with a long K (896 x
//     4864, m 277: 29.0 against 36.1; 3584 x 3584, m 128: 21.4 against 25.6); four row tiles
//     sharing the decode from six tiles per CU (3584 x 3584, m 511: 63.6 against 84.4; at m 277
//     60.7 against 43.0).
//   gate/up: own decode up to 64 rows (2 x 18944 x 3584, m 64: 89.8 against 97.1), two row tiles
//     sharing it beyond (m 128: 151 against 162; 2 x 4864 x 896, m 277: 25.8 against 31.2), four
//     for long prompts at large FFNs (m 511: 521 against 574).
//   Q/K/V: own decode, 4 K shares (54.5 against 59..68 for the others at 7B, m 277; 9.5 at 0.5B).
template <int T>
int x3_plain_t(const X3Args& p, hipStream_t s) {
    const int64_t tiles = (int64_t)((p.m + 31) / 32) * ((p.seg[0].n + 31) / 32);
    if (tiles >= 1536 && p.m >= 128) return x3_launch<T, T, 2, 4, 2, kX3Plain>(p, s);
    if (tiles > 512 || (tiles > 224 && p.kb >= 64)) return x3_launch<T, T, 2, 1, 8, kX3Plain>(p, s);
    return x3_launch<T, T, 1, 1, 8, kX3Plain>(p, s);
}
template <int T>
int x3_silu_t(const X3Args& p, hipStream_t s) {
    if (p.m <= 64) return x3_launch<T, T, 2, 1, 4, kX3Silu>(p, s);
    if (p.m > 400 && p.out_kb >= 256) return x3_launch<T, T, 2, 4, 1, kX3Silu>(p, s);
    return x3_launch<T, T, 2, 2, 2, kX3Silu>(p, s);
}
template <int T, int TV>
int x3_qkv_t(const X3Args& p, hipStream_t s) {
    return x3_launch<T, TV, 2, 1, 4, kX3Qkv>(p, s);
}

#define PE_X3_DECLARE(name)                              \
    int x3_plain_##name(const X3Args& p, hipStream_t s); \
    int x3_silu_##name(const X3Args& p, hipStream_t s);  \
    int x3_qkv_##name(int tv, const X3Args& p, hipStream_t s);
PE_X3_DECLARE(q5_0)
PE_X3_DECLARE(q8_0)
PE_X3_DECLARE(q4_k)
PE_X3_DECLARE(q6_k)
#undef PE_X3_DECLARE

// T: the format; TO: the other format of its family (attn_v's)
#define PE_X3_DEFINE(name, T, TO)                                                                \
    int x3_plain_##name(const X3Args& p, hipStream_t s) { return x3_plain_t<T>(p, s); }          \
    int x3_silu_##name(const X3Args& p, hipStream_t s) { return x3_silu_t<T>(p, s); }            \
    int x3_qkv_##name(int tv, const X3Args& p, hipStream_t s) {                                  \
        return tv == T ? x3_qkv_t<T, T>(p, s) : tv == TO ? x3_qkv_t<T, TO>(p, s) : PE_ERR_TYPE;  \
    }

#define PE_X3_SWITCH(type, call)                 \
    switch (type) {                              \
        case PE_TYPE_Q5_0: return call(q5_0);    \
        case PE_TYPE_Q8_0: return call(q8_0);    \
        case PE_TYPE_Q4_K: return call(q4_k);    \
        case PE_TYPE_Q6_K: return call(q6_k);    \
        default: return PE_ERR_TYPE;             \
    }
inline int x3_plain(int type, const X3Args& p, hipStream_t s) {
#define PE_CALL(f) x3_plain_##f(p, s)
    PE_X3_SWITCH(type, PE_CALL)
#undef PE_CALL
}
inline int x3_silu(int type, const X3Args& p, hipStream_t s) {
#define PE_CALL(f) x3_silu_##f(p, s)
    PE_X3_SWITCH(type, PE_CALL)
#undef PE_CALL
}
inline int x3_qkv(int type, int tv, const X3Args& p, hipStream_t s) {
#define PE_CALL(f) x3_qkv_##f(tv, p, s)
    PE_X3_SWITCH(type, PE_CALL)
#undef PE_CALL
}
#undef PE_X3_SWITCH

}  // namespace pe
