// fp32-grade products of quantized weights on the bf16 matrix cores (the short-prompt prefill).
//
// An fp32 activation is the exact sum of three bf16 values (its 24-bit significand cut into
// 8 + 8 + 8 bits), and the integer code of a Q8_0 / Q5_0 / Q4_K / Q6_K weight is exact in bf16,
// so a block's sum of code x activation is three bf16 MFMA passes whose products are all exact
// and whose sums are fp32; the block's scale is applied to that sum in fp32. Nothing is held or
// multiplied at less than fp32. The matrix cores round their sums downwards, though, not to nearest:
// the scales' signs alternate by block to take the bias out of ordinary rows (codes_bf16). In rows
// whose energy sits in blocks of one parity it stays, below half a unit in the last place of each
// block's sum for each of two additions (measured: mean error 1.4e-7 of the mean result at k =
// 18944 with the other parity's blocks 1000 times smaller, the error in all at most that of the
// dot-product kernel, 1.7e-7). Rows of one sign, whose sums do not cancel: 5.3e-8 against that
// kernel's 4.6e-8 (Q4_K, k = 3584).
//
// Activations travel between kernels in the "x3" form: per 32-row tile and 32-column block,
// 6 KiB = [half of the block][plane hi, mid, lo][lane][8 bf16], lane = row + 32 g, elements
// 16 half + 8 g + 0..7: the A operand of v_mfma_f32_32x32x16_bf16, so a wave loads an operand
// with one contiguous 1 KiB read and no conversion. Rows past m in the last tile are never
// stored to memory by a consumer (row i of A only reaches row i of the product) and may hold
// anything. "xs" holds each row's fp32 sum over every 32-column block, [tile][block / 4][row][4],
// for the minimums of Q4_K (w = a q - m: the second term is m times that sum); it exists when
// the columns are a multiple of 128.
#pragma once

#include <type_traits>

#include "pe_common.h"

namespace pe {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));

constexpr int kX3Block = 6144;  // bytes of one (32-row tile, 32-column block)

// hi + mid + lo = x exactly, each with at most 8 significant bits (truncation: hi never
// overflows); below 2^-110 lo ends at bf16's last bit, 2^-133. An infinity or a NaN stays whole in hi (a NaN whose payload sits in the low bits
// is made quiet).
PE_DEV void split3(float x, uint32_t& h, uint32_t& m, uint32_t& l) {
    const uint32_t u = __float_as_uint(x);
    h = u & 0xFFFF0000u;
    float r = x - __uint_as_float(h);
    if ((u & 0x7F800000u) == 0x7F800000u) {
        h |= (u & 0xFFFFu) ? 0x00400000u : 0u;
        r = 0.f;
    }
    m = __float_as_uint(r) & 0xFFFF0000u;
    l = __float_as_uint(r - __uint_as_float(m));
}

// The upper halves of a (low word) and b (high word).
PE_DEV uint32_t pack_hi(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

// Eight consecutive columns of one row, c8 = their chunk (column / 8), into the x3 form.
PE_DEV void x3_store8(uint8_t* x3, int64_t kb_per_row, int64_t row, int64_t c8, const float* v) {
    uint32_t h[8], m[8], l[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) split3(v[i], h[i], m[i], l[i]);
    uint8_t* p = x3 + ((row >> 5) * kb_per_row + (c8 >> 2)) * kX3Block + ((c8 >> 1) & 1) * 3072 +
                 ((row & 31) + 32 * (c8 & 1)) * 16;
    *reinterpret_cast<u4v*>(p) = u4v{pack_hi(h[0], h[1]), pack_hi(h[2], h[3]), pack_hi(h[4], h[5]), pack_hi(h[6], h[7])};
    *reinterpret_cast<u4v*>(p + 1024) =
        u4v{pack_hi(m[0], m[1]), pack_hi(m[2], m[3]), pack_hi(m[4], m[5]), pack_hi(m[6], m[7])};
    *reinterpret_cast<u4v*>(p + 2048) =
        u4v{pack_hi(l[0], l[1]), pack_hi(l[2], l[3]), pack_hi(l[4], l[5]), pack_hi(l[6], l[7])};
}
// Where the sum of block kb of a row goes.
PE_DEV int64_t xs_index(int64_t kb_per_row, int64_t row, int64_t kb) {
    return (((row >> 5) * (kb_per_row >> 2) + (kb >> 2)) * 32 + (row & 31)) * 4 + (kb & 3);
}

// ---------------------------------------------------------------------------------------
// Weight operands. A step is kBlocks 32-column blocks of the wave's 32 weight rows (lane n =
// lane & 31); g = lane >> 5 picks the 8 columns 16 half + 8 g.. of a block the lane holds. Lane
// (n, g) reads whole 16-byte pieces of block (or chunk) 2 s + g and the two lanes of a row then
// exchange halves (v_permlane32_swap), instead of reading 8-byte pieces.
PE_DEV void swap32(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
PE_DEV u4v gld4(const PE_GLOBAL uint8_t* p) { return *reinterpret_cast<const PE_GLOBAL u4v*>(p); }
PE_DEV u2v gld2(const PE_GLOBAL uint8_t* p) { return *reinterpret_cast<const PE_GLOBAL u2v*>(p); }

// Eight byte codes minus z as bf16 (exact: at most 8 significant bits), negated in odd blocks,
// whose scales are negated too: the bf16 MFMAs' sums round downwards (measured: with every scale
// positive the error grows with the number of blocks), and half of the blocks pulling the other
// way takes the bias out (Q4_K, k = 18944: relative error 1.94e-7 -> 1.13e-7; the
// dot-product kernel's is 1.75e-7).
PE_DEV bf8 codes_bf16(uint32_t a, uint32_t b, float z, bool neg) {
    uint32_t f[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[i] = __float_as_uint(neg ? z - fbyte(a, i) : fbyte(a, i) - z);
        f[4 + i] = __float_as_uint(neg ? z - fbyte(b, i) : fbyte(b, i) - z);
    }
    return __builtin_bit_cast(bf8, u4v{pack_hi(f[0], f[1]), pack_hi(f[2], f[3]), pack_hi(f[4], f[5]), pack_hi(f[6], f[7])});
}

// pin(): what a step's loads brought is used from here on only. Without it the compiler computes
// on the values ahead of the loop's back edge, which waits for the prefetch it has just issued.

PE_DEV float signed_by(int b, float s) { return b & 1 ? -s : s; }

template <int T>
struct W3;

template <>
struct W3<PE_TYPE_Q5_0> {
    static constexpr int kBlocks = 2;
    static constexpr bool kHalfScales = false, kMins = false;
    uint32_t v[4], qh[2], d;
    PE_DEV void load(const Tiled& t, int64_t row, int s, int g) {
        const int64_t blk = row * t.nb + 2 * s, nblk = t.nrows * t.nb;
        const u4v a = gld4(t.base + (blk + g) * 16);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        const u2v q = gld2(t.base + nblk * 16 + blk * 4);
        qh[0] = q.x; qh[1] = q.y;
        d = *reinterpret_cast<const PE_GLOBAL uint32_t*>(t.base + nblk * 20 + blk * 2);
    }
    PE_DEV void prepare() {
        swap32(v[0], v[2]);
        swap32(v[1], v[3]);
    }
    PE_DEV bf8 frag(int b, int half, int g) const {
        const uint32_t bits = __builtin_amdgcn_ubfe(qh[b], 16 * half + 8 * g, 8);
        const uint32_t a = (half ? v[2 * b] >> 4 : v[2 * b]) & 0x0F0F0F0Fu;
        const uint32_t c = (half ? v[2 * b + 1] >> 4 : v[2 * b + 1]) & 0x0F0F0F0Fu;
        return codes_bf16(a | spread4_to_bit4(bits & 15u), c | spread4_to_bit4(bits >> 4), 16.f, b & 1);
    }
    PE_DEV float scale(int b, int) const { return b ? -h2f_fast(d >> 16) : h2f_fast(d & 0xFFFFu); }
    PE_DEV void pin() { asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(qh[0]), "+v"(qh[1]), "+v"(d)); }
};

template <>
struct W3<PE_TYPE_Q8_0> {
    static constexpr int kBlocks = 2;
    static constexpr bool kHalfScales = false, kMins = false;
    uint32_t v[8], d;
    PE_DEV void load(const Tiled& t, int64_t row, int s, int g) {
        const int64_t blk = row * t.nb + 2 * s;
        const u4v a = gld4(t.base + (blk + g) * 32), b = gld4(t.base + (blk + g) * 32 + 16);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        d = *reinterpret_cast<const PE_GLOBAL uint32_t*>(t.base + t.nrows * t.nb * 32 + blk * 2);
    }
    PE_DEV void prepare() {
        swap32(v[0], v[2]);
        swap32(v[1], v[3]);
        swap32(v[4], v[6]);
        swap32(v[5], v[7]);
    }
    PE_DEV bf8 frag(int b, int half, int) const {
        return codes_bf16(v[4 * half + 2 * b] ^ 0x80808080u, v[4 * half + 2 * b + 1] ^ 0x80808080u, 128.f, b & 1);
    }
    PE_DEV float scale(int b, int) const { return b ? -h2f_fast(d >> 16) : h2f_fast(d & 0xFFFFu); }
    PE_DEV void pin() { asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]), "+v"(d)); }
};

// One step = half a super-block (128 columns: 32-byte chunks 2 p, 2 p + 1 of the codes).
template <>
struct W3<PE_TYPE_Q4_K> {
    static constexpr int kBlocks = 4;
    static constexpr bool kHalfScales = false, kMins = true;
    uint32_t v[8], dd, sc, mn;
    u4v hd;
    int hi;
    PE_DEV void load(const Tiled& t, int64_t row, int s, int g) {
        const int64_t blk = row * t.nb + (s >> 1);
        const PE_GLOBAL uint8_t* q = t.base + blk * 128 + 64 * (s & 1) + 32 * g;
        const u4v a = gld4(q), b = gld4(q + 16);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        hd = gld4(t.base + t.nrows * t.nb * 128 + blk * 16);
        hi = s & 1;
    }
    PE_DEV void prepare() {
        // the 6-bit scales and minimums of sub-blocks 4 p .. 4 p + 3, a byte each (k4_scale_min)
        dd = hd.x;
        sc = hi ? (hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u) : hd.y & 0x3F3F3F3Fu;
        mn = hi ? ((hd.w >> 4) & 0x0F0F0F0Fu) | ((hd.z >> 2) & 0x30303030u) : hd.z & 0x3F3F3F3Fu;
        swap32(v[0], v[2]);
        swap32(v[1], v[3]);
        swap32(v[4], v[6]);
        swap32(v[5], v[7]);
    }
    PE_DEV bf8 frag(int b, int half, int) const {
        const uint32_t a = v[4 * half + 2 * (b >> 1)], c = v[4 * half + 2 * (b >> 1) + 1];
        return codes_bf16(((b & 1) ? a >> 4 : a) & 0x0F0F0F0Fu, ((b & 1) ? c >> 4 : c) & 0x0F0F0F0Fu, 8.f, b & 1);
    }
    PE_DEV float scale(int b, int) const { return signed_by(b, h2f_fast(dd & 0xFFFFu) * fbyte(sc, b)); }  // exact
    // a q - m = a (q - 8) - (m - 8 a): codes around zero keep the block sums as small as the
    // result (0..15 codes would round at about three times its magnitude)
    PE_DEV float offset(int b) const { return fmaf(8.f, h2f_fast(dd & 0xFFFFu) * fbyte(sc, b), -(h2f_fast(dd >> 16) * fbyte(mn, b))); }
    PE_DEV void pin() { asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]), "+v"(hd)); }
};

// One step = half a super-block: 64 ql bytes (chunks q & 1), 32 qh bytes, eight scales.
template <>
struct W3<PE_TYPE_Q6_K> {
    static constexpr int kBlocks = 4;
    static constexpr bool kHalfScales = true, kMins = false;
    uint32_t v[8], h[4], sc[2], d;
    PE_DEV void load(const Tiled& t, int64_t row, int s, int g) {
        const int64_t blk = row * t.nb + (s >> 1), nblk = t.nrows * t.nb;
        const int hf = s & 1;
        const PE_GLOBAL uint8_t* q = t.base + blk * 128 + 64 * hf + 32 * g;
        const u4v a = gld4(q), b = gld4(q + 16);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        const PE_GLOBAL uint8_t* qh = t.base + nblk * 128 + blk * 64 + 32 * hf + 8 * g;
        const u2v c = gld2(qh), e = gld2(qh + 16);
        h[0] = c.x; h[1] = c.y; h[2] = e.x; h[3] = e.y;
        const u2v s8 = gld2(t.base + nblk * 192 + blk * 16 + 8 * hf);
        sc[0] = s8.x; sc[1] = s8.y;
        d = *reinterpret_cast<const PE_GLOBAL uint16_t*>(t.base + nblk * 208 + blk * 2);
    }
    PE_DEV void prepare() {
        swap32(v[0], v[2]);
        swap32(v[1], v[3]);
        swap32(v[4], v[6]);
        swap32(v[5], v[7]);
    }
    PE_DEV uint32_t code(uint32_t l, uint32_t hi, int b) const {
        const uint32_t top = b < 2 ? hi << (4 - 2 * b) : hi >> (2 * b - 4);
        return ((b >= 2 ? l >> 4 : l) & 0x0F0F0F0Fu) | (top & 0x30303030u);
    }
    PE_DEV bf8 frag(int b, int half, int) const {
        const int i = 4 * half + 2 * (b & 1);
        return codes_bf16(code(v[i], h[2 * half], b), code(v[i + 1], h[2 * half + 1], b), 32.f, b & 1);
    }
    PE_DEV float scale(int b, int half) const {  // exact: 11-bit x 8-bit
        return signed_by(b, h2f_fast(d) * (float)sext8(sc[b >> 1], 2 * (b & 1) + half));
    }
    PE_DEV void pin() { asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]), "+v"(h[0]), "+v"(h[1]), "+v"(h[2]), "+v"(h[3]), "+v"(sc[0]), "+v"(sc[1]), "+v"(d)); }
};

// ---------------------------------------------------------------------------------------
enum { kX3Plain = 0, kX3Silu = 1, kX3Qkv = 2 };

struct X3Seg {
    Tiled w;
    int64_t n;          // rows (kX3Silu: ffn, the gate rows; the up rows follow them)
    int tile0;          // first column tile of the segment
    const float* bias;  // or null
};

struct X3Args {
    const uint8_t* a;  // x3 activations, kb blocks per row
    const float* xs;
    int m, kb, n_tiles;
    X3Seg seg[3];
    // kX3Plain: y[m][n] = acc + bias + res
    const float* res;
    int64_t res_stride;
    float* y;
    int64_t y_stride;
    // kX3Silu: silu(gate) * up in the x3 form (out_kb blocks per row) and its block sums
    uint8_t* out3;
    float* out_xs;
    int out_kb;
    // kX3Qkv: segments q, k, v; heads of hd, rotation pairs (j, j + hd / 2)
    const float *cos_rows, *sin_rows;
    float *q_out, *k_cache, *v_cache;
    int64_t capacity, pos0;
    int n_head, hd;
};

// One 32-column block of a 32 x 32 tile: in (+)= scale * (codes . activations), af = the block's
// six activation operands. Small planes first: only the last additions round at the magnitude
// of the block's sum.
template <bool HALF>
PE_DEV void x3_block(const u4v (&af)[6], bf8 w0, bf8 w1, float s0, float s1, bool first, f16v& in) {
    auto op = [&](int f) { return __builtin_bit_cast(bf8, af[f]); };
    f16v c = {};
    if constexpr (HALF) {
        f16v e = {};
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op(2), w0, c, 0, 0, 0);
        e = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op(5), w1, e, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op(1), w0, c, 0, 0, 0);
        e = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op(4), w1, e, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op(0), w0, c, 0, 0, 0);
        e = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op(3), w1, e, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; ++r) in[r] = fmaf(s1, e[r], first ? s0 * c[r] : fmaf(s0, c[r], in[r]));
    } else {
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op(2), w0, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op(5), w1, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op(1), w0, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op(4), w1, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op(0), w0, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op(3), w1, c, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; ++r) in[r] = first ? s0 * c[r] : fmaf(s0, c[r], in[r]);
    }
}

// The Q4_K offsets of two blocks times the rows' block sums, both cut into three bf16 planes, as
// one 16-column MFMA: columns (plane pair, block) = hh, mh, lh, hl | hm, mm, 0, 0.
PE_DEV bf8 x3_min_a(float x0, float x1, int g) {
    uint32_t h[2], m[2], l[2];
    split3(x0, h[0], m[0], l[0]);
    split3(x1, h[1], m[1], l[1]);
    const uint32_t hp = pack_hi(h[0], h[1]), mp = pack_hi(m[0], m[1]), lp = pack_hi(l[0], l[1]);
    return __builtin_bit_cast(bf8, u4v{hp, mp, g ? 0u : lp, g ? 0u : hp});
}
PE_DEV bf8 x3_min_b(float o0, float o1, int g) {
    uint32_t h[2], m[2], l[2];
    split3(o0, h[0], m[0], l[0]);
    split3(o1, h[1], m[1], l[1]);
    const uint32_t hp = pack_hi(h[0], h[1]), mp = pack_hi(m[0], m[1]), lp = pack_hi(l[0], l[1]);
    return __builtin_bit_cast(bf8, g ? u4v{mp, mp, 0u, 0u} : u4v{hp, hp, hp, lp});
}

// The wave's share of the K loop, every wave decoding for itself: steps [s0, s1) of its row tile
// rt and NT column tiles.
template <int T, int NT>
PE_DEV void x3_loop(const X3Args& p, const Tiled& w, const int64_t (&row)[NT], int rt, int s0, int s1, int lane,
                    f16v (&acc)[NT]) {
    constexpr int B = W3<T>::kBlocks;
    const int g = lane >> 5;
    if (s0 >= s1) return;
    const PE_GLOBAL uint8_t* const ap = (const PE_GLOBAL uint8_t*)p.a + (int64_t)rt * p.kb * kX3Block + lane * 16;
    const PE_GLOBAL uint8_t* const xp = (const PE_GLOBAL uint8_t*)p.xs + (int64_t)rt * (p.kb >> 2) * 512 + (lane & 31) * 16;
    W3<T> raw[NT], nxt[NT];
    u4v xv[2];
    auto fetch = [&](int s) {
        s = s < s1 ? s : s1 - 1;
#pragma unroll
        for (int j = 0; j < NT; ++j) nxt[j].load(w, row[j], s, g);
        if constexpr (W3<T>::kMins) xv[1] = gld4(xp + s * 512);
    };
    fetch(s0);
    for (int s = s0; s < s1; ++s) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            nxt[j].pin();
            raw[j] = nxt[j];
            raw[j].prepare();
        }
        xv[0] = xv[1];
        fetch(s + 1);
        // the step's own sums, added to the tile's once per step: a K-long chain of additions
        // rounds at the full sum every time
        f16v in[NT];
        if constexpr (W3<T>::kMins) {
            const bf8 a0 = x3_min_a(__uint_as_float(xv[0].x), __uint_as_float(xv[0].y), g);
            const bf8 a1 = x3_min_a(__uint_as_float(xv[0].z), __uint_as_float(xv[0].w), g);
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                in[j] = f16v{};
                in[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, x3_min_b(raw[j].offset(0), raw[j].offset(1), g), in[j], 0, 0, 0);
                in[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, x3_min_b(raw[j].offset(2), raw[j].offset(3), g), in[j], 0, 0, 0);
            }
        }
#pragma unroll
        for (int b0 = 0; b0 < B; b0 += 2) {
            u4v af[2][6];
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int f = 0; f < 6; ++f) af[b][f] = gld4(ap + (int64_t)(s * B + b0 + b) * kX3Block + f * 1024);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int b = b0; b < b0 + 2; ++b)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    x3_block<W3<T>::kHalfScales>(af[b - b0], raw[j].frag(b, 0, g), raw[j].frag(b, 1, g), raw[j].scale(b, 0),
                                                 W3<T>::kHalfScales ? raw[j].scale(b, 1) : 0.f, b == 0 && !W3<T>::kMins,
                                                 in[j]);
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[j] += in[j];
    }
}

// What one wave decodes for the shared loop: half of every block (16 columns) of 32 weight rows,
// a step at a time.
template <int T>
struct W3Half;

template <>
struct W3Half<PE_TYPE_Q5_0> {
    uint32_t v[4], qh[2], d;
    PE_DEV void load(const Tiled& t, int64_t row, int s, int g, int half) {
        const int64_t blk = row * t.nb + 2 * s, nblk = t.nrows * t.nb;
        const u4v a = gld4(t.base + (blk + g) * 16);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        const u2v q = gld2(t.base + nblk * 16 + blk * 4);
        qh[0] = q.x; qh[1] = q.y;
        d = *reinterpret_cast<const PE_GLOBAL uint32_t*>(t.base + nblk * 20 + blk * 2);
    }
    PE_DEV void prepare() {
        swap32(v[0], v[2]);
        swap32(v[1], v[3]);
    }
    PE_DEV bf8 frag(int b, int half, int g) const {
        const uint32_t bits = qh[b] >> (16 * half + 8 * g);
        const uint32_t a = (v[2 * b] >> (4 * half)) & 0x0F0F0F0Fu, c = (v[2 * b + 1] >> (4 * half)) & 0x0F0F0F0Fu;
        return codes_bf16(a | spread4_to_bit4(bits & 15u), c | spread4_to_bit4((bits >> 4) & 15u), 16.f, b & 1);
    }
    PE_DEV float scale(int b) const { return b ? -h2f_fast(d >> 16) : h2f_fast(d & 0xFFFFu); }
    PE_DEV void pin() { asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(qh[0]), "+v"(qh[1]), "+v"(d)); }
};

template <>
struct W3Half<PE_TYPE_Q8_0> {
    uint32_t v[4], d;
    PE_DEV void load(const Tiled& t, int64_t row, int s, int g, int half) {
        const int64_t blk = row * t.nb + 2 * s;
        const u4v a = gld4(t.base + (blk + g) * 32 + 16 * half);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        d = *reinterpret_cast<const PE_GLOBAL uint32_t*>(t.base + t.nrows * t.nb * 32 + blk * 2);
    }
    PE_DEV void prepare() {
        swap32(v[0], v[2]);
        swap32(v[1], v[3]);
    }
    PE_DEV bf8 frag(int b, int, int) const {
        return codes_bf16(v[2 * b] ^ 0x80808080u, v[2 * b + 1] ^ 0x80808080u, 128.f, b & 1);
    }
    PE_DEV float scale(int b) const { return b ? -h2f_fast(d >> 16) : h2f_fast(d & 0xFFFFu); }
    PE_DEV void pin() { asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(d)); }
};

template <>
struct W3Half<PE_TYPE_Q4_K> {
    uint32_t v[4];
    u4v h;
    uint32_t sc, mn;
    int hi;
    PE_DEV void load(const Tiled& t, int64_t row, int s, int g, int half) {
        const int64_t blk = row * t.nb + (s >> 1);
        const u4v a = gld4(t.base + blk * 128 + 64 * (s & 1) + 32 * g + 16 * half);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        h = gld4(t.base + t.nrows * t.nb * 128 + blk * 16);
        hi = s & 1;
    }
    PE_DEV void prepare() {
        sc = hi ? (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u) : h.y & 0x3F3F3F3Fu;
        mn = hi ? ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u) : h.z & 0x3F3F3F3Fu;
        swap32(v[0], v[2]);
        swap32(v[1], v[3]);
    }
    PE_DEV bf8 frag(int b, int, int) const {
        const uint32_t a = v[2 * (b >> 1)], c = v[2 * (b >> 1) + 1];
        return codes_bf16(((b & 1) ? a >> 4 : a) & 0x0F0F0F0Fu, ((b & 1) ? c >> 4 : c) & 0x0F0F0F0Fu, 8.f, b & 1);
    }
    PE_DEV float scale(int b) const { return signed_by(b, h2f_fast(h.x & 0xFFFFu) * fbyte(sc, b)); }
    PE_DEV float offset(int b) const { return fmaf(8.f, h2f_fast(h.x & 0xFFFFu) * fbyte(sc, b), -(h2f_fast(h.x >> 16) * fbyte(mn, b))); }
    PE_DEV void pin() { asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(h)); }
};

template <>
struct W3Half<PE_TYPE_Q6_K> {
    uint32_t v[4], c[2], s8[2], d;
    int hf_;
    PE_DEV void load(const Tiled& t, int64_t row, int s, int g, int half) {
        const int64_t blk = row * t.nb + (s >> 1), nblk = t.nrows * t.nb;
        const int hf = s & 1;
        const u4v a = gld4(t.base + blk * 128 + 64 * hf + 32 * g + 16 * half);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        const u2v q = gld2(t.base + nblk * 128 + blk * 64 + 32 * hf + 16 * half + 8 * g);
        c[0] = q.x; c[1] = q.y;
        const u2v e = gld2(t.base + nblk * 192 + blk * 16 + 8 * hf);
        s8[0] = e.x; s8[1] = e.y;
        d = *reinterpret_cast<const PE_GLOBAL uint16_t*>(t.base + nblk * 208 + blk * 2);
        hf_ = half;
    }
    PE_DEV void prepare() {
        swap32(v[0], v[2]);
        swap32(v[1], v[3]);
    }
    PE_DEV uint32_t code(uint32_t l, uint32_t hi, int b) const {
        const uint32_t top = b < 2 ? hi << (4 - 2 * b) : hi >> (2 * b - 4);
        return ((b >= 2 ? l >> 4 : l) & 0x0F0F0F0Fu) | (top & 0x30303030u);
    }
    PE_DEV bf8 frag(int b, int, int) const {
        const int i = 2 * (b & 1);
        return codes_bf16(code(v[i], c[0], b), code(v[i + 1], c[1], b), 32.f, b & 1);
    }
    PE_DEV float scale(int b) const {  // of this half
        return signed_by(b, h2f_fast(d) * (float)(int8_t)(s8[b >> 1] >> (16 * (b & 1) + 8 * hf_)));
    }
    PE_DEV void pin() { asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(c[0]), "+v"(c[1]), "+v"(s8[0]), "+v"(s8[1]), "+v"(d)); }
};

// The K loop of a workgroup with WM waves in each K share: a wave multiplies its own row tile with
// the two column tiles. The weights are decoded once per workgroup, two blocks
// (a sub-step) at a time, into bf16 operands in LDS (double-buffered, one barrier per sub-step)
// while the previous sub-step is multiplied: a decode costs about as many VALU cycles as one row
// tile's MFMAs take, so sharing it is what lets the matrix cores run. The activations are each
// wave's own and come straight from memory, a sub-step ahead. A sub-step runs as four stages
// (block, column tile): six MFMAs, the scaling of the previous stage's sums and a quarter of the
// decode, fenced so that the scheduler overlaps them and keeps the loads in front.
template <int T>
struct X3Lds {  // of two column tiles
    static constexpr int kFrag = 2 * 4096, kScale = 2 * 512, kMin = W3<T>::kMins ? 2 * 1024 : 0;
    static constexpr int kBuf = kFrag + kScale + kMin;
};

template <int T, int WM, int WK>
PE_DEV void x3_loop_shared(const X3Args& p, const Tiled& w, const int64_t (&row)[2], int rt, int wm, int wk,
                           uint8_t* lds, int lane, f16v (&acc)[2]) {
    constexpr int TU = 4 / WM;  // (column tile, half) units a wave decodes
    static_assert(WM == 2 || WM == 4, "four units spread over the waves");
    using L = X3Lds<T>;
    constexpr int SB = W3<T>::kBlocks / 2;
    const int g = lane >> 5, n = lane & 31;
    const int steps = p.kb / W3<T>::kBlocks;
    const int s0 = steps * wk / WK, s1 = steps * (wk + 1) / WK;
    const int nsub = (steps + WK - 1) / WK * SB;  // the longest share: every wave meets every barrier
    const int mine = (s1 - s0) * SB;
    uint8_t* const base = lds + wk * 2 * L::kBuf;
    const PE_GLOBAL uint8_t* ap = (const PE_GLOBAL uint8_t*)p.a + ((int64_t)rt * p.kb + s0 * W3<T>::kBlocks) * kX3Block + lane * 16;
    const PE_GLOBAL uint8_t* const xp = (const PE_GLOBAL uint8_t*)p.xs + (int64_t)rt * (p.kb >> 2) * 512 + n * 16;
    const int kb0 = s0 * W3<T>::kBlocks;
    // this wave's units: TU == 2: both halves of one tile, else one half
    const int ut = TU == 2 ? wm : wm >> 1, uh = TU == 2 ? 0 : wm & 1;
    int64_t wrow = row[0];
    if (ut == 1) wrow = row[1];  // (a select of the two would put the array into LDS)
    W3Half<T> raw[TU], nxt[TU];
    auto fetch = [&](int s) {
        s = s < s1 ? s : s1 - 1;
#pragma unroll
        for (int t = 0; t < TU; ++t) nxt[t].load(w, wrow, s, g, uh + t);
    };
    auto take = [&] {  // the fetched step becomes the current one
#pragma unroll
        for (int t = 0; t < TU; ++t) {
            nxt[t].pin();
            raw[t] = nxt[t];
            raw[t].prepare();
        }
    };
    // part q (0..3) of the decode of sub-step SUB of raw into buffer buf
    auto decode = [&](auto sub, auto part, int buf) {
        constexpr int S2 = 2 * decltype(sub)::value, Q = decltype(part)::value;
        uint8_t* const o = base + buf * L::kBuf;
        auto one = [&](int t, int b) {
            const int half = uh + t;
            *reinterpret_cast<u4v*>(o + ((ut * 2 + b) * 2 + half) * 1024 + lane * 16) =
                __builtin_bit_cast(u4v, raw[t].frag(S2 + b, half, g));
            if (W3<T>::kHalfScales || half == 0) {  // one scale per row: half a wave writes
                if (g == 0) reinterpret_cast<float*>(o + L::kFrag)[((ut * 2 + b) * 2 + half) * 32 + n] = raw[t].scale(S2 + b);
            }
        };
        if constexpr (TU == 2) {
            one(Q >> 1, Q & 1);
        } else if constexpr (Q < 2) {
            one(0, Q);
        }
        if constexpr (W3<T>::kMins) {
            if (Q == 3 && uh == 0)
                *reinterpret_cast<u4v*>(o + L::kFrag + L::kScale + ut * 1024 + lane * 16) =
                    __builtin_bit_cast(u4v, x3_min_b(raw[0].offset(S2), raw[0].offset(S2 + 1), g));
        }
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    if (mine > 0) {
        fetch(s0);
        take();
        fetch(s0 + 1);
        decode(I0{}, I0{}, 0);
        decode(I0{}, I1{}, 0);
        decode(I0{}, I2{}, 0);
        decode(I0{}, I3{}, 0);
    }
    f16v in[2];
    auto body = [&](auto par, int i) {
        constexpr int P = decltype(par)::value & 1;
        constexpr bool kFirst = decltype(par)::value == 0;
        __syncthreads();
        if (i >= mine) return;
        // decode of the next sub-step (past the end: a repeat nobody reads)
        using NS = std::conditional_t<SB == 2 && P == 0, I1, I0>;
        constexpr bool kTake = SB == 1 || P == 1;
        u4v af[2][6];
        float xs[2];
        const PE_GLOBAL uint8_t* const ab = ap + (int64_t)i * 2 * kX3Block;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
#pragma unroll
            for (int f = 0; f < 6; ++f) af[b][f] = gld4(ab + b * kX3Block + f * 1024);
            if constexpr (W3<T>::kMins) {
                const int kb = kb0 + 2 * i + b;
                xs[b] = *reinterpret_cast<const PE_GLOBAL float*>(xp + (kb >> 2) * 512 + (kb & 3) * 4);
            }
        }
        if constexpr (kTake) {
            take();
            fetch(SB == 1 ? s0 + i + 2 : s0 + (i + 1) / 2 + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        decode(NS{}, I0{}, 1 - P);
        decode(NS{}, I1{}, 1 - P);
        decode(NS{}, I2{}, 1 - P);
        decode(NS{}, I3{}, 1 - P);
        const uint8_t* const o = base + P * L::kBuf;
        const uint8_t* const fr = o + lane * 16;
        const float* const sc = reinterpret_cast<const float*>(o + L::kFrag) + n;
        if constexpr (W3<T>::kMins) {
            const bf8 ma = x3_min_a(xs[0], xs[1], g);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const bf8 mb = __builtin_bit_cast(bf8, *reinterpret_cast<const u4v*>(
                    o + L::kFrag + L::kScale + j * 1024 + lane * 16));
                if constexpr (kFirst) in[j] = f16v{};
                in[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ma, mb, in[j], 0, 0, 0);
            }
        }
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const bf8 w0 = __builtin_bit_cast(bf8, *reinterpret_cast<const u4v*>(fr + ((j * 2 + b) * 2) * 1024));
                const bf8 w1 = __builtin_bit_cast(bf8, *reinterpret_cast<const u4v*>(fr + ((j * 2 + b) * 2 + 1) * 1024));
                x3_block<W3<T>::kHalfScales>(af[b], w0, w1, sc[(j * 2 + b) * 64],
                                             W3<T>::kHalfScales ? sc[(j * 2 + b) * 64 + 32] : 0.f,
                                             kFirst && b == 0 && !W3<T>::kMins, in[j]);
            }
        if (decltype(par)::value == 3 || i + 1 >= mine) {  // every eight blocks: short chains of additions
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[j] += in[j];
        }
    };
    for (int i = 0; i < nsub; i += 4) {
        body(I0{}, i);
        if (i + 1 < nsub) body(I1{}, i + 1);
        if (i + 2 < nsub) body(I2{}, i + 2);
        if (i + 3 < nsub) body(I3{}, i + 3);
    }
}

// One element of the product from the dequantized fp32 weights, as the dot-product kernel forms it.
template <int T>
PE_DEV float x3_dot(const X3Args& p, const Tiled& w, int64_t row, int64_t m) {
    const PE_GLOBAL uint8_t* a = (const PE_GLOBAL uint8_t*)p.a + (m >> 5) * p.kb * kX3Block + (m & 31) * 16;
    float acc = 0.f;
#pragma unroll 1
    for (int u = 0; u < p.kb && acc == acc; ++u) {  // a NaN stays one
        typename Fmt<T>::Raw r;
        Fmt<T>::load(w, row, u, r);
        float wv[32];
        Fmt<T>::dequant(r, wv);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const PE_GLOBAL uint8_t* q = a + (int64_t)u * kX3Block + (c >> 1) * 3072 + (c & 1) * 512;
            const u4v h = gld4(q), md = gld4(q + 1024), l = gld4(q + 2048);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const auto part = [&](const u4v& v) {
                    return __uint_as_float(i & 1 ? v[i >> 1] & 0xFFFF0000u : v[i >> 1] << 16);
                };
                acc = fmaf(wv[8 * c + i], (part(h) + part(md)) + part(l), acc);
            }
        }
    }
    return acc;
}

// Whether any of the eight is an infinity or a NaN.
PE_DEV bool x3_odd8(const float* v) {
    float z = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) z = fmaf(v[i], 0.f, z);
    return z != 0.f;
}

// Elements of v (weight rows n .. n + 7) and, for PAIR, u (rows n + gap ..) that are not finite,
// formed again by x3_dot: a block's sum of codes and activations is larger than the product (by the
// reciprocal of the scale) and may overflow where the product does not, and Q4_K's two terms turn
// an infinite activation into inf - inf.
template <int T, int T1, bool PAIR>
PE_DEV void x3_mend(const X3Args& p, const Tiled& w, bool last, int64_t n, int64_t gap, int64_t m, float* v, float* u) {
#pragma unroll 1
    for (int j = 0; j < (PAIR ? 16 : 8); ++j) {
        float e = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) e = j == i ? v[i] : PAIR && j == 8 + i ? u[i] : e;
        const int64_t row = n + (j & 7) + (j < 8 ? 0 : gap);
        if ((__float_as_uint(e) & 0x7F800000u) != 0x7F800000u || row >= w.nrows) continue;
        e = T1 != T && last ? x3_dot<T1>(p, w, row, m) : x3_dot<T>(p, w, row, m);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[i] = j == i ? e : v[i];
            if (PAIR) u[i] = j == 8 + i ? e : u[i];
        }
    }
}

// One workgroup: a 32 MT x 32 NT tile of the product whose K steps are divided over WK waves
// (a launch at prompt sizes has few tiles and long rows: the split keeps the chip's SIMDs busy
// and each wave's chain of loads short). The waves' partial tiles meet in LDS and are added in
// wave order, so the result does not depend on timing. Workgroups of the same weight rows run
// on one XCD (its L2 then reads the weights once).
// T1 is the format of the last segment where it differs (attn_v beside attn_q and attn_k).
constexpr int x3_max(int a, int b) { return a > b ? a : b; }

template <int T, int T1, int NT, int WM, int WK, int EPI>
__global__ __launch_bounds__(64 * WM * WK, 2) void k_x3(X3Args p, int m_tiles) {
    constexpr bool kShared = WM > 1;
    static_assert(!kShared || NT == 2, "column tiles of the workgroup");
    constexpr int R = WM;            // row tiles of the workgroup
    constexpr int LS = 32 * NT + 8;  // row stride of the partial tiles: rows 4 apart land 32 banks apart
    constexpr int kPart = WK * 32 * R * LS * 4;
    constexpr int kLoop = !kShared ? 0 : WK * 2 * x3_max(X3Lds<T>::kBuf, X3Lds<T1>::kBuf);
    __shared__ __attribute__((aligned(16))) uint8_t lds[x3_max(kPart, kLoop)];
    auto part = reinterpret_cast<float(*)[32 * R][LS]>(lds);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wk = wave / WM, wm = wave % WM;
    const int local = blockIdx.x >> 3;
    const int ct = (blockIdx.x & 7) + 8 * (local / m_tiles);
    if (ct >= p.n_tiles) return;
    const int rt0 = (local % m_tiles) * R;
    int si = 0;
    if constexpr (EPI != kX3Silu) si = ct < p.seg[1].tile0 ? 0 : ct < p.seg[2].tile0 ? 1 : 2;
    const X3Seg sg = p.seg[si];
    const int t = ct - sg.tile0;
    // kX3Silu and kX3Qkv take weight rows in pairs of 32: gate and up rows of the same columns,
    // the two halves of 32 rotation pairs of a head (hd / 64 such pairs per head)
    const int64_t gap = EPI == kX3Silu ? sg.n : EPI == kX3Qkv ? p.hd >> 1 : 32;
    auto pair_row = [&](int q) -> int64_t {
        const int pr = t * (NT / 2) + q;
        if constexpr (EPI == kX3Qkv) return (int64_t)(pr / (p.hd >> 6)) * p.hd + 32 * (pr % (p.hd >> 6));
        return 32 * (int64_t)pr;
    };
    const int64_t n0 = 32 * (int64_t)NT * t;  // kX3Plain: the first row
    int64_t row[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        row[j] = (EPI == kX3Plain ? n0 + j * 32 : pair_row(j >> 1) + (j & 1) * gap) + (lane & 31);
        if (row[j] >= sg.w.nrows) row[j] = sg.w.nrows - 1;
    }
    f16v acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = f16v{};
    auto loop = [&](auto tag) {
        constexpr int TT = decltype(tag)::value;
        const int rt_last = (p.m - 1) >> 5;
        if constexpr (!kShared) {
            const int steps = p.kb / W3<TT>::kBlocks;
            x3_loop<TT, NT>(p, sg.w, row, rt0, steps * wk / WK, steps * (wk + 1) / WK, lane, acc);
        } else {
            x3_loop_shared<TT, WM, WK>(p, sg.w, row, rt0 + wm < rt_last ? rt0 + wm : rt_last, wm, wk, lds, lane, acc);
            __syncthreads();  // the partial tiles reuse the operands' LDS
        }
    };
    if constexpr (T1 != T) {
        if (si == 2) loop(std::integral_constant<int, T1>{});
        else loop(std::integral_constant<int, T>{});
    } else {
        loop(std::integral_constant<int, T>{});
    }
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            part[wk][32 * wm + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)][32 * j + (lane & 31)] = acc[j][r];
    __syncthreads();
    // items: (row, 8 columns), the columns fastest
    constexpr int CH = EPI == kX3Plain ? 4 * NT : 2 * NT;
    for (int it = threadIdx.x; it < 32 * R * CH; it += 64 * WM * WK) {
        const int lr = it / CH, c = 8 * (it % CH);
        const int64_t m = (int64_t)rt0 * 32 + lr;
        if ((m >> 5) > ((p.m - 1) >> 5)) continue;  // a whole tile past the rows
        auto sum8 = [&](int col, float* v) {
#pragma unroll
            for (int i = 0; i < 8; i += 4) {
                float4 a = *reinterpret_cast<const float4*>(&part[0][lr][col + i]);
#pragma unroll
                for (int q = 1; q < WK; ++q) {
                    const float4 b = *reinterpret_cast<const float4*>(&part[q][lr][col + i]);
                    a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
                }
                v[i] = a.x; v[i + 1] = a.y; v[i + 2] = a.z; v[i + 3] = a.w;
            }
        };
        if constexpr (EPI == kX3Plain) {
            if (m >= p.m) continue;
            float v[8];
            sum8(c, v);
            const int64_t n = n0 + c;
            if (__builtin_expect(x3_odd8(v), 0)) x3_mend<T, T1, false>(p, sg.w, false, n, 0, m, v, nullptr);
            float* yp = p.y + m * p.y_stride + n;
            const float* rp = p.res ? p.res + m * p.res_stride + n : nullptr;
            const float* bp = sg.bias ? sg.bias + n : nullptr;
            if (n + 8 <= sg.n && !(((uintptr_t)yp | (uintptr_t)rp | (uintptr_t)bp) & 15)) {
                float4 b0 = {}, b1 = {}, r0 = {}, r1 = {};
                if (bp) {
                    b0 = *reinterpret_cast<const float4*>(bp);
                    b1 = *reinterpret_cast<const float4*>(bp + 4);
                }
                if (rp) {
                    r0 = *reinterpret_cast<const float4*>(rp);
                    r1 = *reinterpret_cast<const float4*>(rp + 4);
                }
                *reinterpret_cast<float4*>(yp) = make_float4(r0.x + (v[0] + b0.x), r0.y + (v[1] + b0.y),
                                                             r0.z + (v[2] + b0.z), r0.w + (v[3] + b0.w));
                *reinterpret_cast<float4*>(yp + 4) = make_float4(r1.x + (v[4] + b1.x), r1.y + (v[5] + b1.y),
                                                                 r1.z + (v[6] + b1.z), r1.w + (v[7] + b1.w));
            } else {
                for (int i = 0; i < 8; ++i)
                    if (n + i < sg.n) yp[i] = (rp ? rp[i] : 0.f) + (v[i] + (bp ? bp[i] : 0.f));
            }
        } else {
            const int pq = c >> 5, cc8 = c & 31;  // the pair and its column
            float v[8], u[8];
            sum8(64 * pq + cc8, v);
            sum8(64 * pq + 32 + cc8, u);
            const int64_t n = pair_row(pq) + cc8;
            // (rows past the last hold anything)
            if (__builtin_expect((x3_odd8(v) | x3_odd8(u)) && m < p.m, 0))
                x3_mend<T, T1, true>(p, sg.w, si == 2, n, gap, m, v, u);
            if constexpr (EPI == kX3Silu) {
                const int64_t ob = t * (NT / 2) + pq;  // the output's 32-column block
                if (ob >= p.out_kb) continue;
                float s = 0.f;
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = silu_mul_prefill(v[i], u[i]);
#pragma unroll
                for (int i = 0; i < 8; ++i) s += v[i];
                if (p.out_xs) {  // the four lanes of a row add their parts of the block sum
                    s += dpp_mov<0xB1>(s);
                    s += dpp_mov<0x4E>(s);
                    if (cc8 == 0) p.out_xs[xs_index(p.out_kb, m, ob)] = s;
                }
                x3_store8(p.out3, p.out_kb, m, 4 * ob + (cc8 >> 3), v);
            } else {
                if (m >= p.m) continue;
                if (sg.bias) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        v[i] += sg.bias[n + i];
                        u[i] += sg.bias[n + gap + i];
                    }
                }
                const int head = (int)(n / p.hd), d0 = (int)(n - (int64_t)head * p.hd);
                if (si < 2) {
                    const float* cr = p.cos_rows + m * gap + d0;
                    const float* sr = p.sin_rows + m * gap + d0;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const float x1 = v[i], x2 = u[i], co = cr[i], si_ = sr[i];
                        v[i] = x1 * co - x2 * si_;
                        u[i] = x1 * si_ + x2 * co;
                    }
                }
                float* base = si == 0 ? p.q_out + (m * p.n_head + head) * p.hd
                                      : (si == 1 ? p.k_cache : p.v_cache) + ((int64_t)head * p.capacity + p.pos0 + m) * p.hd;
                float* o = base + d0;
                *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
                *reinterpret_cast<float4*>(o + 4) = make_float4(v[4], v[5], v[6], v[7]);
                o += gap;
                *reinterpret_cast<float4*>(o) = make_float4(u[0], u[1], u[2], u[3]);
                *reinterpret_cast<float4*>(o + 4) = make_float4(u[4], u[5], u[6], u[7]);
            }
        }
    }
}

}  // namespace pe
