// fp32 causal attention of the prefill on the fp32 matrix cores (v_mfma_f32_32x32x2_f32: fp32
// operands, products and sums, nothing is rounded to fewer bits). Replaces the SDPA of
// model.py:201-209 on the fp32 path; pe_prefill_attn (attn.hip) keeps the general kernel for
// operands that are not 16-byte aligned.
//
// One workgroup per (32 queries, query head); its four waves take the 32-key tiles t, t + 4, ..
// and merge their partial softmaxes at the end, so that short prompts (few query tiles) still use
// four SIMDs per tile. A wave works alone on its tiles: K and V come into its own LDS with
// direct-to-LDS loads, V while the scores are formed, the next K during the softmax and the
// P V products, with no barrier in the loop. Scores are formed transposed (keys x queries), so a
// query's scores sit in one lane pair and P^T is the second product's operand as it stands.
// Bound by each wave's chain of load, product, softmax and product, which little runs beside: at
// head size 128 a workgroup's K and V tiles take 128 KiB of LDS, so a CU holds one workgroup and a
// SIMD one wave. 28/4 heads of 128 at 1537 tokens in the model's prefill: 2823 -> 262 us, 16.9 GFLOP
// of keys that are seen, 65 TFLOP/s of the fp32 matrix cores' 157; 14/2 heads of 64 at 277 tokens:
// 46.7 -> 15.3 us (before: one workgroup per query and head on the vector ALU).
#include "qgemm_x3_launch.h"

namespace pe {

constexpr int kPaWaves = 4;

struct PaArgs {
    const float* q;
    int64_t q_stride;
    const float* k;
    const float* v;
    int group, n_head;
    int64_t capacity, pos0;
    int L;
    float scale;
    float* out;  // fp32 rows, or
    int64_t out_stride;
    _Float16* out16;  // fp16 rows (the o-projection's operand), or
    uint8_t* x3;  // the x3 form of the rows (columns n_head * HD) and its block sums
    float* sums;
};

// 16 bytes per lane from global g into LDS at m0 + 16 lane (one wave instruction: 1 KB)
PE_DEV void pa_load16(const void* g, uint32_t m0) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(m0) : "memory", "m0");
}
template <int N>
PE_DEV void pa_wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
PE_DEV void pa_wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// LDS image of a 32-row tile: row r's 16-byte chunk c sits at chunk position c ^ (r & 7) (eight
// rows read at one chunk then cover eight chunk positions of the banks).
template <int HD>
PE_DEV void pa_stage(const float* base, int row0, int last, uint32_t lds, int lane) {
    constexpr int C = HD / 4;
#pragma unroll
    for (int f = 0; f < HD / 8; ++f) {
        const int slot = f * 64 + lane, r = slot / C, c = (slot % C) ^ (r & 7);
        const int row = row0 + r < last ? row0 + r : last;  // past the keys: the last one again (masked)
        pa_load16(base + (int64_t)row * HD + 4 * c, __builtin_amdgcn_readfirstlane(lds + f * 1024));
    }
}

template <int HD>
__global__ __launch_bounds__(64 * kPaWaves) void k_prefill_attn_mfma(PaArgs p) {
    constexpr int kTile = 32 * HD * 4, D = HD / 32, OS = HD + 4;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kPaWaves][2 * kTile];
    __shared__ float ml[kPaWaves][2][32];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 5, li = lane & 31;
    const int head = blockIdx.x;
    const int q0 = 32 * (gridDim.y - 1 - blockIdx.y);  // the queries with the most keys first
    const int ql = q0 + li < p.L ? q0 + li : p.L - 1;
    const int64_t qpos = p.pos0 + ql;
    const int q_last = q0 + 31 < p.L ? q0 + 31 : p.L - 1;
    const int last = (int)(p.pos0 + q_last);  // the last key any of the queries sees
    const int tiles = last / 32 + 1;
    const int diag = (int)((p.pos0 + q0) / 32);  // tiles from here on hold keys some query must not see
    const float* kb = p.k + (int64_t)(head / p.group) * p.capacity * HD;
    const float* vb = p.v + (int64_t)(head / p.group) * p.capacity * HD;
    const float* qr = p.q + (int64_t)ql * p.q_stride + (int64_t)head * HD;
    float4 q[HD / 8];
#pragma unroll
    for (int j = 0; j < HD / 8; ++j) q[j] = *reinterpret_cast<const float4*>(qr + 8 * j + 4 * g);
    uint8_t* const kt = lds[w];
    uint8_t* const vt = lds[w] + kTile;
    const uint32_t kt_a = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)kt, vt_a = kt_a + kTile;
    const float NEG_INF = -__builtin_huge_valf();
    float m = NEG_INF, l = 0.f;
    f16v o[D];
#pragma unroll
    for (int d = 0; d < D; ++d) o[d] = f16v{};
    // this lane's columns in the V rows 4 g + i (mod 8): (chunk ^ row) * 16 + column in the chunk
    int vcol[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) vcol[i] = (((li >> 2) ^ (4 * g + i)) & 7) * 16 + (li & 3) * 4;
    pa_wait_loads<0>();
    if (w < tiles) {
        pa_stage<HD>(kb, 32 * w, last, kt_a, lane);
        pa_stage<HD>(vb, 32 * w, last, vt_a, lane);
    }
    for (int t = w; t < tiles; t += kPaWaves) {
        pa_wait_loads<HD / 8>();  // K is there, V may be in flight
        f16v s = {}, s2 = {};  // two chains of half the head's dims: fewer roundings in a row
#pragma unroll
        for (int j = 0; j < HD / 8; ++j) {
            const float4 kf = *reinterpret_cast<const float4*>(kt + li * (HD * 4) + (((2 * j + g) ^ (li & 7)) * 16));
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf.x, q[j].x, s, 0, 0, 0);
            s2 = __builtin_amdgcn_mfma_f32_32x32x2f32(kf.y, q[j].y, s2, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf.z, q[j].z, s, 0, 0, 0);
            s2 = __builtin_amdgcn_mfma_f32_32x32x2f32(kf.w, q[j].w, s2, 0, 0, 0);
        }
        s += s2;
        const bool more = t + kPaWaves < tiles;
        pa_wait_lds();
        if (more) pa_stage<HD>(kb, 32 * (t + kPaWaves), last, kt_a, lane);
        // online softmax: register r = key 32 t + 8 (r / 4) + 4 g + r % 4 of query li
        const bool edge = t >= diag;
        float mx = NEG_INF;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float v = s[r] * p.scale;
            if (edge && 32 * t + 8 * (r >> 2) + 4 * g + (r & 3) > qpos) v = NEG_INF;
            s[r] = v;
            mx = fmaxf(mx, v);
        }
        mx = swap32_max(mx);
        const float mn = fmaxf(m, mx);
        const float ms = mn == NEG_INF ? 0.f : mn;  // a query none of whose keys came yet
        const float alpha = expf(m - ms);
        l *= alpha;
        if (__any(alpha != 1.f)) {
#pragma unroll
            for (int d = 0; d < D; ++d) o[d] *= alpha;
        }
        m = mn;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s[r] = expf(s[r] - ms);
            l += s[r];
        }
        if (more) pa_wait_loads<HD / 8>();  // V is there, the next K may be in flight
        else pa_wait_loads<0>();
        bool odd = false;
        if (edge) {
            // a probability of zero must not meet an infinity or a NaN of a key the query does
            // not see
            bool bad = false;
            for (int i = 0; i < kTile / 1024; ++i) {
                const u4v x = *reinterpret_cast<const u4v*>(vt + i * 1024 + lane * 16);
#pragma unroll
                for (int e = 0; e < 4; ++e) bad |= (x[e] & 0x7F800000u) == 0x7F800000u;
            }
            odd = __any(bad);
        }
        if (!odd) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint8_t* vr = vt + (8 * (r >> 2) + 4 * g + (r & 3)) * (HD * 4) + vcol[r & 3];
#pragma unroll
                for (int d = 0; d < D; ++d)
                    o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(*reinterpret_cast<const float*>(vr + 128 * d), s[r], o[d], 0, 0, 0);
            }
        } else {
            for (int key = 0; key < 32; ++key) {
                const int own = key >> 2 & 1;  // the lane half that holds this key's probability
                float pr = 0.f;
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (8 * (r >> 2) + 4 * own + (r & 3) == key) pr = s[r];
                pr = __shfl(pr, li + 32 * own, 64);
                const bool sees = 32 * t + key <= qpos;
#pragma unroll
                for (int d = 0; d < D; ++d)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int col = 32 * d + 8 * (r >> 2) + 4 * g + (r & 3);
                        const float v = *reinterpret_cast<const float*>(vt + key * (HD * 4) + (((col >> 2) ^ (key & 7)) * 16) + (col & 3) * 4);
                        if (sees) o[d][r] = fmaf(pr, v, o[d][r]);
                    }
            }
        }
        pa_wait_lds();
        if (more) pa_stage<HD>(vb, 32 * (t + kPaWaves), last, vt_a, lane);
    }
    l = swap32_sum(l);
    // the wave's partial: unnormalised rows [query][dim], running maximum and sum
    float* const po = reinterpret_cast<float*>(lds[w]);
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
        for (int r = 0; r < 16; r += 4)
            *reinterpret_cast<float4*>(po + li * OS + 32 * d + 8 * (r >> 2) + 4 * g) =
                make_float4(o[d][r], o[d][r + 1], o[d][r + 2], o[d][r + 3]);
    if (g == 0) {
        ml[w][0][li] = m;
        ml[w][1][li] = l;
    }
    __syncthreads();
    for (int it = threadIdx.x; it < 32 * (HD / 8); it += 64 * kPaWaves) {
        const int qi = it / (HD / 8), c = it % (HD / 8);
        if (q0 + qi >= p.L) continue;
        float M = ml[0][0][qi];
#pragma unroll
        for (int s = 1; s < kPaWaves; ++s) M = fmaxf(M, ml[s][0][qi]);
        float v[8] = {}, sum = 0.f;
#pragma unroll
        for (int s = 0; s < kPaWaves; ++s) {
            const float ms = ml[s][0][qi];
            // No key of this wave has a share. A wave whose visible scores are all NaN keeps the
            // maximum -inf as well (fmaxf passes over a NaN), but its sum is NaN and has to reach
            // the row.
            if (ms == NEG_INF && ml[s][1][qi] == 0.f) continue;
            const float f = expf(ms - M);
            sum = fmaf(f, ml[s][1][qi], sum);
            const float* r = reinterpret_cast<const float*>(lds[s]) + qi * OS + 8 * c;
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = fmaf(f, r[i], v[i]);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = v[i] / sum;
        const int64_t row = q0 + qi;
        if (p.x3) {
            const int64_t kbr = (int64_t)p.n_head * D, c8 = (int64_t)head * (HD / 8) + c;
            if (p.sums) {
                float s = 0.f;
#pragma unroll
                for (int i = 0; i < 8; ++i) s += v[i];
                s += dpp_mov<0xB1>(s);  // the four lanes of a 32-column block
                s += dpp_mov<0x4E>(s);
                if (!(c & 3)) p.sums[xs_index(kbr, row, c8 >> 2)] = s;
            }
            x3_store8(p.x3, kbr, row, c8, v);
        } else if (p.out16) {
            typedef _Float16 h8 __attribute__((ext_vector_type(8)));
            h8 h;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                asm volatile("" : "+v"(v[i]));  // the fp32 value is rounded as a value of its own
                h[i] = (_Float16)v[i];
            }
            *reinterpret_cast<h8*>(p.out16 + row * p.out_stride + (int64_t)head * HD + 8 * c) = h;
        } else {
            float* op = p.out + row * p.out_stride + (int64_t)head * HD + 8 * c;
            if (!((uintptr_t)op & 15)) {
                *reinterpret_cast<float4*>(op) = make_float4(v[0], v[1], v[2], v[3]);
                *reinterpret_cast<float4*>(op + 4) = make_float4(v[4], v[5], v[6], v[7]);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) op[i] = v[i];
            }
        }
    }
}

int launch_prefill_attn_mfma(const float* q, int64_t q_stride, const float* k, const float* v, int n_head, int n_kv,
                             int hd, int64_t capacity, int64_t L, int64_t pos0, float scale, float* out,
                             int64_t out_stride, void* out16, void* x3, hipStream_t s) {
    PaArgs p{q, q_stride, k, v, n_head / n_kv, n_head, capacity, pos0, (int)L, scale, out, out_stride,
             (_Float16*)out16, (uint8_t*)x3, nullptr};
    const int64_t cols = (int64_t)n_head * hd;
    if (x3 && cols % 128 == 0) p.sums = x3_sums(x3, L, cols);
    const dim3 grid((unsigned)n_head, (unsigned)((L + 31) / 32));
    if (hd == 64)
        hipLaunchKernelGGL(k_prefill_attn_mfma<64>, grid, dim3(64 * kPaWaves), 0, s, p);
    else
        hipLaunchKernelGGL(k_prefill_attn_mfma<128>, grid, dim3(64 * kPaWaves), 0, s, p);
    return launch_status();
}

// What the matrix-core kernel takes: 16-byte loads of q, K and V rows, 32-bit key numbers.
bool prefill_attn_mfma_ok(const float* q, int64_t q_stride, const float* k, const float* v, int64_t L, int64_t pos0) {
    return aligned(q, 16) && q_stride % 4 == 0 && aligned(k, 16) && aligned(v, 16) && pos0 + L <= 0x7FFFFF00LL &&
           (L + 31) / 32 <= 65535;
}

}  // namespace pe

using namespace pe;

extern "C" int pe_prefill_attn_x3(const float* q, int64_t q_stride, const float* k_cache, const float* v_cache,
                                  int n_head, int n_kv, int head_dim, int64_t capacity, int64_t L, int64_t pos0,
                                  float scale, void* out_x3, pe_stream_t stream) {
    if (n_head <= 0 || n_kv <= 0 || n_head % n_kv || (head_dim != 64 && head_dim != 128) || capacity <= 0 || L <= 0 ||
        pos0 < 0 || pos0 + L > capacity || q_stride < (int64_t)n_head * head_dim)
        return PE_ERR_SHAPE;
    if (!q || !k_cache || !v_cache || !out_x3) return PE_ERR_NULL;
    if (!aligned(out_x3, 16)) return PE_ERR_ALIGN;
    if (!prefill_attn_mfma_ok(q, q_stride, k_cache, v_cache, L, pos0)) return PE_ERR_ALIGN;
    return launch_prefill_attn_mfma(q, q_stride, k_cache, v_cache, n_head, n_kv, head_dim, capacity, L, pos0, scale,
                                    nullptr, 0, nullptr, out_x3, (hipStream_t)stream);
}

extern "C" int pe_prefill_attn_h16(const float* q, int64_t q_stride, const float* k_cache, const float* v_cache,
                                   int n_head, int n_kv, int head_dim, int64_t capacity, int64_t L, int64_t pos0,
                                   float scale, void* out_f16, int64_t out_stride, pe_stream_t stream) {
    if (n_head <= 0 || n_kv <= 0 || n_head % n_kv || (head_dim != 64 && head_dim != 128) || capacity <= 0 || L <= 0 ||
        pos0 < 0 || pos0 + L > capacity || q_stride < (int64_t)n_head * head_dim ||
        out_stride < (int64_t)n_head * head_dim)
        return PE_ERR_SHAPE;
    if (!q || !k_cache || !v_cache || !out_f16) return PE_ERR_NULL;
    if (!aligned(out_f16, 16) || out_stride % 8) return PE_ERR_ALIGN;
    if (!prefill_attn_mfma_ok(q, q_stride, k_cache, v_cache, L, pos0)) return PE_ERR_ALIGN;
    return launch_prefill_attn_mfma(q, q_stride, k_cache, v_cache, n_head, n_kv, head_dim, capacity, L, pos0, scale,
                                    nullptr, out_stride, out_f16, nullptr, (hipStream_t)stream);
}
