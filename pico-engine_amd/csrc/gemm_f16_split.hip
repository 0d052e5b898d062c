// Prefill products with few output tiles (mid-size prompts, narrow matrices), on the matrix cores.
//
// C = A W^T (+ bias) (+ R) with the operands and conventions of gemm_f16.hip. Its 128 x 128 and
// 256-row tiles leave most of the 256 CUs idle here (1021 x 896: 56 tiles) and walk the whole of
// a long K one step after another. A workgroup here computes a 64 x 64 tile with its K divided
// over kSpW waves: each wave holds the whole tile's accumulators and reads its operands straight
// from memory in MFMA order (16 rows x 64 contiguous bytes per load), the next step's loads in
// flight while the current step's sixteen MFMAs run; no barrier in the loop. The waves' tiles meet
// in LDS and are added in wave order (the result does not depend on timing). Bound by the operand
// reads from L2, (64 + 64) K values per tile: 1021 x 896 x 4864 107 -> 41.7 us, 1021 x 896 x 896
// 26.9 -> 12.8 us.
#include "gemm_f16.h"

namespace pe {

constexpr int kSpT = 64;        // tile rows and columns
constexpr int kSpW = 4;         // waves, each with a share of K
constexpr int kSpS = kSpT + 4;  // row stride of the partial tiles in LDS

// SILU, CH: as k_gemm_f16's (interleaved gate / up rows in groups of 16; fp16 output); the same
// shares and order as the plain product of the same sizes, so gemm then silu_mul gives its bits.
template <bool AH, bool SILU, bool CH>
__global__ __launch_bounds__(64 * kSpW, 2) void k_gemm_split(GemmF16Args p, int m_tiles, int n_tiles) {
    __shared__ __attribute__((aligned(16))) float part[kSpW][kSpT][kSpS];
    const int lane = threadIdx.x & 63, wk = threadIdx.x >> 6, li = lane & 15, lq = lane >> 4;
    // an XCD takes an eighth of the tiles in column order: its workgroups share column tiles, whose
    // weight rows its L2 reads once, and no XCD gets more than one tile per CU while the chip has
    // room (with whole column tiles per XCD, 4096 x 64 x 3584 ran on one XCD: 56.3 us)
    const int tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (tile >= m_tiles * n_tiles) return;
    const int tn = tile / m_tiles, tm = tile % m_tiles;
    const int64_t bm = (int64_t)tm * kSpT, bn = (int64_t)tn * kSpT;
    // a step is 64 columns of fp16 A: whole 128-byte lines of both operands (half lines came back
    // from L2 twice, the workgroup's operands being larger than L1); 32 of fp32 A, for the registers
    constexpr int U = AH ? 2 : 1;
    // shares of whole 64 columns for both, so that fp16 and fp32 A give the same bits
    const int64_t s64 = p.K / 64, s0 = s64 * wk / kSpW * (2 / U), s1 = s64 * (wk + 1) / kSpW * (2 / U);
    const PE_GLOBAL uint8_t* ap[4];
    const PE_GLOBAL uint8_t* wp[4];
    constexpr int AE = AH ? 2 : 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // rows past M or N repeat the last one
        const int64_t m = bm + 16 * i + li < p.M ? bm + 16 * i + li : p.M - 1;
        const int64_t n = bn + 16 * i + li < p.N ? bn + 16 * i + li : p.N - 1;
        ap[i] = (AH ? (const PE_GLOBAL uint8_t*)p.ah : (const PE_GLOBAL uint8_t*)p.a) + (m * p.lda + 8 * lq + 32 * U * s0) * AE;
        wp[i] = (const PE_GLOBAL uint8_t*)p.w + (n * p.K + 8 * lq + 32 * U * s0) * 2;
    }
    f4v acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f4v{0.f, 0.f, 0.f, 0.f};
    typedef h8 __attribute__((address_space(1))) gh8;
    typedef f4v __attribute__((address_space(1))) gf4;
    h8 av[2][U][4], wv[2][U][4];
    f4v af[2][4][2];
    const int64_t n = s1 - s0;
    auto load = [&](auto buf, int64_t s) {
        constexpr int B = decltype(buf)::value;
        s = s < n ? s : n - 1;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                wv[B][u][i] = *reinterpret_cast<const gh8*>(wp[i] + s * (64 * U) + 64 * u);
                if constexpr (AH) {
                    av[B][u][i] = *reinterpret_cast<const gh8*>(ap[i] + s * (64 * U) + 64 * u);
                } else {
                    af[B][i][0] = *reinterpret_cast<const gf4*>(ap[i] + s * 128);
                    af[B][i][1] = *reinterpret_cast<const gf4*>(ap[i] + s * 128 + 16);
                }
            }
        __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the other buffer's MFMAs
    };
    auto mul = [&](auto buf) {
        constexpr int B = decltype(buf)::value;
        if constexpr (!AH) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e) av[B][0][i][e] = (_Float16)af[B][i][e >> 2][e & 3];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[B][u][i], wv[B][u][j], acc[i][j], 0, 0, 0);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    if (n > 0) {
        load(I0{}, 0);
        for (int64_t s = 0; s < n; s += 2) {
            load(I1{}, s + 1);
            mul(I0{});
            load(I0{}, s + 2);
            if (s + 1 < n) mul(I1{});
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[wk][16 * i + 4 * lq + r][16 * j + li] = acc[i][j][r];
    __syncthreads();
    auto sum4 = [&](int lr, int c) {
        float4 v = *reinterpret_cast<const float4*>(&part[0][lr][c]);
#pragma unroll
        for (int q = 1; q < kSpW; ++q) {
            const float4 b = *reinterpret_cast<const float4*>(&part[q][lr][c]);
            v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w;
        }
        return v;
    };
    if constexpr (SILU) {
        for (int it = threadIdx.x; it < kSpT * (kSpT / 8); it += 64 * kSpW) {
            const int lr = it / (kSpT / 8), c = 4 * (it % (kSpT / 8));  // the tile's 32 output columns
            const int64_t m = bm + lr, col = bn / 2 + c;
            if (m >= p.M || col >= p.N / 2) continue;  // N / 2 is a multiple of 16
            const float4 g = sum4(lr, 32 * (c >> 4) + (c & 15)), u = sum4(lr, 32 * (c >> 4) + 16 + (c & 15));
            float e[4] = {silu_mul_prefill(g.x, u.x), silu_mul_prefill(g.y, u.y), silu_mul_prefill(g.z, u.z),
                          silu_mul_prefill(g.w, u.w)};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (CH) {
                    asm volatile("" : "+v"(e[i]));  // the fp32 value is rounded as a value of its own
                    p.ch[m * p.ldc + col + i] = (_Float16)e[i];
                } else {
                    p.c[m * p.ldc + col + i] = e[i];
                }
            }
        }
        return;
    }
    for (int it = threadIdx.x; it < kSpT * (kSpT / 4); it += 64 * kSpW) {
        const int lr = it / (kSpT / 4), c = 4 * (it % (kSpT / 4));
        const int64_t m = bm + lr, col = bn + c;
        if (m >= p.M || col >= p.N) continue;
        float4 v = sum4(lr, c);
        float* cp = p.c + m * p.ldc + col;
        const float* rp = p.res ? p.res + m * p.ldr + col : nullptr;
        const float* bp = p.bias ? p.bias + col : nullptr;
        if (col + 4 <= p.N && !(((uintptr_t)cp | (uintptr_t)rp | (uintptr_t)bp) & 15)) {
            if (bp) {
                const float4 b = *reinterpret_cast<const float4*>(bp);
                v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w;
            }
            if (rp) {
                const float4 r = *reinterpret_cast<const float4*>(rp);
                v.x += r.x; v.y += r.y; v.z += r.z; v.w += r.w;
            }
            *reinterpret_cast<float4*>(cp) = v;
        } else {
            const float e[4] = {v.x, v.y, v.z, v.w};
            for (int i = 0; i < 4; ++i)
                if (col + i < p.N) cp[i] = (e[i] + (bp ? bp[i] : 0.f)) + (rp ? rp[i] : 0.f);
        }
    }
}

// Up to 256 tiles of 64 x 64, one workgroup per CU. The time is that of one tile's K, and twice that
// from 257 on; then it is still faster where K is long or k_gemm_f16 would add a bias or a residual
// (its epilogue takes 5 us for that), except where k_gemm_h16_dl takes the product (wide). Either
// side in us, fp16 A, weights not in L2 (as a model's are not):
//   1021 x 896 x 896 (224 tiles) 12.8 | 26.9     1537 x 1152 x 896 (wide) 20.9 | 14.0
//   1021 x 896 x 4864 (224) 41.7 | 107.3         445 x 2560 x 256 (280) 13.8 | 9.3
//   1021 x 1152 x 896 (288, bias) 21.6 | 26.9, without 21.0 | 20.6; 573 x 2048 x 896 (288) 21.0 | 19.5
//   957 x 1152 x 1536 (270) 28.0 | 31.1          200 x 4608 x 3584 (288) 56.0 | 80.5
// fp32 A, 600 x 896 x 4864 (140): 55.6 | 152.3. K from 256 on, so that each wave has a step.
bool gemm_split_ok(int64_t M, int64_t N, int64_t K, bool added, bool wide) {
    if (K % 64 || K < 256 || M > 320 * kSpT || N > 320 * kSpT) return false;
    const int64_t tiles = ((M + kSpT - 1) / kSpT) * ((N + kSpT - 1) / kSpT);
    return tiles <= 256 || (tiles <= 320 && !wide && K >= (added ? 512 : 1536));
}

template <bool AH, bool SILU, bool CH>
static int split_launch(const GemmF16Args& p, hipStream_t s) {
    const int mt = (int)((p.M + kSpT - 1) / kSpT), nt = (int)((p.N + kSpT - 1) / kSpT);
    hipLaunchKernelGGL((k_gemm_split<AH, SILU, CH>), dim3(8u * (unsigned)((mt * nt + 7) / 8)), dim3(64 * kSpW),
                       0, s, p, mt, nt);
    return launch_status();
}

int gemm_split_launch(const GemmF16Args& p, bool silu, hipStream_t s) {
    if (!silu) return p.ah ? split_launch<true, false, false>(p, s) : split_launch<false, false, false>(p, s);
    if (p.ch) return p.ah ? split_launch<true, true, true>(p, s) : split_launch<false, true, true>(p, s);
    return split_launch<false, true, false>(p, s);  // an fp16 A comes with an fp16 output
}

}  // namespace pe
