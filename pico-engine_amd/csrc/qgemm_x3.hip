// Short-prompt prefill products on the matrix cores at fp32 grade (qgemm_x3.h): the x3 forms
// of activations, and the C entry points of the products.
#include "qgemm_x3_launch.h"

namespace pe {

// One workgroup per row: RMSNorm (norm weights given) or a plain copy into the x3 form.
// Bandwidth- and latency-bound; a thread keeps its first 8-column chunk between the sum of squares
// and the store (rows of up to 8 * blockDim = 4096 columns are read once), and reads the others again.
template <bool NORM>
__global__ void k_x3_rows(const float* __restrict__ x, int64_t xs_, const float* __restrict__ w, int64_t n,
                          float eps, uint8_t* __restrict__ x3, float* __restrict__ sums) {
    __shared__ float red[8];
    const int64_t r = blockIdx.x;
    const float* xr = x + r * xs_;
    const int64_t chunks = n >> 3, kb = n >> 5;
    float rstd = 1.f;
    auto load8 = [&](const float* p, float* v) {
        const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    };
    float first[8];
    if (NORM) {
        float ss = 0.f;
        for (int64_t c = threadIdx.x; c < chunks; c += blockDim.x) {
            float v[8];
            load8(xr + 8 * c, v);
#pragma unroll
            for (int i = 0; i < 8; ++i) ss = fmaf(v[i], v[i], ss);
            if (c == threadIdx.x) {
#pragma unroll
                for (int i = 0; i < 8; ++i) first[i] = v[i];
            }
        }
        ss = wave_sum<64>(ss);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
        __syncthreads();
        ss = 0.f;
        for (int i = 0; i < (int)(blockDim.x >> 6); ++i) ss += red[i];
        rstd = 1.0f / sqrtf(ss / (float)n + eps);
    }
    for (int64_t c = threadIdx.x; c < chunks; c += blockDim.x) {
        float v[8];
        if (NORM) {
            float wv[8];
            load8(w + 8 * c, wv);
            if (c == threadIdx.x) {
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = first[i];
            } else {
                load8(xr + 8 * c, v);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = (v[i] * rstd) * wv[i];
        } else {
            load8(xr + 8 * c, v);
        }
        x3_store8(x3, kb, r, c, v);
        if (sums) {
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) s += v[i];
            s += dpp_mov<0xB1>(s);  // the four lanes of a 32-column block (n % 128 == 0)
            s += dpp_mov<0x4E>(s);
            if (!(c & 3)) sums[xs_index(kb, r, c >> 2)] = s;
        }
    }
}

static int x3_rows(const float* x, int64_t x_stride, const float* w, int64_t m, int64_t n, float eps, void* x3,
                   hipStream_t s) {
    const int64_t chunks = n / 8;
    const unsigned threads = chunks <= 64 ? 64 : chunks <= 128 ? 128 : chunks <= 256 ? 256 : 512;
    if (m * threads > 0xFFFFFFFFLL) return PE_ERR_SHAPE;  // more than one grid holds
    float* sums = n % 128 ? nullptr : x3_sums(x3, m, n);
    if (w)
        hipLaunchKernelGGL(k_x3_rows<true>, dim3((unsigned)m), dim3(threads), 0, s, x, x_stride, w, n, eps,
                           (uint8_t*)x3, sums);
    else
        hipLaunchKernelGGL(k_x3_rows<false>, dim3((unsigned)m), dim3(threads), 0, s, x, x_stride, w, n, eps,
                           (uint8_t*)x3, sums);
    return launch_status();
}

}  // namespace pe

using namespace pe;

extern "C" int64_t pe_x3_bytes(int64_t m, int64_t k) {
    if (m <= 0 || m > 0x7FFFFFFF || k <= 0 || k % 32 || k > 0x7FFFFFFF) return -PE_ERR_SHAPE;
    return x3_plane_bytes(m, k) + (k % 128 ? 0 : x3_plane_bytes(m, k) / 48);
}

extern "C" int pe_x3_split(const float* x, int64_t x_stride, int64_t m, int64_t k, void* x3, pe_stream_t stream) {
    if (pe_x3_bytes(m, k) < 0 || x_stride < k || x_stride % 4) return PE_ERR_SHAPE;
    if (!x || !x3) return PE_ERR_NULL;
    if (!aligned(x, 16) || !aligned(x3, 16)) return PE_ERR_ALIGN;
    return x3_rows(x, x_stride, nullptr, m, k, 0.f, x3, (hipStream_t)stream);
}

extern "C" int pe_x3_rmsnorm(const float* x, int64_t x_stride, const float* w, float eps, int64_t m, int64_t k,
                             void* x3, pe_stream_t stream) {
    if (pe_x3_bytes(m, k) < 0 || x_stride < k || x_stride % 4) return PE_ERR_SHAPE;
    if (!x || !w || !x3) return PE_ERR_NULL;
    if (!aligned(x, 16) || !aligned(w, 16) || !aligned(x3, 16)) return PE_ERR_ALIGN;
    return x3_rows(x, x_stride, w, m, k, eps, x3, (hipStream_t)stream);
}

extern "C" int pe_qgemm_x3_supported(int type, int64_t n, int64_t k) { return x3_weight_ok(type, n, k); }

// A tiled matrix of the x3 kernels: the type and shape, and the alignment of its planes' loads.
static int check_x3(int type, const void* w, int64_t n, int64_t k, const void* x3, int64_t m) {
    int st = x3_weight_ok(type, n, k);
    if (st) return st;
    if (m <= 0 || m > 65535LL * 8) return PE_ERR_SHAPE;  // pe_qgemm's rows
    if (!w || !x3) return PE_ERR_NULL;
    if (!aligned(w, 16) || !aligned(x3, 16)) return PE_ERR_ALIGN;
    return PE_OK;
}

static X3Args x3_args(int64_t k, const void* x3, int64_t m) {
    X3Args p{};
    p.a = (const uint8_t*)x3;
    p.xs = x3_sums((void*)x3, m, k);
    p.m = (int)m;
    p.kb = (int)(k / 32);
    return p;
}

extern "C" int pe_qgemm_x3(int type, const void* w, int64_t n, int64_t k, const void* x3, int64_t m,
                           const float* bias, const float* residual, int64_t res_stride, float* y,
                           int64_t y_stride, pe_stream_t stream) {
    int st = check_x3(type, w, n, k, x3, m);
    if (st) return st;
    if (y_stride < n || (residual && res_stride < n)) return PE_ERR_SHAPE;
    if (!y) return PE_ERR_NULL;
    if (!aligned(y, 4) || !aligned(residual, 4) || !aligned(bias, 4)) return PE_ERR_ALIGN;
    X3Args p = x3_args(k, x3, m);
    p.seg[0] = X3Seg{make_tiled(w, n, k / block_elems(type)), n, 0, bias};
    p.res = residual;
    p.res_stride = res_stride;
    p.y = y;
    p.y_stride = y_stride;
    return x3_plain(type, p, (hipStream_t)stream);
}

extern "C" int pe_qgemm_x3_rows(int type, const void* w, int64_t n, int64_t k, const float* x, int64_t x_stride,
                                int64_t m, const float* bias, const float* residual, int64_t res_stride, float* y,
                                int64_t y_stride, void* scratch, int64_t scratch_bytes, pe_stream_t stream) {
    int st = check_x3(type, w, n, k, scratch, m);
    if (st) return st;
    // whole row tiles that the scratch holds and whose grid stays below 2^32 threads (512 per 32 x
    // 64 columns; 32 rows of 2^28 columns do)
    int64_t step = scratch_bytes / pe_x3_bytes(32, k) * 32;
    const int64_t most = (1LL << 33) / n / 32 * 32;
    if (step <= 0) return PE_ERR_SPACE;
    if (step > most) step = most > 32 ? most : 32;
    for (int64_t r = 0; r < m; r += step) {
        const int64_t c = m - r < step ? m - r : step;
        st = pe_x3_split(x ? x + r * x_stride : x, x_stride, c, k, scratch, stream);
        if (!st)
            st = pe_qgemm_x3(type, w, n, k, scratch, c, bias, residual ? residual + r * res_stride : nullptr, res_stride,
                             y ? y + r * y_stride : y, y_stride, stream);
        if (st) return st;
    }
    return PE_OK;
}

extern "C" int pe_qgemm_x3_silu(int type, const void* w, int64_t ffn, int64_t k, const void* x3, int64_t m,
                                void* act_x3, pe_stream_t stream) {
    int st = check_x3(type, w, 2 * ffn, k, x3, m);
    if (st) return st;
    if (ffn % 32) return PE_ERR_SHAPE;
    if (!act_x3) return PE_ERR_NULL;
    if (!aligned(act_x3, 16)) return PE_ERR_ALIGN;
    X3Args p = x3_args(k, x3, m);
    p.seg[0] = X3Seg{make_tiled(w, 2 * ffn, k / block_elems(type)), ffn, 0, nullptr};
    p.out3 = (uint8_t*)act_x3;
    p.out_kb = (int)(ffn / 32);
    p.out_xs = ffn % 128 ? nullptr : x3_sums(act_x3, m, ffn);
    p.n_tiles = (int)(ffn / 32);
    return x3_silu(type, p, (hipStream_t)stream);
}

extern "C" int pe_qkv_x3_supported(int q_type, int k_type, int v_type, int64_t k, int n_head, int n_kv, int hd) {
    if (n_head <= 0 || n_kv <= 0 || hd <= 0 || hd % 64) return PE_ERR_SHAPE;
    int st = x3_weight_ok(q_type, (int64_t)n_head * hd, k);
    if (!st) st = x3_weight_ok(k_type, (int64_t)n_kv * hd, k);
    if (!st) st = x3_weight_ok(v_type, (int64_t)n_kv * hd, k);
    if (st) return st;
    return q_type == k_type && x3_qkv_pair(q_type, v_type) ? PE_OK : PE_ERR_TYPE;
}

extern "C" int pe_qkv_x3(int q_type, int k_type, int v_type, const void* wq, const void* wk, const void* wv,
                         const float* bq, const float* bk, const float* bv, int64_t k, const void* x3, int64_t m,
                         const float* cos_rows, const float* sin_rows, int n_head, int n_kv, int hd,
                         int64_t pos0, float* q_out, float* k_cache, float* v_cache, int64_t capacity,
                         pe_stream_t stream) {
    int st = pe_qkv_x3_supported(q_type, k_type, v_type, k, n_head, n_kv, hd);
    if (st) return st;
    const int64_t nq = (int64_t)n_head * hd, nk = (int64_t)n_kv * hd;
    if ((st = check_x3(q_type, wq, nq, k, x3, m))) return st;
    if ((st = check_x3(k_type, wk, nk, k, x3, m))) return st;
    if ((st = check_x3(v_type, wv, nk, k, x3, m))) return st;
    if (pos0 < 0 || capacity <= 0 || pos0 + m > capacity) return PE_ERR_SHAPE;
    if (!cos_rows || !sin_rows || !q_out || !k_cache || !v_cache) return PE_ERR_NULL;
    if (!aligned(bq, 4) || !aligned(bk, 4) || !aligned(bv, 4) || !aligned(cos_rows, 4) || !aligned(sin_rows, 4) ||
        !aligned(q_out, 16) || !aligned(k_cache, 16) || !aligned(v_cache, 16))
        return PE_ERR_ALIGN;
    X3Args p = x3_args(k, x3, m);
    p.seg[0] = X3Seg{make_tiled(wq, nq, k / block_elems(q_type)), nq, 0, bq};
    p.seg[1] = X3Seg{make_tiled(wk, nk, k / block_elems(k_type)), nk, (int)(nq / 64), bk};
    p.seg[2] = X3Seg{make_tiled(wv, nk, k / block_elems(v_type)), nk, (int)((nq + nk) / 64), bv};
    p.n_tiles = (int)((nq + 2 * nk) / 64);
    p.cos_rows = cos_rows;
    p.sin_rows = sin_rows;
    p.q_out = q_out;
    p.k_cache = k_cache;
    p.v_cache = v_cache;
    p.capacity = capacity;
    p.pos0 = pos0;
    p.n_head = n_head;
    p.hd = hd;
    return x3_qkv(q_type, v_type, p, (hipStream_t)stream);
}
