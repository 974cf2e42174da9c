// Asymmetric-activation side of the W4A4 path for gfx950: the per-token
// uint4 quantizer (dynamic, MoE sign rows, or with a given scale and zero),
// the per-row int4 code sums of the weights and the zero-point outer product
// of the reference's Linear4bit zeros_x branch (signrot/nn/linear.py:35-43).
// The unsigned-A GEMM lives in gemm.hip (srq_matmul_u4s4, and the fused
// srq_w4a4_linear_asym with the zero correction in its epilogue).
//
// Quantizer arithmetic (fused.cu:143-195, quant.cu:133-207, moe.cu:104-152):
// per row vmin / vmax exact, then asym_row_params (common.h), then per
// element q = clamp(__half2int_rn(fp16(x / scale)) + __half2int_rn(zero),
// lo, hi) with [lo, hi] = [0, 15] (uint4) or [-8, 7] (int4, given-parameter
// form only).  One 256-thread block per row, two passes over the row.
#include "common.h"

#include <float.h>

namespace {

constexpr int kT = 256;

SRQ_DEV float block_min(float v, float *red) {
    v = wave_min(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return fminf(fminf(red[0], red[1]), fminf(red[2], red[3]));
}

SRQ_DEV float block_max(float v, float *red) {
    v = wave_max(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

struct AsymArgs {
    const f16 *x;
    int64_t rows, cols, cols_dst;  // cols_dst = ceil(cols / 2) bytes per row
    float clip;
    // dynamic form: scale/zero outputs; given form: scale/zero inputs
    f16 *scale;
    f16 *zero;                     // dynamic form: null with zero8
    int8_t *zero8;                 // dynamic form: the zero points as int8, or null
    int given;
    int lo, hi;                    // code range
    const int8_t *sign;            // MoE: [n_sign_rows, cols] or null
    const int32_t *sign_row;       // MoE: expert id per row
    int64_t n_sign_rows;
    uint8_t *q;
};

__global__ __launch_bounds__(kT) void asym_quant_kernel(AsymArgs a) {
    __shared__ float red[4];
    const int64_t row = blockIdx.x;
    const f16 *xr = a.x + row * a.cols;
    // MoE: x times sign[expert_ids[row]] (exact); an id outside the table
    // takes sign +1, as the symmetric MoE quantizer does
    const int8_t *sr = nullptr;
    if (a.sign) {
        const int64_t e = a.sign_row[row];
        if (e >= 0 && e < a.n_sign_rows) sr = a.sign + e * a.cols;
    }
    auto load = [&](int64_t i) {
        const float v = (float)xr[i];
        return (sr && sr[i] < 0) ? -v : v;
    };
    float s, zf;
    if (a.given) {
        s = (float)a.scale[row];
        zf = (float)a.zero[row];
    } else {
        float vmin = FLT_MAX, vmax = -FLT_MAX;
        for (int64_t i = threadIdx.x; i < a.cols; i += kT) {
            const float v = load(i);
            vmin = fminf(vmin, v);
            vmax = fmaxf(vmax, v);
        }
        vmin = block_min(vmin, red);
        vmax = block_max(vmax, red);
        f16 sh, zh;
        asym_row_params(vmin, vmax, a.clip, sh, zh);
        if (threadIdx.x == 0) {
            a.scale[row] = sh;
            if (a.zero) a.zero[row] = zh;
            if (a.zero8) a.zero8[row] = zero_i8(zh);
        }
        s = (float)sh;
        zf = (float)zh;
    }
    const int zi = h2i_rn(zf);
    uint8_t *qr = a.q + row * a.cols_dst;
    for (int64_t b = threadIdx.x; b < a.cols_dst; b += kT) {
        const int64_t c0 = 2 * b;
        const int lo = asym_code(load(c0), s, zi, a.lo, a.hi);
        const int hi = c0 + 1 < a.cols ? asym_code(load(c0 + 1), s, zi, a.lo, a.hi) : 0;
        qr[b] = (uint8_t)((lo & 0xF) | ((hi & 0xF) << 4));
    }
}

// Dynamic form for rows of 8 VPT 256 values at most, 16-byte aligned: the row
// stays in registers between the reduction and the codes, 16-byte loads,
// packed fp16 arithmetic for rows that are finite (the fused rotation's
// quantizer), asym_code per element otherwise.  The general kernel reads
// every row twice by 2-byte loads and divides per element; 1024 x 14336 with
// signs 59.6 -> 11.5 us, 512 x 4096 9.6 -> 4.0, 48 x 14336 23.6 -> 4.2 us.
template <int VPT>
__global__ __launch_bounds__(kT) void asym_quant_vec_kernel(AsymArgs a) {
    __shared__ float red[3][4];
    const int64_t row = blockIdx.x;
    const int nvec = (int)(a.cols / 8);
    const v8h *xr = reinterpret_cast<const v8h *>(a.x + row * a.cols);
    const int8_t *sr = nullptr;
    if (a.sign) {
        const int64_t e = a.sign_row[row];
        if (e >= 0 && e < a.n_sign_rows) sr = a.sign + e * a.cols;
    }
    union {
        v8h h;
        v2h p[4];
        u32 w[4];
    } v[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int k = threadIdx.x + kT * i;
        v[i].h = k < nvec ? xr[k] : (v8h){};
    }
    if (sr) {
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int k = threadIdx.x + kT * i;
            if (k < nvec) {
                int8_t s[8];
                __builtin_memcpy(s, sr + 8 * k, 8);
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (s[e] < 0) v[i].h[e] = -v[i].h[e];
            }
        }
    }
    const f16 inf = (f16)__builtin_inff();
    v2h mn = {inf, inf}, mx = -mn, ab = {0, 0};
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        if ((int)threadIdx.x + kT * i >= nvec) continue;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            mn = __builtin_elementwise_min(mn, v[i].p[p]);   // NaN-ignoring
            mx = __builtin_elementwise_max(mx, v[i].p[p]);
            ab = __builtin_elementwise_maximum(ab, __builtin_elementwise_abs(v[i].p[p]));
        }
    }
    const bool badl = !((float)ab[0] <= 65504.f) || !((float)ab[1] <= 65504.f);
    const float wmn = -wave_max_dpp(-fminf((float)mn[0], (float)mn[1]));
    const float wmx = wave_max_dpp(fmaxf((float)mx[0], (float)mx[1]));
    const bool wbad = __builtin_amdgcn_ballot_w64(badl) != 0;
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = wmn;
        red[1][threadIdx.x >> 6] = wmx;
        red[2][threadIdx.x >> 6] = wbad ? 1.f : 0.f;
    }
    __syncthreads();
    const float vmin = fminf(fminf(red[0][0], red[0][1]), fminf(red[0][2], red[0][3]));
    const float vmax = fmaxf(fmaxf(red[1][0], red[1][1]), fmaxf(red[1][2], red[1][3]));
    const bool bad = red[2][0] + red[2][1] + red[2][2] + red[2][3] != 0.f;
    f16 sh, zh;
    asym_row_params(vmin, vmax, a.clip, sh, zh);
    if (threadIdx.x == 0) {
        a.scale[row] = sh;
        if (a.zero) a.zero[row] = zh;
        if (a.zero8) a.zero8[row] = zero_i8(zh);
    }
    const float sf = (float)sh;
    const int zi = h2i_rn((float)zh);
    u32 *qr = reinterpret_cast<u32 *>(a.q + row * a.cols_dst);
    if (!bad && sf > 0.f && zi >= -511 && zi <= 511) {
        const float rcp = 1.0f / fmaxf(sf, 0x1p-126f);
        const f16 l1 = (f16)(float)(-zi), h1 = (f16)(float)(15 - zi), z1 = (f16)(float)zi;
        const v2h lo = {l1, l1}, hi = {h1, h1}, zo = {z1, z1};
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int k = threadIdx.x + kT * i;
            u32 o[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) o[p] = asym_offset_codes(quot2(v[i].w[p], rcp), lo, hi, zo);
            if (k < nvec) qr[k] = pack8_raw(o[0], o[1], o[2], o[3]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int k = threadIdx.x + kT * i;
            if (k >= nvec) continue;
            u32 o = 0;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                o |= (u32)(asym_code((float)v[i].h[e], sf, zi, 0, 15) & 0xF) << (4 * e);
            qr[k] = o;
        }
    }
}

// Sum of every nibble of a packed row (sign-extended when SIGNED), int32
// with wrapping adds (signrot/kernels/quant.cu:233-321).
template <bool SIGNED>
__global__ __launch_bounds__(kT) void sum_i4_kernel(const uint8_t *__restrict__ x,
                                                    int64_t packed_cols,
                                                    int32_t *__restrict__ out) {
    __shared__ int red[4];
    const int64_t row = blockIdx.x;
    const uint8_t *xr = x + row * packed_cols;
    u32 acc = 0;
    for (int64_t i = threadIdx.x; i < packed_cols; i += kT) {
        const int byte = xr[i];
        int lo = byte & 0xF, hi = byte >> 4;
        if (SIGNED) {
            lo = lo >= 8 ? lo - 16 : lo;
            hi = hi >= 8 ? hi - 16 : hi;
        }
        acc += (u32)(lo + hi);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += (u32)__shfl_xor((int)acc, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = (int)acc;
    __syncthreads();
    if (threadIdx.x == 0)
        out[row] = (int)((u32)red[0] + (u32)red[1] + (u32)red[2] + (u32)red[3]);
}

// out[r, c] = int32(a[r]) * b[c], wrapping (quant.cu:341-383).
__global__ __launch_bounds__(kT) void colrow_kernel(const int8_t *__restrict__ a,
                                                    const int32_t *__restrict__ b,
                                                    int64_t rows, int64_t cols,
                                                    int32_t *__restrict__ out) {
    const int64_t total = rows * cols;
    for (int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * kT) {
        const int64_t r = i / cols, c = i - r * cols;
        out[i] = (int)((u32)(int)a[r] * (u32)b[c]);
    }
}

int launch_asym(const AsymArgs &a, hipStream_t st, const char *name) {
    const int64_t nvec = a.cols / 8;
    if (!a.given && a.cols % 8 == 0 && nvec <= 8 * kT && srq_aligned(a.x, 16) &&
        srq_aligned(a.q, 4)) {
        const dim3 grid((unsigned)a.rows), block(kT);
        if (nvec <= kT) asym_quant_vec_kernel<1><<<grid, block, 0, st>>>(a);
        else if (nvec <= 2 * kT) asym_quant_vec_kernel<2><<<grid, block, 0, st>>>(a);
        else if (nvec <= 4 * kT) asym_quant_vec_kernel<4><<<grid, block, 0, st>>>(a);
        else asym_quant_vec_kernel<8><<<grid, block, 0, st>>>(a);
        SRQ_LAUNCH_CHECK(name);
        return SRQ_OK;
    }
    asym_quant_kernel<<<dim3((unsigned)a.rows), dim3(kT), 0, st>>>(a);
    SRQ_LAUNCH_CHECK(name);
    return SRQ_OK;
}

int asym_dynamic(const char *name, const void *x, const int8_t *sign, const int32_t *expert_ids,
                 int64_t num_experts, int64_t rows, int64_t cols, float clip_ratio, void *q,
                 void *scale, void *zero, int8_t *zero8, void *stream) {
    SRQ_CHECK_ARG(rows >= 0 && cols >= 0 && num_experts >= 0, "%s: negative shape", name);
    if (rows == 0) return SRQ_OK;
    SRQ_CHECK_ARG(rows <= 0x7fffffffLL, "%s: rows > 2^31-1", name);
    SRQ_CHECK_ARG(cols > 0, "%s: empty rows", name);
    SRQ_CHECK_ARG(x && q && scale && (zero || zero8), "%s: null pointer", name);
    SRQ_CHECK_ARG(!sign || expert_ids, "%s: sign needs expert_ids", name);
    AsymArgs a{};
    a.x = (const f16 *)x;
    a.rows = rows;
    a.cols = cols;
    a.cols_dst = (cols + 1) / 2;
    a.clip = clip_ratio;
    a.scale = (f16 *)scale;
    a.zero = (f16 *)zero;
    a.zero8 = zero8;
    a.lo = 0;
    a.hi = 15;
    a.sign = sign;
    a.sign_row = expert_ids;
    a.n_sign_rows = num_experts;
    a.q = (uint8_t *)q;
    return launch_asym(a, (hipStream_t)stream, name);
}

}  // namespace

extern "C" int srq_asym_quant_dynamic(const void *x, int64_t rows, int64_t cols,
                                      float clip_ratio, void *q, void *scale, void *zero,
                                      void *stream) {
    SRQ_CHECK_ARG(zero || rows == 0, "asym_quant_dynamic: null pointer");
    return asym_dynamic("asym_quant_dynamic", x, nullptr, nullptr, 0, rows, cols, clip_ratio, q,
                        scale, zero, nullptr, stream);
}

extern "C" int srq_asym_quant_dynamic_moe(const void *x, const int8_t *sign,
                                          const int32_t *expert_ids, int64_t num_experts,
                                          int64_t rows, int64_t cols, float clip_ratio, void *q,
                                          void *scale, void *zero, void *stream) {
    SRQ_CHECK_ARG(zero || rows == 0, "asym_quant_dynamic_moe: null pointer");
    return asym_dynamic("asym_quant_dynamic_moe", x, sign, expert_ids, num_experts, rows, cols,
                        clip_ratio, q, scale, zero, nullptr, stream);
}

extern "C" int srq_asym_quant_dynamic_i8(const void *x, const int8_t *sign,
                                         const int32_t *expert_ids, int64_t num_experts,
                                         int64_t rows, int64_t cols, float clip_ratio, void *q,
                                         void *scale, int8_t *zero, void *stream) {
    SRQ_CHECK_ARG(zero || rows == 0, "asym_quant_dynamic_i8: null pointer");
    return asym_dynamic("asym_quant_dynamic_i8", x, sign, expert_ids, num_experts, rows, cols,
                        clip_ratio, q, scale, nullptr, zero, stream);
}

extern "C" int srq_asym_quant(const void *x, const void *scale, const void *zero, int64_t rows,
                              int64_t cols, int is_signed, void *q, void *stream) {
    SRQ_CHECK_ARG(rows >= 0 && cols >= 0, "asym_quant: negative shape");
    if (rows == 0 || cols == 0) return SRQ_OK;
    SRQ_CHECK_ARG(rows <= 0x7fffffffLL, "asym_quant: rows > 2^31-1");
    SRQ_CHECK_ARG(x && q && scale && zero, "asym_quant: null pointer");
    AsymArgs a{};
    a.x = (const f16 *)x;
    a.rows = rows;
    a.cols = cols;
    a.cols_dst = (cols + 1) / 2;
    a.scale = (f16 *)scale;
    a.zero = (f16 *)zero;
    a.given = 1;
    a.lo = is_signed ? -8 : 0;
    a.hi = is_signed ? 7 : 15;
    a.q = (uint8_t *)q;
    return launch_asym(a, (hipStream_t)stream, "asym_quant");
}

extern "C" int srq_sum_i4(const void *x, int64_t rows, int64_t packed_cols, int is_signed,
                          int32_t *out, void *stream) {
    SRQ_CHECK_ARG(rows >= 0 && packed_cols >= 0, "sum_i4: negative shape");
    if (rows == 0) return SRQ_OK;
    SRQ_CHECK_ARG(rows <= 0x7fffffffLL, "sum_i4: rows > 2^31-1");
    SRQ_CHECK_ARG(out && (x || packed_cols == 0), "sum_i4: null pointer");
    hipStream_t st = (hipStream_t)stream;
    if (is_signed)
        sum_i4_kernel<true><<<dim3((unsigned)rows), dim3(kT), 0, st>>>(
            (const uint8_t *)x, packed_cols, out);
    else
        sum_i4_kernel<false><<<dim3((unsigned)rows), dim3(kT), 0, st>>>(
            (const uint8_t *)x, packed_cols, out);
    SRQ_LAUNCH_CHECK("sum_i4");
    return SRQ_OK;
}

extern "C" int srq_matmul_colrow_i8_i32(const int8_t *a_col, const int32_t *b_row, int64_t rows,
                                        int64_t cols, int32_t *out, void *stream) {
    SRQ_CHECK_ARG(rows >= 0 && cols >= 0, "matmul_colrow_i8_i32: negative shape");
    if (rows == 0 || cols == 0) return SRQ_OK;
    SRQ_CHECK_ARG(a_col && b_row && out, "matmul_colrow_i8_i32: null pointer");
    const int64_t blocks = std::min<int64_t>(srq_cdiv(rows * cols, kT), 4096);
    colrow_kernel<<<dim3((unsigned)blocks), dim3(kT), 0, (hipStream_t)stream>>>(a_col, b_row, rows,
                                                                              cols, out);
    SRQ_LAUNCH_CHECK("matmul_colrow_i8_i32");
    return SRQ_OK;
}
