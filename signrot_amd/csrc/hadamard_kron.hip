// MFMA rotation for n = K * m outside the 512 / 1024 chunk forms of
// hadamard_mfma.hip: K a multiple of 4 up to 176 (every Kronecker factor of
// the table: 12 ... 172), m = n / K one of 64, 128, 256, 512 -- the FFN sizes
// 11008 = 172 x 64, 13824 = 108 x 128, 18944 = 148 x 128, 5120 = 20 x 256 and
// their like -- optionally fused with the SignRot sign and the per-token
// symmetric int4 or asymmetric uint4 quantizer.
//
// A row is the matrix X [K, m]; the result is hadK . fp16((X . H_m) / sqrt n)
// with the reference's two fp16 rounding points.  Both products are fp16
// MFMA 32x32x16 with fp32 accumulation (the inputs are fp16, H_m is +-1).
// One block per row at a time, persistent over rows; wave (ct, wi) owns the
// 32 chunks c = 32 ct + 0..31 and the columns i2 of its Q 32-column tiles
// nt = Q wi + q of each 128-column group (m < 128: of the one group).
//
// Stage A, D[c][i] = sum_i' X[c][i'] H[i'][i]: the A operand (8 consecutive
// i' of chunk c per lane) comes straight from global memory, 16 bytes per
// lane, the next row's being in flight during this row's stage K; the B
// operand is one 8-entry +-1 pattern per lane and a sign per step.  For
// m = 128 P the P groups are combined by butterflies over the accumulators
// (index bits in ascending order).  y = fp16(D / sqrt n) goes to LDS
// transposed, yT[i][c] (4 consecutive chunks per lane: 8-byte stores), rows
// padded by 8 halves: the row stride is an odd number of 16-byte units, so
// the 16-byte reads of stage K are free of bank conflicts.
// Stage K, out^T[i][c] = sum_c' yT[i][c'] hadK[c][c']: the wave's hadK
// fragments stay in registers for all rows; operand row ln reads
// i = 16 ((ln >> 2) & 1) + 4 (ln >> 3) + (ln & 3), so that a lane's 16
// results are 16 consecutive outputs of chunk c = 32 ct + ln: 32 bytes of
// the rotated row, 8 bytes of codes, stored directly.
//
// What bounds it: with few rows the chain load -> stage A -> barrier ->
// stage K -> row reduction -> codes; with many, the VALU work per element
// beside the MFMAs and the two barriers of each row (1.4-1.9 TB/s).  The LDS
// kernel that had these sizes does the K-mix on the VALU, a thread per
// column, for K > 64 with hadK from global memory.  Rotation + quantizer, us
// at 1 / 137 / 2048 rows, that kernel -> this one (one MI355X, graph replay):
//   172 x 64   3938 / 4053 / 32330 -> 6.9 / 7.4 / 30.3
//   108 x 128  1572 / 1612 / 12801 -> 7.3 / 8.1 / 38.1
//   60 x 256   97 / 99 / 432       -> 8.1 / 9.4 / 49.4
//   28 x 128   27.7 / 28.9 / 85.9  -> 3.6 / 4.2 / 13.1
//   12 x 64    13.1 / 13.6 / 33.1  -> 3.0 / 3.6 / 5.5
#include "common.h"

#include <algorithm>
#include <type_traits>

namespace {

typedef float v2f __attribute__((ext_vector_type(2)));
typedef u32 v2u __attribute__((ext_vector_type(2)));
typedef u32 v4u __attribute__((ext_vector_type(4)));

SRQ_DEV v16f mfma32(v8h a, v8h b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

SRQ_DEV int parity(int v) { return __builtin_popcount(v) & 1; }

SRQ_DEV u32 pk16(float a, float b) {
    return __builtin_bit_cast(u32, __builtin_convertvector((v2f){a, b}, v2h));
}

SRQ_DEV void lds_barrier() {
    // LDS only: the loads of the next row stay in flight
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

struct KronArgs {
    const f16 *x;
    int64_t rows;
    int K;
    int nc;               // 32-chunk tiles, ceil(K / 32)
    const f16 *hadK;      // [K, K]
    const int8_t *sign;   // [n] or null
    float scale;          // fp32 1 / sqrt(n)
    float clip;
    uint8_t *q;           // MODE 1, 2: packed codes, rows of n / 2 bytes
    f16 *qscale;          // MODE 1, 2: [rows]
    f16 *qzero;           // MODE 2: [rows] or null
    int8_t *qzero8;       // MODE 2: the same as int8 or null
    f16 *out;             // MODE 0: rows of n
};

// KS: stage-K steps of 16 chunks (16 KS >= K); KA: stage-A steps of 16
// columns, min(m, 128) / 16; P = m / 128 (1 below 128); Q: column tiles per
// wave and group.  MODE: 0 rotation (fp16 out), 1 + symmetric int4 quantizer,
// 2 + asymmetric uint4 quantizer.
template <int KS, int KA, int P, int Q, int MODE, int MAXT>
__global__ __launch_bounds__(MAXT) void had_kron_kernel(KronArgs a) {
    constexpr int M = KA * 16 * P;         // chunk length m
    constexpr int LD = KS * 16 + 8;        // yT row stride, halves
    constexpr int T = P * Q;               // output tiles per wave
    __shared__ __attribute__((aligned(16))) f16 yT[M * LD];
    __shared__ float red[3][16];
    const int lane = threadIdx.x & 63;
    const int g = lane >> 5, ln = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    const int ct = wave % a.nc, wi = wave / a.nc;
    const int c = 32 * ct + ln;            // stage-A operand row, stage-K column
    const bool live = c < a.K;
    const int n = a.K * M;

    // chunks past K never get a value: they stay zero (hadK is zero there)
    for (int i = threadIdx.x; i < M * LD / 8; i += blockDim.x)
        reinterpret_cast<v4u *>(yT)[i] = (v4u){0, 0, 0, 0};

    // H operand: entry e of step ks, column i2 = 32 nt + ln, is
    // (-1)^(parity(e & ln) ^ parity((16 ks + 8 g) & i2))
    union Frag {
        v8h h;
        u32 w[4];
    } pat;
#pragma unroll
    for (int e = 0; e < 8; ++e) pat.h[e] = parity(e & ln) ? (f16)-1 : (f16)1;
    const u32 flip_g = parity((8 * g) & ln) ? 0x80008000u : 0u;
    const u32 flip_16 = (ln & 16) ? 0x80008000u : 0u;
    // hadK fragments of column c: c' = 16 s + 8 g + e (K is a multiple of 4,
    // so a run of 4 is wholly inside the row or past it)
    v8h hb[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int cp = 16 * s + 8 * g + 4 * h;
            v4h v = {};
            if (live && cp < a.K) v = *reinterpret_cast<const v4h *>(a.hadK + c * a.K + cp);
#pragma unroll
            for (int e = 0; e < 4; ++e) hb[s][4 * h + e] = v[e];
        }
    // first output of tile (i1, q) of this lane: 16 consecutive from here
    auto out_at = [&](int i1, int q) { return c * M + i1 * 128 + 32 * (wi * Q + q) + 16 * g; };
    // its signs as fp16 factors (any int8 value: the product of a fp16 and a
    // small integer rounds once, as the fp32 product rounded to fp16 does)
    u32 sg[T][8];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int p = 0; p < 8; ++p) sg[t][p] = 0x3C003C00u;
    if (a.sign && live) {
        const bool al = (reinterpret_cast<uintptr_t>(a.sign) & 15) == 0;
#pragma unroll
        for (int i1 = 0; i1 < P; ++i1)
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int8_t *sp = a.sign + out_at(i1, q);
                union {
                    v4u w;
                    int8_t b[16];
                } s;
                if (al) {
                    s.w = *reinterpret_cast<const v4u *>(sp);
                } else {
#pragma unroll
                    for (int e = 0; e < 16; ++e) s.b[e] = sp[e];
                }
#pragma unroll
                for (int p = 0; p < 8; ++p)
                    sg[i1 * Q + q][p] = pk16((float)s.b[2 * p], (float)s.b[2 * p + 1]);
            }
    }

    // stage-A operands of one row: xa[i1][ks] = X[c][128 i1 + 16 ks + 8 g ..]
    v4i xa[P][KA];
    auto fetch = [&](int64_t row) __attribute__((always_inline)) {
        // the resource covers the row: chunks past K read zeros
        const __amdgpu_buffer_rsrc_t xr = make_rsrc(a.x + row * n, (int64_t)n * 2);
        const uint32_t off = (uint32_t)(c * M + 8 * g) * 2;
#pragma unroll
        for (int i1 = 0; i1 < P; ++i1)
#pragma unroll
            for (int ks = 0; ks < KA; ++ks)
                xa[i1][ks] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                                                         xr, off + i1 * 256 + ks * 32, 0, 0));
    };
    // the next row is prefetched where its registers fit beside the rest
    constexpr bool PRE = P * KA * 4 + KS * 4 + T * 16 <= 160;
    int64_t row = blockIdx.x;
    if (PRE && row < a.rows) fetch(row);
    lds_barrier();

    for (; row < a.rows; row += gridDim.x) {
        if (!PRE) fetch(row);
        // ---- stage A
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int nt = wi * Q + q;
            v16f d[P];
#pragma unroll
            for (int i1 = 0; i1 < P; ++i1) d[i1] = (v16f){};
#pragma unroll
            for (int ks = 0; ks < KA; ++ks) {
                const u32 f = flip_g ^ ((ks & 1) ? flip_16 : 0u) ^
                              (parity((ks >> 1) & nt) ? 0x80008000u : 0u);
                Frag b;
#pragma unroll
                for (int i = 0; i < 4; ++i) b.w[i] = pat.w[i] ^ f;
#pragma unroll
                for (int i1 = 0; i1 < P; ++i1)
                    d[i1] = mfma32(__builtin_bit_cast(v8h, xa[i1][ks]), b.h, d[i1]);
            }
#pragma unroll
            for (int h = 1; h < P; h <<= 1)
#pragma unroll
                for (int i1 = 0; i1 < P; ++i1)
                    if (!(i1 & h))
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            const float lo = d[i1][v], hi = d[i1 + h][v];
                            d[i1][v] = lo + hi;
                            d[i1 + h][v] = lo - hi;
                        }
            // register v of the lane: chunk 32 ct + 8 (v / 4) + 4 g + v % 4
#pragma unroll
            for (int i1 = 0; i1 < P; ++i1) {
                f16 *dst = yT + (i1 * 128 + 32 * nt + ln) * LD + 32 * ct + 4 * g;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float y[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        y[r] = d[i1][4 * j + r] * a.scale;
                        // pin the fp32 product: fp16(fp32(x * s)), two roundings
                        asm volatile("" : "+v"(y[r]));
                    }
                    if (32 * ct + 8 * j + 8 <= KS * 16)
                        *reinterpret_cast<v2u *>(dst + 8 * j) =
                            (v2u){pk16(y[0], y[1]), pk16(y[2], y[3])};
                }
            }
        }
        if (PRE && row + gridDim.x < a.rows) fetch(row + gridDim.x);
        lds_barrier();

        // ---- stage K
        u32 w[T][8];
        const int ip = 16 * ((ln >> 2) & 1) + 4 * (ln >> 3) + (ln & 3);
#pragma unroll
        for (int i1 = 0; i1 < P; ++i1)
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const f16 *src = yT + (i1 * 128 + 32 * (wi * Q + q) + ip) * LD + 8 * g;
                v16f z = {};
#pragma unroll
                for (int s = 0; s < KS; ++s)
                    z = mfma32(*reinterpret_cast<const v8h *>(src + 16 * s), hb[s], z);
#pragma unroll
                for (int p = 0; p < 8; ++p) {
                    const v2h v = __builtin_bit_cast(v2h, pk16(z[2 * p], z[2 * p + 1]));
                    w[i1 * Q + q][p] = __builtin_bit_cast(
                        u32, v * __builtin_bit_cast(v2h, sg[i1 * Q + q][p]));
                }
            }

        if constexpr (MODE == 0) {
            if (live) {
#pragma unroll
                for (int i1 = 0; i1 < P; ++i1)
#pragma unroll
                    for (int q = 0; q < Q; ++q) {
                        v4u *o = reinterpret_cast<v4u *>(a.out + row * n + out_at(i1, q));
                        const u32 *t = w[i1 * Q + q];
                        o[0] = (v4u){t[0], t[1], t[2], t[3]};
                        o[1] = (v4u){t[4], t[5], t[6], t[7]};
                    }
            }
            lds_barrier();  // every wave has read yT
        } else {
            // row reduction.  ab: NaN-propagating max |x|, beyond 65504 (or
            // NaN) when the lane holds a non-finite value; mx / mn ignore
            // NaN, as the reference's fmaxf / fminf do.
            v2h ab = {0, 0}, mx, mn;
            mx = (v2h){(f16)-__builtin_inff(), (f16)-__builtin_inff()};
            mn = -mx;
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int p = 0; p < 8; ++p) {
                    const v2h v = __builtin_bit_cast(v2h, w[t][p]);
                    ab = __builtin_elementwise_maximum(ab, __builtin_elementwise_abs(v));
                    if (MODE == 2) {
                        mx = __builtin_elementwise_max(mx, v);
                        mn = __builtin_elementwise_min(mn, v);
                    }
                }
            float al = __builtin_elementwise_maximum((float)ab[0], (float)ab[1]);
            if (!live) al = 0.f;
            const bool wbad = __builtin_amdgcn_ballot_w64(!(al <= 65504.f)) != 0;
            if (MODE == 1) {
                if (wbad) {  // the NaN-ignoring max
                    al = 0.f;
                    if (live) {
#pragma unroll
                        for (int t = 0; t < T; ++t)
#pragma unroll
                            for (int p = 0; p < 8; ++p) {
                                u32 u = w[t][p];
                                asm volatile("" : "+v"(u));  // keep behind the branch
                                const v2h v = __builtin_bit_cast(v2h, u);
                                al = fmaxf(fmaxf(al, fabsf((float)v[0])), fabsf((float)v[1]));
                            }
                    }
                }
                al = wave_max_dpp(al);
                if (lane == 0) {
                    red[0][wave] = al;
                    red[1][wave] = wbad ? 1.f : 0.f;
                }
            } else {
                float fmx = fmaxf((float)mx[0], (float)mx[1]);
                float fmn = fminf((float)mn[0], (float)mn[1]);
                if (!live) {
                    fmx = -__builtin_inff();
                    fmn = __builtin_inff();
                }
                fmx = wave_max_dpp(fmx);
                fmn = -wave_max_dpp(-fmn);
                if (lane == 0) {
                    red[0][wave] = fmx;
                    red[1][wave] = wbad ? 1.f : 0.f;
                    red[2][wave] = fmn;
                }
            }
            lds_barrier();  // and every wave has read yT
            float rmax = red[0][0], rbad = red[1][0], rmin = MODE == 2 ? red[2][0] : 0.f;
            for (int i = 1; i < nwaves; ++i) {
                rmax = fmaxf(rmax, red[0][i]);
                rbad += red[1][i];
                if (MODE == 2) rmin = fminf(rmin, red[2][i]);
            }
            const bool bad = __builtin_amdgcn_readfirstlane(rbad != 0.f);
            uint8_t *qr = a.q + row * (int64_t)(n / 2);
            if constexpr (MODE == 1) {
                const f16 s16 = sym_row_scale(rmax, a.clip);
                const float sf = (float)s16, rcp = sym_rcp_safe(sf);
                if (threadIdx.x == 0) a.qscale[row] = s16;
                const bool clampit = __builtin_amdgcn_readfirstlane(sym_row_needs_clamp(rmax, sf));
                const float rx = sym_recip(sf);
                auto codes = [&](const u32 *t) __attribute__((always_inline)) {
                    if (bad) {
                        v2u r = {0, 0};
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            const float x = (float)__builtin_bit_cast(v2h, t[e / 2])[e & 1];
                            r[e / 8] |= (u32)(sym_code_r(x, rx) & 0xF) << (4 * (e % 8));
                        }
                        return r;
                    }
                    u32 o[8];
                    if (clampit) {
#pragma unroll
                        for (int p = 0; p < 8; ++p) o[p] = offset_codes<true>(quot2(t[p], rcp));
                    } else {
#pragma unroll
                        for (int p = 0; p < 8; ++p) o[p] = offset_codes<false>(quot2(t[p], rcp));
                    }
                    return (v2u){pack8(o[0], o[1], o[2], o[3]), pack8(o[4], o[5], o[6], o[7])};
                };
                if (live) {
#pragma unroll
                    for (int i1 = 0; i1 < P; ++i1)
#pragma unroll
                        for (int q = 0; q < Q; ++q)
                            __builtin_nontemporal_store(
                                codes(w[i1 * Q + q]),
                                reinterpret_cast<v2u *>(qr + out_at(i1, q) / 2));
                }
            } else {
                f16 sh, zh;
                asym_row_params(rmin, rmax, a.clip, sh, zh);
                if (threadIdx.x == 0) {
                    a.qscale[row] = sh;
                    if (a.qzero) a.qzero[row] = zh;
                    if (a.qzero8) a.qzero8[row] = zero_i8(zh);
                }
                const float sf = (float)sh;
                const int zi = h2i_rn((float)zh);
                const bool fast = __builtin_amdgcn_readfirstlane(!bad && sf > 0.f && zi >= -511 &&
                                                                 zi <= 511);
                const float rcp = 1.0f / fmaxf(sf, 0x1p-126f);
                const f16 l1 = (f16)(float)(-zi), h1 = (f16)(float)(15 - zi), z1 = (f16)(float)zi;
                const v2h lo = {l1, l1}, hi = {h1, h1}, zo = {z1, z1};
                auto codes = [&](const u32 *t) __attribute__((always_inline)) {
                    v2u r = {0, 0};
                    if (fast) {
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            u32 o[4];
#pragma unroll
                            for (int p = 0; p < 4; ++p)
                                o[p] = asym_offset_codes(quot2(t[4 * h + p], rcp), lo, hi, zo);
                            r[h] = pack8_raw(o[0], o[1], o[2], o[3]);
                        }
                    } else {
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            const float x = (float)__builtin_bit_cast(v2h, t[e / 2])[e & 1];
                            r[e / 8] |= (u32)(asym_code(x, sf, zi, 0, 15) & 0xF) << (4 * (e % 8));
                        }
                    }
                    return r;
                };
                if (live) {
#pragma unroll
                    for (int i1 = 0; i1 < P; ++i1)
#pragma unroll
                        for (int q = 0; q < Q; ++q)
                            __builtin_nontemporal_store(
                                codes(w[i1 * Q + q]),
                                reinterpret_cast<v2u *>(qr + out_at(i1, q) / 2));
                }
            }
        }
    }
}

}  // namespace

// Launches the kernel above for n = K * m (rotation into `out`; with q, the
// symmetric quantizer; with q and a zero-point output, the asymmetric one).  Returns 1 if
// it launched, 0 if the size or an alignment is not covered.
int srq_had_kron_mfma(const void *x, int64_t rows, int64_t n, int64_t K, const void *hadK,
                      const int8_t *sign, float clip, void *q, void *qscale, void *qzero,
                      int8_t *qzero8, void *out, hipStream_t st) {
    if (K < 12 || K > 176 || K % 4 || n % K) return 0;
    // sizes that the LDS kernel refuses (two fp32 rows beyond 160 KiB) stay
    // refused
    if (K > 64 && n > 20480) return 0;
    const int64_t m = n / K;
    if (!srq_aligned(x, 16) || !srq_aligned(hadK, 8)) return 0;
    if (q ? !srq_aligned(q, 8) : !srq_aligned(out, 16)) return 0;
    KronArgs a{};
    a.x = (const f16 *)x;
    a.rows = rows;
    a.K = (int)K;
    a.nc = (int)srq_cdiv(K, 32);
    a.hadK = (const f16 *)hadK;
    a.sign = sign;
    a.scale = 1.0f / sqrtf((float)n);
    a.clip = clip;
    a.q = (uint8_t *)q;
    a.qscale = (f16 *)qscale;
    a.qzero = (f16 *)qzero;
    a.qzero8 = qzero8;
    a.out = (f16 *)out;
    bool done = false;
    auto go = [&](auto ks, auto ka, auto p, auto qq, auto maxt, int wi) {
        constexpr int KS = decltype(ks)::value, KA = decltype(ka)::value, P = decltype(p)::value,
                      Q = decltype(qq)::value, MT = decltype(maxt)::value;
        const dim3 block((unsigned)(64 * a.nc * wi));
        // persistent blocks: enough for the resident ones of 256 CUs
        const int per_cu = std::max<int>(1, 1024 / (int)block.x);
        const dim3 grid((unsigned)std::min<int64_t>(rows, 256 * per_cu));
        if (q && (qzero || qzero8)) had_kron_kernel<KS, KA, P, Q, 2, MT><<<grid, block, 0, st>>>(a);
        else if (q) had_kron_kernel<KS, KA, P, Q, 1, MT><<<grid, block, 0, st>>>(a);
        else had_kron_kernel<KS, KA, P, Q, 0, MT><<<grid, block, 0, st>>>(a);
        done = true;
    };
#define C(v) std::integral_constant<int, v>{}
    // waves = nc * wi; wi * Q = the column tiles of a group (min(m, 128) / 32)
    if (K <= 32) {
        if (m == 64) go(C(2), C(4), C(1), C(1), C(128), 2);
        else if (m == 128) go(C(2), C(8), C(1), C(1), C(256), 4);
        else if (m == 256) go(C(2), C(8), C(2), C(1), C(256), 4);
    } else if (K <= 64) {
        if (m == 64) go(C(4), C(4), C(1), C(1), C(256), 2);
        else if (m == 128) go(C(4), C(8), C(1), C(2), C(256), 2);
        else if (m == 256) go(C(4), C(8), C(2), C(1), C(512), 4);
        else if (m == 512) go(C(4), C(8), C(4), C(1), C(512), 4);
    } else if (K <= 112) {
        if (m == 64) go(C(7), C(4), C(1), C(2), C(256), 1);
        else if (m == 128) go(C(7), C(8), C(1), C(2), C(512), 2);
    } else {
        if (m == 64) go(C(11), C(4), C(1), C(2), C(384), 1);
        else if (m == 128) go(C(11), C(8), C(1), C(2), C(768), 2);
    }
#undef C
    return done ? 1 : 0;
}
