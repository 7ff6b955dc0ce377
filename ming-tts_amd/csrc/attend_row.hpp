// The row kernel's attention: one 256-thread workgroup over one (query row, head) item, shared by
// attention_kernel (attention.hip) and by the tile kernel's fallback (attention_mfma.hip).
#pragma once

#include "mt_device.hpp"

namespace mt {

constexpr int ATT_THREADS = 256;
constexpr int ATT_MAXKEYS = 4096;

template <int CT>
__device__ __forceinline__ float4 load4(const void *base, size_t off) {
    if constexpr (CT == DT_F32) {
        return *reinterpret_cast<const float4 *>(static_cast<const float *>(base) + off);
    } else {
        const uint2 v = *reinterpret_cast<const uint2 *>(static_cast<const uint16_t *>(base) + off);
        return make_float4(dec_lo<CT>(v.x), dec_hi<CT>(v.x), dec_lo<CT>(v.y), dec_hi<CT>(v.y));
    }
}

// Max / sum over the 64 lanes, the same bits in every lane: quad swaps and the half-row and
// row mirrors on DPP (rows of 16), then two exchanges between rows.
__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, dpp_mov<0xB1>(v));
    v = fmaxf(v, dpp_mov<0x4E>(v));
    v = fmaxf(v, dpp_mov<0x141>(v));
    v = fmaxf(v, dpp_mov<0x140>(v));
    v = fmaxf(v, __shfl_xor(v, 16, 64));
    return fmaxf(v, __shfl_xor(v, 32, 64));
}
__device__ __forceinline__ float wave_sum(float v) { return group_sum(v, 64); }

// The 16-byte raw loads of eight cached values (one of fp16, two of fp32) and their decode.
template <int CT>
struct Raw8 {
    uint4 a, b;
};
template <int CT>
__device__ __forceinline__ Raw8<CT> load8_raw(const void *base, size_t off) {
    Raw8<CT> r;
    if constexpr (CT == DT_F32) {
        const uint4 *p = reinterpret_cast<const uint4 *>(static_cast<const float *>(base) + off);
        r.a = p[0];
        r.b = p[1];
    } else {
        r.a = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(base) + off);
        r.b = make_uint4(0u, 0u, 0u, 0u);
    }
    return r;
}
template <int CT>
__device__ __forceinline__ void decode8(const Raw8<CT> &r, float *o) {
    if constexpr (CT == DT_F32) {
        o[0] = __uint_as_float(r.a.x); o[1] = __uint_as_float(r.a.y); o[2] = __uint_as_float(r.a.z); o[3] = __uint_as_float(r.a.w);
        o[4] = __uint_as_float(r.b.x); o[5] = __uint_as_float(r.b.y); o[6] = __uint_as_float(r.b.z); o[7] = __uint_as_float(r.b.w);
    } else {
        unpack8<CT>(r.a, o);
    }
}

// Its LDS: the scores, the waves' maxima and sums, the phases' partial p.v sums.
struct RowLds {
    float sc[ATT_MAXKEYS];
    float red[ATT_THREADS / 64];
    float4 part[16][16];
};

// Attention of one row: queries qrow[64], keys and values at elements kvbase .. of the caches (nk
// rows of 64), the result to orow[64].  KU / VU: key passes and value rows requested at a time (no
// result depends on them).
template <int CT, int KU, int VU>
__device__ __forceinline__ void attend_row(const float *qrow, const void *kc, const void *vc, size_t kvbase, int nk,
                                           float scale, float *orow, float *sc, float *red, float4 (*part)[16]) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    // Scores.
    const int r = tid & 7;
    float qf[8];
    {
        const float4 *qp = reinterpret_cast<const float4 *>(qrow + 8 * r);
        const float4 a = qp[0], b = qp[1];
        qf[0] = a.x; qf[1] = a.y; qf[2] = a.z; qf[3] = a.w;
        qf[4] = b.x; qf[5] = b.y; qf[6] = b.z; qf[7] = b.w;
    }
    // KU passes of 32 keys per round, all requested before any is used (keys past the end
    // re-read the last key and are skipped).
    float mx = -INFINITY;
    constexpr int KP = ATT_THREADS / 8;
    for (int t0 = tid >> 3; t0 < nk; t0 += KU * KP) {
        Raw8<CT> kr[KU];
#pragma unroll
        for (int u = 0; u < KU; u++) {
            const int t = min(t0 + u * KP, nk - 1);
            kr[u] = load8_raw<CT>(kc, kvbase + static_cast<size_t>(t) * 64 + 8 * r);
        }
#pragma unroll
        for (int u = 0; u < KU; u++) {
            const int t = t0 + u * KP;
            if (t < nk) {  // the 8 lanes of a key agree
                float kf[8];
                decode8<CT>(kr[u], kf);
                float s = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) s = fmaf(qf[e], kf[e], s);
                s = octet_sum(s);
                s *= scale;
                if (r == 0) sc[t] = s;
                mx = fmaxf(mx, s);
            }
        }
    }
    mx = wave_max(mx);
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    __syncthreads();

    // Softmax numerators and their sum.
    float sum = 0.0f;
    for (int t = tid; t < nk; t += ATT_THREADS) {
        const float e = exp_hw(sc[t] - mx);
        sc[t] = e;
        sum += e;
    }
    sum = wave_sum(sum);
    if (lane == 0) red[wave] = sum;
    __syncthreads();
    sum = (red[0] + red[1]) + (red[2] + red[3]);

    // p . v: 16 lanes per V row (4 dims each), 16 key phases, keys t = ks, ks + 16, ... in
    // order; VU rows per round requested before any is used (rows past the end re-read
    // the last row and are skipped).
    const int d4 = tid & 15, ks = tid >> 4;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int t0 = ks; t0 < nk; t0 += 16 * VU) {
        float4 v[VU];
#pragma unroll
        for (int u = 0; u < VU; u++)
            v[u] = load4<CT>(vc, kvbase + static_cast<size_t>(min(t0 + 16 * u, nk - 1)) * 64 + 4 * d4);
#pragma unroll
        for (int u = 0; u < VU; u++) {
            const int t = t0 + 16 * u;
            if (t < nk) {
                const float p = sc[t];
                acc.x = fmaf(p, v[u].x, acc.x);
                acc.y = fmaf(p, v[u].y, acc.y);
                acc.z = fmaf(p, v[u].z, acc.z);
                acc.w = fmaf(p, v[u].w, acc.w);
            }
        }
    }
    part[ks][d4] = acc;
    __syncthreads();
    if (tid < 16) {
        float4 o = part[0][tid];
        for (int k = 1; k < 16; k++) {
            const float4 pp = part[k][tid];
            o.x += pp.x; o.y += pp.y; o.z += pp.z; o.w += pp.w;
        }
        const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
        float4 res = make_float4(o.x * inv, o.y * inv, o.z * inv, o.w * inv);
        *reinterpret_cast<float4 *>(orow + 4 * tid) = res;
    }
}

}  // namespace mt
