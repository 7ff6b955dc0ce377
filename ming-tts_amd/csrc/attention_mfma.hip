// Causal GQA attention over many rows of one sequence (mt_attention) on the matrix cores.
//
// Reference kernel replaced: attention_cache<SPLIT> (Shaders.swift:490-596), for the rows that
// attention_tiles in attention.hip routes here; attention.hip keeps the row kernels.
//
// One 256-thread workgroup per (head, block of 32 rows); its four waves share the block's
// rows and take every fourth 32-key tile each, so the loop has no barrier and no LDS: a wave
// reads its keys and values straight into MFMA operand registers and keeps an online softmax.
//   - Scores: S^T = K Q^T with v_mfma_f32_32x32x16.  Lane l holds key l % 32's dims 8 (l / 32)
//     + 16 kk .. + 7 (the A operand is 16-byte loads of the row-major cache) and query row
//     l % 32's same dims (B).  The accumulator gives the lane 16 keys of its own row, so the row
//     maximum is an in-lane maximum and one swap of the wave's halves, and the softmax weights,
//     the rescaling and the sums are per-lane values.
//   - p . v: O^T = V^T P^T.  The contraction's order is free as long as both operands agree, so
//     the weights stay where the scores' accumulator put them: slot j of step kk and half g is
//     key 16 kk + 8 (j / 4) + 4 g + j % 4.  A lane loads the dims 2 i, 2 i + 1 (i = l % 32) of
//     those eight keys (each load instruction covers two whole rows) and two byte permutes a
//     pair make the A operands of the even and the odd dims.
//   - Precision: q (scaled per row by a power of two) and the weights p (scaled by 2^14) meet an
//     fp16 cache as hi + lo fp16 halves (22 bits, 2 MFMAs a product); an fp32 cache, q and p as
//     three bf16 pieces (all 24 bits) and the 6 products above 2^-24.  Sums are fp32, but an MFMA
//     rounds its sums towards zero, so the weights' sum takes the same way as p . v (ones in place of the
//     values): the same rounded weights and nearly the same loss stand above and below the fraction.
//     Normwise error against fp64 over that of the row kernel, fp16 / fp32 cache: 0.64-1.04 / 0.59-0.88
//     at 400 to 2048 rows, windows of 5 and 65 and none, queries of 0.1 to 40; values with a mean
//     0.89-1.01 / 0.82-0.87 (1.3 / 1.05 with the weights summed beside the MFMAs, which takes 0.1-1 us
//     less, 4 less at 4000 fp16 keys, and 1.1 more at 1600 fp16 rows of window 65).
//   - Tiles start at multiples of 32 keys, a tile without keys of a row adds exact zeros to it, and
//     the four waves' parts meet in wave order: a row's result does not depend on the block it falls
//     into while the cache rows that the block reads are finite.
//   - Bound: a wave's own instructions (about 240 vector instructions a tile with an fp16 cache, its 20
//     MFMAs and a share of the set-up among them: MFMAs busy 25 % of the time, waves waiting 34 %) and,
//     with few tiles a wave, its loads' latency.  2048 rows from position 0 (14 / 2 heads, graph
//     replay): 31 us with an fp16 cache, 66 us with an fp32 one (row kernels 432 and 771).  Two row
//     tiles a wave, which halve the key and value reads, took 256 registers and 36-59 us.
//   - A row with an output that is not finite (infinities and NaN in its query or keys, or in cache
//     rows that it does not attend but its block reads) is done again with the row kernel's arithmetic,
//     which touches only the row's own keys.
#include "attend_row.hpp"
#include "mt_device.hpp"
#include "mt_internal.hpp"
#include "tiled_kernel.hpp"

namespace mt {

namespace {

using tiled::f32x16t;
using tiled::u32x4t;
typedef uint32_t u32x2t __attribute__((ext_vector_type(2)));

constexpr int AM_THREADS = 256, AM_WAVES = 4;
constexpr uint32_t AM_ROWS = 32;  // query rows of a workgroup
constexpr int AM_OLD = 68;  // floats of a row in the waves' hand-over (64 and a 16-byte skew)

// x = p0 + p1 + p2 to 2^-26 or so, three bf16 pieces rounded to nearest (a truncated piece leaves
// remainders of one sign, whose dropped products add up), for a pair of values packed in one word
// a piece.
__device__ __forceinline__ void split3(float x0, float x1, uint32_t (&p)[3]) {
    p[0] = __builtin_bit_cast(uint32_t, __builtin_convertvector(tiled::f32x2t{x0, x1}, tiled::bf16x2t));
    const float r0 = x0 - bf16_lo(p[0]), r1 = x1 - bf16_hi(p[0]);
    p[1] = __builtin_bit_cast(uint32_t, __builtin_convertvector(tiled::f32x2t{r0, r1}, tiled::bf16x2t));
    const float s0 = r0 - bf16_lo(p[1]), s1 = r1 - bf16_hi(p[1]);
    p[2] = __builtin_bit_cast(uint32_t, __builtin_convertvector(tiled::f32x2t{s0, s1}, tiled::bf16x2t));
}

// v and its counterpart 32 lanes away.
__device__ __forceinline__ float swap_max(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

template <int CT>
struct AmType {
    static constexpr int MT = CT == DT_F16 ? DT_F16 : DT_BF16;  // the MFMA's type
    static constexpr int NQ = CT == DT_F16 ? 2 : 3;             // pieces of q and p
    static constexpr int NC = CT == DT_F16 ? 1 : 3;             // pieces of k and v
    static constexpr float PS = CT == DT_F16 ? 16384.0f : 1.0f;  // the weights' scale
    static constexpr uint32_t ONE = CT == DT_F16 ? 0x3C003C00u : 0x3F803F80u;  // two ones
};

// Eight values of q or p as the operand's pieces.
template <int CT>
__device__ __forceinline__ void pieces(const float (&x)[8], u32x4t (&p)[AmType<CT>::NQ]) {
    if constexpr (CT == DT_F16) {
        tiled::split8<DT_F16, true>(x, p[0], p[1]);
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            uint32_t w[3];
            split3(x[2 * e], x[2 * e + 1], w);
#pragma unroll
            for (int i = 0; i < 3; i++) p[i][e] = w[i];
        }
    }
}

// The products of a sum: every piece of q (or p) against an fp16 k (or v); of three pieces against
// three, the six that are not below 2^-24.  am_small adds all but the largest (all below 2^-8 of
// it); a sum takes those of every step first and then the largest, so it rounds at its own size
// only once a step of the latter.
template <int CT>
__device__ __forceinline__ f32x16t am_small(const u32x4t (&c)[AmType<CT>::NC], const u32x4t (&q)[AmType<CT>::NQ], f32x16t acc) {
    constexpr int T = AmType<CT>::MT;
    if constexpr (CT == DT_F16) {
        return tiled::mfma32x<T>(c[0], q[1], acc);
    } else {
        acc = tiled::mfma32x<T>(c[2], q[0], acc);
        acc = tiled::mfma32x<T>(c[0], q[2], acc);
        acc = tiled::mfma32x<T>(c[1], q[1], acc);
        acc = tiled::mfma32x<T>(c[1], q[0], acc);
        return tiled::mfma32x<T>(c[0], q[1], acc);
    }
}

template <int CT>
__global__ __launch_bounds__(AM_THREADS, 2) void attention_mfma_kernel(
    const float *q, uint32_t ldq, uint32_t hq, uint32_t hkv, uint32_t pos0, uint32_t rows, uint32_t window, const void *kc,
    const void *vc, uint32_t cache_len, float *out, uint32_t ldo, float scale) {
    typedef AmType<CT> TY;
    constexpr int ES = CT == DT_F16 ? 2 : 4;  // bytes of a cached value
    __shared__ __attribute__((aligned(16))) float part[AM_WAVES * 32 * AM_OLD];
    __shared__ float mls[2][AM_WAVES][32];
    __shared__ uint32_t redo;  // the block's rows (bits) whose outputs are not finite
    static_assert(sizeof(part) >= sizeof(RowLds), "the row kernel's scratch overlays the hand-over");
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t l32 = lane & 31, g = lane >> 5;
    const uint32_t h = blockIdx.x, kvh = h / (hq / hkv);
    const uint32_t m0 = (gridDim.y - 1 - blockIdx.y) * AM_ROWS;  // the longest rows first
    const uint32_t rn = min(AM_ROWS, rows - m0);
    const uint32_t kend = pos0 + m0 + rn;  // keys the block attends end here

    // The query rows (rows past the end repeat the last one and are never stored), their keys
    // [lo, lo + span) and the factor that turns a dot into a base-2 exponent.
    const uint32_t m = m0 + min(l32, rn - 1);
    const uint32_t hi = pos0 + m + 1;
    const uint32_t lo = window > 0 && hi > window ? hi - window : 0, span = hi - lo;
    const float *qp = q + static_cast<size_t>(m) * ldq + h * 64 + 8 * g;
    float x[4][8];
#pragma unroll
    for (int kk = 0; kk < 4; kk++) {
        const float4 a = *reinterpret_cast<const float4 *>(qp + 16 * kk), b = *reinterpret_cast<const float4 *>(qp + 16 * kk + 4);
        x[kk][0] = a.x; x[kk][1] = a.y; x[kk][2] = a.z; x[kk][3] = a.w;
        x[kk][4] = b.x; x[kk][5] = b.y; x[kk][6] = b.z; x[kk][7] = b.w;
    }
    float f = 1.0f, inv = 1.0f;
    if constexpr (CT == DT_F16) {  // the row's largest |q| to 2^13 .. 2^14
        float mx = 0.0f;
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
            for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf(x[kk][e]));
        mx = swap_max(mx);
        const int ex = min(267 - static_cast<int>(__float_as_uint(mx) >> 23), 253);
        f = __uint_as_float(static_cast<uint32_t>(ex) << 23);
        inv = __uint_as_float(static_cast<uint32_t>(254 - ex) << 23);
    }
    if (scale < 0.0f) f = -f;
    const float cexp = fabsf(scale) * 1.4426950408889634f * inv;
    u32x4t qf[4][TY::NQ];
#pragma unroll
    for (int kk = 0; kk < 4; kk++) {
#pragma unroll
        for (int e = 0; e < 8; e++) x[kk][e] *= f;
        pieces<CT>(x[kk], qf[kk]);
    }

    f32x16t o[2];
    float sub = INFINITY, ls = 0.0f;  // minus the running maximum's exponent (+infinity: no key yet), the weights' sum
#pragma unroll
    for (int r = 0; r < 16; r++) o[0][r] = o[1][r] = 0.0f;

    const char *kbase = static_cast<const char *>(kc) + static_cast<size_t>(kvh) * cache_len * 64 * ES;
    const char *vbase = static_cast<const char *>(vc) + static_cast<size_t>(kvh) * cache_len * 64 * ES;
    // A tile's raw keys (16-byte chunks of the lane's key) and values (two dims of 16 keys).  Keys
    // past the block's last one re-read it.
    u32x4t kr[4 * (ES / 2)];
    u32x2t vr[16];
    auto loadk = [&](uint32_t tile) {
        const uint32_t key = min(32 * tile + l32, kend - 1);
        const u32x4t *p = reinterpret_cast<const u32x4t *>(kbase + (key * (64 * ES) + 8 * ES * g));
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
            for (int i = 0; i < ES / 2; i++) kr[kk * (ES / 2) + i] = p[kk * ES + i];
    };
    auto ldv = [&](const char *p) {
        if constexpr (CT == DT_F16) return u32x2t{*reinterpret_cast<const uint32_t *>(p), 0u};
        else return *reinterpret_cast<const u32x2t *>(p);
    };
    auto loadv = [&](uint32_t tile) {
        if (32 * tile + 32 <= kend) {
            const char *p = vbase + ((32 * tile + 4 * g) * (64 * ES) + 2 * ES * l32);
#pragma unroll
            for (int s = 0; s < 16; s++) vr[s] = ldv(p + (8 * (s >> 2) + (s & 3)) * (64 * ES));
        } else {
#pragma unroll
            for (int s = 0; s < 16; s++) {
                const uint32_t key = min(32 * tile + 4 * g + 8 * (s >> 2) + (s & 3), kend - 1);
                vr[s] = ldv(vbase + (key * (64 * ES) + 2 * ES * l32));
            }
        }
    };

    // Tiles [t0, t1) of the block, this wave's every fourth.
    const uint32_t hi0 = pos0 + m0 + 1, lo1 = window > 0 && kend > window ? kend - window : 0;
    const uint32_t t0 = (window > 0 && hi0 > window ? hi0 - window : 0) / 32, t1 = (kend + 31) / 32;
    uint32_t tile = t0 + ((wave - t0) & (AM_WAVES - 1));
    if (tile < t1) {
        loadk(tile);
        loadv(tile);
    }
    for (; tile < t1; tile += AM_WAVES) {
        const uint32_t next = tile + AM_WAVES;
        // Scores, then the keys' registers take the next tile.
        f32x16t s, sb;
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = sb[r] = 0.0f;
        u32x4t c0[4];
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            u32x4t c[TY::NC];
            if constexpr (CT == DT_F16) {
                c[0] = kr[kk];
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const u32x4t w = kr[2 * kk + (e >> 1)];
                    uint32_t p[3];
                    split3(__uint_as_float(w[2 * (e & 1)]), __uint_as_float(w[2 * (e & 1) + 1]), p);
#pragma unroll
                    for (int i = 0; i < 3; i++) c[i][e] = p[i];
                }
            }
            c0[kk] = c[0];
            s = am_small<CT>(c, qf[kk], s);
        }
        // The largest products as two chains (dims 0-31 and 32-63).
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            s = tiled::mfma32x<TY::MT>(c0[kk], qf[kk][0], s);
            sb = tiled::mfma32x<TY::MT>(c0[2 + kk], qf[2 + kk][0], sb);
        }
        s += sb;
        if (next < t1) loadk(next);

        // Does every key of the tile belong to every row (the last row's window, the first row's end)?
        const bool whole = 32 * tile >= lo1 && 32 * tile + 32 <= hi0;
        if (!whole) {
            const uint32_t k0 = 32 * tile + 4 * g - lo;
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = k0 + (8 * (r >> 2) + (r & 3)) < span ? s[r] : -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; r++) mx = fmaxf(mx, s[r]);
        mx = swap_max(mx);
        const float sn = fminf(sub, -(mx * cexp));
        const float al = sn == sub ? 1.0f : __builtin_amdgcn_exp2f(sn - sub);  // brings older sums to the new maximum
        sub = sn;
        const float su = sub == INFINITY ? 0.0f : sub;
        float p[16];
#pragma unroll
        for (int r = 0; r < 16; r++) p[r] = __builtin_amdgcn_exp2f(fmaf(s[r], cexp, su));
        u32x4t pf[2][TY::NQ];
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            float x8[8];
#pragma unroll
            for (int e = 0; e < 8; e++) x8[e] = p[8 * kk + e] * TY::PS;
            pieces<CT>(x8, pf[kk]);
        }

        // The weights' sum: p . v with ones for v.
        f32x16t lt;
#pragma unroll
        for (int r = 0; r < 16; r++) lt[r] = 0.0f;
        const u32x4t ones = {TY::ONE, TY::ONE, TY::ONE, TY::ONE};
#pragma unroll
        for (int i = TY::NQ - 1; i > 0; i--)
#pragma unroll
            for (int kk = 0; kk < 2; kk++) lt = tiled::mfma32x<TY::MT>(ones, pf[kk][i], lt);
#pragma unroll
        for (int kk = 0; kk < 2; kk++) lt = tiled::mfma32x<TY::MT>(ones, pf[kk][0], lt);
        ls = fmaf(ls, al, lt[0]);

        // p . v: d = 0 the even dims, 1 the odd ones.  A tile's sum starts from zero and joins the
        // running one in one rounding.
#pragma unroll
        for (int d = 0; d < 2; d++) {
            u32x4t c[2][TY::NC];
#pragma unroll
            for (int kk = 0; kk < 2; kk++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const u32x2t a = vr[8 * kk + 2 * e], b = vr[8 * kk + 2 * e + 1];
                    if constexpr (CT == DT_F16) {
                        c[kk][0][e] = __builtin_amdgcn_perm(b[0], a[0], d == 0 ? 0x05040100u : 0x07060302u);
                    } else {
                        uint32_t w[3];
                        split3(__uint_as_float(a[d]), __uint_as_float(b[d]), w);
#pragma unroll
                        for (int i = 0; i < 3; i++) c[kk][i][e] = w[i];
                    }
                }
            f32x16t ot;
#pragma unroll
            for (int r = 0; r < 16; r++) ot[r] = 0.0f;
#pragma unroll
            for (int kk = 0; kk < 2; kk++) ot = am_small<CT>(c[kk], pf[kk], ot);
#pragma unroll
            for (int kk = 0; kk < 2; kk++) ot = tiled::mfma32x<TY::MT>(c[kk][0], pf[kk][0], ot);
#pragma unroll
            for (int r = 0; r < 16; r++) o[d][r] = fmaf(o[d][r], al, ot[r]);
        }
        if (next < t1) loadv(next);
    }

    // The waves' parts of each row meet in wave order: thread (row, d8) joins dims 8 d8 .. + 7.
    float *op = part + (wave * 32 + l32) * AM_OLD + 8 * g;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        *reinterpret_cast<float4 *>(op + 16 * r) = make_float4(o[0][4 * r], o[1][4 * r], o[0][4 * r + 1], o[1][4 * r + 1]);
        *reinterpret_cast<float4 *>(op + 16 * r + 4) =
            make_float4(o[0][4 * r + 2], o[1][4 * r + 2], o[0][4 * r + 3], o[1][4 * r + 3]);
    }
    if (tid == 0) redo = 0;
    if (g == 0) {
        mls[0][wave][l32] = sub;
        mls[1][wave][l32] = ls;
    }
    __syncthreads();
    const int row = tid >> 3, d8 = tid & 7;
    const bool mine = row < static_cast<int>(rn);
    float mm = mls[0][0][row];
#pragma unroll
    for (int w = 1; w < AM_WAVES; w++) mm = fminf(mm, mls[0][w][row]);
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, total = 0.0f;
#pragma unroll
    for (int w = 0; w < AM_WAVES; w++) {
        const float mw = mls[0][w][row];
        const float wt = mw == INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mm - mw);
        total = fmaf(mls[1][w][row], wt, total);
        const float *pp = part + (w * 32 + row) * AM_OLD + 8 * d8;
        const float4 a = *reinterpret_cast<const float4 *>(pp), b = *reinterpret_cast<const float4 *>(pp + 4);
        acc[0] = fmaf(a.x, wt, acc[0]); acc[1] = fmaf(a.y, wt, acc[1]);
        acc[2] = fmaf(a.z, wt, acc[2]); acc[3] = fmaf(a.w, wt, acc[3]);
        acc[4] = fmaf(b.x, wt, acc[4]); acc[5] = fmaf(b.y, wt, acc[5]);
        acc[6] = fmaf(b.z, wt, acc[6]); acc[7] = fmaf(b.w, wt, acc[7]);
    }
    const float il = 1.0f / total;
    bool ok = true;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        acc[e] *= il;
        ok = ok && fabsf(acc[e]) < INFINITY;
    }
    if (mine && !ok) atomicOr(&redo, 1u << row);
    __syncthreads();
    const uint32_t again = redo;
    if (mine && !((again >> row) & 1)) {
        float *orow = out + static_cast<size_t>(m0 + row) * ldo + h * 64 + 8 * d8;
        *reinterpret_cast<float4 *>(orow) = make_float4(acc[0], acc[1], acc[2], acc[3]);
        *reinterpret_cast<float4 *>(orow + 4) = make_float4(acc[4], acc[5], acc[6], acc[7]);
    }
    // The rest once more, a row's query still in place also where out is q.
    for (uint32_t left = again; left; left &= left - 1) {
        RowLds *rl = reinterpret_cast<RowLds *>(part);
        const uint32_t r = __builtin_ctz(left);
        const uint32_t end = pos0 + m0 + r + 1, first = window > 0 && end > window ? end - window : 0;
        attend_row<CT, 2, 2>(q + static_cast<size_t>(m0 + r) * ldq + h * 64, kc, vc,
                             (static_cast<size_t>(kvh) * cache_len + first) * 64, static_cast<int>(end - first), scale,
                             out + static_cast<size_t>(m0 + r) * ldo + h * 64, rl->sc, rl->red, rl->part);
        __syncthreads();
    }
}

}  // namespace

int launch_attention_mfma(const float *q, uint32_t ldq, uint32_t rows, uint32_t hq, uint32_t hkv, uint32_t pos0,
                          uint32_t window, const void *kc, const void *vc, int ct, uint32_t cache_len, float *out,
                          uint32_t ldo, float scale, hipStream_t stream) {
    const dim3 grid(hq, (rows + AM_ROWS - 1) / AM_ROWS);
    if (ct == DT_F32)
        hipLaunchKernelGGL(attention_mfma_kernel<DT_F32>, grid, dim3(AM_THREADS), 0, stream, q, ldq, hq, hkv, pos0, rows,
                           window, kc, vc, cache_len, out, ldo, scale);
    else
        hipLaunchKernelGGL(attention_mfma_kernel<DT_F16>, grid, dim3(AM_THREADS), 0, stream, q, ldq, hq, hkv, pos0, rows,
                           window, kc, vc, cache_len, out, ldo, scale);
    return check_launch("attention (mfma)");
}

}  // namespace mt
