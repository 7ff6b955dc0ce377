// MFMA GEMM of mt_linear for fp32 activations over many rows (prefill, the audio encoder's frames,
// the clone path's latents): the activations go from memory straight to the operand registers of
// the one wave that multiplies them, and only the weights pass through LDS.
//
// Reference kernel replaced: gemm_kernel<32,64,32,4> (Shaders.swift:297-410), whose X is fp32.
//
// y[m][n] = epilogue(sum_k x[m][k] w[n][k]) on a workgroup of 2 WM waves per tile of 32 WM rows x 32
// CB weight rows (GATED: blocks of 32 rows of W and W2 for the same features alternate), K a multiple
// of 64.
//   - Wave (wm, kh) owns x rows 32 wm .. + 31 and half of every 64-k stage, against all CB weight
//     blocks on v_mfma_f32_32x32x16.  No other wave needs those x values: the lane loads its row's
//     eight k of each 16-k step (two 16-byte loads), multiplies them by the norm gain (NORM) while
//     summing x^2, and splits them into hi + lo halves of the weights' type in the registers the
//     MFMA reads.  Staged through LDS instead (ring_split_kernel, tiled_kernel), the two planes are
//     written once and read once, more LDS traffic than the weights', and the conversion stands
//     between two barriers.
//   - A step's x registers take the stage after the next as soon as they are converted, and the weights
//     travel global -> LDS (buffer_load ... lds) NS stages ahead; a request past the last stage has an offset
//     outside the buffer, which reads nothing, so the loop has no branch and the compiler's waits for
//     x are exact.  One barrier a stage.
//   - The two halves' sums meet through LDS (first + second), each wave finishing half of the
//     accumulator registers.
//   - Bound: the x loads (a lane's 16 bytes are its row's own, so an instruction takes a cycle for each
//     of its 64 pieces) and, with one tile a CU, a tile's first loads and epilogue.  The same tiles
//     with x through LDS as fp32 (direct loads) were bound by LDS writes instead and no faster
//     (gate|up at 2048 rows 101 us), nor were persistent workgroups that load the next tile during the
//     epilogue (97 us against 96-104).  Graph replay over six sets of operands, fp16 weights, against
//     ring_split_kernel or tiled_kernel: rmsnorm+gate|up 115 -> 106 us at 2048 rows, 89 -> 79 at 1600,
//     61 -> 52 at 1024, 30.9 -> 26.6 at 512, 25.4 -> 19.0 at 256; rmsnorm+qkv 26.4 -> 19.7 at 2048; the DiT
//     block's qkv (bf16) 27.4 -> 22.0 and ff1 28.4 -> 27.3 at 800.  One layer over 2048 rows 252 -> 243
//     us, the DiT block over 800 rows 107 -> 102 us.  MFMAs busy 29 % of the time (gate|up at 2048 rows),
//     waves waiting 31 %, 71 % of the reads hit L2.
#pragma once

#include "tiled_kernel.hpp"

namespace mt {
namespace direct {

using tiled::f32x16t;
using tiled::f32x4t;
using tiled::u32x4t;

constexpr int SK = 64, NS = 3;     // k of a stage, stages of weights in LDS
constexpr int QN = 2, XN = 2 * QN;  // 16-k steps a wave takes of a stage, its x loads
constexpr uint32_t NORM_K = 2048;  // longest K of a normed linear (its gain is held in LDS)

struct DirectArgs {
    const float *x;
    const uint16_t *w, *w2, *bias, *norm;
    float *y;
    uint32_t M, N, K, ldx, ldy, flags;
    float eps;
    uint32_t tiles_m, tiles_n;
    uint32_t x_bytes, w_bytes;  // extents of x and of each weight matrix
};

// One wave-wide load to LDS: lane l's 16 bytes at offset voff + soff of the buffer land at LDS byte
// lds + 16 l (lds wave-uniform).  An offset past the buffer reads nothing.
__device__ __forceinline__ void buffer_to_lds(__amdgpu_buffer_rsrc_t r, uint32_t lds, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, reinterpret_cast<__attribute__((address_space(3))) void *>(lds), 16, voff, soff,
                                             0, 0);
}

template <int WM, int CB>
struct Shape {
    static constexpr int NW = 2 * WM, NT = 64 * NW;
    static constexpr int BM = 32 * WM, BR = 32 * CB;  // x rows, weight rows
    static constexpr int SB = BR * 128;               // bytes of a stage
    static constexpr int LPW = SB / 1024 / NW;        // 1 KB loads per wave per stage
    static constexpr int XB = WM * 8192;              // hand-over bytes of one weight block
    static constexpr int XC = NS * SB / XB < CB ? NS * SB / XB : CB;  // blocks handed over at a time
    static_assert(LPW * NW * 1024 == SB && NS * SB <= 152 * 1024 && XC >= 1, "direct shape");
};

template <int WT, int WM, int CB, bool GATED, bool NORM>
__global__ __launch_bounds__(128 * WM, 2) void direct_kernel(DirectArgs a) {
    typedef Shape<WM, CB> S;
    constexpr int FN = GATED ? S::BR / 2 : S::BR;
    static_assert(!GATED || CB % 2 == 0, "gate and up blocks alternate");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[NS * S::SB];
    __shared__ __attribute__((aligned(16))) uint16_t gain[NORM ? NORM_K : 8];
    __shared__ float rs[NORM ? 2 * S::BM : 1];
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = wave % WM, kh = wave / WM;
    const uint32_t fr = lane & 31, fh = lane >> 5;

    const uint32_t t = tiled::xcd_order(blockIdx.x, gridDim.x);
    const uint32_t tm = t % a.tiles_m, tn = t / a.tiles_m;
    const uint32_t m0 = tm * S::BM, n0 = tn * FN;
    const uint32_t M = a.M, N = a.N, K = a.K;
    const uint32_t nsteps = K / SK;

    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.x), 0, static_cast<int>(a.x_bytes), 0x00020000);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(a.w), 0, static_cast<int>(a.w_bytes), 0x00020000);
    const __amdgpu_buffer_rsrc_t ur = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(GATED ? a.w2 : a.w), 0, static_cast<int>(a.w_bytes), 0x00020000);

    // Weight loads: load i of this wave fills rows 8 b .. + 7 of a stage, b = wave + NW i; the lane slot
    // lane & 7 of row r with chunk (lane & 7) ^ (r & 7) ^ ((r >> 3) & 1), so that the operand reads (32
    // rows of one chunk) are free of bank conflicts.  Rows past N repeat the last one (their sums are not stored).
    uint32_t woff[S::LPW];
    bool up[S::LPW];
#pragma unroll
    for (int i = 0; i < S::LPW; i++) {
        const uint32_t b = wave + S::NW * i, r = 8 * b + (lane >> 3), ch = (lane & 7) ^ (r & 7) ^ ((r >> 3) & 1);
        up[i] = GATED && ((b >> 2) & 1);
        const uint32_t n = n0 + (GATED ? 32 * (b >> 3) + (r & 31) : r);
        woff[i] = (min(n, N - 1) * K + 8 * ch) * 2;
    }
    const uint32_t lds0 =
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void *)(lds)));
    auto issue = [&](uint32_t s, uint32_t slot) {
        const uint32_t out = s < nsteps ? 0u : 0x80000000u, so = s < nsteps ? s * (2 * SK) : 0u;
#pragma unroll
        for (int i = 0; i < S::LPW; i++) {
            const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + slot * S::SB + (wave + S::NW * i) * 1024);
            buffer_to_lds(up[i] ? ur : wr, dst, woff[i] | out, so);
        }
    };

    // x: row 32 wm + fr of the tile (rows past M repeat the last one), k 16 q + 8 fh of the wave's
    // part of a stage.
    const uint32_t xoff = (min(m0 + 32 * wm + fr, M - 1) * a.ldx + (SK / 2) * kh + 8 * fh) * 4;
    u32x4t xv[2][QN][2];  // stages s and s + 1, by the stage's parity
    float ss[2] = {0.0f, 0.0f};  // the lane's sums of x^2, k even and odd (NORM)
    // after: a value that needs all of the registers' old contents (a request that the compiler
    // moves ahead of a last use gets other registers, and the copies back wait for it).
    auto loadx = [&](uint32_t s, u32x4t (&xq)[2], int q, uint32_t after) {
        const uint32_t so = s < nsteps ? s * (4 * SK) : 0u;
        uint32_t vo = xoff | (s < nsteps ? 0u : 0x80000000u);
        asm volatile("" : "+v"(vo) : "v"(after), "v"(ss[0]), "v"(ss[1]));
        xq[0] = __builtin_bit_cast(u32x4t, __builtin_amdgcn_raw_buffer_load_b128(xr, vo + 64 * q, so, 0));
        xq[1] = __builtin_bit_cast(u32x4t, __builtin_amdgcn_raw_buffer_load_b128(xr, vo + 64 * q + 16, so, 0));
    };

    // Weight operand reads: row fr of a 32-row block, chunk 2 q + fh of the wave's half.
    uint32_t boff[QN];
#pragma unroll
    for (int q = 0; q < QN; q++) {
        boff[q] = fr * 128 + (((2 * (QN * kh + q) + fh) ^ (fr & 7) ^ ((fr >> 3) & 1)) << 4);
    }
    f32x16t acc[CB];
#pragma unroll
    for (int j = 0; j < CB; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[j][r] = 0.0f;

    if constexpr (NORM) {
        for (uint32_t i = tid; i < K / 8; i += S::NT)
            reinterpret_cast<u32x4t *>(gain)[i] = reinterpret_cast<const u32x4t *>(a.norm)[i];
    }
    float bv[CB];
#pragma unroll
    for (int j = 0; j < CB; j++) {
        const uint32_t n = n0 + (GATED ? 32 * (j >> 1) : 32 * j) + fr;
        bv[j] = (a.flags & F_BIAS) && n < N && !(GATED && (j & 1)) ? dec1<WT>(a.bias[n]) : 0.0f;
    }
    // The order of the loop's requests (x of a stage, then weights two stages on), so that the
    // compiler's waits at its head are those of the back edge.
#pragma unroll
    for (int i = 0; i < NS - 1; i++) issue(i, i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int q = 0; q < QN; q++) loadx(s, xv[s][q], q, 0u);
    __builtin_amdgcn_sched_barrier(0);
    issue(NS - 1, NS - 1);
    tiled::wait_vm<(NS - 1) * S::LPW + 2 * XN>();
    tiled::tiled_bar();

    uint32_t slot = 0;
    auto stage = [&](uint32_t s, u32x4t (&xs)[QN][2]) {
        const uint8_t *st = lds + slot * S::SB;
#pragma unroll
        for (int q = 0; q < QN; q++) {
            u32x4t b[CB];
#pragma unroll
            for (int j = 0; j < CB; j++) b[j] = *reinterpret_cast<const u32x4t *>(st + boff[q] + j * 4096);
            float x[8];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                x[e] = __uint_as_float(xs[q][0][e]);
                x[4 + e] = __uint_as_float(xs[q][1][e]);
            }
            if constexpr (NORM) {
                const u32x4t gv = *reinterpret_cast<const u32x4t *>(gain + s * SK + 16 * (QN * kh + q) + 8 * fh);
#pragma unroll
                for (int e = 0; e < 8; e++) ss[e & 1] = fmaf(x[e], x[e], ss[e & 1]);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if constexpr (WT == DT_F16) {  // x times the fp16 gain in one mixed fma each
                        float p0, p1;
                        asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[0,1,0]" : "=v"(p0) : "v"(x[2 * e]), "v"(gv[e]));
                        asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[0,1,0] op_sel_hi:[0,1,0]"
                            : "=v"(p1) : "v"(x[2 * e + 1]), "v"(gv[e]));
                        x[2 * e] = p0;
                        x[2 * e + 1] = p1;
                    } else {
                        x[2 * e] *= dec_lo<WT>(gv[e]);
                        x[2 * e + 1] *= dec_hi<WT>(gv[e]);
                    }
                }
            }
            u32x4t ah, al;
            tiled::split8<WT, true>(x, ah, al);
            loadx(s + 2, xs[q], q, al[3]);
#pragma unroll
            for (int j = 0; j < CB; j++) acc[j] = tiled::mfma32x<WT>(al, b[j], acc[j]);
#pragma unroll
            for (int j = 0; j < CB; j++) acc[j] = tiled::mfma32x<WT>(ah, b[j], acc[j]);
            __builtin_amdgcn_sched_barrier(0);
        }
        // Stage s + 1 is in once the stages after it and the x requested since are the only loads in
        // flight; the barrier also tells that every wave has read stage s, whose slot takes s + NS.
        tiled::wait_vm<(NS - 2) * S::LPW + (NS - 1) * XN>();
        tiled::tiled_bar();
        issue(s + NS, slot);
        slot = slot + 1 == NS ? 0 : slot + 1;
    };
    for (uint32_t s = 0;; s += 2) {
        stage(s, xv[0]);
        if (s + 1 >= nsteps) break;
        stage(s + 1, xv[1]);
        if (s + 2 >= nsteps) break;
    }
    tiled::wait_vm<0>();

    // The rows' scales, and the parts' sums.
    if constexpr (NORM) {
        const uint32_t sb = __float_as_uint(ss[0] + ss[1]);
        const auto r2 = __builtin_amdgcn_permlane32_swap(sb, sb, false, false);
        if (fh == 0) rs[kh * S::BM + 32 * wm + fr] = __uint_as_float(r2[0]) + __uint_as_float(r2[1]);
    }
    tiled::tiled_bar();
    constexpr int RK = 8;  // accumulator registers of a block that a wave finishes
    float sc[NORM ? RK : 1];
    auto finish = [&](auto khc) {
        constexpr int KC = decltype(khc)::value;
        auto row_of = [&](int r) { return 32 * wm + 8 * ((KC * RK + r) >> 2) + 4 * fh + ((KC * RK + r) & 3); };
        if constexpr (NORM) {
#pragma unroll
            for (int r = 0; r < RK; r++) {
                sc[r] = rsqrt_hw((rs[row_of(r)] + rs[S::BM + row_of(r)]) / static_cast<float>(K) + a.eps);
            }
        }
        float sm[CB][RK];
        // Hand-over area: [wm][giving half][block of the batch][quad of the half][lane] float4.
        float *red = reinterpret_cast<float *>(lds);
        auto at = [&](int giver, int j, int u) { return red + ((((wm * 2 + giver) * S::XC + j) * 2 + u) * 64 + lane) * 4; };
#pragma unroll
        for (int j0 = 0; j0 < CB; j0 += S::XC) {
            if (j0) tiled::tiled_bar();
#pragma unroll
            for (int j = j0; j < j0 + S::XC && j < CB; j++)
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    constexpr int G = RK * (1 - KC);
                    *reinterpret_cast<f32x4t *>(at(KC, j - j0, u)) =
                        f32x4t{acc[j][G + 4 * u], acc[j][G + 4 * u + 1], acc[j][G + 4 * u + 2], acc[j][G + 4 * u + 3]};
                }
            tiled::tiled_bar();
#pragma unroll
            for (int j = j0; j < j0 + S::XC && j < CB; j++)
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const f32x4t p = *reinterpret_cast<const f32x4t *>(at(1 - KC, j - j0, u));
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float own = acc[j][KC * RK + 4 * u + e];
                        sm[j][4 * u + e] = KC == 0 ? own + p[e] : p[e] + own;
                    }
                }
        }
        const bool full = m0 + S::BM <= M && n0 + FN <= N;
        const uint32_t flags = a.flags;
        with_flag_set(flags, [&](auto set) {
            constexpr uint32_t FL = decltype(set)::value;
            constexpr int NO = GATED ? CB / 2 : CB;
            const bool accum = accumulates<FL>(flags);
#pragma unroll
            for (int o = 0; o < NO; o++) {
                const uint32_t gn = n0 + 32 * o + fr;
                float v[RK];
#pragma unroll
                for (int r = 0; r < RK; r++) {
                    const uint32_t gm = m0 + row_of(r);
                    v[r] = accum ? a.y[full || (gm < M && gn < N) ? static_cast<size_t>(gm) * a.ldy + gn : 0u] : 0.0f;
                }
#pragma unroll
                for (int r = 0; r < RK; r++) {
                    float c = GATED ? sm[2 * o][r] : sm[o][r], c2 = GATED ? sm[2 * o + 1][r] : 0.0f;
                    if constexpr (NORM) {
                        c *= sc[r];
                        c2 *= sc[r];
                    }
                    v[r] += epilogue_set<FL>(c, c2, bv[GATED ? 2 * o : o], flags);
                }
#pragma unroll
                for (int r = 0; r < RK; r++) {
                    const uint32_t gm = m0 + row_of(r);
                    if (full || (gm < M && gn < N)) a.y[static_cast<size_t>(gm) * a.ldy + gn] = v[r];
                }
            }
        });
    };
    if (kh == 0)
        finish(std::integral_constant<int, 0>{});
    else
        finish(std::integral_constant<int, 1>{});
}

typedef void (*direct_fn)(DirectArgs);

}  // namespace direct
}  // namespace mt
