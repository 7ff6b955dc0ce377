// Instances, tile choice and launcher of the direct GEMM for fp32 x (direct_kernel.hpp).
//
// Reference kernel replaced: gemm_kernel<32,64,32,4> (Shaders.swift:297-410).
#include <algorithm>

#include "direct_kernel.hpp"

namespace mt {

namespace {

using direct::direct_fn;
using direct::DirectArgs;

// Tiles of 32 wm x rows by 32 cb weight rows.
struct Tile {
    uint32_t wm, cb;
};
constexpr Tile TILES[] = {{0, 0}, {2, 6}, {4, 6}, {4, 4}};

template <int WT, bool GATED, bool NORM>
direct_fn pick(int tile) {
    using direct::direct_kernel;
    if (tile == 1) return direct_kernel<WT, 2, 6, GATED, NORM>;
    if (GATED || tile == 2) return direct_kernel<WT, 4, 6, GATED, NORM>;
    return direct_kernel<WT, 4, 4, false, NORM>;
}
template <int WT>
direct_fn pick_wt(bool gated, bool norm, int tile) {
    if (gated) return norm ? pick<WT, true, true>(tile) : pick<WT, true, false>(tile);
    return norm ? pick<WT, false, true>(tile) : pick<WT, false, false>(tile);
}

}  // namespace

// What the kernel takes: whole 64-k stages, the gain in LDS, and 31-bit offsets into x and the
// weights (the upper half of an offset marks a request that reads nothing).
bool direct_takes(const LinearArgs &a) {
    const uint64_t xb = (static_cast<uint64_t>(a.M - 1) * a.ldx + a.K) * 4, wb = static_cast<uint64_t>(a.N) * a.K * 2;
    return a.K % direct::SK == 0 && (!a.norm || a.K <= direct::NORM_K) && xb < 0x7FFFFFFFu && wb < 0x7FFFFFFFu;
}

// The tile for an fp32-x linear, or 0 for the kernels of tiled_plan.  Measured on 256 CUs (graph
// replay over six sets of operands, K = 896 and 1024, fp16 weights), in us by the number r of waves of
// workgroups:
//   gated      64 x 96 features 17 (r = 1), 29 (2), then 15 a wave; 128 x 96 26, 48, 80, 108;
//              tiled_kernel's 64 x 64 features 13.5, 24, 30 and 12 a wave.
//   not gated  64 x 192 17-20, 30-37, 49-55; 128 x 192 25-33, 53; 128 x 128 20-24, 44-55;
//              tiled_kernel's 64 x 128 15.5-18, 25-28, 44, 56.
// So a gated linear goes here once tiled_kernel's tiles no longer fit the CUs at once (gate|up above
// 192 rows), on the 128-row tiles where ring_fills (linear_gemm_lds.hip) says that they fill the
// chip; others once tiled_kernel's 64 x 128 tiles no longer do, and the tile with the least estimate
// takes it.  64 x 128 tiles of this kernel were ahead of tiled_kernel's in a graph of their own (qkv at
// 1600 rows 15.7 against 16.5 us) but not where x comes from the kernel before (19.7 against 17.4), and
// with long K they were behind (down at 2048 rows 70 against 63 us): tiled_kernel keeps x further ahead.
int direct_tile(const LinearArgs &a, int cus, bool ring_fills) {
    if (!direct_takes(a) || a.K < 512 || a.K >= 2048) return 0;
    const bool gated = (a.flags & F_SILU_GATE) != 0;
    const uint32_t ncu = static_cast<uint32_t>(cus);
    const auto waves = [&](uint32_t bm, uint32_t fn) {
        return (((a.M + bm - 1) / bm) * ((a.N + fn - 1) / fn) + ncu - 1) / ncu;
    };
    if (gated) {
        if (waves(64, 64) <= 1) return 0;
        if (ring_fills) return 2;
        const uint32_t r1 = waves(64, 96), r2 = waves(128, 96);
        return (r1 == 1 ? 175 : 290 + 150 * (r1 - 2)) <= 260 * r2 ? 1 : 2;  // tenths of a us
    }
    if (waves(64, 128) <= 1) return 0;
    const uint32_t c1 = 20 + 170 * waves(64, 192), c2 = 30 + 260 * waves(128, 192), c3 = 245 * waves(128, 128);
    return c1 <= c2 && c1 <= c3 ? 1 : c2 <= c3 ? 2 : 3;
}

int launch_gemm_direct(const LinearArgs &a, int wt, int tile, hipStream_t stream) {
    const bool gated = (a.flags & F_SILU_GATE) != 0;
    const uint32_t bm = 32 * TILES[tile].wm, fn = (gated ? 16 : 32) * TILES[tile].cb;
    DirectArgs t;
    t.x = static_cast<const float *>(a.x);
    t.w = a.w;
    t.w2 = a.w2;
    t.bias = a.bias;
    t.norm = a.norm;
    t.y = a.y;
    t.M = a.M; t.N = a.N; t.K = a.K; t.ldx = a.ldx; t.ldy = a.ldy; t.flags = a.flags;
    t.eps = a.eps;
    t.tiles_m = (a.M + bm - 1) / bm;
    t.tiles_n = (a.N + fn - 1) / fn;
    t.x_bytes = static_cast<uint32_t>((static_cast<uint64_t>(a.M - 1) * a.ldx + a.K) * 4);
    t.w_bytes = a.N * a.K * 2;
    const uint64_t G = static_cast<uint64_t>(t.tiles_m) * t.tiles_n;
    if (G == 0 || G > 0x7FFFFFFFu) return set_error(MT_EINVAL, "gemm: %llu direct tiles", static_cast<unsigned long long>(G));
    direct_fn kernel = wt == DT_BF16 ? pick_wt<DT_BF16>(gated, a.norm != nullptr, tile) : pick_wt<DT_F16>(gated, a.norm != nullptr, tile);
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(G)), dim3(128 * TILES[tile].wm), 0, stream, t);
    return check_launch("gemm (direct)");
}

}  // namespace mt
