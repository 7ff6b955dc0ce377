"""The direct GEMM for fp32 x over many rows (mt_linear / mt_linear_rmsnorm): each of its tiles at the
sizes where the choice takes it, against fp64."""
import numpy as np
import pytest
import torch

import mingtts as mt
import oracle as O
from _gpu_util import say

pytestmark = pytest.mark.gpu

# M, N, K, gated, norm and the tile on 256 CUs (1: 64 x 96 features or 64 x 192 weight rows, 2: 128 x 96
# or 128 x 192, 3: 128 x 128), with ragged rows and features, one gated past its last wave; odd and even
# stage counts (8, 14, 15, 16, 31); the shortest and the longest K.
CASES = [(257, 4864, 896, True, True, 1), (330, 4800, 512, True, False, 2), (513, 4850, 896, True, True, 2),
         (1025, 4864, 896, True, True, 2), (1793, 1152, 896, False, True, 1), (1601, 3072, 1024, False, True, 2),
         (900, 4096, 1024, False, True, 3), (1100, 4099, 512, False, False, 2), (2047, 1031, 1984, False, False, 1),
         (1300, 4099, 960, False, True, 2)]


def _tile(M, N, K, gated, norm, cus):
    """linear_gemm_direct.hip's choice: the kernel's tile, 0 for the tiled kernel's linears."""
    if K % 64 or K < 512 or K >= 2048:
        return 0
    tiles = lambda bm, fn: -(-M // bm) * -(-N // fn)  # noqa: E731
    waves = lambda bm, fn: -(-tiles(bm, fn) // cus)  # noqa: E731
    if gated:
        if waves(64, 64) <= 1:
            return 0
        if 4 * tiles(128, 96) >= 3 * waves(128, 96) * cus:
            return 2
        r1 = waves(64, 96)
        return 1 if (175 if r1 == 1 else 290 + 150 * (r1 - 2)) <= 260 * waves(128, 96) else 2
    if waves(64, 128) <= 1:
        return 0
    cost = [20 + 170 * waves(64, 192), 30 + 260 * waves(128, 192), 245 * waves(128, 128)]
    return 1 + cost.index(min(cost))


@pytest.mark.parametrize("wt", [O.F16, O.BF16], ids=["wf16", "wbf16"])
@pytest.mark.parametrize("M,N,K,gated,norm,tile", CASES)
def test_direct_gemm_matches_fp64(gpu, M, N, K, gated, norm, tile, wt):
    """x in a wider matrix (ldx > K) with NaN between its rows, y in a wider one that keeps what lies
    between, bias and accumulate; normwise within the bound of x in two halves (2^-22 of x with fp16,
    2^-17 with bf16) plus fp32 sums, and twice the same bits.  The bits are those of no tile of the tiled
    kernel, which sums in another order, and mt_linear_static gives them too."""
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    assert _tile(M, N, K, gated, norm, cus) == tile or cus != 256
    say(f"direct gemm {M}x{N}x{K} gated={gated} norm={norm} w{wt}")
    dt = torch.float16 if wt == O.F16 else torch.bfloat16
    g = torch.Generator(device=gpu)
    g.manual_seed(M + N + K)
    rand = lambda *s, sc=1.0: torch.randn(*s, generator=g, device=gpu) * sc  # noqa: E731
    ldx, ldy = K + 8, N + 5
    xs = torch.full((M, ldx), float("nan"), device=gpu)
    xs[:, :K] = rand(M, K)
    w, w2 = rand(N, K, sc=0.02).to(dt), rand(N, K, sc=0.02).to(dt)
    b, gain = rand(N, sc=0.1).to(dt), (1.0 + 0.1 * rand(K)).to(dt)
    y0 = rand(M, ldy)
    flags = mt.GemvFlags.accumulate | (mt.GemvFlags.siluGate if gated else 0)

    def run(tile=0):
        y = y0.clone()
        old = mt.set_tuning(mt.TUNE_GEMM_TILE, tile)
        try:
            mt.linear(xs, w, y, flags=flags, w2=w2 if gated else None, bias=b, ldx=ldx, ldy=ldy, norm=gain if norm else None)
        finally:
            mt.set_tuning(mt.TUNE_GEMM_TILE, old)
        torch.cuda.synchronize()
        return y

    runs = [run(), run()]
    assert torch.equal(runs[0], runs[1])
    assert torch.equal(runs[0][:, N:], y0[:, N:])
    for tiled in (1, 2) if gated else (1, 2, 3):
        assert not torch.equal(runs[0], run(tiled)), tiled
    if not norm:
        y = y0.clone()
        rc = mt.linear_static_raw(xs, mt.F32, w, w2 if gated else None, mt.F16 if wt == O.F16 else mt.BF16, b, y, M, N, K, ldx,
                                  ldy, flags)
        assert rc == mt.OK, mt.last_error()
        torch.cuda.synchronize()
        assert torch.equal(runs[0], y)
    x = xs[:, :K].double()
    if norm:
        x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * gain.double()
    v = x @ w.double().t().contiguous() + b.double()
    if gated:
        v = v / (1.0 + torch.exp(-v)) * (x @ w2.double().t().contiguous())
    want = y0[:, :N].double() + v
    got = runs[0][:, :N].double()
    # halves: 2^-22 / 2^-17 of each product; sums: K / 16 roundings of 2^-24 each way
    bound = (2.0 ** -22 if wt == O.F16 else 2.0 ** -17) + 2.0 ** -24 * (K / 16) ** 0.5
    assert ((got - want).norm() / want.norm()).item() <= 2 * bound
    scale = v.pow(2).mean().sqrt()
    assert ((got - want).abs().max() / scale).item() <= 40 * bound


def test_long_k_needs_no_workspace(gpu):
    """fp32 x with long K over rows whose tiles nearly fill the chip (down at 1600 rows) runs without a
    workspace: captured on a stream that has none, eagerly on that stream, on one that owns a workspace
    and through mt_linear_static it gives the same bits, and it allocates nothing."""
    M, N, K = 1600, 896, 4864
    say("gemm: long K without a workspace")
    g = torch.Generator(device=gpu)
    g.manual_seed(9)
    x = torch.randn(M, K, generator=g, device=gpu)
    w = (torch.randn(N, K, generator=g, device=gpu) * 0.02).half()
    want = x.double() @ w.double().t().contiguous()
    y = [torch.zeros(M, N, device=gpu) for _ in range(4)]
    s = torch.cuda.Stream()
    mt.linear(x[:512], w, y[0][:512])  # parts of K: the current stream owns a workspace from here on
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        mt.linear(x, w, y[1], stream=s)
    assert mt.linear_static_raw(x, mt.F32, w, None, mt.F16, None, y[3], M, N, K, K, N, 0) == mt.OK, mt.last_error()
    torch.cuda.synchronize()  # the static scratch is there once its code is loaded
    free = torch.cuda.mem_get_info(gpu)[0]
    mt.linear(x, w, y[2], stream=s)
    mt.linear(x, w, y[0])
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info(gpu)[0] == free
    assert ((y[0].double() - want).norm() / want.norm()).item() <= 2e-6
    for _ in range(3):
        y[1].zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for i in (1, 2, 3):
            assert torch.equal(y[0], y[i]), i
