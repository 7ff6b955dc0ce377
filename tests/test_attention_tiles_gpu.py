"""mt_attention over many rows of one sequence (32-row blocks on the matrix cores) against the
fp64 oracle and against the row kernels."""
import numpy as np
import pytest
import torch

import mingtts as mt
import oracle as O
from _gpu_util import say

pytestmark = pytest.mark.gpu


def _inputs(device, ct, M, hq, hkv, cap, seed, scale=1.5):
    rng = np.random.default_rng(seed)
    q = (rng.standard_normal((M, hq * 64)) * scale).astype(np.float32)
    kc = torch.from_numpy(rng.standard_normal((hkv, cap, 64)).astype(np.float32)).to(device).to(ct)
    vc = torch.from_numpy(rng.standard_normal((hkv, cap, 64)).astype(np.float32)).to(device).to(ct)
    return q, kc, vc


def _tiles(M, pos0, window):
    """Whether mt_attention takes the matrix cores: more than 64 rows, unless every row's keys start at
    position 0 and end by 1024 (those keep the bits of one call per row)."""
    return M > 64 and not (pos0 + M <= 1024 and (window == 0 or pos0 + M <= window))


@pytest.mark.parametrize("ct,M,pos0,window", [
    (torch.float16, 320, 0, 0),
    (torch.float16, 1024, 0, 0),     # the last key within the contract
    (torch.float16, 500, 524, 0),
    (torch.float16, 400, 0, 400),    # a window as long as the last row's span
    (torch.float32, 65, 192, 0),
    (torch.float32, 512, 0, 0),
    (torch.float32, 700, 324, 0),
])
def test_rows_within_1024_keys_have_the_bits_of_one_call_each(gpu, ct, M, pos0, window):
    """mt_attention's contract for M >= 8 rows whose keys start at position 0 and end by 1024, at row
    counts and spans where the matrix cores would take the rows otherwise."""
    assert not _tiles(M, pos0, window)
    q, kc, vc = _inputs(gpu, ct, M, 2, 1, 1024, M + pos0)
    qd = torch.from_numpy(q).to(gpu)
    o1, o2 = torch.full((M, 128), 7.0, device=gpu), torch.full((M, 128), 7.0, device=gpu)
    say(f"rows within 1024 keys ct={ct} M={M} pos0={pos0} window={window}")
    mt.attention(qd, 128, M, 2, 1, pos0, window, kc, vc, 1024, o1, 128, 0.125)
    for m in range(M):
        mt.attention(qd[m:], 128, 1, 2, 1, pos0 + m, window, kc, vc, 1024, o2[m:], 128, 0.125)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(o1.cpu().numpy(), o2.cpu().numpy())


@pytest.mark.parametrize("ct,M,pos0,window,cap,hq,hkv", [
    (torch.float16, 65, 960, 0, 1025, 14, 2),     # the fewest rows, one key past the row kernels' 1024
    (torch.float16, 333, 800, 0, 1136, 14, 2),    # a ragged last block, tiles cut by the block's end
    (torch.float16, 65, 31, 65, 96, 14, 2),       # the fewest rows with a window; the cache's last slot
    (torch.float16, 97, 200, 1, 400, 3, 3),       # a window of the row itself
    (torch.float16, 81, 0, 80, 81, 14, 2),        # a window that cuts the last row alone
    (torch.float32, 65, 960, 0, 1025, 14, 2),
    (torch.float32, 130, 100, 65, 512, 4, 1),
    (torch.float32, 70, 4026, 0, 4096, 2, 2),     # the longest cache
])
def test_tiles_match_fp64(gpu, ct, M, pos0, window, cap, hq, hkv):
    """Sampled rows against fp64 on the stored cache values (the reference's tolerance, atol 2e-5 and
    rtol 1e-4); cache rows no row attends hold NaN; a second run gives the same bits; out = q works."""
    assert _tiles(M, pos0, window)
    q, kc, vc = _inputs(gpu, ct, M, hq, hkv, cap, M * 5 + pos0 + window)
    kg, vg = kc.double().cpu().numpy(), vc.double().cpu().numpy()
    kc[:, pos0 + M:] = float("nan")
    vc[:, pos0 + M:] = float("nan")
    first = max(0, pos0 + 1 - window) if window else 0
    kc[:, :first] = float("nan")
    vc[:, :first] = float("nan")
    qd = torch.from_numpy(q).to(gpu)
    o = [torch.full((M, hq * 64), 7.0, device=gpu) for _ in range(2)]
    say(f"attention tiles ct={ct} M={M} pos0={pos0} window={window} cap={cap} heads {hq}/{hkv}")
    for out in o:
        mt.attention(qd, hq * 64, M, hq, hkv, pos0, window, kc, vc, cap, out, hq * 64, 0.125)
    mt.attention(qd, hq * 64, M, hq, hkv, pos0, window, kc, vc, cap, qd, hq * 64, 0.125)
    torch.cuda.synchronize()
    got = o[0].cpu().numpy()
    np.testing.assert_array_equal(got, o[1].cpu().numpy())
    np.testing.assert_array_equal(got, qd.cpu().numpy())
    for m in sorted({0, 1, 31, 32, M // 2, M - 2, M - 1}):
        want = O.attention_f64(q[m].reshape(hq, 64), kg, vg, pos0 + m, window, 0.125)
        ex, i, g, w = O.worst_violation(got[m].reshape(hq, 64), want, 2e-5)
        assert ex <= 0, f"row {m} index {i} got {g} want {w}"


@pytest.mark.parametrize("ct", [torch.float16, torch.float32])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_values_that_are_not_finite_reach_only_the_rows_that_attend_them(gpu, ct, bad):
    """A cached key or value, or a query, that is not finite: every row gets what the same row gets
    from a call of its own (NaN in the same places), so rows before it stay finite."""
    M, pos0, cap, at = 330, 800, 1152, 150
    assert _tiles(M, pos0, 0)
    for where in ("k", "v", "q"):
        q, kc, vc = _inputs(gpu, ct, M, 2, 1, cap, 11)
        qd = torch.from_numpy(q).to(gpu)
        (dict(k=kc, v=vc)[where][0, pos0 + at] if where != "q" else qd[at])[5] = bad
        o1 = torch.full((M, 128), 7.0, device=gpu)
        o2 = torch.full((M, 128), 7.0, device=gpu)
        say(f"attention tiles ct={ct} {bad} in {where}")
        mt.attention(qd, 128, M, 2, 1, pos0, 0, kc, vc, cap, o1, 128, 0.125)
        for m in range(128, 192):
            mt.attention(qd[m:], 128, 1, 2, 1, pos0 + m, 0, kc, vc, cap, o2[m:], 128, 0.125)
        torch.cuda.synchronize()
        a, b = o1.cpu().numpy()[128:192], o2.cpu().numpy()[128:192]
        assert np.isfinite(a[:at - 128]).all()
        np.testing.assert_allclose(a, b, rtol=1e-4, atol=2e-5)


@pytest.mark.parametrize("ct", [torch.float16, torch.float32])
def test_rows_beside_one_that_is_not_finite_keep_their_bits(gpu, ct):
    """Queries with a NaN and an infinity in rows of their own: every other row of their blocks has the
    bits of a call without them, also where out is q."""
    M, pos0, cap = 330, 800, 1152
    assert _tiles(M, pos0, 0)
    q, kc, vc = _inputs(gpu, ct, M, 2, 1, cap, 12)
    qd = torch.from_numpy(q).to(gpu)
    want = torch.full((M, 128), 7.0, device=gpu)
    say(f"attention tiles ct={ct} rows beside NaN")
    mt.attention(qd, 128, M, 2, 1, pos0, 0, kc, vc, cap, want, 128, 0.125)
    qd[150, 5], qd[159, 70], qd[329, 0] = float("nan"), float("inf"), float("nan")
    out = torch.full((M, 128), 7.0, device=gpu)
    mt.attention(qd, 128, M, 2, 1, pos0, 0, kc, vc, cap, out, 128, 0.125)
    mt.attention(qd, 128, M, 2, 1, pos0, 0, kc, vc, cap, qd, 128, 0.125)
    torch.cuda.synchronize()
    bad = np.zeros((M, 2), bool)  # (row, head)
    bad[150, 0] = bad[159, 1] = bad[329, 0] = True
    for got in (out, qd):
        a, b = got.cpu().numpy().reshape(M, 2, 64), want.cpu().numpy().reshape(M, 2, 64)
        np.testing.assert_array_equal(a[~bad], b[~bad])
        assert np.isnan(a[bad]).all()


@pytest.mark.parametrize("M,pos0,window", [(700, 1024, 0), (400, 0, 65)])
@pytest.mark.parametrize("ct", [torch.float16, torch.float32])
def test_values_with_a_mean_are_as_exact_as_by_the_row_kernel(gpu, ct, M, pos0, window):
    """Values of one sign: sums that round towards zero above the fraction and to nearest below it would
    show.  The error against fp64 stays within that of the same rows in calls of their own (a tenth more
    for the sample's size: 0.8 to 1.0 of it measured)."""
    assert _tiles(M, pos0, window)
    cap = pos0 + M
    q, kc, vc = _inputs(gpu, ct, M, 2, 1, cap, 13, 3.0)
    vc += 5.0
    qd = torch.from_numpy(q).to(gpu)
    o1, o2 = torch.full((M, 128), 7.0, device=gpu), torch.full((M, 128), 7.0, device=gpu)
    say(f"attention tiles ct={ct} values with a mean M={M} pos0={pos0} window={window}")
    mt.attention(qd, 128, M, 2, 1, pos0, window, kc, vc, cap, o1, 128, 0.125)
    for m in range(M):
        mt.attention(qd[m:], 128, 1, 2, 1, pos0 + m, window, kc, vc, cap, o2[m:], 128, 0.125)
    torch.cuda.synchronize()
    kg, vg = kc.double().cpu().numpy(), vc.double().cpu().numpy()
    want = np.stack([O.attention_f64(q[m].reshape(2, 64), kg, vg, pos0 + m, window, 0.125).reshape(128) for m in range(M)])
    e1, e2 = (np.linalg.norm(o.double().cpu().numpy() - want) for o in (o1, o2))
    assert e1 <= 1.1 * e2, f"{e1 / e2:.2f}"


def test_large_and_small_queries(gpu):
    """The halves of q are scaled by the row's own power of two: queries of 1e-6 and of 1e5 (past
    fp16's range), with a score scale that keeps the scores ordinary, and a negative scale.  q rows
    stand in rows of q | k | v, as the engine's do."""
    M, pos0, cap, ld = 320, 760, 1080, 256
    assert _tiles(M, pos0, 0)
    for size, scale in ((1e-6, 1.2e5), (1e5, 1.2e-6), (1.0, -0.125)):
        q, kc, vc = _inputs(gpu, torch.float16, M, 2, 1, cap, 3, size)
        out = torch.full((M, 128), 7.0, device=gpu)
        qkv = torch.full((M, ld), float("nan"), device=gpu)
        qkv[:, :128] = torch.from_numpy(q).to(gpu)
        say(f"attention tiles q {size} scale {scale}")
        mt.attention(qkv, ld, M, 2, 1, pos0, 0, kc, vc, cap, out, 128, scale)
        torch.cuda.synchronize()
        for m in (0, 100, M - 1):
            want = O.attention_f64(q[m].reshape(2, 64), kc.double().cpu().numpy(), vc.double().cpu().numpy(), pos0 + m, 0,
                                   scale)
            ex, i, g, w = O.worst_violation(out[m].cpu().numpy().reshape(2, 64), want, 2e-5)
            assert ex <= 0, f"row {m} index {i} got {g} want {w}"


@pytest.mark.parametrize("ct,cap", [(torch.float32, 1600), (torch.float16, 2100), (torch.float16, 40)])
def test_decode_rounds_match_fp64(gpu, ct, cap):
    """mt_attention_decode at the edges of its rounds (512 keys of an fp32 cache, 1024 of an fp16 one) and
    of its octets, NaN in the cache rows past each length, a maximum that moves in the last round, and
    more query heads than a wave has octets."""
    lens = np.array([n for n in (1, 7, 9, 128, 129, 511, 512, 513, 1023, 1024, 1025, cap) if n <= cap], np.uint32)
    B, hq, hkv = len(lens), 14, 2
    rng = np.random.default_rng(cap)
    q = (rng.standard_normal((B, hq * 64)) * 1.5).astype(np.float32)
    kc = torch.from_numpy(rng.standard_normal((B, hkv, cap, 64)).astype(np.float32)).to(gpu).to(ct)
    vc = torch.from_numpy(rng.standard_normal((B, hkv, cap, 64)).astype(np.float32)).to(gpu).to(ct)
    for b, n in enumerate(lens):
        kc[b, 0, int(n) - 1] *= 4.0
        kc[b, :, int(n):] = float("nan")
        vc[b, :, int(n):] = float("nan")
    out = torch.full((B, hq * 64), 7.0, device=gpu)
    say(f"decode rounds ct={ct} cap={cap} lens={lens.tolist()}")
    mt.attention_decode(torch.from_numpy(q).to(gpu), hq * 64, B, hq, hkv, torch.from_numpy(lens.astype(np.int32)).to(gpu), 0,
                        kc, vc, cap, hkv * cap * 64, out, hq * 64, 0.125)
    torch.cuda.synchronize()
    got = out.cpu().numpy().reshape(B, hq, 64)
    for b, n in enumerate(lens):
        want = O.attention_f64(q[b].reshape(hq, 64), kc[b].double().cpu().numpy(), vc[b].double().cpu().numpy(), int(n) - 1, 0,
                               0.125)
        ex, i, g, w = O.worst_violation(got[b], want, 2e-5)
        assert ex <= 0, f"len {n} index {i} got {g} want {w}"
