"""The GEMM for at most 16 rows and short K (csrc/gemm_rows16.hip): edges of
its slices, columns and waves, any alignment, values past the ends of A and B,
and the residual Add in its epilogue, against the FP64 oracle."""
import numpy as np
import pytest

import oracle_binding as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,waves", [
    (1, 1, 1, 4), (8, 256, 128, 4), (8, 128, 256, 4), (16, 33, 31, 4), (7, 100, 257, 8), (16, 512, 512, 8),
    (3, 31, 32, 4), (16, 2016, 65, 4), (5, 1999, 511, 8), (15, 64, 129, 4), (2, 30, 33, 4)])
def test_rows16_shapes(runtime, m, n, k, waves):
    launch = runtime.compile({"op": "gemm", "m": m, "n": n, "k": k, "tiled": True}).launch
    assert launch["kernel"] == f"gemm_f32_rows16_w{waves}" and launch["grid"][0] == (n + 31) // 32, launch
    a, b, x = orc.values(m * k, 0x61, 1.0), orc.values(k * n, 0x62, 1.0), orc.values(m * n, 0x63, 1.0)
    # Values that loads past a row or past the ends could bring into other outputs: the starts of the second rows of A
    # (read past the end of the first row's last slice) and of B (past its first row's last column), and B's last value.
    for special in (False, True):
        if special and (m < 2 or n < 2 or k < 2):
            continue
        a2, b2 = a.copy(), b.copy()
        if special:
            a2[k] = np.inf        # A[1][0]
            b2[n] = np.nan        # B[1][0]
            b2[-1] = np.inf       # B[k-1][n-1]
        bufs = [runtime.resident(t) for t in (a2, b2, x)] + [runtime.alloc(m * n), runtime.alloc(m * n)]
        gemm = runtime.compile({"op": "gemm", "m": m, "n": n, "k": k, "tiled": True})
        add = runtime.compile({"op": "add", "len": m * n})
        jobs = [(gemm, [bufs[0], bufs[1], bufs[3]]), (add, [bufs[3], bufs[2], bufs[4]])]
        assert runtime.plan(jobs) == [("gemm_residual", 0)]
        print(f"rows16 {m}x{n}x{k} special {special}", flush=True)
        runtime.execute(jobs, 2)
        got, total = runtime.download(bufs[3]).reshape(m, n), runtime.download(bufs[4]).reshape(m, n)
        for t in bufs:
            t.free()
        want = np.asarray(orc.gemm_reference(m, n, k, a, b)).reshape(m, n)
        keep = np.ones((m, n), bool)
        if special:
            keep[1], keep[:, 0], keep[:, -1] = False, False, False
        # K products of values in [-1, 1): each rounding is at most 2^-24 of a partial sum of at most K, and the sums of
        # uniform values stay near sqrt(K / 9), so 2^-23 (K + 8) is far above what FP32 leaves.
        assert np.abs(got[keep] - want[keep]).max(initial=0) <= 2.0 ** -23 * (k + 8)
        if special:
            assert np.isnan(got[:, 0]).all() and not np.isfinite(got[1]).any() and not np.isfinite(got[:, -1]).any()
        np.testing.assert_array_equal(total[keep], got[keep] + x.reshape(m, n)[keep])


@pytest.mark.parametrize("m,n,k", [(8, 256, 128), (16, 33, 31), (3, 31, 48), (7, 100, 257)])
def test_rows16_pairs(runtime, m, n, k):
    # Two products of one shape run as one launch, each output bit for bit its own launch's.
    gemm = runtime.compile({"op": "gemm", "m": m, "n": n, "k": k, "tiled": True})
    assert gemm.launch["kernel"].startswith("gemm_f32_rows16"), gemm.launch
    x, wg, wu = (runtime.resident(orc.values(c, s, 1.0)) for c, s in ((m * k, 0x64), (k * n, 0x65), (k * n, 0x66)))
    c = [runtime.alloc(m * n) for _ in range(2)]
    jobs = [(gemm, [x, wg, c[0]]), (gemm, [x, wu, c[1]])]
    assert runtime.plan(jobs) == [("pair", 0)]
    print(f"rows16 pair {m}x{n}x{k}", flush=True)
    runtime.execute(jobs, 2)
    both = [runtime.download(t) for t in c]
    for job in jobs:
        runtime.execute([job], 1)
    alone = [runtime.download(t) for t in c]
    for t in (x, wg, wu, *c):
        t.free()
    for got, want in zip(both, alone):
        np.testing.assert_array_equal(got, want)
