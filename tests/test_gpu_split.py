"""Products on bf16 parts (csrc/split_bf16.hpp) where the parts alone are not
enough: values below 2^-100 (their third part meets bf16's smallest
subnormal), infinities and NaN (an infinity minus its own first part), and the
top of the FP32 range (the partial products overflow one by one). The kernels
must notice each and give what FP32 arithmetic gives.

Tolerance: sums of K products within K * 2^-24 of the sum of |a||b| is what
FP32 sums in any order keep; 2^-24 sqrt(K) * 8 of it is asserted (eight
standard deviations of K independent roundings).
"""
import numpy as np
import pytest

import oracle_binding as orc

pytestmark = pytest.mark.gpu


def scaled(name, m, n, k):
    a = orc.values(m * k, 0x71, 1.0).reshape(m, k)
    b = orc.values(k * n, 0x72, 1.0).reshape(k, n)
    if name == "non-finite":
        a[5, 3], a[m - 1, k - 1], a[m // 2, 1] = np.inf, -np.inf, np.nan
        b[k // 2, 7], b[0, n - 1] = -np.inf, np.nan
    elif name == "tiny":  # every product ~1e-16, every A below 2^-100
        a, b = a * np.float32(1e-36), b * np.float32(1e20)
    elif name == "tiny rows":  # subnormals among ordinary rows; tiny columns of B
        a[m // 2 : m // 2 + 3] *= np.float32(1e-39)
        b[:, 9] *= np.float32(1e-33)
    elif name == "zeros":  # zeros are exact: not tiny
        a[:, ::2] = 0
        b[::3] = 0
        a[0] = 0
    elif name == "huge":
        a, b = a * np.float32(3.4e38), b * np.float32(1e-30)
    elif name == "largest":
        a[0, 0] = np.finfo(np.float32).max
        b[0] = 0.99
    return np.ascontiguousarray(a, np.float32), np.ascontiguousarray(b, np.float32)


CASES = ["non-finite", "tiny", "tiny rows", "zeros", "huge", "largest"]


def check(got, a, b, k):
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
        size = np.abs(np.where(np.isfinite(a), a, 0)).astype(np.float64) @ np.abs(np.where(np.isfinite(b), b, 0)).astype(np.float64)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    infinite = np.isinf(want)
    np.testing.assert_array_equal(got[infinite], want[infinite].astype(np.float32))
    finite = np.isfinite(want)
    # A result in the subnormal range keeps an absolute 2^-149.
    bound = 8 * 2.0 ** -24 * np.sqrt(k) * size[finite] + k * 2.0 ** -149
    assert (np.abs(got[finite].astype(np.float64) - want[finite]) <= bound).all()


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("m,n,k", [(2048, 2048, 512), (2560, 2560, 1024)])  # one tile a workgroup; runs of one and two
def test_persistent_gemm_special_values(runtime, name, m, n, k):
    kernel = runtime.compile({"op": "gemm", "m": m, "n": n, "k": k, "tiled": True})
    assert kernel.launch["kernel"] == "gemm_f32_ring_128x128x32"
    a, b = scaled(name, m, n, k)
    bufs = [runtime.resident(a), runtime.resident(b), runtime.alloc(m * n)]
    print(f"ring {m}x{n}x{k} {name}", flush=True)
    runtime.execute([(kernel, bufs)], 1)
    got = runtime.download(bufs[2]).reshape(m, n)
    for x in bufs:
        x.free()
    check(got, a, b, k)


@pytest.mark.parametrize("name", CASES[:4])
def test_persistent_gate_up_special_values(runtime, name):
    m, n, k = 2048, 2048, 512
    a, b = scaled(name, m, n, k)
    gemm = runtime.compile({"op": "gemm", "m": m, "n": n, "k": k, "tiled": True})
    swiglu = runtime.compile({"op": "swi_glu", "len": m * n})
    x, wg, wu = (runtime.resident(t) for t in (a, b, b[:, ::-1]))
    g, u, d = (runtime.alloc(m * n) for _ in range(3))
    jobs = [(gemm, [x, wg, g]), (gemm, [x, wu, u]), (swiglu, [g, u, d])]
    assert runtime.plan(jobs) == [("gate_up_swiglu", 0)]
    print(f"dual ring {m}x{n}x{k} {name}", flush=True)
    runtime.execute(jobs, 1)
    got_g, got_u = runtime.download(g).reshape(m, n), runtime.download(u).reshape(m, n)
    for t in (x, wg, wu, g, u, d):
        t.free()
    check(got_g, a, b, k)
    check(got_u, a, np.ascontiguousarray(b[:, ::-1]), k)
