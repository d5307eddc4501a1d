"""Products on bf16 parts (csrc/split_bf16.hpp) where the parts alone are not
enough: values whose own parts would meet bf16's smallest subnormal (which
the scale ahead of the split lifts above it), infinities and NaN (an infinity minus its own first part), and the
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


def product(runtime, m, n, k, a, b):
    kernel = runtime.compile({"op": "gemm", "m": m, "n": n, "k": k, "tiled": True})
    assert kernel.launch["kernel"] == "gemm_f32_ring_128x128x32"
    bufs = [runtime.resident(a), runtime.resident(b), runtime.alloc(m * n)]
    print(f"ring {m}x{n}x{k}", flush=True)
    runtime.execute([(kernel, bufs)], 1)
    got = runtime.download(bufs[2]).reshape(m, n)
    for x in bufs:
        x.free()
    return got


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


@pytest.mark.parametrize("side", ["a", "b"])
@pytest.mark.parametrize("m,n,k", [(2048, 2048, 512), (2560, 2560, 1024)])
def test_persistent_gemm_keeps_subnormals(runtime, side, m, n, k):
    # Every nonzero of one operand lies below 2^-134, where bf16 holds nothing.
    tiny = (orc.values(m * k if side == "a" else k * n, 0x73, 1.0).astype(np.float64) * 2.0 ** -134).astype(np.float32)
    other = orc.values(k * n if side == "a" else m * k, 0x74, 1.0) * np.float32(1e30)
    a, b = (tiny, other) if side == "a" else (other, tiny)
    got = product(runtime, m, n, k, a, b)
    assert np.abs(got).max() > 1e-11
    check(got, a.reshape(m, k), b.reshape(k, n), k)


def test_persistent_gemm_small_products(runtime):
    # Products near the smallest normals: products of their parts lie below them.
    m, n, k = 2048, 2048, 512
    a, b = orc.values(m * k, 0x75, 1.0) * np.float32(2.0 ** -55), orc.values(k * n, 0x76, 1.0) * np.float32(2.0 ** -55)
    check(product(runtime, m, n, k, a, b), a.reshape(m, k), b.reshape(k, n), k)


@pytest.mark.parametrize("special", [1e-35, 1e-41, np.inf, 3e38])
def test_persistent_gemm_special_value_stays_in_its_row_and_column(runtime, special):
    # How an output is computed depends on its own row and column alone, so one
    # tiny, infinite or huge operand leaves all other outputs' bits (and so
    # the work done for them) as they were.
    m, n, k = 2560, 2560, 512  # two tiles in some workgroups
    a, b = orc.values(m * k, 0x77, 1.0).reshape(m, k), orc.values(k * n, 0x78, 1.0).reshape(k, n)
    plain = product(runtime, m, n, k, a, b)
    a[5, 3] = b[k // 2, 700] = special
    got = product(runtime, m, n, k, a, b)
    plain[5], plain[:, 700] = got[5], got[:, 700]
    np.testing.assert_array_equal(got, plain)
    check(got, a, b, k)


@pytest.mark.parametrize("special", [1e-35, 1e-41, np.inf, np.nan, 3e38])
@pytest.mark.parametrize("where", ["x", "gate", "up"])
def test_persistent_gate_up_bits_with_a_special_value(runtime, special, where):
    # A special value in one operand: the fused launch's bits stay those of
    # each product launched alone.
    m, n, k = 2048, 2048, 512  # two tiles of 128x64 a workgroup fused, one of 128x128 alone
    data = {"x": orc.values(m * k, 0x79, 1.0), "gate": orc.values(k * n, 0x7A, 1.0), "up": orc.values(k * n, 0x7B, 1.0)}
    data[where][(m * k if where == "x" else k * n) // 2 + 77] = special
    gemm = runtime.compile({"op": "gemm", "m": m, "n": n, "k": k, "tiled": True})
    assert gemm.launch["kernel"] == "gemm_f32_ring_128x128x32"
    swiglu = runtime.compile({"op": "swi_glu", "len": m * n})
    x, wg, wu = (runtime.resident(t) for t in data.values())
    g, u, d = (runtime.alloc(m * n) for _ in range(3))
    jobs = [(gemm, [x, wg, g]), (gemm, [x, wu, u]), (swiglu, [g, u, d])]
    assert runtime.plan(jobs) == [("gate_up_swiglu", 0)]
    print(f"dual ring {special} in {where}", flush=True)
    runtime.execute(jobs, 1)
    fused = [runtime.download(t) for t in (g, u, d)]
    for job in jobs:
        runtime.execute([job], 1)
    alone = [runtime.download(t) for t in (g, u, d)]
    for t in (x, wg, wu, g, u, d):
        t.free()
    for f, w, name in zip(fused, alone, ("gate", "up", "act")):
        np.testing.assert_array_equal(f, w, err_msg=name)


def attend(runtime, heads, seq, dim, causal, q, k, v):
    kernel = runtime.compile({"op": "attention_online", "heads": heads, "seq": seq, "dim": dim, "causal": causal})
    print(f"attention H{heads} S{seq} D{dim} causal {causal}: {kernel.launch}", flush=True)
    bufs = [runtime.resident(x) for x in (q, k, v)] + [runtime.alloc(heads * seq * dim)]
    assert kernel.launch["kernel"].startswith("attention_flash"), kernel.launch
    runtime.execute([(kernel, bufs)], 2)
    got = runtime.download(bufs[3])
    for x in bufs:
        x.free()
    return got, kernel.launch


@pytest.mark.parametrize("heads,seq,dim,causal,threads", [
    (24, 1531, 80, False, 512),  # eight waves: one round of 144 blocks against two of 288
    (33, 1020, 128, False, 512), (33, 1020, 128, True, 256),  # heads not a multiple of the XCDs
    (256, 300, 72, True, 512), (171, 513, 128, True, 512),  # eight waves, causal
    (32, 1024, 100, True, 256), (32, 1000, 96, True, 256),  # four waves, one per SIMD
    (40, 900, 64, True, 256), (9, 3700, 20, False, 256),  # head dims to 64 and 32
    (304, 1, 64, False, 256), (304, 33, 96, True, 256), (304, 31, 128, False, 256), (272, 32, 4, True, 256),
    (272, 129, 36, False, 256),  # one key; the edges of a tile; one block and a row more
])
def test_flash_on_parts_shapes(runtime, heads, seq, dim, causal, threads):
    n = heads * seq * dim
    q, k, v = orc.normal(n, 0x81), orc.normal(n, 0x82), orc.normal(n, 0x83)
    got, launch = attend(runtime, heads, seq, dim, causal, q, k, v)
    assert launch["block"][0] == threads and launch["kernel"] == f"attention_flash_d{(dim + 31) // 32 * 32}", launch
    want = orc.attention_reference(heads, seq, dim, causal, q, k, v)
    # FP32 rounding of scores of a few units and of sums of weights: 1e-5 of the unit-sized values.
    assert orc.compare(got, want, 1e-5, 1e-5).status == 0


FLASH = [(32, 1000, 96, True), (24, 1531, 80, False), (40, 900, 64, True)]  # four waves, eight, two a SIMD


@pytest.mark.parametrize("heads,seq,dim,causal", FLASH)
def test_flash_on_parts_scaled_operands(runtime, heads, seq, dim, causal):
    # Operands at the ends of the FP32 range whose scores are ordinary, and
    # values of V near the smallest normals: as FP32 arithmetic has them.
    n = heads * seq * dim
    q, k, v = orc.normal(n, 0x91), orc.normal(n, 0x92), orc.normal(n, 0x93)
    for sq, sk, sv in ((1e30, 1e-30, 1.0), (1e-30, 1e30, 1.0), (1.0, 1.0, 1e-36)):
        a, b, c = (np.asarray(x * np.float32(s), np.float32) for x, s in ((q, sq), (k, sk), (v, sv)))
        got, _ = attend(runtime, heads, seq, dim, causal, a, b, c)
        want = orc.attention_reference(heads, seq, dim, causal, a, b, c)
        assert orc.compare(got / np.float32(sv), np.asarray(want) / sv, 2e-5, 2e-5).status == 0, (sq, sk, sv)


@pytest.mark.parametrize("heads,seq,dim,causal", FLASH)
def test_flash_on_parts_non_finite(runtime, heads, seq, dim, causal):
    n = heads * seq * dim
    q, k, v = (orc.normal(n, s).reshape(heads, seq, dim).copy() for s in (0xA1, 0xA2, 0xA3))
    key = seq // 2
    q[1, :, 0] = np.abs(q[1, :, 0]) + 0.5
    k[1, key] = 0
    k[1, key, 0] = -np.inf  # scores of -inf: the key has no weight
    v[2, key, 3] = np.inf
    q[3, key, 1] = np.nan
    got, _ = attend(runtime, heads, seq, dim, causal, q.ravel(), k.ravel(), v.ravel())
    got = got.reshape(heads, seq, dim)
    want = np.asarray(orc.attention_reference(heads, seq, dim, causal, *(np.where(np.isfinite(x), x, 0).ravel()
                                                                       for x in (q, k, v)))).reshape(heads, seq, dim)
    clean = [h for h in range(heads) if h not in (1, 2, 3)]
    assert orc.compare(got[clean].ravel(), want[clean].ravel(), 1e-5, 1e-5).status == 0
    # Head 1: finite everywhere, and what the other keys give.
    rows = [0, key - 1, key, seq - 1]
    for r in rows:
        keys = np.arange(r + 1 if causal else seq)
        keys = keys[keys != key] if len(keys) > 1 else keys
        s = q[1, r].astype(np.float64) @ k[1, keys].astype(np.float64).T / np.sqrt(dim)
        w = np.exp(s - s.max())
        np.testing.assert_allclose(got[1, r], (w / w.sum()) @ v[1, keys].astype(np.float64), rtol=2e-5, atol=2e-5)
    assert np.isfinite(got[1]).all()
    # Head 2: column 3 of every query that weighs the key, the other columns as they were.
    first = key if causal else 0
    assert not np.isfinite(got[2, first:, 3]).any()
    other = [d for d in range(dim) if d != 3]
    assert orc.compare(got[2][:, other].ravel(), want[2][:, other].ravel(), 1e-5, 1e-5).status == 0
    # Head 3: the one query.
    assert np.isnan(got[3, key]).all()
    rest = [r for r in range(seq) if r != key]
    assert orc.compare(got[3, rest].ravel(), want[3, rest].ravel(), 1e-5, 1e-5).status == 0


@pytest.mark.parametrize("heads,seq,dim,causal", FLASH)
def test_flash_on_parts_subnormal_values(runtime, heads, seq, dim, causal):
    # Every V below 2^-134, where bf16 holds nothing; outputs keep FP32's
    # absolute 2^-149 (and the sum of the weights its rounding).
    n = heads * seq * dim
    q, k = orc.normal(n, 0xB1), orc.normal(n, 0xB2)
    v = (orc.values(n, 0xB3, 1.0).astype(np.float64) * 2.0 ** -134).astype(np.float32)
    got, _ = attend(runtime, heads, seq, dim, causal, q, k, v)
    want = np.asarray(orc.attention_reference(heads, seq, dim, causal, q, k, v * np.float32(2.0 ** 64)), np.float64)
    assert np.abs(got.astype(np.float64) * 2.0 ** 64 - want).max() <= 4 * 2.0 ** -85


@pytest.mark.parametrize("heads,seq,dim,causal", FLASH)
@pytest.mark.parametrize("special", [1e-35, 1e-41])
def test_flash_on_parts_tiny_value_costs_nothing(runtime, heads, seq, dim, causal, special):
    # One tiny V in place of a zero: the other dims' bits (and so the work done
    # for them) stay as they were.
    n = heads * seq * dim
    q, k, v = (orc.normal(n, s).reshape(heads, seq, dim).copy() for s in (0xB4, 0xB5, 0xB6))
    v[:, seq // 2, 3] = 0
    plain, _ = attend(runtime, heads, seq, dim, causal, q.ravel(), k.ravel(), v.ravel())
    v[:, seq // 2, 3] = special
    got, _ = attend(runtime, heads, seq, dim, causal, q.ravel(), k.ravel(), v.ravel())
    other = [d for d in range(dim) if d != 3]
    np.testing.assert_array_equal(got.reshape(n // dim, dim)[:, other], plain.reshape(n // dim, dim)[:, other])


@pytest.mark.parametrize("heads,seq,dim,causal", FLASH)
@pytest.mark.parametrize("special", [1e-25, 1e-42])
def test_flash_on_parts_tiny_query_costs_nothing(runtime, heads, seq, dim, causal, special):
    # One tiny Q element in place of a zero moves no score, so all bits (and so
    # the work done) stay as they were.
    n = heads * seq * dim
    q, k, v = (orc.normal(n, s).reshape(heads, seq, dim).copy() for s in (0xB7, 0xB8, 0xB9))
    q[:, ::20, 3] = 0
    plain, _ = attend(runtime, heads, seq, dim, causal, q.ravel(), k.ravel(), v.ravel())
    q[:, ::20, 3] = special
    got, _ = attend(runtime, heads, seq, dim, causal, q.ravel(), k.ravel(), v.ravel())
    np.testing.assert_array_equal(got, plain)


@pytest.mark.parametrize("heads,seq,dim,causal", FLASH)
def test_flash_on_parts_subnormal_operands(runtime, heads, seq, dim, causal):
    # Q (or K) below 2^-110, subnormals among it, against K (or Q) as large: ordinary scores.
    n = heads * seq * dim
    v = orc.normal(n, 0xBC)
    for tiny_q in (True, False):
        small = (orc.normal(n, 0xBA).astype(np.float64) * 2.0 ** -126).astype(np.float32)
        large = orc.normal(n, 0xBB) * np.float32(2.0 ** 124)
        q, k = (small, large) if tiny_q else (large, small)
        got, _ = attend(runtime, heads, seq, dim, causal, q, k, v)
        s = (np.float32(2.0 ** 64), np.float32(2.0 ** -64))
        want = orc.attention_reference(heads, seq, dim, causal, *((q * s[0], k * s[1]) if tiny_q else (q * s[1], k * s[0])), v)
        assert orc.compare(got, want, 2e-5, 2e-5).status == 0, tiny_q
