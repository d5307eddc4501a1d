"""CPU restatement of the persistent GEMM's staging on bf16 parts
(gemm_f32_ring in jade-compute_amd/csrc/gemm_ring.hip): the LDS writes of a
stage fill each part's 128 rows of A and of B once; the operand reads of both
half-stages return the k and the row or column that the MFMA layout needs; the
reads cover every bank evenly; the buffer offsets stay inside a tile; and no
buffer is written while a wave may still read it. And of the split itself
(csrc/split_bf16.hpp): exact for every finite value in range, and how much the
three products of parts that are not taken can amount to."""
import numpy as np
import pytest

PART, B_REGION, STAGE = 8192, 3 * 8192, 6 * 8192


def parts_of(x):
    """The three bf16 parts of FP32 values, each held in FP32, and what they leave."""
    parts, rest = [], x
    for _ in range(3):
        bits = rest.view(np.uint32).astype(np.uint64)
        part = ((bits + 0x7FFF + ((bits >> 16) & 1)) >> 16 << 16).astype(np.uint32).view(np.float32)
        parts.append(part)
        rest = rest - part
    return parts, rest


# The operands' scale and the largest exponent that stays in range with it: GEMM; attention's V and Q.
@pytest.mark.parametrize("scale,top,least", [(2.0 ** 16, 110, 0.0), (2.0 ** 24, 102, 2.0 ** -126)])
def test_split_of_scaled_values_is_exact(scale, top, least):
    rng = np.random.default_rng(1)
    mantissas = np.unique(np.concatenate([rng.integers(0, 1 << 23, 4096), [0, 1, 2, 0x7FFF, 0x8000, 0x8001, 0x7F7FFF,
                                                                           0x7F8000, 0x7FFFFF]])).astype(np.uint32)
    for exponent in range(0, 127 + top + 1):  # 0: subnormals and zero
        x = (mantissas | np.uint32(exponent << 23)).view(np.float32)
        parts, rest = parts_of(x * np.float32(scale))
        assert not rest.any() and np.isfinite(parts[0]).all()
        sizes = np.abs(np.stack(parts))
        # No part below what the instructions on the way keep (0: bf16's subnormals).
        assert (sizes[sizes > 0] >= least).all()


def test_products_left_out_stay_below_half_an_ulp():
    x = (np.arange(1 << 23, dtype=np.uint32) | np.uint32(0x3F800000)).view(np.float32)
    (_, second, third), _ = parts_of(x)
    p1, p2 = (np.abs(p.astype(np.float64)) / x for p in (second, third))
    assert 2 * p1.max() * p2.max() + p2.max() ** 2 < 0.996 * 2.0 ** -24
    rng = np.random.default_rng(2)
    i, j = rng.integers(0, 1 << 23, (2, 1 << 20))
    s, t, x = second.astype(np.float64), third.astype(np.float64), x.astype(np.float64)
    lost = (s[i] * t[j] + t[i] * s[j] + t[i] * t[j]) / (x[i] * x[j])
    assert np.sqrt((lost ** 2).mean()) < 2.0 ** -27.4


def swz(row):
    return (row >> 2) & 3


def staged(dual):
    """(LDS byte of every 2-byte element of part 0) -> (matrix, row or column, k), as the threads write it."""
    lds = {}
    for tid in range(512):
        wave, lane = tid >> 6, tid & 63
        ar, aq = tid >> 2, tid & 3
        for e in range(8):
            at = ar * 64 + ((aq ^ swz(ar)) << 4) + 2 * e
            assert at not in lds
            lds[at] = ("A", ar, 8 * aq + e)
        br = (lane >> 5) * 64 + (lane & 31)
        for col in range(2):
            for e in range(4):
                at = B_REGION + br * 64 + (((wave >> 1) ^ swz(br)) << 4) + (wave & 1) * 8 + col * 2048 + 2 * e
                assert at not in lds
                name, column = (("gate", "up")[col], lane) if dual else ("B", 2 * lane + col)
                lds[at] = (name, column, 4 * wave + e)
    return lds


@pytest.mark.parametrize("dual", [False, True])
def test_operand_reads_return_what_was_staged(dual):
    lds = staged(dual)
    assert len(lds) == 2 * 128 * 32
    assert max(lds) < STAGE
    for wave in range(8):
        wm, wn = wave >> 1, wave & 1
        for lane in range(64):
            h, c = lane >> 5, lane & 31
            for half in range(2):
                ra = (32 * wm + c) * 64 + (((2 * half + h) ^ swz(c)) << 4)
                rb = B_REGION + (64 * wn + c) * 64 + (((2 * half + h) ^ swz(c)) << 4)
                for e in range(8):
                    k = 16 * half + 8 * h + e
                    assert lds[ra + 2 * e] == ("A", 32 * wm + c, k)
                    for j in range(2):
                        want = (("gate", "up")[j], 32 * wn + c, k) if dual else ("B", 64 * wn + 2 * c + j, k)
                        assert lds[rb + 2048 * j + 2 * e] == want


def test_reads_spread_over_the_banks():
    # ds_read_b128 serves 16 consecutive lanes from 256 bytes of banks.
    for first in range(0, 64, 16):
        lanes = np.arange(first, first + 16)
        h, c = lanes >> 5, lanes & 31
        for half in range(2):
            at = c * 64 + (((2 * half + h) ^ swz(c)) << 4)
            assert len(set((at % 256) // 16)) == 16


@pytest.mark.parametrize("n,k", [(4096, 4096), (11008, 4096), (1024, 2816), (128, 512)])
def test_loads_stay_inside_the_stage(n, k):
    tid = np.arange(512)
    wave, lane = tid >> 6, tid & 63
    va = ((tid >> 2) * k + 8 * (tid & 3)) * 4
    seen = np.concatenate([va + 16 * x for x in range(2)])
    assert len(set(seen.tolist())) == 1024 and seen.max() + 16 <= (127 * k + 32) * 4
    vb = (4 * wave * n + 2 * lane) * 4
    seen = np.concatenate([vb + e * n * 4 for e in range(4)])
    assert len(set(seen.tolist())) == 2048 and seen.max() + 8 <= (31 * n + 128) * 4


def test_stage_buffers_are_free_when_written():
    # Events of one wave in program order; a barrier opens half 1 of every
    # stage. Between two waves only the barriers order anything, so a write
    # may fall anywhere from the barrier before it to the barrier after it, and
    # so may a read.
    writes, reads, barrier = [], [], 0
    writes += [("B", 0, 0, 0), ("A", 0, 0, 0), ("A", 1, 1, 0)]  # prologue: matrix, stage, buffer, barriers passed
    barrier = 1
    reads += [(0, 0, 0, barrier)]  # stage, half, buffer, barriers passed
    for g in range(12):
        p = g & 1
        reads.append((g, 1, p, barrier))  # half 0 reads half 1's operands
        writes.append(("B", g + 1, p ^ 1, barrier))
        barrier += 1
        reads.append((g + 1, 0, p ^ 1, barrier))
        writes.append(("A", g + 2, p, barrier))
    for matrix, stage, buf, when in writes:
        assert buf == stage & 1
        for s, half, b, at in reads:
            if b != buf:
                continue
            if s == stage:
                assert when < at  # published by a barrier before the read
            if s < stage:
                assert at < when  # the older stage's reads lie a barrier back
            if s > stage:
                assert when < at
