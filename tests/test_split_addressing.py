"""CPU restatement of the persistent GEMM's staging on bf16 parts
(gemm_f32_ring in jade-compute_amd/csrc/gemm_ring.hip): the LDS writes of a
stage fill each part's 128 rows of A and of B once; the operand reads of both
half-stages return the k and the row or column that the MFMA layout needs; the
reads cover every bank evenly; the buffer offsets stay inside a tile; and no
buffer is written while a wave may still read it."""
import numpy as np
import pytest

PART, B_REGION, STAGE = 8192, 3 * 8192, 6 * 8192


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
