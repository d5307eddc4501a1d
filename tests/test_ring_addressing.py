"""CPU restatement of the persistent 128x128 GEMM's schedule
(gemm_f32_ring in jade-compute_amd/csrc/gemm_ring.hip): the workgroup-to-tile
map covers every tile once and gives every workgroup a run of whole tiles; the
load cursors bring each stage of each tile in turn, past the last one too, from
inside A and B; no register set is loaded before its stage is converted, none
converted before it is loaded; the epilogue's stores cover a tile once in every
form, and the FP32 recomputation reads the rows, columns and k of the outputs
that it replaces. The LDS side is restated in test_split_addressing.py."""
import numpy as np
import pytest

BK, BM, BN = 32, 128, 128
CUS, GROUP_M = 256, 8
WAVES, LANES = 8, 64


def xcd_order(bid, count):
    per, rem = divmod(count, 8)
    xcd, idx = bid % 8, bid // 8
    return xcd * per + min(xcd, rem) + idx


def grouped_tile(logical, tiles_m, tiles_n):
    span = GROUP_M * tiles_n
    group, inside = divmod(logical, span)
    first = group * GROUP_M
    rows = min(tiles_m - first, GROUP_M)
    return first + inside % rows, inside // rows


@pytest.mark.parametrize("tiles_m,tiles_n", [(32, 32), (32, 86), (16, 16), (40, 40), (34, 32), (96, 8), (32, 22)])
def test_persistent_map_covers_every_tile_once(tiles_m, tiles_n):
    # Workgroup b takes tiles pos(b) + j * G of the grouped order, j < mine:
    # every tile once, and the runs differ in length by at most one tile.
    tiles = tiles_m * tiles_n
    nwg = min(tiles, CUS)
    count, runs = {}, []
    for b in range(nwg):
        pos = xcd_order(b, nwg)
        mine = (tiles - pos + nwg - 1) // nwg
        runs.append(mine)
        for j in range(mine):
            key = grouped_tile(j * nwg + pos, tiles_m, tiles_n)
            count[key] = count.get(key, 0) + 1
    assert len(count) == tiles and set(count.values()) == {1}
    assert max(runs) - min(runs) <= 1 and sum(runs) == tiles


class Cursor:
    """load_a's or load_b's cursor: (tile, stage) of the next load."""

    def __init__(self, nk):
        self.nk, self.tile, self.stage = nk, 0, 0

    def take(self, next_tile):
        at = (self.tile, self.stage)
        self.stage += 1
        if self.stage == self.nk:
            self.tile, self.stage = next_tile, 0
        return at


@pytest.mark.parametrize("n,k", [(4096, 4096), (11008, 4096), (1024, 2816), (128, 512)])
def test_stage_loads_fill_their_slot_once(n, k):
    # One stage's loads of all threads: rows [0, 128) x k [0, 32) of A and rows
    # [0, 32) x columns [0, 128) of B (of 64 columns of each product, fused),
    # each element once, from 32-bit offsets.
    tid = np.arange(512)
    wave, lane = tid >> 6, tid & 63
    a = ((tid >> 2) * k + 8 * (tid & 3))[:, None] + np.arange(8)
    assert len(set(a.ravel().tolist())) == BM * BK
    assert (a // k).max() == BM - 1 and (a % k).max() == BK - 1 and 4 * int(a.max()) + 4 < 2 ** 31
    for cols, width in ((2 * lane, 2), (lane, 1)):
        b = (4 * wave * n + cols)[:, None, None] + n * np.arange(4)[:, None] + np.arange(width)
        assert len(set(b.ravel().tolist())) == BK * 64 * width
        assert (b // n).max() == BK - 1 and (b % n).max() == 64 * width - 1 and 4 * int(b.max()) + 4 < 2 ** 31


@pytest.mark.parametrize("nk,mine", [(16, 1), (16, 3), (88, 2), (24, 5)])
def test_ring_schedule_never_overwrites_a_live_slot(nk, mine):
    # Two register sets for A and two for B. Stage g converts B of g + 1, then
    # loads g + 3 into that set, then converts A of g + 2 and loads g + 4. Every
    # conversion must find its own stage of its own tile in the set.
    aim = {"next": min(1, mine - 1)}
    cursors, sets = {"a": Cursor(nk), "b": Cursor(nk)}, {}
    done = {"a": [], "b": []}

    def load(matrix, which):
        assert sets.get((matrix, which)) is None  # the stage before was converted
        sets[matrix, which] = cursors[matrix].take(aim["next"])

    def convert(matrix, which):
        done[matrix].append(sets[matrix, which])
        sets[matrix, which] = None

    for step, matrix, which in ((load, "a", 0), (load, "b", 0), (load, "a", 1), (load, "b", 1), (convert, "a", 0),
                                (load, "a", 0), (convert, "b", 0), (load, "b", 0), (convert, "a", 1), (load, "a", 1)):
        step(matrix, which)
    for tile in range(mine):
        if tile > 0:
            aim["next"] = min(tile + 1, mine - 1)
        for stage in range(nk):
            p = stage & 1
            convert("b", p ^ 1)
            load("b", p ^ 1)
            convert("a", p)
            load("a", p)
    stages = [(tile, stage) for tile in range(mine) for stage in range(nk)]
    for matrix in ("a", "b"):
        assert done[matrix][:len(stages)] == stages
        assert all(tile == mine - 1 for tile, _ in done[matrix][len(stages):])  # read again, never multiplied


def outputs(dual):
    """(wave, lane, accumulator, value) -> (product, row, column) of the tile, as `store` writes them."""
    for wave in range(WAVES):
        wm, wn = wave >> 1, wave & 1
        for lane in range(LANES):
            h, c = lane >> 5, lane & 31
            for v in range(16):
                row = 32 * wm + 4 * h + 8 * (v >> 2) + (v & 3)
                for j in range(2):
                    yield (wave, lane, j, v), ((j, row, 32 * wn + c) if dual else (0, row, 64 * wn + 2 * c + j))


@pytest.mark.parametrize("dual", [False, True])
def test_epilogue_covers_the_tile_once(dual):
    seen = [place for _, place in outputs(dual)]
    assert len(seen) == len(set(seen)) == BM * BN
    assert max(row for _, row, _ in seen) == BM - 1 and max(col for _, _, col in seen) == (63 if dual else 127)


@pytest.mark.parametrize("dual", [False, True])
def test_operand_reads_return_the_mfma_layout(dual):
    # The FP32 recomputation: lane (h, c) reads A row 32 wm + c and, for
    # accumulator j, B column 64 wn + 2c + j (fused: column 32 wn + c of product
    # j), k 4h + e of every eight. v_mfma_f32_32x32x2_f32 puts row
    # 8 (v >> 2) + 4h + (v & 3) of A's 32 rows and column c of B's 32 into value v
    # of lane (h, c): those must be the row and column that `store` writes.
    assert sorted(4 * h + e for h in range(2) for e in range(4)) == list(range(8))
    for (wave, lane, j, v), (product, row, col) in outputs(dual):
        wm, wn, h, c = wave >> 1, wave & 1, lane >> 5, lane & 31
        a_rows = [32 * wm + i for i in range(32)]
        b_cols = [(j, 32 * wn + i) if dual else (0, 64 * wn + 2 * i + j) for i in range(32)]
        assert a_rows[8 * (v >> 2) + 4 * h + (v & 3)] == row and b_cols[c] == (product, col)
