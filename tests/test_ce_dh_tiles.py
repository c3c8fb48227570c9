"""The cross-entropy dH's work list (``DhTiles``, ``dh_slots`` in
``siq_vl_amd/csrc/flce.hip``), as a Python model: every token tile of a chunk
gets each of its vocab ranges, or parts of one, exactly once, within the slots
the workspace and the grid hold, and whether a row's ranges are cut depends on
the batch's counted rows alone, not on the chunk."""

import random

import pytest

BJ, XCDS, SUB, ROUND = 256, 8, 4, 32


def ceil(a, b):
    return -(-a // b)


class Tiles:
    def __init__(self, nvalid, c0, nv, n_i, splits, run):
        self.t0 = c0 // BJ
        self.t1 = ceil(c0 + nv, BJ) if nv > 0 else self.t0
        self.run, self.nj = run, ceil(nvalid, BJ)

        def cut(n):
            return min(n, (n * n_i % ROUND + n_i - 1) // n_i) if splits == XCDS else 0

        self.full, self.last = cut(run), cut(self.nj % run)

    def cut_before(self, t):
        g, i, whole = t // self.run, t % self.run, self.nj // self.run
        return g * self.full + max(0, i - (self.run - self.full) if g < whole
                                   else i - (self.nj - whole * self.run - self.last))

    def at(self, t):
        return t - self.t0 + (SUB - 1) * (self.cut_before(t) - self.cut_before(self.t0))

    def cut(self, t):
        return self.cut_before(t + 1) > self.cut_before(t)


def slots(c0, nc, n_i, splits, run):
    t0, t1 = c0 // BJ, ceil(c0 + nc, BJ)
    if splits < XCDS:
        return (t1 - t0) * splits
    cut = min(run, (ROUND - 1 + n_i - 1) // n_i) * ((t1 - 1) // run - t0 // run + 1)
    return XCDS * (t1 - t0 + (SUB - 1) * min(t1 - t0, cut))


@pytest.mark.parametrize("seed", range(8))
def test_every_range_once_and_the_cut_independent_of_the_chunk(seed):
    rng = random.Random(seed)
    for _ in range(250):
        n = rng.randint(1, 20000)
        chunk = min(n, rng.choice([n, rng.randint(1, n), BJ * rng.randint(1, 60)]))
        if n / chunk > 40:
            continue
        n_i, run, nvalid = rng.randint(1, 20), rng.choice([1, 2, 4, 27, 80, 8000]), rng.randint(0, n)
        splits = max(1, min(XCDS, ceil(2048, n_i * ceil(chunk, BJ))))
        batch = Tiles(nvalid, 0, nvalid, n_i, splits, run)
        for c0 in range(0, n, chunk):
            nc = min(chunk, n - c0)
            nv = min(nc, nvalid - c0)
            t = Tiles(nvalid, c0, nv, n_i, splits, run)
            held = slots(c0, nc, n_i, splits, run)
            got = {}
            for unit in range(XCDS * ceil(held, XCDS)):
                u, x = unit // XCDS, unit % XCDS
                if splits < XCDS:
                    tile, part = t.t0 + unit // splits, unit % splits
                    if tile >= t.t1:
                        continue
                else:
                    if t.t1 == t.t0 or u >= t.at(t.t1):
                        continue
                    tile, end = t.t0, t.t1
                    while end - tile > 1:
                        mid = (tile + end) // 2
                        tile, end = (mid, end) if t.at(mid) <= u else (tile, mid)
                    part = (u - t.at(tile), x)
                    assert 0 <= part[0] < (SUB if t.cut(tile) else 1)
                assert unit < held
                got.setdefault(tile, []).append(part)
            assert sorted(got) == list(range(t.t0, t.t1))
            for tile, parts in got.items():
                want = splits if splits < XCDS else XCDS * (SUB if t.cut(tile) else 1)
                assert len(parts) == len(set(parts)) == want
                assert t.cut(tile) == batch.cut(tile)
                # the rows of a slot: the tile's rows of the chunk
                rows = min((tile + 1) * BJ - c0, nv) - max(tile * BJ - c0, 0)
                assert 0 < rows <= min(chunk, BJ)
