"""CPU model of the cell exchange of csrc/hip/sor_resident.h: tiles of several waves, three planes
whose cells are marked until they are given, each wave at its own pace.  A wave's rows are also read by
tiles that it takes nothing from itself, so when a wave marks its cells again on its own account --
straight after its take -- a slow reader can find them marked and the solve stands still; behind the next
barrier of its tile it cannot.  Every schedule is one that the GPU could run: at each turn any wave
whose next operation does not have to wait may go on."""
import random

import pytest

MARK = None
WAVES = 4  # rows of one wave each: 0 and 3 hold the halo, 1 and 2 are owned


class Tile:
    def __init__(self, i, j, grid, order):
        self.i, self.j, self.grid, self.order = i, j, grid, order
        self.at = [(0, 0)] * WAVES  # epoch, operation
        self.arrived = [0] * WAVES  # barriers

    def sources(self, w):
        """(tile, row) pairs whose cells wave w takes."""
        rows, cols = self.grid["shape"]
        out = []
        for di in (-1, 0, 1):
            for dj in (-1, 0, 1):
                i, j = self.i + di, self.j + dj
                if (di or dj) and 0 <= i < rows and 0 <= j < cols:
                    if w == 0 and di == -1:
                        out += [((i, j), 1), ((i, j), 2)]  # thicker halos than a wave: both owned rows
                    if w == WAVES - 1 and di == 1:
                        out += [((i, j), 1), ((i, j), 2)]
                    if w in (1, 2) and di == 0:
                        out.append(((i, j), w))
        return out

    def ready(self, w):
        e, op = self.at[w]
        name = self.order[op]
        if name == "barrier":
            return True
        if name == "pass":
            return min(self.arrived) >= self.arrived[w]
        if name == "take":
            plane = self.grid["planes"][(e + 1) % 3]
            return all(plane[s] is not MARK for s in self.sources(w))
        return True

    def run(self, w):
        e, op = self.at[w]
        name, planes, me = self.order[op], self.grid["planes"], (self.i, self.j)
        owned = w in (1, 2)
        if name == "barrier":
            self.arrived[w] += 1
        elif name == "give" and owned:
            assert planes[(e + 1) % 3][me, w] is MARK, "a cell is given before it was marked again"
            planes[(e + 1) % 3][me, w] = e
        elif name == "take":
            for s in self.sources(w):
                assert planes[(e + 1) % 3][s] == e, "cells of another epoch"
        elif name == "mark own" and owned and e > 0:   # what epoch e - 1 gave, straight after the take
            planes[e % 3][me, w] = MARK
        elif name == "mark tile" and owned and e > 1:  # what epoch e - 2 gave, behind the next barrier
            planes[(e - 1) % 3][me, w] = MARK
        self.at[w] = (e, op + 1) if op + 1 < len(self.order) else (e + 1, 0)


def solve(shape, order, seed, epochs=8):
    """Runs `epochs` epochs under a random schedule; False: no wave could go on."""
    rng = random.Random(seed)
    grid = {"shape": shape}
    tiles = [Tile(i, j, grid, order) for i in range(shape[0]) for j in range(shape[1])]
    grid["planes"] = [{((t.i, t.j), w): MARK for t in tiles for w in (1, 2)} for _ in range(3)]
    waves = [(t, w) for t in tiles for w in range(WAVES)]
    slow = set(rng.sample(range(len(waves)), max(1, len(waves) // 6)))  # these get few turns
    while True:
        left = [x for x in range(len(waves)) if waves[x][0].at[waves[x][1]][0] < epochs]
        if not left:
            return True
        can = [x for x in left if waves[x][0].ready(waves[x][1])]
        if not can:
            return False
        quick = [x for x in can if x not in slow]
        t, w = waves[rng.choice(quick if quick and rng.random() < 0.99 else can)]
        t.run(w)


# an epoch: the sweeps' barriers (the last half-sweep's is none: a wave goes on to give), give, take
PER_TILE = ("barrier", "pass", "mark tile", "barrier", "pass", "give", "take")
PER_WAVE = ("barrier", "pass", "barrier", "pass", "give", "take", "mark own")


@pytest.mark.parametrize("shape", [(2, 1), (3, 1), (3, 2), (3, 3)])
def test_marks_behind_the_tiles_barrier_never_stop_a_reader(shape):
    assert all(solve(shape, PER_TILE, seed) for seed in range(30))


@pytest.mark.parametrize("shape", [(3, 1), (3, 3)])
def test_marks_by_each_wave_on_its_own_would(shape):
    assert not all(solve(shape, PER_WAVE, seed) for seed in range(30))
