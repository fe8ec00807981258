"""How a resident sweep splits an RVE over workgroups and lanes, followed on the
host with the kernel's own functions: every interior node belongs to one item, and
every word that a neighbouring rank reads is published by one lane, into the place
where the reader's product looks for that node."""
import collections
import ctypes as C
import random

import pytest

from madmax_amd import _lib


def split(n, fp64, nrhs, max_rves, slab_nodes=128, ncu=256):
    """(ranks, shares of the rows, planes per item, items per column); 0 ranks: not swept on chip."""
    return split_meet(n, fp64, nrhs, max_rves, slab_nodes, ncu)[:4]


def split_meet(n, fp64, nrhs, max_rves, slab_nodes, ncu):
    """The same and how the ranks meet before they wait for each other: 1 with patience, 2 without, 0 not (one)."""
    out = (C.c_int * 5)()
    assert _lib.lib().mm_sweep_split(*n, int(fp64), nrhs, max_rves, slab_nodes, ncu, out) == 0
    return tuple(out)


def faults(n, fp64, s):
    out = (C.c_int * 4)()
    assert _lib.lib().mm_sweep_check(*n, int(fp64), (C.c_int * 4)(*s), out) == 0
    return tuple(out)


def runs(n, s):
    """Of the ranks' shares of the planes: does one end in a run shorter than the others, and in an empty one?"""
    cw, ty, lp, nch = s
    niz, cz = n[2] - 1, cw // ty
    shares = {(r + 1) * niz // cz - r * niz // cz for r in range(cz)}
    used = {-(-p // lp) for p in shares}
    return any(p % lp for p in shares), min(used) < nch


# cells whose smaller shares leave the last run of every column empty
EMPTY_RUN = [((26, 26, 26), True, 1, 4096), ((19, 19, 26), True, 6, 4), ((19, 19, 26), False, 6, 4),
             ((4, 4, 44), False, 6, 8)]


@pytest.mark.parametrize("n,fp64,nrhs,max_rves", EMPTY_RUN)
def test_an_empty_last_run(n, fp64, nrhs, max_rves):
    s = split(n, fp64, nrhs, max_rves)
    assert s[0] > 1 and runs(n, s)[1], s
    assert faults(n, fp64, s) == (0, 0, 0, 0)


def test_every_word_that_is_read_is_published():
    rng = random.Random(5)
    kinds, lengths, shared = collections.Counter(), set(), 0
    for _ in range(4000):
        n = tuple(rng.randint(2, rng.choice([8, 24, 60, 110])) for _ in range(3))
        fp64, nrhs = rng.random() < 0.5, rng.choice([1, 6, 7])
        max_rves, slab_nodes = rng.choice([1, 2, 4, 8, 16, 32, 64, 256, 4096]), rng.choice([64, 128, 256])
        s = split(n, fp64, nrhs, max_rves, slab_nodes)
        if s[0] == 0:
            continue
        assert faults(n, fp64, s) == (0, 0, 0, 0), (n, fp64, nrhs, max_rves, slab_nodes, s)
        if s[0] > 1:
            kinds[runs(n, s)] += 1
            shared += s[1] > 1
        lengths.add((fp64, s[2]))
    # every kind of split was among them
    assert kinds[True, False] > 100 and kinds[False, False] > 100 and kinds[True, True] + kinds[False, True] > 20
    assert shared > 100 and lengths >= {(False, i) for i in range(1, 9)} | {(True, i) for i in range(1, 5)}


@pytest.mark.parametrize("ncu", [1, 8, 32, 64, 128, 256, 304])
def test_splits_fit_the_device(ncu):
    """A cluster never has more ranks than the device can run at once, all but single workgroups meet first, and one
    that waits with patience is small enough that four of them leave room for a missing rank."""
    rng, some = random.Random(ncu), 0
    for _ in range(1500):
        n = tuple(rng.randint(2, rng.choice([24, 60, 110])) for _ in range(3))
        fp64, nrhs, max_rves = rng.random() < 0.5, rng.choice([1, 6, 7]), rng.choice([1, 4, 16, 64, 4096])
        s = split_meet(n, fp64, nrhs, max_rves, 128, ncu)
        if s[0] == 0:
            continue
        some += 1
        assert s[0] <= max(1, min(ncu - 1, 240)) and faults(n, fp64, s[:4]) == (0, 0, 0, 0)
        assert (s[4] > 0) == (s[0] > 1)
        if s[4] == 1:
            assert s[0] <= 16 and 4 * (s[0] - 1) < ncu
    assert some > 100


def test_cells_without_an_interior_or_too_wide_are_not_swept():
    for n in ((1, 4, 5), (4, 1, 5), (4, 5, 1), (4098, 2, 2), (2, 4098, 2), (130, 130, 130)):
        assert split(n, False, 6, 16)[0] == 0
    assert split((100, 100, 100), False, 1, 9)[0] > 0 and split((85, 85, 85), True, 1, 9)[0] > 0


@pytest.mark.parametrize("n", [(32, 3, 4), (10, 9, 6), (9, 8, 40), (20, 17, 11), (31, 32, 6), (32, 32, 3), (34, 33, 3),
                               (24, 23, 12), (40, 36, 3), (7, 7, 7), (21, 22, 19), (12, 10, 17), (33, 34, 2),
                               (37, 35, 5), (70, 40, 4), (130, 9, 6), (5, 300, 3), (34, 38, 21), (2, 2, 2), (2, 3, 9)])
def test_cells_of_the_sweep_tests_are_swept(n):
    for fp64 in (False, True):
        for max_rves in (32, 64):
            assert split(n, fp64, 6, max_rves)[0] > 0


@pytest.mark.parametrize("fp64,n,max_rves,large", [
    (False, (24, 22, 20), 4, False), (False, (44, 41, 39), 200, False), (False, (60, 52, 50), 4, True),
    (False, (82, 80, 78), 2, True), (True, (30, 28, 26), 2, False), (True, (50, 47, 45), 200, True),
    (False, (72, 70, 68), 3, True), (False, (100, 100, 100), 9, True)])
def test_cells_of_the_one_load_case_tests_are_swept(fp64, n, max_rves, large):
    """And those that are to be split over large clusters are."""
    s = split_meet(n, fp64, 1, max_rves, 128, 256)
    assert s[0] > 1 and s[4] == (2 if large else 1)
