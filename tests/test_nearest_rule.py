"""The start slot of k_nearest_insert's cascades (csrc/ud_gather.hip), modelled on the CPU
under random interleavings of the row's reads and atomic minima.

A candidate word starts at the number of smaller words known: those of the row as its
pixel's lanes read it, and those of the pixel's other candidates that are not in it.  With
one copy of the row per pixel the rows come out as the K smallest distinct words in order,
whatever the interleaving.  With a copy per lane they do not: a mate's word that another
pixel inserts between two lanes' reads is counted twice."""
import random

import pytest

EMPTY = 1 << 64


def read_row(row, K):
    """One read per word, each an event of its own."""
    copy = []
    for j in range(K):
        copy.append(row[j])
        yield
    return copy


def start_slot(copy, key):
    """(distinct smaller words of the copy as the kernel counts them, key is there)"""
    pos, top = 0, 0
    for j, v in enumerate(copy):
        pos += v < key and (j == 0 or v > top)
        top = max(top, v)
    return pos, key in copy


def cascade(row, K, pos, key):
    for j in range(pos, K):
        old = row[j]
        row[j] = min(old, key)                      # atomicMin
        if old == key or old == EMPTY:
            return
        key = max(old, key)
        yield


def interleave(rng, tasks):
    """Runs generators one event at a time in random order."""
    tasks = list(tasks)
    while tasks:
        t = rng.randrange(len(tasks))
        try:
            next(tasks[t])
        except StopIteration:
            tasks.pop(t)


def pixel(rng, row, K, keys, per_lane):
    """A wavefront's pixel: the lanes read (in step or each for itself), then all cascade."""
    if per_lane:
        copies = [[] for _ in keys]
        for j in range(K):                          # one load instruction, served lane by lane
            for copy in rng.sample(copies, len(copies)):
                copy.append(row[j])
                yield
    else:
        copy = yield from read_row(row, K)
        copies = [copy] * len(keys)
    found = [start_slot(c, key) for c, key in zip(copies, keys)]
    mine = [EMPTY if there else key for key, (_, there) in zip(keys, found)]
    mine = [EMPTY if key in mine[:q] else key for q, key in enumerate(mine)]
    runs = [cascade(row, K, pos + sum(m < key for m in mine), key)
            for key, (pos, _) in zip(mine, found) if key != EMPTY]
    while runs:                                     # the lanes' atomics, in any order
        r = rng.choice(runs)
        try:
            next(r)
        except StopIteration:
            runs.remove(r)
        yield


def wrong_rows(per_lane, trials, seed):
    rng = random.Random(seed)
    wrong = 0
    for _ in range(trials):
        K, pixels, lanes, words = rng.randint(1, 6), rng.randint(1, 5), rng.randint(1, 5), rng.randint(1, 9)
        row = [EMPTY] * K
        keys = [[rng.randrange(words) for _ in range(lanes)] for _ in range(pixels)]
        interleave(rng, [pixel(rng, row, K, k, per_lane) for k in keys])
        ref = sorted({x for k in keys for x in k})[:K]
        wrong += row != ref + [EMPTY] * (K - len(ref))
    return wrong


@pytest.mark.parametrize("seed", range(4))
def test_rows_whatever_the_interleaving(seed):
    assert wrong_rows(False, 5000, seed) == 0


def test_model_shows_a_row_read_per_lane():
    assert wrong_rows(True, 5000, 0) > 0
