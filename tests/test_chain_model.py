"""The hand-over of a row that two logical waves share (chain_add in
bhs_kernels.h), every interleaving of the two waves' memory operations: one wave
finishes the row with both of the other's halves, it waits for nothing, and the
words are empty afterwards (CPU only)."""
import itertools

import pytest

CALL = 7
STALE = (3 << 1 | 1, "stale")            # in a pair word, left behind by another call


def wave(side, order, halves):
    """One wave as a generator of memory operations; returns the value it finishes
    the row with, or None.  Words: pair[0..1], count; an empty word is (0, None)."""
    tag, n = CALL << 1 | side, len(halves)
    got = [None] * n
    for h in order:                       # the lanes' exchanges, in either order
        got[h] = yield "xchg", ("pair", h), (tag, halves[h])
    found = [g[0] == tag ^ 1 for g in got]
    if not any(found):
        return None
    if not all(found):
        seen = yield "xchg", "count", (CALL, 1)
        if seen[0] != CALL:
            return None
        for h in range(n):
            if not found[h]:
                got[h] = yield "load", ("pair", h), None
        yield "store", "count", (0, None)
    for h in range(n):
        yield "store", ("pair", h), (0, None)
    return [g[1] for g in got]


def run(mem, waves, schedule):
    """Steps the waves as `schedule` says, then whichever is left."""
    results, todo, reply = [None, None], [0, 1], [None, None]
    steps = itertools.chain(schedule, itertools.cycle([0, 1]))
    while todo:
        i = next(steps)
        if i not in todo:
            continue
        try:
            op, word, value = waves[i].send(reply[i])
        except StopIteration as e:
            results[i] = e.value
            todo.remove(i)
            continue
        old = mem[word]
        if op != "load":
            mem[word] = value
        reply[i] = old
    return results


@pytest.mark.parametrize("n", [1, 2])     # halves: 4-byte values have one
@pytest.mark.parametrize("left", [(0, None), STALE])
def test_one_wave_finishes_with_both_halves(n, left):
    values = [[f"{s}{h}" for h in range(n)] for s in "ab"]
    orders = list(itertools.permutations(range(n)))
    for oa, ob in itertools.product(orders, orders):
        for schedule in itertools.product([0, 1], repeat=10):
            mem = {("pair", h): left for h in range(n)}
            count = mem["count"] = (left[0] >> 1, left[1])
            for _ in range(2):            # a replay of the same call finds empty words
                out = run(mem, [wave(0, oa, values[0]), wave(1, ob, values[1])], schedule)
                assert sorted(o is None for o in out) == [False, True]
                who = 0 if out[0] is not None else 1
                assert out[who] == values[1 - who]
                assert all(mem["pair", h] == (0, None) for h in range(n))
                assert mem["count"] in ((0, None), count)
