"""The lookups an example of the forward combiner sums (csrc/lookup_range.h), for example ids in any order: a replay of the
workgroup's check, which refuses lookups out of order, leaves no range outside the lookups it looked at, and the right ones
where the ids are in order.  Host code, compiled here by itself."""
import ctypes
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tensornet_amd", "csrc")
SOURCE = """
#include "lookup_range.h"
extern "C" void range(unsigned first, unsigned behind, unsigned lo, unsigned* out) {
    const tn::LookupRange r = tn::lookup_range(first, behind, lo);
    out[0] = r.from;
    out[1] = r.to;
}
"""


@pytest.fixture(scope="module")
def lookup_range(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("lookup_range")
    (tmp / "r.cc").write_text(SOURCE)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, str(tmp / "r.cc"), "-o", str(tmp / "r.so")])
    f = ctypes.CDLL(str(tmp / "r.so")).range

    def call(first, behind, lo):
        out = (ctypes.c_uint * 2)()
        f(first, behind, lo, out)
        return out[0], out[1]

    return call


def ranges(lookup_range, ex, lo, hi, b0, nb, order):
    """What the check of lookups [lo, hi) by the workgroup of examples b0 .. b0 + nb - 1 leaves, lookups taken in `order`."""
    first, behind = [0] * nb, [0] * nb
    for i in order:
        x, prev, after = ex[i], ex[i - 1] if i else -1, ex[i + 1] if i + 1 < len(ex) else b0 + nb
        if x < b0 or x >= b0 + nb or prev > x:
            continue
        if prev != x or i == lo:
            first[x - b0] = i
        if after != x or i + 1 == hi:
            behind[x - b0] = i + 1
    return [lookup_range(f, b, lo) for f, b in zip(first, behind)]


def test_a_run_behind_its_neighbour(lookup_range):
    ex = [i // 3 for i in range(256 * 3)]
    ex[210:216] = [71] * 3 + [70] * 3
    for f, t in ranges(lookup_range, ex, 192, 384, 64, 64, range(192, 384)):
        assert f == t or 192 <= f < t <= 384


@pytest.mark.parametrize("seed", range(40))
def test_no_range_leaves_the_lookups(lookup_range, seed):
    rng = random.Random(seed)
    n, batch = rng.randint(1, 120), rng.randint(1, 40)
    for _ in range(50):
        ex = sorted(rng.randrange(batch) for _ in range(n))
        kind = rng.randrange(3)
        if kind == 1:
            rng.shuffle(ex)
        elif kind == 2:  # one run moved
            a, b, c = sorted(rng.randrange(n + 1) for _ in range(3))
            ex = ex[:a] + ex[b:c] + ex[a:b] + ex[c:]
        b0 = rng.randrange(batch)
        nb = rng.randint(1, batch - b0)
        if kind == 0:
            lo, hi = sum(x < b0 for x in ex), sum(x < b0 + nb for x in ex)
        else:
            lo = rng.randrange(n + 1)
            hi = rng.randint(lo, n)
        order = list(range(lo, hi))
        rng.shuffle(order)
        got = ranges(lookup_range, ex, lo, hi, b0, nb, order)
        for e, (f, t) in enumerate(got):
            assert f == t or lo <= f < t <= hi
            if kind == 0:
                assert list(range(f, t)) == [i for i in range(n) if ex[i] == b0 + e]
