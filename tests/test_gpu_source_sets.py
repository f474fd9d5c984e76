"""GPU tests of the particle source's sizing by each set's own entry count:
sets of growing and shrinking size on one handle, an empty set, sets of which
nothing reaches a cell, and a set above the entry limit, which is refused (as
is its repeat) and leaves the handle usable. Bit for bit the oracle's."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(__file__))
from test_gpu_parity import B, compare, pair, random_state, settings  # noqa: E402

pytestmark = pytest.mark.gpu


def particles(n, seed, dx, cells):
    rng = np.random.default_rng(seed)
    a = np.zeros((n, 8), np.float32)
    a[:, 0:3] = rng.uniform(-0.1, 1.1, (n, 3))
    a[:, 3:6] = rng.standard_normal((n, 3))
    a[:, 6] = rng.uniform(*cells, n) * dx
    a[:, 7] = rng.uniform(0.1, 2.0, n)
    return a


def test_sets_in_turn():
    s = settings(B, (32, 24, 20), smoke_density=0.5)
    g, o = pair(s, random_state(s, 6, smoke=True))
    dx = float(s.dx)
    sets = [particles(700, 1, dx, (0.4, 3.0)), particles(9000, 2, dx, (0.45, 0.8)), np.zeros((0, 8), np.float32),
            particles(3, 3, dx, (1.0, 6.0)), particles(500, 4, dx, (0.1, 0.5)), particles(4097, 5, dx, (0.3, 2.5))]
    for q, p in enumerate(sets):
        print(f"[source] set {q}: {len(p)} particles", flush=True)
        for x in (g, o):
            x.add_source(p)
            x.add_source(None)
        for w in range(5):
            compare(f"set {q} field {w}", g.field(w), o.field(w))


def test_set_above_the_entry_limit():
    s = settings(B, (16, 16, 16))
    g, o = pair(s, random_state(s, 7))
    dx = float(s.dx)
    big = particles(8, 1, dx, (1.0, 2.0))
    big[3, 6] = 1e5 * dx
    for _ in range(2):
        with pytest.raises(B.BlazeError, match="2\\^31 entries"):
            g.add_source(big)
        with pytest.raises(B.BlazeError, match="2\\^31 entries"):
            g.add_source(None)
    p = particles(300, 2, dx, (1.0, 3.0))
    g.add_source(p)
    o.add_source(p)
    for w in range(4):
        compare(f"field {w}", g.field(w), o.field(w))
