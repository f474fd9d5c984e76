"""Several sweeps per launch (the default sweeps, variant 2000) against the
oracle bit for bit: every tile size the grid can get, one-column and clipped
tiles at both rims, one to many slab groups (partly filled last groups), a
sweep count that leaves one to the colour passes, and calls of fewer than four
sweeps, which run one sweep per launch."""
import numpy as np
import pytest

B = pytest.importorskip("blaze_amd")
O = pytest.importorskip("oracle")
from helpers import compare, random_state, settings  # noqa: E402

pytestmark = pytest.mark.gpu

# 4x4 tiles up to 64x64 columns, then 8x4, 8x8, 16x8, 16x12 and 16x16
SHAPES = [(4, 4, 4), (6, 5, 9), (34, 33, 32), (64, 61, 6), (66, 90, 13), (90, 75, 5), (130, 66, 22), (122, 128, 8),
          (162, 133, 7), (200, 98, 18), (200, 180, 7), (250, 220, 6)]


def pair(s, st):
    g, o = B.Solver(s), O.Oracle(s)
    for w, a in st.items():
        g.set_field(w, a)
        o.set_field(w, a)
    return g, o


@pytest.mark.parametrize("res", SHAPES, ids=["x".join(map(str, r)) for r in SHAPES])
@pytest.mark.parametrize("iters", [3, 5, 7, 10, 22])
def test_tile_sweeps_bitwise(res, iters):
    print(f"[tiles] res={res} iters={iters}", flush=True)
    s = settings(B, res, max_iter_solve=iters)
    g, o = pair(s, random_state(s, seed=iters + sum(res)))
    for x in (g, o):
        x.run_stage(B.STAGE_PRESSURE, 0.0, 1.0 / 24.0)
    compare("tile sweeps", g.field(B.FIELD_P), o.field(B.FIELD_P))
    assert g.stats().rbgs_kernel == (4 if iters >= 4 else 3)


@pytest.mark.parametrize("every", [1, 2, 3])
@pytest.mark.parametrize("res", [(18, 7, 4), (64, 61, 6), (90, 75, 22), (256, 256, 9), (40, 36, 52)],
                         ids=lambda r: "x".join(map(str, r)))
def test_calls_of_few_sweeps(res, every):
    """Two or three sweeps between checks, or a cap of them: row-pair sweeps
    (an odd one as colour passes), reported as such, whose launches are timed:
    one per sweep and two per colour-passed sweep."""
    print(f"[few sweeps] res={res} every={every}", flush=True)
    s = settings(B, res, max_iter_solve=8, residual_tol=1e-30, residual_check_every=every)
    g, o = pair(s, random_state(s, seed=every + sum(res)))
    g.set_timing(True)
    for x in (g, o):
        x.run_stage(B.STAGE_PRESSURE, 0.0, 1.0 / 24.0)
    st, batches = g.stats(), [every] * (8 // every) + [8 % every] * (8 % every > 0)
    assert st.rbgs_iters_last == o.stats()["rbgs_iters_last"] == 8
    assert st.rbgs_kernel == (1 if batches[-1] == 1 else 3)
    assert st.rbgs_launches == sum(n + n % 2 for n in batches)
    compare("few sweeps", g.field(B.FIELD_P), o.field(B.FIELD_P))


@pytest.mark.parametrize("sweeps", [2, 20])
def test_autotune_times_tile_sweeps(sweeps):
    """However few sweeps the tuner is asked to time, the tiles are timed as a
    solve runs them (at 128^3 they take under half of any other variant's
    time); a solve that checks every two sweeps cannot use them."""
    for every, want in ((10, True), (2, False)):
        s = settings(B, (128, 128, 128), max_iter_solve=20, residual_tol=1e-30, residual_check_every=every)
        g = B.Solver(s)
        v, times = g.autotune(sweeps)
        print(f"[tiles-autotune] {sweeps} sweeps, checks every {every}: {v} {times}", flush=True)
        assert len(times) == 17
        assert (v == 2000) == want


@pytest.mark.parametrize("res,every,want", [((1024, 1024, 8), 10, (1, 2, 3)), ((1024, 1024, 8), 2, (1, 2, 3)),
                                            ((274, 258, 33), 10, (4,)), ((274, 258, 33), 3, (1, 2, 3)),
                                            ((512, 512, 88), 2, (1, 2, 3)), ((256, 256, 5), 10, (4,))],
                         ids=["flat", "flat-2", "wide", "wide-3", "large-2", "tile-per-CU"])
def test_default_sweeps_of_wide_slabs(res, every, want):
    """More than one 16x16 tile per CU: the tiles, except on few slabs, where
    a launch's filling and draining steps cost more than they save (1.5 times
    the best one-sweep variant's time at 1024x1024x8)."""
    print(f"[tiles-wide] res={res} every={every}", flush=True)
    s = settings(B, res, max_iter_solve=every, residual_tol=1e-30, residual_check_every=every)
    rng = np.random.default_rng(every)
    W, H, D = res
    st = {w: rng.random((D, H, W), dtype=np.float32) - np.float32(0.5) for w in (B.FIELD_P, B.FIELD_RHS)}
    g, o = pair(s, st)
    for x in (g, o):
        x.run_stage(B.STAGE_PRESSURE, 0.0, 1.0 / 24.0)
    assert g.stats().rbgs_kernel in want
    compare("wide slab", g.field(B.FIELD_P), o.field(B.FIELD_P))


@pytest.mark.parametrize("kind", ["tiny", "negzero", "decay", "inf"])
@pytest.mark.parametrize("res", [(40, 36, 24), (90, 75, 10), (162, 133, 9), (200, 180, 9), (250, 220, 9)],
                         ids=["4x4", "8x4", "16x8", "16x12", "16x16"])
def test_tile_sweeps_exact_division(kind, res):
    """Numerators outside the fast division's range in some lanes, groups or
    slabs only, and an infinity that spreads."""
    print(f"[tiles-exact] {kind} res={res}", flush=True)
    s = settings(B, res, max_iter_solve=10)
    st = random_state(s, seed=3)
    p, r = st[B.FIELD_P], st[B.FIELD_RHS]
    if kind == "tiny":
        st[B.FIELD_P], st[B.FIELD_RHS] = p * np.float32(1e-38), r * np.float32(3e-38)
    elif kind == "negzero":
        st[B.FIELD_P], st[B.FIELD_RHS] = np.full_like(p, -0.0), np.full_like(r, -0.0)
        st[B.FIELD_RHS][3, 5, 7] = np.float32(1e-3)
    elif kind == "decay":
        st[B.FIELD_P], st[B.FIELD_RHS] = np.zeros_like(p), np.zeros_like(r)
        st[B.FIELD_RHS][1, 20, 21] = np.float32(1e-30)
    else:
        st[B.FIELD_P][4, 9, 11] = np.float32(np.inf)
    g, o = pair(s, st)
    for x in (g, o):
        x.run_stage(B.STAGE_PRESSURE, 0.0, 1.0 / 24.0)
    compare(f"tile sweeps {kind}", g.field(B.FIELD_P), o.field(B.FIELD_P))


@pytest.mark.parametrize("sizes", [((32, 24, 20), (16, 40, 9)), ((96, 88, 12), (130, 66, 7)),
                                   ((162, 133, 8), (34, 36, 16)), ((200, 98, 6), (162, 133, 5)),
                                   ((162, 133, 8), (162, 133, 5), (34, 36, 16)), ((274, 258, 5), (34, 36, 30))],
                         ids=["small", "middle", "16x8", "16x12", "16x16", "over-256-tiles"])
def test_batch_tile_sweeps_equal_single_scenes(sizes):
    """Scenes of unlike sizes share a tile in the batch and each get what
    they get alone; the variant can be set by its number."""
    print(f"[tiles-batch] {sizes}", flush=True)
    sets = [settings(B, r, max_iter_solve=30, residual_tol=1e-6, residual_check_every=10, buoyancy=1.0, gravity=-9.8)
            for r in sizes]
    b = B.Batch(sets)
    assert b.stats().variant == 2000
    b.set_variant(2000)
    states = [random_state(s, seed=q, vel_scale=0.5) for q, s in enumerate(sets)]
    single = [B.Solver(s) for s in sets]
    for q, st in enumerate(states):
        for w, a in st.items():
            b.scenes[q].set_field(w, a)
            single[q].set_field(w, a)
    for _ in range(2):
        b.step(0.0)
        for g in single:
            g.step(0.0)
    for q, g in enumerate(single):
        for w in (B.FIELD_T, B.FIELD_U, B.FIELD_V, B.FIELD_W, B.FIELD_P):
            compare(f"scene {q} field {w}", b.scenes[q].field(w), g.field(w))
