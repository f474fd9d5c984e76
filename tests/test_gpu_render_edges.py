"""GPU tests of the renderer where its work is cut: bricks of empty space
passed over (of 4, 8 and 16 cells, none clear, all clear, a NaN in one), the
samples taken at a time for 0, 1, 4 and 10 lights, grids of 4 and 6 cells
(scatter volumes of one texel), and the tiles that a frame's pixels and lights
choose, at their edges. The oracle's image, bit for bit."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(__file__))
from test_gpu_render import B, O, compare, render_settings, settings  # noqa: E402

pytestmark = pytest.mark.gpu


def blob(res, seed, size=None):
    """A small ball in an empty grid, its edge falling through the cutoff."""
    W, H, D = res
    rng = np.random.default_rng(seed)
    z, y, x = np.meshgrid(np.arange(D), np.arange(H), np.arange(W), indexing="ij")
    r2 = ((x - 0.35 * W) ** 2 + (y - 0.55 * H) ** 2 + (z - 0.6 * D) ** 2) / (0.2 * (size or min(res))) ** 2
    T = np.where(r2 < 1.5, 2.0 * np.exp(-4.0 * r2) * (0.5 + rng.random((D, H, W))), 0.0)
    return T.astype(np.float32)


CASES = {
    "brick4": ((32, 40, 36), 2, {}),
    "brick8": ((160, 128, 128), 1, {}),
    "brick16": ((1024, 1032, 9), 1, {"ball": 400}),
    "no-cutoff": ((16, 12, 20), 2, {"cutoff": 0.0}),
    "nan": ((24, 24, 24), 2, {"nan": True}),
    "empty": ((24, 24, 24), 3, {"empty": True}),
    "no-light": ((32, 32, 32), 0, {}),
    "4-lights": ((24, 20, 28), 4, {}),
    "10-lights": ((24, 20, 28), 10, {"gain": 0.0}),
    "smallest": ((4, 4, 4), 2, {}),
    "one-texel": ((6, 7, 5), 2, {"gain": 0.0}),
    "thin-shadow": ((32, 32, 32), 2, {"shadow_density_scale": 0.25, "emission_scale": 0.0}),
}


def add_lights(r, lights):
    rng = np.random.default_rng(2)
    for l in range(2, lights):
        d = rng.standard_normal(3)
        d /= np.linalg.norm(d)
        for a in range(3):
            r.light_dir[l][a], r.light_color[l][a] = d[a], 0.5
        r.light_intensity[l] = 0.3
    r.light_count = lights


@pytest.mark.parametrize("name", list(CASES))
def test_render_edges(name):
    res, lights, opt = CASES[name]
    print(f"[render] {name} {res} lights {lights}", flush=True)
    s = settings(B, res)
    g = B.Solver(s)
    T = blob(res, 11, opt.get("ball"))
    if opt.get("nan"):
        T[3, 4, 5] = np.nan
    if opt.get("empty"):
        T[:] = 0.0
    g.set_field(B.FIELD_T, T)
    r = render_settings(64, 48, float(s.dx))
    for k in ("cutoff", "gain", "shadow_density_scale", "emission_scale"):
        if k in opt:
            setattr(r, k, opt[k])
    add_lights(r, lights)
    want = O.render(T, float(s.dx), list(s.domain_min), list(s.domain_max), r)
    compare(f"render {name}", g.render(r), want)
    compare(f"render noalloc {name}", g.render_noalloc(r), want)


# width, height, lights: 4x4 tiles from 200000 pixels on (30000 without
# lights), a thread per pixel from 200000 and 500000 more per light
FRAMES = [(200, 144, 0), (208, 152, 0), (624, 320, 0), (632, 320, 0), (624, 320, 2), (632, 320, 1), (632, 320, 10),
          (992, 704, 1), (1000, 704, 1)]


@pytest.mark.parametrize("w,h,lights", FRAMES, ids=lambda v: str(v))
@pytest.mark.parametrize("res", [(16, 12, 20), (18, 9, 7)], ids=["pow2dx", "18x9x7"])
def test_render_tiles(res, w, h, lights):
    print(f"[render-tiles] {res} {w}x{h} lights {lights}", flush=True)
    s = settings(B, res)
    g = B.Solver(s)
    T = blob(res, 5)
    T[2, 1, 3] = np.nan if lights == 2 else 0.5
    g.set_field(B.FIELD_T, T)
    r = render_settings(w, h, float(s.dx))
    add_lights(r, lights)
    want = O.render(T, float(s.dx), list(s.domain_min), list(s.domain_max), r)
    compare(f"render {w}x{h}", g.render(r), want)
