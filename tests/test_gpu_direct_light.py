"""The direct light of many light records: a diffuse floor under K
directional lights, of which some are blocked by a wall and some lie below
the floor, so every pixel is the sum of the others' color * cos * diffuse / pi.
Bar: float64 sums within the rounding of K + 16 float32 operations at two
rounding steps each, with the same value for both ways to weight the light
(no light has an area)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from muon_amd import Context, DeviceScene, HostScene  # noqa: E402
from muon_amd.renderer import render_device  # noqa: E402

FLOOR = """film_size 37 21
integrator pathtracer
next_event_estimation {nee}
importance_sampling cosine
max_depth 1
pixel_samples 3
camera 0 0 5  0 0 0  0 1 0  20
brdf lambertian
ambient 0 0 0
diffuse 0.4 0.55 0.7
specular 0 0 0
vertex -50 -50 0
vertex 50 -50 0
vertex 50 50 0
vertex -50 50 0
tri 0 1 2
tri 0 2 3
vertex 20 -500 -1
vertex 20 500 -1
vertex 20 500 60
vertex 20 -500 60
tri 4 5 6
tri 4 6 7
"""


def lights(k):
    rng = np.random.default_rng(k)
    kind = np.arange(k) % 3  # 0 lit, 1 blocked by the wall, 2 below the floor
    kind[-1] = 0  # the last record counts
    dirs = np.where(kind[:, None] == 0, [0.1, 0.2, 1.0], np.where(kind[:, None] == 1, [1.0, 0.1, 0.3], [0.3, 0.1, -1.0]))
    dirs = dirs + rng.uniform(-0.05, 0.05, (k, 3))
    dirs = dirs / np.linalg.norm(dirs, axis=1, keepdims=True)
    return dirs.astype(np.float32), rng.uniform(0.1, 1.0, (k, 3)).astype(np.float32), kind


@pytest.mark.parametrize("nee", ["on", "mis"])
@pytest.mark.parametrize("k", [1, 2, 63, 64, 65, 130])
def test_sum_of_lights(k, nee):
    """Up to and past the 64 rays that a path's mask of shadow rays holds."""
    dirs, color, kind = lights(k)
    text = FLOOR.format(nee=nee) + "".join(
        "directional_light %r %r %r %r %r %r\n" % tuple(float(x) for x in (*d, *c)) for d, c in zip(dirs, color))
    ctx = Context(0)
    hs = HostScene.from_text(text)
    acc, st = render_device(DeviceScene(ctx, hs), hs.params)
    torch.cuda.synchronize()
    want = (color.astype(np.float64) * dirs[:, 2:].astype(np.float64))[kind == 0].sum(axis=0) * np.array([0.4, 0.55, 0.7]) / np.pi
    got = acc.cpu().numpy().astype(np.float64) / 3
    assert np.abs(got / want - 1).max() < (k + 16) * 2.0 ** -23 + 2.0 ** -24 / want.min()
    assert st.shadow_rays == 37 * 21 * 3 * int((kind < 2).sum())
