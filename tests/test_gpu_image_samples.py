"""The deterministic integrators' images where their samples are split over
launches: every sample of an image that sees one albedo everywhere adds the
same colour, so the film is the float32 sum of that colour in order.
Bar: bit-exact films, one primary ray per sample."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from muon_amd import Context, DeviceScene, HostScene  # noqa: E402
from muon_amd.renderer import render_device  # noqa: E402

ROOM = """film_size {w} {h}
integrator albedo
pixel_samples {spp}
camera 0 0 0.3  0 0 -1  0 1 0  40
ambient 0 0 0
diffuse 0.1 0.37 0.7
specular 0.2 0.0 0.11
sphere 0 0 0 5
"""


@pytest.mark.parametrize("w,h,spp", [(9, 7, 1), (9, 7, 2), (70, 33, 11), (512, 513, 25), (2001, 1500, 2)],
                         ids=["one", "two_buffered", "buffered", "two_batches", "unbuffered"])
def test_samples_add_in_order(w, h, spp):
    """Samples in one buffer, in two batches of it, and added directly where
    the buffer holds no two of them."""
    ctx = Context(0)
    hs = HostScene.from_text(ROOM.format(w=w, h=h, spp=spp))
    acc, st = render_device(DeviceScene(ctx, hs), hs.params)
    torch.cuda.synchronize()
    colour = np.array([0.1, 0.37, 0.7], np.float32) + np.array([0.2, 0.0, 0.11], np.float32)
    want = np.zeros(3, np.float32)
    for _ in range(spp):
        want = want + colour
    got = acc.cpu().numpy()
    assert got.shape == (h, w, 3) and np.array_equal(got, np.broadcast_to(want, got.shape))
    assert st.primary_rays == w * h * spp
