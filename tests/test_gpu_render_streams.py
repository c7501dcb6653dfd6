"""Renders of one context on several streams without stats, which return while
their work runs: the counters and the sample buffer that the deterministic
integrators share go from one to the next in order.
Bar: every film has the bits of the render run alone."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from muon_amd import Context, DeviceScene, HostScene, scenes  # noqa: E402
from muon_amd import _lib  # noqa: E402
from muon_amd.renderer import render_device  # noqa: E402

NORMALS, DEPTH, RAYTRACER, PATHTRACER = 0, 2, 3, 5  # MUONX_INTEGRATOR_*


def _scene(ctx, integrator, w, h, spp, seed):
    text = scenes.icosphere_text(w, h, spp, 3, level=4) + "directional_light 0.2 0.3 1 0.5 0.6 0.7\n"
    hs = HostScene.from_text(text)
    p = hs.params
    p.integrator = integrator
    p.seed = seed
    return DeviceScene(ctx, hs), p


# (integrator, width, height, samples) of the renders, issued to the streams in turn
SETS = {
    # samples in the buffer, claimed chunks (more than 1,572,864 samples), then few samples and a buffer that grows
    "buffered": [(RAYTRACER, 801, 603, 4), (NORMALS, 1001, 600, 3), (DEPTH, 99, 65, 5), (NORMALS, 1003, 700, 5),
                 (RAYTRACER, 640, 480, 2)],
    # films above half of the buffer's limit: samples added directly, counters cleared for each
    "direct": [(NORMALS, 2001, 1500, 2), (RAYTRACER, 2001, 1499, 2), (DEPTH, 1999, 1500, 2)],
    # a path-traced render among them
    "path": [(RAYTRACER, 801, 603, 4), (PATHTRACER, 64, 64, 2), (NORMALS, 1001, 600, 3)],
}


@pytest.mark.parametrize("name", list(SETS))
def test_two_streams(name):
    ctx = Context(0)
    jobs = [_scene(ctx, *spec, seed=3 + k) for k, spec in enumerate(SETS[name])]
    want = []
    for ds, p in jobs:
        acc, _ = render_device(ds, p)
        want.append(acc.clone())
    torch.cuda.synchronize()
    fresh = Context(0)  # its buffers are allocated while other renders run
    jobs = [_scene(fresh, *spec, seed=3 + k) for k, spec in enumerate(SETS[name])]
    films = [torch.full_like(w, -3.0) for w in want]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for rep in range(3):
        for k, (ds, p) in enumerate(jobs):
            s = streams[(rep + k) % 2]
            films[k].record_stream(s)
            _lib.check(_lib.lib.muonx_render(ds.h, C.byref(p), films[k].data_ptr(), None, s.cuda_stream))
    st = _lib.TraceStatsC()  # a render with stats behind them counts its own samples only
    ds, p = jobs[0]
    last = torch.empty_like(want[0])
    _lib.check(_lib.lib.muonx_render(ds.h, C.byref(p), last.data_ptr(), C.byref(st), streams[0].cuda_stream))
    assert st.primary_rays == p.width * p.height * p.spp
    torch.cuda.synchronize()
    assert torch.equal(last, want[0])
    for k in range(len(jobs)):
        assert torch.equal(films[k], want[k]), (name, k)
