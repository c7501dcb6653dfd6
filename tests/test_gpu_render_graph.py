"""Renders by the deterministic integrators recorded into a HIP graph: a
replay uses nothing of the context that other calls clear, overwrite or move.
Bar: every replay's film has the bits of the plain render."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from muon_amd import Context, DeviceScene, HostScene, scenes  # noqa: E402
from muon_amd import _lib  # noqa: E402
from muon_amd.renderer import render_device  # noqa: E402


NORMALS, RAYTRACER, PATHTRACER = 0, 3, 5  # MUONX_INTEGRATOR_*


def _scene(ctx, integrator, w, h, spp):
    hs = HostScene.from_text(scenes.cornell_text(w, h, spp, 3) + "directional_light 0.2 0.3 1 0.5 0.6 0.7\n")
    p = hs.params
    p.integrator = integrator
    return DeviceScene(ctx, hs), p


def _render(ds, p, acc, stream):
    _lib.check(_lib.lib.muonx_render(ds.h, C.byref(p), acc.data_ptr(), None, stream))


@pytest.mark.parametrize("integrator", [NORMALS, RAYTRACER], ids=["normals", "raytracer"])
@pytest.mark.parametrize("w,h,spp", [(9, 7, 1), (121, 67, 3), (1303, 1301, 2)], ids=["small", "samples", "claims"])
def test_captured_render_replays(integrator, w, h, spp):
    """The largest image has more samples than its wavefronts take without
    claim counters (1,572,864 on 256 CUs); between replays another render
    grows the sample buffer and clears the counters."""
    ctx = Context(0)
    ds, p = _scene(ctx, integrator, w, h, spp)
    other, po = _scene(ctx, NORMALS, 640, 480, 1)
    want, _ = render_device(ds, p)
    want = want.clone()
    acc = torch.empty((h, w, 3), device="cuda:0")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        _render(ds, p, acc, torch.cuda.current_stream().cuda_stream)
    for k in range(4):
        acc.fill_(float(k) - 7.0)
        po.spp = 2 + 4 * k
        render_device(other, po)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(acc, want), k
    again, _ = render_device(ds, p)  # and the context renders on as before
    assert torch.equal(again, want)


def test_captured_path_tracer_is_refused():
    """Its loop runs on the host. The context renders on after the refusal, to the same bits."""
    ctx = Context(0)
    ds, p = _scene(ctx, PATHTRACER, 64, 48, 2)
    want, _ = render_device(ds, p)
    want = want.clone()
    acc = torch.zeros_like(want)
    marker = torch.zeros(1, device="cuda:0")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        marker.add_(1.0)
        rc = _lib.lib.muonx_render(ds.h, C.byref(p), acc.data_ptr(), None, torch.cuda.current_stream().cuda_stream)
    assert rc == -5 and b"captured" in _lib.lib.muonx_last_error()
    g.replay()
    torch.cuda.synchronize()
    assert marker.item() == 1.0 and not acc.any()
    again, _ = render_device(ds, p)
    assert torch.equal(again, want)
