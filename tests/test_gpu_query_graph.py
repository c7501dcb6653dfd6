"""Ray queries recorded into a HIP graph. Bar: every replay's results have the
bits of the plain call, with other queries of the context run between the
replays; sizes on both sides of what the wavefronts take without claim
counters (1,572,864 exact and 2,097,152 fast rays on 256 CUs)."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from muon_amd import Context, DeviceScene, HostScene, scenes  # noqa: E402


@pytest.fixture(scope="module")
def scene():
    ctx = Context(0)
    ds = DeviceScene(ctx, HostScene.from_text(scenes.icosphere_text(64, 64, 1, 2, level=3)))
    n = 2_500_009
    o, d = scenes.microbench_rays(n, (-0.5, 0.1, -0.5), (0.5, 1.1, 0.5), seed=6)
    return ctx, ds, torch.from_numpy(o).cuda(), torch.from_numpy(d).cuda()


@pytest.mark.parametrize("noalloc", [False, True], ids=["plain", "noalloc"])
@pytest.mark.parametrize("any_hit", [False, True], ids=["closest", "any"])
@pytest.mark.parametrize("exact", [True, False], ids=["exact", "fast"])
@pytest.mark.parametrize("n", [1, 1003, 2_500_009])
def test_captured_query_replays(scene, n, exact, any_hit, noalloc):
    ctx, ds, o, d = scene
    o, d = o[:n], d[:n]
    tmax = torch.full((n,), 0.7, device="cuda:0") if any_hit else None
    out = lambda: dict(prim=torch.empty(n, dtype=torch.int32, device="cuda:0"),
                       t=torch.empty(n, device="cuda:0"), occ=torch.empty(n, dtype=torch.uint8, device="cuda:0"))
    want, got = out(), out()
    ds.query(o, d, tmax, any_hit, exact, noalloc=noalloc, **want)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ds.query(o, d, tmax, any_hit, exact, noalloc=noalloc, **got)
    keys = ("occ",) if any_hit else ("prim", "t")
    for k in range(4):
        for name in keys:
            got[name].fill_(5)
        other = out()
        ds.query(o, d, tmax, any_hit, exact, noalloc=noalloc, **other)  # leaves its counts in the counters
        g.replay()
        torch.cuda.synchronize()
        for name in keys:
            assert torch.equal(got[name], want[name]), (k, name)
            assert torch.equal(other[name], want[name]), (k, name)
