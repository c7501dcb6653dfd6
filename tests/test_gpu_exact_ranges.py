"""Exact-mode queries outside the range of the reciprocal quotients
(exact_div.h): rays with tiny direction components or origins, and a scene
with a tiny plane, take the division path lane by lane beside ordinary rays.
Bar: ids, distance bits and any-hit flags equal the oracle's."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from muon_amd import Context, DeviceScene, HostScene, scenes  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    assert torch.cuda.is_available(), "GPU tests need a ROCm device"
    return Context(0)


def _rays(kind, n=1500):
    rng = np.random.default_rng(11)
    o = rng.uniform(-0.9, 0.9, (n, 3)).astype(np.float32)
    o[:, 1] += 1.0
    d = rng.normal(size=(n, 3)).astype(np.float32)
    odd = rng.random(n) < 0.5
    axis = rng.integers(0, 3, n)
    rows = np.nonzero(odd)[0]
    if kind == "tiny_direction":
        d[rows, axis[rows]] = np.float32(1e-24) * rng.choice([-1, 1], len(rows)).astype(np.float32)
    elif kind == "tiny_origin":
        o[rows, axis[rows]] = np.float32(3e-31)
    elif kind == "zero_direction":
        d[rows, axis[rows]] = rng.choice(np.array([0.0, -0.0], np.float32), len(rows))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return o, d.astype(np.float32)


@pytest.mark.parametrize("tiny_plane", [False, True], ids=["planes", "tiny_plane"])
@pytest.mark.parametrize("kind", ["ordinary", "tiny_direction", "tiny_origin", "zero_direction"])
def test_exact_mode_everywhere(ctx, oracle, kind, tiny_plane):
    text = scenes.cornell_text(64, 64, 1, 2)
    if tiny_plane:  # one plane of the tree at 1e-27
        text += "start_mesh\nvertex 1e-27 0.2 0\nvertex 0.5 0.2 0\nvertex 0.5 0.9 0.3\ntri 0 1 2\nend_mesh\n"
    ds = DeviceScene(ctx, HostScene.from_text(text))
    orc = oracle.load_text(text)
    o, d = _rays(kind)
    pr, tr, _, _, _ = orc.intersect(o, d)
    to, td = torch.from_numpy(o).cuda(), torch.from_numpy(d).cuda()
    prim, t = ds.intersect_closest(to, td, exact=True)
    tm = np.full(len(o), 0.8, np.float32)
    occ = ds.intersect_any(to, td, torch.from_numpy(tm).cuda(), exact=True)
    torch.cuda.synchronize()
    assert np.array_equal(prim.cpu().numpy(), pr)
    hit = pr >= 0
    assert hit.any() and np.array_equal(t.cpu().numpy()[hit].view(np.uint32), tr[hit].view(np.uint32))
    oref, _ = orc.occluded(o, d, tm)
    assert np.array_equal(occ.cpu().numpy() != 0, oref != 0)


@pytest.mark.parametrize("n", [1, 2, 129, 4097, 131073, 500009])
def test_exact_mode_batch_sizes(ctx, oracle, n):
    """From two rays to a wavefront, over all first chunks filled, to chunks
    claimed from the counter (past 393,216 rays on 256 CUs)."""
    text = scenes.icosphere_text(64, 64, 1, 2, level=3)
    ds = DeviceScene(ctx, HostScene.from_text(text))
    orc = oracle.load_text(text)
    o, d = scenes.microbench_rays(n, (-0.5, 0.1, -0.5), (0.5, 1.1, 0.5), seed=n)
    pr, tr, _, _, _ = orc.intersect(o, d)
    prim, t = ds.intersect_closest(torch.from_numpy(o).cuda(), torch.from_numpy(d).cuda(), exact=True)
    torch.cuda.synchronize()
    assert np.array_equal(prim.cpu().numpy(), pr)
    hit = pr >= 0
    assert np.array_equal(t.cpu().numpy()[hit].view(np.uint32), tr[hit].view(np.uint32))
