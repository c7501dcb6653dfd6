"""Exact queries of more rays than their wavefronts take without claim counters
(256 chunks' rays for each of 24 wavefronts per CU: 1,572,864 on 256 CUs), plain
and without allocation. Bar: ids, distance bits and any-hit flags equal the
oracle's, twice in a row, so that counters left as they were would show."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from muon_amd import Context, DeviceScene, HostScene, scenes  # noqa: E402


@pytest.fixture(scope="module")
def batch(oracle):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n = cus * 12 * 2 * 64 * 4 + 27_139  # blocks per CU, wavefronts per block, rays per chunk, chunks
    text = scenes.icosphere_text(64, 64, 1, 2, level=3)
    o, d = scenes.microbench_rays(n, (-0.5, 0.1, -0.5), (0.5, 1.1, 0.5), seed=12)
    tmax = np.random.default_rng(12).uniform(0.05, 1.5, n).astype(np.float32)
    orc = oracle.load_text(text)
    prim, t, _, _, _ = orc.intersect(o, d)
    occ, _ = orc.occluded(o, d, tmax)
    ds = DeviceScene(Context(0), HostScene.from_text(text))
    return ds, [torch.from_numpy(x).cuda() for x in (o, d, tmax)], prim, t, occ != 0


@pytest.mark.parametrize("noalloc", [False, True], ids=["plain", "noalloc"])
def test_claimed_chunks(batch, noalloc):
    ds, (o, d, tmax), want_prim, want_t, want_occ = batch
    hit = want_prim >= 0
    assert hit.mean() > 0.5 and 0.1 < want_occ.mean() < 0.9
    for rep in range(2):
        prim = torch.full((o.shape[0],), -9, dtype=torch.int32, device="cuda:0")
        occ = torch.full((o.shape[0],), 9, dtype=torch.uint8, device="cuda:0")
        _, t = ds.query(o, d, None, False, True, prim=prim, noalloc=noalloc)
        ds.query(o, d, tmax, True, True, occ=occ, noalloc=noalloc)
        torch.cuda.synchronize()
        assert np.array_equal(prim.cpu().numpy(), want_prim), rep
        assert np.array_equal(t.cpu().numpy()[hit].view(np.uint32), want_t[hit].view(np.uint32)), rep
        assert np.array_equal(occ.cpu().numpy(), want_occ.astype(np.uint8)), rep
