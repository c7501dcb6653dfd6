"""Batches past 2^32 / 3 rays, whose coordinates need more than 32-bit indices:
the same million rays over and over. Bar: every repetition has the bits of the
million alone, the ragged end included."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from muon_amd import Context, DeviceScene, HostScene, scenes  # noqa: E402

BLOCK = 1_000_003
REPS = 1500  # 1,500,004,500 rays and a part of a block: past 2^32 / 3 = 1,431,655,765
END = 12_345


@pytest.fixture(scope="module")
def rays():
    if torch.cuda.get_device_properties(0).total_memory < 100 << 30:
        pytest.skip("needs 60 GB of device memory")
    o, d = scenes.microbench_rays(BLOCK, (-0.8, 0.2, -0.8), (0.8, 1.8, 0.8), seed=9)
    o, d = torch.from_numpy(o).cuda(), torch.from_numpy(d).cuda()
    n = BLOCK * REPS + END
    big = []
    for x in (o, d):
        y = torch.empty((n, 3), device="cuda:0")
        y[:BLOCK * REPS].view(REPS, BLOCK, 3).copy_(x.expand(REPS, BLOCK, 3))
        y[BLOCK * REPS:].copy_(x[:END])
        big.append(y)
    yield o, d, big[0], big[1]
    del big, y
    torch.cuda.empty_cache()


@pytest.mark.parametrize("exact,fetch", [(False, 16), (False, 0), (True, 16)], ids=["fast", "gridstride", "exact"])
def test_past_32_bit_coordinates(rays, exact, fetch):
    o, d, bo, bd = rays
    ctx = Context(0)
    ctx.set_tuning(ray_fetch=fetch)
    ds = DeviceScene(ctx, HostScene.from_text(scenes.cornell_text(64, 64, 1, 2)))
    want, _ = ds.intersect_closest(o, d, exact=exact)
    prim = torch.full((bo.shape[0],), -9, dtype=torch.int32, device="cuda:0")
    t = torch.empty(0, device="cuda:0")  # no distances
    got = ds.query(bo, bd, None, False, exact, prim=prim, t=t)[0]
    torch.cuda.synchronize()
    assert len(torch.unique(want)) > 5
    rows = got[:BLOCK * REPS].view(REPS, BLOCK)
    for k in range(0, REPS, 100):
        assert torch.equal(rows[k:k + 100], want.expand(min(100, REPS - k), BLOCK)), k
    assert torch.equal(got[BLOCK * REPS:], want[:END])
    del prim, got, rows
    torch.cuda.empty_cache()
