"""Every place of the traversal stacks past their LDS part: a ring of 16 with its
older entries in HBM, of 8 with them in private memory, and the whole stack in
LDS, with per-lane ray fetch and without it, in queries and in the engine.

The trees are chains: every internal node has a leaf beside the rest of the
tree, and the boxes of the overlapping spheres all hold the rays' origins, so a
walk that goes down the chain first keeps an entry per level. Bar: ids, distance
bits and films equal those of the whole stack in LDS, and the distances those of
the exact walk in the host's own tree (no two spheres meet a ray at the same
distance but by chance: ids differ on at most one ray in a thousand)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from muon_amd import Context, DeviceScene, HostScene, scenes  # noqa: E402
from muon_amd.renderer import render_device  # noqa: E402


def _text(n, w=40, h=30):
    lines = []
    scenes.cornell_header(lines, w, h, 2, 4)
    lines.append("diffuse 0.5 0.6 0.7")
    rng = np.random.default_rng(n)
    for c, r in zip(rng.uniform(-0.05, 0.05, (n, 3)), rng.uniform(0.5, 0.9, n)):
        lines.append("sphere %r %r %r %r" % (float(c[0]), float(c[1] + 1.0), float(c[2]), float(r)))
    return "\n".join(lines) + "\n"


def _prim_boxes(hs):
    """World boxes of the primitives, from the leaves of the host's tree (one primitive each or their leaf's)."""
    a = hs.arrays()
    box = np.zeros((hs.desc.num_prims, 6), np.float32)
    for b, s, c in zip(a["node_bounds"], a["node_start"], a["node_count"]):
        for k in a["leaf_prims"][s:s + c]:
            box[k] = b
    return box


def _chain(ctx, hs, depth):
    """The scene under a chain of `depth` levels."""
    n = hs.desc.num_prims
    box = _prim_boxes(hs)
    parts = np.array_split(np.arange(n, dtype=np.int32), depth)
    assert all(len(p) for p in parts)
    union = lambda ids: np.concatenate([box[ids, :3].min(axis=0), box[ids, 3:].max(axis=0)])
    bounds, left, right, axis, start, count = [], [], [], [], [], []
    for k in range(depth - 1):  # node 2k: internal, 2k + 1: its leaf, 2k + 2: the rest
        bounds += [union(np.arange(parts[k][0], n)), union(parts[k])]
        # whichever direction a ray goes along the axis, half of the levels send it down the chain first
        a, b = (2 * k + 2, 2 * k + 1) if k % 7 < 6 else (2 * k + 1, 2 * k + 2)
        left += [a, -1]
        right += [b, -1]
        axis += [0, 0]
        start += [0, int(parts[k][0])]
        count += [0, len(parts[k])]
    bounds.append(union(parts[-1]))
    left.append(-1)
    right.append(-1)
    axis.append(0)
    start.append(int(parts[-1][0]))
    count.append(len(parts[-1]))
    i32 = lambda x: np.array(x, np.int32)
    ds = DeviceScene.from_arrays(ctx, hs, num_nodes=len(bounds), node_bounds=np.array(bounds, np.float32), node_left=i32(left),
                                 node_right=i32(right), node_axis=i32(axis), node_start=i32(start), node_count=i32(count),
                                 leaf_prims=np.arange(n, dtype=np.int32))
    assert ds.info()["bvh_depth"] == depth
    return ds


def _rays(n):
    rng = np.random.default_rng(5)
    o = np.array([0, 1, 0], np.float32) + rng.uniform(-0.2, 0.2, (n, 3)).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return torch.from_numpy(o).cuda(), torch.from_numpy(d.astype(np.float32)).cuda()


# past the ring of 16; the private stack's last depth and the first past it; the deepest that LDS alone holds
@pytest.mark.parametrize("depth", [24, 72, 73, 96])
@pytest.mark.parametrize("width,bits", [(2, 32), (4, 32), (4, 8)], ids=["binary", "wide", "quantized"])
def test_stack_places_agree(depth, width, bits):
    ctx = Context(0)
    hs = HostScene.from_text(_text(100))
    ds = _chain(ctx, hs, depth)
    n = 20_011
    o, d = _rays(n)
    tmax = torch.full((n,), 0.6, device="cuda:0")
    plain_prim, plain_t = DeviceScene(ctx, hs).intersect_closest(o, d, exact=True)
    want = None
    for stack in (0, 8, 16):
        for fetch in (16, 0):
            ctx.set_tuning(stack_entries=stack, ray_fetch=fetch, bvh_width=width, node_bits=bits)
            for noalloc in (False, True):
                prim, t = ds.query(o, d, None, False, noalloc=noalloc)
                occ = ds.query(o, d, tmax, True, noalloc=noalloc)
                torch.cuda.synchronize()
                if want is None:
                    want = prim.clone(), t.clone(), occ.clone()
                    assert torch.equal(t, plain_t) and (prim != plain_prim).sum() <= n // 1000
                    assert torch.equal(occ != 0, (plain_prim >= 0) & (plain_t < 0.6))
                assert torch.equal(prim, want[0]) and torch.equal(t, want[1]) and torch.equal(occ, want[2]), (stack, fetch, noalloc)


@pytest.mark.parametrize("depth", [24, 73, 96])
def test_engine_stack_places_agree(depth):
    ctx = Context(0)
    hs = HostScene.from_text(_text(100))
    ds = _chain(ctx, hs, depth)
    want = None
    for stack in (0, 8, 16):
        for fetch in (16, 0):
            ctx.set_tuning(stack_entries=stack, ray_fetch=fetch, bvh_width=2, node_bits=32, path_budget_mb=64)
            film, st = render_device(ds, hs.params)
            torch.cuda.synchronize()
            if want is None:
                want = film.clone()
                assert st.shadow_rays > 0 and st.secondary_rays > 0 and want.max() > 0
            assert torch.equal(film, want), (stack, fetch)
