"""muonx_intersect_noalloc takes no device memory, from the runtime neither: the
free memory around the first query of a fresh process. A stack of even eight
entries per lane in private memory would be set aside for every resident
wavefront at the first dispatch: 8 * 8 B * 64 lanes * 32 wavefronts * 256 CUs =
32 MiB. Bar: less than half of that."""
import os
import subprocess
import sys

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SCRIPT = """
import sys
import torch
from muon_amd import Context, DeviceScene, HostScene, scenes
exact, any_hit, width, stack, fetch = (int(a) for a in sys.argv[1:])
ctx = Context(0)
ctx.set_tuning(bvh_width=width, node_bits=8 if width == 4 else 32, stack_entries=stack, ray_fetch=fetch)
ds = DeviceScene(ctx, HostScene.from_text(scenes.icosphere_text(64, 64, 1, 2, level=5)))
n = 1 << 20
o, d = scenes.microbench_rays(n, (-0.5, 0.1, -0.5), (0.5, 1.1, 0.5), seed=1)
o, d = torch.from_numpy(o).cuda(), torch.from_numpy(d).cuda()
out = dict(prim=torch.empty(n, dtype=torch.int32, device="cuda"), t=torch.empty(n, device="cuda"),
           occ=torch.empty(n, dtype=torch.uint8, device="cuda"))
torch.cuda.synchronize()
before = torch.cuda.mem_get_info()[0]
ds.query(o, d, None, bool(any_hit), bool(exact), noalloc=True, **out)
torch.cuda.synchronize()
print("taken", before - torch.cuda.mem_get_info()[0])
"""


# exact, any_hit, bvh_width, stack_entries, ray_fetch
@pytest.mark.parametrize("form", [(0, 0, 4, 8, 16), (0, 1, 4, 8, 16), (0, 0, 2, 8, 0), (0, 0, 4, 16, 16), (1, 0, 4, 8, 16),
                                  (1, 1, 4, 8, 16)],
                         ids=["default", "default-any", "binary-gridstride", "ring16", "exact", "exact-any"])
def test_first_query_takes_no_memory(form):
    r = subprocess.run([sys.executable, "-c", SCRIPT, *map(str, form)], cwd=ROOT, capture_output=True, text=True,
                       timeout=100, env={**os.environ, "PYTHONPATH": ROOT})
    assert r.returncode == 0, r.stdout + r.stderr
    taken = int(r.stdout.split("taken")[1])
    assert taken < 16 << 20
