"""A process whose first call of the producers is recorded into a graph: the pinned block of the totals (mstf_landing_take) is not
there yet."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import torch
from mustafar_amd import ops
g = torch.Generator(device="cuda").manual_seed(1)
k, v = (torch.randn((12, 1024, 128), generator=g, device="cuda", dtype=torch.float16) for _ in range(2))
ws = ops.Workspace("cuda", 1 << 22)
torch.cuda.synchronize()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    c = ops.compress_kv(k, v, 89, 10, ws=ws)
print("recorded", flush=True)
for _ in range(3):
    for t in c[0].bmp, c[0].idx, c[0].nz, c[1].bmp, c[1].idx, c[1].nz:
        t.zero_()
    graph.replay()
    want = ops.compress_kv(k, v, 89, 10, ws=ws)
    assert want[0]._landing is not None and want[0].used_halfs() > 0     # landings are there for the calls behind it
    for a, b in zip(c, want):
        assert all(torch.equal(x, y) for x, y in ((a.bmp, b.bmp), (a.idx, b.idx), (a.nz_off, b.nz_off), (a.packed(), b.packed())))
print("replayed", flush=True)
"""


def test_the_first_call_is_recorded():
    r = subprocess.run([sys.executable, "-u", "-c", CHILD], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0 and "replayed" in r.stdout, r.stdout[-2000:]
