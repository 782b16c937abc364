"""wh_modwt_inv_adj needs no library scratch: as the first library call of a
process it can be captured into a graph (an arena that grew there would call
hipMalloc), and replays give the adjoint's values, zeros in the S slots that
carried the level hand-off included.  In a process of its own: other tests'
calls have grown this one's arenas."""
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

PROGRAM = """
import ctypes as C, torch
from wavecuda_amd import _lib as W
n, count, J, f = {n}, {count}, {J}, W.{filt}
dt, code = torch.{dtype}, W.WH_{code}
p = lambda t: C.c_void_p(t.data_ptr())
g = torch.Generator(device="cuda").manual_seed(3)
x = torch.randn(count, n, dtype=dt, device="cuda", generator=g)
w = torch.full((count, 2 * n * J), 7.0, dtype=dt, device="cuda")
torch.cuda.synchronize()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    W.check(W.lib().wh_modwt_inv_adj(p(x), p(w), n, count, J, f, code, s), "captured call")
want = torch.empty_like(w)
for seed in range(3):
    x.copy_(torch.randn(count, n, dtype=dt, device="cuda", generator=g))
    graph.replay()
    W.check(W.lib().wh_modwt_fwd_many(p(x), p(want), n, count, J, f, code,
                                      C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    v = want.view(count, J, 2, n)
    v *= torch.tensor([2.0 ** -l for l in range(1, J + 1)], dtype=dt, device="cuda").view(J, 1, 1)
    v[:, : J - 1, 0] = 0
    torch.cuda.synchronize()
    assert torch.equal(w, want), seed
print("equal")
"""


@pytest.mark.parametrize("case", [
    dict(n=1 << 14, count=4, J=8, filt="LA8", dtype="float64", code="F64"),
    dict(n=1 << 13, count=8, J=12, filt="HAAR", dtype="float32", code="F32")])
def test_captured_as_first_call(case):
    root = Path(__file__).resolve().parents[1]
    r = subprocess.run([sys.executable, "-c", PROGRAM.format(**case)], cwd=root, text=True,
                       capture_output=True, timeout=100)
    assert r.returncode == 0 and "equal" in r.stdout, r.stderr[-2000:]
