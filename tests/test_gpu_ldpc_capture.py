"""A program that has decoded once may capture decoder calls of other batch
sizes into a graph: one call loads the tables of every kernel that a later one
may take.  In a process of its own, since any handle's creation loads them too."""
import subprocess
import sys
from pathlib import Path

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parents[1]

PROGRAM = """
import sys
import torch
from puschrx import abi, ops
z, k, rows = 384, 22 * 384, 8
gen = torch.Generator(device="cuda")
gen.manual_seed(1)
sizes = [1000, 400, 3]  # beyond two blocks a compute unit, between one and two, below
lam = torch.randint(-3000, 3000, (max(sizes) * 68 * z,), generator=gen, device="cuda").to(torch.int16)
s = torch.cuda.Stream()
call = lambda n: ops.ldpc_decode(lam, n, z, k, 3, rows, abi.LDPC_MODE_FP16, False)
with torch.cuda.stream(s):
    call(sizes[int(sys.argv[1])])
    s.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        got = [call(n) for n in sizes]
    for replay in range(3):
        graph.replay()
        s.synchronize()
        for n, (bits, _, it) in zip(sizes, got):
            want, _, want_it = call(n)
            s.synchronize()
            assert torch.equal(bits, want) and torch.equal(it, want_it), (replay, n)
            bits.zero_()
print("captured")
"""


@pytest.mark.parametrize("first", [0, 1])
def test_capture_after_one_call(first):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    r = subprocess.run([sys.executable, "-c", PROGRAM, str(first)], cwd=ROOT / "ai-ran-npu-kernels_amd",
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "captured" in r.stdout, r.stdout + r.stderr
