"""Scratch of the row kernels' paths: the first triangle attention forward of a
process takes the gated output's buffer and a quarter more to grow into, and
nothing for the normalised rows that stay on chip."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import numpy as np, torch
from bindcraft2_amd import ops, params as bparams
from tests.helpers import weights_dir
name = "triangle_attention_starting_node"
prm = bparams.init_block_params(0, np.random.default_rng(0), modules=[name])
mod = ops.TriangleAttention(weights_dir(prm, "scratch"), f"param/block0/{name}/", False)
def buffers(n):
    x = torch.randn(n, n, 128, device="cuda")
    return (x, torch.ones(n, n, device="cuda"), None, torch.empty_like(x),
            torch.empty(mod.save_bytes(n), dtype=torch.uint8, device="cuda"))
mod.forward(*buffers(32))
big = buffers(448)
torch.cuda.synchronize()
free = torch.cuda.mem_get_info()[0]
mod.forward(*big)
torch.cuda.synchronize()
print("TOOK", free - torch.cuda.mem_get_info()[0])
"""


def test_attention_forward_scratch(cuda):
    r = subprocess.run([sys.executable, "-c", CHILD], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    took = int(r.stdout.split("TOOK")[1])
    og = 448 * 448 * 128 * 2
    print(f"{took / 2**20:.1f} MB, the gated output {og / 2**20:.1f}", flush=True)
    assert took <= 1.25 * og + (4 << 20)
