"""Device memory of the pair track's weights: a block's triangle attention, triangle
multiplication and transition hold the binary16 forms that their kernels read and no
others."""
import numpy as np
import pytest
import torch

from bindcraft2_amd import ops, params as bparams
from tests.helpers import weights_dir

pytestmark = pytest.mark.gpu
BLOCKS = 24


def test_weight_forms(cuda):
    names = ["triangle_attention_starting_node", "triangle_multiplication_outgoing", "pair_transition"]
    rng, prm = np.random.default_rng(0), {}
    for b in range(BLOCKS):
        prm.update(bparams.init_block_params(b, rng, modules=names))
    wdir = weights_dir(prm, "forms")
    x, m = torch.randn(32, 32, 128, device=cuda), torch.ones(32, 32, device=cuda)

    def block(b):
        p = f"param/block{b}/"
        ops.TriangleAttention(wdir, p + names[0] + "/", False).forward(x, m)
        ops.TriangleMultiplication(wdir, p + names[1] + "/", True).forward(x, m)
        ops.Transition(wdir, p + names[2] + "/", 128).forward(x)

    block(0)  # and every scratch buffer
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    for b in range(1, BLOCKS):
        block(b)
    torch.cuda.synchronize()
    used = free - torch.cuda.mem_get_info()[0]
    # attention: q|k|v|g forward, dX twice, out both ways; multiplication: projections
    # forward, the tail's 4C and 5C, out both ways; transition: both ways of both
    matrices = (3 * 4 + 2) + (5 + 4 + 5 + 2) + 4 * 4
    need = (BLOCKS - 1) * matrices * 128 * 128 * 2
    print(f"{used / 2**20:.1f} MB of weights, {need / 2**20:.1f} MB read", flush=True)
    assert used <= 1.1 * need + (4 << 20)  # biases, norms; the allocator's granules
