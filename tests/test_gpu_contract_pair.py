"""Triangle multiplication's two backward contractions in one launch: both
directions (the second product with both operands k-major or both K-contiguous)
at every channel plane of the launch, 32 to 256, and the first size beyond it,
against the fp64 oracle at the module's bars."""
import numpy as np
import pytest
import torch

from bindcraft2_amd import ops, params as bparams
from oracle import af2
from tests.helpers import assert_grad, random_mask, weights_dir

pytestmark = pytest.mark.gpu
D = torch.float64


@pytest.mark.parametrize("outgoing", [True, False])
@pytest.mark.parametrize("n", [32, 64, 96, 128, 160, 192, 224, 256, 288])
def test_backward(cuda, n, outgoing):
    print(f"n={n} outgoing={outgoing}", flush=True)
    name = "triangle_multiplication_" + ("outgoing" if outgoing else "incoming")
    rng = np.random.default_rng(2 * n + outgoing)
    prm = bparams.init_template_block_params(0, rng, gates="random", ln="random")
    prefix = f"param/block0/{name}/"
    mod = ops.TriangleMultiplication(weights_dir(prm, f"cp_{n}_{outgoing}"), prefix, outgoing, c=64,
                                     hidden=64)
    x = torch.as_tensor(rng.standard_normal((n, n, 64)).astype(np.float32), device=cuda)
    dout = torch.as_tensor(rng.standard_normal((n, n, 64)).astype(np.float32), device=cuda)
    mask = torch.as_tensor(random_mask(n, 0.1, rng)[0], device=cuda)
    _, save = mod.forward(x, mask, None)
    din = mod.backward(x, mask, None, save, dout)
    P = af2.Params(prm, prefix)
    p = lambda v: P(v).to(cuda)
    p.sub = lambda s: (lambda v: P.sub(s)(v).to(cuda))
    xd = x.double().requires_grad_(True)
    ref = af2.triangle_multiplication(xd, mask.double(), p, outgoing)
    (g,) = torch.autograd.grad(ref, xd, dout.double())
    print(" ", assert_grad((din - dout).cpu().double(), g.cpu(), 0.99999, "dpair"))
