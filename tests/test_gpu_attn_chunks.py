"""Triangle attention at the edges of the attention kernels' launch forms: N =
256 (the dK/dV partials over the row's own buffer), whole and partial last
64- and 96-key chunks and idle query waves beyond 256, each with residues whose
rows are fully masked (uniform attention) among partially masked ones, forward
and backward against the fp64 oracle run on the device."""
import numpy as np
import pytest
import torch

from bindcraft2_amd import ops, params as bparams
from oracle import af2
from tests.helpers import assert_act, assert_grad, weights_dir

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,flip", [(256, False), (256, True), (288, False), (320, True),
                                    (352, False), (384, True), (480, False), (512, True)])
def test_attention_chunks(cuda, n, flip):
    print(f"attention chunks n={n} flip={flip}", flush=True)
    name = "triangle_attention_" + ("ending_node" if flip else "starting_node")
    rng = np.random.default_rng(n + flip)
    prm = bparams.init_block_params(0, rng, modules=[name], gates="random", ln="random")
    prefix = f"param/block0/{name}/"
    wdir = weights_dir(prm, f"chunks_{n}_{int(flip)}")
    m = np.ones(n, np.float32)
    m[rng.choice(n, n // 8, replace=False)] = 0.0
    T = lambda a: torch.as_tensor(np.asarray(a, np.float32), device=cuda)
    pair, dout = T(rng.standard_normal((n, n, 128))), T(rng.standard_normal((n, n, 128)))
    mask = T(np.outer(m, m))
    mod = ops.TriangleAttention(wdir, prefix, flip)
    out, save = mod.forward(pair, mask)
    din = mod.backward(pair, mask, None, save, dout)
    P = af2.Params(prm, prefix)
    x = pair.double().requires_grad_(True)
    ref = af2.triangle_attention(x, mask.double(), lambda v: P(v).to(cuda), flip)
    (g,) = torch.autograd.grad(ref, x, dout.double())
    print(" ", assert_act((out - pair).cpu().double(), ref.detach().cpu(), 2e-3, "delta"),
          assert_grad((din - dout).cpu().double(), g.cpu(), 0.99999, "dpair"))
