"""The template stack's widths (C = 64: heads of 16) beyond 256 residues: the
attention's forward and dQ with 64- and 96-key chunks, whole and partial last ones,
and idle query waves, with residues whose rows are fully masked, and the
multiplication's 64-row centre-norm form, forward and backward against the fp64 oracle
run on the device."""
import numpy as np
import pytest
import torch

from bindcraft2_amd import ops, params as bparams
from oracle import af2
from tests.helpers import assert_act, assert_grad, weights_dir

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n,flip", [("attention", 288, True), ("attention", 320, False),
                                         ("attention", 352, False), ("attention", 416, True),
                                         ("attention", 480, False), ("attention", 512, True),
                                         ("multiplication", 352, True), ("multiplication", 416, False)])
def test_template_lengths(cuda, kind, n, flip):
    print(f"c=64 {kind} n={n} flip={flip}", flush=True)
    name = {"attention": ("triangle_attention_starting_node", "triangle_attention_ending_node"),
            "multiplication": ("triangle_multiplication_incoming", "triangle_multiplication_outgoing")}[kind][flip]
    rng = np.random.default_rng(n + flip)
    prm = bparams.init_template_block_params(0, rng, gates="random", ln="random")
    prefix = f"param/block0/{name}/"
    wdir = weights_dir(prm, f"tl_{kind}_{n}")
    m = np.ones(n, np.float32)
    m[rng.choice(n, n // 8, replace=False)] = 0.0
    T = lambda a: torch.as_tensor(np.asarray(a, np.float32), device=cuda)
    pair, dout = T(rng.standard_normal((n, n, 64))), T(rng.standard_normal((n, n, 64)))
    mask = T(np.outer(m, m))
    if kind == "attention":
        mod, oracle = ops.TriangleAttention(wdir, prefix, flip, c=64), af2.triangle_attention
    else:
        mod = ops.TriangleMultiplication(wdir, prefix, flip, c=64, hidden=64)
        oracle = af2.triangle_multiplication
    out, save = mod.forward(pair, mask)
    din = mod.backward(pair, mask, None, save, dout)
    P = af2.Params(prm, prefix)
    p = lambda v: P(v).to(cuda)
    p.sub = lambda s: (lambda v: P.sub(s)(v).to(cuda))
    x = pair.double().requires_grad_(True)
    ref = oracle(x, mask.double(), p, flip)
    (g,) = torch.autograd.grad(ref, x, dout.double())
    print(" ", assert_act((out - pair).cpu().double(), ref.detach().cpu(), 2e-3, "delta"),
          assert_grad((din - dout).cpu().double(), g.cpu(), 0.99999, "dpair"))
