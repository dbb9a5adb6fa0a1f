"""The template stack's transition (C = 64, factor 2) as one kernel a direction:
row counts at the edges of its row tiles (32 rows, and 64 for the last case), with and without the shared dropout
table, against the fp64 oracle at the module's bars."""
import numpy as np
import pytest
import torch

from bindcraft2_amd import ops, params as bparams
from oracle import af2
from tests.helpers import assert_act, assert_grad, weights_dir

pytestmark = pytest.mark.gpu
D = torch.float64


@pytest.mark.parametrize("b,n,drop", [(1, 1, False), (1, 31, True), (3, 11, False), (1, 64, True),
                                      (5, 13, True), (32, 32, False), (96, 96, True), (182, 181, True)])
def test_template_transition(cuda, b, n, drop):
    print(f"b={b} n={n} drop={drop}", flush=True)
    rng = np.random.default_rng(64 * b + n)
    prm = bparams.init_template_block_params(0, rng, gates="random", ln="random")
    mod = ops.Transition(weights_dir(prm, f"tt_{b}_{n}"), "param/block0/pair_transition/", 64, 2)
    act = rng.standard_normal((b, n, 64)).astype(np.float32)
    dout = rng.standard_normal((b, n, 64)).astype(np.float32)
    tbl = ((rng.random((n, 64)) > 0.25) / 0.75).astype(np.float32) if drop else None
    T = lambda a: None if a is None else torch.as_tensor(a, device=cuda)
    ta, td, tt = T(act), T(dout), T(tbl)
    out, save = mod.forward(ta, tt)
    din = mod.backward(ta, tt, save, td)
    P = af2.Params(prm, "param/block0/pair_transition/")
    x = torch.tensor(act, dtype=D, requires_grad=True)
    ref = af2.transition(x, None, P)
    if drop:
        ref = ref * torch.as_tensor(tbl, dtype=D)[None]
    (g,) = torch.autograd.grad(ref, x, torch.as_tensor(dout, dtype=D))
    print(assert_act((out - ta).cpu().double(), ref.detach(), what="delta"),
          assert_grad((din - td).cpu().double(), g, what="dact"))
