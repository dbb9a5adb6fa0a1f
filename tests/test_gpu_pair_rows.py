"""The pair track's row-tile kernels at the edges of their launch rules: the
32-, 48- and 64-row forms of triangle attention's and triangle multiplication's
products and the two forms of triangle attention's dX product, forward and
backward, at C = 128 (an Evoformer block) and C = 64 (the template stack),
with and without a dropout table, against the fp64 oracle at the modules' bars."""
import numpy as np
import pytest
import torch

from bindcraft2_amd import ops, params as bparams
from oracle import af2, jax_prng as J
from tests.helpers import assert_act, assert_grad, random_mask, weights_dir

pytestmark = pytest.mark.gpu
D = torch.float64


@pytest.mark.parametrize("kind", ["triattn", "trimul"])
# 128 / 160: 32- to 64-row LayerNorm tiles; 192 / 224: the last of the dX
# kernel; 288: 64-row cotangent tiles.  C = 64: as far as the fp64 oracle is quick.
@pytest.mark.parametrize("c,n,drop", [(128, 32, True), (128, 128, False), (128, 160, True),
                                      (128, 192, True), (128, 288, False), (64, 32, False),
                                      (64, 96, True), (64, 160, False), (64, 224, True)])
def test_row_kernels(cuda, kind, c, n, drop):
    print(f"{kind} c={c} n={n} drop={drop}", flush=True)
    flip = (n // 32) % 2 == 1  # ending node / outgoing at odd multiples of 32
    name = {"triattn": ("triangle_attention_starting_node", "triangle_attention_ending_node"),
            "trimul": ("triangle_multiplication_incoming", "triangle_multiplication_outgoing")}[kind][flip]
    rng = np.random.default_rng(c + n)
    if c == 128:
        prm = bparams.init_block_params(0, rng, modules=[name], gates="random", ln="random")
    else:
        prm = bparams.init_template_block_params(0, rng, gates="random", ln="random")
    prefix = f"param/block0/{name}/"
    wdir = weights_dir(prm, f"rows_{kind}_{c}_{n}")
    pair = rng.standard_normal((n, n, c)).astype(np.float32)
    dout = rng.standard_normal((n, n, c)).astype(np.float32)
    mask, _ = random_mask(n, 0.1, rng)
    tbl = af2.dropout_table(J.prng_key(n), 0.25, n, c) if drop else None
    if kind == "triattn":
        mod = ops.TriangleAttention(wdir, prefix, flip, c=c)
    else:
        mod = ops.TriangleMultiplication(wdir, prefix, flip, c=c, hidden=c)
    T = lambda a: None if a is None else torch.as_tensor(a, device=cuda)
    tp, tm, tt, td = T(pair), T(mask), T(tbl), T(dout)
    out, save = mod.forward(tp, tm, tt)
    din = mod.backward(tp, tm, tt, save, td)
    torch.cuda.synchronize()
    # the oracle on the device, in fp64
    P = af2.Params(prm, prefix)
    p = lambda v: P(v).to(cuda)
    p.sub = lambda s: (lambda v: P.sub(s)(v).to(cuda))
    x = tp.double().requires_grad_(True)
    if kind == "triattn":
        ref = af2.triangle_attention(x, tm.double(), p, flip)
    else:
        ref = af2.triangle_multiplication(x, tm.double(), p, flip)
    if drop:
        ref = ref * (tt.double()[:, None] if kind == "triattn" and flip else tt.double()[None])
    (g,) = torch.autograd.grad(ref, x, td.double())
    print(" ", assert_act((out - tp).cpu().double(), ref.detach().cpu(), 2e-3, "delta"),
          assert_grad((din - td).cpu().double(), g.cpu(), 0.99999, "dpair"))
