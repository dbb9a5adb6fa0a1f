"""Triangle attention and multiplication at widths without a row kernel (eight heads
of 16 or 32, a hidden width other than the channels'): LayerNorm, products and
LayerNorm backward as launches of their own, forward and backward, with and without a
dropout table, against the fp64 oracle run on the device."""
import numpy as np
import pytest
import torch

from bindcraft2_amd import ops, params as bparams
from oracle import af2, jax_prng as J
from tests.helpers import assert_act, assert_grad, random_mask, weights_dir

pytestmark = pytest.mark.gpu


# (channels, heads): head widths 16 and 32; 288: the attention's long forms
@pytest.mark.parametrize("c,h,n,flip,drop", [(128, 8, 32, False, True), (128, 8, 96, True, False),
                                             (128, 8, 288, False, False), (256, 8, 64, True, True),
                                             (256, 8, 160, False, False)])
def test_triangle_attention(cuda, c, h, n, flip, drop):
    print(f"triattn c={c} h={h} n={n} flip={flip} drop={drop}", flush=True)
    name = "triangle_attention_" + ("ending_node" if flip else "starting_node")
    rng = np.random.default_rng(c + n)
    prm = bparams.init_block_params(0, rng, modules=[name], gates="random", ln="random", c_z=c, tri_heads=h)
    prefix = f"param/block0/{name}/"
    mod = ops.TriangleAttention(weights_dir(prm, f"gen_a_{c}_{n}"), prefix, flip, c=c, heads=h)
    _compare(cuda, rng, prm, prefix, mod, c, n, drop,
             lambda x, m, p: af2.triangle_attention(x, m, p, flip), flip)


# (channels, hidden): 288: contractions as tiled products
@pytest.mark.parametrize("c,i,n,out,drop", [(128, 64, 32, True, True), (128, 64, 96, False, False),
                                            (64, 128, 64, True, False), (256, 128, 64, False, True),
                                            (128, 64, 288, True, False)])
def test_triangle_multiplication(cuda, c, i, n, out, drop):
    print(f"trimul c={c} i={i} n={n} out={out} drop={drop}", flush=True)
    name = "triangle_multiplication_" + ("outgoing" if out else "incoming")
    rng = np.random.default_rng(c + i + n)
    prm = bparams.init_block_params(0, rng, modules=[name], gates="random", ln="random", c_z=c,
                                    trimul_hidden=i)
    prefix = f"param/block0/{name}/"
    mod = ops.TriangleMultiplication(weights_dir(prm, f"gen_m_{c}_{i}_{n}"), prefix, out, c=c, hidden=i)
    _compare(cuda, rng, prm, prefix, mod, c, n, drop,
             lambda x, m, p: af2.triangle_multiplication(x, m, p, out), False)


def _compare(cuda, rng, prm, prefix, mod, c, n, drop, oracle, per_column):
    T = lambda a: None if a is None else torch.as_tensor(np.asarray(a, np.float32), device=cuda)
    pair, dout = T(rng.standard_normal((n, n, c))), T(rng.standard_normal((n, n, c)))
    mask = T(random_mask(n, 0.1, rng)[0])
    tbl = T(af2.dropout_table(J.prng_key(n), 0.25, n, c)) if drop else None
    out, save = mod.forward(pair, mask, tbl)
    din = mod.backward(pair, mask, tbl, save, dout)
    P = af2.Params(prm, prefix)
    p = lambda v: P(v).to(cuda)
    p.sub = lambda s: (lambda v: P.sub(s)(v).to(cuda))
    x = pair.double().requires_grad_(True)
    ref = oracle(x, mask.double(), p)
    if drop:
        ref = ref * (tbl.double()[:, None] if per_column else tbl.double()[None])
    (g,) = torch.autograd.grad(ref, x, dout.double())
    print(" ", assert_act((out - pair).cpu().double(), ref.detach().cpu(), 2e-3, "delta"),
          assert_grad((din - dout).cpu().double(), g.cpu(), 0.99999, "dpair"))
