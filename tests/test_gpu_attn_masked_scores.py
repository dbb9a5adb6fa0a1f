"""Masked keys weigh nothing however large their scores: triangle attention whose
masked residues, where a live query's score against them counted, would win by
far more than 8192 log2 units, on both sides of N = 256 and at both head widths,
forward and backward against the fp64 oracle run on the device (whose rows
without a live key attend uniformly)."""
import numpy as np
import pytest
import torch

from bindcraft2_amd import ops, params as bparams
from oracle import af2
from tests.helpers import assert_act, assert_grad, weights_dir

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c,n,flip", [(128, 256, False), (128, 288, True), (128, 480, False),
                                      (64, 256, True), (64, 320, False), (64, 512, True)])
def test_masked_scores(cuda, c, n, flip):
    print(f"masked scores c={c} n={n} flip={flip}", flush=True)
    name = "triangle_attention_" + ("ending_node" if flip else "starting_node")
    rng = np.random.default_rng(n + c)
    if c == 128:
        prm = bparams.init_block_params(0, rng, modules=[name], gates="random", ln="random")
    else:
        prm = bparams.init_template_block_params(0, rng, gates="random", ln="random")
    prefix = f"param/block0/{name}/"
    # channels 0 and 1 mark a token as masked or live; a masked key answers a
    # live query with a score of some 1e5, live keys do not see the markers
    for w, ch, v in (("key_w", 0, 800.0), ("key_w", 1, 0.0), ("query_w", 0, 0.0), ("query_w", 1, 0.5)):
        prm[prefix + "attention/" + w][ch] = v
    prm[prefix + "feat_2d_weights"][:2] = 0.0
    prm[prefix + "query_norm/scale"][:2], prm[prefix + "query_norm/offset"][:2] = 1.0, 0.0
    wdir = weights_dir(prm, f"masked_{c}_{n}")
    m = np.ones(n, np.float32)
    m[rng.choice(n, n // 8, replace=False)] = 0.0
    mask = np.outer(m, m)
    pair = rng.standard_normal((n, n, c))
    pair[..., 0], pair[..., 1] = 20.0 * (1 - mask), 3.0 * mask
    # rows of mean 0: the LayerNorm leaves the absent marker at 0
    pair[..., 2:] -= pair.sum(-1, keepdims=True) / (c - 2)
    T = lambda a: torch.as_tensor(np.asarray(a, np.float32), device=cuda)
    pair, dout, mask = T(pair), T(rng.standard_normal((n, n, c))), T(mask)
    P = af2.Params(prm, prefix)
    p = lambda v: P(v).to(cuda)
    # the premise, from the oracle's own operands: a live row's masked scores
    xr = af2.layer_norm((pair.transpose(0, 1) if flip else pair)[int(m.argmax())].double(),
                        p("query_norm/scale"), p("query_norm/offset"))
    live = torch.as_tensor(m, device=cuda) > 0
    s = torch.einsum("qhd,khd->hqk", torch.einsum("qc,chd->qhd", xr, p("attention/query_w")),
                     torch.einsum("kc,chd->khd", xr, p("attention/key_w")))
    s = s * (c // 4) ** -0.5 * np.log2(np.e)
    assert (s[:, live][..., ~live].amax(-1) - s[:, live][..., live].amax(-1)).min() > 2 * 8192
    mod = ops.TriangleAttention(wdir, prefix, flip, c=c)
    out, save = mod.forward(pair, mask)
    din = mod.backward(pair, mask, None, save, dout)
    x = pair.double().requires_grad_(True)
    ref = af2.triangle_attention(x, mask.double(), p, flip)
    (g,) = torch.autograd.grad(ref, x, dout.double())
    print(" ", assert_act((out - pair).cpu().double(), ref.detach().cpu(), 2e-3, "delta"),
          assert_grad((din - dout).cpu().double(), g.cpu(), 0.99999, "dpair"))
