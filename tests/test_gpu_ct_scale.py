"""The backward's power-of-two cotangent scale: d(in) of 2^k times a cotangent is
2^k times d(in), bit for bit (the scaled cotangent that every product sees is the
same), and a zero cotangent gives zeros -- where the first row kernel reduces the
partial maxima itself and where a launch of its own does (the MSA's width; eight
heads, or a hidden width other than the channels', which have no row kernel)."""
import numpy as np
import pytest
import torch

from bindcraft2_amd import ops, params as bparams
from tests.helpers import random_mask, weights_dir

pytestmark = pytest.mark.gpu


def _module(kind, c, n, rng):
    kind, _, general = kind.partition("/")
    names = {"triattn": "triangle_attention_starting_node",
             "trimul": "triangle_multiplication_outgoing",
             "transition": "pair_transition", "msa_transition": "msa_transition"}
    if c == 64:
        prm = bparams.init_template_block_params(0, rng, gates="random", ln="random")
    else:
        kw = {"tri_heads": 8, "trimul_hidden": 64} if general else {}
        prm = bparams.init_block_params(0, rng, modules=[names[kind]], gates="random", ln="random", **kw)
    wdir, prefix = weights_dir(prm, f"ct_{kind}{general}_{c}_{n}"), f"param/block0/{names[kind]}/"
    if kind == "triattn":
        return ops.TriangleAttention(wdir, prefix, False, c=c, heads=8 if general else 4)
    if kind == "trimul":
        return ops.TriangleMultiplication(wdir, prefix, True, c=c, hidden=64 if general else c)
    return ops.Transition(wdir, prefix, c, 2 if c == 64 else 4)


@pytest.mark.parametrize("kind,c,n", [("triattn", 128, 32), ("triattn", 64, 96), ("trimul", 128, 64),
                                      ("trimul", 64, 32), ("transition", 128, 33),
                                      ("transition", 64, 32), ("msa_transition", 256, 64),
                                      ("triattn/general", 128, 32), ("trimul/general", 128, 64)])
def test_power_of_two(cuda, kind, c, n):
    print(f"{kind} c={c} n={n}", flush=True)
    rng = np.random.default_rng(n + c)
    mod = _module(kind, c, n, rng)
    rows = (2, n, c) if kind == "msa_transition" else (n, n, c)
    x = torch.as_tensor(rng.standard_normal(rows).astype(np.float32), device=cuda)
    dout = torch.as_tensor(rng.standard_normal(rows).astype(np.float32), device=cuda)
    mask = torch.as_tensor(random_mask(n, 0.1, rng)[0], device=cuda)
    args = (x, mask, None) if kind.startswith("tri") else (x, None)
    _, save = mod.forward(*args)
    ref = mod.backward(*args, save, dout)
    assert torch.isfinite(ref).all() and ref.abs().max() > 0
    for k in (-40, 13, 60):
        got = mod.backward(*args, save, dout * 2.0 ** k)
        assert torch.equal(got * 2.0 ** -k, ref), k
    assert not mod.backward(*args, save, torch.zeros_like(dout)).any()
