"""The MSA row attention beyond N = 256 on both sides of the line between the
forms for few workgroups and for many (two a CU: 16 rows at N = 512 and 17, 21
rows at N = 288 and 22), with whole and partial last key chunks, partially masked
rows and one without a live key, forward and backward against the fp64 oracle run
on the device."""
import numpy as np
import pytest
import torch

from bindcraft2_amd import ops, params as bparams
from oracle import af2
from tests.helpers import assert_act, assert_grad, weights_dir

pytestmark = pytest.mark.gpu
NAME = "msa_row_attention_with_pair_bias"


@pytest.mark.parametrize("n,s", [(288, 1), (288, 21), (288, 22), (320, 2), (384, 3), (416, 1),
                                 (512, 16), (512, 17), (544, 2), (1024, 1)])
def test_few_rows(cuda, n, s):
    print(f"msa row attention n={n} s={s}", flush=True)
    rng = np.random.default_rng(n + s)
    prm = bparams.init_block_params(0, rng, modules=[NAME], gates="random", ln="random")
    prefix = f"param/block0/{NAME}/"
    mask = (rng.random((s, n)) > 0.2).astype(np.float32)
    if s > 1:
        mask[s - 1] = 0.0
    T = lambda a: torch.as_tensor(np.asarray(a, np.float32), device=cuda)
    msa, dout = T(rng.standard_normal((s, n, 256))), T(rng.standard_normal((s, n, 256)))
    pair, mask = T(rng.standard_normal((n, n, 128))), T(mask)
    mod = ops.MSARowAttentionWithPairBias(weights_dir(prm, f"few_{n}_{s}"), prefix)
    out, save = mod.forward(msa, mask, pair)
    din, dpair = mod.backward(msa, mask, pair, None, save, dout)
    P = af2.Params(prm, prefix)
    x, z = msa.double().requires_grad_(True), pair.double().requires_grad_(True)
    ref = af2.msa_row_attention(x, mask.double(), z, lambda v: P(v).to(cuda))
    gx, gz = torch.autograd.grad(ref, (x, z), dout.double())
    print(" ", assert_act((out - msa).cpu().double(), ref.detach().cpu(), 2e-3, "delta"),
          assert_grad((din - dout).cpu().double(), gx.cpu(), 0.99999, "dmsa"),
          assert_grad(dpair.cpu().double(), gz.cpu(), 0.99999, "dpair"))
