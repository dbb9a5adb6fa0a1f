"""Which launch a product of few tiles takes: row counts on both sides of each
line of the rule, against the exact product of the binary16 operands (the bound
of f32 sums of K products in any order); past the lines no launch whose time
grows faster than its rows do, and the MSA side's split launches on the second
stream with the bits of one stream."""
import numpy as np
import pytest
import torch

from bindcraft2_amd import ops, params as bparams
from tests.helpers import random_mask, weights_dir

pytestmark = pytest.mark.gpu


def _operands(cuda, m, n, k):
    g = torch.Generator(device=cuda).manual_seed(m + n + k)
    return (torch.randn(m, k, generator=g, device=cuda).half(),
            torch.randn(n, k, generator=g, device=cuda).half())


# the lines on 256 CUs: unsplit 1792 tiles of 16 x 32; two and three slices 80
# steps; four and more 288 steps, 128 beyond K = 1024
@pytest.mark.parametrize("m,n,k", [(7168, 128, 128), (7184, 128, 128), (4779, 192, 64), (4800, 192, 64),
                                   (13648, 64, 384), (13664, 64, 384), (48, 12288, 512), (49, 12288, 512),
                                   (4607, 256, 1024), (4609, 256, 1024),
                                   (2048, 128, 2048), (2049, 128, 2048), (40, 12288, 1024)])
def test_both_sides(cuda, m, n, k):
    print(f"few-tile rule m={m} n={n} k={k}", flush=True)
    a, b = _operands(cuda, m, n, k)
    c = ops.probe_gemm(a, b).cpu().double()
    a, b = a.cpu().double(), b.cpu().double()
    bound = (k + 1) * 2.0 ** -24 * (a.abs() @ b.abs().T)
    assert ((c - a @ b.T).abs() <= bound).all()


@pytest.mark.parametrize("m,n,k", [(3584, 256, 1024), (768, 1024, 1024), (8128, 128, 2048)])
def test_time_follows_rows(cuda, m, n, k):
    """Twice the rows in at most 2.5 times the time (an even split would be 2)."""
    def us(rows):
        a, b = _operands(cuda, rows, n, k)
        best = float("inf")
        for _ in range(8):
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            t0.record()
            for _ in range(40):
                ops.probe_gemm(a, b)
            t1.record()
            t1.synchronize()
            best = min(best, t0.elapsed_time(t1) * 25)
        return best
    half, whole = us(m), us(2 * m)
    print(f"m={m} n={n} k={k}: {half:.1f} us, twice the rows {whole:.1f}", flush=True)
    assert whole < 2.5 * half


# 5120 and 4896 rows, past the line of K = 1024 (4608), beside the pair track; N = 288:
# the row attention's few-workgroup forms as well
@pytest.mark.parametrize("n,s", [(160, 32), (288, 17)])
def test_split_on_the_second_stream(cuda, n, s):
    print(f"stack n={n} s={s}", flush=True)
    rng = np.random.default_rng(n)
    prm = {}
    for b in range(2):
        prm.update(bparams.init_block_params(b, rng, gates="random", ln="random"))
    st = ops.EvoformerStack(weights_dir(prm, f"split_side_{n}"), 2)
    T = lambda a: torch.as_tensor(np.asarray(a, np.float32), device=cuda)
    pm, m1 = random_mask(n, 0.1, rng)
    pmask, mmask = T(pm), T(np.tile(m1, (s, 1)))
    pair, msa = T(rng.standard_normal((n, n, 128))), T(rng.standard_normal((s, n, 256)))
    ct_p, ct_m = torch.randn_like(pair), torch.randn_like(msa)
    seed = ops.seed_tensor((3, 4), True, cuda)
    res = []
    for on in (False, True, True):
        with ops.msa_overlap(on):
            po, mo, sv = st.forward(pair, msa, pmask, mmask, seed)
            res.append([t.clone() for t in (po, mo, *st.backward(ct_p, ct_m, pmask, mmask, sv, seed))])
    for r in res[1:]:
        for a, b in zip(res[0], r):
            assert torch.isfinite(a).all() and torch.equal(a, b)
