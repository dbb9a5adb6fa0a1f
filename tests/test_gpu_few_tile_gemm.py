"""Products of a few tiles (the MSA's S x N rows): every form of the launch --
one chain a wave, slices over waves, both tile heights -- at the edges of its
tiles and at odd row counts, against the exact product of the binary16
operands.  The sum of K products in f32, in whatever order, is off by at most
(K + 1) 2^-24 sum |a b| to first order."""
import pytest
import torch

from bindcraft2_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (1, 8, 32), (15, 64, 64), (16, 256, 64), (17, 72, 224), (33, 128, 128),   # unsplit, K < 256
    (127, 64, 256), (160, 256, 256), (160, 1024, 256), (129, 256, 1024),      # slices over waves
    (640, 1024, 256), (1025, 1024, 256),                                      # to the 32 x 64 tile
    (9216, 64, 256), (1500, 256, 1024), (1400, 1024, 288), (2049, 768, 320),  # two, three slices
    (224, 256, 2048),                                                         # past the slice limit
])
def test_few_tile_gemm(cuda, m, n, k):
    print(f"few-tile gemm m={m} n={n} k={k}", flush=True)
    g = torch.Generator().manual_seed(m * 7 + n * 3 + k)
    a = torch.randn(m, k, generator=g).half()
    b = torch.randn(n, k, generator=g).half()
    c = ops.probe_gemm(a.to(cuda), b.to(cuda)).cpu().double()
    a, b = a.double(), b.double()
    bound = (k + 1) * 2.0 ** -24 * (a.abs() @ b.abs().T)
    assert ((c - a @ b.T).abs() <= bound).all()
