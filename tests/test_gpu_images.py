"""Factors of 128-wide tiles: what lies below the diagonal is the image of what lies above, to the bit, up to the last
row and column and not beyond; with old values, in one piece and in pieces of the reduction."""
import pytest
import torch

from torchsso import _ops as ops

pytestmark = pytest.mark.gpu


# (rows, columns with the one of the bias): one tile and its edges, ragged ones, 32-row blocks that are cut
@pytest.mark.parametrize('rows,d', [(64, 256), (49, 257), (96, 385), (33, 415), (256, 511), (20, 1000), (4096, 321)])
@pytest.mark.parametrize('grouped', [False, True])
def test_images(rows, d, grouped):
    dev = torch.device('cuda', 0)
    gen = torch.Generator().manual_seed(d)
    x = torch.randn(rows, d - 1, generator=gen)
    prev = torch.randn(d, d, generator=gen)
    prev = prev + prev.t()
    ones = torch.cat([x, torch.ones(rows, 1)], 1).double()
    want = 0.25 * ones.t() @ ones + 0.5 * prev.double()
    # each output is a sum of `rows` products of float32 values: rounding of sqrt(rows) units, with room
    tol = 6e-8 * (4 + rows ** 0.5)
    guard = torch.full((d * d + 64,), 7., device=dev)
    out = guard[:d * d].view(d, d)
    xd, old = x.to(dev), prev.to(dev)
    if grouped:
        job = ops.factor_job('linear', xd, 0.25, out, beta=0.5, prev=old, add_bias=True)
        ops.factor_grouped([job], dev)
    else:
        ops.factor_linear(xd, True, 0.25, out=out, beta=0.5, prev=old)
    assert torch.equal(out, out.t())
    assert ((out.double().cpu() - want).norm() / want.norm()).item() < tol
    assert bool((guard[d * d:] == 7.).all())
