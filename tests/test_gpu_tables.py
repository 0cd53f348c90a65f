"""Device tables of grouped factor calls that take one short, one long and several uploads."""
import pytest
import torch

from torchsso import _ops as ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('count', [1, 20, 30, 60, 120, 250])
def test_tables_of_many_products(count):
    dev = torch.device('cuda', 0)
    gen = torch.Generator().manual_seed(count)
    xs = [torch.randn(5 + i % 7, 1 + i % 40, generator=gen) for i in range(count)]
    dxs = [x.to(dev) for x in xs]
    outs = [torch.full((x.shape[1], x.shape[1]), float('nan'), device=dev) for x in xs]
    ops.factor_grouped([ops.factor_job('linear', x, 0.5, o) for x, o in zip(dxs, outs)], dev)
    for x, o in zip(xs, outs):
        ref = 0.5 * x.double().t() @ x.double()
        # (sums of at most 11 products: a few roundings of 2^-24 of the largest entry)
        assert (o.double().cpu() - ref).abs().max() <= 16 * 2. ** -24 * ref.abs().max()
