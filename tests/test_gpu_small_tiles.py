"""Products of small factors on 64-wide tiles (four waves, a 32x32 block each) of the bf16 matrix cores:
at the edges of blocks and tiles, of chunks and short reductions, single and in one grouped call, with
odd runs and elements that are not finite; and where single products change to 128-wide tiles."""
import pytest
import torch

from test_gpu_split_products import _assert_float32_sum, dev, ops  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


def randn(dev, *shape):
    gen = torch.Generator(device=dev).manual_seed(sum(shape))
    return torch.randn(*shape, device=dev, generator=gen)


@pytest.mark.parametrize('rows', [1, 15, 16, 17, 48, 49, 300, 2049])
@pytest.mark.parametrize('f', [1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 192])
def test_dense(ops, dev, f, rows):  # noqa: F811
    x = randn(dev, rows, f)
    a = torch.cat([x.double(), torch.ones(rows, 1, device=dev, dtype=torch.float64)], 1)
    old = torch.rand(f + 1, f + 1, device=dev)
    old = old + old.t()
    grouped = [torch.full((f + b,) * 2, float('nan'), device=dev) for b in (0, 1)]
    ops.factor_grouped([ops.factor_job('linear', x, 1., grouped[0], add_bias=False),
                        ops.factor_job('linear', x, 1., grouped[1], add_bias=True)], dev)
    torch.cuda.synchronize()
    for out, a64, plus in ((ops.factor_linear(x, False, 1.), a[:, :f], 0.),
                           (ops.factor_linear(x, True, 1., out=old.clone(), beta=1.), a, old.double()),
                           (grouped[0], a[:, :f], 0.), (grouped[1], a, 0.)):
        _assert_float32_sum(out, a64, a64, '%d rows of %d' % (rows, f), plus=plus)
        assert torch.equal(out, out.t())


# both sides of the change of tile
@pytest.mark.parametrize('f', [193, 256])
@pytest.mark.parametrize('rows', [24576, 24577, 32768, 32769])
def test_long_reductions(ops, dev, f, rows):  # noqa: F811
    x = randn(dev, rows, f)
    out = ops.factor_linear(x, False, 1.)
    _assert_float32_sum(out, x.double(), x.double(), '%d rows of %d' % (rows, f))
    assert torch.equal(out, out.t())


# runs of one row, padded ones, and short ones that are not; 9 to 1587 terms
@pytest.mark.parametrize('c', [3, 33, 64, 65, 130])
@pytest.mark.parametrize('hw', [(1, 3), (3, 3), (5, 7), (4, 4), (23, 23)])
def test_convolutions(ops, dev, c, hw):  # noqa: F811
    x = randn(dev, 3, c, *hw)
    positions = x.double().permute(0, 2, 3, 1).reshape(-1, c)
    cols = {}
    for k, s in ((3, 1), (3, 2)):
        u = torch.nn.functional.unfold(x.double(), k, padding=1, stride=s)
        cols[k, s] = u.permute(0, 2, 1).reshape(-1, u.shape[1])
    jobs, outs = [], []
    for kind, a, geometry in (('conv_g', positions, {}),
                              ('conv_a', positions, dict(kernel_size=1, stride=1, padding=0, dilation=1)),
                              ('conv_a', cols[3, 1], dict(kernel_size=3, stride=1, padding=1, dilation=1)),
                              ('conv_a', cols[3, 2], dict(kernel_size=3, stride=2, padding=1, dilation=1))):
        out = torch.full((a.shape[1],) * 2, float('nan'), device=dev)
        jobs.append(ops.factor_job(kind, x, 1., out, **geometry))
        outs.append((out, a))
    ops.factor_grouped(jobs, dev)
    torch.cuda.synchronize()
    outs += [(ops.factor_conv_g(x, 1.), positions)]
    outs += [(ops.factor_conv_a(x, (k, k), (s, s), (1, 1), (1, 1), False, 1.), a) for (k, s), a in cols.items()]
    for i, (out, a) in enumerate(outs):
        _assert_float32_sum(out, a, a, 'product %d, %d channels of %dx%d' % ((i, c) + hw))
        assert torch.equal(out, out.t())


@pytest.mark.parametrize('rows', [20, 147])
def test_not_finite(ops, dev, rows):  # noqa: F811
    x = randn(dev, rows, 100).abs() + 0.1
    x[1, 10], x[0, 40], x[2, 70], x[3, 90] = float('inf'), -float('inf'), float('nan'), 1.1e25
    x[4, 99], x[5, 3] = 2. ** 64 - 2. ** 54, 3.4e38 * 1e-20
    want = x.cpu().t() @ x.cpu()
    for out in (ops.factor_linear(x, False, 1.), ops.factor_conv_g(x.t().reshape(1, 100, 1, rows), 1.)):
        out = out.cpu()
        assert torch.equal(out.isnan(), want.isnan())
        assert torch.equal(out.isposinf(), want.isposinf()) and torch.equal(out.isneginf(), want.isneginf())
        ok = want.isfinite()
        # (sums of positive terms: either side within rows roundings of the exact sum)
        assert ((out - want)[ok] / want[ok]).abs().max().item() < 2 * rows * 2. ** -24


# one term apiece in sums of up to, and of more than, a rolled loop's length; magnitudes around 1, and from
# below the range of split elements to sums beyond that of scaled ones
@pytest.mark.parametrize('rows', [5, 48, 49, 300, 5000])
@pytest.mark.parametrize('exponents', [(0, 0), (-36, 3), (-36, 18)])
def test_single_terms_are_rounded_once(ops, dev, rows, exponents):  # noqa: F811
    """Sums of which all terms but one are zero (inputs behind a ReLU, one-hot rows) are that product, rounded to
    float32.  Allowed beyond that: the seven partial products added to the corrections, at most 2^-8 of the
    product, each rounded by 2^-23 of those."""
    f = 130
    x = torch.zeros(rows, f, device=dev)
    gen = torch.Generator(device=dev).manual_seed(rows)
    lo, hi = exponents
    x[rows // 2] = torch.randn(f, device=dev, generator=gen).sign() * 10. ** (
        lo + (hi - lo) * torch.rand(f, device=dev, generator=gen, dtype=torch.float64)).float() * (
        1 + torch.rand(f, device=dev, generator=gen))
    want = x[rows // 2].double()[:, None] * x[rows // 2].double()
    bound = want.abs() * 2. ** -24 * (1 + 7 * 2. ** -7) + 2. ** -149
    grouped = torch.full((f, f), float('nan'), device=dev)
    ops.factor_grouped([ops.factor_job('linear', x, 1., grouped)], dev)
    positions = x.t().reshape(1, f, 1, rows).contiguous()
    torch.cuda.synchronize()
    for got in (ops.factor_linear(x, False, 1.), grouped, ops.factor_conv_g(positions, 1.)):
        # (what a float32 cannot hold as a normal number is not looked at)
        over = ((got.double() - want).abs() / bound)[want.abs() >= 2. ** -126]
        assert over.max().item() <= 1., 'error %.2f times the bound' % over.max().item()
