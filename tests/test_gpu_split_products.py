"""Products on the bf16 matrix cores with float32 results (csrc/gemm_split.h): every element
within the rounding of a float32 sum of its exact products, at the edges of tiles, chunks and
runs, and over the range of magnitudes of the data type."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def dev():
    return torch.device('cuda:0')


@pytest.fixture(scope='module')
def ops():
    from torchsso import _ops
    return _ops


def _assert_float32_sum(got, a, b, what, where=None, plus=0.):
    """got = a^T b (+ plus) for float64 copies a [K, m], b [K, n] of float32 operands.  An element is a
    sum of exact products, of which the terms of relative size 2^-23 and below are left
    out, added to float32 accumulators in at most K / 16 + 1 steps each for the leading and
    the correction terms (16 products per step, each step within 2^-23 of the running sum of
    absolute values), over at most K / 128 + 1 partial sums.  At the small end of the range an
    element below 2^-109 is rounded to a multiple of 2^-133, the smallest bf16 number, and
    a sum to one of 2^-149 at every step of either accumulator."""
    K = a.shape[0]
    want = a.t() @ b + plus
    mass = a.abs().t() @ b.abs() + abs(plus)
    tiny = lambda x: ((x.abs() < 2. ** -109) & (x != 0)).double()
    rounded = 2. ** -134 * (tiny(a).t() @ b.abs() + a.abs().t() @ tiny(b))
    bound = mass * (2. ** -23) * (2 * (K // 16 + 1) + K // 128 + 4) + rounded \
        + 2. ** -149 * (2 * (K // 16 + 1) + K // 128 + 4)
    over = (got.double() - want).abs() / bound
    over = (over if where is None else over[where]).max().item()
    assert over <= 1., '%s: error %.2f times the bound' % (what, over)


@pytest.mark.parametrize('bias', [False, True])
@pytest.mark.parametrize('rows', [1, 15, 16, 17, 33, 47, 130])
@pytest.mark.parametrize('f', [193, 255, 256, 257, 384])
def test_dense_symmetric(ops, dev, f, rows, bias):
    gen = torch.Generator(device=dev).manual_seed(f * 1000 + rows)
    x = torch.randn(rows, f, device=dev, generator=gen)
    out = ops.factor_linear(x, bias, 1.)
    a = x.double()
    if bias:
        a = torch.cat([a, torch.ones(rows, 1, device=dev, dtype=torch.float64)], 1)
    _assert_float32_sum(out, a, a, 'factor of %d x %d' % (rows, f))
    assert torch.equal(out, out.t())


# the last reduction in one rolled loop (48 steps) and the first that is not, of products of one
# operand, of two, and of operands whose consecutive k are next to each other
@pytest.mark.parametrize('rows', [31, 32, 48, 49, 64])
def test_short_reductions(ops, dev, rows):
    gen = torch.Generator(device=dev).manual_seed(rows)
    x = torch.randn(rows, 300, device=dev, generator=gen)
    g = torch.randn(rows, 200, device=dev, generator=gen)
    a = torch.cat([x.double(), torch.ones(rows, 1, device=dev, dtype=torch.float64)], 1)
    _assert_float32_sum(ops.factor_linear(x, True, 1.), a, a, 'factor, %d rows' % rows)
    w, b = ops.diag_cov_linear(g, x, True, 1.)
    # (the squares are float32 too: another rounding of either factor)
    _assert_float32_sum(torch.cat([w, b[:, None]], 1), g.double() ** 2, a ** 2, 'squares, %d' % rows)
    c = torch.randn(1, 300, 1, rows, device=dev, generator=gen)
    a = c.double().reshape(300, rows).t()
    _assert_float32_sum(ops.factor_conv_g(c, 1.), a, a, 'positions, %d' % rows)


# one run of a multiple of 4, padded runs (5 = 8 - 3, 6, 7, 9, ...), runs left as they are (1 .. 3)
@pytest.mark.parametrize('hw', [(1, 1), (1, 3), (2, 2), (1, 5), (2, 3), (1, 7), (3, 3), (2, 5), (3, 5),
                                (7, 7), (5, 13), (8, 8)])
@pytest.mark.parametrize('n', [1, 2, 5, 40])
def test_positions_in_runs_of_a_grouped_call(ops, dev, n, hw):
    """Output gradients of two sizes, a pointwise and a strided convolution's input in one call;
    nothing but the positions themselves may reach the sums, whatever lies beside a run."""
    gen = torch.Generator(device=dev).manual_seed(n * 100 + hw[0] * hw[1])
    randn = lambda *shape: torch.randn(*shape, device=dev, generator=gen)
    positions = lambda t: t.double().permute(0, 2, 3, 1).reshape(-1, t.shape[1])
    g, h, x = randn(n, 200, *hw), randn(n, 65, *hw), randn(n, 257, *hw)
    s = randn(n, 23, 2 * hw[0] + 1, 2 * hw[1] + 1)          # 3x3, stride 2: hw output positions
    g[0, 199], g[0, 198] = 1e18, 1.
    cols = torch.nn.functional.unfold(s.double(), 3, stride=2)         # [n, 23 * 9, positions]
    jobs, outs, rows = [], [], []
    for kind, t, rows64, geometry in (
            ('conv_g', g, positions(g), {}), ('conv_g', h, positions(h), {}),
            ('conv_a', x, positions(x), dict(kernel_size=1, stride=1, padding=0, dilation=1)),
            ('conv_a', s, cols.permute(0, 2, 1).reshape(-1, cols.shape[1]),
             dict(kernel_size=3, stride=2, padding=0, dilation=1))):
        out = torch.full((rows64.shape[1],) * 2, float('nan'), device=dev)
        jobs.append(ops.factor_job(kind, t, 1., out, **geometry))
        outs.append(out)
        rows.append(rows64)
    ops.factor_grouped(jobs, dev)
    torch.cuda.synchronize()
    for k, (out, a) in enumerate(zip(outs, rows)):
        _assert_float32_sum(out, a, a, 'product %d, %d images of %dx%d' % ((k, n) + hw))
        assert torch.equal(out, out.t())


@pytest.mark.parametrize('hw', [(1, 1), (1, 3), (2, 2), (3, 3), (7, 7), (5, 13), (8, 8)])
@pytest.mark.parametrize('n', [1, 5])
def test_positions_in_runs(ops, dev, n, hw):
    c = 200
    gen = torch.Generator(device=dev).manual_seed(n * 100 + hw[0] * hw[1])
    g = torch.randn(n, c, *hw, device=dev, generator=gen)
    out = ops.factor_conv_g(g, 1.)
    a = g.double().permute(0, 2, 3, 1).reshape(-1, c)
    _assert_float32_sum(out, a, a, 'output gradients %dx%dx%d' % ((n,) + hw))
    assert torch.equal(out, out.t())


# single products on 128-wide tiles (more than 256 rows), with the old contents of the output, and
# with the reduction cut into pieces
@pytest.mark.parametrize('hw', [(1, 1), (1, 3), (1, 5), (2, 3), (1, 7), (3, 3), (7, 7), (5, 13), (8, 8)])
@pytest.mark.parametrize('n', [1, 5, 60])
def test_positions_in_runs_of_a_single_call(ops, dev, n, hw):
    c = 300
    gen = torch.Generator(device=dev).manual_seed(n * 100 + hw[0] * hw[1])
    g = torch.randn(n, c, *hw, device=dev, generator=gen)
    old = torch.rand(c, c, device=dev, generator=gen)
    old = old + old.t()
    a = g.double().permute(0, 2, 3, 1).reshape(-1, c)
    for out in (ops.factor_conv_g(g, 1., out=old.clone(), beta=1.),
                ops.factor_conv_a(g, 1, 1, 0, 1, False, 1., out=old.clone(), beta=1.)):
        _assert_float32_sum(out, a, a, 'positions %dx%dx%d' % ((n,) + hw), plus=old.double())
        assert torch.equal(out, out.t())


# rows of the correlations' rectangles: W - 2 inside, 1 at the edges (runs of 1 .. 12)
@pytest.mark.parametrize('w', [3, 5, 6, 7, 8, 9, 11, 13, 14])
@pytest.mark.parametrize('c', [66, 200])
def test_correlations_in_runs(ops, dev, c, w):
    gen = torch.Generator(device=dev).manual_seed(100 * c + w)
    x = torch.randn(3, c, 6, w, device=dev, generator=gen)
    x[1, c - 1, 2, w - 1], x[1, c - 1, 3, 0] = 1e18, -1e18
    a = torch.nn.functional.unfold(x.double(), 3, padding=1).permute(0, 2, 1).reshape(-1, 9 * c)
    single = ops.factor_conv_a(x, (3, 3), (1, 1), (1, 1), (1, 1), False, 1.)
    out = torch.full((9 * c,) * 2, float('nan'), device=dev)
    ops.factor_grouped([ops.factor_job('conv_a', x, 1., out, kernel_size=3, stride=1, padding=1,
                                       dilation=1)], dev)
    torch.cuda.synchronize()
    for got in (single, out):
        # (a block is the sum of up to 9 rectangles' products)
        _assert_float32_sum(got, a, a, 'correlations of %d channels of 6x%d' % (c, w))


@pytest.mark.parametrize('exponent', [-15, 0, 15])
def test_magnitudes(ops, dev, exponent):
    # columns of very different sizes: each keeps its own 24 bits
    gen = torch.Generator(device=dev).manual_seed(3)
    x = torch.randn(200, 300, device=dev, generator=gen)
    x *= 10. ** torch.linspace(exponent - 3, exponent + 3, 300, device=dev)
    out = ops.factor_linear(x, False, 1.)
    _assert_float32_sum(out, x.double(), x.double(), 'magnitudes around 1e%d' % exponent)


@pytest.mark.parametrize('rows', [20, 200])
def test_smallest_elements(ops, dev, rows):
    # columns from 1e-38 to 1e18: subnormal parts, subnormal products and elements of less than 24 bits
    gen = torch.Generator(device=dev).manual_seed(5)
    x = torch.randn(rows, 300, device=dev, generator=gen)
    x *= 10. ** torch.linspace(-38, 18, 300, device=dev, dtype=torch.float64).float()
    out = ops.factor_linear(x, False, 1.)
    _assert_float32_sum(out, x.double(), x.double(), 'columns from 1e-38 on')


@pytest.mark.parametrize('hw', [(4, 8), (7, 7)])
def test_infinities_and_overflow(ops, dev, hw):
    """What a float32 sum gives where it is not finite: inf with its sign, NaN only for
    NaN and for inf - inf; everything else as if those elements were not there."""
    gen = torch.Generator(device=dev).manual_seed(6)
    g = torch.rand(3, 300, *hw, device=dev, generator=gen) + 0.1
    g[1, 10, 1, 2] = float('inf')
    g[0, 140, -1, -3] = -float('inf')    # (brought twice by a padded run's last load)
    g[2, 270, -1, -1] = float('nan')
    g[:, 20] *= 1.1e25                        # its square overflows, nothing else does
    x = g.permute(0, 2, 3, 1).reshape(-1, 300).contiguous()
    want = x.cpu().t() @ x.cpu()
    for out in (ops.factor_conv_g(g, 1.), ops.factor_linear(x, False, 1.)):
        out = out.cpu()
        assert torch.equal(out.isnan(), want.isnan())
        assert torch.equal(out.isposinf(), want.isposinf())
        assert torch.equal(out.isneginf(), want.isneginf())
        ok = want.isfinite()
        assert ((out - want)[ok] / want[ok]).abs().max().item() < 1e-5


@pytest.mark.parametrize('hw', [(4, 8), (7, 7)])
def test_finite_elements_beyond_the_largest_bf16(ops, dev, hw):
    """3.4e38 is a float32 like any other, though its nearest bf16 number is infinite: its products
    with small elements are finite, and only its square overflows."""
    gen = torch.Generator(device=dev).manual_seed(7)
    g = 1e-30 * (torch.rand(3, 300, *hw, device=dev, generator=gen) + 0.1)
    g[1, 10, 1, 2] = 3.4e38
    g[0, 140, -1, -3] = -3.4e38
    g[2, 270, -1, -1] = 3.3962e38            # (the smallest ones that round up: 3.39618e38)
    x = g.permute(0, 2, 3, 1).reshape(-1, 300).contiguous()
    pointwise = ops.factor_conv_a(g, 1, 1, 0, 1, False, 1.)
    for out in (ops.factor_conv_g(g, 1.), ops.factor_linear(x, False, 1.), pointwise):
        a = x.double()
        large = (a.abs() > 1e38).any(0)
        finite = (a.t() @ a).abs() < 3.4e38
        assert torch.equal(out.isfinite(), finite) and int((~finite).sum()) == 3
        _assert_float32_sum(torch.where(finite, out, 0.), a * ~large, a, 'small elements by all',
                            where=finite & ~large[:, None])
        _assert_float32_sum(torch.where(finite, out, 0.), a * large, a, 'large elements by all',
                            where=finite & large[:, None])
    # (in sums of two operands too)
    Gi = torch.randn(300, 300, device=dev, generator=gen)
    Gi = Gi + Gi.t()
    w = 1e-30 * torch.randn(300, 200, device=dev, generator=gen)
    Gi[:, 5], Gi[5, :] = 1e-9, 1e-9
    w[5, 7] = 3.4e38
    want = Gi.double() @ w.double()
    ops.precondition_batched([Gi], [torch.eye(200, device=dev)], [w], [None])
    assert ((w.double() - want).abs() / (want.abs() + 1e-30)).max().item() < 1e-4


@pytest.mark.parametrize('rows', [3, 100])
def test_sums_just_below_the_largest_float32(ops, dev, rows):
    """2^64 - 2^54 is 2^64 in bf16: its square is finite, that of its leading part is not.  In a
    reduction in one rolled loop and in the pipelined one, with the sign, and in a sum of two."""
    big = 2. ** 64 - 2. ** 54
    x = torch.zeros(rows, 300, device=dev)
    x[1, 5], x[1, 290] = big, -big                                  # products of both signs
    x[0, 100], x[2, 100] = big * 0.75, big * 0.65                   # 0.985 of it
    x[0, 200], x[1, 200] = big, big                                 # overflows in float32 too
    want = x.double().t() @ x.double()
    over = want > 3.4028235e38
    assert int(over.sum()) == 1 and (want[5, 5] > 3.39e38) and (want[5, 290] < -3.39e38)
    for out in (ops.factor_linear(x, False, 1.), ops.factor_conv_g(x.t().reshape(1, 300, 1, rows), 1.)):
        assert torch.equal(out.isposinf(), over) and not out.isneginf().any() and not out.isnan().any()
        # (each product here is a float32 number up to its last bits)
        assert ((out.double() - want)[~over].abs() <= 2. ** -22 * want[~over].abs()).all()


def test_positive_terms(ops, dev):
    # no drift where all terms have one sign
    gen = torch.Generator(device=dev).manual_seed(4)
    x = torch.rand(4096, 256, device=dev, generator=gen)
    out = ops.factor_linear(x, False, 1.)
    want = x.double().t() @ x.double()
    assert ((out.double() - want) / want).mean().abs().item() < 2. ** -22


@pytest.mark.parametrize('shape', [(1, 2), (129, 258), (300, 77), (128, 513)])
def test_preconditioned_gradient(ops, dev, shape):
    dG, dA = shape
    gen = torch.Generator(device=dev).manual_seed(dG + dA)
    Gi = torch.randn(dG, dG, device=dev, generator=gen)
    Ai = torch.randn(dA, dA, device=dev, generator=gen)
    Gi, Ai = Gi + Gi.t(), Ai + Ai.t()
    w = torch.randn(dG, dA - 1, device=dev, generator=gen)
    b = torch.randn(dG, device=dev, generator=gen)
    full = torch.cat([w, b[:, None]], 1).double()
    want = Gi.double() @ full @ Ai.double()
    ops.precondition_batched([Gi], [Ai], [w], [b])
    got = torch.cat([w, b[:, None]], 1).double()
    # two products, each a float32 sum; the bound in the 2-norm
    mass = Gi.double().abs() @ full.abs() @ Ai.double().abs()
    steps = 2 * (dG // 16 + dA // 16 + 2) + 8
    assert (got - want).abs().div(mass * 2. ** -23 * steps).max().item() <= 1.
