"""The two ways a batch is inverted (csrc/inverse.hip): batches whose tiles fit beside a diagonal
block by the sweep, larger ones by the recursive triangular inverse.  The same matrices go both
ways, the second time beside a matrix whose tiles alone are over the line, in each form of
the result."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D = torch.float64

# one block, tile edges, ragged last blocks, several widths in a batch, more tiles in a step than
# compute units, and a row panel of more than 64 tiles
BATCHES = [(130,), (128, 256), (129, 255, 257, 384, 385), (1, 127, 1000, 641, 37),
           (2945, 300), (1153, 1300, 1281, 1408, 1025, 1100, 1200)]


@pytest.fixture(scope='module')
def dev():
    return torch.device('cuda:0')


@pytest.fixture(scope='module')
def ops():
    from torchsso import _ops
    return _ops


@pytest.fixture(scope='module')
def large(dev):
    return 2 * torch.eye(39 * 128, device=dev)          # 780 tiles


@pytest.mark.parametrize('form', ['inverse', 'factor', 'std'])
@pytest.mark.parametrize('sizes', BATCHES)
def test_sweep_and_recursive_inverse(ops, dev, large, sizes, form):
    gen = torch.Generator().manual_seed(sum(sizes))
    mats = []
    for n in sizes:
        a = torch.randn(n, n + 8, generator=gen).to(dev)
        mats.append(a @ a.t() / (n + 8) + 0.05 * torch.eye(n, device=dev))
    damping = 1e-3

    def invert(As):
        nan = lambda: [torch.full_like(a, float('nan')) for a in As]
        # (every matrix the A of a layer whose G is a multiple of the identity, 1x1)
        Gs = [torch.ones(1, 1, device=dev) for _ in As]
        Gi = [torch.empty(1, 1, device=dev) for _ in As]
        none = [None] * len(As)
        damp = [damping] * len(As)
        if form == 'factor':
            out = nan()
            info = ops.pi_damped_inverse_factored_batched(As, Gs, damp, none, Gi, out, none)
            res = [(y,) for y in out]
        else:
            out, std = nan(), nan() if form == 'std' else none
            info = ops.pi_damped_inverse_std_batched(As, Gs, damp, out, Gi, std, none)
            res = [(x,) if w is None else (x, w) for x, w in zip(out, std)]
        assert int(info.abs().sum()) == 0
        return res

    alone, beside = invert(mats), invert(mats + [large])
    for m, one, two in zip(mats, alone, beside):
        n = m.shape[0]
        shift = (damping * m.double().diagonal().mean()).sqrt()
        x = m.double() + shift * torch.eye(n, device=dev, dtype=D)
        ref = torch.linalg.inv(x)
        if form == 'factor':
            want = (torch.linalg.inv(torch.linalg.cholesky(x).mT),)
        else:
            want = (ref, torch.linalg.cholesky(ref).mT)
        # rounding of n-term float32 sums, as the condition number magnifies it: of random sign,
        # sqrt(n) u per entry (a Cholesky factor of the inverse: another factor of 2)
        cond = (torch.linalg.matrix_norm(x, 1) * torch.linalg.matrix_norm(ref, 1)).item()
        bound = 2 * n ** 0.5 * 2. ** -24 * cond
        for got, other, w in zip(one, two, want):
            for y in (got, other):
                err = ((y.double() - w).norm() / w.norm()).item()
                assert err < bound, (sizes, n, err, bound)
            if w is ref:
                assert torch.equal(got, got.t())
            else:
                assert torch.equal(got, torch.triu(got)) and torch.equal(other, torch.triu(other))
