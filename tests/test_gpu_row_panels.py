"""Row panels of the blocked factorisation in launches of more than 64 tiles (a workgroup to a tile)
and of fewer (four to a tile), at ragged last blocks, in a sweep and outside of one, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
U = 2. ** -24


@pytest.fixture(scope='module')
def ops():
    from torchsso import _ops
    return _ops


@pytest.fixture(scope='module')
def dev():
    return torch.device('cuda:0')


def matrix(n, dev):
    g = torch.Generator().manual_seed(n)
    x = torch.randn(2 * n + 8, n, generator=g, dtype=torch.float64)
    return (x.t() @ x / (2 * n + 8) + 0.1 * torch.eye(n, dtype=torch.float64)).float().to(dev)


# (matrices, sizes): row panels of 33 * 2 and 33 tiles in a sweep; of 110 * 3, 110 * 2 and 110 outside
# of one (more than 765 tiles in all); a single matrix with four workgroups to every tile
@pytest.mark.parametrize('count,sizes', [(33, (257, 300, 383, 384)), (33, (258, 288, 289, 321)),
                                         (110, (385, 416, 511, 512)), (110, (386, 449, 450, 481)),
                                         (1, (641,)), (1, (897,))])
def test_inverse_and_factor_against_float64(ops, dev, count, sizes):
    distinct = [matrix(n, dev) for n in sizes]
    mats = [distinct[i % len(sizes)] for i in range(count)]
    us, info = ops.cholesky_upper_batched(mats)
    xs, info2 = ops.damped_inverse_batched(mats, [0.] * count)
    assert not info.any().item() and not info2.any().item()
    eigs = [torch.linalg.eigvalsh(m.double().cpu()) for m in distinct]
    for i, m in enumerate(mats):
        n, m64, eig = m.shape[0], m.double(), eigs[i % len(sizes)]
        # backward error of a Cholesky factor computed in float32, (n + 1) u |U|^T |U| with
        # | |U|^T |U| |_F <= n^(1/2) |M|_F; the inverse's is that times the condition number, twice
        bound = (n + 1) * U * n ** 0.5
        u, x = us[i].double(), xs[i].double()
        assert torch.equal(us[i], us[i].triu())
        assert ((u.t() @ u - m64).norm() / m64.norm()).item() <= bound
        rest = x @ m64 - torch.eye(n, dtype=torch.float64, device=dev)
        assert (rest.norm() / n ** 0.5).item() <= 2 * bound * (eig[-1] / eig[0]).item()
        assert torch.equal(xs[i], xs[i].t())


# panels of 66 tiles in a sweep, of 240, 160 and 80 outside of one
@pytest.mark.parametrize('count,sizes', [(33, (257, 300, 383, 384)), (80, (385, 416, 511, 512))])
def test_matrices_of_any_magnitude(ops, dev, count, sizes):
    """The same matrices times 2^-116 (many entries below 2^-118), 2^90 and 2^106 (beyond what the panels' elements
    are multiplied with: computed in another way): errors as those of the matrices themselves, but for the few
    entries that are rounded to multiples of 2^-149."""
    distinct = [matrix(n, dev) for n in sizes]
    eye = [torch.eye(n, dtype=torch.float64, device=dev) for n in sizes]

    def errors(exponent):
        mats = [distinct[i % len(sizes)] * 2. ** exponent for i in range(count)]
        us, info = ops.cholesky_upper_batched(mats)
        xs, info2 = ops.damped_inverse_batched(mats, [0.] * count)
        assert not info.any().item() and not info2.any().item()
        out = []
        for i in range(count):
            m, u, x = mats[i].double(), us[i].double(), xs[i].double()
            out += [((u.t() @ u - m).norm() / m.norm()).item(), (x @ m - eye[i % len(sizes)]).norm().item()]
        return torch.tensor(out)

    base = errors(0)
    for exponent in (-116, 90, 106):
        assert (errors(exponent) / base).max().item() < 2.
