"""The diagonal block of the blocked Cholesky at the sizes where its strips, steps and columns end,
on its own (n <= 128) and with the panel above it pending (n > 128), against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
U = 2. ** -24

SIZES = [1, 2, 3, 5, 30, 31, 32, 33, 34, 35, 62, 63, 64, 65, 66, 94, 95, 96, 97, 98, 126, 127, 128,
         129, 130, 131, 132, 159, 160, 161, 191, 192, 193, 223, 224, 225, 254, 255, 256, 257, 261]


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


@pytest.mark.parametrize('n', SIZES)
def test_factor_and_inverse_against_float64(ops, dev, n):
    m = matrix(n, dev)
    # (what lies below the diagonal is not read)
    poisoned = torch.where(torch.ones_like(m).triu().bool(), m, torch.full_like(m, float('nan')))
    (u,), info = ops.cholesky_upper_batched([poisoned])
    (x,), info2 = ops.damped_inverse_batched([m], [0.])
    assert info.item() == 0 and info2.item() == 0
    m64 = m.double()
    # backward error of a Cholesky factor computed in float32: (n + 1) u |U|^T |U| element by
    # element, and | |U|^T |U| |_F <= n^(1/2) |M|_F; the inverse's relative error is that times the condition
    # number, once more for the product with the inverse factor
    bound = (n + 1) * U * n ** 0.5
    assert torch.equal(u, u.triu())
    assert ((u.double().t() @ u.double() - m64).norm() / m64.norm()).item() <= bound
    ref = torch.linalg.inv(m64)
    assert ((x.double() - ref).norm() / ref.norm()).item() <= 2 * bound * torch.linalg.cond(m64).item()
    assert torch.equal(x, x.t())


@pytest.mark.parametrize('n', [1, 33, 97, 128, 200, 256, 300])
def test_the_first_bad_pivot_is_reported(ops, dev, n):
    at = sorted({k for k in (0, 1, 30, 31, 32, 33, 64, 95, 96, 127, 128, 129, 160, 255, n - 1) if k < n})
    mats = []
    for k in at:
        m = matrix(n, dev)
        m[k, k] = -1.
        mats.append(m)
    mats.append(matrix(n, dev))
    _, info = ops.cholesky_upper_batched(mats)
    assert info.cpu().tolist() == [k + 1 for k in at] + [0]


def test_values_that_are_not_finite_end_and_are_reported(ops, dev):
    for value in (float('nan'), float('inf'), -float('inf')):
        mats = []
        for k in (0, 31, 40, 127, 130, 255):
            m = matrix(256, dev)
            m[k, k] = value
            mats.append(m)
        outs, info = ops.damped_inverse_batched(mats + [matrix(256, dev)], [0.] * 7)
        assert info[6].item() == 0 and bool(torch.isfinite(outs[6]).all())
        if value != float('inf'):
            assert (info[:6] > 0).all()


def test_entries_close_to_the_largest_float(ops, dev):
    """A second block that the first one explains but for 1e-3: the sums of squares that the pending panel takes
    from it lie above 0.995 of the largest float32."""
    g = torch.Generator().manual_seed(5)
    x = torch.randn(600, 128, generator=g, dtype=torch.float64)
    x = torch.cat([x, x + 0.03 * torch.randn(600, 128, generator=g, dtype=torch.float64)], 1)
    x = x / x.norm(dim=0)
    m = (x.t() @ x * (0.9995 * torch.finfo(torch.float32).max)).float().to(dev)
    (u,), info = ops.cholesky_upper_batched([m])
    assert info.item() == 0 and bool(u.isfinite().all())
    m64, u64 = m.double(), u.double()
    assert ((u64.t() @ u64 - m64).norm() / m64.norm()).item() <= 257 * U * 16
