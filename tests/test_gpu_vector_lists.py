"""The element-wise engine calls over lists whose tensors travel as a kernel argument: short and long
lists, more tensors than one launch holds, sizes next to the edges of a workgroup's block, views that
are not 16-byte aligned, against the same arithmetic in torch float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
# one rounding per product and sum (at most three of them) of values up to 8 in size
TOL = 4 * 8 * 2. ** -24
SIZES = [1, 3, 4, 5, 1023, 1024, 1025, 2047, 2048, 2052, 4095, 4096, 4097, 4100, 8192, 40000]


@pytest.fixture(scope='module')
def ops():
    from torchsso import _ops
    return _ops


@pytest.fixture(scope='module')
def dev():
    return torch.device('cuda:0')


def tensors(count, seed, dev, positive=False):
    """`count` tensors of the sizes above, every third one starting 4 bytes past an aligned address"""
    g = torch.Generator().manual_seed(seed)
    out = []
    for i in range(count):
        n = SIZES[(i * 7 + count) % len(SIZES)]
        t = torch.randn(n + 1, generator=g).clamp_(-4, 4)
        t = (t.abs() + 0.1 if positive else t).to(dev)
        out.append(t[1:] if i % 3 == 0 else t[:-1].clone())
    return out


def same(got, want):
    for a, b in zip(got, want):
        assert (a.double() - b).abs().max().item() <= TOL


@pytest.mark.parametrize('count', [1, 2, 8, 9, 64, 65, 130])
def test_lists_against_float64(ops, dev, count):
    x, y = tensors(count, 1, dev), tensors(count, 2, dev)
    for a, b in ((0.25, 0.75), (0.5, 0.)):
        ref = [a * u.double() + b * v.double() for u, v in zip(x, y)]
        out = [v.clone() if i % 2 else v for i, v in enumerate(y)]
        y = [v.clone() for v in y]
        ops.axpby_batched(x, out, a, b)
        same(out, ref)

    p, g, m = tensors(count, 3, dev), tensors(count, 4, dev), tensors(count, 5, dev)
    lr, mom, wd = [0.1] * count, [0.9 if i % 4 else 0. for i in range(count)], [0.01 * (i % 2) for i in range(count)]
    g64 = [gi.double() + w * pi.double() for gi, pi, w in zip(g, p, wd)]
    g64 = [mu * mi.double() + gi if mu else gi for gi, mi, mu in zip(g64, m, mom)]
    p64 = [pi.double() - 0.1 * gi for pi, gi in zip(p, g64)]
    m64 = [gi if mu else mi.double() for gi, mi, mu in zip(g64, m, mom)]
    ops.sgd_update_batched(p, g, [mi if mu else None for mi, mu in zip(m, mom)], lr, mom, wd)
    same(p, p64)
    same(g, g64)
    same(m, m64)

    v = tensors(count, 6, dev, positive=True)
    out = [torch.empty_like(t) for t in v]
    ops.sqrt_batched(v, out)
    same(out, [t.double().sqrt() for t in v])


# 130: with tensors of more blocks than a tensor's share of a launch, accessed by 4 and by 16 bytes
@pytest.mark.parametrize('count', [8, 9, 64, 65, 130])
def test_other_operations_against_float64(ops, dev, count):
    def lists(seed, positive=False):
        out = tensors(count, seed, dev, positive)
        if count == 130:
            big = torch.randn(300000, generator=torch.Generator().manual_seed(seed)).clamp_(-4, 4)
            big = (big.abs() + 0.1 if positive else big).to(dev)
            out[1], out[count - 2] = big, big[1:70002]
            assert out[1].data_ptr() % 16 == 0 and out[count - 2].data_ptr() % 16 == 4
        return [t.clone() if i % 5 == 1 else t for i, t in enumerate(out)]      # (aligned next to others that are not)

    inv, grad = lists(11, True), lists(12)
    want = [a.double() * b.double() for a, b in zip(inv, grad)]
    ops.diag_precondition_batched(inv, grad)
    same(grad, want)

    x, y = lists(13), lists(14)
    want = [torch.maximum(a.double(), b.double()) for a, b in zip(x, y)]
    ops.max_batched(x, y)
    same(y, want)

    ema = lists(15, True)
    for use_sqrt in (False, True):
        out = [torch.full_like(t, float('nan')) for t in ema]
        ops.diag_inverse_batched(ema, out, [1. + i % 3 for i in range(count)], use_sqrt)
        same(out, [1 / ((t.double().sqrt() if use_sqrt else t.double()) + 1. + i % 3) for i, t in enumerate(ema)])

    mean, std, noise = lists(16), lists(17, True), lists(18)
    scales = [0.25 * (i % 4) for i in range(count)]
    want = [m.double() + s * n.double() * d.double() for m, d, n, s in zip(mean, std, noise, scales)]
    ops.diag_sample_batched(mean, std, noise, scales)
    same(noise, want)
