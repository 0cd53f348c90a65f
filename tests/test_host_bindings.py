"""The native host side of the engine calls: what it packs, what it refuses, and that the Python path
names the tensor at fault."""
import ctypes
import struct

import pytest
import torch

from torchsso import _hip, _host, _ops


def test_values_are_packed_as_the_library_takes_them():
    assert _host.ints([1, -2, True]) == struct.pack('=3i', 1, -2, 1)
    assert _host.int64s((2 ** 40,)) == struct.pack('=q', 2 ** 40)
    assert _host.floats([1, 0.1, -2.5]) == struct.pack('=3f', 1, 0.1, -2.5)
    assert _host.numels([torch.ones(3, 4), torch.ones(0)]) == struct.pack('=2q', 12, 0)
    assert _host.ints([]) == b''
    assert _host.ints([2 ** 31]) is None            # (does not fit)
    with pytest.raises(TypeError):
        _host.ints([1.5])
    with pytest.raises(TypeError):
        _host.floats(['1'])


def test_tensors_the_engine_cannot_take_are_refused_and_named():
    host = torch.ones(3)
    assert _host.pointer(host) is None and _host.pointer(3) is None and _host.pointer(None) is None
    assert _host.pointers([None], True) == bytes(8) and _host.pointers([None], False) is None
    assert _host.pointers([host], True) is None
    with pytest.raises(_hip.KfacHipError, match='x 0 is on cpu'):
        _hip.ptr_array([host], 'x')
    with pytest.raises(_hip.KfacHipError, match='x 0 is None'):
        _hip.ptr_array([None], 'x')
    job = _hip.FactorJob()
    assert not _host.update_job(ctypes.addressof(job), host, host, None, 1., 0.)
    with pytest.raises(_hip.KfacHipError, match='input is on cpu'):
        _ops.factor_job_update(job, host, 1., host)


@pytest.mark.gpu
def test_addresses_and_jobs_of_device_tensors():
    dev = torch.device('cuda:0')
    a, b = torch.ones(6, 5, device=dev), torch.ones(7, device=dev)
    assert _host.pointers([a, None, b[2:], torch.nn.Parameter(b)], True) == struct.pack(
        '=4Q', a.data_ptr(), 0, b.data_ptr() + 8, b.data_ptr())
    for bad in (a.t(), a.double(), a.half(), a[:, 1]):
        assert _host.pointer(bad) is None
        with pytest.raises(_hip.KfacHipError, match='t 1'):
            _hip.ptr_array([a, bad], 't')
    out, prev = torch.ones(5, 5, device=dev), torch.ones(5, 5, device=dev)
    job = _ops.factor_job('linear', a, 1., out)
    for beta, p, want in ((0., None, None), (0.5, None, out), (0.25, prev, prev)):
        _ops.factor_job_update(job, a, 2., out, beta, p)
        assert (job.x, job.C, job.alpha, job.beta) == (a.data_ptr(), out.data_ptr(), 2., beta)
        assert job.C_prev == (None if want is None else want.data_ptr())
    assert _host.jobs([ctypes.addressof(job)] * 2) == bytes(job) * 2


@pytest.mark.gpu
def test_a_lazily_copied_tensor_is_not_written_through():
    dev = torch.device('cuda:0')
    for through in ('call', 'job'):
        a = torch.zeros(8, 8, device=dev)
        b = torch._lazy_clone(a)
        x = torch.ones(3, 8, device=dev)
        if through == 'call':
            _ops.axpby_batched([torch.full((8, 8), 3., device=dev)], [b], 1., 0.)
        else:
            job = _ops.factor_job('linear', x, 1., x.new_empty(8, 8))
            _ops.factor_job_update(job, x, 1., b)
            _ops.factor_grouped([job], dev)
        assert not a.any().item() and bool((b == 3.).all())


@pytest.mark.gpu
def test_order_of_two_streams():
    dev = torch.device('cuda:0')
    x = torch.zeros(1 << 24, device=dev)
    first, second = torch.cuda.Stream(dev), torch.cuda.Stream(dev)
    torch.cuda.synchronize()
    for k in range(1, 6):
        with torch.cuda.stream(first):
            for _ in range(20):
                x.add_(1.)
        _hip.order_streams(0, second, first)
        with torch.cuda.stream(second):
            y = x.clone()
        _hip.order_streams(0, first, second)
        torch.cuda.synchronize()
        assert bool((y == 20. * k).all())
    with pytest.raises(TypeError):
        _host.order(0, 0)
