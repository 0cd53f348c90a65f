"""Which device and stream the queued factor products run on, and what waits for what (torchsso._lanes), with
stand-ins for the streams and events of two devices."""
import types

import pytest
import torch

from torchsso import _lanes


class Stream(object):
    made = 0

    def __init__(self, device=None, handle=None):
        Stream.made += 1
        self.device_index = device if isinstance(device, int) else device.index
        self.cuda_stream = 1000 + Stream.made if handle is None else handle
        self.stream_id, self.device_type = self.cuda_stream, 1

    def __eq__(self, other):
        return (self.device_index, self.cuda_stream) == (other.device_index, other.cuda_stream)

    __hash__ = None

    def wait_event(self, event):
        event.log.append(('wait', self, event))

    def synchronize(self):
        pass


class World(object):
    """Two devices with a null stream each; records what is launched and ordered."""

    def __init__(self):
        self.device, self.streams, self.log = 0, [Stream(0, 0), Stream(1, 0)], []
        world = self

        class Event(object):
            def __init__(self):
                self.device, self.log = None, world.log

            def record(self, stream):
                # (an event belongs to the device of its first record)
                assert self.device in (None, stream.device_index), 'event of another device'
                self.device = stream.device_index
                world.log.append(('record', stream, self))

            def query(self):
                return True

        class device(object):
            def __init__(self, i):
                self.i = i

            def __enter__(self):
                self.before, world.device = world.device, self.i

            def __exit__(self, *args):
                world.device = self.before

        self.torch = types.SimpleNamespace(
            device=torch.device,
            _C=types.SimpleNamespace(_cuda_getCurrentStream=lambda i: ident(self.streams[i])),
            cuda=types.SimpleNamespace(Stream=Stream, Event=Event, device=device,
                                       current_device=lambda: self.device,
                                       current_stream=lambda i: self.streams[i]))

        def ident(st):
            return st.stream_id, st.device_index, st.device_type

    def factor_grouped(self, jobs, device, stream=None):
        # (without a stream: the current one of `device`; handle 0 is the null stream of the current device)
        st = self.streams[device.index] if stream is None else stream
        at = self.device if st.cuda_stream == 0 else st.device_index
        self.log.append(('call', st, [job.C for job in jobs]))
        assert at == device.index, 'a product of device %d on device %d' % (device.index, at)

    def calls(self):
        return [(st, c) for kind, st, c in self.log if kind == 'call']


@pytest.fixture
def world(monkeypatch):
    w = World()
    monkeypatch.setattr(_lanes, 'torch', w.torch)
    monkeypatch.setattr(_lanes._ops, 'factor_grouped', w.factor_grouped)
    monkeypatch.setattr(_lanes._ops, 'bn_diag_cov_batched', lambda jobs, device: None)
    monkeypatch.setattr(_lanes._hip, 'order_streams', lambda i, a, b: w.log.append(('order', a, b)))
    for name in ('_deferred', '_calls', '_inflight', '_streams', '_pending', '_stream_objects'):
        monkeypatch.setattr(_lanes, name, {})
    monkeypatch.setattr(_lanes, '_events', type(_lanes._events)())
    monkeypatch.setattr(_lanes, '_count', 2)
    return w


def defer(device, key, address, **kw):
    job = types.SimpleNamespace(C=address, C_prev=None)
    _lanes.defer(torch.device('cuda', device), key, job, (), **kw)


def test_events_are_recorded_on_their_own_device(world):
    for step in range(3):
        for i in (0, 1):
            world.device = i        # (two programs, or one that goes from device to device)
            defer(i, ('A', i), 100 + i)
            defer(i, ('G', i), 200 + i, backward=True)      # (runs the input factors on a side stream)
            _lanes.join(torch.device('cuda', i))
    assert [(st.device_index, c) for st, c in world.calls()] == 3 * [(0, [100]), (0, [200]), (1, [101]), (1, [201])]


def test_products_of_two_devices_keep_to_their_devices(world):
    for step in range(3):
        for i in (0, 1):
            defer(i, ('A', i), 100 + i)
            defer(i, ('G', i), 200 + i, backward=True)      # (runs the input factors on a side stream)
        _lanes.join()
    assert [(st.device_index, c) for st, c in world.calls()] == 3 * [(0, [100]), (1, [101]), (0, [200]), (1, [201])]
    assert world.device == 0


def test_a_hooks_stream_waits_for_the_products_a_reader_runs(world):
    """Its next pass may write the same factors, and the allocator hands what the products read out again there."""
    reader, hook = world.streams[0], Stream(0)
    world.streams[0] = hook
    defer(0, ('A', 0), 100)
    world.streams[0] = reader
    _lanes.join()
    (call, _), = world.calls()
    at = [kind for kind, *_ in world.log].index('call')
    behind = [(entry[1], entry[2]) for entry in world.log[at:] if entry[0] == 'order']
    recorded = {id(event): st for kind, st, event in world.log[at:] if kind == 'record'}
    behind += [(st, recorded[id(event)]) for kind, st, event in world.log[at:] if kind == 'wait']
    assert (hook, call) in behind
    assert call == reader or (reader, call) in behind
