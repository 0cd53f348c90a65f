"""Native shape checks of the batched calls against the wrappers' own loops (on host tensors: nothing is
launched)."""
import pytest
import torch

from torchsso import _hip, _host, _ops


@pytest.mark.parametrize('shapes', [[], [(3, 3)], [(1, 1), (700, 700)], [(3, 3), (3, 4)], [(9,)], [(2, 2, 2)], [()],
                                    [(0, 0)]])
def test_square_dims(monkeypatch, shapes):
    mats = [torch.empty(s) for s in shapes]
    expected = [s[0] for s in shapes] if all(len(s) == 2 and s[0] == s[1] for s in shapes) else None
    assert _host.square_dims(mats) == expected == _host.square_dims(tuple(mats))
    if expected is None:
        with pytest.raises(_hip.KfacHipError, match='not square'):
            _ops._square_dims(mats, 'matrix')
    else:
        assert _ops._square_dims(mats, 'matrix') == expected
    assert _host.square_dims([torch.ones(2, 2), None]) is None


@pytest.mark.parametrize('weight, bias', [((5, 7), None), ((5, 6), (5,)), ((5, 2, 3), (5,)), ((5, 7), (5,)),
                                          ((5, 6), (4,)), ((7, 5), None), ((35,), None), ((5, 6), None)])
def test_kron_dims(monkeypatch, weight, bias):
    G, A = torch.empty(5, 5), torch.empty(7, 7)
    lists = ([G, G], [A, A], [torch.empty(5, 7), torch.empty(weight)],
             [None, None if bias is None else torch.empty(bias)])

    def outcome():
        try:
            dG, dA = _ops._kron_dims(*lists, 'call')
            return list(dG), list(dA)
        except _hip.KfacHipError as e:
            return str(e)
    native = outcome()
    fits = _host.kron_dims(*lists)
    monkeypatch.setattr(_hip, '_host', None)
    assert outcome() == native
    assert (fits is None) == isinstance(native, str)
    assert fits is None or fits == ([5, 5], [7, 7])


def test_outputs_fit():
    x, y, bad = torch.empty(3, 3), torch.empty(3, 3), torch.empty(3, 2)
    fit = _host.outputs_fit
    assert fit([x, x], [y, None], [None, y], True)
    assert not fit([x], [y], [y], True) and not fit([x], [None], [None], True)
    assert fit([x, x], [y, y], [y, None], False) and not fit([x], [None], [y], False)
    for flag in (True, False):
        assert not fit([x], [bad], [None], flag) and not fit([x], [torch.empty(9)], [None], flag)
        assert not fit([x, x], [y], [None, None], flag)
        assert fit([], [], [], flag)
    assert not fit([x], [None], [bad], True) and not fit([x], [y], [bad], False)
    with pytest.raises(TypeError):
        fit(3, [y], [None], True)


def test_vectors_and_sums_on_the_host():
    made = _ops.vectors(torch.empty(2, dtype=torch.float64), 5, 2)
    assert [tuple(v.shape) for v in made] == [(5,), (5,)]
    assert all(v.dtype == torch.float32 and not v.requires_grad for v in made)
    assert _ops.vectors(made[0], 0, 1)[0].numel() == 0
    # (what the engine cannot take is left to the wrapper, which raises)
    assert _host.rowsq_sum(0, torch.ones(2, 3, 4), 3, None, None) is None
    with pytest.raises(TypeError):
        _host.rowsq_sum(0, torch.ones(2, 3, 4), 3)
