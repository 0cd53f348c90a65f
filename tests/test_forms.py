"""How long the factor of an inverse is bound to the form that a recorded graph was captured with
(KronCurvature._form_captured): as long as it lies in the buffers that the graph knows."""
import copy
import pickle

import pytest
import torch
import torch.nn as nn

from torchsso.curv.cov.linear import KronCovLinear


def bound():
    c = KronCovLinear(nn.Linear(3, 2))
    c.ema = [torch.eye(4), torch.eye(2)]
    c._inv = [None, torch.eye(2)]
    c._inv_factors = [torch.eye(4), None]
    c._a_in_halves = True
    c._form_captured = True
    return c


@pytest.mark.parametrize('value', [None, [torch.eye(4), torch.eye(2)]])
def test_inverses_from_outside_are_in_other_buffers(value):
    c = bound()
    c.inv = value
    assert c._form_captured is None and not c._a_in_halves


def test_loaded_state_is_in_other_buffers():
    c = bound()
    c._inv[0] = torch.eye(4)         # (formed: a host tensor's factor is not multiplied here)
    c.load_state_dict(c.state_dict())
    assert c._form_captured is None and not c._a_in_halves


def test_an_inversion_keeps_the_form_with_the_buffer():
    c = bound()
    c.factored_inverse_min_dim = 4
    factor = c._inv_factors[0]
    _, facs, _ = c._inverse_outputs(False)
    assert facs[0] is factor and c._form_captured is True and c._a_in_halves
    c._inverse_outputs(True)         # (explicit inverses, beside their Cholesky factors)
    assert c._inv_factors[0] is None and c._form_captured is None and not c._a_in_halves


@pytest.mark.parametrize('copied', [copy.deepcopy, lambda c: pickle.loads(pickle.dumps(c))])
def test_copies_have_buffers_of_their_own(copied):
    c = bound()
    d = copied(c)
    assert c._form_captured is True
    assert d._form_captured is None and d._a_in_halves
    assert torch.equal(d._inv_factors[0], c._inv_factors[0]) and d._inv_factors[0] is not c._inv_factors[0]
