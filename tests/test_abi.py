"""The C-ABI library: it loads without a GPU, exports every function that
include/kfac_hip.h declares, the ctypes binding covers exactly those, and the
argument checks that need no device reject bad input with an error code."""
import ctypes
import os
import re

import pytest

from torchsso import _hip

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, 'include', 'kfac_hip.h')


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r'/\*.*?\*/', '', text, flags=re.S)
    return sorted(set(re.findall(r'\b(kfac_[a-z0-9_]+)\s*\(', text)))


def test_library_is_built_and_loads():
    assert os.path.exists(_hip.lib_path()), 'run python pytorch-sso_amd/build_ext.py'
    lib = _hip.load()
    assert lib.kfac_abi_version() == 2


def test_every_declared_symbol_is_exported_and_bound():
    names = declared_functions()
    assert len(names) >= 15
    raw = ctypes.CDLL(_hip.lib_path())
    for n in names:
        assert hasattr(raw, n), 'header declares %s but the library does not export it' % n
    assert sorted(_hip.signatures()) == names


def test_header_cites_the_reference_for_each_entry_point():
    text = open(HEADER).read()
    for n in declared_functions():
        if n.endswith(('_workspace_bytes', '_executed_flops')) or n == 'kfac_abi_version':
            continue
        idx = text.index(n + '(')
        comment = text[:idx].rsplit('/*', 1)[1]
        flat = ' '.join(comment.replace('*', ' ').split())
        if 'no counterpart in the reference' in flat:
            # says so instead of citing, and names the callers it exists for
            assert 'cannot allocate' in flat
            continue
        assert re.search(r'\.py:\d+', comment), '%s: no reference file:line in its comment' % n


def test_workspace_queries_need_no_device():
    lib = _hip.load()
    assert lib.kfac_factor_workspace_bytes(4608, 1568) >= 0
    assert lib.kfac_factor_workspace_bytes(64, 401408) > 0          # split-k partials
    dims = _hip.int_array([100, 300])
    assert lib.kfac_inverse_workspace_bytes(2, dims) >= 4 * (100 * 100 + 300 * 300)
    assert lib.kfac_precondition_workspace_bytes(1, _hip.int_array([10]), _hip.int_array([20])) >= 800
    assert lib.kfac_vector_workspace_bytes(3) > 0


def test_argument_errors_are_codes_not_crashes():
    lib = _hip.load()
    # null pointers / bad sizes are rejected before anything touches a device
    assert lib.kfac_factor_linear(None, 8, 4, 4, 1, 1.0, 0.0, None, None, None, 0, None) == 1
    assert lib.kfac_factor_conv_g(None, 1, 1, 1, 1, 1.0, 0.0, None, None, None, 0, None) == 1
    assert lib.kfac_rowsq_sum(None, 1, 1, 1, None, None, None, None) == 1
    assert lib.kfac_bn_diag_cov(None, 1, 1, 1, None, 1.0, None, None, None, 0, None) == 1
    assert lib.kfac_bn_diag_cov_workspace_bytes(32, 64) == 32 * 64 * 4
    assert lib.kfac_bn_diag_cov_workspace_bytes(0, 64) == 0
    # the entry point with built-in scratch refuses what does not fit it, before any launch
    assert lib.kfac_static_workspace_bytes() == 8 << 20
    big = _hip.int_array([2000])
    one = (ctypes.c_void_p * 1)(1 << 20)
    two = (ctypes.c_void_p * 1)(2 << 20)
    assert lib.kfac_inverse_workspace_bytes(1, big) > lib.kfac_static_workspace_bytes()
    assert lib.kfac_damped_inverse_batched_static(1, big, one, None, two, one, None) == 4
    assert lib.kfac_damped_inverse_batched_static(1, big, one, None, one, one, None) == 1
    with pytest.raises(_hip.KfacHipError):
        _hip.check(2, 'x')


def _job(kind, c, rows, H=1, W=1, k=1, stride=1, pad=0, x=256, C=512):
    j = _hip.FactorJob()
    j.kind, j.c, j.rows, j.H, j.W = kind, c, rows, H, W
    j.kh = j.kw = k
    j.sh = j.sw = stride
    j.ph = j.pw = pad
    j.dh = j.dw = 1
    j.alpha, j.x, j.C = 1., x, C
    return j


@pytest.mark.parametrize('n,c,side', [(32, 128, 28), (32, 256, 14), (64, 128, 14)])
def test_correlation_plan_fits_one_round(n, c, side):
    """A correlation launch of 128-wide tiles holds about as many items as two resident
    workgroups per compute unit (512), the last of each job rounded up: their number follows from
    the scratch, one c x c partial per split and 45 block sums."""
    lib = _hip.load()
    size = lib.kfac_factor_conv_a_workspace_bytes(n, c, side, side, 3, 3, 1, 1, 1, 1, 1, 1, 0)
    splits = size // (4 * c * c) - 45
    tiles = (-(-c // 128)) ** 2
    assert 256 < splits * tiles <= 512 + 64 // 2


@pytest.mark.parametrize('n,c,side', [(39, 400, 16), (2, 324, 52)])
def test_correlation_plan_of_many_tiles(n, c, side):
    """Where whole splits make a good deal more than one round of items in any case, they are shorter."""
    size = _hip.load().kfac_factor_conv_a_workspace_bytes(n, c, side, side, 3, 3, 1, 1, 1, 1, 1, 1, 0)
    assert (size // (4 * c * c) - 45) * (-(-c // 128)) ** 2 > 1.375 * 512


@pytest.mark.parametrize('d,rows,splits', [(1600, 8192, 5), (2176, 8192, 3), (2304, 8192, 4),
                                           (2304, 2000, 2)])
def test_splits_of_a_single_product(d, rows, splits):
    """Two workgroups per compute unit are resident: three on the fullest one pay off where they are a
    good deal shorter than two (2304 rows of a factor), not in exchange for little."""
    tiles = -(-d // 128) * (-(-d // 128) + 1) // 2
    assert _hip.load().kfac_factor_workspace_bytes(d, rows) == 4 * 128 * 128 * tiles * splits


def test_grouped_factor_plan_needs_no_device():
    """The plan of a grouped call (scratch, executed flops) is host arithmetic; bad lists are
    refused before anything is launched."""
    lib = _hip.load()
    jobs = [_job(_hip.FACTOR_LINEAR, 784, 128, C=1 << 20),
            _job(_hip.FACTOR_CONV_G, 64, 32, 56, 56, C=2 << 20),          # long reduction: k-splits
            _job(_hip.FACTOR_CONV_A, 64, 32, 56, 56, k=3, pad=1, C=3 << 20),   # correlation kernels
            _job(_hip.FACTOR_CONV_A, 128, 32, 28, 28, k=3, stride=2, pad=1, C=4 << 20)]
    arr = (_hip.FactorJob * len(jobs))(*jobs)
    assert lib.kfac_factor_grouped_workspace_bytes(len(jobs), arr) > 64 * 64 * 4
    # executed flops: the same tiles and reduction chunks as the single-product plans
    single = (lib.kfac_factor_executed_flops(784, 128) + lib.kfac_factor_executed_flops(64, 32 * 56 * 56)
              + lib.kfac_factor_conv_a_executed_flops(32, 64, 56, 56, 3, 3, 1, 1, 1, 1, 1, 1, 0)
              + lib.kfac_factor_conv_a_executed_flops(32, 128, 28, 28, 3, 3, 2, 2, 1, 1, 1, 1, 0))
    assert abs(lib.kfac_factor_grouped_executed_flops(len(jobs), arr) - single) <= 1e-9 * single
    # images of odd length: single products pad their runs as grouped ones do, within the scratch
    # of a product of as many terms
    for c, n, h, w in ((600, 8, 3, 3), (300, 32, 1, 7), (2048, 32, 7, 7), (512, 1, 1, 5)):
        odd = (_hip.FactorJob * 1)(_job(_hip.FACTOR_CONV_A, c, n, h, w))
        assert lib.kfac_factor_conv_a_executed_flops(n, c, h, w, 1, 1, 1, 1, 0, 0, 1, 1, 0) \
            == lib.kfac_factor_grouped_executed_flops(1, odd)
        assert lib.kfac_factor_conv_a_workspace_bytes(n, c, h, w, 1, 1, 1, 1, 0, 0, 1, 1, 0) \
            == lib.kfac_factor_workspace_bytes(c, n * h * w)
    # a launch too small for 1.5 rounds of items of 8 chunks is one round (512), not a little more
    # (the scratch is one 128 x 128 partial per item, and a little for the tables)
    pointwise = (_hip.FactorJob * 1)(_job(_hip.FACTOR_CONV_A, 256, 32, 56, 56, stride=2))
    assert 256 < lib.kfac_factor_grouped_workspace_bytes(1, pointwise) / 4. / 128 ** 2 < 513
    assert lib.kfac_factor_grouped(0, None, None, 0, None) == 0
    assert lib.kfac_factor_grouped(1, None, None, 0, None) == 1
    assert lib.kfac_factor_grouped(len(jobs), arr, None, 0, None) == 2            # no scratch
    bad = (_hip.FactorJob * 1)(_job(7, 4, 4))
    assert lib.kfac_factor_grouped(1, bad, None, 0, None) == 1                    # unknown kind
    twice = (_hip.FactorJob * 2)(_job(_hip.FACTOR_LINEAR, 4, 4), _job(_hip.FACTOR_LINEAR, 4, 4))
    assert lib.kfac_factor_grouped(2, twice, None, 0, None) == 1                  # one output twice
