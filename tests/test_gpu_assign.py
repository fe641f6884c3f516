"""The MFMA assignment (assign_mfma.hip) against the oracle: every operand
form (1 to 8 k steps in registers, long vectors in small and large tiles),
ragged rows, lists and k, near ties, and rows with more near lists than the
re-check keeps."""
import numpy as np
import pytest

import pyoracle as po

import jhq_gpu_amd as jg

pytestmark = pytest.mark.gpu


def _t(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _assign(gpu, f, y, cent, norms):
    import torch
    a = torch.full((y.shape[0],), -7, dtype=torch.int32, device=gpu)
    f(_t(y, gpu), _t(cent, gpu), _t(norms, gpu), a)
    torch.cuda.synchronize()
    return a.cpu().numpy()


@pytest.mark.parametrize("n,d,nlist", [
    (1, 4, 1), (255, 32, 63), (257, 60, 65), (300, 96, 129), (1025, 128, 1000),   # 1 .. 4 steps
    (129, 132, 33), (300, 192, 31), (127, 200, 100), (640, 256, 1000),            # 5 .. 8 steps
    (130, 260, 65), (70, 388, 300),                                               # small tiles
    (22001, 292, 257),                                                            # large tiles
])
def test_assign_forms(gpu, n, d, nlist):
    rng = np.random.default_rng(n + d + nlist)
    cent = rng.standard_normal((nlist, d)).astype(np.float32)
    y = rng.standard_normal((n, d)).astype(np.float32)
    m = n // 3  # midpoints of two lists: near ties
    y[:m] = 0.5 * (cent[rng.integers(0, nlist, m)] + cent[rng.integers(0, nlist, m)])
    norms = po.cent_norms(cent)
    got = _assign(gpu, jg.k_assign, y, cent, norms)
    assert np.array_equal(got, po.assign(y, cent, norms))


@pytest.mark.parametrize("d", [64, 288])
def test_assign_many_equal_lists(gpu, d):
    """40 copies of one centroid: more near lists than kept per row, so the
    rows near it take the fixed-order argmin over every list."""
    rng = np.random.default_rng(d)
    cent = rng.standard_normal((200, d)).astype(np.float32)
    cent[100:140] = cent[3]
    y = rng.standard_normal((700, d)).astype(np.float32)
    y[::2] = cent[3] + 0.01 * rng.standard_normal((350, d)).astype(np.float32)
    norms = po.cent_norms(cent)
    got = _assign(gpu, jg.k_assign, y, cent, norms)
    assert np.array_equal(got, po.assign(y, cent, norms))


@pytest.mark.parametrize("d", [32, 132, 320])
def test_assign_non_finite(gpu, d):
    """Rows and a list with infinities and NaN: the lists of the fixed-order
    argmin alone (k_assign_noalloc)."""
    rng = np.random.default_rng(d)
    cent = rng.standard_normal((150, d)).astype(np.float32)
    y = rng.standard_normal((500, d)).astype(np.float32)
    y[3, 1], y[77, 0], y[200] = np.nan, np.inf, 3e38
    cent[60, 2], cent[61, 0] = np.nan, -np.inf
    norms = np.square(cent.astype(np.float64)).sum(1).astype(np.float32)
    got = _assign(gpu, jg.k_assign, y, cent, norms)
    want = _assign(gpu, jg.k_assign_noalloc, y, cent, norms)
    ok = np.isfinite(y).all(1)
    assert np.array_equal(got[ok], want[ok]) and np.array_equal(got[~ok], want[~ok])


@pytest.mark.parametrize("d", [32, 132, 320])
@pytest.mark.parametrize("first", [True, False], ids=["before", "behind"])
def test_assign_nan_lists(gpu, d, first):
    """Lists with a NaN among finite ones, and finite rows: the bound stays finite,
    so the rows are accepted or re-checked by their own scores.  The NaN lists,
    before or behind the others, are no row's."""
    rng = np.random.default_rng(d)
    cent = rng.standard_normal((150, d)).astype(np.float32)
    nan = np.arange(0, 20, 3) if first else np.arange(130, 150, 3)
    cent[nan, rng.integers(0, d, len(nan))] = np.nan
    y = rng.standard_normal((500, d)).astype(np.float32)
    y[:100] = 0.5 * (cent[50] + cent[rng.integers(20, 130, 100)])  # near ties
    norms = po.cent_norms(cent)
    got = _assign(gpu, jg.k_assign, y, cent, norms)
    finite = np.setdiff1d(np.arange(150), nan)
    assert np.array_equal(got, finite[po.assign(y, cent[finite], norms[finite])])
    assert np.array_equal(got, _assign(gpu, jg.k_assign_noalloc, y, cent, norms))
