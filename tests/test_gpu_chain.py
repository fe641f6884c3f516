"""The fixed-order GEMM on fp32 MFMA (gemm_chain.hip) against the oracle's
fmaf chain, bit for bit: both tile sizes, vector and scalar loads, rows,
columns and k past the last whole tile."""
import numpy as np
import pytest

import pyoracle as po

import jhq_gpu_amd as jg

pytestmark = pytest.mark.gpu


def _t(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


@pytest.mark.parametrize("n,d", [
    (1, 1), (65, 3), (63, 32), (130, 65),      # 64 x 64 tiles, k tails 1 .. 31
    (22001, 260), (21900, 259),                # 128 x 128 tiles, vector / scalar loads
    (65537, 128),                              # whole k steps only, a last tile of one row
])
def test_rotate_chain(gpu, n, d):
    import torch
    rng = np.random.default_rng(n + d)
    x = rng.standard_normal((n, d)).astype(np.float32)
    x[:, 0] *= 1e-40  # subnormal products
    P = rng.standard_normal((d, d)).astype(np.float32)
    y = torch.empty((n, d), dtype=torch.float32, device=gpu)
    jg.k_rotate(_t(P, gpu), _t(x, gpu), y)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy().view(np.uint32), po.rotate(P, x).view(np.uint32))


@pytest.mark.parametrize("n,d,nlist", [(70, 5, 3), (64, 36, 129), (4101, 36, 2101), (4095, 33, 2049)])
def test_argmin_chain(gpu, n, d, nlist):
    """k_assign_noalloc runs the fixed-order argmin on every row."""
    import torch
    rng = np.random.default_rng(n + d + nlist)
    y = rng.integers(-2, 3, (n, d)).astype(np.float32)      # many exact ties
    cent = rng.integers(-2, 3, (nlist, d)).astype(np.float32)
    norms = po.cent_norms(cent)
    a = torch.empty((n,), dtype=torch.int32, device=gpu)
    jg.k_assign_noalloc(_t(y, gpu), _t(cent, gpu), _t(norms, gpu), a)
    torch.cuda.synchronize()
    assert np.array_equal(a.cpu().numpy(), po.assign(y, cent, norms))
