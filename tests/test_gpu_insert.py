"""Encode kernels of insert.hip against the oracle, bit for bit: every digit
width that packs in words, d past the last whole octet and chunk, both residual
widths, and vector counts around a workgroup's 16."""
import numpy as np
import pytest

import pyoracle as po

import jhq_gpu_amd as jg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 17, 100])
@pytest.mark.parametrize("d,M,Br,Kr", [
    (8, 1, 4, 16), (136, 17, 4, 16), (1032, 129, 8, 256),    # Ds 8
    (4, 1, 4, 16), (132, 33, 4, 16), (260, 65, 8, 200),      # Ds 4
    (12, 6, 4, 16), (140, 70, 8, 256),                       # Ds 2
    (4, 4, 8, 256), (268, 268, 4, 16),                       # Ds 1
    (136, 17, 4, 9), (129, 129, 4, 16),                      # the general kernel
])
def test_encode_words(gpu, n, d, M, Br, Kr):
    import torch

    def t(a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(gpu)

    rng = np.random.default_rng(n * 1000 + d + M)
    y = (rng.standard_normal((n, d)) * 0.05).astype(np.float32)
    c1d = po.lloyd_max_c1d(0.05, 1 << (8 // (d // M)))
    rc = np.sort(rng.standard_normal(Kr).astype(np.float32) * 0.02)
    # values on the thresholds
    mids = np.float32(0.5) * (c1d[:-1] + c1d[1:])
    y[0, :min(d, len(mids))] = mids[:min(d, len(mids))]
    codes = torch.empty((n, M), dtype=torch.uint8, device=gpu)
    res = torch.empty((n, (d * Br + 7) // 8), dtype=torch.uint8, device=gpu)
    corr = torch.empty((n,), dtype=torch.float32, device=gpu)
    jg.k_primary_encode(t(y), codes, t(c1d), M)
    jg.k_residual_encode(t(y), codes, res, corr, t(c1d), t(rc), M, Br)
    torch.cuda.synchronize()
    oc = po.primary_encode(y, M, c1d)
    ores, ocorr = po.residual_encode(y, oc, M, c1d, rc, Br)
    assert np.array_equal(codes.cpu().numpy(), oc)
    assert np.array_equal(res.cpu().numpy(), ores)
    assert np.array_equal(corr.cpu().numpy().view(np.uint32), ocorr.view(np.uint32))
