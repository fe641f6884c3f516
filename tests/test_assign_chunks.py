"""The chunked accumulation of the MFMA assignment (jhq_gpu_amd/csrc/assign_mfma.hip):
the MFMAs sum 4 steps of 32 k from zero, and each chunk is added to the dot
with one rounding.  The scores' bound, with
    e_dot = (2u * 1.02 * 33 * 3 * min(dp/32, 4) + 1.02 u chunks + 3.01 * 2^-16
             + (d + 4) u) ||y|| Cmax,
must cover the difference to the fixed-order chain in any order the MFMA can
take, and must not cover a dropped chunk."""
import numpy as np
import pytest

from test_assign_bound import U, chain_dot, make, mfma_dot, score


def chunk_dot(y, c, rng, mode, drop=None):
    total = None
    for j, k0 in enumerate(range(0, y.shape[0], 128)):
        if j == drop:
            continue
        part = mfma_dot(y[k0:k0 + 128], c[k0:k0 + 128], rng, mode)
        total = part if total is None else np.float32(total + part)
    return total


def bound(y, nmax, K):
    ny = np.sqrt(np.sum(y.astype(np.float64) ** 2)) * (1 + 4 * U)
    nm = nmax * (1 + 4 * U)
    cm = np.sqrt(nm)
    steps = (K + 31) // 32
    e_dot = (2 * U * 1.02 * 33 * 3 * min(steps, 4) + 1.02 * U * ((steps + 3) // 4) + 3.01 / 65536.0 +
             (K + 4) * U) * ny * cm
    tiny = 6.0 * K * (2.0 ** -126 * (ny + cm) + 2.0 ** -149)
    return 2.0 * (2.0 * e_dot + 2.0 * U * nm + 4.0 * U * ny * cm) + tiny


@pytest.mark.parametrize("K,offset,spread", [(128, 100.0, 30.0), (132, 0.0, 1.0), (300, 2.0, 1.0),
                                            (1024, 0.0, 1.0), (768, 5.0, 1e3)])
def test_chunks_within_half_bound(K, offset, spread):
    rng, y, c, norms = make(K, offset, spread, 11 * K + int(offset), rows=8, cols=12)
    nmax = float(norms.max())
    worst = 0.0
    for i in range(y.shape[0]):
        E = bound(y[i], nmax, K)
        for j in range(c.shape[0]):
            fixed = score(chain_dot(y[i], c[j], range(K)), norms[j])
            for mode in ("one", "seq"):
                alt = score(chunk_dot(y[i], c[j], rng, mode), norms[j])
                worst = max(worst, abs(float(fixed) - float(alt)) / E)
    # E holds twice the summed worst cases
    assert worst < 0.5, worst


def test_bound_catches_a_dropped_chunk():
    rng = np.random.default_rng(5)
    K = 512
    y, c = (rng.standard_normal(K).astype(np.float32) for _ in range(2))
    norm = np.float32(np.sum(c.astype(np.float64) ** 2))
    E = bound(y, float(norm), K)
    good = score(chain_dot(y, c, range(K)), norm)
    assert abs(float(good) - float(score(chunk_dot(y, c, rng, "one", drop=2), norm))) > 4 * E
