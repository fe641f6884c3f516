"""Inserts and reservations that do not get a device buffer: the row-major copy
of the primary codes is optional to an insert, and a failed reservation leaves
the lists whole."""
import contextlib

import numpy as np
import pytest

import jhq_gpu_amd as jg

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def refused(lo, hi, skip=0, count=1 << 40):
    """Buffers of lo <= bytes < hi fail; yields a list that then holds how many."""
    n = []
    jg.lib().jhq_debug_fail_alloc(lo, hi, skip, count)
    try:
        yield n
    finally:
        n.append(int(jg.lib().jhq_debug_fail_alloc(0, 0, 0, 0)))


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


def _make(x, d=512, M=64, **kw):
    p = dict(M=M, B=8, Br=4, alpha=4.0, nlist=8, nprobe=4, ivf_iters=2, batch_size=16, seed=42)
    p.update(kw)
    ix = jg.JHQGpuIndex(d, jg.Params(**p))
    ix.train(x[:1000])
    return ix


def _same(a, b, q, k=10):
    la, lb = a.lists(), b.lists()
    assert all(np.array_equal(la[n], lb[n]) for n in la)
    for kind in (0, 1, 2):  # 2: the pre-scan, whose re-check reads the copy
        a.set_scan_kind(kind)
        b.set_scan_kind(kind)
        (da, ia), (db, ib) = a.search(q, k), b.search(q, k)
        assert np.array_equal(ia, ib) and np.array_equal(_bits(da), _bits(db))
    a.set_scan_kind(0)
    b.set_scan_kind(0)


@pytest.fixture(scope="module")
def data():
    g = np.random.default_rng(3)
    return (g.standard_normal((4000, 512)).astype(np.float32),
            g.standard_normal((40, 512)).astype(np.float32))


def _copy_bytes(ix):
    """The row-major copy of an index's pool (the codes' own buffer has 16
    bytes more)."""
    return (ix.pool()[1] + 15) // 16 * 16 * 64


def test_add_without_row_copy(gpu, data):
    x, q = data
    want, got = _make(x), _make(x)
    want.add(x)
    n = _copy_bytes(want)
    with refused(n, n + 1, count=1) as hit:
        got.add(x)
    assert hit == [1]
    _same(got, want, q)


def test_append_without_row_copy(gpu, data):
    """An append that re-packs the pool while its copy's new buffer is refused,
    then appends in place."""
    x, q = data
    want, got = _make(x), _make(x)
    want.add(x[:2000])
    got.add(x[:2000])
    want.append(x[2000:3900])
    n = _copy_bytes(want)
    with refused(n, n + 1, count=1) as hit:
        got.append(x[2000:3900])
    assert hit == [1]
    _same(got, want, q)
    for ix in (want, got):
        ix.append(x[3900:])
    _same(got, want, q)


def test_shortage_of_the_reservation_leaves_the_lists(gpu, data):
    """The copy stays refused, also to the reservation behind the insert: the
    call fails, the vectors are in, and the index works again with memory."""
    x, q = data
    want, got = _make(x), _make(x)
    want.add(x[:2000])
    want.append(x[2000:])
    got.add(x[:2000])
    n = _copy_bytes(want)
    with refused(n, n + 1) as hit:
        with pytest.raises(jg.JHQDeviceError):
            got.append(x[2000:])
    assert hit[0] >= 2
    assert got.ntotal == want.ntotal
    _same(got, want, q)
