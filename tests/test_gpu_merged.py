"""Search calls with more queries than batch_size run in merged batches of up
to 512 queries: the ids and distances of every call are, bit for bit, those of
calls of batch_size queries (host and device, each scan kind, sizes around the
merged batch, the lanes and a ragged last batch, and shapes whose products are
split over K by the number of rows)."""
import numpy as np
import pytest

import jhq_gpu_amd as jg

pytestmark = pytest.mark.gpu

# d, M, Br, nlist, nprobe, batch, alpha, k
SHAPES = {
    "one_bit_prescan": (128, 16, 4, 24, 6, 16, 4.0, 10),
    # merged calls past the pre-scan's pair limit where it is not the scan
    "one_bit_many_probes": (128, 16, 4, 80, 70, 32, 4.0, 10),
    "two_bit": (100, 25, 4, 24, 5, 32, 4.0, 10),
    "flat": (96, 12, 8, 1, 1, 7, 4.0, 1),
    "long_lists": (128, 32, 4, 16, 16, 100, 4.0, 100),
    "batch_over_512": (64, 16, 4, 16, 4, 600, 4.0, 10),
    # d not a multiple of 64: the rows would choose the split of the scores (2 at
    # 64 rows, 1 at 512; only near ties of the probes show it) and of the
    # rotation (8 and 2; every distance shows it)
    "split_scores": (200, 50, 4, 2048, 8, 64, 4.0, 10),
    "split_rotation": (520, 65, 4, 16, 4, 64, 4.0, 10),
}


@pytest.fixture(scope="module", params=sorted(SHAPES))
def built(request, gpu):
    d, M, Br, nlist, nprobe, batch, alpha, k = SHAPES[request.param]
    g = np.random.default_rng(5)
    x = g.standard_normal((6000, d)).astype(np.float32)
    ix = jg.JHQGpuIndex(d, jg.Params(M=M, B=8, Br=Br, alpha=alpha, nlist=nlist, nprobe=nprobe,
                                     ivf_iters=2, batch_size=batch, seed=42))
    ix.train(x[:3000])
    ix.add(x)
    ix.reserve(k)
    q = g.standard_normal((2100, d)).astype(np.float32)
    return ix, q, batch, k


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


@pytest.mark.parametrize("kind", [0, 1, 2])
def test_merged_batches_equal_single_ones(built, gpu, kind):
    import torch
    ix, q, B, k = built
    ix.set_scan_kind(kind)
    try:
        parts = [ix.search(q[i:i + B], k) for i in range(0, len(q), B)]
        want_d = np.concatenate([p[0] for p in parts])
        want_i = np.concatenate([p[1] for p in parts])
        for nq in sorted({B, B + 1, 511, 512, 513, 1029, 2100}):
            d, i = ix.search(q[:nq], k)
            assert np.array_equal(i, want_i[:nq]), nq
            assert np.array_equal(_bits(d), _bits(want_d[:nq])), nq
            qt = torch.from_numpy(q[:nq]).to(gpu)
            od = torch.full((nq, k), -1.0, device=gpu)
            oi = torch.full((nq, k), -2, dtype=torch.int32, device=gpu)
            for _ in range(2):
                ix.search_device(qt, k, od, oi, stream=torch.cuda.current_stream())
            assert np.array_equal(oi.cpu().numpy(), want_i[:nq]), nq
            assert np.array_equal(_bits(od.cpu().numpy()), _bits(want_d[:nq])), nq
    finally:
        ix.set_scan_kind(0)


@pytest.mark.parametrize("d,M,nprobe", [(1024, 128, 32), (1024, 128, 64), (512, 64, 64)])
def test_batches_sharing_a_query_product(gpu, d, M, nprobe):
    """Batches of at most 128 queries: a lane takes two at a time with one query
    product (4 split sums a query at d 1024, 2 at 512), the last pair ragged, or
    its last batch alone."""
    import torch
    g = np.random.default_rng(6)
    x = g.standard_normal((3000, d)).astype(np.float32)
    ix = jg.JHQGpuIndex(d, jg.Params(M=M, B=8, Br=4, alpha=4.0, nlist=96, nprobe=nprobe,
                                     ivf_iters=2, batch_size=64, seed=42))
    ix.train(x[:1000])
    ix.add(x)
    ix.set_scan_kind(2)
    rows = ix.call_plan(1 << 16, 10)["rows"]
    assert rows == 4096 // nprobe
    L = ix.call_plan(1 << 16, 10)["lanes"]
    assert L > 1
    q = g.standard_normal((4 * L * rows, d)).astype(np.float32)
    parts = [ix.search(q[i:i + 64], 10) for i in range(0, len(q), 64)]
    want_d = np.concatenate([p[0] for p in parts])
    want_i = np.concatenate([p[1] for p in parts])
    qt = torch.from_numpy(q).to(gpu)
    # in batches: whole pairs, a ragged last one, a last batch alone
    for nq in (len(q), len(q) - rows // 2, len(q) - rows, L * rows + 1):
        plan = ix.call_plan(nq, 10)
        assert plan["shared"] == 2 and plan["lanes"] > 1, (nq, plan)
        od = torch.full((nq, 10), -1.0, device=gpu)
        oi = torch.full((nq, 10), -2, dtype=torch.int32, device=gpu)
        for _ in range(2):
            ix.search_device(qt[:nq], 10, od, oi, stream=torch.cuda.current_stream())
            assert np.array_equal(oi.cpu().numpy(), want_i[:nq]), nq
            assert np.array_equal(_bits(od.cpu().numpy()), _bits(want_d[:nq])), nq
    # pairs where they lengthen no lane: 2 or 4 batches on the fullest one, not 1
    # or 3
    for nb in range(1, 4 * L + 1):
        assert ix.call_plan(nb * rows, 10)["shared"] == (1 if (nb + L - 1) // L % 2 else 2), nb


@pytest.mark.parametrize("kind", [0, 2])
def test_long_short_lists_leave_the_others_their_scan(gpu, kind):
    """Reserving a k past the pre-scan's short lists changes neither the scan nor
    the batches of calls with small k (one size serves every reserved k)."""
    g = np.random.default_rng(8)
    x = g.standard_normal((4000, 1024)).astype(np.float32)
    q = g.standard_normal((600, 1024)).astype(np.float32)
    ix = jg.JHQGpuIndex(1024, jg.Params(M=128, B=8, Br=4, alpha=10.0, nlist=64, nprobe=32,
                                        ivf_iters=2, batch_size=16, seed=42))
    ix.train(x[:1000])
    ix.add(x)
    ix.set_scan_kind(kind)
    plan = ix.call_plan(600, 10)
    assert plan["scan"] == "mfma_scan_kernel" and plan["rows"] == 128
    want = ix.search(q, 10)
    ix.reserve(130)
    assert ix.call_plan(600, 10) == plan
    assert ix.call_plan(600, 130)["scan"] != "mfma_scan_kernel"
    got = ix.search(q, 10)
    assert np.array_equal(got[1], want[1]) and np.array_equal(_bits(got[0]), _bits(want[0]))


def test_workspaces_stay_within_their_bound(gpu):
    """The workspaces of merged batches: at most 640 MB on each lane that a call
    uses (one list of 131072 and k 100: 577 MB of distances for 512 queries)."""
    import torch

    def used():
        torch.cuda.synchronize()
        free, total = torch.cuda.mem_get_info()
        return total - free

    g = np.random.default_rng(9)
    x = g.standard_normal((131072, 64)).astype(np.float32)
    ix = jg.JHQGpuIndex(64, jg.Params(M=16, B=8, Br=4, alpha=4.0, nlist=1, nprobe=1, ivf_iters=1,
                                      batch_size=32, seed=42))
    ix.train(x[:2000])
    ix.add(x)
    before = used()
    ix.reserve(100)
    plan = ix.call_plan(1 << 16, 100)
    assert plan["rows"] == 512 and plan["scan"] == "scan_dump_kernel"
    assert used() - before <= plan["lanes"] * (640 << 20)
