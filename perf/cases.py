"""Timing cases of the JHQ engine: what a program does with it through jhq_gpu_amd.

Three kinds of work, each through the public entry points:

* ``search``  queries against a trained and filled index, device-resident
  (``search_device``) or host to host (``search``);
* ``stream``  one step of a growing index: ``append`` a few thousand host
  vectors, then search a batch of queries in the grown index;
* ``encode``  the device-resident encoding of a block of vectors: rotation,
  primary codes, residual codes and corrections, list assignment;
* ``build``   an index from nothing: create, train, add and a first search.

The data is the benchmark's family (Gaussian mixtures, L2-normalised float32
rows, or byte-valued ones), smaller.  A search case's index stands for the one
that a serving program keeps: it depends on the case alone and is shared by
the states of all seeds; a seed draws the queries.
"""
import collections
import math

import numpy as np
import torch

import jhq_gpu_amd as jg

DEV = "cuda:0"

# (d, M) of the shapes that the configurations and tests use, and generic
# ones: Ds = d / M in {1, 2, 4, 8}, d multiples of 64 and not
SHAPES = ((1024, 128), (768, 96), (512, 64), (384, 96), (256, 32), (200, 50), (128, 16),
          (100, 25), (96, 12), (64, 16))


def _search(name, **kw):
    c = dict(name=name, kind="search", d=1024, M=128, Br=4, per_subspace=0, data="f32", n=262144,
             nlist=2048, nprobe=16, batch=64, alpha=4.0, k=10, nq=64, host=0)
    c.update(kw)
    return c


def listed():
    return [
        # a single query against a flat index, the lowest latency a caller sees
        _search("one_query_flat_1024", n=65536, nlist=1, nprobe=1, batch=1, nq=1),
        # a small index answering a ragged host request (8-bit residual codes,
        # a batch size that does not divide the queries)
        _search("small_host_96", d=96, M=12, Br=8, n=20011, nlist=100, nprobe=8, batch=16, nq=37,
                host=1),
        # the headline shape, 262 144 of its vectors: many device-resident
        # queries in batches of 64, alpha 10
        _search("ivf_1024", alpha=10.0, nq=4096),
        # the reference's protocol at the parameters' defaults (M 96, nlist 1024,
        # nprobe 8, batch 256, alpha 4): host arrays in, host arrays out
        _search("host_768_defaults", d=768, M=96, n=200003, nlist=1024, nprobe=8, batch=256,
                nq=1000, host=1),
        # byte vectors with many candidates per query: the scan-bound shape
        _search("u8_128_scan", d=128, M=16, data="u8", n=4000000, nlist=4096, nprobe=64, nq=2048),
        # heavy-tailed int8 rows, d and M no powers of two, two bits per digit
        _search("i8_100_scan", d=100, M=25, data="i8", n=1000000, nlist=4096, nprobe=48, batch=32,
                nq=320),
        # long result lists (k 100, short list 400) on two-bit digits
        _search("k100_384", d=384, M=96, n=300007, nlist=1024, nprobe=8, batch=128, k=100, nq=500),
        # streaming: 2000 vectors in, 128 queries answered (k 100, one residual
        # codebook per subspace)
        dict(name="stream_768", kind="stream", d=768, M=96, Br=4, per_subspace=1, data="f32",
             n=200000, nlist=1024, nprobe=32, batch=128, alpha=4.0, k=100, nq=128, rows=2000),
        # one full add() block of the headline shape
        dict(name="encode_1024", kind="encode", d=1024, M=128, Br=4, n=65536, nlist=4096),
        # the byte configurations' add() block: short vectors, very many lists
        dict(name="encode_128", kind="encode", d=128, M=16, Br=4, n=65536, nlist=65536),
        # a small insert, d not a multiple of 16
        dict(name="encode_small_100", kind="encode", d=100, M=25, Br=4, n=1000, nlist=1000),
        # a small index from nothing
        dict(name="build_u8_128", kind="build", d=128, M=16, Br=4, per_subspace=0, data="u8",
             n=100000, ntrain=20000, nlist=512, nprobe=16, batch=64, alpha=4.0, k=10, nq=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("search",) * 5 + ("encode",) * 3 + ("stream",))
    d, M = rng.choice(SHAPES)
    if kind == "encode":
        n = _log(rng, 500, 65536)
        # no more score arithmetic than the largest listed block
        nlist = min(_log(rng, 16, 65536), int(2.5e11 / (n * d)))
        return dict(kind="encode", d=d, M=M, Br=rng.choice((4, 4, 8)), n=n, nlist=max(nlist, 8))
    data = rng.choice(("u8", "i8")) if d <= 128 and rng.random() < 0.5 else "f32"
    nlist = _log(rng, 16, 2048)
    k = rng.choice((1, 10, 10, 10, 20, 100))
    if kind == "stream":
        return dict(kind="stream", d=d, M=M, Br=4, per_subspace=rng.randint(0, 1), data=data,
                    n=_log(rng, 50000, 200000), nlist=min(nlist, 1024),
                    nprobe=rng.randint(4, 16), batch=128, alpha=4.0, k=min(k, 20),
                    nq=rng.randint(1, 128), rows=_log(rng, 100, 2000))
    if rng.random() < 0.15:
        nlist = 1
    n = _log(rng, 10000, min(4000000, int(2.0e8 / d)))
    nlist = min(nlist, n // 64)
    nprobe = min(nlist, rng.choice((1, 4, 8, 16, 32, 64)))
    cand = max(1.0, n * nprobe / nlist)
    batch = min(rng.choice((1, 16, 32, 64, 64, 100, 128, 256)), max(1, int(3e7 / cand)))
    # no more code bytes per call than the largest listed search
    nq = max(1, min(_log(rng, 1, 4096), int(1.0e9 / (cand * M))))
    c = _search("", d=d, M=M, Br=rng.choice((4, 4, 4, 8)), data=data, n=n, nlist=nlist,
                nprobe=nprobe, batch=batch,
                alpha=rng.choice((2.0, 4.0) if k > 20 else (4.0, 4.0, 10.0)), k=k, nq=nq,
                host=rng.randint(0, 1))
    del c["name"]
    return c


# ---- data -------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _mixture(c, n, seed, comp_seed=11):
    """n rows of the case's distribution on the device, the components drawn
    from comp_seed: float32 L2-normalised anisotropic Gaussian mixture rows;
    uint8 with means N(34, 60^2) and deviation 20, clipped (about 30% zeros);
    int8 with means N(0, 32^2) and 16 x Student-t (nu = 4) noise."""
    d, data = c["d"], c["data"]
    ncomp = max(64, min(4096, 2 * c["nlist"]))
    g = _gen(comp_seed)
    means = torch.randn(ncomp, d, device=DEV, generator=g)
    scales = torch.empty(ncomp, d, device=DEV).uniform_(math.log(0.1), 0.0, generator=g).exp_()
    g = _gen(seed)
    out = torch.empty(n, d, device=DEV,
                      dtype={"f32": torch.float32, "u8": torch.uint8, "i8": torch.int8}[data])
    step = max(1, (1 << 27) // d)
    for i in range(0, n, step):
        m = min(step, n - i)
        comp = torch.randint(0, ncomp, (m,), device=DEV, generator=g)
        z = torch.randn(m, d, device=DEV, generator=g)
        if data == "f32":
            x = means[comp] + scales[comp] * z
            out[i:i + m] = x / x.norm(dim=1, keepdim=True)
        elif data == "u8":
            x = 34.0 + 60.0 * means[comp] + 20.0 * z
            out[i:i + m] = x.round_().clamp_(0, 255).to(torch.uint8)
        else:
            chi = torch.zeros(m, d, device=DEV)
            for _ in range(4):
                chi += torch.randn(m, d, device=DEV, generator=g) ** 2
            x = 32.0 * means[comp] + 16.0 * z / (chi / 4.0).sqrt()
            out[i:i + m] = x.round_().clamp_(-128, 127).to(torch.int8)
    return out


def _ntrain(c):
    """Training rows: at least four per list, at most 6 M values beyond that."""
    return c.get("ntrain") or min(c["n"], max(4 * c["nlist"], 6_000_000 // c["d"]))


def _params(c):
    return jg.Params(M=c["M"], B=8, Br=c["Br"], alpha=c["alpha"], nlist=c["nlist"],
                     nprobe=c["nprobe"], ivf_iters=4, batch_size=c["batch"], seed=42,
                     residual_per_subspace=c["per_subspace"])


def _build(c):
    base = _mixture(c, c["n"], 101).cpu().numpy()
    ix = jg.JHQGpuIndex(c["d"], _params(c))
    ix.train(base[:_ntrain(c)])
    ix.add(base)
    ix.reserve(c["k"])
    return ix


# The indexes that searches share, the least recently used one dropped.
_KEEP = 16
_indexes = collections.OrderedDict()


def _index(c):
    key = tuple(sorted((k, v) for k, v in c.items() if k not in ("name", "nq", "host")))
    if key not in _indexes:
        while len(_indexes) >= _KEEP:
            _indexes.popitem(last=False)
        _indexes[key] = _build(c)
    _indexes.move_to_end(key)
    return _indexes[key]


def _queries(c, seed):
    return _mixture(c, c["nq"], 1000 + seed)


def _encode_inputs(c, seed):
    """A rotation, rotated-space centroids and codebooks as training leaves
    them, and n vectors."""
    d, K1D = c["d"], 1 << (8 * c["M"] // c["d"])
    Kr = 1 << c["Br"]
    P = torch.linalg.qr(torch.randn(d, d, generator=torch.Generator().manual_seed(7)))[0].to(DEV)
    P = P.contiguous()
    mix = dict(c, data="f32")
    x = _mixture(mix, c["n"], 1000 + seed)
    y0 = _mixture(mix, c["nlist"] * 2, 5)
    cent = ((y0[::2] + y0[1::2]) * 0.5) @ P.T
    norms = cent.double().square().sum(1).float()
    sigma = d ** -0.5

    def quantiles(m, s):
        p = (torch.arange(m, dtype=torch.float64) + 0.5) / m
        return (s * math.sqrt(2.0) * torch.erfinv(2.0 * p - 1.0)).float().to(DEV)

    return dict(P=P, x=x, cent=cent.contiguous(), norms=norms, c1d=quantiles(K1D, sigma),
                res_c1d=quantiles(Kr, sigma * (0.6 if K1D == 2 else 1.1 / K1D)))


# ---- the measured interface ------------------------------------------------------

def prepare(case, seed):
    c = case
    if c["kind"] == "search":
        q = _queries(c, seed)
        s = dict(c=c, ix=_index(c))
        if c["host"]:
            s["q"] = q.cpu().numpy()
        else:
            s["q"] = q.float().contiguous()
            s["d"] = torch.empty(c["nq"], c["k"], device=DEV)
            s["i"] = torch.empty(c["nq"], c["k"], dtype=torch.int32, device=DEV)
        return s
    if c["kind"] == "stream":
        # the index grows: every state has one of its own
        return dict(c=c, ix=_build(c), rows=_mixture(c, c["rows"], 5000 + seed).cpu().numpy(),
                    q=_queries(c, seed).cpu().numpy())
    if c["kind"] == "build":
        return dict(c=c, x=_mixture(c, c["n"], 5000 + seed).cpu().numpy(),
                    q=_queries(c, seed).cpu().numpy())
    s = _encode_inputs(c, seed)
    n, d, M = c["n"], c["d"], c["M"]
    s.update(c=c, y=torch.empty(n, d, device=DEV),
             codes=torch.empty(n, M, dtype=torch.uint8, device=DEV),
             res=torch.empty(n, (d * c["Br"] + 7) // 8, dtype=torch.uint8, device=DEV),
             corr=torch.empty(n, device=DEV),
             assign=torch.empty(n, dtype=torch.int32, device=DEV))
    return s


def run(s):
    c = s["c"]
    if c["kind"] == "search":
        if c["host"]:
            return s["ix"].search(s["q"], c["k"])
        s["ix"].search_device(s["q"], c["k"], s["d"], s["i"])
        return s["d"], s["i"]
    if c["kind"] == "stream":
        s["ix"].append(s["rows"])
        return s["ix"].search(s["q"], c["k"])
    if c["kind"] == "build":
        ix = jg.JHQGpuIndex(c["d"], _params(c))
        ix.train(s["x"][:c["ntrain"]])
        ix.add(s["x"])
        dists, ids = ix.search(s["q"], c["k"])
        return dists, ids, {k: v for k, v in ix.codebooks().items() if k != "P"}
    jg.k_rotate(s["P"], s["x"], s["y"])
    jg.k_primary_encode(s["y"], s["codes"], s["c1d"], c["M"])
    jg.k_residual_encode(s["y"], s["codes"], s["res"], s["corr"], s["c1d"], s["res_c1d"], c["M"],
                         c["Br"])
    jg.k_assign(s["y"], s["cent"], s["norms"], s["assign"])
    return s["y"], s["codes"], s["res"], s["corr"], s["assign"]


def work(case):
    c = case
    d, M, n, nlist = c["d"], c["M"], c["n"], c["nlist"]
    bpv = (d * c["Br"] + 7) // 8
    if c["kind"] == "encode":
        # vectors, rotation and centroids in; rotated vectors, codes,
        # corrections and lists out
        return dict(bytes=4.0 * (2 * n * d + d * d + nlist * d) + n * (M + bpv + 8.0),
                    flops=2.0 * n * d * (d + nlist))
    nq, k = c["nq"], c["k"]
    ck = max(k, math.ceil(c["alpha"] * k))
    cand = n * c["nprobe"] / nlist  # candidates per query, lists of equal size
    # queries, [rotation ; centroids], the probed codes once however many
    # queries share them, the short lists' residual codes, results
    nbytes = (4.0 * (nq * d + (d + nlist) * d) + min(float(n), nq * cand) * M
              + nq * min(ck, cand) * (bpv + 8.0) + 8.0 * nq * k)
    flops = 2.0 * nq * d * (d + nlist) + nq * cand * M + 2.0 * nq * min(ck, cand) * d
    if c["kind"] == "stream":
        m = c["rows"]
        nbytes += m * (d * (4.0 if c["data"] == "f32" else 1.0) + M + bpv + 8.0)
        flops += 2.0 * m * d * (d + nlist)
    if c["kind"] == "build":
        m = c["ntrain"]
        nbytes += n * (d * (4.0 if c["data"] == "f32" else 1.0) + M + bpv + 8.0)
        # rotations, four k-means assignments, the final assignment, and the
        # rotation's QR
        flops += 2.0 * (m + n) * d * d + 2.0 * (4 * m + n) * d * nlist + 4.0 * d ** 3
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    # add and train are pinned bit for bit (codes, lists and codebooks do not
    # depend on a summation order)
    if case["kind"] == "encode":
        return "exact"
    # the query rotation and the centroid scores may sum in any order; ids may
    # swap where two distances agree to that rounding
    return {"rel": 2e-6, "max": 2e-5, "differ": 2e-3}


# ---- the same in 64 bits ------------------------------------------------------------

def _nearest(book, v):
    """Index of the nearest word of a sorted codebook (midpoint thresholds)."""
    return torch.bucketize(v, (book[:-1] + book[1:]) * 0.5, right=True)


def _exact_encode(c, seed):
    s = _encode_inputs(c, seed)
    c1d, rc = s["c1d"].double(), s["res_c1d"].double()
    y = torch.empty(c["n"], c["d"], dtype=torch.float64, device=DEV)
    corr = torch.empty(c["n"], dtype=torch.float64, device=DEV)
    for i in range(0, c["n"], 8192):
        y[i:i + 8192] = s["x"][i:i + 8192].double() @ s["P"].double().T
        t = y[i:i + 8192]
        yhat = c1d[_nearest(c1d, t)]
        corr[i:i + 8192] = 2.0 * (yhat * rc[_nearest(rc, t - yhat)]).sum(1)
    return y, None, None, corr, None


def _exact_search(c, ix, q):
    """The search of q in the stored lists of ix, every sum in float64.  The
    index's trained state and stored codes are inputs."""
    d, M, Br, k, P = c["d"], c["M"], c["Br"], c["k"], c["nprobe"]
    n, bpd = ix.ntotal, 8 * M // d
    ck = max(k, math.ceil(c["alpha"] * k))
    cb, L = ix.codebooks(), ix.lists()

    def dev(a, t=None):
        a = torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
        return a if t is None else a.to(t)

    qr = dev(q, torch.float64) @ dev(cb["P"], torch.float64).T
    cent = dev(cb["centroids"], torch.float64)
    score = cent.square().sum(1)[None, :] - 2.0 * (qr @ cent.T)
    probes = score.topk(P, dim=1, largest=False).indices
    sizes = dev(np.diff(L["offsets"].astype(np.int64)))
    lists = torch.repeat_interleave(torch.arange(c["nlist"], device=DEV), sizes)
    c1d, rc = dev(cb["c1d"], torch.float64), dev(cb["res_c1d"], torch.float64)
    codes, res = dev(L["codes"]), dev(L["res"])
    corr = dev(L["corr"], torch.float64)
    shift = (torch.arange(d // M, device=DEV) * bpd).to(torch.int32)

    def decode(codes):
        dig = (codes.to(torch.int32)[..., None] >> shift) & ((1 << bpd) - 1)
        return c1d[dig.flatten(-2)]

    # primary distances of every vector, the probed ones kept, block by block
    nq = qr.shape[0]
    best_d = torch.full((nq, ck), math.inf, dtype=torch.float64, device=DEV)
    best_i = torch.full((nq, ck), -1, dtype=torch.int64, device=DEV)
    on = torch.zeros(nq, c["nlist"], dtype=torch.bool, device=DEV).scatter_(1, probes, True)
    step = max(1024, 200_000_000 // max(nq, d))
    for i in range(0, n, step):
        yh = decode(codes[i:i + step])
        dd = qr.square().sum(1)[:, None] + yh.square().sum(1)[None, :] - 2.0 * (qr @ yh.T)
        dd.masked_fill_(~on[:, lists[i:i + step]], math.inf)
        v, j = dd.topk(min(ck, dd.shape[1]), dim=1, largest=False)
        v, at = torch.cat((best_d, v), 1).topk(ck, dim=1, largest=False)
        best_i = torch.cat((best_i, j + i), 1).gather(1, at)
        best_d = v
    out = torch.full((nq, k), math.inf, dtype=torch.float64, device=DEV)
    for b in range(0, nq, 64):
        at = best_i[b:b + 64].clamp(min=0)
        r = res[at].to(torch.int64)
        if Br == 4:
            r = torch.stack((r & 15, r >> 4), -1).flatten(-2)[..., :d]
        if rc.dim() == 2:
            rhat = rc[torch.arange(d, device=DEV) // (d // M), r]
        else:
            rhat = rc[r]
        comp = best_d[b:b + 64] + (qr[b:b + 64, None, :] - rhat).square().sum(2) + corr[at]
        comp[torch.isinf(best_d[b:b + 64])] = math.inf
        out[b:b + 64] = comp.topk(k, dim=1, largest=False).values
    return out.cpu().numpy(), None


def exact(case, seed):
    c = case
    if c["kind"] == "encode":
        return _exact_encode(c, seed)
    if c["kind"] == "search":
        return _exact_search(c, _index(c), _queries(c, seed).cpu().numpy())
    if c["kind"] == "stream":
        s = prepare(c, seed)
        s["ix"].append(s["rows"])
        return _exact_search(c, s["ix"], s["q"])
    return None  # training's discrete choices have no 64-bit counterpart
