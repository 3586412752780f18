"""Performance cases of the search paths: what is timed, on which inputs, and how far results may differ.

Every case goes through the package's public entry points on device-resident data, as a serving
program does: the index, the inverted lists, the codes or the codebooks are in hand before the
call, queries and output buffers are on the device, and a pass is one call (or the two calls that
always go together, such as packing the queries and scanning the codes).  All cases of a process
share one GPUContext, as one serving process would.

A case is a dict with "kind" and sizes (N rows, D dimensions, Q queries, k results):

  index    AcceleratedVectorIndex.searchDevice over inserted rows; "metric"; "removed" rows are
           deleted first and not compacted (the index then searches with its deletion mask)
  rows     FusedTopKKernel.encode over raw fp32 rows (no index); "metric"
  int8     ScalarQuantizationKernel: quantize the queries, then the int8 scan + top-k
  hamming  BinaryQuantizationKernel: pack the queries, then the Hamming scan + top-k (D bits)
  ivf      IVFSearchPipeline.encodeSearch: coarse probe, list scan, top-k ("lists", "nprobe")
  pq       ProductQuantizationKernel's search: ADC tables, code scan, top-k (M x K codebooks)
  encode   ScalarQuantizationKernel: per-dimension parameters, then the codes of N rows
"""
from __future__ import annotations

import functools

import torch

from vectoraccelerate_amd import (
    AcceleratedVectorIndex,
    BinaryQuantizationKernel,
    FusedTopKKernel,
    FusedL2TopKParameters,
    GPUContext,
    HammingDistanceKernel,
    IndexConfiguration,
    IVFSearchConfiguration,
    IVFSearchPipeline,
    Metric,
    ScalarQuantizationKernel,
    VectorHandle,
)

_METRIC = {
    "euclidean": Metric.euclideanSquared,
    "cosine": Metric.cosine,
    "dotProduct": Metric.dotProduct,
}


def listed():
    return [
        # one interactive query over a small collection (the index of a desktop application or of
        # one tenant): nothing but launches and latency
        {"name": "index_5k_q1", "kind": "index", "metric": "euclidean", "N": 5000, "D": 128, "Q": 1, "k": 10},
        # one interactive query over a large collection: the rows are streamed once
        {"name": "index_1m_q1", "kind": "index", "metric": "euclidean", "N": 1_000_000, "D": 768, "Q": 1, "k": 10},
        # a serving batch over a collection of ordinary size; row count with no round factor
        {"name": "index_100k_q100", "kind": "index", "metric": "cosine", "N": 100_003, "D": 768, "Q": 100, "k": 10},
        # an offline batch over a large collection of long embeddings (the headline benchmark)
        {"name": "index_1m_q1024", "kind": "index", "metric": "cosine", "N": 1_000_000, "D": 1536, "Q": 1024, "k": 100},
        # maximum inner product over a plain array of rows, no index built: odd counts, short word vectors
        {"name": "rows_50k_q37", "kind": "rows", "metric": "dotProduct", "N": 49_999, "D": 300, "Q": 37, "k": 25},
        # a serving batch over int8 codes
        {"name": "int8_10m_q32", "kind": "int8", "N": 10_000_000, "D": 512, "Q": 32, "k": 10},
        # an offline batch over int8 codes
        {"name": "int8_10m_q4096", "kind": "int8", "N": 10_000_000, "D": 512, "Q": 4096, "k": 10},
        # candidate generation over sign bits (100 candidates a query, to be re-ranked by the caller)
        {"name": "hamming_10m_q100", "kind": "hamming", "N": 10_000_000, "D": 768, "Q": 100, "k": 100},
        # a serving batch over inverted lists, the configuration's "standard" preset
        {"name": "ivf_1m_q16", "kind": "ivf", "N": 1_000_000, "D": 768, "Q": 16, "k": 10, "lists": 1024, "nprobe": 16},
        # an offline batch over many inverted lists, the "large" preset
        {"name": "ivf_4m_q1024", "kind": "ivf", "N": 4_000_000, "D": 768, "Q": 1024, "k": 10, "lists": 4096, "nprobe": 32},
        # a serving batch over product-quantized codes
        {"name": "pq_10m_q64", "kind": "pq", "N": 10_000_000, "D": 768, "Q": 64, "k": 10, "M": 16, "K": 256},
        # coding a collection before it is scanned as int8
        {"name": "encode_1m", "kind": "encode", "N": 1_000_000, "D": 768, "Q": 0, "k": 0},
    ]


def _log_int(rng, lo, hi):
    """A whole number whose logarithm is uniform on [lo, hi]."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["index", "index", "index", "rows", "int8", "int8", "hamming", "ivf", "ivf", "pq", "encode"])
    k = rng.choice([1, 5, 10, 10, 20, 50, 100])
    if kind == "index":
        D = rng.choice([96, 128, 200, 256, 300, 384, 512, 768, 768, 1024, 1536])
        Q = _log_int(rng, 1, 1024)
        N = _log_int(rng, 5000, 1_000_000)
        removed = rng.choice([0, 0, 0, max(1, N // 100)])
        metric = rng.choice(["euclidean", "euclidean", "cosine", "dotProduct"])
        return {"kind": kind, "metric": metric, "N": N, "D": D, "Q": Q, "k": k, "removed": removed}
    if kind == "rows":
        D = rng.choice([50, 100, 127, 128, 300, 384, 513, 768])
        metric = rng.choice(["euclidean", "cosine", "dotProduct"])
        return {"kind": kind, "metric": metric, "N": _log_int(rng, 2000, 500_000), "D": D, "Q": _log_int(rng, 1, 512), "k": k}
    if kind == "int8":
        D = rng.choice([64, 128, 200, 256, 384, 512, 512, 768, 1024])
        return {"kind": kind, "N": _log_int(rng, 100_000, 5_000_000), "D": D, "Q": _log_int(rng, 1, 4096), "k": k}
    if kind == "hamming":
        D = rng.choice([128, 256, 384, 512, 768, 768, 1000, 1024])
        return {"kind": kind, "N": _log_int(rng, 100_000, 20_000_000), "D": D, "Q": _log_int(rng, 1, 256), "k": k}
    if kind == "ivf":
        lists, nprobe = rng.choice([(256, 8), (1024, 16), (1024, 8), (2048, 32)])
        N = _log_int(rng, lists * 100, 2_000_000)
        return {"kind": kind, "N": N, "D": rng.choice([96, 128, 384, 768, 768]), "Q": _log_int(rng, 1, 1024),
                "k": min(k, 50), "lists": lists, "nprobe": nprobe}
    if kind == "pq":
        D, M = rng.choice([(128, 8), (128, 16), (384, 32), (768, 16), (768, 32), (768, 64), (768, 48)])
        return {"kind": kind, "N": _log_int(rng, 100_000, 10_000_000), "D": D, "Q": _log_int(rng, 1, 256), "k": min(k, 50),
                "M": M, "K": 256}
    return {"kind": kind, "N": _log_int(rng, 10_000, 1_500_000), "D": rng.choice([100, 127, 128, 384, 512, 768, 1024]),
            "Q": 0, "k": 0}


# ---------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _context() -> GPUContext:
    return GPUContext(0)


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _removed_rows(case, g):
    """Rows deleted from the index before the search."""
    n = int(case.get("removed", 0))
    return torch.randperm(case["N"], device="cuda", generator=g)[:n]


def _vectors(case, g):
    """Rows N(0, 1), normalised for cosine; queries are rows with noise (a user's query lies near
    some rows of the collection)."""
    N, D, Q = case["N"], case["D"], case["Q"]
    x = torch.randn(N, D, device="cuda", generator=g)
    src = torch.randint(0, N, (Q,), device="cuda", generator=g)
    if case["metric"] == "cosine":
        x /= x.norm(dim=1, keepdim=True)
        q = x[src] + 0.05 * torch.randn(Q, D, device="cuda", generator=g)
        q /= q.norm(dim=1, keepdim=True)
    else:
        q = x[src] + torch.randn(Q, D, device="cuda", generator=g)
    return x, q.contiguous()


def _clustered(case, g):
    """Centroids, rows around them with Zipf(1.1) cluster sizes, and queries of the same mixture."""
    N, D, Q, C = case["N"], case["D"], case["Q"], case["lists"]
    cen = torch.randn(C, D, device="cuda", generator=g) * 4.0
    p = torch.tensor(_zipf(C), device="cuda")
    x = torch.randn(N, D, device="cuda", generator=g)
    lab = torch.multinomial(p, N, replacement=True, generator=g)
    for s in range(0, N, 1 << 19):
        x[s:s + (1 << 19)] += cen[lab[s:s + (1 << 19)]]
    qlab = torch.multinomial(p, Q, replacement=True, generator=g)
    q = (cen[qlab] + torch.randn(Q, D, device="cuda", generator=g)).contiguous()
    return cen, x, q


@functools.lru_cache(maxsize=None)
def _zipf(n: int):
    w = [1.0 / (i + 1) ** 1.1 for i in range(n)]
    total = sum(w)
    return tuple(v / total for v in w)


def _int8(case, g):
    """Database codes over the whole signed range (what the per-dimension min/max map gives for
    evenly spread values), the map's parameters, and fp32 queries inside the range."""
    N, D, Q = case["N"], case["D"], case["Q"]
    codes = torch.empty(N, D, device="cuda", dtype=torch.int8)
    for s in range(0, N, 1 << 20):
        e = min(N, s + (1 << 20))
        codes[s:e] = torch.randint(-128, 128, (e - s, D), device="cuda", generator=g, dtype=torch.int8)
    span = torch.rand(D, device="cuda", generator=g) * 1.5 + 0.5
    scale = (2.0 * span / 255.0).contiguous()
    zero_point = torch.zeros(D, device="cuda", dtype=torch.int32)
    q = ((torch.rand(Q, D, device="cuda", generator=g) * 2 - 1) * span).contiguous()
    return codes, scale, zero_point, q


def _bits(case, g):
    """Sign-bit codes of independent normal values (fair bits; the bits past D are zero) and fp32 queries."""
    N, D, Q = case["N"], case["D"], case["Q"]
    words = (D + 31) // 32
    codes = torch.randint(-2**31, 2**31 - 1, (N, words), device="cuda", generator=g, dtype=torch.int32)
    if D % 32:
        codes[:, -1] &= (1 << (D % 32)) - 1
    return codes, torch.randn(Q, D, device="cuda", generator=g)


def _pq(case, g):
    N, D, Q, M, K = case["N"], case["D"], case["Q"], case["M"], case["K"]
    books = torch.randn(M, K, D // M, device="cuda", generator=g)
    codes = torch.randint(0, K, (N, M), device="cuda", generator=g, dtype=torch.uint8)
    return books, codes, torch.randn(Q, D, device="cuda", generator=g)


def _encode_rows(case, g):
    N, D = case["N"], case["D"]
    span = torch.rand(D, device="cuda", generator=g) * 1.5 + 0.5
    return (torch.randn(N, D, device="cuda", generator=g) * span).contiguous()


def prepare(case, seed):
    c, g, kind = _context(), _generator(seed), case["kind"]
    N, D, Q, k = case["N"], case["D"], case["Q"], case["k"]
    s = {"case": case, "ctx": c}
    if kind == "encode":
        s.update(x=_encode_rows(case, g), mn=c.empty((D,), torch.float32), mx=c.empty((D,), torch.float32),
                 scale=c.empty((D,), torch.float32), zp=c.empty((D,), torch.int32),
                 codes=c.empty((N, D), torch.int8), sq=ScalarQuantizationKernel(c))
        return s
    s.update(idx=c.empty((Q, k), torch.int32),
             dist=c.empty((Q, k), torch.int32 if kind in ("int8", "hamming") else torch.float32))
    if kind == "index":
        x, s["q"] = _vectors(case, g)
        ix = AcceleratedVectorIndex(IndexConfiguration.flat(D, N, metric=case["metric"]), c)
        ix.insert(vectors=x)
        gone = _removed_rows(case, g).tolist()
        if gone:
            ix.remove([VectorHandle(r) for r in gone])
        s["index"] = ix
    elif kind == "rows":
        s["x"], s["q"] = _vectors(case, g)
        s.update(kernel=FusedTopKKernel(c), params=FusedL2TopKParameters(Q, N, D, k), metric=_METRIC[case["metric"]])
    elif kind == "int8":
        s["codes"], s["scale"], s["zp"], s["q"] = _int8(case, g)
        s.update(qcodes=c.empty((Q, D), torch.int8), sq=ScalarQuantizationKernel(c))
    elif kind == "hamming":
        s["codes"], s["q"] = _bits(case, g)
        s.update(qcodes=c.empty((Q, s["codes"].shape[1]), torch.int32), bq=BinaryQuantizationKernel(c),
                 hamming=HammingDistanceKernel(c))
    elif kind == "ivf":
        cen, x, s["q"] = _clustered(case, g)
        pipe = IVFSearchPipeline(c, IVFSearchConfiguration(case["lists"], case["nprobe"], D))
        s.update(pipe=pipe, structure=pipe.prepareIndexStructure(cen, x))
    else:
        s["books"], s["codes"], s["q"] = _pq(case, g)
    return s


def run(s):
    case, c = s["case"], s["ctx"]
    kind, N, D, Q, k = case["kind"], case["N"], case["D"], case["Q"], case["k"]
    if kind == "index":
        s["index"].searchDevice(s["q"], k, s["idx"], s["dist"])
    elif kind == "rows":
        s["kernel"].encode(s["q"], s["x"], s["idx"], s["dist"], s["params"], s["metric"])
    elif kind == "int8":
        s["sq"].encodeQuantize(s["q"], s["qcodes"], s["scale"], s["zp"], Q, D)
        s["sq"].encodeScanTopK(s["qcodes"], s["codes"], s["idx"], s["dist"], Q, N, D, k)
    elif kind == "hamming":
        s["bq"].encodeQuantize(s["q"], s["qcodes"], Q, D)
        s["hamming"].encodeTopK(s["qcodes"], s["codes"], s["idx"], s["dist"], Q, N, s["codes"].shape[1], k)
    elif kind == "ivf":
        s["pipe"].encodeSearch(s["q"], s["structure"], s["idx"], s["dist"], k)
    elif kind == "pq":
        c.check(c.lib.va_pq_search(c.handle, s["q"].data_ptr(), Q, D, case["M"], case["K"], s["books"].data_ptr(),
                                   s["codes"].data_ptr(), N, k, s["idx"].data_ptr(), s["dist"].data_ptr()),
                "va_pq_search")
    else:
        s["sq"].encodeComputeParameters(s["x"], N, D, s["mn"], s["mx"], s["scale"], s["zp"])
        s["sq"].encodeQuantize(s["x"], s["codes"], s["scale"], s["zp"], N, D)
        return {"min": s["mn"], "max": s["mx"], "scale": s["scale"], "zero_point": s["zp"], "codes": s["codes"]}
    return {"ids": s["idx"], "distances": s["dist"]}


def work(case):
    kind, N, D, Q, k = case["kind"], case["N"], case["D"], case["Q"], case["k"]
    out = 8.0 * Q * k
    if kind == "index":  # the fp16 copy the index keeps (fp32 rows where D % 4 != 0)
        return {"bytes": (2.0 if D % 4 == 0 else 4.0) * N * D + 4.0 * Q * D + out, "flops": 2.0 * Q * N * D}
    if kind == "rows":
        return {"bytes": 4.0 * N * D + 4.0 * Q * D + out, "flops": 2.0 * Q * N * D}
    if kind == "int8":
        return {"bytes": 1.0 * N * D + 4.0 * Q * D + out, "flops": 2.0 * Q * N * D}
    if kind == "hamming":
        return {"bytes": N * ((D + 31) // 32) * 4.0 + 4.0 * Q * D + out, "flops": 2.0 * Q * N * D}
    if kind == "ivf":
        # a query probes its own cluster's list and nprobe - 1 others; a list is read once a call
        C, nprobe = case["lists"], case["nprobe"]
        rows = pairs = 0.0
        for p in _zipf(C):
            hit = min(1.0, p + (nprobe - 1) / C)
            rows += N * p * (1.0 - (1.0 - hit) ** Q)
            pairs += N * p * hit * Q
        return {"bytes": 2.0 * rows * D + 4.0 * (C + Q) * D + out, "flops": 2.0 * D * (pairs + Q * C)}
    if kind == "pq":  # one addition per looked-up entry
        return {"bytes": 1.0 * N * case["M"] + 4.0 * (Q + case["K"]) * D + out,
                "flops": 1.0 * Q * N * case["M"] + 3.0 * Q * case["K"] * D}
    return {"bytes": 5.0 * N * D + 16.0 * D, "flops": 4.0 * N * D}


def tolerance(case):
    """Whole-number paths are exact.  A float search returns fp32 distances, about four times what
    the fp32 results measure against 64 bits: rel 6e-7 at most, ids swapped only where distances tie
    within that.  The inverted lists hold rows whose norms are several times their distances
    (|q|^2 + |x|^2 - 2 q.x cancels), which measures 8e-6 and 0.3% of ids in another order."""
    if case["kind"] in ("int8", "hamming", "encode"):
        return "exact"
    if case["kind"] == "ivf":
        return {"rel": 3.3e-5, "max": 1.3e-4, "differ": 0.01}
    return {"rel": 2.5e-6, "max": 1e-5, "differ": 0.002}


# ---------------------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------------------
def _chunks(n, step):
    return [(s, min(n, s + step)) for s in range(0, n, step)]


def _smallest(blocks, k):
    """The k smallest columns over blocks of a Q x N matrix, ascending, +inf where there are fewer."""
    best = None
    for d in blocks:
        if d.shape[1] > k:
            d = torch.topk(d, k, dim=1, largest=False).values
        best = d if best is None else torch.cat([best, d], 1)
    best = torch.sort(best, dim=1).values[:, :k]
    if best.shape[1] < k:
        pad = torch.full((best.shape[0], k - best.shape[1]), float("inf"), device=best.device, dtype=best.dtype)
        best = torch.cat([best, pad], 1)
    return best


def _distances(metric, q, x):
    dot = q @ x.T
    if metric == "dotProduct":
        return -dot
    if metric == "cosine":
        return 1.0 - dot / (q.norm(dim=1)[:, None] * x.norm(dim=1)[None, :])
    return ((q * q).sum(1)[:, None] + (x * x).sum(1)[None, :] - 2.0 * dot).clamp_(min=0.0)


def exact(case, seed):
    kind, N, Q, k = case["kind"], case["N"], case["Q"], case["k"]
    g = _generator(seed)
    if kind in ("int8", "hamming"):
        return None
    if kind == "encode":
        x = _encode_rows(case, g)
        mn, mx = x.amin(0).double(), x.amax(0).double()
        return {"min": mn, "max": mx, "scale": ((mx - mn) / 255.0).clamp(min=1e-8), "zero_point": None, "codes": None}
    step = max(1 << 12, min(1 << 18, (1 << 28) // max(Q, 1)))
    if kind == "pq":
        books, codes, q = _pq(case, g)
        M, K = case["M"], case["K"]
        sub = q.double().view(Q, M, -1)
        tables = torch.stack([((sub[:, m, None, :] - books[m].double()[None]) ** 2).sum(-1) for m in range(M)])

        def blocks():
            for s, e in _chunks(N, step):
                acc = torch.zeros(Q, e - s, device="cuda", dtype=torch.float64)
                for m in range(M):
                    acc += tables[m][:, codes[s:e, m].long()]
                yield acc

        return {"ids": None, "distances": _smallest(blocks(), k).sqrt()}
    if kind == "ivf":
        cen, x, q = _clustered(case, g)
        cen, q = cen.double(), q.double()
        probes = torch.topk(_distances("euclidean", q, cen), case["nprobe"], dim=1, largest=False).indices
        probed = torch.zeros(Q, case["lists"], device="cuda", dtype=torch.bool).scatter_(1, probes, True)

        def blocks():
            for s, e in _chunks(N, step):
                xs = x[s:e].double()
                near = torch.cat([_distances("euclidean", xs[a:b], cen).argmin(1) for a, b in _chunks(e - s, 1 << 16)])
                yield _distances("euclidean", q, xs).masked_fill_(~probed[:, near], float("inf"))

        return {"ids": None, "distances": _smallest(blocks(), k)}
    x, q = _vectors(case, g)
    gone = torch.zeros(N, device="cuda", dtype=torch.bool)
    if kind == "index":
        gone[_removed_rows(case, g)] = True
    q = q.double()

    def blocks():
        for s, e in _chunks(N, step):
            yield _distances(case["metric"], q, x[s:e].double()).masked_fill_(gone[s:e][None, :], float("inf"))

    return {"ids": None, "distances": _smallest(blocks(), k)}
