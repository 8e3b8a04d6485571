"""What this library is timed on: the jobs of its users at the sizes they come in.

Five paths, each through the Python binding's public entry points:

  nmf       one logged window of the factorisation A ~ W H: log_every = 10 multiplicative updates
            of W and H and the loss (MuNmf.run), matrix and factors resident on the GPU
  job       a whole small factorisation from host buffers to host buffers: load, normalise, drop
            empty columns, create the context, 50 updates with their logged losses, W and H back
  fit       new examples against a fixed sparse H: first stage, 25 updates of W with the logged
            loss, W back (Learner)
  load      a PEF block from host buffers to a normalised, pruned device matrix, and that matrix
            back for host tools
  topk      the k largest entries of dense per-example Fisher rows (topk_rows)
  sparsify  unit-norm components of H cut at a threshold (op_dot, op_threshold_compact)

Everything is fp32 with 32-bit column ids: the one data type of the path."""

import math

import numpy as np
import torch

import npeff_ref_amd as d

NMF_ITERS = 10
FIT_ITERS = 25
JOB_ITERS = 50


def listed():
    return [
        # a toy matrix, as in a first try or a unit test: launches and host work are all there is
        dict(name="nmf_toy", path="nmf", n=48, m_full=2000, k=64, k_min=0, zipf=1.1, r=8),
        # the smallest configuration of the benchmark
        dict(name="nmf_512x1M_r16", path="nmf", n=512, m_full=1 << 20, k=4096, k_min=0, zipf=1.1, r=16),
        # a rank and sizes that no tile divides
        dict(name="nmf_ragged_sizes_r50", path="nmf", n=777, m_full=3_000_017, k=5003, k_min=0, zipf=1.1, r=50),
        # an ordinary run at the rank the analyses use most: the benchmark's downscaled configuration
        dict(name="nmf_1000x11M_r128", path="nmf", n=1000, m_full=11_000_000, k=16_384, k_min=0, zipf=1.1, r=128),
        # a large one: a steeper column law, twice the rank, factors of several GB
        dict(name="nmf_2000x20M_r256", path="nmf", n=2000, m_full=20_000_000, k=32_768, k_min=0, zipf=1.3, r=256),
        # rows of very different lengths at a high rank
        dict(name="nmf_ragged_rows_r512", path="nmf", n=1500, m_full=6_000_000, k=65_536, k_min=1024, zipf=1.1,
             r=512),
        # everything the factorisation tool does between reading its input file and writing its output file
        dict(name="job_300x400k_r20", path="job", n=300, m_full=400_000, k=2048, k_min=0, zipf=1.1, r=20),
        # coefficients of a handful of new examples
        dict(name="fit_100x200k_r20", path="fit", n=100, m_full=200_000, k=1000, zipf=1.1, r=20, density=0.02),
        # a large batch of new examples: the benchmark's shape with fewer examples and columns
        dict(name="fit_2000x22M_r256", path="fit", n=2000, m_full=22_000_000, k=32_768, zipf=1.1, r=256,
             density=0.01),
        # the loader of both tools: transfer, normalisation, pruning of rare columns
        dict(name="load_1000x16384", path="load", n=1000, m_full=11_000_000, k=16_384, zipf=1.1, keep="count"),
        # the sparsifier at the size of a full model: few rows of 1e8 values each
        dict(name="topk_2x110M", path="topk", n=2, count=110_000_000, k=65_536),
        # components of H of a mid-sized model
        dict(name="sparsify_4x6M", path="sparsify", n=4, count=6_000_000, density=0.01),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rank(rng, hi):
    """Half the users take a round rank, the others what their analysis asks for."""
    if rng.random() < 0.5:
        return rng.choice([q for q in (8, 16, 32, 64, 128, 256, 512) if q <= hi])
    return _log_int(rng, 4, hi)


def draw(rng):
    path = rng.choice(["nmf", "nmf", "nmf", "nmf", "job", "fit", "fit", "load", "topk", "topk", "sparsify"])
    zipf = rng.choice([1.1, 1.1, 1.3])
    if path == "nmf":
        r = _rank(rng, 512)
        n = _log_int(rng, 32, 2000)
        k = _log_int(rng, max(n, 64), 32_768)
        m_full = _log_int(rng, 8 * k, min(20_000_000, 2000 * k))
        # no more factor than the largest listed case holds
        m_full = max(8 * k, min(m_full, 5_000_000_000 // r))
        ragged = rng.random() < 0.25
        return dict(path=path, n=n, m_full=m_full, k=k, k_min=max(n, k // 64) if ragged and n < k else 0, zipf=zipf,
                    r=r)
    if path == "job":
        n = _log_int(rng, 32, 400)
        k = _log_int(rng, n, 4096)
        return dict(path=path, n=n, m_full=_log_int(rng, 8 * k, 500_000), k=k, k_min=0, zipf=zipf, r=_rank(rng, 64))
    if path == "fit":
        n = _log_int(rng, 16, 2000)
        k = _log_int(rng, 256, 32_768)
        return dict(path=path, n=n, m_full=_log_int(rng, 16 * k, 22_000_000) if 16 * k < 22_000_000 else 16 * k, k=k,
                    zipf=zipf, r=_rank(rng, 256), density=rng.choice([0.005, 0.01, 0.02]))
    if path == "load":
        n = _log_int(rng, 16, 1000)
        k = _log_int(rng, 64, 16_384)
        return dict(path=path, n=n, m_full=_log_int(rng, 8 * k, 11_000_000), k=k, zipf=zipf,
                    keep=rng.choice(["count", "list"]))
    if path == "topk":
        count = _log_int(rng, 20_000, 110_000_000)
        n = max(1, min(64, _log_int(rng, 1, 220_000_000 // count)))
        return dict(path=path, n=n, count=count, k=_log_int(rng, 64, min(65_536, count // 8)))
    return dict(path=path, n=rng.randint(1, 4), count=_log_int(rng, 20_000, 6_000_000),
                density=rng.choice([0.002, 0.01, 0.05]))


class _Mem:
    """Device memory of the library as torch sees it; a tensor on it keeps its owner alive."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<f4", data=(int(ptr), False), version=2)


def _tensor(owner, ptr, shape):
    return torch.as_tensor(_Mem(owner, ptr, shape), device="cuda")


def _quiet(_line):
    pass


def _synth(case, seed):
    if case.get("k_min", 0) > 0:
        return d.Csr.synth(case["n"], case["m_full"], k_min=case["k_min"], k_max=case["k"], zipf_s=case["zipf"],
                           seed=seed)
    return d.Csr.synth(case["n"], case["m_full"], k_fixed=case["k"], zipf_s=case["zipf"], seed=seed)


def _entries(case, seed):
    """Rows as the producer writes them, on the host: (rowptr, cols, vals, norms).  Distinct columns by
    a Zipf law, log-normal values, row norms.  The examples come in another order and with other values
    for every seed; how many columns they hold between them, and so the shape of H, is the case's."""
    A, _ = _synth(case, 20230)
    rowptr, cols, _ = A.download()
    A.close()
    n, lens = case["n"], np.diff(rowptr)
    order = np.random.default_rng(seed).permutation(n)
    if case.get("k_min", 0) > 0:
        first = np.concatenate(([0], np.cumsum(lens[order])))
        cols = np.concatenate([cols[rowptr[i]:rowptr[i + 1]] for i in order])
        rowptr = first.astype(np.int64)
    else:
        cols = cols.reshape(n, -1)[order].reshape(-1)
    g = torch.Generator(device="cuda").manual_seed(seed)
    v = torch.empty(len(cols), device="cuda").normal_(-8.0, 2.0, generator=g).exp_()
    sq = torch.cumsum(v.double() ** 2, 0)
    ends = torch.cat([sq.new_zeros(1), sq])[torch.from_numpy(rowptr).cuda()]
    norms = (ends[1:] - ends[:-1]).clamp_(min=0).sqrt_().float().cpu().numpy()
    return rowptr, cols, v.cpu().numpy(), norms


def _pef_on_host(case, seed):
    _, cols, vals, norms = _entries(case, seed)
    return cols.reshape(case["n"], -1), vals.reshape(case["n"], -1), norms


def _sparse_H(r, m, density, seed):
    """r x m in CSR on the host, every entry present with the given probability, values in [0, 1)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    many = int(r * m * density * 1.02) + 4096
    u = torch.rand(many, generator=g, device="cuda", dtype=torch.float64).clamp_(min=1e-12)
    at = torch.cumsum(torch.ceil(torch.log(u) / math.log1p(-density)).clamp_(min=1).to(torch.int64), 0) - 1
    at = at[at < r * m]
    rowptr = torch.searchsorted(at, torch.arange(r + 1, device="cuda", dtype=torch.int64) * m)
    vals = torch.rand(at.numel(), generator=g, device="cuda")
    return rowptr.cpu().numpy(), (at % m).to(torch.int32).cpu().numpy(), vals.cpu().numpy()


def _dense_rows(n, count, seed, shuffle=None):
    """Per-example squared gradients: log-normal over many orders of magnitude; `shuffle`: in another order
    for every such seed."""
    x = d.DeviceArray((n, count))
    t = _tensor(x, x.ptr.value, (n, count))
    g = torch.Generator(device="cuda").manual_seed(seed)
    t.normal_(-8.0, 2.0, generator=g).exp_()
    if shuffle is not None:
        t.copy_(t[:, torch.randperm(count, generator=g.manual_seed(shuffle), device="cuda")])
    torch.cuda.synchronize()
    return x


def prepare(case, seed):
    path = case["path"]
    if path == "nmf":
        rowptr, cols, vals, norms = _entries(case, seed)
        A = d.Csr.from_host(rowptr, cols, vals, case["m_full"])
        A.normalize_rows(norms)
        A.compact_columns(1)
        nmf = d.MuNmf(A, d.MuNmfParams(rank=case["r"], max_iters=NMF_ITERS, seed=seed, log_every=NMF_ITERS))
        nmf.initialize()
        return dict(path=path, A=A, nmf=nmf)
    if path == "job":
        cols, vals, norms = _pef_on_host(case, seed)
        params = d.MuNmfParams(rank=case["r"], max_iters=JOB_ITERS, seed=seed)
        return dict(path=path, cols=cols, vals=vals, norms=norms, m_full=case["m_full"], params=params)
    if path == "fit":
        A, norms = _synth(case, seed)
        A.normalize_rows(norms)
        rowptr, cols, vals = _sparse_H(case["r"], case["m_full"], case["density"], seed)
        H = d.Csr.from_host(rowptr, cols, vals, case["m_full"])
        return dict(path=path, A=A, H=H, params=d.LearnerParams(max_iters=FIT_ITERS, seed=seed))
    if path == "load":
        cols, vals, norms = _pef_on_host(case, seed)
        kept = None
        if case["keep"] == "list":  # the columns an earlier factorisation kept
            rng = np.random.default_rng(20230)
            kept = np.flatnonzero(rng.random(case["m_full"], dtype=np.float32) < 0.6).astype(np.int32)
        return dict(path=path, cols=cols, vals=vals, norms=norms, m_full=case["m_full"], kept=kept)
    if path == "topk":
        return dict(path=path, x=_dense_rows(case["n"], case["count"], seed), k=case["k"])
    rows = [_dense_rows(1, case["count"], 20230 + i, shuffle=seed + i) for i in range(case["n"])]
    # the threshold that leaves about the density asked for on unit-norm log-normal rows
    t = math.sqrt(2.0) * float(torch.erfinv(torch.tensor(1.0 - 2.0 * case["density"], dtype=torch.float64)))
    return dict(path=path, rows=rows, threshold=math.exp(2.0 * t - 4.0) / math.sqrt(case["count"]))


def run(state):
    path = state["path"]
    if path == "nmf":
        nmf = state["nmf"]
        history = nmf.run(log=_quiet)
        w, h = nmf.device_factors()
        r = nmf.params.rank
        return dict(losses=[loss for _, loss, _ in history], W=_tensor(nmf, w, (nmf.n_rows, r)),
                    H=_tensor(nmf, h, (nmf.n_cols, r)))
    if path == "job":
        A = d.Csr.from_pef(state["cols"], state["vals"], state["m_full"])
        A.normalize_rows(state["norms"])
        A.compact_columns(1)
        nmf = d.MuNmf(A, state["params"])
        history = nmf.run(log=_quiet)
        out = dict(losses=[loss for _, loss, _ in history], W=nmf.loadWToHostSync(), H=nmf.loadHToHostSync(),
                   kept=A.kept_indices())
        nmf.close()
        A.close()
        return out
    if path == "fit":
        learner = d.Learner(state["A"], state["H"], state["params"])
        history = learner.Run(log=_quiet)
        out = dict(losses=[[ref, true] for _, ref, true, _ in history], W=learner.GetOnHost_W())
        learner.close()
        return out
    if path == "load":
        A = d.Csr.from_pef(state["cols"], state["vals"], state["m_full"])
        A.normalize_rows(state["norms"])
        if state["kept"] is None:
            A.compact_columns(2)
        else:
            A.retain_columns(state["kept"])
        out = dict(csr=A.download(), kept=A.kept_indices(), sq_norm=A.sq_norm())
        A.close()
        return out
    if path == "topk":
        vals, idx, norms = d.topk_rows(state["x"], state["k"])
        return dict(vals=vals, idx=idx, norms=norms)
    out = []
    for x in state["rows"]:
        norm = math.sqrt(d.op_dot(x, x))
        idx, vals = d.op_threshold_compact(x, norm, state["threshold"])
        out.append(dict(norm=norm, idx=idx, vals=vals))
    return out


def _mean_entries(case):
    """Entries per row on average (ragged rows: uniform in the logarithm between the two bounds)."""
    lo, hi = case.get("k_min", 0), case["k"]
    return float(hi) if lo <= 0 or lo >= hi else (hi - lo) / math.log(hi / lo)


def _kept_columns(case, at_least=1):
    """Columns that at least so many rows are expected to hold (1 or 2), from the Zipf law the entries are drawn by."""
    n, m, k = case["n"], case["m_full"], min(_mean_entries(case), case["m_full"] - 1.0)
    edges = np.unique(np.floor(np.geomspace(1, m + 1, 600)))
    width = np.diff(edges)
    mid = np.sqrt(edges[:-1] * np.maximum(edges[1:] - 1, edges[:-1]))
    p = mid ** -case["zipf"]
    p /= (p * width).sum()
    lo, hi = 0.0, 60.0
    for _ in range(60):  # draws per row that leave k distinct columns
        t = math.exp((lo + hi) / 2)
        lo, hi = (lo, (lo + hi) / 2) if (width * -np.expm1(-t * p)).sum() > k else ((lo + hi) / 2, hi)
    held = -np.expm1(-math.exp(lo) * p)
    none = (1.0 - held) ** n
    one = n * held * (1.0 - held) ** (n - 1) if at_least > 1 else 0.0
    return max(1.0, float((width * (1.0 - none - one)).sum()))


def work(case):
    path, n = case["path"], float(case["n"])
    if path in ("nmf", "job"):
        r, z, m = float(case["r"]), case["n"] * _mean_entries(case), _kept_columns(case)
        # an iteration reads A in either order, reads H for A H^T, reads and writes H and W in their updates
        step_bytes = 2 * 8 * z + 4 * r * (3 * m + 3 * n)
        step_flops = 4 * z * r + (m + n) * (r * (r + 1) + 2 * r * r)
        if path == "nmf":
            return dict(bytes=NMF_ITERS * step_bytes, flops=NMF_ITERS * step_flops)
        # and once: the block and the norms in, both factors and the kept ids out
        return dict(bytes=JOB_ITERS * step_bytes + 8 * z + 4 * n + 4 * r * (m + n) + 4 * m,
                    flops=JOB_ITERS * step_flops)
    if path == "fit":
        r, z, m = float(case["r"]), n * case["k"], float(case["m_full"])
        zh = r * m * case["density"]
        first = 8 * z + 8 * zh + 4 * n * r + 4 * r * r
        # an update reads W and A H^T, writes W and (W itself being read for the next) nothing else
        return dict(bytes=first + FIT_ITERS * 12 * n * r + 4 * n * r,
                    flops=2 * z * r * case["density"] + zh * r * case["density"] + (FIT_ITERS + 1) * 2 * n * r * r)
    if path == "load":
        z = n * case["k"]
        if case["keep"] == "list":
            left, m, extra = 0.6 * z, 0.6 * case["m_full"], 0.6 * 4 * case["m_full"]
        else:
            m = _kept_columns(case, 2)
            left, extra = z - (_kept_columns(case) - m), 0.0
        return dict(bytes=8 * z + 4 * n + extra + 8 * left + 8 * n + 4 * m, flops=2 * z)
    if path == "topk":
        return dict(bytes=n * (4 * case["count"] + 8 * case["k"] + 4), flops=2 * n * case["count"])
    return dict(bytes=n * case["count"] * (4 + 8 * case["density"]), flops=3 * n * case["count"])


def tolerance(case):
    if case["path"] == "load":  # IEEE division and moves; ||A||^2 is a sum in fp64
        return dict(rel=1e-9, max=1e-9)
    if case["path"] in ("topk", "sparsify"):  # moves, fp32 division and fp64 sums rounded to fp32
        return dict(rel=2e-7, max=2e-7)
    return dict(rel=2e-5)  # fp32 sums in another order, carried through the updates
