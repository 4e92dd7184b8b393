"""Performance cases of the library's public entry points on one GPU.

Each case is one call as a program makes it, with the matrices it brings:

* ``plain``    ``lu_batched_inverse`` (one n, in place).  The program keeps its
  matrices, so a pass copies them into the working buffer (``copy_kernel``)
  and inverts that.
* ``lapack``   ``lu_batched_inverse_lapack``: the same with ``ipiv`` / ``info``.
* ``refined``  ``lu_batched_inverse_refined``: out of place, one refinement step.
* ``verify``   ``residual``: the library's check of computed inverses.
* ``ragged``   ``lu_batched_inverse_ragged`` with a kept plan: mixed n, packed
  in the order of arrival.
* ``serve``    a burst of requests through ``Server``: submit, progress until
  all are done, take the results, release.

Sizes are those of the reference's sweep (n up to 32, up to a million
matrices), of the benchmark's workloads (1M x n = 32; 500k mixed n in 2..32;
100k refined; requests of up to 4096 matrices of n in 4..32), and small calls.

Matrices hold U[-1,1) entries plus 2 sqrt(n) on the diagonal, their rows in
random order where the rule finds any row (not for ``none``, nor for ``tree``,
which at most sizes cannot reach every row): condition numbers of a few units
and no growth at every n, so every entry of the result has a meaning in FP32.
"""
import math
from types import SimpleNamespace

import torch

import matrixinversion_amd as mia
from matrixinversion_amd._native import check, lib
from matrixinversion_amd.serve import Server

DEV = "cuda"
RULES = {"none": mia.PIVOT_NONE, "parallel": mia.PIVOT_PARALLEL, "serial": mia.PIVOT_SERIAL, "tree": mia.PIVOT_TREE,
         "gepp": mia.PIVOT_GEPP}
EXACT_CHUNK = 1 << 25  # matrix entries inverted at once in 64 bits


def listed():
    return [
        # one small system of an interactive program: latency
        {"name": "plain_n16_b100", "kind": "plain", "n": 16, "batch": 100, "pivot": "parallel"},
        # a million tiny odd-sized matrices (finite elements, 6-dof + 1 blocks)
        {"name": "plain_n7_1M", "kind": "plain", "n": 7, "batch": 1000000, "pivot": "parallel"},
        # positive definite inputs that need no pivoting, batch not a multiple of a tile
        {"name": "plain_n20_none_333k", "kind": "plain", "n": 20, "batch": 333333, "pivot": "none"},
        # the benchmark's headline configuration
        {"name": "plain_n32_1M", "kind": "plain", "n": 32, "batch": 1000000, "pivot": "parallel"},
        # the reference's exact tree rule at an odd size
        {"name": "plain_n27_tree_150k", "kind": "plain", "n": 27, "batch": 150001, "pivot": "tree"},
        # a LAPACK program: partial pivoting, interchanges and info
        {"name": "lapack_n32_gepp_250k", "kind": "lapack", "n": 32, "batch": 250000, "pivot": "gepp"},
        # the benchmark's refinement batch
        {"name": "refined_n32_100k", "kind": "refined", "n": 32, "batch": 100000, "pivot": "parallel"},
        # refinement of small matrices
        {"name": "refined_n12_300k", "kind": "refined", "n": 12, "batch": 300000, "pivot": "parallel"},
        # the check of a sweep's results, as the harness makes it after each size
        {"name": "verify_n32_500k", "kind": "verify", "n": 32, "batch": 500000},
        # a mid-sized mixed batch, as a server coalesces it
        {"name": "ragged_3k", "kind": "ragged", "n_lo": 4, "n_hi": 32, "batch": 3000, "pivot": "parallel"},
        # the benchmark's mixed batch
        {"name": "ragged_500k", "kind": "ragged", "n_lo": 2, "n_hi": 32, "batch": 500000, "pivot": "parallel"},
        # a burst of mixed requests at the server
        {"name": "serve_32req", "kind": "serve", "n_lo": 4, "n_hi": 32, "requests": 32, "batch": 8192,
         "pivot": "parallel"},
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["plain", "plain", "plain", "lapack", "refined", "verify", "ragged", "ragged", "serve"])
    if kind in ("ragged", "serve"):
        n_lo = rng.randint(1, 24)
        case = {"kind": kind, "n_lo": n_lo, "n_hi": rng.randint(n_lo + 1, 32)}
        if kind == "ragged":
            case["batch"] = _log_uniform(rng, 32, 500000)
        else:
            case["requests"] = rng.randint(4, 64)
            case["batch"] = _log_uniform(rng, 256, 32768)
        case["pivot"] = rng.choice(["parallel", "parallel", "none", "tree", "gepp"])
        return case
    most = {"plain": 1000000, "lapack": 500000, "refined": 300000, "verify": 500000}[kind]
    case = {"kind": kind, "n": rng.randint(1, 32), "batch": _log_uniform(rng, 16, most)}
    if kind == "lapack":
        case["pivot"] = rng.choice(["parallel", "gepp"])
    elif kind != "verify":
        case["pivot"] = rng.choice(["parallel", "parallel", "none", "serial", "tree", "gepp"])
    return case


# ------------------------------------------------------------------ inputs


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _permutations(gen, ns, permute):
    """(len(ns), 32) int64: row i holds a random permutation of 0..ns[i]-1
    (the identity without `permute`), then 32s up to column 31."""
    cols = torch.arange(32, device=DEV)
    out = torch.where(cols < ns[:, None], cols, 32)
    if permute:
        key = torch.rand(out.shape, generator=gen, device=DEV) + (out == 32)
        out = torch.where(cols < ns[:, None], key.argsort(dim=1), 32)
    return out


def _packed(gen, ns, permute):
    """Packed matrices of sizes ns: (flat FP32, offsets, pivot offsets)."""
    sizes = ns * ns
    ends, pends = sizes.cumsum(0), ns.cumsum(0)
    offsets, poffs = ends - sizes, pends - ns
    flat = torch.rand(int(ends[-1]), generator=gen, device=DEV).mul_(2).sub_(1)
    for lo in range(0, ns.numel(), 1 << 18):  # bounded index tensors
        s, o = ns[lo:lo + (1 << 18)], offsets[lo:lo + (1 << 18)]
        perm = _permutations(gen, s, permute)
        live = perm < 32
        at = (o[:, None] + perm * s[:, None] + torch.arange(32, device=DEV))[live]
        flat[at] += (2.0 * s.double().sqrt()).float()[:, None].expand(-1, 32)[live]
    return flat, offsets, poffs


def _sizes(case, gen):
    """The sizes of a case's matrices, int64: equally many of each, in random order."""
    if "n" in case:
        return torch.full((case["batch"],), case["n"], dtype=torch.int64, device=DEV)
    order = torch.rand(case["batch"], generator=gen, device=DEV).argsort()
    return case["n_lo"] + order % (case["n_hi"] - case["n_lo"] + 1)


def _inputs(case, seed):
    """(sizes, packed matrices, offsets, pivot offsets) of an inversion case."""
    gen = _generator(seed)
    ns = _sizes(case, gen)
    return (ns, *_packed(gen, ns, case["pivot"] not in ("none", "tree")))


def _verify_inputs(case, seed):
    """A = D + u v^T and its inverse in FP32 (Sherman-Morrison in FP64); one
    matrix in eight carries an error that the check's threshold sees."""
    gen = _generator(seed)
    b, n = case["batch"], case["n"]

    def rand(*shape):
        return torch.rand(*shape, generator=gen, device=DEV)

    d, u, v = 1 + rand(b, n), (rand(b, n) * 2 - 1) / math.sqrt(n), (rand(b, n) * 2 - 1) / math.sqrt(n)
    a, x = torch.empty(b, n, n, device=DEV), torch.empty(b, n, n, device=DEV)
    scale = (rand(b) < 0.125) * 1e-2 * rand(b)
    step = max(1, EXACT_CHUNK // (n * n))
    for lo in range(0, b, step):
        s = slice(lo, lo + step)
        d64, u64, v64 = d[s].double(), u[s].double(), v[s].double()
        a[s] = (torch.diag_embed(d64) + u64[:, :, None] * v64[:, None, :]).float()
        w = 1 + (u64 * v64 / d64).sum(1)
        x64 = torch.diag_embed(1 / d64) - (u64 / d64)[:, :, None] * (v64 / d64)[:, None, :] / w[:, None, None]
        x[s] = (x64 * (1 + scale[s].double()[:, None, None])).float()
    return a, x


def _view(t):
    """A tensor's memory as the library's buffer argument."""
    return SimpleNamespace(ptr=t.data_ptr(), nbytes=t.numel() * t.element_size())


def prepare(case, seed):
    kind = case["kind"]
    s = SimpleNamespace(case=case, stream=SimpleNamespace(handle=torch.cuda.current_stream().cuda_stream))
    if kind == "verify":
        s.a, s.x = _verify_inputs(case, seed)
        return s
    s.ns, s.a, offsets, poffs = _inputs(case, seed)
    s.flags = RULES[case["pivot"]]
    s.x = torch.empty_like(s.a)
    s.piv = torch.zeros(int(s.ns.sum()), dtype=torch.int32, device=DEV)
    s.va, s.vx, s.vpiv = _view(s.a), _view(s.x), _view(s.piv)
    if kind == "lapack":
        s.info = torch.zeros(case["batch"], dtype=torch.int32, device=DEV)
    elif kind == "ragged":
        s.ns32 = s.ns.int()
        s.offsets, s.poffs = offsets, poffs
        s.vns, s.voff, s.vpoff = _view(s.ns32), _view(offsets), _view(poffs)
        s.plan = mia.RaggedPlan(case["batch"])
    elif kind == "serve":
        budget = 2 * (s.a.numel() + s.piv.numel()) * 4 + (1 << 20)
        s.server = Server(budget, max_batch=case["batch"], ring_slots=2 * case["batch"])
        cuts = torch.linspace(0, case["batch"], case["requests"] + 1).long().tolist()
        host_ns = s.ns.int().cpu().numpy()
        at, pat, s.requests = 0, 0, []
        for lo, hi in zip(cuts[:-1], cuts[1:]):
            ns = host_ns[lo:hi]
            floats, pivs = int((ns.astype("int64") ** 2).sum()), int(ns.sum())
            s.requests.append((s.a.data_ptr() + at * 4, ns, s.x.data_ptr() + at * 4, floats * 4,
                               s.piv.data_ptr() + pat * 4, pivs * 4))
            at, pat = at + floats, pat + pivs
    return s


# ----------------------------------------------------------------- one pass


def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "plain":
        n, batch = case["n"], case["batch"]
        mia.device.copy_kernel(s.vx, s.va, batch * n * n, s.stream)
        mia.lu_batched_inverse(s.vx, n, batch, s.flags, s.vpiv, s.stream)
        return s.x, s.piv
    if kind == "lapack":
        n, batch = case["n"], case["batch"]
        mia.device.copy_kernel(s.vx, s.va, batch * n * n, s.stream)
        check(lib().lu_batched_inverse_lapack(s.vx.ptr, s.vpiv.ptr, s.info.data_ptr(), n, batch, s.flags,
                                              s.stream.handle), "lu_batched_inverse_lapack")
        return s.x, s.piv, s.info
    if kind == "refined":
        check(lib().lu_batched_inverse_refined(s.va.ptr, s.vx.ptr, s.vpiv.ptr, case["n"], case["batch"], s.flags,
                                               s.stream.handle), "lu_batched_inverse_refined")
        return s.x, s.piv
    if kind == "verify":
        return mia.residual(_view(s.a), _view(s.x), case["n"], case["batch"])
    if kind == "ragged":
        mia.device.copy_kernel(s.vx, s.va, s.a.numel(), s.stream)
        mia.lu_batched_inverse_ragged(s.vx, s.voff, s.vns, case["batch"], s.flags, s.vpiv, s.vpoff, s.plan, s.stream)
        return s.x, s.piv
    return _serve(s)


def _serve(s):
    server, waiting = s.server, {}
    for r in s.requests:
        t = server.submit(r[0], r[1], s.flags)
        if t is None:
            raise RuntimeError("the server's budget holds every request of the burst")
        waiting[t] = r
        server.progress()
    done = []
    while waiting:
        server.progress()
        for t in server.poll():
            _, _, dst, nbytes, pdst, pbytes = waiting.pop(t)
            _, res, piv, _ = server.query(t)
            check(lib().lubx_memcpy_dtod_async(dst, res, nbytes, s.stream.handle), "memcpy D2D")
            if piv:
                check(lib().lubx_memcpy_dtod_async(pdst, piv, pbytes, s.stream.handle), "memcpy D2D")
            done.append(t)
    torch.cuda.current_stream().synchronize()  # the results have left the arena
    for t in done:
        server.release(t)
    return s.x, s.piv


# ------------------------------------------------------------- what it is


def _moments(case):
    """(sum of n, sum of n^2, sum of n^3) over the case's matrices (up to the
    last incomplete round of sizes)."""
    ns = [case["n"]] if "n" in case else range(case["n_lo"], case["n_hi"] + 1)
    per = case["batch"] / len(ns)
    return tuple(per * sum(n ** p for n in ns) for p in (1, 2, 3))


def work(case):
    s1, s2, s3 = _moments(case)
    if case["kind"] == "verify":
        return {"bytes": 8 * s2, "flops": 2 * s3}
    pivots = 0 if case["pivot"] == "none" and case["kind"] == "serve" else 4 * s1
    extra = {"lapack": 4, "ragged": 20}.get(case["kind"], 0) * case["batch"]  # info; offset, size, pivot offset
    return {"bytes": 8 * s2 + pivots + extra, "flops": (6 if case["kind"] == "refined" else 2) * s3}


def tolerance(case):
    if case["kind"] == "verify":
        return "exact"  # counts, and FP32 sums in a stated order
    # four times the errors measured against `exact` over listed and drawn cases
    # (FP32 elimination: 1.5e-7 and 1.1e-6; refined: 2.9e-8 and 6e-8)
    return {"rel": 1.2e-7, "max": 2.5e-7} if case["kind"] == "refined" else {"rel": 6e-7, "max": 4e-6}


def exact(case, seed):
    if case["kind"] == "verify":
        a, x = _verify_inputs(case, seed)
        n, worst = case["n"], 0.0
        step = max(1, EXACT_CHUNK // (n * n))
        eye = torch.eye(n, dtype=torch.float64, device=DEV)
        for lo in range(0, case["batch"], step):
            r = torch.bmm(a[lo:lo + step].double(), x[lo:lo + step].double()) - eye
            worst = max(worst, float(r.abs().max()))
        return None, worst
    ns, flat, offsets, _ = _inputs(case, seed)
    out = torch.empty(flat.numel(), dtype=torch.float64, device=DEV)
    for n in sorted(set(ns.tolist())):
        entries = torch.arange(n * n, device=DEV)
        of_n = offsets[ns == n]
        step = max(1, EXACT_CHUNK // (n * n))
        for lo in range(0, of_n.numel(), step):
            at = of_n[lo:lo + step, None] + entries
            out[at] = _inverse64(flat[at].double().view(-1, n, n)).view(-1, n * n)
    return (out, None, None) if case["kind"] == "lapack" else (out, None)


def _inverse64(a):
    """Inverses by Gauss-Jordan with partial pivoting, rows in place."""
    b, n, _ = a.shape
    m = torch.cat([a, torch.eye(n, dtype=a.dtype, device=a.device).repeat(b, 1, 1)], 2)
    rows = torch.arange(b, device=a.device)
    for k in range(n):
        p = m[:, k:, k].abs().argmax(1) + k
        top = m[rows, p].clone()
        m[rows, p] = m[:, k].clone()
        top = top / top[:, k:k + 1]
        m = m - m[:, :, k:k + 1] * top[:, None, :]
        m[:, k] = top
    return m[:, :, n:].contiguous()
