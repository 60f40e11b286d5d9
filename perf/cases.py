"""Performance cases: the SpGEMM work a program has this package do, through
its public entry points.

  listed()             the named cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  operands (and the plan or server a program keeps)
  run(state)           one pass; returns the products whole
  work(case)           bytes and operations one pass cannot do without
  exact(case, seed)    the same products from plain torch in 64 bits

Operands are made on the GPU with torch, in torch's memory, and handed to the
package as DeviceCSR views.  The case fixes the sparsity pattern up to a
relabelling of rows and columns, so that nnz(C) is the case's own; the seed
draws the relabelling and the values.  Products are returned as torch views of
the package's device arrays (row pointer, columns, values).
"""
import math

import numpy as np
import torch

import brmerge_amd as bm
from brmerge_amd.spgemm import DeviceArray

DEV = "cuda"


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest calls: coarse AMG levels, small graphs; launches and
        # host round trips are what they cost
        {"name": "er_2048", "kind": "product", "family": "er", "rows": 2048, "dmin": 8, "dmax": 8, "upper": False},
        # 16,384^2, 8 per row: the Erdos-Renyi product of the benchmark
        {"name": "er_16384", "kind": "product", "family": "er", "rows": 16384, "dmin": 8, "dmax": 8, "upper": False},
        # AMG setup on a 96^3 grid: R = P^T, A*P, R*(A*P) with a 27-point
        # stencil and a 3x3x3 aggregation
        {"name": "galerkin_96", "kind": "galerkin", "n": 96, "g": 3},
        # a banded operator times another: 4-32 entries per row, half-width 64
        {"name": "banded_40009", "kind": "product", "family": "banded", "rows": 40009, "dmin": 4, "dmax": 32,
         "upper": False},
        # more than a million unknowns, ragged rows of 4-20 entries
        {"name": "er_1500007", "kind": "product", "family": "er", "rows": 1500007, "dmin": 4, "dmax": 20,
         "upper": False},
        # power-law graphs A*A (R-MAT 0.57/0.19/0.19/0.05, 16 edges per row):
        # a small one, a large one, and BRMerge-Upper's row waves of C-bar
        {"name": "rmat_14", "kind": "product", "family": "rmat", "scale": 14, "upper": False},
        {"name": "rmat_18", "kind": "product", "family": "rmat", "scale": 18, "upper": False},
        {"name": "rmat_17_upper", "kind": "product", "family": "rmat", "scale": 17, "upper": True},
        # many independent products (rows 256-65,536, half Erdos-Renyi, half
        # banded): fused in one call, and replayed by a plan kept for fixed
        # patterns
        {"name": "batch_192", "kind": "batch", "pairs": 192, "plan": False},
        {"name": "plan_192", "kind": "batch", "pairs": 192, "plan": True},
        # a burst of requests (log-normal rows, median 4,096, 8-24 per row)
        # against resident R-MAT-18 operands
        {"name": "serve_20", "kind": "serve", "requests": 20, "resident": 4, "scale": 18},
        # the drop-in call on host arrays, as a program of the reference makes it
        {"name": "host_rmat_12", "kind": "host", "scale": 12},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["er", "er", "banded", "rmat", "rmat", "galerkin", "batch", "serve", "host"])
    if kind in ("er", "banded"):
        rows = _log_int(rng, 700, 1400000)
        dmin = rng.randint(1, 12)
        return {"kind": "product", "family": kind, "rows": rows, "dmin": dmin, "dmax": dmin + rng.randint(0, 16),
                "upper": rng.random() < 0.3}
    if kind == "rmat":
        return {"kind": "product", "family": "rmat", "scale": rng.randint(10, 17), "edges": rng.randint(5, 19),
                "upper": rng.random() < 0.4}
    if kind == "galerkin":
        return {"kind": "galerkin", "n": _log_int(rng, 12, 120), "g": rng.choice([2, 3, 4])}
    if kind == "batch":
        return {"kind": "batch", "pairs": _log_int(rng, 3, 190), "plan": rng.random() < 0.5}
    if kind == "serve":
        return {"kind": "serve", "requests": rng.randint(2, 20), "resident": rng.randint(1, 4),
                "scale": rng.randint(14, 18)}
    return {"kind": "host", "scale": rng.randint(9, 13), "edges": rng.randint(5, 16)}


# ------------------------------------------------------------------ operands
class Mat:
    """A CSR operand in torch's device memory, and the package's view of it."""

    def __init__(self, rpt, col, val, M, N):
        self.rpt, self.col, self.val, self.M, self.N, self.nnz = rpt, col, val, M, N, int(col.numel())
        self.dev = bm.DeviceCSR(DeviceArray(rpt.data_ptr(), M + 1, np.int32),
                                DeviceArray(col.data_ptr(), self.nnz, np.int32),
                                DeviceArray(val.data_ptr(), self.nnz, np.float64), M, N, self.nnz)

    def bytes(self):
        return 4 * (self.M + 1) + 12 * self.nnz


def _gen(seed, k=0):
    return torch.Generator(device=DEV).manual_seed((seed * 1000003 + k * 7919 + 17) % (1 << 62))


def _pattern_gen(k):
    """Draws operand k's pattern: the same for every seed."""
    return torch.Generator(device=DEV).manual_seed(424243 + 7919 * k)


def _shift(seed, M):
    """Rows and columns are relabelled i -> (i + shift) mod M, a small shift
    that depends on M alone beside the seed, so that hubs and bands stay where
    they are and A's columns keep naming the same rows of B."""
    return (seed * 2654435761 >> 7) % min(64, M)


def _from_keys(keys, M, N, gen):
    """CSR of the distinct keys row * N + column; values uniform in [-1, 1]."""
    keys = torch.unique(keys)
    rows = torch.div(keys, N, rounding_mode="floor")
    rpt = torch.zeros(M + 1, dtype=torch.int64, device=DEV)
    rpt[1:] = torch.cumsum(torch.bincount(rows, minlength=M), 0)
    col = (keys - rows * N).to(torch.int32)
    val = torch.rand(col.numel(), dtype=torch.float64, device=DEV, generator=gen) * 2 - 1
    return rpt.to(torch.int32), col, val


def _ragged_rows(M, dmin, dmax, gen):
    """Row index of every drawn entry: dmin to dmax of them per row."""
    deg = torch.randint(dmin, dmax + 1, (M,), device=DEV, generator=gen)
    return torch.repeat_interleave(torch.arange(M, device=DEV), deg)


def _relabelled(rows, cols, M, N, seed, k):
    keys = (rows + _shift(seed, M)) % M * N + (cols + _shift(seed, N)) % N
    return Mat(*_from_keys(keys, M, N, _gen(seed, k)), M, N)


def er(M, N, dmin, dmax, seed, k=0):
    gen = _pattern_gen(k)
    rows = _ragged_rows(M, dmin, dmax, gen)
    cols = torch.randint(0, N, (rows.numel(),), device=DEV, generator=gen)
    return _relabelled(rows, cols, M, N, seed, k)


def banded(M, dmin, dmax, seed, k=0, half=64):
    gen = _pattern_gen(k)
    rows = _ragged_rows(M, dmin, dmax, gen)
    cols = rows + torch.randint(-half, half + 1, (rows.numel(),), device=DEV, generator=gen)
    return _relabelled(rows, cols.clamp_(0, M - 1), M, M, seed, k)


def rmat(scale, seed, k=0, edges=16):
    gen = _pattern_gen(k)
    n = 1 << scale
    row = torch.zeros(n * edges, dtype=torch.int64, device=DEV)
    col = torch.zeros_like(row)
    for _ in range(scale):
        u = torch.rand(row.numel(), dtype=torch.float64, device=DEV, generator=gen)
        down = u >= 0.76  # quadrants a, b above; c, d below
        right = ((u >= 0.57) & (u < 0.76)) | (u >= 0.95)
        row = row * 2 + down
        col = col * 2 + right
    return _relabelled(row, col, n, n, seed, k)


def stencil27(n, seed):
    """27-point stencil on an n^3 grid, 26 on the diagonal and -1 off it, with
    coefficients perturbed by up to a tenth."""
    gen = _gen(seed, 1)
    i = torch.arange(n ** 3, device=DEV)
    z, y, x = i // (n * n), (i // n) % n, i % n
    keys = []
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                ok = ((z + dz >= 0) & (z + dz < n) & (y + dy >= 0) & (y + dy < n) & (x + dx >= 0) & (x + dx < n))
                keys.append((i * n ** 3 + i + (dz * n + dy) * n + dx)[ok])
    rpt, col, val = _from_keys(torch.cat(keys), n ** 3, n ** 3, gen)
    rows = torch.repeat_interleave(torch.arange(n ** 3, device=DEV), torch.diff(rpt).long())
    val = torch.where(col.long() == rows, 26.0, -1.0) * (1.0 + 0.1 * val)
    return Mat(rpt, col, val, n ** 3, n ** 3)


def aggregation(n, g, seed):
    """n^3 x ceil(n/g)^3 prolongator: one entry per row."""
    gen = _gen(seed, 2)
    m = -(-n // g)
    i = torch.arange(n ** 3, device=DEV)
    agg = ((i // (n * n)) // g * m + ((i // n) % n) // g) * m + (i % n) // g
    val = 1.0 + 0.1 * torch.rand(n ** 3, dtype=torch.float64, device=DEV, generator=gen)
    return Mat(torch.arange(n ** 3 + 1, dtype=torch.int32, device=DEV), agg.to(torch.int32), val, n ** 3, m ** 3)


def _spread(i, n, lo, hi):
    """The i-th of n sizes spread evenly over the logarithm of [lo, hi], in a
    fixed shuffled order."""
    step = next(s for s in range(int(0.618 * n) | 1, 2 * n + 3) if math.gcd(s, n) == 1)
    return int(round(math.exp(math.log(lo) + (((i * step) % n) + 0.5) / n * (math.log(hi) - math.log(lo)))))


def batch_pairs(n, seed):
    """Square pairs, rows 256 to 65,536, 4-32 entries per row; even ones
    Erdos-Renyi, odd ones banded."""
    pairs = []
    for i in range(n):
        M = _spread(i, n, 256, 65536)
        if i % 2 == 0:
            pairs.append((er(M, M, 4, 32, seed, 2 * i), er(M, M, 4, 32, seed, 2 * i + 1)))
        else:
            pairs.append((banded(M, 4, 32, seed, 2 * i), banded(M, 4, 32, seed, 2 * i + 1)))
    return pairs


def serve_requests(n, scale, seed):
    """A operands of n requests: rows log-normal (median 4,096, sigma 1.5, the
    n quantiles in a fixed shuffled order), 8-24 columns per row."""
    step = next(s for s in range(int(0.618 * n) | 1, 2 * n + 3) if math.gcd(s, n) == 1)
    out = []
    for i in range(n):
        q = (((i * step) % n) + 0.5) / n
        z = float(torch.erfinv(torch.tensor(2.0 * q - 1.0, dtype=torch.float64))) * math.sqrt(2.0)
        M = max(1, int(round(math.exp(math.log(4096) + 1.5 * z))))
        out.append(er(M, 1 << scale, 8, 24, seed, 100 + i))
    return out


def operands(case, seed):
    """(A, B) of a single product."""
    f = case["family"]
    if f == "rmat":
        A = rmat(case["scale"], seed, edges=case.get("edges", 16))
        return A, A
    if f == "er":
        A = er(case["rows"], case["rows"], case["dmin"], case["dmax"], seed, 1)
        return A, (A if case["dmin"] == case["dmax"] else
                   er(case["rows"], case["rows"], case["dmin"], case["dmax"], seed, 2))
    A = banded(case["rows"], case["dmin"], case["dmax"], seed, 1)
    return A, banded(case["rows"], case["dmin"], case["dmax"], seed, 2)


# ------------------------------------------------------------------ results
class _Span:
    """A device array of the package as torch sees it; keeps its owner alive."""

    def __init__(self, owner, ptr, n, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False), "version": 2}


class Held:
    """What one state keeps between passes: the last pass's products (given
    back before the next pass), its plan or server.  The products' torch views
    keep it alive.  When the last state is gone, the package's cached device
    memory goes back to the driver, for torch to use."""

    alive = 0

    def __init__(self):
        Held.alive += 1
        self.free = []
        self.plan = None
        self.server = None

    def release(self):
        for C in self.free:
            C.free()
        self.free = []

    def __del__(self):
        try:
            self.release()
            if self.plan is not None:
                self.plan.close()
            if self.server is not None:
                self.server.close()
            Held.alive -= 1
            if Held.alive == 0:
                bm.lib().brm_dev_trim()
        except Exception:
            pass


_TYPES = {"<i4": torch.int32, "<i8": torch.int64, "<f8": torch.float64}


def _view(st, slot, ptr, n, typestr):
    """Torch view of n elements at ptr; made again only when they moved."""
    if n == 0:
        return torch.empty(0, dtype=_TYPES[typestr], device=DEV)
    got = st["views"].get(slot)
    if got is None or got[0] != (ptr, n):
        got = ((ptr, n), torch.as_tensor(_Span(st["held"], ptr, n, typestr), device=DEV))
        st["views"][slot] = got
    return got[1]


def _csr(st, slot, C):
    t = "<i8" if C.rpt.dtype == np.int64 else "<i4"
    return [_view(st, (slot, 0), C.rpt.ptr, C.M + 1, t), _view(st, (slot, 1), C.col.ptr, C.nnz, "<i4"),
            _view(st, (slot, 2), C.val.ptr, C.nnz, "<f8")]


# ------------------------------------------------------------------ the passes
def prepare(case, seed):
    if bm.lib().brm_init(0) != 0:
        raise RuntimeError("no HIP device")
    kind = case["kind"]
    st = {"case": case, "held": Held(), "views": {}}
    if kind == "product":
        st["A"], st["B"] = operands(case, seed)
    elif kind == "galerkin":
        st["A"], st["P"] = stencil27(case["n"], seed), aggregation(case["n"], case["g"], seed)
    elif kind == "batch":
        st["pairs"] = batch_pairs(case["pairs"], seed)
        st["dev"] = [(A.dev, B.dev) for A, B in st["pairs"]]
        torch.cuda.synchronize()
        if case["plan"]:
            # the default tier shapes, without the tuner: a plan tuned anew by
            # timing would not be the same plan twice
            st["held"].plan = bm.BatchPlan(st["dev"], autotune=False)
    elif kind == "serve":
        st["B"] = [rmat(case["scale"], seed, k) for k in range(case["resident"])]
        st["A"] = serve_requests(case["requests"], case["scale"], seed)
        torch.cuda.synchronize()
        srv = bm.Server(budget_bytes=64 << 30)
        st["held"].server = srv
        st["ids"] = [srv.add_b(B.dev) for B in st["B"]]
        st["rids"] = []
    else:
        A = rmat(case["scale"], seed, edges=case.get("edges", 16))
        st["host"] = bm.CSR(A.rpt.cpu().numpy(), A.col.cpu().numpy(), A.val.cpu().numpy(), A.M, A.N)
    torch.cuda.synchronize()
    return st


def run(st):
    case, held = st["case"], st["held"]
    kind = case["kind"]
    held.release()
    if kind == "product":
        C = bm.spgemm_dev(st["A"].dev, st["B"].dev, upper=case["upper"])
        held.free = [C]
        return _csr(st, "C", C)
    if kind == "galerkin":
        P = st["P"].dev
        R = P.transpose()
        AP = bm.spgemm_dev(st["A"].dev, P)
        op = AP.as_operand()
        RAP = bm.spgemm_dev(R, op)
        held.free = [R, AP, op.rpt, RAP]
        return {"R": _csr(st, "R", R), "AP": _csr(st, "AP", AP), "RAP": _csr(st, "RAP", RAP)}
    if kind == "batch":
        if case["plan"]:
            held.plan.execute()
            C, _ = held.plan.result()
        else:
            C, _ = bm.spgemm_batched(st["dev"])
            held.free = [C]
        return _csr(st, "C", C)
    if kind == "serve":
        srv = held.server
        for r in st["rids"]:
            srv.release(r)
        st["rids"] = [srv.submit(st["ids"][i % len(st["ids"])], A.dev) for i, A in enumerate(st["A"])]
        out = []
        for i, r in enumerate(st["rids"]):
            g = srv.wait(r)
            out.append([_view(st, (i, 0), g.crpt, g.M + 1, "<i8"), _view(st, (i, 1), g.ccol, g.nnz, "<i4"),
                        _view(st, (i, 2), g.cval, g.nnz, "<f8")])
        return out
    C = bm.brmerge_precise(st["host"], st["host"])
    return [C.rpt, C.col, C.val]


# ------------------------------------------------------------------ what a pass cannot do without
def _products(A, B):
    return int(torch.diff(B.rpt)[A.col.long()].sum())


def _size(v):
    if isinstance(v, dict):
        return sum(_size(x) for x in v.values())
    if isinstance(v, (list, tuple)):
        return sum(_size(x) for x in v)
    return v.nbytes if isinstance(v, np.ndarray) else v.numel() * v.element_size()


def work(case):
    """Bytes: every operand read once, every product written once.  Operations:
    a multiply and an add per intermediate product.  Counted on seed 0."""
    st = prepare(case, 0)
    kind = case["kind"]
    out = _size(run(st))
    if kind == "product":
        A, B = st["A"], st["B"]
        return {"bytes": out + A.bytes() + (B.bytes() if B is not A else 0), "flops": 2 * _products(A, B)}
    if kind == "galerkin":
        A, P = st["A"], st["P"]
        # P is read to be transposed and as an operand; R*(A*P) has one product per entry of A*P
        ap = int(run(st)["AP"][1].numel())
        return {"bytes": out + A.bytes() + P.bytes(), "flops": 2 * (_products(A, P) + ap)}
    if kind == "batch":
        return {"bytes": out + sum(A.bytes() + B.bytes() for A, B in st["pairs"]),
                "flops": 2 * sum(_products(A, B) for A, B in st["pairs"])}
    if kind == "serve":
        nb = len(st["B"])
        # the B rows that the requests select
        bts = sum(A.bytes() for A in st["A"])
        for k, B in enumerate(st["B"]):
            used = torch.zeros(B.M, dtype=torch.bool, device=DEV)
            for A in st["A"][k::nb]:
                used[A.col.long()] = True
            bts += int(torch.diff(B.rpt)[used].sum()) * 12
        return {"bytes": out + bts, "flops": 2 * sum(_products(A, st["B"][i % nb]) for i, A in enumerate(st["A"]))}
    A = st["host"]
    lens = np.diff(A.rpt)
    return {"bytes": out + 4 * (A.M + 1) + 12 * A.nnz, "flops": 2 * int(lens[A.col].sum())}


# ------------------------------------------------------------------ the same products in 64 bits
EXACT_PRODUCTS = 3 * 10 ** 8
_CHUNK = 5 * 10 ** 7


def _multiply(Arpt, Acol, Aval, Brpt, Bcol, Bval, M, N):
    """C = A * B: expand, sort by (row, column), add up; in chunks of rows."""
    Arpt, Acol, Brpt = Arpt.long(), Acol.long(), Brpt.long()
    blen = torch.diff(Brpt)
    ends = torch.zeros(Acol.numel() + 1, dtype=torch.int64, device=DEV)
    ends[1:] = torch.cumsum(blen[Acol], 0)
    row_end = ends[Arpt]
    lens = torch.zeros(M, dtype=torch.int64, device=DEV)
    cols, vals = [], []
    r0 = 0
    row_end_h = row_end.cpu().numpy()
    while r0 < M:
        r1 = max(r0 + 1, int(np.searchsorted(row_end_h, row_end_h[r0] + _CHUNK, side="right")) - 1)
        r1 = min(r1, M)
        e0, e1 = int(Arpt[r0]), int(Arpt[r1])
        e = torch.arange(e0, e1, device=DEV)
        n = blen[Acol[e0:e1]]
        src = torch.repeat_interleave(e, n)
        at = torch.arange(int(n.sum()), device=DEV) - (ends[src] - ends[e0]) + Brpt[Acol[src]]
        rows = torch.repeat_interleave(torch.arange(r0, r1, device=DEV), torch.diff(Arpt[r0:r1 + 1]))
        rows = torch.repeat_interleave(rows, n)
        key, perm = torch.sort(rows * N + Bcol[at].long(), stable=True)
        v = (Aval[src] * Bval[at])[perm]
        del rows, src, at, perm
        uk, inv = torch.unique_consecutive(key, return_inverse=True)
        s = torch.zeros(uk.numel(), dtype=torch.float64, device=DEV).index_add_(0, inv, v)
        ur = torch.div(uk, N, rounding_mode="floor")
        lens += torch.bincount(ur, minlength=M)
        cols.append((uk - ur * N).to(torch.int32))
        vals.append(s)
        r0 = r1
    rpt = torch.zeros(M + 1, dtype=torch.int64, device=DEV)
    rpt[1:] = torch.cumsum(lens, 0)
    return [rpt, torch.cat(cols), torch.cat(vals)]


def _mul(A, B):
    return _multiply(A.rpt, A.col, A.val, B.rpt, B.col, B.val, A.M, B.N)


def _transposed(A):
    rows = torch.repeat_interleave(torch.arange(A.M, device=DEV), torch.diff(A.rpt).long())
    key, perm = torch.sort(A.col.long() * A.M + rows)
    rpt = torch.zeros(A.N + 1, dtype=torch.int64, device=DEV)
    rpt[1:] = torch.cumsum(torch.bincount(A.col.long(), minlength=A.N), 0)
    return [rpt.to(torch.int32), (key % A.M).to(torch.int32), A.val[perm]]


def exact(case, seed):
    kind = case["kind"]
    if kind == "product":
        A, B = operands(case, seed)
        return None if _products(A, B) > EXACT_PRODUCTS else _mul(A, B)
    if kind == "galerkin":
        A, P = stencil27(case["n"], seed), aggregation(case["n"], case["g"], seed)
        R = _transposed(P)
        AP = _mul(A, P)
        return {"R": R, "AP": AP, "RAP": _multiply(*R, *AP, P.N, P.N)}
    if kind == "batch":
        parts = [_mul(A, B) for A, B in batch_pairs(case["pairs"], seed)]
        rpt, base = [torch.zeros(1, dtype=torch.int64, device=DEV)], 0
        for p in parts:
            rpt.append(p[0][1:] + base)
            base += int(p[0][-1])
        return [torch.cat(rpt), torch.cat([p[1] for p in parts]), torch.cat([p[2] for p in parts])]
    if kind == "serve":
        Bs = [rmat(case["scale"], seed, k) for k in range(case["resident"])]
        return [_mul(A, Bs[i % len(Bs)]) for i, A in enumerate(serve_requests(case["requests"], case["scale"], seed))]
    A = rmat(case["scale"], seed, edges=case.get("edges", 16))
    r, c, v = _mul(A, A)
    return [r.to(torch.int32).cpu().numpy(), c.cpu().numpy(), v.cpu().numpy()]
