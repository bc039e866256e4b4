"""What the speed of this framework is measured on: sparse tensor contractions
through the public Python entry points (SpTC, Plan, Batch, Server), from calls
of a few thousand nonzeros, where launches and waits are the time, to 1e9
intermediate products, where HBM is.

A case is a dict of plain values.  `kind` says how the call is made:
  contract  SpTC on device tensors, the result's entries left on the device
  plan      Plan kept, execute(), the entries decoded into torch tensors
  host      SpTC on numpy tensors, the entries decoded into numpy arrays
  count     SpTC count_only under a memory budget (nnz and value sum)
  chain     SpTC, its result contracted again from device memory
  batch     Batch kept, one hipGraph replay over all its instances
  serve     a burst of requests to a Server that holds the tensors
Tensors are drawn like the synthetic workloads of gsparc_amd/workloads.py:
distinct coordinates, Zipf or uniform modes, uniform(0, 1] or lognormal
values.
"""
import functools
import math

import numpy as np
import torch

from gsparc_amd import sptc
from gsparc_amd.coo import COOTensor

GIB = 1 << 30


# ---- cases -----------------------------------------------------------------

def _pair(name, kind, dims_x, zipf_x, nnz_x, cx, dims_y=None, zipf_y=None, nnz_y=0, cy=None, idx_bytes=4,
          values="uniform", acc=0, **more):
    """One contraction; without dims_y the tensor is contracted with itself."""
    c = {"name": name, "kind": kind, "dims_x": _text(dims_x), "zipf_x": _text(zipf_x), "nnz_x": nnz_x, "cx": _text(cx),
         "dims_y": _text(dims_y or ()), "zipf_y": _text(zipf_y or ()), "nnz_y": nnz_y, "cy": _text(cy or cx),
         "idx_bytes": idx_bytes, "values": values, "acc": acc}
    c.update(more)
    return c


def _text(v):
    return ",".join(str(x) for x in v)


def listed():
    return [
        # a script's small tensor, numpy in and numpy out: the default form of the API
        _pair("host_small", "host", (300, 200, 60), (1.1, 1.1, 0), 2_000, (2,)),
        # the same kind of call inside a GPU program: launches and waits only
        _pair("device_tiny", "contract", (300, 200, 60), (1.1, 1.1, 0), 3_001, (2,)),
        # the framework's small configuration: rows of one or two owners, 8e7 products
        _pair("plain_small", "contract", (2000, 2000, 500), (1.1, 1.1, 0), 200_000, (2,)),
        # operands prepared once, executed often, order 4 with two contracted modes, ragged sizes
        _pair("plan_order4", "plan", (1213, 347, 5003, 91), (1.1, 1.1, 1.1, 1.1), 250_007, (2, 3)),
        # the benchmark's shape at a third of its nonzeros: long rows of many owners, 1e9 products
        _pair("nips_third", "contract", (2482, 2862, 14036, 17), (1.2, 1.2, 1.2, 0), 1_000_000, (2, 3), values="lognormal"),
        # rows of a large tensor against the whole of it, counted under a budget that cuts it into chunks
        _pair("nell2_rows", "count", (12092, 9184, 28818), (1.1, 1.1, 1.1), 30_000, (2,), (12092, 9184, 28818),
              (1.1, 1.1, 1.1), 1_000_000, (2,), budget_gib=8),
        # large operands, 64-bit indices, a contract field too wide for a table and few matches: linearize, sort and match
        _pair("sparse_match", "contract", (9001, 6007, 12007, 9011), (0, 0, 0, 0), 8_000_000, (2, 3), (12007, 9011, 5003, 701),
              (0, 0, 0, 0), 3_000_001, (0, 1), idx_bytes=8, values="lognormal"),
        # tensor times a sparse matrix: narrow output columns, the dense row accumulator's case
        _pair("ttm_narrow", "contract", (4001, 301, 64), (0, 0, 0), 600_000, (2,), (64, 901), (0, 0), 19_000, (0,)),
        # the dense accumulator asked for (-d 1) over a wide column space: its tiled form
        _pair("dense_tiled", "contract", (2003, 1500, 400), (0, 1.1, 1.1), 40_000, (2,), acc=1),
        # Z = (X x Y) x W with the intermediate kept on the device
        _pair("chain_two", "chain", (400, 300, 50), (1.1, 1.1, 0), 9_000, (2,), (50, 250), (0, 1.1), 2_000, (0,),
              dims_w="250,111", zipf_w="1.1,0", nnz_w=6_000),
        # many contractions of the batch distribution in one launch sequence
        {"name": "batch_16", "kind": "batch", "instances": 16, "shape_seed": 3, "ir_cap": 4_000_000},
        # requests that arrive together at the server
        {"name": "serve_12", "kind": "serve", "instances": 12, "shape_seed": 11, "ir_cap": 1_000_000},
    ]


def _self_share(dims, zipf, modes):
    """Chance that two draws agree on `modes`: products per pair of nonzeros."""
    q = 1.0
    for m in modes:
        if zipf[m]:
            p = np.arange(1, dims[m] + 1, dtype=np.float64) ** -zipf[m]
            p /= p.sum()
            q *= float((p * p).sum())
        else:
            q /= dims[m]
    return q


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["contract"] * 8 + ["plan"] * 3 + ["host", "count", "count", "chain", "ttm", "ttm", "tiled", "match", "match",
                      "batch", "batch", "serve"])
    if kind in ("batch", "serve"):
        return {"kind": kind, "instances": rng.randint(4, 16), "shape_seed": rng.randrange(1 << 20),
                "ir_cap": int(_log(rng, 1e5, 4e6 if kind == "batch" else 1e6))}
    idx_bytes, values = rng.choice([4, 4, 8]), rng.choice(["uniform", "uniform", "lognormal"])
    if kind == "ttm":
        c, cols = rng.randint(20, 200), rng.randint(60, 4000)
        rows = (rng.randint(50, 5000), rng.randint(20, 400))
        nx = int(min(_log(rng, 2e3, 6e5), rows[0] * rows[1] * c // 8))
        per = max(16, cols // rng.randint(3, 8))
        nx = min(nx, 200_000_000 // per)
        return _pair("", "contract", rows + (c,), (0, 0, 0), nx, (2,), (c, cols), (0, 0), int(c * per * 0.9), (0,), idx_bytes, values)
    if kind == "match":
        dx = (rng.randint(3000, 12000), rng.randint(3000, 12000))
        cd = (rng.randint(3000, 13000), rng.randint(3000, 13000))
        nx, ny = int(_log(rng, 1e5, 8e6)), int(_log(rng, 1e5, 4e6))
        return _pair("", "contract", dx + cd, (0, 0, 0, 0), nx, (2, 3), cd + (rng.randint(300, 6000), rng.randint(300, 900)),
                     (0, 0, 0, 0), ny, (0, 1), idx_bytes, values)
    order = rng.choice([3, 3, 4])
    dims = tuple(int(_log(rng, 100, 20000)) for _ in range(order))
    zipf = tuple(rng.choice([0, 1.1, 1.1, 1.2]) for _ in range(order))
    cx = tuple(sorted(rng.sample(range(order), rng.choice([1, 1, 2]) if order == 4 else 1)))
    q = _self_share(dims, zipf, cx)
    top = {"contract": 6e8, "plan": 2e8, "host": 2e5, "count": 8e8, "chain": 3e5, "tiled": 4e6}[kind]
    space = math.prod(dims) // 8
    if kind == "count":
        ny = int(min(1_000_000, space, _log(rng, 1e5, 1e6)))
        nx = max(500, min(ny, int(_log(rng, 1e7, top) / (ny * q))))
        return _pair("", "count", dims, zipf, nx, cx, dims, zipf, ny, cx, idx_bytes, values, budget_gib=rng.choice([8, 16, 64]))
    nnz = int(max(500, min(math.sqrt(_log(rng, 3e4, top) / q), 1_500_000, space)))
    if kind == "chain":
        m = rng.randint(60, 400)
        w = rng.randint(30, 300)
        c = dims[cx[0]]
        return _pair("", "chain", dims, zipf, min(nnz, 20_000), cx[:1], (c, m), (0, 0), max(100, min(c * m // 9, 3_000)), (0,), idx_bytes,
                     values, dims_w=_text((m, w)), zipf_w="0,0", nnz_w=m * w // 8 + 1)
    if kind == "tiled":
        return _pair("", "contract", dims, zipf, nnz, cx, idx_bytes=idx_bytes, values=values, acc=rng.choice([1, 2]))
    return _pair("", kind, dims, zipf, nnz, cx, idx_bytes=idx_bytes, values=values)


# ---- tensors -----------------------------------------------------------------

class Tensor:
    """A COO tensor on the device, as the entry points take it (on_device=True)."""

    def __init__(self, dims, idx, val):
        self.dims, self.order, self.idx, self.val, self.nnz = dims, len(dims), idx, val, int(val.numel())


def _numbers(text, of=int):
    return tuple(of(x) for x in text.split(",")) if text else ()


def _zipf_cdf(d, s):
    return torch.cumsum(torch.arange(1, d + 1, dtype=torch.float64, device="cuda") ** -s, 0)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _make(dims, zipf, nnz, values, idx_bytes, seed, k, labels):
    """nnz distinct coordinates (fewer when the modes' heads are full) drawn
    from the sizes and k, so that every seed's tensors hold as many entries and
    give as many outputs; the seed turns each mode's indices by a shift
    (labels[m]: modes of one label turn together), orders the entries and draws
    the values."""
    g = _generator(nnz * 64 + k)
    nnz = min(nnz, max(1, math.prod(dims) // 2))
    cdf = [_zipf_cdf(d, s) if s else None for d, s in zip(dims, zipf)]
    have = torch.empty(0, dtype=torch.int64, device="cuda")
    for _ in range(12):
        n = int((nnz - have.numel()) * 1.2) + 64
        key = torch.zeros(n, dtype=torch.int64, device="cuda")
        for d, c in zip(dims, cdf):
            u = torch.rand(n, dtype=torch.float64, device="cuda", generator=g)
            i = (u * d).long() if c is None else torch.searchsorted(c, u * c[-1], right=True)
            key = key * d + i.clamp_(max=d - 1)
        have = torch.unique(torch.cat([have, key]))
        if have.numel() >= nnz:
            break
    have = have[torch.randperm(have.numel(), device="cuda", generator=g)[:nnz]]
    g = _generator(seed * 64 + k)
    have = have[torch.randperm(have.numel(), device="cuda", generator=g)]
    idx = []
    for d, label in reversed(list(zip(dims, labels))):
        turn = np.random.RandomState([seed & 0xFFFFFFFF, label]).randint(d)
        idx.append(((have % d + turn) % d).to(torch.int64 if idx_bytes == 8 else torch.int32).contiguous())
        have = have // d
    n = idx[0].numel()
    if values == "lognormal":
        val = torch.randn(n, dtype=torch.float64, device="cuda", generator=g).exp().float()
    else:
        val = 1.0 - torch.rand(n, dtype=torch.float32, device="cuda", generator=g)
    return Tensor(tuple(dims), idx[::-1], val)


def _operands(c, seed):
    """X and Y of a contraction (Y is X for a self-contraction), W of a chain."""
    def one(s, k, shared):
        dims = _numbers(c["dims_" + s])
        return _make(dims, _numbers(c["zipf_" + s], float), c["nnz_" + s], c["values"], c["idx_bytes"], seed, k,
                     [shared.get(m, 16 * k + m) for m in range(len(dims))])
    X = one("x", 1, {})
    Y = one("y", 2, {b: 16 + a for a, b in zip(_numbers(c["cx"]), _numbers(c["cy"]))}) if c["dims_y"] else X
    # W's first mode is contracted with the last mode of X x Y, which is Y's last
    return X, Y, one("w", 3, {0: 32 + len(Y.dims) - 1}) if c["kind"] == "chain" else None


@functools.lru_cache(maxsize=32)
def _shapes(shape_seed, instances, ir_cap):
    """The instances of a batch or of a server's requests: order 3-4, dims
    log-uniform in [100, 20000], nnz log-uniform in [1e3, 2e6] cut so that the
    self-contraction has about ir_cap products at most, 1-2 contracted modes,
    Zipf(1.1)."""
    r = np.random.RandomState(shape_seed)
    out = []
    for _ in range(instances):
        order = 3 + r.randint(2)
        dims = tuple(int(math.exp(r.uniform(math.log(100), math.log(20000)))) for _ in range(order))
        nnz = math.exp(r.uniform(math.log(1e3), math.log(2e6)))
        cm = tuple(sorted(int(m) for m in r.choice(order, 1 + r.randint(2), replace=False)))
        zipf = (1.1,) * order
        nnz = int(min(nnz, math.sqrt(ir_cap / _self_share(dims, zipf, cm)), math.prod(dims) // 8))
        out.append((dims, zipf, max(nnz, 200), cm))
    return tuple(out)


def _instances(c, seed):
    return [(_make(d, z, n, "uniform", 4, seed, k, [64 * k + m for m in range(len(d))]), cm)
            for k, (d, z, n, cm) in enumerate(_shapes(c["shape_seed"], c["instances"], c["ir_cap"]))]


# ---- the framework's calls ---------------------------------------------------------

class _Device:
    """Device memory of a result as torch sees it; holds the result."""

    def __init__(self, owner, ptr, n, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": kind, "data": (ptr, False), "version": 2}


def _view(owner, ptr, n, kind):
    if not n:
        return torch.empty(0, dtype={"<i4": torch.int32, "<i8": torch.int64, "<f4": torch.float32}[kind], device="cuda")
    return torch.as_tensor(_Device(owner, ptr, n, kind), device="cuda")


def _entries(r):
    """(row, col, val) of a result: views of its device memory."""
    parts = [(_view(r, a, n, "<i4"), _view(r, b, n, "<i8"), _view(r, v, n, "<f4")) for n, a, b, v in r.chunks()]
    if len(parts) == 1:
        return list(parts[0])
    if not parts:
        return [_view(r, 0, 0, k) for k in ("<i4", "<i8", "<f4")]
    return [torch.cat([p[j] for p in parts]) for j in range(3)]


def _whole(r):
    return _entries(r) + [_view(r, r.info.row_key, int(r.info.nrows), "<i8")]


def prepare(case, seed):
    c = dict(case)
    k = c["kind"]
    if k == "batch":
        items = [(t, t, list(cm), list(cm)) for t, cm in _instances(c, seed)]
        b = sptc.Batch(items, on_device=True)
        results = [b.result(i) for i in range(len(items))]
        return {"kind": k, "batch": b, "results": results, "keep": items, "views": [_entries(r) for r in results]}
    if k == "serve":
        s = sptc.Server(budget_bytes=24 * GIB, workers=2)
        return {"kind": k, "server": s, "requests": [(s.add_tensor(t, on_device=True), list(cm)) for t, cm in _instances(c, seed)]}
    X, Y, W = _operands(c, seed)
    s = {"kind": k, "X": X, "Y": Y, "W": W, "cx": list(_numbers(c["cx"])), "cy": list(_numbers(c["cy"])), "acc": c["acc"],
         "budget": c.get("budget_gib", 0) * GIB}
    if k == "host":
        def to_host(t):
            return COOTensor(t.dims, [i.cpu().numpy().astype(np.uint64 if c["idx_bytes"] == 8 else np.uint32) for i in t.idx], t.val.cpu().numpy())
        s["X"] = to_host(X)
        s["Y"] = s["X"] if Y is X else to_host(Y)
    if k == "plan":
        s["plan"] = sptc.Plan(X, Y, s["cx"], s["cy"], on_device=True)
    return s


def run(state):
    s = state
    k = s["kind"]
    if k == "batch":
        s["batch"].run(use_graph=True)
        s["batch"].sync()
        return s["views"]
    if k == "serve":
        srv = s["server"]
        ids = [srv.submit(t, t, cm, cm) for t, cm in s["requests"]]
        return [_entries(srv.wait(i)[0]) for i in ids]
    if k == "host":
        idx, val = sptc.SpTC(s["X"], s["Y"], s["cx"], s["cy"]).decode()
        return idx + [val]
    if k == "plan":
        r = s["plan"].execute()
        idx = [torch.empty(r.nnz, dtype=torch.int32, device="cuda") for _ in range(r.info.out_order)]
        val = torch.empty(r.nnz, dtype=torch.float32, device="cuda")
        r.decode_device([i.data_ptr() for i in idx], val.data_ptr())
        return idx + [val]
    if k == "count":
        r = sptc.SpTC(s["X"], s["Y"], s["cx"], s["cy"], count_only=True, mem_budget_bytes=s["budget"], on_device=True)
        return {"nnz": r.nnz, "ir_nnz": r.ir_nnz, "value_sum": float(r.info.value_sum)}
    r = sptc.SpTC(s["X"], s["Y"], s["cx"], s["cy"], dense_accumulator=s["acc"], on_device=True)
    if k == "chain":
        # the intermediate's modes: X's free modes, then Y's; its last is contracted with W's first
        z = sptc.SpTC(r, s["W"], [r.info.out_order - 1], [0], on_device=True)
        return _whole(r) + _whole(z)
    return _whole(r)


# ---- the same in 64 bits, by torch alone ------------------------------------------

def _bits(d):
    return max(0, (int(d) - 1).bit_length())


def _pack(t, modes, widths=None):
    key = torch.zeros(t.idx[0].numel(), dtype=torch.int64, device="cuda")
    for j, m in enumerate(modes):
        key = (key << (widths[j] if widths else _bits(t.dims[m]))) | t.idx[m].long()
    return key


def _pieces(X, Y, cx, cy, most=120_000_000):
    """The contraction's outputs in (row, column) order, row range by row
    range: first row_key, then (row, col, value in 64 bits, products) tuples."""
    w = [max(_bits(X.dims[a]), _bits(Y.dims[b])) for a, b in zip(cx, cy)]
    xf, yf = (_pack(t, [m for m in range(t.order) if m not in c]) for t, c in ((X, cx), (Y, cy)))
    xc, yc = _pack(X, cx, w), _pack(Y, cy, w)
    rows, xrow = torch.unique(xf, return_inverse=True)
    yield rows
    cols, ycol = torch.unique(yf, return_inverse=True)
    yc, o = torch.sort(yc)
    ycol, yval = ycol[o], Y.val.double()[o]
    xrow, o = torch.sort(xrow, stable=True)
    xc, xval = xc[o], X.val.double()[o]
    lo = torch.searchsorted(yc, xc)
    cnt = torch.searchsorted(yc, xc, right=True) - lo
    del yc, xc, o
    pre = torch.cumsum(cnt, 0)
    first = torch.searchsorted(xrow, torch.arange(rows.numel() + 1, device="cuda"))  # first nonzero of each row
    before = torch.cat([pre.new_zeros(1), pre])[first].cpu().numpy()  # products before each row
    first = first.cpu().numpy()
    a = 0
    while a < rows.numel():
        b = max(a + 1, int(np.searchsorted(before, before[a] + most, side="right")) - 1)
        i0, i1, n = int(first[a]), int(first[b]), int(before[b] - before[a])
        a = b
        if not n:
            continue
        c = cnt[i0:i1]
        x = torch.repeat_interleave(torch.arange(i0, i1, device="cuda"), c, output_size=n)
        y = torch.arange(n, device="cuda") - (pre[i0:i1] - c)[x - i0] + int(pre[i0 - 1] if i0 else 0) + lo[x]
        key = xrow[x] * cols.numel() + ycol[y]
        val = xval[x] * yval[y]
        del x, y
        key, o = torch.sort(key)
        val = val[o]
        del o
        key, inv = torch.unique_consecutive(key, return_inverse=True)
        out = torch.zeros(key.numel(), dtype=torch.float64, device="cuda").index_add_(0, inv, val)
        del inv, val
        yield (key // cols.numel()).int(), cols[key % cols.numel()], out, n


def _contract64(X, Y, cx, cy):
    """[row, col, value in 64 bits, row_key]."""
    it = _pieces(X, Y, cx, cy)
    rows = next(it)
    got = [p[:3] for p in it]
    if not got:
        e = torch.empty(0, device="cuda")
        return [e.int(), e.long(), e.double(), rows]
    return [torch.cat([p[j] for p in got]) for j in range(3)] + [rows]


def _unpack(key, t, modes):
    out, s = {}, 0
    for m in reversed(modes):
        out[m] = ((key >> s) & ((1 << _bits(t.dims[m])) - 1)).int()
        s += _bits(t.dims[m])
    return [out[m] for m in modes]


def _decoded(z, X, Y, cx, cy):
    fx, fy = ([m for m in range(t.order) if m not in c] for t, c in ((X, cx), (Y, cy)))
    return _unpack(z[3][z[0].long()], X, fx) + _unpack(z[1], Y, fy), tuple(X.dims[m] for m in fx) + tuple(Y.dims[m] for m in fy)


def exact(case, seed):
    c = dict(case)
    k = c["kind"]
    if k in ("batch", "serve"):
        return [_contract64(t, t, cm, cm)[:3] for t, cm in _instances(c, seed)]
    X, Y, W = _operands(c, seed)
    cx, cy = _numbers(c["cx"]), _numbers(c["cy"])
    if k == "count":
        it = _pieces(X, Y, cx, cy)
        next(it)
        nnz, ir, total = 0, 0, 0.0
        for row, _, val, n in it:
            nnz, ir, total = nnz + row.numel(), ir + n, total + float(val.sum())
        return {"nnz": nnz, "ir_nnz": ir, "value_sum": total}
    z = _contract64(X, Y, cx, cy)
    if k in ("host", "plan"):
        return _decoded(z, X, Y, cx, cy)[0] + [z[2]]
    if k == "chain":
        idx, dims = _decoded(z, X, Y, cx, cy)
        return z + _contract64(Tensor(dims, idx, z[2]), W, (len(dims) - 1,), (0,))
    return z


# ---- the bytes and operations a pass cannot do without ------------------------------

def _one(X, Y, cx, cy):
    """(operand bytes, outputs, products) of one contraction."""
    def size(t):
        return t.idx[0].numel() * (sum(i.element_size() for i in t.idx) + t.val.element_size())
    it = _pieces(X, Y, cx, cy)
    rows = next(it).numel()
    out = ir = 0
    for row, _, _, n in it:
        out, ir = out + row.numel(), ir + n
    return size(X) + (0 if Y is X else size(Y)), out, ir, rows


@functools.lru_cache(maxsize=64)
def _work(items):
    """Counted on the case's tensors: each operand read once, each output
    (row 4, column 8, value 4 bytes; row keys 8) written once; a multiply and an
    add for each product."""
    c = dict(items)
    k = c["kind"]
    if k in ("batch", "serve"):
        n = [_one(t, t, cm, cm) for t, cm in _instances(c, 5)]
        return sum(i + 16 * o for i, o, _, _ in n), 2 * sum(p for _, _, p, _ in n)
    X, Y, W = _operands(c, 5)
    cx, cy = _numbers(c["cx"]), _numbers(c["cy"])
    i, o, p, rows = _one(X, Y, cx, cy)
    if k == "count":
        return i + 24, 2 * p
    if k in ("host", "plan"):
        return i + 4 * o * (X.order + Y.order - 2 * len(cx) + 1), 2 * p
    if k == "chain":
        z = _contract64(X, Y, cx, cy)
        idx, dims = _decoded(z, X, Y, cx, cy)
        i2, o2, p2, r2 = _one(Tensor(dims, idx, z[2]), W, (len(dims) - 1,), (0,))
        return i + 16 * o + 8 * rows + i2 + 16 * o2 + 8 * r2, 2 * (p + p2)
    return i + 16 * o + 8 * rows, 2 * p


def work(case):
    b, f = _work(tuple(sorted((k, v) for k, v in case.items() if k != "name")))
    return {"bytes": b, "flops": f}
