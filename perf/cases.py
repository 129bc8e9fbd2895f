"""Performance cases of the scan / mapreduce path: what a user's program has it do.

Five families, each through the Python entry points (which call the C ABI):

  scan    scan_(op, dst, src): prefix sums, running maxima, the affine
          recurrence x_t = a_t x_{t-1} + b_t and quaternion products, over
          whole vectors, views that start off the 16-byte grid, and one
          channel of interleaved records (a strided view).
  reduce  mapreduce(f, op, x): sums, sums of squares and maxima of a vector,
          as a host scalar (a residual, a norm) or into a device element.
  multi   mapreduce1d(f, op, (x, y)): dot products and squared distances of
          two vectors or two views of one series.
  dims    mapreduce(f, op, A, dims=..., g=...): sums, sums of squares, norms
          and maxima along dims of 2- to 4-dimensional column-major arrays
          and of every second column of a matrix.
  mv      matvec(A, x) / vecmat(x, A) over column-major matrices of any
          aspect, the shapes of the library's matvec / vecmat sweep.

Sizes run from a few thousand elements (one launch, latency only) to the
2^28 and 2^30 elements of the headline benchmark. `draw` spreads sizes over
that range by their logarithm, odd ones included.
"""
import math

import torch

import __graft_entry__

kf = __graft_entry__.load_package()

DTYPES = {"f32": torch.float32, "f64": torch.float64, "i32": torch.int32, "u8": torch.uint8,
          "affine": torch.float32, "quat": torch.float32}
SIZE = {"f32": 4, "f64": 8, "i32": 4, "u8": 1, "affine": 8, "quat": 16}
LANES = {"affine": 2, "quat": 4}  # float32 values per element


def listed():
    return [
        # a short prefix sum, as in stream compaction or a histogram's offsets: latency only
        {"name": "scan f32 1e4", "kind": "scan", "dtype": "f32", "op": "+", "exclusive": False, "n": 10_007,
         "off": 0, "stride": 1},
        # a linear recurrence (IIR filter, discounted return) over an ordinary series
        {"name": "scan affine 4e6", "kind": "scan", "dtype": "affine", "op": "affine", "exclusive": False,
         "n": 4_000_037, "off": 0, "stride": 1},
        # offsets from one channel of interleaved three-value records
        {"name": "scan i32 channel 8e6", "kind": "scan", "dtype": "i32", "op": "+", "exclusive": True,
         "n": 8_000_009, "off": 0, "stride": 3},
        # the headline scan
        {"name": "scan f32 2^28", "kind": "scan", "dtype": "f32", "op": "+", "exclusive": False, "n": 1 << 28,
         "off": 0, "stride": 1},
        # a small sum a program branches on: the result comes back to the host
        {"name": "sum f64 4e3 to host", "kind": "reduce", "dtype": "f64", "f": "identity", "op": "+", "n": 4_099,
         "off": 0, "stride": 1, "host": True},
        # the headline reduction: a sum of squares over 2^30 elements
        {"name": "sumsq f32 2^30", "kind": "reduce", "dtype": "f32", "f": "abs2", "op": "+", "n": 1 << 30,
         "off": 0, "stride": 1, "host": False},
        # lag-1 product sum of one series: two views of it, one element apart
        {"name": "lag dot f32 3e7", "kind": "multi", "dtype": "f32", "f": "mul", "n": 30_000_001, "lag": 1},
        # column norms of a matrix whose columns are no multiple of 16 bytes
        {"name": "column norms f32", "kind": "dims", "dtype": "f32", "f": "abs2", "op": "+", "g": "sqrt",
         "shape": "5003x20011", "dims": "1", "every": 1},
        # row sums of every second column of a matrix
        {"name": "row sums f32 view", "kind": "dims", "dtype": "f32", "f": "identity", "op": "+", "g": "identity",
         "shape": "65536x2049", "dims": "2", "every": 2},
        # per-channel statistics of a (W, H, C, N) batch
        {"name": "channel sumsq f32", "kind": "dims", "dtype": "f32", "f": "abs2", "op": "+", "g": "identity",
         "shape": "57x61x64x100", "dims": "1,2,4", "every": 1},
        # a dense matrix-vector product with an odd row count
        {"name": "matvec f64", "kind": "mv", "dtype": "f64", "which": "matvec", "rows": 10_007, "cols": 3_001},
        # a vector-matrix product over bytes, mid-sized
        {"name": "vecmat u8", "kind": "mv", "dtype": "u8", "which": "vecmat", "rows": 1_000, "cols": 100_003},
    ]


def _log_int(rng, lo, hi):
    """An integer spread over [lo, hi] by its logarithm, odd more often than not."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        v |= 1
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choice(["scan", "scan", "reduce", "multi", "dims", "dims", "mv"])
    if kind == "scan":
        dtype = rng.choice(["f32", "f32", "f64", "i32", "u8", "affine", "quat"])
        top = (1 << 30) // SIZE[dtype]
        op = {"affine": "affine", "quat": "*", "u8": "+"}.get(dtype) or rng.choice(["+", "+", "max"])
        stride = rng.choice([1, 1, 1, 2, 3, 4])
        return {"kind": kind, "dtype": dtype, "op": op, "exclusive": rng.random() < 0.3,
                "n": _log_int(rng, 4_000, top // stride), "off": rng.choice([0, 0, 1]), "stride": stride}
    if kind == "reduce":
        dtype = rng.choice(["f32", "f32", "f64", "i32", "u8"])
        stride = rng.choice([1, 1, 1, 2, 3, 10])
        op = "+" if dtype == "u8" else rng.choice(["+", "+", "max"])
        return {"kind": kind, "dtype": dtype, "f": rng.choice(["identity", "abs2"]), "op": op,
                "n": _log_int(rng, 2_000, (1 << 31) // SIZE[dtype] // stride), "off": rng.choice([0, 0, 1]),
                "stride": stride, "host": rng.random() < 0.5}
    if kind == "multi":
        dtype = rng.choice(["f32", "f32", "f64"])
        return {"kind": kind, "dtype": dtype, "f": rng.choice(["mul", "mul", "sqdiff"]),
                "n": _log_int(rng, 2_000, (1 << 30) // SIZE[dtype]), "lag": rng.choice([0, 1, 1, 2, 3, 7])}
    if kind == "dims":
        dtype = rng.choice(["f32", "f32", "f64", "i32", "u8"])
        total = _log_int(rng, 10_000, (1 << 30) // SIZE[dtype])
        nd = rng.choice([2, 2, 3, 4])
        cut = sorted(rng.uniform(0.0, 1.0) for _ in range(nd - 1))
        parts = [b - a for a, b in zip([0.0] + cut, cut + [1.0])]
        shape = [max(2, int(round(total ** p))) for p in parts]
        dims = sorted(rng.sample(range(1, nd + 1), rng.randint(1, nd - 1)))
        op = "+" if dtype == "u8" else rng.choice(["+", "+", "max"])
        g = rng.choice(["identity", "identity", "sqrt"]) if dtype in ("f32", "f64") else "identity"
        return {"kind": kind, "dtype": dtype, "f": "abs2" if g == "sqrt" else rng.choice(["identity", "abs2"]), "op": op,
                "g": g, "shape": "x".join(map(str, shape)), "dims": ",".join(map(str, dims)),
                "every": rng.choice([1, 1, 2]) if nd == 2 else 1}
    dtype = rng.choice(["f32", "f64", "u8"])
    total = _log_int(rng, 10_000, (1 << 30) // SIZE[dtype])
    rows = max(2, int(round(total ** rng.uniform(0.1, 0.9))))
    return {"kind": kind, "dtype": dtype, "which": rng.choice(["matvec", "vecmat"]), "rows": rows,
            "cols": max(2, total // rows)}


# ---- inputs -----------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _values(case, n, gen):
    """n elements of the case's type: measurements or weights in [0, 1), signed values for sums of squares and
    distances, signed values in units of their own for maxima, small counts for the integer types (their sums
    wrap as the type does)."""
    dtype = case["dtype"]
    if case.get("op") == "max":
        if dtype == "i32":
            return torch.randint(-2 ** 30, 2 ** 30, (n,), generator=gen, device="cuda", dtype=torch.int32)
        unit = 0.5 + torch.rand((1,), generator=gen, device="cuda", dtype=DTYPES[dtype])
        return torch.randn((n,), generator=gen, device="cuda", dtype=DTYPES[dtype]).mul_(unit)
    if dtype == "i32":
        return torch.randint(0, 16, (n,), generator=gen, device="cuda", dtype=torch.int32)
    if dtype == "u8":
        return torch.randint(0, 256, (n,), generator=gen, device="cuda", dtype=torch.uint8)
    if dtype == "affine":
        p = torch.randn((n, 2), generator=gen, device="cuda")
        p[:, 0].uniform_(0.9, 1.0, generator=gen)
        return p
    if dtype == "quat":  # unit quaternions: rotations
        q = torch.randn((n, 4), generator=gen, device="cuda")
        return q.div_(q.norm(dim=1, keepdim=True))
    if case.get("f") in ("abs2", "sqdiff"):
        return torch.randn((n,), generator=gen, device="cuda", dtype=DTYPES[dtype])
    return torch.rand((n,), generator=gen, device="cuda", dtype=DTYPES[dtype])


def _shape(case):
    return tuple(int(v) for v in case["shape"].split("x"))


def _dims(case):
    return tuple(int(v) for v in case["dims"].split(","))


def _inputs(case, seed):
    """The operands alone, as tuples of tensors (views included)."""
    gen = _generator(seed)
    kind = case["kind"]
    if kind in ("scan", "reduce"):
        n, off, stride = case["n"], case["off"], case["stride"]
        return (_values(case, (n - 1) * stride + 1 + off, gen)[off::stride],)
    if kind == "multi":
        n, lag = case["n"], case["lag"]
        if lag:
            base = _values(case, n + lag, gen)
            return base[lag:], base[:n]
        return _values(case, n, gen), _values(case, n, gen)
    if kind == "dims":
        shape, every = list(_shape(case)), case["every"]
        shape[-1] = (shape[-1] - 1) * every + 1
        count = math.prod(shape)
        A = _values(case, count, gen).view(*reversed(shape)).permute(*reversed(range(len(shape))))
        return (A[..., ::every],)
    rows, cols = case["rows"], case["cols"]
    A = _values(case, rows * cols, gen).view(cols, rows).t()
    return A, _values(case, cols if case["which"] == "matvec" else rows, gen)


def prepare(case, seed):
    """The operands and, as a program that repeats the call keeps them, the destination (and a scan's scratch)."""
    ops = _inputs(case, seed)
    state = {"case": dict(case), "in": ops}
    kind = case["kind"]
    if kind == "scan":
        src = ops[0]
        state["dst"] = torch.empty(src.shape, dtype=src.dtype, device="cuda")
        state["tmp"] = kf.get_allocation(kf.Scan1D, kf.identity, case["op"], src)
    elif kind == "reduce" and not case["host"]:
        state["dst"] = torch.empty(1, dtype=ops[0].dtype, device="cuda")
    elif kind == "mv":
        A = ops[0]
        state["dst"] = torch.empty(A.shape[0] if case["which"] == "matvec" else A.shape[1], dtype=A.dtype, device="cuda")
    return state


_MAPS = {"identity": kf.identity, "abs2": kf.abs2}
_POST = {"identity": None, "sqrt": math.sqrt}


def run(state):
    case, ops = state["case"], state["in"]
    kind = case["kind"]
    if kind == "scan":
        return kf.scan_(case["op"], state["dst"], ops[0], exclusive=case["exclusive"], tmp=state["tmp"])
    if kind == "reduce":
        if case["host"]:
            return kf.mapreduce(_MAPS[case["f"]], case["op"], ops[0])
        return kf.mapreduce_(_MAPS[case["f"]], case["op"], state["dst"], ops[0])
    if kind == "multi":
        return kf.mapreduce1d(case["f"] if case["f"] == "mul" else kf.sqdiff, "+", ops, to_cpu=False)
    if kind == "dims":
        return kf.mapreduce(_MAPS[case["f"]], case["op"], ops[0], dims=_dims(case), g=_POST[case["g"]])
    if case["which"] == "matvec":
        return kf.matvec_(state["dst"], ops[0], ops[1])
    return kf.vecmat_(state["dst"], ops[1], ops[0])


# ---- what a pass cannot do without ------------------------------------------
def work(case):
    kind, es = case["kind"], SIZE[case["dtype"]]
    if kind == "scan":
        return {"bytes": 2 * case["n"] * es, "flops": case["n"] * {"affine": 3, "quat": 28}.get(case["dtype"], 1)}
    if kind == "reduce":
        return {"bytes": (case["n"] + 1) * es, "flops": case["n"] * (2 if case["f"] == "abs2" else 1)}
    if kind == "multi":  # two views of one series share its elements
        read = case["n"] + case["lag"] if case["lag"] else 2 * case["n"]
        return {"bytes": (read + 1) * es, "flops": 2 * case["n"]}
    if kind == "dims":
        shape, dims = _shape(case), _dims(case)
        count = math.prod(shape)
        out = math.prod(s for i, s in enumerate(shape) if i + 1 not in dims)
        return {"bytes": (count + out) * es, "flops": count * (2 if case["f"] == "abs2" else 1)}
    rows, cols = case["rows"], case["cols"]
    return {"bytes": (rows * cols + rows + cols) * es, "flops": 2 * rows * cols}


def tolerance(case):
    """Whole numbers and maxima are exact; sums and products carry the rounding of their order. Measured against
    64 bits: Float32 sums and scans at most 3.2e-7 off (2^28 elements), Float64 2e-16 to 2e-15. A product of n
    unit quaternions drifts by about 2e-8 sqrt(n) (1.7e-5 at 8*10^5)."""
    if case["dtype"] == "quat":
        return {"rel": max(2e-6, 8e-8 * math.sqrt(case["n"]))}
    if case["dtype"] in ("i32", "u8"):
        return "exact"
    if case.get("op") == "max" and case.get("g") != "sqrt":
        return "exact"
    return {"rel": 1e-14} if case["dtype"] == "f64" else {"rel": 2e-6}


# ---- the same in 64 bits ----------------------------------------------------
def _compose(case, p, q):
    """p then q, for rows of 64-bit affine pairs or quaternions (older on the left)."""
    if case["dtype"] == "affine":
        return torch.stack([q[:, 0] * p[:, 0], q[:, 0] * p[:, 1] + q[:, 1]], 1)
    a, b, c, d = p.unbind(1)
    e, f, g, h = q.unbind(1)
    return torch.stack([a * e - b * f - c * g - d * h, a * f + b * e + c * h - d * g,
                        a * g - b * h + c * e + d * f, a * h + b * g - c * f + d * e], 1)


def _exact_scan(case, x):
    if case["dtype"] in LANES:
        if case["n"] > 1 << 26:
            return None
        v, step = x.double(), 1
        while step < v.shape[0]:  # every row holds the composition of the last 2*step rows up to it
            v = torch.cat([v[:step], _compose(case, v[:-step], v[step:])])
            step *= 2
    elif case["op"] == "max":
        v = torch.cummax(x, 0).values.to(torch.float64 if x.dtype.is_floating_point else torch.int64)
    else:
        v = torch.cumsum(x, 0, dtype=torch.float64 if x.dtype.is_floating_point else torch.int64)
    if case["exclusive"]:
        first = torch.zeros_like(v[:1])
        if case["dtype"] in LANES:
            first[:, 0] = 1
        elif case["op"] == "max":
            first.fill_({"f32": -math.inf, "f64": -math.inf, "i32": -2 ** 31, "u8": 0}[case["dtype"]])
        v = torch.cat([first, v[:-1]])
    return v


def _wrap(x, dtype):
    """64-bit whole numbers as the type holds them."""
    return x.to(dtype) if dtype in (torch.uint8, torch.int32) else x


def exact(case, seed):
    ops = _inputs(case, seed)
    kind = case["kind"]
    floating = ops[0].dtype.is_floating_point
    if kind == "scan":
        v = _exact_scan(case, ops[0])
        return None if v is None else _wrap(v, ops[0].dtype)
    wide = torch.float64 if floating else torch.int64
    if kind in ("reduce", "dims"):
        x = ops[0]
        over = tuple(d - 1 for d in _dims(case)) if kind == "dims" else tuple(range(x.dim()))
        parts = []
        # the last dim in pieces, so that the wide copies stay small
        for piece in x.split(max(1, (1 << 26) * x.shape[-1] // max(1, x.numel())), dim=-1):
            w = piece.to(wide)
            w = _wrap(w * w, x.dtype).to(wide) if case["f"] == "abs2" else w
            parts.append(w.amax(over, keepdim=True) if case["op"] == "max" else w.sum(over, keepdim=True))
        v = torch.cat(parts, -1)
        if x.dim() - 1 in over:
            v = v.amax(-1, keepdim=True) if case["op"] == "max" else v.sum(-1, keepdim=True)
        v = _wrap(v, x.dtype)
        if kind == "reduce":
            v = v.reshape(1)
            return v.item() if case["host"] else v
        return torch.sqrt(v) if case["g"] == "sqrt" else v
    if kind == "multi":
        total = 0.0
        for x, y in zip(ops[0].split(1 << 26), ops[1].split(1 << 26)):
            x, y = x.double(), y.double()
            total = total + ((x * y) if case["f"] == "mul" else (x - y) ** 2).sum()
        return total.reshape(1)
    A, x = ops
    along = 1 if case["which"] == "matvec" else 0
    w = x.to(wide)
    out = None
    for lo in range(0, A.shape[1], max(1, (1 << 26) // A.shape[0])):
        hi = min(A.shape[1], lo + max(1, (1 << 26) // A.shape[0]))
        if along == 1:
            part = (A[:, lo:hi].to(wide) * w[lo:hi][None, :]).sum(1)
            out = part if out is None else out + part
        else:
            part = (A[:, lo:hi].to(wide) * w[:, None]).sum(0)
            out = part if out is None else torch.cat([out, part])
    return _wrap(out, A.dtype)
