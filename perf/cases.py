"""The work that array programs have this framework do, case by case, through its public entry points: the skeletons
of the C ABI on arrays in device memory (`acchip.Skeleton`), and a whole program of the array language from host arrays
to a host array (`accelerate_hip.run1`).

    listed()           the cases: the smallest calls, ordinary ones and large ones, odd sizes among them
    draw(rng)          another case of the same ranges
    prepare(case, s)   inputs made from the seed `s`, result arrays, and the compiled instances, which a program keeps
    run(state)         one pass, as a program makes it; returns the results
    work(case)         the bytes and operations that a pass cannot do without
    tolerance(case)    how far another correct implementation of the same precision may be off

Fragments are written as the array language's code generator writes them: a linear read of an array that is wanted once
is `acc_stream(array, ix)`, extents are the kernel's own names for them.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "accelerate-cuda_amd"))

import acchip as A  # noqa: E402

SIZE = {"Word8": 1, "Int32": 4, "Int64": 8, "float": 4, "double": 8}
TORCH = {"Word8": torch.uint8, "Int32": torch.int32, "Int64": torch.int64, "float": torch.float32, "double": torch.float64}
NUMPY = {"Word8": np.uint8, "Int32": np.int32, "Int64": np.int64, "float": np.float32, "double": np.float64}


def listed():
    return [
        # The smallest call: y <- a x + y over a vector that a program touches between two larger steps.  What counts
        # is what a call costs, not what it computes.
        {"name": "saxpy_1000", "path": "zipwith", "type": "float", "n": 1000},
        # A matrix turned before a step that wants it by columns; neither side is a multiple of a tile.
        {"name": "transpose_5003x3001", "path": "transpose", "type": "float", "h": 5003, "w": 3001},
        # fold (+) 0 (zipWith (*) xs ys): the dot product of the benchmark, 2^24 elements.
        {"name": "dot_16m", "path": "dot", "type": "float", "n": 1 << 24},
        # Column means and norms of a table of samples: a fold down the columns of a row-major matrix.
        {"name": "columns_20000x1000", "path": "fold2d", "type": "float", "h": 20000, "w": 1000, "along": "columns"},
        # scanl (+) 0 over 2^26 Int32: the prefix sum of the benchmark, the largest scan in use here.
        {"name": "scanl_64m", "path": "scan", "type": "Int32", "kind": "scanl", "n": 1 << 26},
        # A cumulative sum in double precision of an ordinary size that is no multiple of anything.
        {"name": "scanl1_3m_double", "path": "scan", "type": "double", "kind": "scanl1", "n": 3000001},
        # permute (+): 2^26 keys counted into 65 536 bins, Zipf(1.1), as in the benchmark: word counts, degrees.
        {"name": "histogram_64m_65536", "path": "histogram", "n": 1 << 26, "bins": 65536, "keys": "zipf"},
        # Stream compaction, the `filter` of the array language: scanl' over the flags gives every element that stays
        # its place, a permute stores it there.
        {"name": "filter_16m", "path": "filter", "n": 1 << 24, "kept": 0.5},
        # A sparse matrix times a vector: foldSeg (+) 0 over a gather, 2^20 rows of Poisson(32) entries.
        {"name": "smvm_1m", "path": "smvm", "type": "float", "rows": 1 << 20, "mean": 32, "lengths": "poisson"},
        # Ten passes of a 3 x 3 Gaussian over an image of 8192 x 8192, clamped at the edges.
        {"name": "gaussian_8192_x10", "path": "stencil2d", "type": "float", "h": 8192, "w": 8192, "points": 9, "boundary": "clamp", "iterations": 10},
        # One explicit step of the heat equation on a volume whose rows are no multiple of a strip.
        {"name": "heat3d_300", "path": "stencil3d", "type": "float", "d": 300, "h": 300, "w": 300, "points": 7, "boundary": "clamp"},
        # A program of the array language on host arrays, as `run1` serves it call after call: both operands to the
        # device, one fused kernel, the result back.
        {"name": "run1_cumulative_1m", "path": "run1", "n": 1 << 20},
    ]


def _size(rng, low, high):
    """a size between `low` and `high`, even over the logarithm: mostly odd ones, sometimes a power of two"""
    n = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if rng.random() < 0.25:
        n = 1 << max(0, n.bit_length() - 1)
    return max(low, min(high, n))


def draw(rng):
    path = rng.choice(["zipwith", "transpose", "dot", "fold2d", "scan", "scan", "histogram", "filter", "smvm", "stencil2d", "stencil3d", "run1"])
    if path == "zipwith":
        return {"path": path, "type": rng.choice(["float", "float", "double", "Int32", "Word8"]), "n": _size(rng, 1000, 1 << 26)}
    if path == "transpose":
        h = _size(rng, 64, 8192)
        return {"path": path, "type": rng.choice(["float", "float", "double"]), "h": h, "w": _size(rng, 64, 8192)}
    if path == "dot":
        return {"path": path, "type": rng.choice(["float", "float", "double", "Int32"]), "n": _size(rng, 1000, 1 << 26)}
    if path == "fold2d":
        h = _size(rng, 64, 1 << 18)
        w = _size(rng, 16, max(16, min(1 << 14, (1 << 25) // h)))
        return {"path": path, "type": rng.choice(["float", "float", "double", "Int32"]), "h": h, "w": w, "along": rng.choice(["rows", "columns"])}
    if path == "scan":
        return {"path": path, "type": rng.choice(["Int32", "float", "double", "Int64"]),
                "kind": rng.choice(["scanl", "scanl1", "scanl'", "scanr", "scanr1", "scanr'"]), "n": _size(rng, 1000, 1 << 26)}
    if path == "histogram":
        bins = _size(rng, 16, 1 << 18)
        return {"path": path, "n": _size(rng, 1000, 1 << 26 if bins <= 65536 else 1 << 24), "bins": bins, "keys": rng.choice(["uniform", "zipf"])}
    if path == "filter":
        return {"path": path, "n": _size(rng, 1000, 1 << 26), "kept": round(rng.uniform(0.05, 0.95), 2)}
    if path == "smvm":
        mean = _size(rng, 4, 128)
        return {"path": path, "type": rng.choice(["float", "float", "double"]), "rows": _size(rng, 1000, (1 << 25) // mean), "mean": mean,
                "lengths": rng.choice(["poisson", "skewed"])}
    boundary = rng.choice(["clamp", "mirror", "wrap", "constant"])
    if path == "stencil2d":
        iterations = rng.choice([1, 1, 2, 5, 10])
        h = _size(rng, 64, 8192)
        return {"path": path, "type": rng.choice(["float", "float", "double"]), "h": h, "w": _size(rng, 64, 8192), "points": rng.choice([5, 9]),
                "boundary": boundary, "iterations": iterations if h <= 4096 else min(iterations, 5)}
    if path == "stencil3d":
        return {"path": path, "type": rng.choice(["float", "float", "double"]), "d": _size(rng, 16, 400), "h": _size(rng, 16, 400), "w": _size(rng, 32, 400),
                "points": rng.choice([7, 27]), "boundary": boundary}
    return {"path": path, "n": _size(rng, 1000, 1 << 22)}


# ------------------------------------------------------------------------------ what a program keeps

_kept = {}


def _context():
    """the program's context and its stream"""
    if "context" not in _kept:
        cx = A.Context(0)
        _kept["context"] = (cx, cx.stream())
    return _kept["context"]


def _skeleton(kind, elt, **description):
    """an instance, compiled once for the program"""
    key = (kind, elt, repr(sorted(description.items())))
    if key not in _kept:
        _kept[key] = _context()[0].skeleton(kind, elt, wait=True, **description)
    return _kept[key]


class _Array(A.DeviceArray):
    """device memory of a tensor as an array of the framework; the tensor stays with it"""

    def __init__(self, tensor, ctype):
        A.DeviceArray.__init__(self, _context()[0], tuple(tensor.shape), NUMPY[ctype], ptr=tensor.data_ptr(), owner=False)
        self.tensor = tensor


def _random(shape, ctype, gen, low=0.0, high=1.0):
    """uniform in [low, high), whole numbers of the whole types"""
    if ctype in ("float", "double"):
        return torch.empty(shape, dtype=TORCH[ctype], device="cuda").uniform_(low, high, generator=gen)
    return torch.randint(int(low), int(high), shape, dtype=TORCH[ctype], device="cuda", generator=gen)


def _input(shape, ctype, gen, low=0.0, high=1.0):
    return _Array(_random(shape, ctype, gen, low, high), ctype)


def _result(shape, ctype):
    return _Array(torch.empty(shape, dtype=TORCH[ctype], device="cuda"), ctype)


def _read(k):
    return "acc_stream(arrIn%d_0, ix)" % k


def _lit(v, ctype):
    return {"float": "%r" % float(v) + "f", "double": "%r" % float(v)}.get(ctype, "((%s)%d)" % (ctype, int(v)))


# ------------------------------------------------------------------------------ inputs

def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    state = dict(_PREPARE[case["path"]](case, gen, int(seed)), path=case["path"], stream=_context()[1])
    return state


def _prepare_zipwith(c, gen, seed):
    t, n = c["type"], c["n"]
    high = 100 if t in ("Word8", "Int32") else 1.0
    get = "(%s)(%s * %s + %s)" % (t, _lit(3, t), _read(0), _read(1))
    return {"sk": _skeleton(A.SKEL_MAP, t, env=[(1, t), (1, t)], out_rank=1, get=get),
            "x": _input((n,), t, gen, 0, high), "y": _input((n,), t, gen, 0, high), "out": _result((n,), t)}


def _prepare_transpose(c, gen, seed):
    t = c["type"]
    sk = _skeleton(A.SKEL_MAP, t, env=[(2, t)], out_rank=2, flags=A.FLAG_TILED, get="arrIn0_0[(ix % shOut_0) * shIn0_0 + (ix / shOut_0)]")
    return {"sk": sk, "x": _input((c["h"], c["w"]), t, gen), "out": _result((c["w"], c["h"]), t)}


def _prepare_dot(c, gen, seed):
    t, n = c["type"], c["n"]
    low, high = (-4, 5) if t == "Int32" else (-1.0, 1.0)
    sk = _skeleton(A.SKEL_FOLD, t, env=[(1, t), (1, t)], out_rank=0, get="%s * %s" % (_read(0), _read(1)), combine="x + y", seed=_lit(0, t))
    x = _random((n,), t, gen, low, high)
    # (the two operands agree in part, so that the sum does not cancel: its relative error says something)
    y = x + _random((n,), t, gen, low, high)
    return {"sk": sk, "x": _Array(x, t), "y": _Array(y, t), "n": n, "out": _result((), t)}


def _prepare_fold2d(c, gen, seed):
    t, h, w = c["type"], c["h"], c["w"]
    x = _input((h, w), t, gen, 0, 16 if t == "Int32" else 1.0)
    if c["along"] == "rows":
        sk = _skeleton(A.SKEL_FOLD, t, env=[(2, t)], out_rank=1, get=_read(0), combine="x + y", seed=_lit(0, t))
        return {"sk": sk, "x": x, "shape": (h, w), "out": _result((h,), t)}
    # the fold of the transposed matrix: its rows lie across memory
    sk = _skeleton(A.SKEL_FOLD, t, env=[(2, t)], out_rank=1, flags=A.FLAG_TILED, get="arrIn0_0[acc_col * shIn0_0 + acc_row]", combine="x + y", seed=_lit(0, t))
    return {"sk": sk, "x": x, "shape": (w, h), "out": _result((w,), t)}


def _prepare_scan(c, gen, seed):
    t, n, kind = c["type"], c["n"], c["kind"]
    sk = _skeleton(A.SCAN_KINDS[kind], t, env=[(1, t)], get=_read(0), combine="x + y", seed=None if kind.endswith("1") else _lit(0, t))
    return {"sk": sk, "x": _input((n,), t, gen, 0, 16 if t in ("Int32", "Int64") else 1.0), "n": n,
            "out": _result((n + 1 if kind in ("scanl", "scanr") else n,), t), "total": _result((), t) if kind.endswith("'") else None}


def _keys(n, bins, kind, gen):
    """key values below `bins`: uniform, or bin k as often as 1 / (k + 1)^1.1"""
    if kind == "uniform":
        return torch.randint(0, bins, (n,), dtype=torch.int32, device="cuda", generator=gen)
    cdf = torch.arange(1, bins + 1, dtype=torch.float64, device="cuda").pow_(-1.1).cumsum(0)
    cdf /= cdf[-1].clone()
    u = torch.empty((n,), dtype=torch.float64, device="cuda").uniform_(0, 1, generator=gen)
    return torch.searchsorted(cdf, u).clamp_(max=bins - 1).to(torch.int32)


def _prepare_histogram(c, gen, seed):
    sk = _skeleton(A.SKEL_PERMUTE, "Int32", env=[(1, "Int32")], out_rank=1, get="1", combine="x + y", permutation=_read(0), combine_hint=A.COMBINE_ADD)
    return {"sk": sk, "x": _Array(_keys(c["n"], c["bins"], c["keys"], gen), "Int32"), "n": c["n"],
            "zeros": _Array(torch.zeros((c["bins"],), dtype=torch.int32, device="cuda"), "Int32"), "out": _result((c["bins"],), "Int32")}


def _prepare_filter(c, gen, seed):
    n = c["n"]
    flags = _skeleton(A.SKEL_SCANLP, "Int32", env=[(1, "float")], get="((%s > 0.0f) ? 1 : 0)" % _read(0), combine="x + y", seed="0")
    store = _skeleton(A.SKEL_PERMUTE, "float", env=[(1, "float"), (1, "Int32")], out_rank=1, get=_read(0), combine="x",
                      permutation="((%s > 0.0f) ? (Int64)%s : ACC_IGNORE)" % (_read(0), _read(1)))
    return {"flags": flags, "store": store, "n": n, "x": _input((n,), "float", gen, c["kept"] - 1.0, c["kept"]), "places": _result((n,), "Int32"),
            "count": _result((), "Int32"), "zeros": _Array(torch.zeros((n,), device="cuda"), "float"), "out": _result((n,), "float")}


def _lengths(c, gen):
    """entries per row: Poisson, or spread over two orders of magnitude round the same mean"""
    rows, mean = c["rows"], float(c["mean"])
    if c["lengths"] == "poisson":
        return torch.poisson(torch.full((rows,), mean, device="cuda"), generator=gen).to(torch.int64)
    z = torch.empty((rows,), device="cuda").normal_(0.0, 1.0, generator=gen)
    return (z.exp_() * (mean * math.exp(-0.5))).round_().clamp_(max=64 * mean).to(torch.int64)


def _prepare_smvm(c, gen, seed):
    t, rows = c["type"], c["rows"]
    offsets = torch.zeros((rows + 1,), dtype=torch.int64, device="cuda")
    torch.cumsum(_lengths(c, gen), 0, out=offsets[1:])
    entries = int(offsets[-1])
    sk = _skeleton(A.SKEL_FOLDSEG, t, env=[(1, t), (1, "Int32"), (1, t)], get="%s * arrIn2_0[%s]" % (_read(0), _read(1)), combine="x + y", seed=_lit(0, t))
    return {"sk": sk, "n": entries, "values": _input((entries,), t, gen, -1.0, 1.0), "columns": _input((entries,), "Int32", gen, 0, rows),
            "x": _input((rows,), t, gen, -1.0, 1.0), "offsets": _Array(offsets.to(torch.int32), "Int32"), "out": _result((rows,), t)}


def _prepare_stencil2d(c, gen, seed):
    t, shape = c["type"], (c["h"], c["w"])
    if c["points"] == 9:
        taps, weights, over = [(dy, dx) for dy in (-1, 0, 1) for dx in (-1, 0, 1)], [1, 2, 1, 2, 4, 2, 1, 2, 1], 16
    else:
        taps, weights, over = [(-1, 0), (0, -1), (0, 0), (0, 1), (1, 0)], [1, 1, 4, 1, 1], 8
    sk = _skeleton(A.SKEL_STENCIL, t, out_rank=2, taps=taps, boundary=c["boundary"], boundary_constant=_lit(0.5, t) if c["boundary"] == "constant" else None,
                   stencil_fn=A.linear_stencil_fn(weights, over, t))
    return {"sk": sk, "x": _input(shape, t, gen), "a": _result(shape, t), "b": _result(shape, t), "iterations": c["iterations"]}


def _prepare_stencil3d(c, gen, seed):
    t, shape = c["type"], (c["d"], c["h"], c["w"])
    if c["points"] == 7:
        taps = [(0, 0, 0), (-1, 0, 0), (1, 0, 0), (0, -1, 0), (0, 1, 0), (0, 0, -1), (0, 0, 1)]
        weights = [0.4] + [0.1] * 6
    else:
        taps = [(dz, dy, dx) for dz in (-1, 0, 1) for dy in (-1, 0, 1) for dx in (-1, 0, 1)]
        weights = [0.5 ** (3 + abs(dz) + abs(dy) + abs(dx)) for dz, dy, dx in taps]
    sk = _skeleton(A.SKEL_STENCIL, t, out_rank=3, taps=taps, boundary=c["boundary"], boundary_constant=_lit(0.5, t) if c["boundary"] == "constant" else None,
                   stencil_fn=A.linear_stencil_fn(weights, None, t))
    return {"sk": sk, "x": _input(shape, t, gen), "out": _result(shape, t)}


def _prepare_run1(c, gen, seed):
    import accelerate_hip as acc
    if "program" not in _kept:
        add, mul = (lambda a, b: a + b), (lambda a, b: a * b)
        _kept["program"] = acc.run1(lambda xs, ys: acc.scanl1(add, acc.zipWith(mul, xs, ys)))
    rng = np.random.default_rng(seed)
    return {"program": _kept["program"], "x": rng.random(c["n"], dtype=np.float32), "y": rng.random(c["n"], dtype=np.float32)}


_PREPARE = {"zipwith": _prepare_zipwith, "transpose": _prepare_transpose, "dot": _prepare_dot, "fold2d": _prepare_fold2d, "scan": _prepare_scan,
            "histogram": _prepare_histogram, "filter": _prepare_filter, "smvm": _prepare_smvm, "stencil2d": _prepare_stencil2d,
            "stencil3d": _prepare_stencil3d, "run1": _prepare_run1}


# ------------------------------------------------------------------------------ one pass

def run(s):
    path, stream = s["path"], s["stream"]
    if path == "zipwith":
        s["sk"].map([s["x"], s["y"]], s["out"], stream=stream)
    elif path == "transpose":
        s["sk"].map([s["x"]], s["out"], stream=stream)
    elif path == "dot":
        s["sk"].fold([s["x"], s["y"]], s["n"], s["out"], stream=stream)
    elif path == "fold2d":
        s["sk"].fold([s["x"]], s["shape"], s["out"], stream=stream)
    elif path == "scan":
        s["sk"].scan([s["x"]], s["n"], s["out"], total=s["total"], stream=stream)
        if s["total"] is not None:
            return {"out": s["out"].tensor, "total": s["total"].tensor}
    elif path == "histogram":
        s["sk"].permute([s["x"]], s["n"], s["zeros"], s["out"], stream=stream)
    elif path == "filter":
        s["flags"].scan([s["x"]], s["n"], s["places"], total=s["count"], stream=stream)
        s["store"].permute([s["x"], s["places"]], s["n"], s["zeros"], s["out"], stream=stream)
        return {"out": s["out"].tensor, "count": s["count"].tensor}
    elif path == "smvm":
        s["sk"].foldseg([s["values"], s["columns"], s["x"]], s["n"], s["offsets"], s["out"], stream=stream)
    elif path == "stencil2d":
        s["sk"].stencil(None, s["x"], s["a"], stream=stream)
        if s["iterations"] > 1:
            return s["sk"].stencil_iterate(None, s["a"], s["b"], s["iterations"] - 1, stream=stream).tensor
        return s["a"].tensor
    elif path == "stencil3d":
        s["sk"].stencil(None, s["x"], s["out"], stream=stream)
    else:
        return s["program"](s["x"], s["y"])
    return s["out"].tensor


# ------------------------------------------------------------------------------ what a pass cannot do without

def work(c):
    path, e = c["path"], SIZE.get(c.get("type"), 4)
    if path == "zipwith":
        return {"bytes": 3 * c["n"] * e, "flops": 2 * c["n"]}
    if path == "transpose":
        return {"bytes": 2 * c["h"] * c["w"] * e, "flops": 0}
    if path == "dot":
        return {"bytes": 2 * c["n"] * e + e, "flops": 2 * c["n"]}
    if path == "fold2d":
        return {"bytes": (c["h"] * c["w"] + (c["h"] if c["along"] == "rows" else c["w"])) * e, "flops": c["h"] * c["w"]}
    if path == "scan":
        return {"bytes": 2 * c["n"] * e + e, "flops": c["n"]}
    if path == "histogram":
        return {"bytes": 4 * (c["n"] + 2 * c["bins"]), "flops": c["n"]}
    if path == "filter":
        return {"bytes": 4 * (3 * c["n"] + 1), "flops": c["n"]}             # elements and defaults in, the result out
    if path == "smvm":
        entries = c["rows"] * c["mean"]
        return {"bytes": entries * (e + 4) + c["rows"] * (4 + 2 * e), "flops": 2 * entries}
    if path == "stencil2d":
        return {"bytes": 2 * c["h"] * c["w"] * e * c["iterations"], "flops": 2 * c["points"] * c["h"] * c["w"] * c["iterations"]}
    if path == "stencil3d":
        return {"bytes": 2 * c["d"] * c["h"] * c["w"] * e, "flops": 2 * c["points"] * c["d"] * c["h"] * c["w"]}
    return {"bytes": 12 * c["n"], "flops": 2 * c["n"]}


def tolerance(c):
    """Whole numbers and moved elements are exact.  Floating results: against the same sums in double precision the
    paths were off by 6e-8 at most, and by 2.3e-7 in a prefix sum of 2^26 Float32; Float64 ones, against sums in
    another order, by 8.4e-16.  About four times that."""
    t = c.get("type", "float")
    if c["path"] in ("transpose", "filter", "histogram") or t in ("Word8", "Int32", "Int64"):
        return "exact"
    return {"rel": 1e-6 if t == "float" else 4e-15}
