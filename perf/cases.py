"""The work this library is used for, as measurable cases.

Every case goes through the public Tensor methods on operands that are already on the GPU, as a training or
evaluation program drives them: activations and parameters are prepared once, the outputs are tensors the
program keeps, and one pass is the calls a program makes for them. Nothing in a pass waits for the GPU except
the calls that return a number.

A case is a dict; "path" says which program it is:

  softmax    class probabilities and predictions of a batch: max, csub, exp, sum, cdiv
  update     one momentum SGD step of a parameter block, in place: mul, cadd, cadd
  pointwise  one elementwise call on dense, windowed, transposed or broadcast operands of any type
  permuted   c = a + b where a is a 3-D tensor seen through permute(3, 2, 1)
  reduce     one reduction along a dim of an (outer, n, inner) tensor
  total      one reduction of a whole tensor to a number
  scan       cumsum along a dim of an (outer, n, inner) tensor
  image      a byte NHWC image batch converted into NCHW activations
"""
import math

import torch

import cutorch_amd as thc

TORCH = {"float": torch.float32, "half": torch.float16, "double": torch.float64, "byte": torch.uint8,
         "char": torch.int8, "short": torch.int16, "int": torch.int32, "long": torch.int64}
SIZE = {"float": 4, "half": 2, "double": 8, "byte": 1, "char": 1, "short": 2, "int": 4, "long": 8}
FLOATING = ("float", "half", "double")
BINARY = ("cadd", "axpy", "cmul", "cdiv", "cmax", "lt")
INTEGER_OPS = ("cadd", "cmul", "cmax", "lt")
ARITHMETIC = ("cadd", "axpy", "cmul", "cdiv", "cmax", "lt", "addcmul", "scale", "copy", "convert")


def listed():
    return [
        # a mini-batch's scores: five calls on a few hundred elements, all launch and call cost
        {"name": "softmax-64x10", "path": "softmax", "type": "float", "rows": 64, "cols": 10},
        # the weights and bias of a 1024-to-1000 layer as one block: the ordinary size of a parameter update
        {"name": "update-1m", "path": "update", "type": "float", "n": 1025000},
        # the plain stream: one flat add of 64 MiB operands
        {"name": "add-2p24", "path": "pointwise", "op": "cadd", "type": "float", "view": "dense", "rows": 4096, "cols": 4096},
        # a product with a transposed matrix accumulated onto a third one
        {"name": "addcmul-t-8192", "path": "pointwise", "op": "addcmul", "type": "float", "view": "transposed", "rows": 8192, "cols": 8192},
        # half activations through a transposed view of odd sizes: no row starts on a 16-byte boundary
        {"name": "exp-half-t-odd", "path": "pointwise", "op": "exp", "type": "half", "view": "transposed", "rows": 8191, "cols": 8193},
        # the largest: more than 2^31 elements, 64-bit offsets, all dims of one operand reversed
        {"name": "permuted-add-26gb", "path": "permuted", "type": "float", "x": 2048, "y": 2048, "z": 520},
        # predictions of a large evaluation batch: value and index of every row's maximum
        {"name": "max-rows-1024", "path": "reduce", "op": "max", "type": "float", "outer": 65536, "n": 1024, "inner": 1},
        # norms over the middle dim of half activations, accumulated in float
        {"name": "norm-middle-half", "path": "reduce", "op": "norm", "type": "half", "outer": 64, "n": 4096, "inner": 512},
        # batch statistics of a tall narrow matrix: one variance per column, rows of 40 bytes
        {"name": "var-tall-10", "path": "reduce", "op": "var", "type": "float", "outer": 1, "n": 6710886, "inner": 10},
        # the whole of 2^28 elements summed to a number the program waits for
        {"name": "sumall-2p28", "path": "total", "op": "sumall", "type": "float", "n": 1 << 28},
        # running totals of one long vector of weights, as sampling needs them
        {"name": "cumsum-2p26", "path": "scan", "type": "float", "outer": 1, "n": 1 << 26, "inner": 1},
        # a byte image batch on its way into a network
        {"name": "image-64x512", "path": "image", "type": "float", "images": 64, "height": 512, "width": 512, "channels": 3},
    ]


def _log(rng, low, high):
    """A whole number between low and high, even over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _odd_or_round(rng, n):
    """n itself two times in three, else the nearest multiple of 64 (or of 8 for small n)."""
    if rng.random() < 2 / 3:
        return n
    step = 64 if n >= 256 else 8
    return max(step, n // step * step)


def _reduced_shape(rng, most):
    """(outer, n, inner) of at most `most` elements: rows, a middle dim, or a tall matrix."""
    kind = rng.choice(("rows", "middle", "tall"))
    if kind == "rows":
        n = _odd_or_round(rng, _log(rng, 2, 65536))
        return _log(rng, 1, max(1, min(1 << 22, most // n))), n, 1
    if kind == "middle":
        n, inner = _odd_or_round(rng, _log(rng, 2, 8192)), _odd_or_round(rng, _log(rng, 2, 2048))
        return _log(rng, 1, max(1, min(4096, most // (n * inner)))), n, inner
    inner = _log(rng, 2, 1024)
    return 1, _log(rng, 1024, max(1024, most // inner)), inner


def draw(rng):
    path = rng.choice(("softmax", "update", "pointwise", "pointwise", "permuted", "reduce", "reduce", "total", "scan", "image"))
    if path == "softmax":
        cols = _log(rng, 2, 16384)
        return {"path": path, "type": rng.choice(("float", "float", "half")), "rows": _log(rng, 1, min(65536, (1 << 26) // cols)), "cols": cols}
    if path == "update":
        return {"path": path, "type": rng.choice(("float", "float", "half", "double")), "n": _log(rng, 64, 1 << 27)}
    if path == "pointwise":
        kind = rng.choice(("float", "float", "half", "half", "double", "byte", "char", "short", "int", "long"))
        ops = BINARY + ("addcmul", "scale", "copy", "convert", "exp", "tanh") if kind in FLOATING else INTEGER_OPS + ("scale", "copy", "convert")
        return {"path": path, "op": rng.choice(ops), "type": kind, "view": rng.choice(("dense", "window", "transposed", "transposed", "bias")),
                "rows": _odd_or_round(rng, _log(rng, 16, 8192)), "cols": _odd_or_round(rng, _log(rng, 16, 8192))}
    if path == "permuted":
        return {"path": path, "type": rng.choice(("float", "half")), "x": _odd_or_round(rng, _log(rng, 32, 1024)),
                "y": _odd_or_round(rng, _log(rng, 4, 1024)), "z": _odd_or_round(rng, _log(rng, 32, 512))}
    if path == "reduce":
        kind = rng.choice(("float", "float", "half", "double", "int", "byte"))
        ops = ("sum", "mean", "norm", "max", "min", "var", "std") if kind in FLOATING else ("sum", "max", "min")
        outer, n, inner = _reduced_shape(rng, 1 << 27)
        return {"path": path, "op": rng.choice(ops), "type": kind, "outer": outer, "n": n, "inner": inner}
    if path == "total":
        kind = rng.choice(("float", "float", "half", "double", "int"))
        ops = ("sumall", "meanall", "normall", "maxall", "varall") if kind in FLOATING else ("sumall", "maxall")
        return {"path": path, "op": rng.choice(ops), "type": kind, "n": _log(rng, 256, 1 << 27)}
    if path == "scan":
        outer, n, inner = _reduced_shape(rng, 1 << 26)
        return {"path": path, "type": rng.choice(("float", "float", "half", "double", "int")), "outer": outer, "n": n, "inner": inner}
    side = _log(rng, 28, 512)
    return {"path": path, "type": rng.choice(("float", "float", "half")), "images": _log(rng, 1, 128), "height": side,
            "width": side + rng.choice((0, 0, 1, 16)), "channels": rng.choice((1, 3, 3, 4))}


# ------------------------------------------------------------------------ operands --
class _Alias(object):
    """What torch needs to see an engine tensor's memory without a copy; keeps the tensor alive."""

    def __init__(self, t):
        item = SIZE[t.kind]
        self.tensor = t
        self.__cuda_array_interface__ = {
            "shape": t.shape, "strides": tuple(s * item for s in t.strides), "data": (t.data_ptr(), False), "version": 2,
            "typestr": {"float": "<f4", "half": "<f2", "double": "<f8", "byte": "|u1", "char": "|i1", "short": "<i2",
                        "int": "<i4", "long": "<i8"}[t.kind]}


def _torch(t):
    return torch.as_tensor(_Alias(t), device="cuda")


def _empty(kind, *shape):
    return thc.Tensor(kind).resize(shape)


class _Maker(object):
    """Operands from one seed: normal values for the floating types, small whole numbers for the others."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def fill(self, t, low=None, high=None):
        a = _torch(t)
        if t.kind in FLOATING and low is None:
            a.normal_(generator=self.g)
        elif t.kind in FLOATING:
            a.uniform_(low, high, generator=self.g)
        else:
            low, high = (0, 256) if t.kind == "byte" else (-100, 101)
            a.random_(low, high, generator=self.g)
        return t

    def new(self, kind, *shape):
        return self.fill(_empty(kind, *shape))

    def view(self, kind, view, rows, cols):
        """A (rows, cols) operand laid out as `view` says."""
        if view == "transposed":
            return self.new(kind, cols, rows).t()
        if view == "window":       # some columns of a wider matrix
            return self.new(kind, rows, cols + 7).narrow(1, 3, cols)
        if view == "bias":         # one row for all
            return self.new(kind, 1, cols).view_as_strided(0, (rows, cols), (0, 1))
        return self.new(kind, rows, cols)


def _convert_target(kind):
    return "half" if kind == "float" else "float"


def _out_kind(case):
    return "byte" if case["op"] == "lt" else _convert_target(case["type"]) if case["op"] == "convert" else case["type"]


def prepare(case, seed):
    make = _Maker(seed)
    path, kind = case["path"], case["type"]
    s = {"case": case}
    if path == "softmax":
        rows, cols = case["rows"], case["cols"]
        s["x"] = make.new(kind, rows, cols)
        s["p"] = _empty(kind, rows, cols)
        s["top"], s["total"], s["at"] = _empty(kind, rows, 1), _empty(kind, rows, 1), _empty("long", rows, 1)
        s["top_all"] = s["top"].view_as_strided(0, (rows, cols), (1, 0))
        s["total_all"] = s["total"].view_as_strided(0, (rows, cols), (1, 0))
        s["out"] = [_torch(s["p"]), _torch(s["at"])]
    elif path == "update":
        n = case["n"]
        s["w"], s["v"], s["g"] = make.new(kind, n), make.new(kind, n), make.new(kind, n)
        s["out"] = [_torch(s["w"]), _torch(s["v"])]
    elif path == "pointwise":
        rows, cols, op, view = case["rows"], case["cols"], case["op"], case["view"]
        s["a"] = make.view(kind, view, rows, cols)
        if op in BINARY or op == "addcmul":
            s["b"] = make.new(kind, rows, cols)
        if op == "addcmul":
            s["d"] = make.new(kind, rows, cols)
        s["c"] = _empty(_out_kind(case), rows, cols)
        s["out"] = [_torch(s["c"])]
    elif path == "permuted":
        x, y, z = case["x"], case["y"], case["z"]
        s["a"] = make.new(kind, z, y, x).view_as_strided(0, (x, y, z), (1, x, x * y))
        s["b"] = make.new(kind, x, y, z)
        s["c"] = _empty(kind, x, y, z)
        s["out"] = [_torch(s["c"])]
    elif path == "reduce":
        outer, n, inner = case["outer"], case["n"], case["inner"]
        s["x"] = make.new(kind, outer, n, inner)
        s["r"] = _empty(kind, outer, 1, inner)
        s["out"] = [_torch(s["r"])]
        if case["op"] in ("max", "min"):
            s["at"] = _empty("long", outer, 1, inner)
            s["out"].append(_torch(s["at"]))
    elif path == "total":
        s["x"] = _empty(kind, case["n"])
        make.fill(s["x"], 0.0, 1.0)
    elif path == "scan":
        shape = (case["outer"], case["n"], case["inner"])
        s["x"] = _empty(kind, *shape)
        # weights that add up to about one along the dim, as a sampler's are
        make.fill(s["x"], 0.0, 2.0 / case["n"])
        s["r"] = _empty(kind, *shape)
        s["out"] = [_torch(s["r"])]
    else:
        b, h, w, c = case["images"], case["height"], case["width"], case["channels"]
        s["x"] = make.new("byte", b, h, w, c).view_as_strided(0, (b, c, h, w), (h * w * c, 1, w * c, c))
        s["r"] = _empty(kind, b, c, h, w)
        s["out"] = [_torch(s["r"])]
    return s


# ------------------------------------------------------------------------ one pass --
def _pointwise(s, op):
    a, c = s["a"], s["c"]
    if op == "cadd":
        c.cadd(a, 1, s["b"])
    elif op == "axpy":
        c.cadd(a, 0.25, s["b"])
    elif op == "cmul":
        c.cmul(a, s["b"])
    elif op == "cdiv":
        c.cdiv(a, s["b"])
    elif op == "cmax":
        c.binary("cmax", a, s["b"])
    elif op == "lt":
        c.compare_tensor("lt", a, s["b"])
    elif op == "addcmul":
        c.addcmul(s["d"], 1, a, s["b"])
    elif op == "scale":
        c.mul(a, 3)
    elif op == "copy":
        c.copy(a)
    elif op == "convert":
        c.copy_from(a)
    else:
        c.unary(op, a)


def run(s):
    case = s["case"]
    path = case["path"]
    if path == "softmax":
        p = s["p"]
        s["top"].max(s["at"], s["x"], 1)
        p.csub(s["x"], 1, s["top_all"])
        p.unary("exp", p)
        s["total"].sum(p, 1)
        p.cdiv(p, s["total_all"])
    elif path == "update":
        s["v"].mul(s["v"], 0.5)
        s["v"].cadd(s["v"], 1, s["g"])
        s["w"].cadd(s["w"], -0.0078125, s["v"])
    elif path == "pointwise":
        _pointwise(s, case["op"])
    elif path == "permuted":
        s["c"].cadd(s["a"], 1, s["b"])
    elif path == "reduce":
        op, x, r = case["op"], s["x"], s["r"]
        if op in ("max", "min"):
            getattr(r, op)(s["at"], x, 1)
        elif op == "norm":
            r.norm(x, 2, 1)
        else:
            getattr(r, op)(x, 1)
    elif path == "total":
        x, op = s["x"], case["op"]
        return x.normall(2) if op == "normall" else getattr(x, op)()
    elif path == "scan":
        s["r"].cumsum(s["x"], 1)
    else:
        s["r"].copy_from(s["x"])
    return s["out"]


# ------------------------------------------------------------------------ measures --
def work(case):
    path, e = case["path"], SIZE[case["type"]]
    if path == "softmax":
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * e * n + 8 * case["rows"], "flops": 5 * n}
    if path == "update":
        return {"bytes": 5 * e * case["n"], "flops": 4 * case["n"]}
    if path == "pointwise":
        n, op = case["rows"] * case["cols"], case["op"]
        first = case["cols"] if case["view"] == "bias" else n
        others = n * (2 if op == "addcmul" else 1 if op in BINARY else 0)
        return {"bytes": e * (first + others) + SIZE[_out_kind(case)] * n, "flops": n * (2 if op in ("addcmul", "axpy") else 1)}
    if path == "permuted":
        n = case["x"] * case["y"] * case["z"]
        return {"bytes": 3 * e * n, "flops": n}
    if path == "reduce":
        rest = case["outer"] * case["inner"]
        n = rest * case["n"]
        return {"bytes": e * (n + rest) + (8 * rest if case["op"] in ("max", "min") else 0), "flops": n * (2 if case["op"] in ("norm", "var", "std") else 1)}
    if path == "total":
        return {"bytes": e * case["n"] + e, "flops": case["n"]}
    if path == "scan":
        n = case["outer"] * case["n"] * case["inner"]
        return {"bytes": 2 * e * n, "flops": n}
    n = case["images"] * case["height"] * case["width"] * case["channels"]
    return {"bytes": (1 + e) * n, "flops": n}


def tolerance(case):
    """Bit for bit where every result is one rounding of exact arithmetic or a choice among the inputs; elsewhere about
    four times what the path differs from float64 arithmetic on the same inputs."""
    path, kind = case["path"], case["type"]
    op = case.get("op")
    if path in ("permuted", "update", "image") or op in ARITHMETIC or op in ("max", "min", "maxall") or kind not in FLOATING:
        return "exact"
    if path == "pointwise":        # exp, tanh
        return {"rel": {"half": 8e-4, "float": 1e-7, "double": 1e-15}[kind]}
    if path == "softmax":
        return {"rel": {"half": 2e-3, "float": 6e-7, "double": 1e-14}[kind]}
    if path == "scan":
        return {"rel": {"half": 8e-4, "float": 8e-7, "double": 1e-13}[kind]}
    if path == "total":            # the number comes back in float, also for half
        return {"rel": {"half": 4e-7, "float": 4e-7, "double": 1e-13}[kind]}
    # sums, norms and moments along a dim: the sums are in float, a half result is rounded once
    return {"rel": {"half": 1.4e-3, "float": 1e-6, "double": 1e-13}[kind]}
