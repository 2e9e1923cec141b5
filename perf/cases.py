"""Workloads that the performance of this backend is judged on.

Each case is one pass of work that a program using the backend has it do: the
statistics of a batch, the top-k or the draw of a decoding step, a softmax and
its gradient, a cross-entropy step, the layout change of an image batch.  Most
call the C entry points of include/tpr_rocm.h with descriptors, outputs and
workspaces made once, as a serving or training loop keeps them; the
cross-entropy step goes through the Python tensors.

`listed()` names the cases, `draw()` makes others of the same ranges,
`prepare()` makes a case's inputs on the GPU from a seed, `run()` is one pass,
and `work()`, `tolerance()` and `exact()` say what a pass has to move, how far
two correct passes may lie apart, and what plain torch gives in 64 bits.
"""
import ctypes
import math

import torch

import tensorplay_amd as tp
from tensorplay_amd import _capi as capi

DEV = "cuda:0"
DTYPES = {"float32": torch.float32, "float64": torch.float64, "int64": torch.int64, "int32": torch.int32,
          "int8": torch.int8, "uint8": torch.uint8}
# the largest pass any drawn case makes, in bytes of its inputs
MOST_BYTES = 1 << 28


def listed():
    return [
        # Metrics of one small batch (64 samples of 1000 scores): every launch is
        # far shorter than its own latency.
        {"name": "stats_small", "kind": "reduce", "shape": "64x1000", "dtype": "float32",
         "plan": "sum:1 mean:1 amax:1 argmax:1 var:1 std:1"},
        # The headline workload of bench.py: a 1 GiB tensor reduced six ways.
        {"name": "stats_flat", "kind": "reduce", "shape": "268435456", "dtype": "float32",
         "plan": "sum: mean: amax: argmax: var: std:"},
        # The strided reductions of bench.py (one per dim) at sizes that are no
        # multiple of anything: rows start at any 4-byte address.
        {"name": "stats_ragged", "kind": "reduce", "shape": "63x1021x1023", "dtype": "float32",
         "plan": "mean:1 amax:0 argmax:0 var:2 std:2"},
        # Batch statistics of an activation [N, C, H, W] over N, H, W, forward and backward.
        {"name": "channel_stats", "kind": "channels", "shape": "64x64x56x56"},
        # An image batch as it is loaded (uint8, channels last): to float32
        # channels first, per-image channel maxima, the sum of all pixels.
        {"name": "image_batch", "kind": "images", "shape": "64x224x224x3"},
        # Top-50 of a decoding step's logits, bench.py's shape.
        {"name": "topk_logits", "kind": "topk", "rows": 256, "cols": 151936, "k": 50, "dtype": "float32",
         "largest": True},
        # A large k over short rows (candidate pruning), bench.py's shape.
        {"name": "topk_large_k", "kind": "topk", "rows": 4096, "cols": 2048, "k": 1000, "dtype": "float32",
         "largest": True},
        # One decoding step of a small batch: top-50, then the top-p nucleus.
        {"name": "sample_decode", "kind": "sample", "rows": 8, "cols": 151936, "k": 50, "temperature": 0.8,
         "top_p": 0.9},
        # Nucleus sampling alone (top-p over the whole vocabulary).
        {"name": "sample_nucleus", "kind": "sample", "rows": 256, "cols": 151936, "k": 151936, "temperature": 0.8,
         "top_p": 0.9},
        # Softmax over an odd vocabulary and its gradient.
        {"name": "softmax_rows", "kind": "softmax", "shape": "2048x50261", "dim": 1, "log": False,
         "dtype": "float32"},
        # Softmax over a middle dim and its gradient, bench.py's shape.
        {"name": "softmax_dim1", "kind": "softmax", "shape": "64x1024x1024", "dim": 1, "log": False,
         "dtype": "float32"},
        # Cross entropy over an odd vocabulary: loss and the gradient of the logits.
        {"name": "cross_entropy", "kind": "cross_entropy", "rows": 2048, "cols": 50261},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _fit(shape, item):
    """`shape` with its largest extent cut so that the tensor is no larger than MOST_BYTES."""
    shape = list(shape)
    n = math.prod(shape)
    if n * item > MOST_BYTES:
        i = max(range(len(shape)), key=lambda j: shape[j])
        shape[i] = max(1, MOST_BYTES * shape[i] // (n * item))
    return shape


def _text(shape):
    return "x".join(str(s) for s in shape)


def draw(rng):
    kind = rng.choice(["reduce", "reduce", "reduce", "channels", "images", "topk", "topk", "sample", "sample",
                       "softmax", "softmax", "cross_entropy"])
    if kind == "reduce":
        dtype = rng.choice(["float32", "float32", "float32", "float32", "float64", "int32", "int8"])
        item = torch.empty(0, dtype=DTYPES[dtype]).element_size()
        form = rng.choice(["flat", "rows", "dims"])
        if form == "flat":
            shape = [_log_int(rng, 1000, 1 << 26)]
            dims = [""]
        elif form == "rows":
            shape = [_log_int(rng, 8, 8192), _log_int(rng, 32, 200000)]
            dims = ["1"]
        else:
            shape = [_log_int(rng, 8, 512), _log_int(rng, 16, 2048), _log_int(rng, 16, 2048)]
            dims = ["0", "1", "2"]
        ops = ["sum", "amax", "argmax"] + (["mean", "var", "std"] if dtype.startswith("float") else [])
        plan = " ".join("%s:%s" % (rng.choice(ops), d) for d in dims for _ in range(2))
        return {"kind": kind, "shape": _text(_fit(shape, item)), "dtype": dtype, "plan": plan}
    if kind == "channels":
        hw = _log_int(rng, 5, 120)
        return {"kind": kind, "shape": _text(_fit([_log_int(rng, 8, 256), _log_int(rng, 8, 512), hw,
                                                   max(3, hw + rng.randint(-2, 2))], 4))}
    if kind == "images":
        return {"kind": kind, "shape": _text(_fit([_log_int(rng, 1, 256), _log_int(rng, 28, 512),
                                                   _log_int(rng, 28, 512), rng.choice([1, 3, 3, 3, 4])], 4))}
    if kind == "topk":
        dtype = rng.choice(["float32", "float32", "float32", "float64", "int32"])
        rows, cols = _log_int(rng, 1, 16384), _log_int(rng, 64, 200000)
        rows, cols = _fit([rows, cols], 8)
        return {"kind": kind, "rows": rows, "cols": cols, "k": min(cols, _log_int(rng, 1, 2048)), "dtype": dtype,
                "largest": rng.random() < 0.8}
    if kind == "sample":
        # Temperatures and nuclei that decoding uses.  Hotter ones draw from the
        # flat tail, where the steps of the cumulative sums are as small as the
        # rounding of a float32 sum and two correct draws often differ.
        rows, cols = _fit([_log_int(rng, 1, 256), _log_int(rng, 1000, 200000)], 8)
        k = rng.choice([_log_int(rng, 5, 500), cols])
        return {"kind": kind, "rows": rows, "cols": cols, "k": k,
                "temperature": round(rng.uniform(0.5, 0.9), 2), "top_p": round(rng.uniform(0.7, 0.95), 2)}
    if kind == "softmax":
        dtype = rng.choice(["float32", "float32", "float32", "float64"])
        item = 8 if dtype == "float64" else 4
        if rng.random() < 0.6:
            shape, dim = [_log_int(rng, 8, 32768), _log_int(rng, 10, 160000)], 1
        else:
            shape, dim = [_log_int(rng, 4, 128), _log_int(rng, 8, 2048), _log_int(rng, 32, 4096)], 1
        return {"kind": kind, "shape": _text(_fit(shape, item)), "dim": dim, "log": rng.random() < 0.5, "dtype": dtype}
    rows, cols = _fit([_log_int(rng, 32, 8192), _log_int(rng, 10, 150000)], 4)
    return {"kind": kind, "rows": rows, "cols": cols}


def _shape(case):
    return [int(s) for s in case["shape"].split("x")]


def _plan(case):
    for item in case["plan"].split():
        op, dims = item.split(":")
        yield op, [int(d) for d in dims.split(",")] if dims else None


def _normal(shape, gen, mean=0.0, std=1.0):
    return torch.empty(shape, device=DEV).normal_(mean, std, generator=gen)


def _logits(rows, cols, gen):
    """Logits as bench.py draws them for its vocabulary rows: N(0, 3) with a few
    likely tokens in each row."""
    x = _normal((rows, cols), gen, 0.0, 3.0)
    at = torch.randint(0, cols, (rows, 8), generator=gen, device=DEV)
    return x.scatter_add_(1, at, torch.full((rows, 8), 15.0, device=DEV))


def _inputs(case, seed):
    """The input tensors of a case."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    kind = case["kind"]
    if kind == "reduce":
        shape, dt = _shape(case), DTYPES[case["dtype"]]
        x = _normal(shape, gen, 0.5, 2.0)
        return [x if dt == torch.float32 else x.double() if dt == torch.float64
                else (x * 20).round_().clamp_(-127, 127).to(dt)]
    if kind == "channels":
        shape = _shape(case)
        return [_normal(shape, gen, 0.5, 2.0), _normal((shape[1],), gen), _normal((shape[1],), gen)]
    if kind == "images":
        return [torch.randint(0, 256, _shape(case), generator=gen, device=DEV, dtype=torch.uint8)]
    if kind == "topk":
        dt = DTYPES[case["dtype"]]
        if case["cols"] > 30000:
            x = _logits(case["rows"], case["cols"], gen)
        else:
            x = torch.rand((case["rows"], case["cols"]), generator=gen, device=DEV) * 2 - 1
        return [x if dt == torch.float32 else x.double() if dt == torch.float64
                else (x * (1 << 24)).to(dt)]
    if kind == "sample":
        return [_logits(case["rows"], case["cols"], gen), torch.rand((case["rows"],), generator=gen, device=DEV)]
    if kind == "softmax":
        shape, dt = _shape(case), DTYPES[case["dtype"]]
        return [_normal(shape, gen, 0.0, 3.0).to(dt), _normal(shape, gen).to(dt)]
    n, c = case["rows"], case["cols"]
    return [_normal((n, c), gen, 0.0, 3.0), torch.randint(0, c, (n,), generator=gen, device=DEV)]


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _work(n):
    return torch.empty(max(int(n), 1), dtype=torch.uint8, device=DEV)


def _reduce(x, op, dims):
    nd = x.dim()
    rd = list(range(nd)) if dims is None else dims
    tmap = capi._torch_dtypes()
    od = capi.default_out_dtype(op, tmap[x.dtype])
    out = torch.empty([x.shape[i] for i in range(nd) if i not in rd], device=DEV,
                      dtype={v: k for k, v in tmap.items()}[od])
    desc = capi.make_desc(op, list(x.shape), list(x.stride()), rd, od, 1, in_dtype=tmap[x.dtype])
    lib = capi.lib()
    n = lib.tpr_reduce_workspace_bytes(ctypes.byref(desc))
    ws = _work(n)
    return lib.tpr_reduce, (ctypes.byref(desc), _ptr(x), _ptr(out), _ptr(ws), n, _stream()), [out], (desc, ws)


def _reduce_backward(grad, x, op, dims):
    desc = capi.make_desc(op, list(x.shape), list(x.stride()), dims, capi.FLOAT32, 1)
    out = torch.empty_like(x)
    lib = capi.lib()
    n = lib.tpr_reduce_backward_workspace_bytes(ctypes.byref(desc))
    ws = _work(n)
    return (lib.tpr_reduce_backward, (ctypes.byref(desc), _ptr(grad), _ptr(x), ctypes.c_void_p(0), _ptr(out),
                                      _ptr(ws), n, _stream()), [out], (desc, ws))


def _copy(src, dtype):
    """A dense copy of the view `src` in `dtype`."""
    out = torch.empty(list(src.shape), dtype=dtype, device=DEV)
    tmap = capi._torch_dtypes()
    desc = capi.make_copy_desc(list(src.shape), list(out.stride()), list(src.stride()), tmap[dtype], tmap[src.dtype])
    return capi.lib().tpr_copy, (ctypes.byref(desc), _ptr(out), _ptr(src), _stream()), [out], (desc,)


def _softmax(a, dim, mode, b=None):
    out = torch.empty_like(a)
    desc = capi.SoftmaxDesc()
    desc.mode, desc.dtype = mode, capi.FLOAT64 if a.dtype == torch.float64 else capi.FLOAT32
    desc.outer, desc.n, desc.inner = math.prod(a.shape[:dim]), a.shape[dim], math.prod(a.shape[dim + 1:])
    for s in (desc.a_strides, desc.b_strides):
        s[0], s[1], s[2] = desc.n * desc.inner, desc.inner, 1
    lib = capi.lib()
    n = lib.tpr_softmax_workspace_bytes(ctypes.byref(desc))
    ws = _work(n)
    return (lib.tpr_softmax, (ctypes.byref(desc), _ptr(a), _ptr(b) if b is not None else ctypes.c_void_p(0),
                              _ptr(out), _ptr(ws), n, _stream()), [out], (desc, ws))


def _topk(x, k, largest):
    rows, cols = x.shape
    dt = capi._torch_dtypes()[x.dtype]
    vals = torch.empty((rows, k), dtype=x.dtype, device=DEV)
    idx = torch.empty((rows, k), dtype=torch.int64, device=DEV)
    lib = capi.lib()
    n = lib.tpr_topk_workspace_bytes(dt, rows, cols, k)
    ws = _work(n)
    return (lib.tpr_topk, (_ptr(x), dt, rows, cols, cols, k, int(largest), 1, _ptr(vals), _ptr(idx), _ptr(ws), n,
                           _stream()), [vals, idx], (ws,))


def _sample(x, u, k, temperature, top_p):
    rows, cols = x.shape
    ids = torch.empty((rows,), dtype=torch.int64, device=DEV)
    lib = capi.lib()
    n = lib.tpr_sample_workspace_bytes(capi.FLOAT32, rows, cols, k)
    ws = _work(n)
    return (lib.tpr_sample, (_ptr(x), capi.FLOAT32, rows, cols, cols, k, ctypes.c_float(temperature),
                             ctypes.c_float(top_p), _ptr(u), _ptr(ids), _ptr(ws), n, _stream()), [ids], (ws,))


class _Exported:
    """A result tensor under the array interface that torch reads."""

    TYPES = {tp.float32: "<f4", tp.float64: "<f8", tp.int64: "<i8"}

    def __init__(self, t):
        self.tensor = t
        self.__cuda_array_interface__ = {"shape": tuple(t.shape), "typestr": self.TYPES[t.dtype], "strides": None,
                                         "data": (t.data_ptr(), False), "version": 2}


def prepare(case, seed):
    kind = case["kind"]
    xs = _inputs(case, seed)
    if kind == "cross_entropy":
        return {"kind": kind, "x": tp.from_torch(xs[0]), "target": tp.from_torch(xs[1]),
                "grad": tp.from_torch(torch.ones((), device=DEV))}
    x = xs[0]
    if kind == "reduce":
        calls = [_reduce(x, op, dims) for op, dims in _plan(case)]
    elif kind == "channels":
        calls = [_reduce(x, "mean", [0, 2, 3]), _reduce(x, "var", [0, 2, 3]),
                 _reduce_backward(xs[1], x, "mean", [0, 2, 3]), _reduce_backward(xs[2], x, "var", [0, 2, 3])]
    elif kind == "images":
        calls = [_copy(x.permute(0, 3, 1, 2), torch.float32), _reduce(x, "amax", [1, 2]), _reduce(x, "sum", None)]
    elif kind == "topk":
        calls = [_topk(x, case["k"], case["largest"])]
    elif kind == "sample":
        calls = [_sample(x, xs[1], case["k"], case["temperature"], case["top_p"])]
    else:
        log = case["log"]
        fwd = _softmax(x, case["dim"], capi.LOG_SOFTMAX_FWD if log else capi.SOFTMAX_FWD)
        calls = [fwd, _softmax(xs[1], case["dim"], capi.LOG_SOFTMAX_BWD if log else capi.SOFTMAX_BWD, fwd[2][0])]
    return {"kind": kind, "inputs": xs, "kept": [c[3] for c in calls], "calls": [(c[0], c[1]) for c in calls],
            "outputs": [t for c in calls for t in c[2]]}


def run(state):
    if state["kind"] == "cross_entropy":
        x, target = state["x"], state["target"]
        log_probs = tp.log_softmax(x, 1)
        loss, total = tp.nll_loss(log_probs, target)
        grad = tp.nll_loss_backward(state["grad"], log_probs, target, total_weight=total)
        grad = tp._log_softmax_backward_data(grad, log_probs, 1)
        return [torch.as_tensor(_Exported(t), device=DEV) for t in (loss, grad)]
    for fn, args in state["calls"]:
        if fn(*args):
            raise RuntimeError(capi.lib().tpr_last_error().decode())
    return state["outputs"]


def _numel(case):
    return math.prod(_shape(case))


def work(case):
    """Bytes: each input of a call chain read once for each call that has to pass
    over it, each result written once.  flops: one for each element and step of
    the definition (add, compare, multiply, exponential)."""
    kind = case["kind"]
    if kind == "reduce":
        shape, item = _shape(case), torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()
        n, by = math.prod(shape), 0
        for op, dims in _plan(case):
            nout = 1 if dims is None else n // math.prod(shape[d] for d in dims)
            by += n * item + nout * (8 if op == "argmax" or (op == "sum" and item < 4) else max(item, 4))
        return {"bytes": by, "flops": 2 * n * len(list(_plan(case)))}
    if kind == "channels":  # x for the two statistics, two gradients written
        n = _numel(case)
        return {"bytes": 3 * n * 4, "flops": 8 * n}
    if kind == "images":
        n = _numel(case)
        return {"bytes": n + 4 * n, "flops": 3 * n}
    if kind == "topk":
        item = torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()
        n = case["rows"] * case["cols"]
        return {"bytes": n * item + case["rows"] * case["k"] * (item + 8), "flops": n}
    if kind == "sample":
        n = case["rows"] * case["cols"]
        return {"bytes": n * 4 + case["rows"] * 12, "flops": 3 * n}
    if kind == "softmax":  # x read and y written, then g and y read and the gradient written
        n = _numel(case)
        return {"bytes": 5 * n * (8 if case["dtype"] == "float64" else 4), "flops": 8 * n}
    n = case["rows"] * case["cols"]
    return {"bytes": 2 * n * 4 + case["rows"] * 8, "flops": 8 * n}


def tolerance(case):
    kind = case["kind"]
    if kind == "topk" or kind == "images":
        return "exact"
    if kind == "sample":  # a draw that falls between two roundings of the cumulative sums
        return {"rel": 0.0, "differ": 0.01}
    if kind == "reduce" and case["dtype"].startswith("int"):
        return "exact"
    if kind == "reduce" or kind == "channels":
        # float32 results of 64-bit sums
        return {"rel": 1e-12 if case.get("dtype") == "float64" else 1e-6}
    if kind == "softmax" and case["dtype"] == "float64":
        return {"rel": 1e-11}
    return {"rel": 1e-6, "max": 1e-4}  # float32 exponentials and sums: 1e-7 to 2e-7 from 64 bits


def exact(case, seed):
    kind = case["kind"]
    xs = _inputs(case, seed)
    x = xs[0]
    if kind == "sample":
        return None
    if kind == "topk":
        return [torch.topk(x, case["k"], dim=1, largest=case["largest"]).values.double(), None]
    if kind == "images":
        return [x.permute(0, 3, 1, 2).double(), x.amax((1, 2)), x.sum(dtype=torch.int64)]
    if kind == "reduce":
        outs = []
        for op, dims in _plan(case):
            if op == "argmax":
                outs.append(None)
                continue
            d = x.double()
            rd = tuple(range(x.dim())) if dims is None else tuple(dims)
            outs.append({"sum": lambda: d.sum(rd), "mean": lambda: d.mean(rd), "amax": lambda: d.amax(rd),
                         "var": lambda: d.var(rd), "std": lambda: d.std(rd)}[op]())
        return outs
    if kind == "channels":
        d, rd = x.double(), (0, 2, 3)
        n = x.numel() // x.shape[1]
        gm, gv = xs[1].double().view(1, -1, 1, 1), xs[2].double().view(1, -1, 1, 1)
        mean = d.mean(rd, keepdim=True)
        return [mean.flatten(), d.var(rd), (gm / n).expand_as(d), gv * 2 / (n - 1) * (d - mean)]
    if kind == "softmax":
        dim, log = case["dim"], case["log"]
        y = (torch.log_softmax if log else torch.softmax)(x.double(), dim)
        g = xs[1].double()
        if log:
            return [y, g - y.exp() * g.sum(dim, keepdim=True)]
        return [y, (g - (g * y).sum(dim, keepdim=True)) * y]
    lp = torch.log_softmax(x.double(), 1)
    at = xs[1].view(-1, 1)
    g = lp.exp().scatter_add_(1, at, torch.full_like(at, -1.0, dtype=torch.float64))
    return [-lp.gather(1, at).mean(), g / x.shape[0]]
