"""The work that users of this package have it do, as cases that a timing harness runs.

``listed()`` names the sizes that stand for each public operator of ``lego_amd.ops``; ``draw(rng)`` gives more
cases of the same ranges, and ``prepare`` / ``run`` make a case's inputs and take one pass through the operator.
"""
import math

import torch

from lego_amd import ops

_DTYPES = {
    "f16": torch.float16,
    "bf16": torch.bfloat16,
    "f32": torch.float32,
    "e4m3": torch.float8_e4m3fn,
    "e5m2": torch.float8_e5m2,
}
_BYTES = {"f16": 2, "bf16": 2, "f32": 4, "e4m3": 1, "e5m2": 1}

# Eight independent products with every side out of {1024, 2048, 4096}: bench.py's grouped launch.
_EIGHT = ("4096x1024x2048 1024x4096x2048 2048x4096x1024 2048x2048x1024 "
          "4096x4096x1024 1024x1024x1024 4096x2048x1024 1024x1024x1024")


def listed():
    return [
        # an ordinary fp32 layout change: the LEGO TileBy transpose, 64 MiB in and out
        {"name": "transpose_f32_4096", "op": "transpose", "dtype": "f32", "rows": 4096, "cols": 4096},
        # a large 16-bit layout change whose rows start at any element: tensors that nobody padded
        {"name": "transpose_f16_odd", "op": "transpose", "dtype": "f16", "rows": 9999, "cols": 10001},
        # attention scores: the row softmax of a large half-precision matrix
        {"name": "softmax_f16_8192", "op": "softmax", "dtype": "f16", "rows": 8192, "cols": 8192},
        # the smallest training step: forward and backward of a LayerNorm over one short sequence; launches and
        # host work are what it costs
        {"name": "layernorm_bf16_small", "op": "layernorm", "dtype": "bf16", "rows": 512, "cols": 768},
        # a LayerNorm training step at the reference benchmark's own row count and a long row
        {"name": "layernorm_f16_4096x8192", "op": "layernorm", "dtype": "f16", "rows": 4096, "cols": 8192},
        # the dense product of a large prefill or training step
        {"name": "gemm_f16_8192", "op": "gemm", "dtype": "f16", "m": 8192, "n": 8192, "k": 8192,
         "layout": "nn", "activation": "", "out": "f16"},
        # decode: a few rows against a large weight stored k-major, bound by reading the weight once
        {"name": "gemm_bf16_decode", "op": "gemm", "dtype": "bf16", "m": 16, "n": 8192, "k": 8192,
         "layout": "nt", "activation": "", "out": "bf16"},
        # an ordinary 8-bit layer with a fused activation, row-major operands, a batch that no tile divides
        {"name": "gemm_e5m2_1000", "op": "gemm", "dtype": "e5m2", "m": 1000, "n": 2048, "k": 2048,
         "layout": "nn", "activation": "leaky_relu", "out": "f16"},
        # independent products of different sizes in one launch (experts, adapters)
        {"name": "grouped_f16_eight", "op": "grouped", "problems": _EIGHT},
        # one time step of a dense 27-point stencil over a row-major field
        {"name": "stencil_f3d_384", "op": "stencil", "kind": "f3d", "n": 384, "radius": 1, "bricks": False},
        # alignment of two long sequences
        {"name": "nw_8192", "op": "nw", "n": 8192, "penalty": 10},
        # factorisation of a dense fp32 matrix, the smallest size the reference publishes
        {"name": "lud_4096", "op": "lud", "n": 4096},
    ]


def _log(rng, lo, hi):
    """A whole number, its logarithm spread evenly."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _side(rng, lo, hi):
    """A matrix side: half of them whole 64s as most tensors have them, a quarter whole 8s, the rest anything."""
    v = _log(rng, lo, hi)
    step = rng.choice((64, 64, 8, 1))
    return max(step, v // step * step) if v >= step else v


def draw(rng):
    op = rng.choice(("transpose",) * 2 + ("softmax",) * 2 + ("layernorm",) * 2 + ("gemm",) * 4 + ("grouped",) * 2 +
                    ("stencil",) * 2 + ("nw", "lud"))
    if op in ("transpose", "softmax"):
        dtype = rng.choice(("f16", "bf16", "f32"))
        rows = _side(rng, 16, 16384)
        cols = _side(rng, 16, min(32768, (1 << 27) // rows))
        return {"op": op, "dtype": dtype, "rows": rows, "cols": cols}
    if op == "layernorm":
        dtype = rng.choice(("f16", "bf16", "f32"))
        rows = _side(rng, 16, 16384)
        cols = _side(rng, 64, min(16384, (1 << 26) // rows))
        return {"op": op, "dtype": dtype, "rows": rows, "cols": cols}
    if op == "gemm":
        dtype = rng.choice(("f16", "f16", "bf16", "bf16", "e4m3", "e5m2"))
        out = rng.choice(("f16", "bf16")) if dtype == "bf16" else "f16"
        m, n, k = _side(rng, 1, 8192), _side(rng, 64, 8192), _side(rng, 64, 8192)
        return {"op": op, "dtype": dtype, "m": m, "n": n, "k": k, "layout": rng.choice(("nn", "nt", "tn", "tt")),
                "activation": rng.choice(("", "", "leaky_relu")), "out": out}
    if op == "grouped":
        problems = ["%dx%dx%d" % tuple(_side(rng, 64, 4096) for _ in range(3)) for _ in range(rng.randint(1, 16))]
        return {"op": op, "problems": " ".join(problems)}
    if op == "stencil":
        kind = rng.choice(("f3d", "laplacian"))
        return {"op": op, "kind": kind, "n": _log(rng, 4, 64) * 8, "radius": rng.randint(1, 3 if kind == "f3d" else 4),
                "bricks": rng.random() < 0.5}
    if op == "nw":
        return {"op": op, "n": _log(rng, 1, 128) * 64, "penalty": rng.randint(1, 16)}
    return {"op": op, "n": _log(rng, 1, 64) * 64}


def _problems(case):
    return [tuple(int(s) for s in p.split("x")) for p in case["problems"].split()]


def _stored(shape, transposed, make):
    """A matrix of this shape, row-major or (a ``.T`` view) column-major."""
    return make(shape[1], shape[0]).t() if transposed else make(*shape)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape):
        return torch.randn(*shape, device="cuda", generator=g)

    op = case["op"]
    if op == "transpose":
        x = torch.rand(case["rows"], case["cols"], device="cuda", generator=g) * 2 - 1
        return {"case": case, "x": x.to(_DTYPES[case["dtype"]])}
    if op == "softmax":
        return {"case": case, "x": (2 * randn(case["rows"], case["cols"])).to(_DTYPES[case["dtype"]])}
    if op == "layernorm":
        dtype, n = _DTYPES[case["dtype"]], case["cols"]
        return {
            "case": case,
            "x": (2 * randn(case["rows"], n)).to(dtype).requires_grad_(),
            "w": (1 + 0.1 * randn(n)).to(dtype).requires_grad_(),
            "b": (0.1 * randn(n)).to(dtype).requires_grad_(),
            "dy": (0.1 * randn(case["rows"], n)).to(dtype),
        }
    if op == "gemm":
        m, n, k, dtype = case["m"], case["n"], case["k"], _DTYPES[case["dtype"]]
        # 8-bit operands as the reference's own 8-bit run makes them; the others scaled so that results stay near one
        scale = 1.0 if _BYTES[case["dtype"]] == 1 else 1 / math.sqrt(k)
        ta, tb = (letter == "t" for letter in case["layout"])
        a = _stored((m, k), ta, lambda *s: (scale * randn(*s)).to(dtype))
        b = _stored((k, n), tb, lambda *s: (scale * randn(*s)).to(dtype))
        return {"case": case, "a": a, "b": b}
    if op == "grouped":
        a, b = [], []
        for m, n, k in _problems(case):
            a.append((randn(m, k) / math.sqrt(k)).half())
            b.append((randn(k, n) / math.sqrt(k)).half())
        return {"case": case, "a": a, "b": b}
    if op == "stencil":
        n, r = case["n"], case["radius"]
        x = torch.rand(n, n, n, device="cuda", generator=g) * 2 - 1
        c = torch.rand((8, 8, 8) if case["kind"] == "f3d" else (r + 1,), device="cuda", generator=g)
        return {"case": case, "x": x, "c": c}
    if op == "nw":
        n = case["n"]
        scores = torch.randint(-4, 12, (n + 1, n + 1), device="cuda", generator=g, dtype=torch.int32)
        matrix = torch.zeros(n + 1, n + 1, device="cuda", dtype=torch.int32)
        border = -torch.arange(n + 1, device="cuda", dtype=torch.int32) * case["penalty"]
        matrix[:, 0] = border
        matrix[0, :] = border
        return {"case": case, "scores": scores, "matrix": matrix}
    m = torch.rand(case["n"], case["n"], device="cuda", generator=g)
    m.diagonal().add_(float(case["n"]))
    return {"case": case, "m": m}


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "transpose":
        return ops.transpose(state["x"])
    if op == "softmax":
        return ops.softmax(state["x"])
    if op == "layernorm":
        # forward and backward; the gradients are asked for and not accumulated
        x, w, b = state["x"], state["w"], state["b"]
        y = ops.lego_layer_norm(x, (case["cols"],), w, b, 1e-5)
        return (y.detach(),) + torch.autograd.grad(y, (x, w, b), state["dy"])
    if op == "gemm":
        return ops.matmul(state["a"], state["b"], activation=case["activation"], out_dtype=_DTYPES[case["out"]])
    if op == "grouped":
        return ops.lego_group_gemm_fn(state["a"], state["b"])
    if op == "stencil":
        call = ops.stencil_f3d if case["kind"] == "f3d" else ops.stencil_laplacian
        return call(state["x"], state["c"], case["radius"], case["bricks"])
    if op == "nw":
        return ops.needleman_wunsch(state["scores"], state["matrix"], case["penalty"])
    return ops.lud(state["m"].clone())      # in place: the factors of a copy, the matrix stays


def work(case):
    op = case["op"]
    if op in ("transpose", "softmax"):
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * n * _BYTES[case["dtype"]], "flops": 0 if op == "transpose" else 5 * n}
    if op == "layernorm":
        # forward: x in, y out; backward: dy and x in, dx out; the vectors beside them
        n, cols, rows = case["rows"] * case["cols"], case["cols"], case["rows"]
        return {"bytes": (5 * n + 5 * cols) * _BYTES[case["dtype"]] + 4 * rows * 4, "flops": 8 * n + 12 * n}
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": (m * k + k * n) * _BYTES[case["dtype"]] + m * n * 2, "flops": 2 * m * n * k}
    if op == "grouped":
        return {"bytes": sum(2 * (m * k + k * n + m * n) for m, n, k in _problems(case)),
                "flops": sum(2 * m * n * k for m, n, k in _problems(case))}
    if op == "stencil":
        n, r = case["n"], case["radius"]
        points = 2 * (2 * r + 1) ** 3 if case["kind"] == "f3d" else 7 * r + 1
        return {"bytes": 2 * 4 * n ** 3, "flops": points * n ** 3}
    if op == "nw":
        return {"bytes": 2 * 4 * case["n"] ** 2, "flops": 5 * case["n"] ** 2}
    return {"bytes": 2 * 4 * case["n"] ** 2, "flops": 2 * case["n"] ** 3 // 3}


def tolerance(case):
    """Four times what the operators' results differ from the same computed in 64 bits.  16-bit results differ by their
    own rounding (rel 2.1e-4 and 1.7e-3, max 4.9e-4 and 3.9e-3), whatever is summed in which order in fp32."""
    op = case["op"]
    if op in ("transpose", "nw"):
        return "exact"
    if op == "stencil":      # fp32 sums of up to 344 products one after another: rel 3.3e-7, max 2.2e-6
        return {"rel": 1.3e-6, "max": 8.7e-6}
    if op == "lud":          # n = 4096: rel 3.9e-7, max 1.2e-6
        return {"rel": 1.6e-6, "max": 4.6e-6}
    out = {"gemm": case.get("out"), "grouped": "f16"}.get(op) or case["dtype"]
    if out == "f32":         # softmax rel 8e-8, max 3.6e-7; gradients of LayerNorm over 1216 rows rel 2.2e-7, max 1.0e-6
        return {"rel": 1e-6, "max": 4e-6}
    return {"rel": 8.3e-4, "max": 2.1e-3} if out == "f16" else {"rel": 6.6e-3, "max": 1.6e-2}


def _rows(x):
    """64-bit slices of a matrix, few enough rows at a time for the temporaries to stay small."""
    step = max(1, (1 << 25) // x.shape[1])
    return [(slice(i, i + step), x[i:i + step].double()) for i in range(0, x.shape[0], step)]


def _exact_layernorm(s):
    x, w, b, dy = (s[k].detach() for k in ("x", "w", "b", "dy"))
    wd, bd = w.double(), b.double()
    y, dx = torch.empty_like(x, dtype=torch.float64), torch.empty_like(x, dtype=torch.float64)
    dw, db = torch.zeros_like(wd), torch.zeros_like(bd)
    for rows, xd in _rows(x):
        d = dy[rows].double()
        mean = xd.mean(1, keepdim=True)
        rstd = (xd.var(1, unbiased=False, keepdim=True) + 1e-5).rsqrt()
        xhat, g = (xd - mean) * rstd, d * wd
        y[rows] = xhat * wd + bd
        dx[rows] = (g - g.mean(1, keepdim=True) - xhat * (g * xhat).mean(1, keepdim=True)) * rstd
        dw += (d * xhat).sum(0)
        db += d.sum(0)
    return y, dx, dw, db


def _exact_product(a, b):
    return a.to(torch.float64) @ b.to(torch.float64)


def _exact_stencil(case, x, c):
    n, r = case["n"], case["radius"]
    x, c = x.double(), c.double().tolist()
    if case["bricks"]:       # 8 x 8 x 8 points after one another, the bricks row-major
        x = x.view(n // 8, n // 8, n // 8, 8, 8, 8).permute(0, 3, 1, 4, 2, 5).reshape(n, n, n)
    out = torch.zeros_like(x)
    core = out[r:n - r, r:n - r, r:n - r]

    def at(di, dj, dk):
        return x[r + di:n - r + di, r + dj:n - r + dj, r + dk:n - r + dk]

    if case["kind"] == "f3d":     # the centre counts once on its own and once more in the window
        core.add_(at(0, 0, 0), alpha=c[r][r][r])
        span = range(-r, r + 1)
        for di in span:
            for dj in span:
                for dk in span:
                    core.add_(at(di, dj, dk), alpha=c[di + r][dj + r][dk + r])
    else:
        core.add_(at(0, 0, 0), alpha=c[0])
        for d in range(1, r + 1):
            for step in ((d, 0, 0), (-d, 0, 0), (0, d, 0), (0, -d, 0), (0, 0, d), (0, 0, -d)):
                core.add_(at(*step), alpha=c[d])
    if case["bricks"]:
        out = out.view(n // 8, 8, n // 8, 8, n // 8, 8).permute(0, 2, 4, 1, 3, 5).reshape(n, n, n)
    return out


def _exact_lu(m):
    """L and U in one matrix, no pivoting: panels of 64 columns, the rest by matrix products."""
    m, n = m.double(), m.shape[0]
    for k in range(0, n, 64):
        e = min(k + 64, n)
        panel = m[k:, k:e]
        for j in range(e - k - 1 if e == n else e - k):
            panel[j + 1:, j] /= panel[j, j]
            panel[j + 1:, j + 1:].addr_(panel[j + 1:, j], panel[j, j + 1:], alpha=-1)
        if e < n:
            lower = m[k:e, k:e].tril(-1) + torch.eye(e - k, device=m.device, dtype=m.dtype)
            m[k:e, e:] = torch.linalg.solve_triangular(lower, m[k:e, e:], upper=False, unitriangular=True)
            m[e:, e:] -= m[e:, k:e] @ m[k:e, e:]
    return m


def exact(case, seed):
    """What ``run`` returns for these inputs, from plain torch operations in 64 bits (None: bits moved or whole numbers)."""
    op = case["op"]
    if op in ("transpose", "nw"):
        return None
    s = prepare(case, seed)
    if op == "softmax":
        out = torch.empty_like(s["x"], dtype=torch.float64)
        for rows, xd in _rows(s["x"]):
            out[rows] = torch.softmax(xd, 1)
        return out
    if op == "layernorm":
        return _exact_layernorm(s)
    if op == "gemm":
        c = _exact_product(s["a"], s["b"])
        return torch.where(c >= 0, c, 0.01 * c) if case["activation"] else c
    if op == "grouped":
        return [_exact_product(a, b) for a, b in zip(s["a"], s["b"])]
    if op == "stencil":
        return _exact_stencil(case, s["x"], s["c"])
    return _exact_lu(s["m"])
