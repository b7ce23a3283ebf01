"""The work a user of this framework has it do, case by case, for timing it.

Every case goes through the Python binding's public entry points on device
buffers the program holds, on one runtime handle that the process keeps:

  gemm      GpuRuntime.gemm_desc: one C = op(A) op(B), bf16 in, fp32 accumulate
  dispatch  the reference-style sequence: a tile kernel, its kernargs and grid
            prepared once, then one asynchronous dispatch per pass
  matmul    the f32 Linear forward, both operands converted on every call
  linear    one training step of an f32 Linear layer: forward and data gradient
            with the weight's bf16 copy from the cache, weight gradient, and the
            invalidation that a weight update brings
  mlp       one training step of a bf16 two-layer MLP: six GEMMs

Sizes are m x n x k of the (forward) product.  `draw` covers the same ranges:
1 to 8192 rows, 64 to 16384 columns, K to 65536, every layout, both output
types, epilogue chains, padded leading dimensions, and sizes that are multiples
of 64, of 8, or odd.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "t0-gpu_amd"))
import t0g  # noqa: E402

_runtime = None


def _rt():
    """The process's runtime handle, opened once, as a program keeps it."""
    global _runtime
    if _runtime is None:
        _runtime = t0g.GpuRuntime.new(0)
    return _runtime


def _gemm(name, m, n, k, layout, out, epilogue="", pad=0):
    return {"name": name, "kind": "gemm", "m": m, "n": n, "k": k, "layout": layout, "out": out,
            "epilogue": epilogue, "pad": pad}


def listed():
    return [
        # the reference's smallest configuration: launch latency decides
        _gemm("gemm_256_nt_f32", 256, 256, 256, "NT", "f32"),
        # a small layer through the reference's own select / kernargs / grid / dispatch sequence
        {"name": "dispatch_512_nt", "kind": "dispatch", "m": 512, "n": 512, "k": 512, "layout": "NT"},
        # odd everywhere: rows that are not 16-byte aligned, a fused bias + ReLU, ragged tiles
        _gemm("gemm_odd_1001x1003x999_nt_f32", 1001, 1003, 999, "NT", "f32", "bias relu"),
        # a few rows through the MLP's wide layer: every weight is read once for little work
        _gemm("rows_16x11008x4096_nt_bf16", 16, 11008, 4096, "NT", "bf16"),
        # the thin benchmark shape: a short batch through a square layer
        _gemm("thin_128x4096x4096_nt_bf16", 128, 4096, 4096, "NT", "bf16"),
        # the split-K benchmark shape: a small output over a long contraction
        _gemm("deepk_256x256x32768_nt_f32", 256, 256, 32768, "NT", "f32"),
        # an ordinary layer with its activation fused
        _gemm("gemm_2048_nn_bf16_bias_silu", 2048, 2048, 2048, "NN", "bf16", "bias silu"),
        # the two headline benchmark shapes
        _gemm("gemm_4096_nn_bf16", 4096, 4096, 4096, "NN", "bf16"),
        _gemm("gemm_8192_nn_bf16", 8192, 8192, 8192, "NN", "bf16"),
        # f32 tensors: an ordinary layer's training step, and the MLP's wide layer, forward only
        {"name": "linear_512x3072x768_f32", "kind": "linear", "m": 512, "n": 3072, "k": 768},
        {"name": "matmul_1024x11008x4096_f32", "kind": "matmul", "m": 1024, "n": 11008, "k": 4096},
        # the MLP benchmark: hidden layer n, width k
        {"name": "mlp_1024x11008x4096_bf16", "kind": "mlp", "m": 1024, "n": 11008, "k": 4096},
    ]


def _size(rng, lo, hi, step):
    """An integer spread over the logarithm of [lo, hi], a multiple of `step` (1: odd)."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    if step == 1:
        return min(hi, max(lo, int(v))) | 1
    return max(step, int(v / step + 0.5) * step)


_EPILOGUES = ["", "", "", "bias", "bias relu", "bias silu", "gelu", "scale", "bias scale clamp"]


def draw(rng):
    kind = rng.choice(["square", "square", "square", "odd", "rows", "thin", "deepk", "dispatch", "linear", "matmul", "mlp"])
    layout = rng.choice(["NT", "NN", "TN", "TT"])
    out = rng.choice(["f32", "bf16"])
    epilogue = rng.choice(_EPILOGUES)
    pad = rng.choice([0, 0, 0, 8, 64])
    if kind in ("square", "odd"):
        step = 1 if kind == "odd" else rng.choice([64, 64, 8])
        cap = 2 ** 31 if kind == "odd" else 2 ** 38
        while True:
            m, n, k = (_size(rng, 64, 2048 if kind == "odd" else 8192, step) for _ in range(3))
            if m * n * k <= cap:
                break
        c = _gemm("", m, n, k, layout, out, epilogue, 0 if kind == "odd" else pad)
    elif kind == "rows":
        m = _size(rng, 1, 63, 1) if rng.random() < 0.5 else _size(rng, 8, 64, 8)
        # with rows stored along K (TN, TT) the row count is A's leading dimension
        c = _gemm("", m, _size(rng, 1024, 16384, 64), _size(rng, 1024, 16384, 64), rng.choice(["NT", "NN"]), out,
                  epilogue, pad)
    elif kind == "thin":
        c = _gemm("", _size(rng, 64, 256, 8), _size(rng, 1024, 8192, 64), _size(rng, 1024, 8192, 64), layout, out,
                  epilogue, pad)
    elif kind == "deepk":
        c = _gemm("", _size(rng, 64, 512, 8), _size(rng, 64, 512, 8), _size(rng, 8192, 65536, 64), layout, out,
                  epilogue, pad)
    elif kind == "dispatch":
        c = {"kind": "dispatch", "m": _size(rng, 64, 2048, 8), "n": _size(rng, 64, 2048, 64),
             "k": _size(rng, 64, 2048, 64), "layout": rng.choice(["NT", "NN"])}
    elif kind == "linear":
        c = {"kind": "linear", "m": _size(rng, 32, 2048, 8), "n": _size(rng, 128, 4096, 8), "k": _size(rng, 128, 4096, 8)}
    elif kind == "matmul":
        c = {"kind": "matmul", "m": _size(rng, 32, 2048, 8), "n": _size(rng, 128, 11008, 8),
             "k": _size(rng, 128, 4096, 8)}
    else:
        c = {"kind": "mlp", "m": _size(rng, 128, 1024, 64), "n": _size(rng, 512, 11008, 64),
             "k": _size(rng, 256, 4096, 64)}
    c.pop("name", None)
    return c


def _normal(g, rows, cols, scale, dtype, pad=0):
    """[rows][cols + pad] normal values of the given deviation; the whole pitch is filled."""
    t = torch.randn((rows, cols + pad), generator=g, device="cuda")
    return (t * scale).to(dtype)


def _shapes(case):
    m, n, k, layout = case["m"], case["n"], case["k"], case["layout"]
    return ((m, k) if layout in ("NT", "NN") else (k, m)), ((n, k) if layout in ("NT", "TT") else (k, n))


def _inputs(case, seed):
    """The case's input tensors, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    m, n, k, kind = case["m"], case["n"], case["k"], case["kind"]
    bf16, f32 = torch.bfloat16, torch.float32
    if kind in ("gemm", "dispatch"):
        sa, sb = _shapes(case)
        pad = case.get("pad", 0)
        return {"a": _normal(g, *sa, 1.0, bf16, pad), "b": _normal(g, *sb, k ** -0.5, bf16, pad),
                "bias": torch.randn(n, generator=g, device="cuda")}
    if kind == "matmul":
        return {"x": _normal(g, m, k, 1.0, f32), "w": _normal(g, k, n, k ** -0.5, f32)}
    if kind == "linear":
        return {"x": _normal(g, m, k, 1.0, f32), "w": _normal(g, k, n, k ** -0.5, f32),
                "dy": _normal(g, m, n, 0.02, f32)}
    return {"x": _normal(g, m, k, 1.0, bf16), "w1": _normal(g, k, n, (2.0 / k) ** 0.5, bf16),
            "w2": _normal(g, n, k, (2.0 / n) ** 0.5, bf16), "dy": _normal(g, m, k, 0.02, bf16)}


_SCALE, _CLAMP = 0.125, (-0.1, 0.1)


def prepare(case, seed):
    rt = _rt()
    s = _inputs(case, seed)
    m, n, k, kind = case["m"], case["n"], case["k"], case["kind"]
    s["rt"], s["case"] = rt, case

    def new(rows, cols, dtype):
        return torch.empty((rows, cols), dtype=dtype, device="cuda")

    def p(t):
        return t.data_ptr()

    if kind == "gemm":
        sa, sb = _shapes(case)
        pad = case["pad"]
        # the padding columns of C are not written: zeroed, so that C is defined as a whole
        s["c"] = torch.zeros((m, n + pad), dtype=torch.bfloat16 if case["out"] == "bf16" else torch.float32, device="cuda")
        ops = case["epilogue"].split()
        s["desc"] = t0g.gemm_desc(p(s["a"]), p(s["b"]), p(s["c"]), m, n, k, transpose=case["layout"],
                                  out_dtype=t0g.BF16 if case["out"] == "bf16" else t0g.F32, lda=sa[1] + pad,
                                  ldb=sb[1] + pad, ldc=n + pad, epilogue_ops=ops or None,
                                  bias=p(s["bias"]) if "bias" in ops else 0, epi_scale=_SCALE, clamp=_CLAMP)
    elif kind == "dispatch":
        s["c"] = new(m, n, torch.float32)
        cfg = t0g.tile_auto_select(m, k, n, t0g.LAYOUTS[case["layout"]])
        s["kernel"] = rt.ensure_tile_kernel(cfg)
        s["grid"] = t0g.tile_compute_grid(cfg, m, n)
        s["kernargs"] = t0g.build_kernargs_m(p(s["a"]), p(s["b"]), p(s["c"]), k, n, m, cfg)
    elif kind == "matmul":
        s["y"] = new(m, n, torch.float32)
    elif kind == "linear":
        s["y"], s["dx"], s["dw"] = new(m, n, torch.float32), new(m, k, torch.float32), new(k, n, torch.float32)
    else:
        bf16 = torch.bfloat16
        s["h"], s["dh"] = new(m, n, bf16), new(m, n, bf16)
        s["y"], s["dx"] = new(m, k, bf16), new(m, k, bf16)
        s["dw1"], s["dw2"] = new(k, n, bf16), new(n, k, bf16)

        def d(a, b, c, mm, nn, kk, layout):
            return t0g.gemm_desc(p(a), p(b), p(c), mm, nn, kk, transpose=layout, out_dtype=t0g.BF16)

        s["descs"] = [d(s["x"], s["w1"], s["h"], m, n, k, "NN"), d(s["h"], s["w2"], s["y"], m, k, n, "NN"),
                      d(s["dy"], s["w2"], s["dh"], m, n, k, "NT"), d(s["dh"], s["w1"], s["dx"], m, k, n, "NT"),
                      d(s["h"], s["dy"], s["dw2"], n, k, m, "TN"), d(s["x"], s["dh"], s["dw1"], k, n, m, "TN")]
    torch.cuda.synchronize()   # the runtime's stream is its own: the inputs are there before it is used
    return s


def run(s):
    rt, case = s["rt"], s["case"]
    kind = case["kind"]
    if kind == "gemm":
        rt.gemm_desc(s["desc"])
        return s["c"]
    if kind == "dispatch":
        rt.dispatch_async(s["kernel"], s["grid"], s["kernargs"])
        return s["c"]
    m, n, k = case["m"], case["n"], case["k"]
    if kind == "matmul":
        rt.matmul_f32(s["x"].data_ptr(), s["w"].data_ptr(), s["y"].data_ptr(), m, k, n)
        return s["y"]
    if kind == "linear":
        x, w, dy = s["x"].data_ptr(), s["w"].data_ptr(), s["dy"].data_ptr()
        rt.matmul_f32_cached(x, w, w, s["y"].data_ptr(), m, k, n)
        rt.matmul_backward_data_f32_cached(dy, w, w, s["dx"].data_ptr(), m, k, n)
        rt.matmul_backward_weight_f32(x, dy, s["dw"].data_ptr(), m, k, n)
        rt.invalidate_bf16(w)   # the update that follows a step changes the weight
        return {"y": s["y"], "dx": s["dx"], "dw": s["dw"]}
    for d in s["descs"]:
        rt.gemm_desc(d)
    return {v: s[v] for v in ("h", "y", "dh", "dx", "dw1", "dw2")}


def work(case):
    m, n, k, kind = case["m"], case["n"], case["k"], case["kind"]
    mnk = float(m) * n * k
    if kind == "gemm":
        return {"bytes": 2.0 * (m * k + k * n) + (2 if case["out"] == "bf16" else 4) * m * n +
                (4 * n if "bias" in case["epilogue"] else 0), "flops": 2 * mnk}
    if kind == "dispatch":
        return {"bytes": 2.0 * (m * k + k * n) + 4.0 * m * n, "flops": 2 * mnk}
    if kind == "matmul":
        return {"bytes": 4.0 * (m * k + k * n + m * n), "flops": 2 * mnk}
    if kind == "linear":
        return {"bytes": 8.0 * (m * k + k * n + m * n), "flops": 6 * mnk}
    # x, dy in and y, dx out; h and dh out; both weights in and their gradients out
    return {"bytes": 2.0 * (4 * m * k + 2 * m * n + 4 * k * n), "flops": 12 * mnk}


def tolerance(case):
    # fp32 sums in another order, then the epilogue; bf16 outputs add their own rounding
    # (2^-9 of a value at most, 1.7e-3 in the norm)
    if case["kind"] == "mlp":
        return {"rel": 1e-2}
    if case["kind"] == "gemm" and case["out"] == "bf16":
        return {"rel": 7e-3}
    return {"rel": 1e-5}


def _chain(x, case, bias):
    for op in case.get("epilogue", "").split():
        if op == "bias":
            x = x + bias.double()
        elif op == "scale":
            x = x * _SCALE
        elif op == "relu":
            x = x.clamp(min=0.0)
        elif op == "silu":
            x = x * torch.sigmoid(x)
        elif op == "gelu":   # the reference's form
            x = x * torch.sigmoid(1.702 * x)
        elif op == "clamp":
            x = x.clamp(torch.tensor(_CLAMP[0], dtype=torch.float32).item(), torch.tensor(_CLAMP[1], dtype=torch.float32).item())
    return x


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("gemm", "dispatch"):
        sa, sb = _shapes(case)
        a, b = s["a"][:, :sa[1]].double(), s["b"][:, :sb[1]].double()
        if case["layout"] in ("TN", "TT"):
            a = a.t().contiguous()
        if case["layout"] in ("NT", "TT"):
            b = b.t().contiguous()
        c = _chain(a @ b, case, s["bias"])
        pad = case.get("pad", 0)
        return torch.nn.functional.pad(c, (0, pad)) if pad else c
    if kind in ("matmul", "linear"):
        # the f32 entry points multiply their operands rounded to bf16
        x, w = s["x"].to(torch.bfloat16).double(), s["w"].to(torch.bfloat16).double()
        y = x @ w
        if kind == "matmul":
            return y
        dy = s["dy"].to(torch.bfloat16).double()
        return {"y": y, "dx": dy @ w.t().contiguous(), "dw": x.t().contiguous() @ dy}
    x, w1, w2, dy = (s[v].double() for v in ("x", "w1", "w2", "dy"))
    h, dh = x @ w1, dy @ w2.t().contiguous()
    return {"h": h, "y": h @ w2, "dh": dh, "dx": dh @ w1.t().contiguous(), "dw1": x.t().contiguous() @ dh,
            "dw2": h.t().contiguous() @ dy}
