"""Operands staged through registers (_u kernels: rows that are not 16-byte aligned),
at the sizes where the staging can go wrong: K tails around whole 64-K stages and around
the stages kept in flight, tiles one short of and one past their edge, rows of fewer than
8 values, split-K slices.  Each operand sits at an odd element offset inside a buffer of
NaN bit patterns, with NaN in its padding columns: a K value taken from outside the operand
makes the result NaN, and so does an output computed from a wrong row."""
import numpy as np
import pytest

import oracle as o
import t0g

pytestmark = pytest.mark.gpu

NAN = np.uint16(0x7FC0)


@pytest.fixture(scope="module")
def rt():
    r = t0g.GpuRuntime.new(0)
    yield r
    r.close()


def _embed(rt, stored, pad, lead):
    rows, cols = stored.shape
    full = np.full((rows, cols + pad), NAN, dtype=np.uint16)
    full[:, :cols] = stored
    # the operand ends at its last value: what follows (guard) is not part of it
    flat = full.reshape(-1)[:(rows - 1) * (cols + pad) + cols]
    host = np.concatenate([np.full(lead, NAN, np.uint16), flat, np.full(64, NAN, np.uint16)])
    addr = rt.upload(host)
    return addr, addr + 2 * lead


# (m, n, k): stage edges with 2 (128x128) and 4 (64x64) stages in flight, tile edges, tiny rows
SHAPES = [(65, 63, 63), (64, 64, 65), (63, 129, 64 * 4 + 1), (127, 66, 64 * 5 - 1), (129, 127, 64 * 8 + 7),
          (130, 70, 64 * 9), (33, 257, 7), (257, 31, 8), (5, 90, 321), (90, 3, 130), (1, 1, 200), (2, 67, 5),
          (70, 130, 1), (129, 65, 3), (1, 66, 5), (3, 2, 2), (1, 1, 1)]


@pytest.mark.parametrize("layout", ["NT", "NN", "TN", "TT"])
@pytest.mark.parametrize("preset", ["gfx950_64x64_k64", "gfx950_128x128_k64"])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_unaligned_operands(rt, layout, preset, m, n, k):
    rng = np.random.default_rng(m * 1000003 + n * 1009 + k)
    a_mk = o.f32_to_bf16_rne(rng.uniform(-0.5, 0.5, (m, k)).astype(np.float32))
    b_nk = o.f32_to_bf16_rne(rng.uniform(-0.5, 0.5, (n, k)).astype(np.float32))
    a = a_mk if layout in ("NT", "NN") else np.ascontiguousarray(a_mk.T)
    b = b_nk if layout in ("NT", "TT") else np.ascontiguousarray(b_nk.T)
    ref = o.gemm("NT", a_mk, b_nk, m, n, k)
    for pad, split in ((0, 1), (3, 1), (1, 3 if k >= 192 else 1)):
        bufs = []
        try:
            ra, da = _embed(rt, a, pad, 5)
            bufs.append(ra)
            rb, db = _embed(rt, b, pad, 3)
            bufs.append(rb)
            dc = rt.alloc(m * n * 4)
            bufs.append(dc)
            kw = dict(transpose=layout, lda=a.shape[1] + pad, ldb=b.shape[1] + pad, split_k=split,
                      config=t0g.GemmConfig.preset(preset))
            assert t0g.gemm_kernel_name(t0g.gemm_desc(da, db, dc, m, n, k, **kw)).endswith("_u")
            rt.memset(dc, 0xFF, m * n * 4)
            rt.gemm(da, db, dc, m, n, k, **kw)
            rt.wait_idle()
            c = rt.read(dc, (m, n), np.float32)
            ok, relf, maxabs, bound = o.parity(c, ref, k)
            assert ok, f"pad={pad} split={split} relF={relf:.3e} max|d|={maxabs:.3e} bound={bound:.3e}"
            rt.gemm(da, db, dc, m, n, k, out_dtype=t0g.BF16, **kw)
            rt.wait_idle()
            c16 = rt.read(dc, (m, n), np.uint16)
            assert np.array_equal(c16, o.f32_to_bf16_rne(c))
        finally:
            for x in bufs:
                rt.free(x)


def test_more_tiles_than_a_grid_row(rt):
    """More 64-column tiles than 2^32 threads hold in 512-thread workgroups: three
    quarters of them along grid y.  One row times a column vector of repeating values, so C repeats as well."""
    period, n = 65521, (1 << 29) + 64 * 5 + 3
    rng = np.random.default_rng(7)
    col = o.f32_to_bf16_rne(rng.uniform(-0.5, 0.5, period).astype(np.float32))
    a = o.f32_to_bf16_rne(np.array([0.6875], np.float32))
    want = o.f32_to_bf16_rne(o.bf16_to_f32(col) * np.float32(0.6875))
    cfg = t0g.GemmConfig.preset("gfx950_64x64_k64")
    da, db, dc = rt.upload(a), rt.upload(np.resize(col, n)), rt.alloc(n * 2)
    try:
        kw = dict(out_dtype=t0g.BF16, config=cfg)
        assert t0g.gemm_compile(t0g.gemm_desc(da, db, dc, 1, n, 1, **kw)).grid[1] == 4
        rt.memset(dc, 0xFF, n * 2)
        rt.gemm(da, db, dc, 1, n, 1, **kw)
        rt.wait_idle()
        c = rt.read(dc, (n,), np.uint16)
        whole = n - n % period
        assert np.all(c[:whole].reshape(-1, period) == want) and np.array_equal(c[whole:], want[:n % period])
        # one tile count further than a grid takes: refused, and the handle goes on working
        with pytest.raises(t0g.T0gError) as e:
            rt.gemm(da, db, dc, 1, 1 << 30, 1, **kw)
        assert e.value.code == t0g.ERR_INVALID_ARG and not rt.is_poisoned()
        rt.gemm(da, db, dc, 1, 5, 1, **kw)
        rt.wait_idle()
        assert np.array_equal(rt.read(dc, (5,), np.uint16), want[:5])
    finally:
        for x in (da, db, dc):
            rt.free(x)


@pytest.mark.parametrize("preset", ["gfx950_64x64_k64", "gfx950_128x128_k64"])
@pytest.mark.parametrize("layout,rows,ld,k", [("NT", 32764, 65537, 200), ("TN", 131, 16392001, 131)])
def test_offsets_to_the_last_bit(rt, layout, preset, rows, ld, k):
    """An unaligned operand of about 2^31 - 2^17 elements, so that 32-bit byte offsets run up to
    their last values: whole stages and the edge stage, a K-contiguous B and an M-contiguous A.  All of it
    is NaN but the rows (columns) of C that are looked at, at both ends of the operand."""
    assert (1 << 31) - (1 << 18) < rows * ld < 1 << 31
    other, size = 3, rows if layout == "NT" else ld          # the operand's M/N extent
    pieces = ((0, 70), (size - 300, 300))                    # where it holds values
    rng = np.random.default_rng(rows)
    few = o.f32_to_bf16_rne(rng.uniform(-0.5, 0.5, (other, k)).astype(np.float32))
    many = {s: o.f32_to_bf16_rne(rng.uniform(-0.5, 0.5, (c, k)).astype(np.float32)) for s, c in pieces}
    big = rt.alloc(rows * ld * 2)
    df = rt.upload(few if layout == "NT" else np.ascontiguousarray(few.T))
    dc = rt.alloc(other * size * 4)
    try:
        rt.memset(big, 0xFF, rows * ld * 2)
        for s, v in many.items():
            if layout == "NT":
                for r in range(len(v)):
                    rt.write(big + (s + r) * ld * 2, v[r])
            else:
                for r in range(k):
                    rt.write(big + (r * ld + s) * 2, np.ascontiguousarray(v[:, r]))
        m, n, a, b = (other, size, df, big) if layout == "NT" else (size, other, big, df)
        d = t0g.gemm_desc(a, b, dc, m, n, k, transpose=layout, lda=k if layout == "NT" else ld,
                          ldb=ld if layout == "NT" else other, split_k=1, config=t0g.GemmConfig.preset(preset))
        assert t0g.gemm_kernel_name(d).endswith("_u")
        rt.memset(dc, 0, other * size * 4)
        rt.gemm_desc(d)
        rt.wait_idle()
        c = rt.read(dc, (m, n), np.float32)
        c = c.T if layout == "NT" else c                     # [operand row][other]
        for s, v in many.items():
            ref = o.gemm("NT", v, few, len(v), other, k)
            ok, relf, maxabs, bound = o.parity(np.ascontiguousarray(c[s:s + len(v)]), ref, k)
            assert ok, f"at {s}: relF={relf:.3e} max|d|={maxabs:.3e} bound={bound:.3e}"
        assert np.all(np.isnan(c[70:size - 300]))
    finally:
        for x in (big, df, dc):
            rt.free(x)


@pytest.mark.parametrize("preset", ["gfx950_64x64_k64", "gfx950_128x128_k64"])
@pytest.mark.parametrize("layout", ["NT", "NN"])
@pytest.mark.parametrize("k", [5, 64, 333])
def test_dispatch_of_no_columns(rt, layout, preset, k):
    """Kernargs with N = 0 under a grid of tiles: nothing is read or stored."""
    m = 70
    cfg = t0g.GemmConfig.preset(preset).copy(transpose=t0g.LAYOUTS[layout])
    kern = rt.ensure_tile_kernel(cfg)
    da, db, dc = rt.alloc(m * k * 2), rt.alloc(256), rt.alloc(4096)
    try:
        rt.memset(dc, 0xA5, 4096)
        rt.dispatch(kern, t0g.tile_compute_grid(cfg, m, 2 * cfg.tile_n), t0g.build_kernargs_m(da, db, dc, k, 0, m, cfg))
        assert np.all(rt.read(dc, (4096,), np.uint8) == 0xA5)
    finally:
        for x in (da, db, dc):
            rt.free(x)


# ---- f32 operands rounded inside the kernel (_ff, _fb) -----------------------------

def _guarded_f32(rt, x):
    host = np.concatenate([np.full(1, np.nan, np.float32), x.reshape(-1), np.full(16, np.nan, np.float32)])
    addr = rt.upload(host)
    return addr, addr + 4


# (m, k, n) of the layer: the contraction is k forward, n for the data gradient, m for the
# weight gradient; stage edges (63, 64, 65, 129 ...), rows of fewer than 4 values, ragged
# tiles.  With each layer the route of its six calls (forward, data and weight gradient, cached
# forward and data gradient, bf16 weight): K slices of a GEMM that rounds the operands, 0 for
# converted first, "?" where it is left to the rule.
LAYERS = [(32, 128, 128, "111111"), (65, 63, 66, "111111"), (64, 64, 64, "111111"), (1, 65, 3, "111111"),
          (3, 2, 130, "111111"), (130, 129, 2, "111111"), (66, 1, 3, "111111"), (1, 2, 1, "111111"), (127, 300, 191, "111111"), (64, 2048, 64, "811818"),
          (5, 1000, 1001, "221???"), (300, 1536, 1544, "220???"), (2048, 2048, 2048, "000000"),
          (64, 1024, 4096, "480080"), (144, 1216, 1920, "??00??")]


@pytest.mark.parametrize("m,k,n,routes", LAYERS)
def test_f32_layers(rt, m, k, n, routes):
    ops = (t0g.MATMUL_FORWARD, t0g.MATMUL_BACKWARD_DATA, t0g.MATMUL_BACKWARD_WEIGHT, t0g.MATMUL_FORWARD_CACHED,
           t0g.MATMUL_BACKWARD_DATA_CACHED, t0g.MATMUL_WT_BF16)
    for op, route in zip(ops, routes):
        name, splits = t0g.matmul_kernel_name(op, m, k, n)
        staged = name.endswith("_ff" if op <= t0g.MATMUL_BACKWARD_WEIGHT else "_fb")
        assert route == "?" or route == (str(splits) if staged else "0"), (op, name, splits)
    rng = np.random.default_rng(m * 1009 + k * 31 + n)
    x = rng.uniform(-0.5, 0.5, (m, k)).astype(np.float32)
    w = rng.uniform(-0.5, 0.5, (k, n)).astype(np.float32)
    dy = rng.uniform(-0.5, 0.5, (m, n)).astype(np.float32)
    xb, wb, dyb = (o.f32_to_bf16_rne(v) for v in (x, w, dy))
    t = np.ascontiguousarray
    y_ref = o.gemm("NT", xb, t(wb.T), m, n, k)
    dx_ref = o.gemm("NT", dyb, wb, m, k, n)
    dw_ref = o.gemm("NT", t(xb.T), t(dyb.T), k, n, m)
    bufs = []
    try:
        (bx, dx_), (bw, dw_), (bd, dd_) = (_guarded_f32(rt, v) for v in (x, w, dy))
        bufs += [bx, bw, bd]
        out = rt.alloc(max(m * n, m * k, k * n) * 4)
        bufs.append(out)

        def check(what, shape, ref, kk, call):
            rt.memset(out, 0xFF, shape[0] * shape[1] * 4)
            call()
            rt.wait_idle()
            ok, relf, maxabs, bound = o.parity(rt.read(out, shape, np.float32), ref, kk)
            assert ok, f"{what}: relF={relf:.3e} max|d|={maxabs:.3e} bound={bound:.3e}"

        check("forward", (m, n), y_ref, k, lambda: rt.matmul_f32(dx_, dw_, out, m, k, n))
        check("data gradient", (m, k), dx_ref, n, lambda: rt.matmul_backward_data_f32(dd_, dw_, out, m, k, n))
        check("weight gradient", (k, n), dw_ref, m, lambda: rt.matmul_backward_weight_f32(dx_, dd_, out, m, k, n))
        check("cached forward", (m, n), y_ref, k, lambda: rt.matmul_f32_cached(dx_, dw_, 77, out, m, k, n))
        check("cached data gradient", (m, k), dx_ref, n,
              lambda: rt.matmul_backward_data_f32_cached(dd_, dw_, 77, out, m, k, n))
        wt = rt.upload(t(wb.T))
        bufs.append(wt)
        check("bf16 weight", (m, n), y_ref, k, lambda: rt.matmul_wt_bf16_f32(dx_, wt, out, m, k, n))
    finally:
        rt.clear_bf16_cache()
        for b in bufs:
            rt.free(b)


def test_f32_rounding_inside_the_kernel(rt):
    """The operand conversion's integer rounding: ties to even, overflow to infinity, denormals, and a
    NaN whose mantissa carries past the exponent becoming -0 (no special case), as t0g_f32_to_bf16."""
    m, k, n = 64, 64, 64
    bits = np.array([0x3F808000, 0x3F818000, 0x3F807FFF, 0x7F7FFFFF, 0xFF7FFFFF, 0x00000001, 0x00008000, 0x00018000,
                     0x807FFFFF, 0x7FFF8001, 0xFFFFFFFF, 0x7F800000, 0x7FC00000, 0x80000000], dtype=np.uint32)
    x = np.zeros((m, k), dtype=np.float32)
    for i, b in enumerate(bits):   # one value per row, so a NaN or an infinity stays in its row
        x[i, i] = np.array([b], np.uint32).view(np.float32)[0]
    w = np.eye(k, n, dtype=np.float32)
    dx_, dw_ = rt.upload(x), rt.upload(w)
    out = rt.alloc(m * n * 4)
    d16 = rt.alloc(m * k * 2)
    try:
        rt.matmul_f32(dx_, dw_, out, m, k, n)
        rt.f32_to_bf16(dx_, d16, m * k)
        rt.wait_idle()
        y = rt.read(out, (m, n), np.float32)
        x16 = o.bf16_to_f32(rt.read(d16, (m, k), np.uint16))
        for i in range(len(bits)):
            v = x16[i, i]
            if np.isfinite(v):
                # bf16 denormals as MFMA operands: kept or flushed, alike for every kernel
                assert y[i, i] == v or (abs(v) < 2.0 ** -126 and y[i, i] == 0.0), f"{bits[i]:08x}: {y[i, i]} for {v}"
            elif np.isinf(v):
                assert y[i, i] == v and np.all(np.isnan(np.delete(y[i], i))), f"{bits[i]:08x}"
            else:
                assert np.all(np.isnan(y[i])), f"{bits[i]:08x}"
    finally:
        for b in (dx_, dw_, out, d16):
            rt.free(b)


# (m, k, n), the call, the operand that the output lies over and by how many values it starts
# past it: layers small enough to be rounded inside the GEMM and one that is converted first
OVERLAPS = [(512, 512, 512, "forward", "x", 0), (1024, 1024, 1024, "forward", "x", 0),
            (1024, 1024, 1024, "forward", "w", 0), (1024, 1024, 1024, "forward", "x", 4096),
            (1024, 1024, 1024, "forward", "w", -4096), (1024, 1024, 1024, "cached forward", "x", 0),
            (1024, 1024, 1024, "bf16 weight", "x", 0), (1024, 1024, 1024, "data gradient", "dy", 0),
            (1024, 1024, 1024, "data gradient", "w", 0), (1024, 1024, 1024, "cached data gradient", "dy", 0),
            (1024, 1024, 1024, "weight gradient", "x", 0), (1024, 1024, 1024, "weight gradient", "dy", 0),
            (512, 768, 3072, "cached forward", "x", 0), (2001, 333, 1777, "bf16 weight", "x", 0),
            (2001, 1777, 333, "cached data gradient", "dy", 0), (640, 512, 512, "forward", "x", 0), (65, 63, 63, "forward", "x", 0), (2048, 2048, 2048, "forward", "x", 0)]


@pytest.mark.parametrize("m,k,n,call,over,shift", OVERLAPS)
def test_f32_output_over_an_operand(rt, m, k, n, call, over, shift):
    """The f32 calls take a private copy of an operand that their output lies over, so the
    result is that of separate buffers."""
    rng = np.random.default_rng(m + 3 * k + 5 * n + len(call))
    host = {"x": rng.uniform(-0.5, 0.5, (m, k)).astype(np.float32),
            "w": rng.uniform(-0.5, 0.5, (k, n)).astype(np.float32),
            "dy": rng.uniform(-0.5, 0.5, (m, n)).astype(np.float32)}
    t = np.ascontiguousarray
    xb, wb, dyb = (o.f32_to_bf16_rne(host[v]) for v in ("x", "w", "dy"))
    shape, ref, kk = {"forward": ((m, n), (xb, t(wb.T)), k), "data gradient": ((m, k), (dyb, wb), n),
                      "weight gradient": ((k, n), (t(xb.T), t(dyb.T)), m)}[
                          call.replace("cached ", "").replace("bf16 weight", "forward")]
    ref = o.gemm("NT", *ref, shape[0], shape[1], kk)
    guard = 8192
    bufs, at = [], {}
    try:
        for v, a in host.items():   # room on both sides, so that a shifted output stays inside the buffer
            room = max(a.size, shape[0] * shape[1]) + 2 * guard
            b = rt.alloc(room * 4)
            bufs.append(b)
            at[v] = b + 4 * guard
        wt = rt.upload(t(wb.T))
        bufs.append(wt)
        out = at[over] + 4 * shift
        x, w, dy = at["x"], at["w"], at["dy"]
        run = {"forward": lambda: rt.matmul_f32(x, w, out, m, k, n),
               "cached forward": lambda: rt.matmul_f32_cached(x, w, 91, out, m, k, n),
               "bf16 weight": lambda: rt.matmul_wt_bf16_f32(x, wt, out, m, k, n),
               "data gradient": lambda: rt.matmul_backward_data_f32(dy, w, out, m, k, n),
               "cached data gradient": lambda: rt.matmul_backward_data_f32_cached(dy, w, 91, out, m, k, n),
               "weight gradient": lambda: rt.matmul_backward_weight_f32(x, dy, out, m, k, n)}[call]
        for _ in range(5):
            for v, a in host.items():
                rt.write(at[v], a)
            run()
            rt.wait_idle()
            ok, relf, maxabs, bound = o.parity(rt.read(out, shape, np.float32), ref, kk)
            assert ok, f"relF={relf:.3e} max|d|={maxabs:.3e} bound={bound:.3e}"
    finally:
        rt.clear_bf16_cache()
        for b in bufs:
            rt.free(b)


# (m, k, n): K slices when the operands are rounded inside the GEMM (forward, data gradient),
# and layers that are converted first
@pytest.mark.parametrize("m,k,n", [(256, 1024, 512), (256, 512, 1024), (2048, 2048, 512)])
def test_f32_calls_under_capture(m, k, n):
    """A handle whose scratch buffers are not grown yet: a captured f32 call allocates nothing,
    and every replay gives the eager result within the parity gate."""
    from hip_rt import Graph, Stream
    h = t0g.GpuRuntime.new(0)
    s = Stream()
    bufs, graphs = [], []
    try:
        rng = np.random.default_rng(m + k + n)
        x = rng.uniform(-0.5, 0.5, (m, k)).astype(np.float32)
        w = rng.uniform(-0.5, 0.5, (k, n)).astype(np.float32)
        dy = rng.uniform(-0.5, 0.5, (m, n)).astype(np.float32)
        xb, wb, dyb = (o.f32_to_bf16_rne(v) for v in (x, w, dy))
        y_ref = o.gemm("NT", xb, np.ascontiguousarray(wb.T), m, n, k)
        dx_ref = o.gemm("NT", dyb, wb, m, k, n)
        ax, aw, ad = (h.upload(v) for v in (x, w, dy))
        out = h.alloc(max(m * n, m * k) * 4)
        bufs += [ax, aw, ad, out]
        h.get_or_create_bf16(5, aw, k * n)
        # loads the kernels; too small to be split or converted
        for warm in (lambda: h.matmul_f32(ax, aw, out, 16, 64, 64), lambda: h.matmul_f32_cached(ax, aw, 6, out, 16, 64, 64),
                     lambda: h.matmul_backward_data_f32(ad, aw, out, 16, 64, 64),
                     lambda: h.matmul_backward_data_f32_cached(ad, aw, 6, out, 16, 64, 64)):
            warm()
        h.wait_idle()
        h.set_stream(s.ptr)
        for shape, ref, kk, call in (((m, n), y_ref, k, lambda: h.matmul_f32(ax, aw, out, m, k, n)),
                                     ((m, n), y_ref, k, lambda: h.matmul_f32_cached(ax, aw, 5, out, m, k, n)),
                                     ((m, k), dx_ref, n, lambda: h.matmul_backward_data_f32(ad, aw, out, m, k, n)),
                                     ((m, k), dx_ref, n, lambda: h.matmul_backward_data_f32_cached(ad, aw, 5, out, m, k, n))):
            before = t0g.device_alloc_count()
            graphs.append(Graph(s, call))
            assert t0g.device_alloc_count() == before
            for _ in range(3):
                h.memset(out, 0xFF, shape[0] * shape[1] * 4)
                graphs[-1].launch(s)
                s.synchronize()
                ok, relf, maxabs, bound = o.parity(h.read(out, shape, np.float32), ref, kk)
                assert ok, f"relF={relf:.3e} max|d|={maxabs:.3e} bound={bound:.3e}"
                h.matmul_f32(ax, aw, out, 16, 64, 64)   # eager work between the replays
                h.wait_idle()
        h.set_stream(None)
    finally:
        for g in graphs:
            g.destroy()
        h.clear_bf16_cache()
        for b in bufs:
            h.free(b)
        h.close()
        s.destroy()
