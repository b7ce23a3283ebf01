"""The deep-ring kernels whose DMA goes out from four waves of their own: bit-identical
to the ordinary kernels of the tile (more workgroups than CUs, the same K order), which run the
same columns as part of a wider product; every layout, both outputs, one stage, fewer stages
than the ring holds, K tails, ragged tiles, split planes with a short last slice."""
import numpy as np
import pytest

import oracle as o
import t0g

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    r = t0g.GpuRuntime.new(0)
    yield r
    r.close()


@pytest.mark.parametrize("tile", [128, 64])
@pytest.mark.parametrize("layout", ["NT", "NN", "TN", "TT"])
@pytest.mark.parametrize("m,k,split", [(200, 8, 1), (136, 64, 1), (264, 136, 1), (128, 192, 1), (256, 264, 1),
                                       (392, 1000, 1), (200, 1096, 4)])
def test_deep_kernels_equal_the_ordinary_one(rt, tile, layout, m, k, split):
    wide, h = 33024, 264          # more than 256 tile columns against a few
    rng = np.random.default_rng(m + k)
    pool = o.f32_to_bf16_rne(rng.uniform(-0.5, 0.5, 1 << 20).astype(np.float32))
    a_shape = (m, k) if layout in ("NT", "NN") else (k, m)
    b_shape = (wide, k) if layout in ("NT", "TT") else (k, wide)
    a = np.resize(pool, a_shape[0] * a_shape[1]).reshape(a_shape)
    b = np.resize(pool[::-1][:-13], b_shape[0] * b_shape[1]).reshape(b_shape)
    cfg = t0g.GemmConfig.preset(f"gfx950_{tile}x{tile}_k64")
    c0 = 264 * 5
    da, db = rt.upload(a), rt.upload(b)
    dc, dh = rt.alloc(m * wide * 4), rt.alloc(m * h * 4)
    try:
        for out, esize in ((t0g.F32, 4), (t0g.BF16, 2)):
            kw = dict(transpose=layout, out_dtype=out, config=cfg, split_k=split, lda=a_shape[1], ldb=b_shape[1])
            boff = c0 * (k if layout in ("NT", "TT") else 1) * 2
            full = t0g.gemm_desc(da, db, dc, m, wide, k, ldc=wide, **kw)
            part = t0g.gemm_desc(da, db + boff, dh, m, h, k, ldc=h, **kw)
            prefix = f"t0g_gemm_{tile}x{tile}_k64_{layout.lower()}_"
            f32 = out == t0g.F32 or split > 1   # split planes are fp32
            assert t0g.gemm_kernel_name(full) == prefix + ("f32" if f32 else "bf16")
            assert t0g.gemm_kernel_name(part) == prefix + ("f32_d" if split > 1 else "f32_df" if f32 else "bf16_d")
            rt.memset(dc, 0xFF, m * wide * esize)
            rt.memset(dh, 0xFF, m * h * esize)
            rt.gemm_desc(full)
            rt.gemm_desc(part)
            rt.wait_idle()
            dt = np.uint32 if esize == 4 else np.uint16
            got, ref = rt.read(dh, (m, h), dt), rt.read(dc, (m, wide), dt)[:, c0:c0 + h]
            assert np.array_equal(got, ref), f"{layout} out={out}: {np.count_nonzero(got != ref)} values differ"
            if out == t0g.F32:
                b_nk = np.ascontiguousarray(b[c0:c0 + h] if layout in ("NT", "TT") else b[:, c0:c0 + h].T)
                a_mk = a if layout in ("NT", "NN") else np.ascontiguousarray(a.T)
                exact = o.gemm("NT", a_mk, b_nk, m, h, k)
                ok, relf, maxabs, bound = o.parity(got.view(np.float32), exact, k)
                assert ok, f"relF={relf:.3e} max|d|={maxabs:.3e} bound={bound:.3e}"
    finally:
        for x in (da, db, dc, dh):
            rt.free(x)


@pytest.mark.parametrize("k,out,suffix", [(320, t0g.F32, "_df"), (320, t0g.BF16, "_d"), (321, t0g.F32, "_u")])
def test_loaded_with_the_configs_workgroup(rt, k, out, suffix):
    """A kernel with operand waves, loaded from the code object with the 256 threads of its
    tile's config: the same workgroups run, those waves included, and the same bits come out."""
    m, n = 136, 200
    rng = np.random.default_rng(k)
    a = o.f32_to_bf16_rne(rng.uniform(-0.5, 0.5, m * k).astype(np.float32))
    b = o.f32_to_bf16_rne(rng.uniform(-0.5, 0.5, n * k).astype(np.float32))
    da, db = rt.upload(a), rt.upload(b)
    dc, dr = rt.alloc(m * n * 4), rt.alloc(m * n * 4)
    try:
        ck = t0g.gemm_compile(t0g.gemm_desc(da, db, dc, m, n, k, out_dtype=out))
        name, tiles = ck.name.decode(), ck.grid[0] // ck.workgroup_size
        assert name.endswith(suffix) and ck.workgroup_size == 512
        kern = rt.load_kernel(ck.elf(), name, (256, 1, 1), ck.lds_size)
        dt = np.uint32 if out == t0g.F32 else np.uint16
        for buf in (dc, dr):
            rt.memset(buf, 0xFF, m * n * dt().itemsize)
        rt.dispatch(kern, (tiles * 256, 1, 1), ck.args())
        rt.gemm(da, db, dr, m, n, k, out_dtype=out)
        rt.wait_idle()
        assert np.array_equal(rt.read(dc, (m, n), dt), rt.read(dr, (m, n), dt))
    finally:
        for x in (da, db, dc, dr):
            rt.free(x)
