"""The 256x256 kernels' L2 prefetch (operands of 96 MB or more): bit-identical to the loop
without it, which runs the same tiles when the problem is cut in two along N, and within
the parity gate on sampled rows; every layout, both outputs, K ranges that end in whole
stages (prefetched) and in a tail (not), two to nine tile rows (the prefetch share's cases), split-K."""
import struct

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


def _prefetches(desc):
    flags = struct.unpack_from("<I", t0g.gemm_compile(desc).args(), 40 + 11 * 4)[0]
    return bool(flags & 32)   # T0G_FLAG_PREFETCH: the prefetching loop, if the K range is whole stages


@pytest.mark.parametrize("layout", ["NT", "NN", "TN", "TT"])
@pytest.mark.parametrize("m,n,k,split", [(264, 12032, 4096, 1), (520, 11776, 4096, 1), (1032, 4608, 9088, 1),
                                         (2056, 10240, 4096, 1), (2056, 10240, 4104, 1), (264, 5888, 8192, 4)])
def test_prefetch_changes_no_bit(rt, layout, m, n, k, split):
    assert 2 * k * (m + n) >= 96e6 and 2 * k * (m + n // 2) < 96e6
    rng = np.random.default_rng(m + n + k)
    # a short random row repeated at odd shifts: distinct values everywhere, made quickly
    pool = o.f32_to_bf16_rne(rng.uniform(-0.5, 0.5, 1 << 20).astype(np.float32))
    a_shape = (m, k) if layout in ("NT", "NN") else (k, m)
    b_shape = (n, k) if layout in ("NT", "TT") else (k, n)
    a = np.resize(pool, a_shape[0] * a_shape[1]).reshape(a_shape)
    b = np.resize(pool[::-1][:-13], b_shape[0] * b_shape[1]).reshape(b_shape)
    cfg = t0g.GemmConfig.preset("gfx950_256x256_k64")
    da, db = rt.upload(a), rt.upload(b)
    dc, dh = rt.alloc(m * n * 4), rt.alloc(m * n * 4)
    try:
        for out, esize in ((t0g.F32, 4), (t0g.BF16, 2)):
            kw = dict(transpose=layout, out_dtype=out, config=cfg, split_k=split, lda=a_shape[1], ldb=b_shape[1], ldc=n)
            h = n // 2
            if split == 1:
                assert _prefetches(t0g.gemm_desc(da, db, dc, m, n, k, **kw))
                assert not _prefetches(t0g.gemm_desc(da, db, dc, m, h, k, **kw))
            rt.memset(dc, 0xFF, m * n * esize)
            rt.memset(dh, 0xFF, m * n * esize)
            rt.gemm(da, db, dc, m, n, k, **kw)
            for c0 in (0, h):
                boff = c0 * (k if layout in ("NT", "TT") else 1) * 2
                rt.gemm(da, db + boff, dh + c0 * esize, m, h, k, **kw)
            rt.wait_idle()
            got = rt.read(dc, (m, n), np.uint32 if esize == 4 else np.uint16)
            half = rt.read(dh, (m, n), np.uint32 if esize == 4 else np.uint16)
            assert np.array_equal(got, half), f"{layout} out={out}: prefetch changed the result"
            if out == t0g.F32:
                rows = np.array([0, m // 2, m - 1])
                a_rows = np.ascontiguousarray(a[rows] if layout in ("NT", "NN") else a[:, rows].T)
                b_nk = b if layout in ("NT", "TT") else np.ascontiguousarray(b.T)
                ref = o.gemm("NT", a_rows, b_nk, len(rows), n, k)
                ok, relf, maxabs, bound = o.parity(got.view(np.float32)[rows], ref, k)
                assert ok, f"relF={relf:.3e} max|d|={maxabs:.3e} bound={bound:.3e}"
    finally:
        for x in (da, db, dc, dh):
            rt.free(x)
