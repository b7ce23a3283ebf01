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
          (130, 70, 64 * 9), (33, 257, 7), (257, 31, 8), (5, 90, 321), (90, 3, 130), (1, 1, 200), (2, 67, 5)]


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
