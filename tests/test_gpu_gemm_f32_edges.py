"""The f64 matrix-core GEMM's staging: K around its 64-k chunks and the six
chunks its loads run ahead, tiles with few rows (chain waves without any) and
few columns, aligned and unaligned lhs rows.  Bit-identical to the host order."""
import numpy as np
import pytest

import nemotron_hip as NH
import oracle_ctypes as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = NH.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("k", [1, 2, 8, 60, 64, 65, 68, 127, 128, 129, 132, 192, 256, 384, 388, 448, 453, 776])
@pytest.mark.parametrize("m,n", [(1, 16), (4, 17), (5, 1), (16, 60), (35, 130)])
def test_gemm_f32_chunk_edges(ctx, m, n, k):
    print(f"gemm_f32 m={m} k={k} n={n}", flush=True)
    lhs, rhs = O.normal_f32(k, m * k), O.normal_f32(k + 1, k * n, 0.0, 0.02)
    rhs[-1] = np.float32(3e38)  # the last k counts
    _, ref, _ = O.gemm_f32(lhs, rhs, m, k, n)
    dr, out = ctx.upload(rhs), ctx.empty(m * n + 8, np.float32)
    for shift in (0, 1):  # shift 1: lhs rows off a 16-byte boundary
        dl = ctx.upload(np.concatenate([np.full(shift, np.nan, np.float32), lhs]))
        out.copy_from(np.full(m * n + 8, 7, np.float32))
        NH.call("nh_gemm_f32", ctx.handle, dl.offset(4 * shift), lhs.size, dr.ptr, rhs.size, m, k, n, out.ptr, m * n,
                None)
        ctx.synchronize()
        got = out.numpy()
        assert np.array_equal(got[: m * n].view(np.uint32), ref.view(np.uint32))
        assert (got[m * n:] == 7).all()
