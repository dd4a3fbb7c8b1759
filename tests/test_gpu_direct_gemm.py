"""The register-direct GEMM (gemm_direct.hip) and the LDS-tiled ones at the edges of their tiles.

Every result is exact (int32 sums, the epilogue's fixed rounding order), so
outputs equal the exact-integer reference bit for bit, and those of the
row-major entry point, whose kernels share no code with it.
"""
import numpy as np
import pytest

import nemotron_hip as NH
import oracle_ctypes as O
from exact_int import linear_w8a8_exact

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = NH.Context(0)
    yield c
    c.close()


# one row tile, one to eight tiles per group, several groups (balanced and not); N not a multiple of 16, 32 or 64, and
# of 4; one K tile, fewer K tiles than waves, K tails; column blocks not a multiple of the 8 XCDs
SHAPES = [(1, 16, 16), (17, 1000, 1024), (33, 4099, 208), (64, 130, 4112), (65, 2688, 2688), (100, 2052, 320),
          (113, 333, 4096), (128, 517, 1040), (129, 1027, 4096), (260, 2690, 1856), (400, 70, 8192), (37, 11008, 4096)]


# shapes whose time model takes the LDS tiles (256, 128 and 64 rows), with ragged edges both ways and rows of odd length
RAGGED = [(1000, 4097, 1024), (2047, 4099, 256), (613, 4099, 2688), (600, 1027, 512), (1025, 8193, 128)]


@pytest.mark.parametrize("m,n,k", SHAPES + RAGGED)
def test_direct_gemm_bit_exact(ctx, m, n, k):
    print(f"direct gemm m={m} n={n} k={k}", flush=True)
    rng = np.random.default_rng(m * 7 + n)
    xq = rng.integers(-127, 128, size=(m, k), dtype=np.int8)
    wq = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
    sx = rng.uniform(1e-3, 2e-2, m).astype(np.float32)
    sw = rng.uniform(1e-4, 2e-3, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    dx, dsx, dsw, db = ctx.upload(xq), ctx.upload(sx), ctx.upload(sw), ctx.upload(bias)
    dxt = NH.tile_weights(ctx, dx, m, k)
    drow = ctx.upload(wq)
    dw = NH.tile_weights(ctx, drow, n, k)
    # 0: aligned rows; 1 element: rows that never start on a vector store's boundary
    for out_dtype, np_dtype, shift in ((NH.BF16, np.uint16, 0), (NH.F32, np.float32, 1), (NH.BF16, np.uint16, 1)):
        for b in (None, bias):
            ref = linear_w8a8_exact(xq, sx, wq, sw, bias=b, out_bf16=out_dtype == NH.BF16)
            guard = ctx.upload(np.full(m * n + 16, 7, dtype=np_dtype))
            row_major = ctx.empty((m, n), np_dtype)
            args = (db.ptr if b is not None else None, m, n, k)
            NH.call("nh_gemm_w8a8_ta", ctx.handle, dxt.ptr, dsx.ptr, dw.ptr, dsw.ptr, *args,
                    guard.offset(shift * guard.dtype.itemsize), out_dtype, None)
            NH.call("nh_gemm_w8a8", ctx.handle, dx.ptr, dsx.ptr, dw.ptr, dsw.ptr, *args, row_major.ptr, out_dtype, None)
            ctx.synchronize()
            got = guard.numpy()
            assert np.array_equal(got[shift:shift + m * n].reshape(m, n), ref)
            assert (got[:shift] == 7).all() and (got[shift + m * n:] == 7).all()  # nothing past the matrix
            assert np.array_equal(row_major.numpy(), ref)


# rows past the fused decode unit, f32 rows of any count, K past it; more rows than columns (the A tiles then go to the
# linear workspace); row groups of 64 and of 128; zero points at both ends
@pytest.mark.parametrize("m,n,k,zp,f32", [(17, 1000, 1024, 8, False), (24, 4096, 8192, 0, False), (1, 517, 4096, 15, True),
                                          (16, 2048, 208, 7, True), (3, 300, 8208, 8, False), (70, 33, 4096, 5, False),
                                          (129, 2050, 1040, 8, True), (300, 4096, 512, 3, False), (100, 16384, 256, 9, False)])
def test_direct_w4a8_bit_exact(ctx, m, n, k, zp, f32):
    print(f"direct w4a8 m={m} n={n} k={k} zp={zp} f32={f32}", flush=True)
    rng = np.random.default_rng(m + n)
    codes = rng.integers(0, 16, size=(k, n), dtype=np.uint8)
    flat = np.append(codes.reshape(-1), 0)[: (k * n + 1) // 2 * 2]
    packed = (flat[0::2] | (flat[1::2] << 4)).astype(np.uint8)
    scale = 0.0137
    xf = O.normal_f32(3 + m, m * k).reshape(m, k)
    x = xf if f32 else O.to_bf16(xf)
    st, xq, sx, _ = (O.quantize_rows_f32 if f32 else O.quantize_rows_bf16)(x)
    assert st == O.OK
    w = (codes.astype(np.int16) - zp).astype(np.int8).T.copy()
    bias = rng.standard_normal(n).astype(np.float32)
    need = NH.lib().nh_tiled_int4_weights_bytes(n, k)
    dp, dt = ctx.upload(packed), ctx.empty(need, np.uint8)
    NH.call("nh_tile_weights_int4", ctx.handle, dp.ptr, packed.size, k, n, zp, dt.ptr, need, None)
    ws_bytes = NH.lib().nh_linear_w4a8_workspace_size(m, n, k)
    ws, dx, db = ctx.empty(ws_bytes, np.uint8), ctx.upload(x), ctx.upload(bias)
    ws.fill_bytes(0x5a)  # rows and columns past the matrix hold anything
    for out_dtype, b in ((NH.BF16, None), (NH.F32, bias)):
        out = ctx.empty((m, n), np.uint16 if out_dtype == NH.BF16 else np.float32)
        NH.call("nh_linear_w4a8", ctx.handle, dx.ptr, NH.F32 if f32 else NH.BF16, dt.ptr, scale, zp,
                db.ptr if b is not None else None, m, n, k, out.ptr, out_dtype, ws.ptr, ws_bytes, None, None)
        ctx.synchronize()
        ref = linear_w8a8_exact(xq, sx, w, np.full(n, scale, np.float32), bias=b, out_bf16=out_dtype == NH.BF16)
        assert np.array_equal(out.numpy(), ref)
