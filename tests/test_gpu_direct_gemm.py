"""The register-direct GEMM (gemm_direct.hip) and the LDS-tiled ones at the edges of their tiles.

Every result is exact (int32 sums, the epilogue's fixed rounding order), so
outputs equal the exact-integer reference bit for bit, and those of the
row-major entry point, whose kernels share no code with it.  Each shape names
the kernels that it is there for; the dispatch is asked first.
"""
import numpy as np
import pytest

import nemotron_hip as NH
import oracle_ctypes as O
from dispatch import Recorder
from exact_int import linear_w8a8_exact

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = NH.Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def rec():
    r = Recorder()
    yield r
    r.close()


D16, D32, D64 = (["gemm_w8a8_direct%d" % c] for c in (16, 32, 64))
T256, T128, T64128, T6464 = (["gemm_w8a8_ta_" + t] for t in ("256x128", "128x128", "64x128", "64x64"))
# one row tile, one to eight tiles per group, several groups (balanced and not); N not a multiple of 16, 32 or 64, and
# of 4; one K tile, fewer K tiles than waves, K tails; column blocks not a multiple of the 8 XCDs
SHAPES = [(1, 16, 16, D16), (17, 1000, 1024, D16), (64, 130, 4112, D16), (65, 2688, 2688, D16), (113, 333, 4096, D16),
          (129, 1027, 4096, D16), (400, 70, 8192, D16), (22, 18, 256, D16), (37, 122, 1040, D16), (188, 124, 2064, D16),
          (260, 2498, 1856, D32), (120, 262, 2064, D32), (17, 5044, 1040, D32), (237, 139, 2064, D32), (372, 191, 2064, D32),
          (37, 11008, 4096, D64), (17, 8486, 2064, D64), (20, 10395, 2064, D64), (136, 4119, 2064, D64), (153, 4277, 2064, D64)]
# the LDS tiles with ragged edges both ways and rows of odd length, the persistent 256 x 224 kernel with few rows in its
# tile, and the launch split in whole rounds of 256 x 128 tiles and 128 x 128 ones for the columns after them, which are
# stored at the whole matrix's row distance
RAGGED = [(33, 4099, 208, T6464), (100, 2052, 320, T6464), (128, 517, 1040, T6464), (600, 1027, 512, T6464), (2047, 4099, 256, T6464),
          (1025, 8193, 128, T6464), (27, 35, 16, T6464), (77, 15091, 16, T64128), (1000, 2003, 192, T64128),
          (613, 4099, 2688, T128), (74, 16813, 528, T128), (1000, 4097, 1024, T256), (460, 12679, 16, T256),
          (668, 18232, 80, ["gemm_w8a8_p256x224"]), (899, 19912, 144, T256 + T128), (1225, 14755, 144, T256 + T128)]


@pytest.mark.parametrize("m,n,k,kernels", SHAPES + RAGGED)
def test_direct_gemm_bit_exact(ctx, rec, m, n, k, kernels):
    print(f"direct gemm m={m} n={n} k={k} {kernels}", flush=True)
    assert rec.gemm_ta(m, n, k) == kernels
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


W16, W32, W64, W128 = (["gemm_w4a8_direct%d" % c] for c in (16, 32, 64, 128))
EXPAND = ["expand_int4_tiles"]
# rows past the fused decode unit, f32 rows of any count, K past it; more rows than columns (the A tiles then go to the
# linear workspace); one row group and several of each width; zero points at both ends; and the weights expanded to int8
# tiles, for a GEMV, one or two LDS-tiled GEMMs and the single-row unit; bf16 rows off a 16-byte boundary with K tails
@pytest.mark.parametrize("m,n,k,zp,f32,offset,kernels", [
    (17, 1000, 1024, 8, False, 0, W16), (24, 4096, 8192, 0, False, 0, W16), (1, 517, 4096, 15, True, 0, W16),
    (16, 2048, 208, 7, True, 0, W16), (3, 300, 8208, 8, False, 0, W16), (70, 33, 4096, 5, False, 0, W16),
    (132, 35, 192, 15, False, 0, W16), (129, 2050, 1040, 8, True, 0, W32), (3, 6167, 16, 0, True, 0, W32),
    (154, 3302, 256, 8, False, 0, W32), (300, 4096, 512, 3, False, 0, W64), (100, 16384, 256, 9, False, 0, W64),
    (1, 8758, 48, 15, True, 0, W64), (206, 6118, 256, 0, False, 0, W64), (6, 19705, 128, 15, True, 0, W128),
    (119, 13821, 192, 8, False, 0, W128), (64, 16390, 3984, 0, False, 0, W128), (2, 16855, 64, 8, True, 0, EXPAND + ["gemv_w8a8_xt"]),
    (77, 44, 16, 15, False, 0, EXPAND + T6464), (165, 7371, 16, 8, False, 0, EXPAND + T64128),
    (275, 6558, 528, 3, False, 0, EXPAND + T128), (923, 19854, 192, 8, False, 0, EXPAND + T256 + T128),
    (1, 128, 15312, 8, True, 0, EXPAND + ["linear_decode_long"]), (16, 100, 208, 15, False, 2, W16), (5, 40, 1040, 7, False, 8, W16)])
def test_direct_w4a8_bit_exact(ctx, rec, m, n, k, zp, f32, offset, kernels):
    print(f"direct w4a8 m={m} n={n} k={k} zp={zp} f32={f32} offset={offset}", flush=True)
    took = [q for q in rec.w4a8(m, n, k, NH.F32 if f32 else NH.BF16, x=(1 << 40) + offset) if not q.startswith("quantize")]
    assert took == kernels
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
    ws, db = ctx.empty(ws_bytes, np.uint8), ctx.upload(bias)
    dx = ctx.upload(np.concatenate([np.zeros(offset // x.itemsize, x.dtype), x.reshape(-1)]))
    ws.fill_bytes(0x5a)  # rows and columns past the matrix hold anything
    for out_dtype, b in ((NH.BF16, None), (NH.F32, bias)):
        out = ctx.empty((m, n), np.uint16 if out_dtype == NH.BF16 else np.float32)
        NH.call("nh_linear_w4a8", ctx.handle, dx.offset(offset), NH.F32 if f32 else NH.BF16, dt.ptr, scale, zp,
                db.ptr if b is not None else None, m, n, k, out.ptr, out_dtype, ws.ptr, ws_bytes, None, None)
        ctx.synchronize()
        ref = linear_w8a8_exact(xq, sx, w, np.full(n, scale, np.float32), bias=b, out_bf16=out_dtype == NH.BF16)
        assert np.array_equal(out.numpy(), ref)
