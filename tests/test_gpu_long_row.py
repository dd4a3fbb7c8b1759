"""The long-row decode unit: one f32 row, or one of more than 8192 values,
quantized inside the GEMV's workgroups.  Codes, scale and outputs equal the
oracle's bit for bit; a non-finite value is reported at its column."""
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


def run(ctx, x, xdt, n, k, out_dtype, bias=None, offset=0, word=None):
    """One call on the row at byte `offset` of a device buffer; returns (out, codes, scale, weights, scales)."""
    rng = np.random.default_rng(n + k)
    wq = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
    sw = rng.uniform(1e-4, 2e-3, n).astype(np.float32)
    drow, dsw = ctx.upload(wq), ctx.upload(sw)
    dw = NH.tile_weights(ctx, drow, n, k)
    dx = ctx.upload(np.concatenate([np.zeros(offset // x.itemsize, x.dtype), x.reshape(-1)]))
    db = ctx.upload(bias) if bias is not None else None
    ws_bytes = NH.lib().nh_linear_w8a8_workspace_size(1, k)
    ws, out = ctx.empty(ws_bytes, np.uint8), ctx.empty(n, np.uint16 if out_dtype == NH.BF16 else np.float32)
    codes, scale = ctx.empty((1, k), np.int8), ctx.empty(1, np.float32)
    NH.call("nh_linear_w8a8", ctx.handle, dx.offset(offset), xdt, dw.ptr, dsw.ptr, db.ptr if db else None, 1, n, k,
            out.ptr, out_dtype, ws.ptr, ws_bytes, codes.ptr, scale.ptr, word.ptr if word else None, None)
    ctx.synchronize()
    return out.numpy(), codes.numpy(), scale.numpy(), wq, sw


# one K tile and a partial one, K tails of 16 and 48, fewer and more K tiles than a ring; one, several and a partial N
# tile; the longest rows the unit holds and the first ones past it; rounds of several workgroups per CU; a row off a
# 16-byte boundary (the two-launch path)
@pytest.mark.parametrize("k,n,f32,offset", [
    (16, 5, True, 0), (80, 16, True, 0), (1072, 130, True, 0), (4096, 4096, True, 0), (4112, 517, True, 0),
    (8256, 33, False, 0), (9648, 1000, False, 0), (21504, 300, True, 0), (22528, 17, True, 0), (22544, 17, True, 0),
    (45056, 16, False, 0), (45072, 16, False, 0), (8192, 4130, True, 0), (4096, 4130, True, 0), (4096, 96, True, 4)])
def test_long_row_bit_exact(ctx, k, n, f32, offset):
    print(f"long row k={k} n={n} f32={f32} offset={offset}", flush=True)
    xf = O.normal_f32(k, k).reshape(1, k)
    x = xf if f32 else O.to_bf16(xf)
    st, xq, sx, _ = (O.quantize_rows_f32 if f32 else O.quantize_rows_bf16)(x)
    assert st == O.OK
    bias = O.normal_f32(3, n)
    for out_dtype, b in ((NH.BF16, bias), (NH.F32, None)):
        out, codes, scale, wq, sw = run(ctx, x, NH.F32 if f32 else NH.BF16, n, k, out_dtype, b, offset)
        assert np.array_equal(codes, xq) and np.array_equal(scale, sx)
        ref = linear_w8a8_exact(xq, sx, wq, sw, bias=b, out_bf16=out_dtype == NH.BF16)
        assert np.array_equal(out, ref[0])


@pytest.mark.parametrize("f32", [True, False])
def test_long_row_zero_and_nonfinite(ctx, f32):
    k, n = 8320, 40
    x = np.zeros((1, k), np.float32 if f32 else np.uint16)
    out, codes, scale, _, _ = run(ctx, x, NH.F32 if f32 else NH.BF16, n, k, NH.F32)
    assert not codes.any() and scale[0] == 0 and not out.any()
    xf = O.normal_f32(5, k).reshape(1, k)
    xf[0, 8301], xf[0, 4003] = np.nan, -np.inf
    word = ctx.upload(np.zeros(1, np.uint64))
    run(ctx, xf if f32 else O.to_bf16(xf), NH.F32 if f32 else NH.BF16, n, k, NH.F32, word=word)
    st, err = NH.call_status("nh_take_nonfinite", ctx.handle, word.ptr, None)
    assert st == NH.NON_FINITE_INPUT and err.argument == b"input" and err.index == 4003 and err.value == -np.inf


def test_long_row_still_asks_for_its_workspace(ctx):
    k, n = 8320, 16
    d = ctx.empty(n * k + 64, np.uint8)
    st, err = NH.call_status("nh_linear_w8a8", ctx.handle, d.ptr, NH.F32, d.ptr, d.ptr, None, 1, n, k, d.ptr, NH.F32,
                             None, 0, None, None, None, None)
    assert st == NH.LENGTH_MISMATCH and err.argument == b"workspace"


@pytest.mark.parametrize("k", [4096, 21504])
def test_long_row_overwritten_by_its_own_outputs(ctx, k):
    """A square f32 layer in place (out = x), and codes written over the row: every value is read before any is written."""
    print(f"long row in place k={k}", flush=True)
    n = k if k == 4096 else 512
    rng = np.random.default_rng(k)
    x = O.normal_f32(k + 1, k).reshape(1, k)
    _, xq, sx, _ = O.quantize_rows_f32(x)
    wq = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
    sw = rng.uniform(1e-4, 2e-3, n).astype(np.float32)
    drow, dsw = ctx.upload(wq), ctx.upload(sw)
    dw = NH.tile_weights(ctx, drow, n, k)
    ref = linear_w8a8_exact(xq, sx, wq, sw)[0]
    ws_bytes = NH.lib().nh_linear_w8a8_workspace_size(1, k)
    ws, out = ctx.empty(ws_bytes, np.uint8), ctx.empty(n, np.float32)
    for codes in (False, True):
        dx = ctx.upload(x)
        NH.call("nh_linear_w8a8", ctx.handle, dx.ptr, NH.F32, dw.ptr, dsw.ptr, None, 1, n, k, out.ptr if codes else dx.ptr,
                NH.F32, ws.ptr, ws_bytes, dx.ptr if codes else None, None, None, None)
        ctx.synchronize()
        got = dx.numpy().reshape(-1)
        if codes:
            assert np.array_equal(got.view(np.int8)[:k], xq[0])
        assert np.array_equal(out.numpy() if codes else got[:n], ref)
