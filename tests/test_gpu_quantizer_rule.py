"""The row quantizer of a GEMM's A tiles at both sides of each line of its rule (rows, row length): codes, scales and outputs
equal the oracle's bit for bit, also from rows off a 16-byte boundary, whose codes past K the tiles do not get."""
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


@pytest.mark.parametrize("m,k,f32,offset,kernel", [
    (17, 16, False, 0, "tiles"), (45, 528, False, 0, "rows_i8"), (33, 256, True, 0, "tiles"), (255, 1024, False, 0, "rows_i8"),
    (256, 1008, False, 0, "tiles"), (511, 592, True, 0, "rows_i8"), (512, 592, True, 0, "tiles"), (600, 2560, False, 0, "tiles"),
    (600, 2576, False, 0, "rows_i8"), (1024, 2576, False, 0, "tiles"), (40, 4112, False, 0, "rows_i8"), (256, 8208, False, 0, "rows_long"),
    (257, 8208, False, 0, "rows_r11"), (257, 11280, True, 0, "rows_i8"), (257, 18448, True, 0, "rows_long"),
    (70, 208, True, 4, "rows_i8"), (70, 208, False, 2, "rows_i8")])
def test_quantizer_rule_bit_exact(ctx, m, k, f32, offset, kernel):
    n = 48
    print(f"quantizer rule m={m} k={k} f32={f32} offset={offset}", flush=True)
    rec = Recorder()
    xdt = NH.F32 if f32 else NH.BF16
    assert rec.linear(m, n, k, xdt, x=(1 << 40) + offset)[0] == "quantize_" + kernel
    rec.close()
    rng = np.random.default_rng(m + k)
    xf = O.normal_f32(m + k, m * k).reshape(m, k)
    x = xf if f32 else O.to_bf16(xf)
    st, xq, sx, _ = (O.quantize_rows_f32 if f32 else O.quantize_rows_bf16)(x)
    assert st == O.OK
    wq = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
    sw = rng.uniform(1e-4, 2e-3, n).astype(np.float32)
    drow, dsw = ctx.upload(wq), ctx.upload(sw)
    dw = NH.tile_weights(ctx, drow, n, k)
    dx = ctx.upload(np.concatenate([np.zeros(offset // x.itemsize, x.dtype), x.reshape(-1)]))
    ws_bytes = NH.lib().nh_linear_w8a8_workspace_size(m, k)
    ws, out = ctx.empty(ws_bytes, np.uint8), ctx.empty((m, n), np.float32)
    ws.fill_bytes(0x5a)
    codes, scale = ctx.empty((m, k), np.int8), ctx.empty(m, np.float32)
    NH.call("nh_linear_w8a8", ctx.handle, dx.offset(offset), xdt, dw.ptr, dsw.ptr, None, m, n, k, out.ptr, NH.F32, ws.ptr, ws_bytes,
            codes.ptr, scale.ptr, None, None)
    ctx.synchronize()
    assert np.array_equal(codes.numpy(), xq) and np.array_equal(scale.numpy(), sx)
    assert np.array_equal(out.numpy(), linear_w8a8_exact(xq, sx, wq, sw))
