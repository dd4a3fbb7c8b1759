"""Bit-exact results at both sides of the in-launch handoff's rule (which side
is which: test_dispatch.py): few columns and long rows take it (here also more
launches than the context has counter slots, each against its own result), the
others run as two launches."""
import ctypes

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


@pytest.mark.parametrize("m,n,k,calls", [(8, 512, 4160, 300), (16, 3840, 6160, 3), (16, 3841, 6160, 3), (8, 6144, 8192, 2),
                                         (8, 6160, 8192, 2), (9, 4096, 8192, 2), (5, 1000, 4080, 3), (5, 1000, 4032, 3),
                                         (8, 5120, 6912, 2), (8, 5120, 6848, 2), (12, 4200, 688, 3)])
def test_handoff_rule_bit_exact(ctx, m, n, k, calls):
    print(f"handoff rule m={m} n={n} k={k}", flush=True)
    rng = np.random.default_rng(n)
    wq = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
    sw = rng.uniform(1e-4, 2e-3, n).astype(np.float32)
    drow, dsw = ctx.upload(wq), ctx.upload(sw)
    dw = NH.tile_weights(ctx, drow, n, k)
    ws_bytes = NH.lib().nh_linear_w8a8_workspace_size(m, k)
    ws, outs = ctx.empty(ws_bytes, np.uint8), ctx.empty((calls, m, n), np.uint16)
    rows = [O.to_bf16(O.normal_f32(40 + i, m * k, 0.0, 1.0 + i)).reshape(m, k) for i in range(3)]
    refs = []
    for x in rows:
        _, xq, sx, _ = O.quantize_rows_bf16(x)
        refs.append(linear_w8a8_exact(xq, sx, wq, sw, out_bf16=True))
    dx = [ctx.upload(x) for x in rows]
    for i in range(calls):
        NH.call("nh_linear_w8a8", ctx.handle, dx[i % 3].ptr, NH.BF16, dw.ptr, dsw.ptr, None, m, n, k,
                outs.offset(i * m * n * 2), NH.BF16, ws.ptr, ws_bytes, None, None, None, None)
    ctx.synchronize()
    got = outs.numpy()
    for i in range(calls):  # back to back: a slot's next user may start as soon as its last one has left it
        assert np.array_equal(got[i], refs[i % 3]), f"call {i}"
    timeouts, busy = ctypes.c_uint32(0), ctypes.c_uint32(0)
    NH.call("nh_handoff_status", ctx.handle, ctypes.addressof(timeouts), ctypes.addressof(busy))
    assert (timeouts.value, busy.value) == (0, 0)
