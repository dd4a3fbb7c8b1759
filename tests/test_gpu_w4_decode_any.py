"""W4A8 decode of 3..16 bf16 rows whose K the 512-wide streaming unit does not take: its padded forms.  Results are exact,
a non-finite value is reported at its index in the whole input, and a caller's workspace is left alone (a program may pass
one buffer to calls on several streams: these shapes never needed it)."""
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


def setup(ctx, m, n, k, zp, seed):
    rng = np.random.default_rng(seed)
    packed = rng.integers(0, 256, size=(k * n + 1) // 2, dtype=np.uint8)
    x = O.to_bf16(O.normal_f32(seed + 1, m * k)).reshape(m, k)
    need = NH.lib().nh_tiled_int4_weights_bytes(n, k)
    dp, dt = ctx.upload(packed), ctx.empty(need, np.uint8)
    NH.call("nh_tile_weights_int4", ctx.handle, dp.ptr, packed.size, k, n, zp, dt.ptr, need, None)
    return rng, packed, x, dt


# one chunk pair, a K tile less and more one 16-group, groups of 64 chunks less and more one chunk pair, both ends of the
# short and of the long form; one to eight and nine to sixteen rows, two launches of the long form with a remainder of one
# row, of four and of more; one column, part of a tile, several rounds of tiles per workgroup; zero points at both ends; three and four
# rows on both sides of their lines, and as the remainder of eleven
@pytest.mark.parametrize("m,n,k,zp", [(5, 1, 16, 8), (16, 40, 48, 15), (8, 100, 80, 0), (9, 517, 496, 7), (16, 256, 528, 8),
                                      (13, 4130, 1040, 3), (8, 33, 4080, 8), (16, 2048, 4080, 15), (5, 64, 4112, 8),
                                      (8, 517, 8176, 1), (8, 4100, 8192, 8), (9, 300, 8192, 15), (12, 96, 5120, 0),
                                      (15, 130, 6160, 9), (16, 517, 8192, 6), (7, 20000, 144, 8),
                                      (3, 33, 1008, 8), (3, 33, 1024 + 16, 8), (4, 4130, 4080, 3), (3, 8200, 4112, 8),
                                      (4, 8192, 4112, 15), (11, 8200, 4160, 0)])
def test_w4a8_decode_any_k_bit_exact(ctx, m, n, k, zp):
    print(f"w4a8 decode any K m={m} n={n} k={k} zp={zp}", flush=True)
    rng, packed, x, dt = setup(ctx, m, n, k, zp, m * 131 + k)
    bias = rng.standard_normal(n).astype(np.float32)
    scale = 0.0137
    dx, db = ctx.upload(x), ctx.upload(bias)
    ws_bytes = NH.lib().nh_linear_w4a8_workspace_size(m, n, k)
    ws = ctx.empty(ws_bytes, np.uint8)
    ws.fill_bytes(0x5a)
    for out_dtype, np_dtype, b, w in ((NH.BF16, np.uint16, None, ws), (NH.F32, np.float32, bias, ws), (NH.BF16, np.uint16, bias, None)):
        out = ctx.upload(np.full(m * n + 16, 7, np_dtype))
        NH.call("nh_linear_w4a8", ctx.handle, dx.ptr, NH.BF16, dt.ptr, scale, zp, db.ptr if b is not None else None, m, n, k,
                out.ptr, out_dtype, w.ptr if w else None, ws_bytes if w else 0, None, None)
        ctx.synchronize()
        st, ref = O.linear_w4a8(x, packed, n, scale, zp, bias=b, out_bf16=out_dtype == NH.BF16)
        assert st == O.OK
        got = out.numpy()
        assert np.array_equal(got[: m * n].reshape(m, n), ref)
        assert (got[m * n:] == 7).all()
    assert (ws.numpy() == 0x5A).all()


@pytest.mark.parametrize("m,k,bad", [(16, 1040, [(15, 1039)]), (8, 6160, [(7, 6150), (7, 6159)]), (16, 8192, [(12, 3), (9, 8191)]),
                                     (9, 8192, [(8, 5)]), (3, 1040, [(2, 1039)]), (16, 4080, [(3, 4079), (11, 0)])])
def test_w4a8_decode_any_k_reports_the_first_nonfinite(ctx, m, k, bad):
    n = 48
    print(f"w4a8 decode any K nonfinite m={m} k={k}", flush=True)
    _, _, x, dt = setup(ctx, m, n, k, 8, m + k)
    for r, c in bad:
        x[r, c] = 0x7FC0  # NaN
    dx, out = ctx.upload(x), ctx.empty((m, n), np.uint16)
    word = ctx.upload(np.zeros(1, np.uint64))
    NH.call("nh_linear_w4a8", ctx.handle, dx.ptr, NH.BF16, dt.ptr, 0.01, 8, None, m, n, k, out.ptr, NH.BF16, None, 0, word.ptr,
            None)
    st, err = NH.call_status("nh_take_nonfinite", ctx.handle, word.ptr, None)
    assert st == NH.NON_FINITE_INPUT and err.argument == b"input" and err.index == min(r * k + c for r, c in bad)


def test_w4a8_decode_any_k_zero_rows(ctx):
    m, n, k = 9, 40, 1072
    _, packed, x, dt = setup(ctx, m, n, k, 15, 3)
    x[4] = 0
    dx, out = ctx.upload(x), ctx.empty((m, n), np.float32)
    NH.call("nh_linear_w4a8", ctx.handle, dx.ptr, NH.BF16, dt.ptr, 0.01, 15, None, m, n, k, out.ptr, NH.F32, None, 0, None, None)
    ctx.synchronize()
    ref = O.linear_w4a8(x, packed, n, 0.01, 15, out_bf16=False)[1]
    assert not out.numpy()[4].any() and np.array_equal(out.numpy(), ref)
