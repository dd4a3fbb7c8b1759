"""Which kernels the entry points launch, and the rules behind that (no GPU: dispatch.py)."""
import pytest

import nemotron_hip as NH
from dispatch import Recorder


@pytest.fixture(scope="module")
def rec():
    r = Recorder()
    yield r
    r.close()


def test_recorder_names_the_launches_of_a_call(rec):
    assert rec.linear(1, 4096, 4096) == ["linear_decode_w8a8_m1"]
    assert rec.linear(8, 4096, 4096) == ["linear_decode_stream_m8"]
    assert rec.linear(2048, 21504, 4096) == ["quantize_tiles", "gemm_w8a8_p256x224"]
    with pytest.raises(NH.NhStatusError):  # refused calls launch nothing
        rec.linear(4, 100, 72)
    assert rec.linear(1, 16, 16) == ["linear_decode_w8a8_m1"]


# A single row's workgroups each read the whole row, so an output laid over it would be written while others still read:
# such calls keep the quantizer launch, which has read the row before anything is written.
@pytest.mark.parametrize("x_dtype,k", [(NH.F32, 4096), (NH.F32, 64), (NH.F32, 21504), (NH.BF16, 12288)])
def test_single_row_under_its_own_outputs_takes_two_launches(rec, x_dtype, k):
    X, row = 1 << 40, k * (2 if x_dtype == NH.BF16 else 4)
    two = ["quantize_rows_long" if row > 16384 else "quantize_rows_i8", "gemv_w8a8_xt"]
    n = 48
    assert rec.linear(1, n, k, x_dtype) == ["linear_decode_long"]
    for out_dtype, size in ((NH.F32, 4 * n), (NH.BF16, 2 * n)):
        for out in (X, X + row - 16, X - size + 16):  # on the row, over its end, over its start
            assert rec.linear(1, n, k, x_dtype, out_dtype, out=out) == two
        for out in (X + row, X - size):  # beside it
            assert rec.linear(1, n, k, x_dtype, out_dtype, out=out) == ["linear_decode_long"]
    assert rec.linear(1, n, k, x_dtype, xq_out=X) == two
    assert rec.linear(1, n, k, x_dtype, xq_out=X + row - 16) == two
    assert rec.linear(1, n, k, x_dtype, xq_out=X + row) == ["linear_decode_long"]
    assert rec.linear(1, n, k, x_dtype, sx_out=X + row - 4) == two
    assert rec.linear(1, n, k, x_dtype, sx_out=X + row) == ["linear_decode_long"]
