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
