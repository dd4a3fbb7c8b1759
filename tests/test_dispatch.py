"""Which kernels the entry points launch, and the rules behind that (no GPU: dispatch.py)."""
import csv
import os
import re

import pytest

import dispatch as D
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


# W4A8 of 3..4 rows, alone or left over from a long-K group of eight: streamed where K is not short, or the output wide.
@pytest.mark.parametrize("m,n,k,kernels", [
    (3, 64, 1008, ["row4"]), (4, 64, 1040, ["stream_w4_any_m8"]), (2, 64, 1040, ["row2"]), (3, 8192, 4112, ["row4"]),
    (4, 8193, 4112, ["stream_w4_long_m8"]), (2, 30000, 4112, ["row2"]), (11, 8208, 4112, ["stream_w4_long_m8"] * 2),
    (12, 256, 8192, ["stream_w4_long_m8", "row4"]), (9, 30000, 8192, ["stream_w4_long_m8", "m1"])])
def test_w4a8_few_rows(rec, m, n, k, kernels):
    assert [q.replace("linear_decode_", "").replace("w4a8_", "") for q in rec.w4a8(m, n, k)] == kernels


# W4A8 decode never writes the workspace, given or not: a buffer that calls on several streams share is not raced on.
@pytest.mark.parametrize("m", range(1, 17))
@pytest.mark.parametrize("k", [16, 288, 512, 1040, 4080, 4096, 4112, 5120, 8176, 8192])
def test_w4a8_decode_ignores_its_workspace(rec, m, k):
    for n in (5, 256, 4096, 300000):
        given, none = rec.w4a8(m, n, k), rec.w4a8(m, n, k, workspace=False)
        assert given == none and all(name.startswith("linear_decode") for name in given)
        # and the weights are streamed once, or once per 8 rows of K > 4096, where a workgroup's run of tiles fits
        if m > 2 and n < 262144:
            assert len(given) <= (1 if k <= 4096 else (m + 7) // 8)


# MoE experts: a slot per (expert, part); fewer slots than experts where the workgroups search for the experts with routes.
# Not where the slots are fewer than the CUs, or a few of a round's are live.
@pytest.mark.parametrize("experts,routes,parts,slots", [(16, 12, 8, 16), (136, 1, 8, 1), (30, 1, 8, 30), (128, 126, 2, 126), (127, 126, 2, 127),
                                                        (128, 48, 4, 48), (128, 3072, 2, 128), (184, 125, 2, 125),
                                                        (512, 300, 2, 300), (1024, 48, 4, 48), (1024, 180, 2, 180),
                                                        (1024, 1428, 2, 1024), (1025, 500, 2, 1025), (4000, 380, 2, 380)])
def test_expert_slots(rec, experts, routes, parts, slots):
    (name, gx, gy), = rec.launches("nh_moe_grouped_gemm_w8a8", 1 << 40, 2 << 40, 0, 1, 3 << 40, 4 << 40, routes, routes, experts,
                                   5 << 40, 6 << 40, 512, 1024, 0, 7 << 40, None)
    assert (name, gx, gy) == ("moe_expert_gemm", parts, slots)


# The GEMM choice against the times of every candidate kernel (us, one MI355X): weights not in any cache, and one matrix
# called over and over.  The "check" shapes took no part in the fit.  The bounds on the mean excess are twice what it is
# (0.8%, 0.9%, 1.7%, 2.1%), those on the worst what it is (1.37, 1.26, 1.47, 1.51) and the times' own noise of 3%.
def choice_table(name):
    with open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "profiles", name)) as f:
        return list(csv.DictReader(f))


@pytest.mark.parametrize("part,mean,worst", [("fit", 1.016, 1.41), ("check", 1.018, 1.30), ("cached fit", 1.034, 1.51),
                                             ("cached check", 1.042, 1.56)])
def test_gemm_choice_is_near_the_best(rec, part, mean, worst):
    excess = []
    for r in choice_table("gemm_choice.csv"):
        if r["part"] != part:
            continue
        times = {k: float(v) for k, v in r.items() if k.startswith("gemm") and v}
        took = rec.gemm_ta(int(r["m"]), int(r["n"]), int(r["k"]), NH.F32 if r["out"] == "f32" else NH.BF16)
        excess.append(times[took[0]] / min(times.values()))
    assert len(excess) >= 300
    assert sum(excess) / len(excess) < mean and max(excess) < worst


# A column block's row groups are on one XCD, so 20 blocks of 11 groups are 33 workgroups on some XCDs of 32 CUs: two
# rounds.  (16 blocks are one.)
@pytest.mark.parametrize("m,n,k,kernel", [(1309, 640, 2048, "gemm_w8a8_ta_64x64"), (1429, 576, 2592, "gemm_w8a8_ta_64x64"),
                                          (1309, 512, 2048, "gemm_w8a8_direct32")])
def test_gemm_choice_counts_the_rounds_of_an_xcd(rec, m, n, k, kernel):
    (name, gx, _), = rec.launches("nh_gemm_w8a8_ta", D.X, D.S, D.W, D.S2, None, m, n, k, D.OUT, NH.BF16, None)
    assert name == kernel and gx <= D.CUS


def test_w4a8_choice_is_near_the_best(rec):
    excess = []
    for r in choice_table("w4a8_choice.csv"):
        times = {k: float(v) for k, v in r.items() if k.startswith(("gemm", "expand")) and v}
        took = rec.w4a8(int(r["m"]), int(r["n"]), int(r["k"]), NH.F32 if r["x"] == "f32" else NH.BF16)
        excess.append(next(times[k] for k in took if k in times) / min(times.values()))
    assert len(excess) >= 700
    assert sum(excess) / len(excess) < 1.015 and max(excess) < 1.34


# The row quantizer of a GEMM's A tiles, against the times of a call with each (its 256-column product included).
def test_quantizer_choice_is_near_the_best(rec):
    excess = []
    for r in choice_table("quantizer_choice.csv"):
        # the forms that the dispatch has for the shape: a wave per row is for gathered rows, 11 chunks per thread past 1024
        times = {k: float(v) for k, v in r.items() if k.startswith("quantize") and v and k != "quantize_rows_wave"}
        took = rec.linear(int(r["m"]), 256, int(r["k"]), NH.F32 if r["x"] == "f32" else NH.BF16)[0]
        excess.append(times[took] / min(times.values()))
    assert len(excess) == 700
    assert sum(1 for e in excess if e > 1.03) <= 25 and sum(excess) / len(excess) < 1.004


# The handoff launch, both clauses of its rule at their edges: the first K of 64 K tiles and the last of 63, the last columns
# whose workgroups all have a CU beside the rows'; the weights per CU, the row count and the columns of the second.
@pytest.mark.parametrize("m,n,k,handoff", [(8, 512, 4048, True), (8, 512, 4032, False), (5, 1000, 4080, True), (12, 4200, 688, False),
                                           (16, 3840, 6160, True), (16, 3841, 6160, False), (8, 4096, 8192, True),
                                           (9, 4096, 8192, False), (8, 4096, 8064, True), (8, 4096, 7680, False),
                                           (8, 5120, 6912, True), (8, 5120, 6848, False), (8, 6144, 6912, True),
                                           (8, 6144, 6144, False), (8, 6145, 8192, False)])
def test_handoff_rule(rec, m, n, k, handoff):
    assert rec.linear(m, n, k) == (["linear_handoff"] if handoff else ["quantize_rows_i8", "gemv_w8a8_xt"])


# The f64 matrix-core GEMM's two-chunk form up to K = 128, by alignment and K.
@pytest.mark.parametrize("k,shift,kernel", [(128, 0, "short"), (132, 0, ""), (127, 0, "short_any"), (129, 0, "any"),
                                            (64, 4, "short_any"), (4, 0, "short")])
def test_gemm_f32_short_k(rec, k, shift, kernel):
    m, n, X = 300, 60, 1 << 40
    assert rec.kernels("nh_gemm_f32", X + shift, m * k, 2 << 40, k * n, m, k, n, 3 << 40, m * n, None) == [
        "gemm_f32_mfma" + ("_" + kernel if kernel else "")]


# Every linear kernel of the library is reached by a shape that the GPU tests check bit for bit: a dispatch that moves on
# must not leave one behind without a test.
def test_gpu_tests_reach_every_linear_kernel(rec):
    import test_gpu_direct_gemm as direct
    import test_gpu_parity as parity
    import test_gpu_random_shapes as drawn
    import test_gpu_w4_decode_any as w4any

    def shapes(fn):
        return next(m.args[1] for m in fn.pytestmark if m.name == "parametrize" and m.args[0].startswith("m,"))

    reached = set()
    for m, n, k, kernels in direct.SHAPES + direct.RAGGED:
        reached.update(kernels)
    for m, n, k, _, f32, offset, _ in shapes(direct.test_direct_w4a8_bit_exact):
        reached.update(rec.w4a8(m, n, k, NH.F32 if f32 else NH.BF16, x=(1 << 40) + offset))
    for m, n, k, _, dtype in shapes(parity.test_linear_w4a8_bit_exact):
        reached.update(rec.w4a8(m, n, k, NH.F32 if dtype == "f32" else NH.BF16))
    for m, n, k, _ in shapes(w4any.test_w4a8_decode_any_k_bit_exact):
        reached.update(rec.w4a8(m, n, k))
    for fn in (parity.test_linear_decode_unit_bit_exact, parity.test_linear_small_m_shapes_bit_exact, parity.test_linear_handoff_bit_exact):
        for s in shapes(fn):
            f32 = fn is parity.test_linear_small_m_shapes_bit_exact and s[3] == "f32"
            reached.update(rec.linear(s[0], s[1], s[2], NH.F32 if f32 else NH.BF16))
    for m, hidden, inter, dtype in shapes(parity.test_mlp_bit_exact):
        reached.update(rec.mlp(m, hidden, inter, NH.F32 if dtype == "f32" else NH.BF16))
    for i in range(40):
        m, n, k, dtype, out_bf16, _, _ = drawn.draw_linear(i)
        reached.update(rec.linear(m, n, k, NH.F32 if dtype == "f32" else NH.BF16, NH.BF16 if out_bf16 else NH.F32))
    for m, n, k in shapes(parity.test_gemm_w8a8_bit_exact):
        reached.update(rec.kernels("nh_gemm_w8a8", 1 << 40, 2 << 40, 3 << 40, 4 << 40, None, m, n, k, 5 << 40, NH.BF16, None))
    source = os.path.join(os.path.dirname(NH.__file__), "csrc", "runtime", "context.cpp")
    every = set(re.findall(r'"nh_((?:linear|gemm_w|expand)\w*)_kernel"', open(source).read()))
    assert len(every) > 30 and every - reached == set()
