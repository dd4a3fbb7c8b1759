"""The MoE expert kernels' split over the chip: how many workgroups an expert
gets, and which workgroup takes which expert, depend on how many experts the
routes reach.  Every output is exact, so each split equals the oracle's
stages bit for bit."""
import numpy as np
import pytest

import nemotron_hip as NH
import oracle_ctypes as O
from exact_int import moe_forward_exact
from tiling import tile_experts

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = NH.Context(0)
    yield c
    c.close()


# one route; a few experts of many (their workgroups packed); more than 64 experts (the search's second step) with the
# only routes at the last of them; every expert reached; parts that leave the last one few tiles or none; one expert
# with every route (several passes of rows); the search's last step of four and the reads after it, up to 1024 experts
# (the up projection in 2, 3, 4, 5, 8, 9 and 17 parts: as many row maxima for the down projection's lane groups to share)
@pytest.mark.parametrize("tokens,hidden,inter,experts,top_k,only", [
    (1, 256, 128, 5, 1, None), (2, 64, 176, 30, 2, None), (2, 512, 1072, 130, 2, None), (7, 1040, 272, 70, 3, (64, 70)), (3, 512, 1072, 192, 2, (184, 192)), (3, 512, 1072, 193, 2, (185, 193)),
    (3, 512, 1072, 256, 2, (248, 256)), (3, 512, 1072, 257, 2, (249, 257)), (20, 512, 256, 16, 2, None),
    (40, 272, 64, 9, 4, None), (130, 256, 528, 3, 1, (1, 2)), (90, 528, 16, 200, 1, (128, 200)), (6, 64, 2048, 40, 6, None),
    (3, 64, 528, 512, 2, None), (5, 64, 272, 1000, 4, (990, 1000)), (1, 128, 256, 1024, 8, None), (9, 64, 256, 513, 1, (512, 513))])
def test_moe_split_bit_exact(ctx, tokens, hidden, inter, experts, top_k, only):
    print(f"moe split t={tokens} h={hidden} i={inter} e={experts} k={top_k} only={only}", flush=True)
    rng = np.random.default_rng(tokens + experts)
    x = O.to_bf16(O.normal_f32(9 + tokens, tokens * hidden)).reshape(tokens, hidden)
    logits = rng.standard_normal((tokens, experts)).astype(np.float32)
    if only:  # every route inside this range of experts
        logits[:, : only[0]] -= 50
        logits[:, only[1]:] -= 50
    up = rng.integers(-127, 128, size=(experts, inter, hidden), dtype=np.int8)
    down = rng.integers(-127, 128, size=(experts, hidden, inter), dtype=np.int8)
    su = rng.uniform(1e-4, 1e-3, (experts, inter)).astype(np.float32)
    sd = rng.uniform(1e-4, 1e-3, (experts, hidden)).astype(np.float32)
    ref = moe_forward_exact(x, logits.reshape(-1), up, su, down, sd, top_k)[0]
    ws_bytes = NH.lib().nh_moe_forward_w8a8_workspace_size(tokens, hidden, inter, experts, top_k)
    ws = ctx.empty(ws_bytes, np.uint8)
    ws.fill_bytes(0x7f)  # row maxima of parts without columns are written, not assumed
    d = [ctx.upload(a) for a in (x, logits, tile_experts(up), su, tile_experts(down), sd)]
    out = ctx.empty((tokens, hidden), np.uint16)
    NH.call("nh_moe_forward_w8a8", ctx.handle, d[0].ptr, NH.BF16, d[1].ptr, tokens, hidden, inter, experts, top_k, 1,
            1.0, *(b.ptr for b in d[2:]), None, out.ptr, NH.BF16, ws.ptr, ws_bytes, None, None)
    ctx.synchronize()
    assert np.array_equal(out.numpy(), ref)
