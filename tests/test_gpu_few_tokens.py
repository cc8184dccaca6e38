"""Gate/up of a few tokens with each selected expert read once (rabbitm2_amd/csrc/experts_decode.hip): every
output keeps the products and sums of the one-token kernel, so a call's rows are those of its tokens' own
calls, bit for bit."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests.common import SynthLayer

pytestmark = pytest.mark.gpu

CASES = [
    # (D, E, K, H, dtype, T, bias on expert 0)
    (2048, 64, 8, 1024, po.DT_BF16, 4, 0),   # below the line: one read per pair
    (2048, 64, 8, 1024, po.DT_BF16, 5, 0),   # at it
    (2048, 64, 8, 1024, po.DT_BF16, 16, 20),  # 128 pairs: both masks full, one expert selected by all
    (2048, 64, 8, 1024, po.DT_BF16, 17, 0),  # 136 pairs: one read per pair again
    (512, 5, 5, 1024, po.DT_BF16, 10, 0),    # one wave-step, every token selects every expert
    (1536, 40, 13, 512, po.DT_BF16, 5, 0),   # 65 pairs
    (1024, 3, 1, 4096, po.DT_BF16, 64, 0),   # 64 pairs: the second mask empty
    (256, 3, 1, 4096, po.DT_F32, 128, 0),    # one place per token
    (768, 9, 3, 2048, po.DT_F32, 21, 0),     # 63 pairs
    (2048, 2, 2, 256, po.DT_F32, 64, 0),     # two experts, 64 pairs each, longest rows
    (4096, 8, 2, 1024, po.DT_BF16, 8, 0),    # rows past the longest: one read per pair
]


@pytest.mark.parametrize("case", CASES, ids=["D%dE%dK%dH%ddt%dT%db%d" % c for c in CASES])
def test_rows_are_the_single_tokens_rows(dev, case):
    D, E, K, H, dt, T, b = case
    bias = np.array([float(b)] + [0.0] * (E - 1), np.float32) if b else None
    layer = SynthLayer(dev, D, E, K, H, dt, 1, seed=51, w_scale=1.0, fan_in=True, bias=bias)
    dev.set_option("prefill_min_tokens", 1000)  # the GEMVs at every T here
    dev.set_option("full_min_tokens", 1000)
    try:
        dev.set_router_order(po.ORDER_AVX2)
        xb, x = layer.make_x(T, seed=52, bf16=False), layer.make_x(T, seed=53)
        got = layer.run_gpu(xb, x=x)
        for t in range(T):
            one = layer.run_gpu(xb[t:t + 1], x=x[t:t + 1])
            for k in ("routing", "weights", "moe", "x"):
                assert got[k][t].tobytes() == one[k][0].tobytes(), (t, k)
    finally:
        dev.set_option("prefill_min_tokens", 12)
        dev.set_option("full_min_tokens", 0)
        layer.close()
