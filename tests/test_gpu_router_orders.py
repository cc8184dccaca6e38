"""The router's logits kernels by order, type and batch size (rabbitm2_amd/csrc/router.hip): routing equal to
the oracle's with no exemption but exact ties, and combine weights bit for bit but for the exp: the
kernels round an exp taken in double, glibc's expf is within 0.502 ulp, so at most 0.4% of exps differ by an
ulp, and a renormalised weight holds K + 1 of them; a logit that is not the engine's own sum moves nearly
every weight. Sizes at the edges of the kernels' ranges: 256 / 257 tokens (a block per token and row pair, then
tiles of 16 rows x 16 tokens or the batch kernel), 16 / 17 (the general kernel, then those tiles, for dims
that the first does not take), ragged rows and tokens, dims at and past a 512-column chunk, and dims that fall
back to the general kernel. The grouped path's fused front end: 512 / 513 (one token per wave, then two).
"""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests.common import SynthLayer, routing_check

pytestmark = pytest.mark.gpu

SHAPES = [(64, 8, 2), (16, 5, 2), (2048, 64, 8), (1040, 20, 4), (100, 7, 3), (516, 33, 4), (4096, 3, 1), (8256, 5, 2)]


@pytest.mark.parametrize("dt", [po.DT_F32, po.DT_BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("order", [po.ORDER_AVX2, po.ORDER_SCALAR], ids=["avx2", "scalar"])
@pytest.mark.parametrize("shape", SHAPES, ids=["D%dE%dK%d" % s for s in SHAPES])
def test_router_logits_exact(dev, shape, order, dt):
    D, E, K = shape
    bias = np.linspace(-0.25, 0.25, E).astype(np.float32) if E % 2 else None
    layer = SynthLayer(dev, D, E, K, 16, dt, 1, seed=51, w_scale=1.0, fan_in=True, bias=bias)
    try:
        dev.set_router_order(order)
        for T in (1, 3, 16, 17, 256, 257, 511, 513) if D <= 1040 else (1, 16, 18, 257):
            xb = layer.make_x(T, seed=52 + T, bf16=False)
            got, want = layer.run_gpu(xb), layer.oracle(xb, order)
            bad, unexplained = routing_check(got["routing"], want["routing"], want["probs"])
            assert unexplained == 0
            if bad == 0:
                g, w = got["weights"], want["weights"].astype(np.float32).reshape(got["weights"].shape)
                off = g != w
                assert off.sum() <= max(1, 0.004 * (K + 1) * off.size), (T, int(off.sum()))
                assert np.max(np.abs(g - w) / w) <= (K + 2) * 2.0 ** -23
    finally:
        layer.close()


@pytest.mark.parametrize("shape", [(64, 64, 8), (1048, 49, 3), (516 * 2, 61, 61)], ids=["D64E64", "D1048E49", "D1032E61"])
@pytest.mark.parametrize("T", [65, 512, 513, 515])
def test_router_front_end_exact(dev, shape, T):
    """Router, softmax and top-k in one launch, as the grouped calls of 48 experts and more take them: blocks of two
    tokens up to 512, of four from 513 on, the last one cut short."""
    D, E, K = shape
    layer = SynthLayer(dev, D, E, K, 16, po.DT_BF16, 1, seed=53, w_scale=1.0, fan_in=True)
    try:
        dev.set_router_order(po.ORDER_AVX2)
        dev.set_option("full_min_tokens", 2)
        xb = layer.make_x(T, seed=54 + T, bf16=False)
        got, want = layer.run_gpu(xb), layer.oracle(xb, po.ORDER_AVX2)
        bad, unexplained = routing_check(got["routing"], want["routing"], want["probs"])
        assert unexplained == 0
        if bad == 0:
            g, w = got["weights"], want["weights"].astype(np.float32).reshape(got["weights"].shape)
            off = g != w
            assert off.sum() <= max(1, 0.004 * (K + 1) * off.size), (T, int(off.sum()))
            assert np.max(np.abs(g - w) / w) <= (K + 2) * 2.0 ** -23
    finally:
        dev.set_option("full_min_tokens", 0)
        layer.close()
