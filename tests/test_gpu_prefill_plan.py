"""The grouped path's plan from the tokens-per-expert histogram (rabbitm2_amd/csrc/prefill.hip): wide 128-row tiles
or 64-row tiles, by the number of rounds that either takes, and the dispatch of many pairs in two launches.

Whatever the plan, the outputs are those of either tile height, bit for bit (both run the same sums), and the
histogram is the routing's. The plan's rule is restated here. Sizes: one
round of wide tiles, both sides of the rule, and 6144 / 6152 pairs around the one-block dispatch.
"""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests.common import SynthLayer

pytestmark = pytest.mark.gpu


def plan_rows(counts, wide_nt):
    ceil = lambda a, b: (a + b - 1) // b
    rw = ceil(int(sum(ceil(c, 128) for c in counts)) * wide_nt, 256)
    rs = ceil(int(sum(ceil(c, 64) for c in counts)) * 2 * wide_nt, 256)
    return 64 if rw > 1 and rs * 10 < rw * 29 else 128


@pytest.fixture(scope="module")
def layers(dev):
    made = {}
    for skew in (False, True):
        bias = np.array([2.0] * 8 + [0.0] * 56, np.float32) if skew else None
        made[skew] = SynthLayer(dev, 2048, 64, 8, 1024, po.DT_BF16, 1, seed=61, bias=bias)
    yield made
    for layer in made.values():
        layer.close()


@pytest.mark.parametrize("T,skew", [(256, False), (400, True), (768, False), (769, False), (777, True), (1024, False),
                                    (1500, True), (2500, False)])
def test_plan_matches_forced_height(dev, layers, T, skew):
    layer = layers[skew]
    dev.set_router_order(po.ORDER_AVX2)
    xb = layer.make_x(T, seed=T)
    try:
        got = layer.run_gpu(xb)
        counts = dev.expert_counts(64)
        assert np.array_equal(counts, np.bincount(got["routing"].ravel(), minlength=64))
        rows = plan_rows(counts, 4)
        dev.set_option("prefill_tile_rows", rows)
        want = layer.run_gpu(xb)
    finally:
        dev.set_option("prefill_tile_rows", 0)
    print(f"T {T} skew {skew}: {rows}-row tiles, longest list {counts.max()}", flush=True)
    assert np.array_equal(got["routing"], want["routing"])
    assert got["moe"].tobytes() == want["moe"].tobytes()


@pytest.mark.parametrize("D,E,K,H,T", [(2048, 64, 8, 1024, 777), (512, 16, 4, 256, 200), (1024, 8, 2, 768, 500)])
def test_rows_do_not_depend_on_the_height(dev, D, E, K, H, T):
    """Both heights run the same chunks in the same order, so the height that the other tokens' routing leads to
    does not show in a token's output."""
    layer = SynthLayer(dev, D, E, K, H, po.DT_BF16, 1, seed=65, w_scale=1.0, fan_in=True)
    dev.set_router_order(po.ORDER_AVX2)
    xb = layer.make_x(T, seed=66, bf16=False)
    got = {}
    try:
        for rows in (0, 64, 128):
            dev.set_option("prefill_tile_rows", rows)
            got[rows] = layer.run_gpu(xb)["moe"].tobytes()
    finally:
        dev.set_option("prefill_tile_rows", 0)
        layer.close()
    assert got[64] == got[128] and got[0] == got[128]


@pytest.mark.parametrize("E,K,T", [(8, 2, 3073), (256, 6, 1025), (61, 7, 20000), (5, 1, 6145)])
def test_dispatch_of_many_pairs(dev, E, K, T):
    """Two-launch dispatch: every pair in its expert's list once, so every token's output is what a call of
    the token alone gives within the two forms' rounding, and the histogram is the routing's."""
    layer = SynthLayer(dev, 64, E, K, 32, po.DT_BF16, 0, seed=62, w_scale=1.0, fan_in=True)
    try:
        dev.set_option("prefill_min_tokens", 12)
        dev.set_router_order(po.ORDER_AVX2)
        xb = layer.make_x(T, seed=63)
        got = layer.run_gpu(xb)
        assert np.array_equal(dev.expert_counts(E), np.bincount(got["routing"].ravel(), minlength=E))
        pick = np.unique(np.r_[0, 1, T - 1, np.random.default_rng(64).integers(0, T, 200)])
        want = layer.oracle(xb[pick], po.ORDER_AVX2)
        rel = np.linalg.norm(got["moe"][pick] - want["moe"], axis=1) / np.linalg.norm(want["moe"], axis=1)
        assert rel.max() <= 1e-5  # sums of at most 64 f32 products in other orders
    finally:
        layer.close()
