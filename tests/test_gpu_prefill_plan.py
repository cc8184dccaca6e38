"""The grouped path's plan from the tokens-per-expert histogram (rabbitm2_amd/csrc/prefill.hip): wide 128-row tiles
or 64-row tiles, by the time that the rounds of either take, and the dispatch of many pairs in two launches.

Whatever the plan, the outputs are those of either tile height, bit for bit (both run the same sums), and the
histogram is the routing's. The plan's rule is restated here and held to measured times. Sizes: one
round of wide tiles, both sides of the rule, and 6144 / 6152 pairs around the one-block dispatch.
"""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests.common import SynthLayer

pytestmark = pytest.mark.gpu


BLOB = dict(full=290, empty2=15, second=80, second_kd=40960, per_group=50, behind=96, part_max=64)
COPY = dict(full=260, empty2=5, second=60, second_kd=20480, per_group=20, behind=32, part_max=256)


def plan_rows(counts, D, H, k=BLOB):
    c = [int(v) for v in counts]
    tiles = lambda rows: sum(-(-v // rows) for v in c)
    m128, m64 = tiles(128), tiles(64)
    if m128 * (H // 256) <= 256:
        return 128
    skewed = max(c) * len(c) > 4 * sum(c)
    per = k["full"] - k["empty2"] * (8 * m128 - tiles(16)) // (2 * m128)
    wide = short = 0
    for nt, kd in ((H // 256, D), (D // 512, H)):
        rounds = -(-m128 * nt // 256)
        part, cost = m128 * nt - (rounds - 1) * 256, rounds * per
        if skewed and rounds == 2 and part <= k["part_max"]:
            need = -(-(part + k["behind"]) // nt)
            q = next((q for q in range(1, 8) if sum(0 < v % 128 <= 16 * q for v in c) >= need), 8)
            cost = min(cost, per + k["second"] + k["second_kd"] // kd + k["per_group"] * max(0, q - 3) +
                       (40 + (part - 64) * 5 // 8 if part > 64 else 0))
        wide += cost * kd
        short += -(-m64 * 2 * nt // 256) * 100 * kd
    return 64 if short < wide else 128


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
        rows = plan_rows(counts, 2048, 1024)
        assert dev.tile_rows() == rows
        dev.set_option("prefill_tile_rows", rows)
        want = layer.run_gpu(xb)
    finally:
        dev.set_option("prefill_tile_rows", 0)
    print(f"T {T} skew {skew}: {rows}-row tiles, longest list {counts.max()}", flush=True)
    assert np.array_equal(got["routing"], want["routing"])
    assert got["moe"].tobytes() == want["moe"].tobytes()


# (bias, experts that have it, tokens, us of gate/up + down measured on wide tiles, on wide tiles reading a tiled
# copy, on 64-row tiles)
FULL = (2048, 64, 8, 1024)
TIMES = {
    FULL: [(0, 0, 777, 195, 184, 264), (0, 0, 1500, 371, 359, 427), (1, 16, 400, 322, 298, 200),
           (2, 8, 512, 232, 197, 239), (2, 8, 450, 230, 196, 246), (2, 8, 777, 324, 298, 249),
           (2, 8, 1500, 368, 345, 436), (4, 4, 1300, 353, 328, 427), (2, 1, 300, 234, 203, 189),
           (30, 8, 1300, 334, 308, 352)],
    (512, 64, 6, 1024): [(4, 4, 600, 105, 92, 79), (2, 1, 400, 116, 109, 65)],
    (4096, 16, 2, 2048): [(4, 4, 1500, 438, 306, 430)],
}


@pytest.mark.parametrize("shape", TIMES, ids=["D%dE%dK%dH%d" % s for s in TIMES])
def test_plan_is_the_faster_height(dev, layers, shape):
    """The device's pick against times measured with either height forced, with and without a tiled copy."""
    D, E, K, H = shape
    layer = layers[False] if shape == FULL else SynthLayer(dev, D, E, K, H, po.DT_BF16, 1, seed=1, w_scale=0.02)
    kept = layer.bias_dev
    dev.set_router_order(po.ORDER_AVX2)
    wrong = []
    try:
        for amp, n, T, wide, copy, short in TIMES[shape]:
            layer.bias_dev = dev.upload_array(np.array([amp] * n + [0.0] * (E - n), np.float32))
            xb = layer.make_x(T, seed=67, bf16=False)
            out = {}
            for tiled, us, k in ((False, wide, BLOB), (True, copy, COPY)):
                if tiled:
                    dev.prefill_layout(layer.desc())
                out[tiled] = layer.run_gpu(xb)["moe"].tobytes()
                rows = dev.tile_rows()
                assert rows == plan_rows(dev.expert_counts(E), D, H, k)
                if (us if rows == 128 else short) > 1.03 * min(us, short):
                    wrong.append((amp, n, T, tiled, rows, us, short))
            dev.prefill_layout_drop(layer.desc())
            assert out[False] == out[True]
            dev.free(layer.bias_dev)
    finally:
        dev.prefill_layout_drop(layer.desc())
        layer.bias_dev = kept
        if layer is not layers[False]:
            layer.close()
    assert not wrong


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
        dev.set_option("full_min_tokens", 12)
        dev.set_router_order(po.ORDER_AVX2)
        xb = layer.make_x(T, seed=63)
        got = layer.run_gpu(xb)
        assert np.array_equal(dev.expert_counts(E), np.bincount(got["routing"].ravel(), minlength=E))
        pick = np.unique(np.r_[0, 1, T - 1, np.random.default_rng(64).integers(0, T, 200)])
        want = layer.oracle(xb[pick], po.ORDER_AVX2)
        rel = np.linalg.norm(got["moe"][pick] - want["moe"], axis=1) / np.linalg.norm(want["moe"], axis=1)
        assert rel.max() <= 1e-5  # sums of at most 64 f32 products in other orders
    finally:
        dev.set_option("full_min_tokens", 0)
        layer.close()
