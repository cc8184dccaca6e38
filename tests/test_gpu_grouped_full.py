"""The full-precision grouped form (rabbitm2_amd/csrc/grouped_full.hip): f32 weights, and bf16 weights of
dims that the bf16 tiles do not divide, where it is faster or from "full_min_tokens" tokens on.

Each output is held to its value in 64 bits within the worst case of its own sums: a sum of n f32 products
in blocks of 64 columns and then over the blocks is off by at most gamma = (64 + n / 32 + 16) * 2^-24 of the
sum of its terms' absolute values (the parts of a bf16 product are exact); the gate and up errors travel
through silu (slope at most 1.1) and W2, and the exp, divide and combine add a few roundings each.
Routing equals the oracle's except at exact ties.
"""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests.common import SynthLayer, routing_check

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def by_size(dev):
    """Every test leaves the choice of the form to the size of the call again."""
    yield
    dev.set_option("full_min_tokens", 0)


SHAPES = [
    # (D, E, K, H, dtype, T, bias on expert 0)
    (36, 5, 2, 25, po.DT_F32, 17, 0),      # partial last k-steps, h rows padded, 4-byte loads
    (36, 4, 2, 25, po.DT_BF16, 20, 0),     # 2-byte loads of W2 rows
    (32, 4, 1, 64, po.DT_F32, 13, 0),      # one k-step
    (8, 4, 2, 7, po.DT_BF16, 12, 0),       # rows shorter than a k-step both ways
    (64, 8, 2, 128, po.DT_BF16, 12, 0),    # 32-row tiles
    (1000, 20, 3, 330, po.DT_BF16, 50, 0),
    (100, 7, 7, 33, po.DT_BF16, 40, 0),    # K = E: every list 40 rows, 64-row tiles
    (256, 8, 2, 256, po.DT_F32, 300, 30),  # one list of 300 rows: five row tiles
    (260, 6, 1, 132, po.DT_BF16, 129, 0),  # past a column tile by 4
    (128, 256, 4, 48, po.DT_F32, 64, 0),   # the most experts, most lists empty
    (2048, 64, 8, 1024, po.DT_F32, 33, 0),
]


def reference(layer, xb, routing, weights):
    """(moe, bound) in 64 bits for the given routing."""
    T, D, H = xb.shape[0], layer.D, layer.H
    u = 2.0 ** -24
    g1, g2 = (64 + D / 32 + 16) * u, (64 + H / 32 + 16) * u
    moe, bound = np.zeros((T, D)), np.zeros((T, D))
    n = H * D
    for e in np.unique(routing):
        raw = layer.experts[e * layer.stride:e * layer.stride + 3 * n * layer.esz]
        w = (po.bf16_to_f32(raw.view(np.uint16)) if layer.dtype == po.DT_BF16 else raw.view(np.float32)).astype(np.float64)
        w1, w3, w2 = w[:n].reshape(H, D), w[n:2 * n].reshape(H, D), w[2 * n:].reshape(D, H)
        t, k = np.nonzero(routing == e)
        x = xb[t].astype(np.float64)
        g, up = x @ w1.T, x @ w3.T
        eg, eu = g1 * (np.abs(x) @ np.abs(w1).T), g1 * (np.abs(x) @ np.abs(w3).T)
        s = g / (1.0 + np.exp(-g))
        h = s * up
        eh = 1.1 * np.abs(up) * eg + (np.abs(s) + 1.1 * eg) * eu + 8 * u * np.abs(h)
        wk = weights[t, k].astype(np.float64)[:, None]
        np.add.at(moe, t, wk * (h @ w2.T))
        np.add.at(bound, t, wk * (eh @ np.abs(w2).T + (g2 + 12 * u) * ((np.abs(h) + eh) @ np.abs(w2).T)))
    return moe, bound


@pytest.mark.parametrize("shape", SHAPES, ids=["D%dE%dK%dH%ddt%dT%db%d" % s for s in SHAPES])
def test_full_grouped_shapes(dev, shape):
    D, E, K, H, dt, T, b = shape
    bias = np.array([float(b)] + [0.0] * (E - 1), np.float32) if b else None
    dev.set_option("full_min_tokens", 12)  # from 12 tokens on whatever the sizes
    layer = SynthLayer(dev, D, E, K, H, dt, 1, seed=31, w_scale=1.0, fan_in=True, bias=bias)
    try:
        dev.set_router_order(po.ORDER_AVX2)
        xb = layer.make_x(T, seed=32, bf16=False)
        x = layer.make_x(T, seed=33)
        got = layer.run_gpu(xb, x=x)
        want = layer.oracle(xb, po.ORDER_AVX2, x=x)
        assert routing_check(got["routing"], want["routing"], want["probs"])[1] == 0
        counts = dev.expert_counts(E)
        assert counts is not None and np.array_equal(counts, np.bincount(got["routing"].ravel(), minlength=E))
        moe, bound = reference(layer, xb, got["routing"], got["weights"])
        worst = np.max(np.abs(got["moe"] - moe) / np.maximum(bound, 1e-30))
        rel = np.linalg.norm(got["moe"] - moe) / np.linalg.norm(moe)
        print(f"D{D}E{E}K{K}H{H}T{T}: error {rel:.2e}, {worst:.3f} of the bound", flush=True)
        assert worst <= 1.0
        assert np.array_equal(got["x"], x + got["moe"])
    finally:
        layer.close()


def test_full_grouped_nonfinite_rows_stay_apart(dev):
    """A token with infinities and NaN leaves the other tokens' rows as they are without it."""
    dev.set_option("full_min_tokens", 12)
    layer = SynthLayer(dev, 68, 4, 4, 36, po.DT_BF16, 0, seed=35, w_scale=1.0, fan_in=True)
    try:
        dev.set_router_order(po.ORDER_AVX2)
        xb = layer.make_x(16, seed=36, bf16=False)
        clean = layer.run_gpu(xb)["moe"]
        xb[5, 3], xb[5, 67] = np.inf, np.nan
        xb[9, :4] = 3.4e38  # rounds past the largest bf16; its parts do not
        got = layer.run_gpu(xb)["moe"]
        keep = [t for t in range(16) if t not in (5, 9)]
        assert got[keep].tobytes() == clean[keep].tobytes()
        assert np.isnan(got[5]).any()
        dev.set_option("full_min_tokens", 65536)  # the GEMVs: token 9's sums are finite, h and y may not be
        want = layer.run_gpu(xb)["moe"][[5, 9]]
        for same in (np.isnan, np.isposinf, np.isneginf):
            assert np.array_equal(same(got[[5, 9]]), same(want))
    finally:
        layer.close()


@pytest.mark.parametrize("dt", [po.DT_F32, po.DT_BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("what", ["inf in w3", "inf in w2", "inf in w1", "overflow in w3", "overflow in w2", "inf in x"])
@pytest.mark.parametrize("shape", [(68, 36), (512, 132)], ids=["D68", "D512"])
def test_full_grouped_infinities_are_the_gemvs(dev, what, dt, shape):
    """Where a weight is infinite or a sum of finite products overflows, the infinities (and their signs) and
    the NaN are those of the per-pair GEMVs. Activations of one bf16 part, whose other parts are zeros."""
    D, H = shape
    layer = SynthLayer(dev, D, 4, 2, H, dt, 0, seed=39, w_scale=1.0, fan_in=True)
    dev.set_router_order(po.ORDER_AVX2)
    try:
        big = 2e19 if "overflow" in what else np.inf
        enc = np.array([big], np.float32)
        enc = enc.view(np.uint16)[1:] if dt == po.DT_BF16 else enc
        mat = D * H
        first = {"w1": 0, "w3": mat, "w2": 2 * mat}[what[-2:]] if what != "inf in x" else None
        xb = layer.make_x(16, seed=40)
        if first is not None:  # one row of the first expert's matrix: every product of it, or its last
            n = H if what.endswith("w2") else D
            row = np.repeat(enc, n if "overflow" in what else 1)
            at = first + 3 * n + (0 if "overflow" in what else n - 1)
            dev.h2d(layer.experts_dev, row, offset=at * layer.esz)
        if what == "overflow in w3":
            xb[3] = 1e19  # products 2e38: any two of them overflow
        elif what == "overflow in w2":
            xb[3] = 1e10
            raw = np.repeat(np.array([1e10], np.float32).view(np.uint16)[1:] if dt == po.DT_BF16
                            else np.array([1e10], np.float32), 2 * mat)
            dev.h2d(layer.experts_dev, raw, offset=0)  # gate and up 1e20 D, h past the largest float
        elif what == "inf in x":
            xb[3, D - 1] = np.inf
        dev.set_option("full_min_tokens", 65536)
        want = layer.run_gpu(xb)["moe"]
        dev.set_option("full_min_tokens", 2)
        got = layer.run_gpu(xb)
        assert dev.expert_counts(4) is not None and dev.expert_counts(4).sum() == 32
        got = got["moe"]
        assert not np.isfinite(want).all()
        assert np.array_equal(np.isnan(got), np.isnan(want))
        assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
        fin = np.isfinite(want)
        g64, w64 = got[fin].astype(np.float64), want[fin].astype(np.float64)
        assert np.linalg.norm(g64 - w64) <= 4e-6 * np.linalg.norm(w64)  # sums of at most 512 f32 products
    finally:
        layer.close()


def test_full_grouped_scratch_limit(dev):
    """rbt_hip_moe_dev_noalloc takes the per-pair GEMVs where the grouped buffers pass its scratch array, so
    the calls that fitted without them still run."""
    D, E, K, H, T = 2048, 8, 8, 64, 1200  # y alone is 75 MiB; the GEMVs need 2.4 MiB
    dev.set_option("full_min_tokens", 12)
    layer = SynthLayer(dev, D, E, K, H, po.DT_F32, 1, seed=37, w_scale=1.0, fan_in=True)
    xb = layer.make_x(T, seed=38)
    xd, moe = dev.upload_array(xb), dev.malloc(4 * T * D)
    try:
        dev.set_router_order(po.ORDER_AVX2)
        dev.moe_dev_noalloc(layer.desc(), xd, T, moe=moe)
        got = dev.d2h(moe, (T, D), np.float32)
        want = layer.run_gpu(xb)["moe"]
        assert np.linalg.norm(got - want) <= 4e-6 * np.linalg.norm(want)
    finally:
        dev.free(xd)
        dev.free(moe)
        layer.close()


# (D, E, K, H, dtype) around the number of tokens from which the grouped form is taken. The lines:
# 100e6 expected saved bytes, 450e6 for the shapes of the specialised GEMVs, 1000e6 where their gate/up reads an
# expert once.
LINES = [(1600, 40, 6, 800, po.DT_BF16), (1000, 20, 3, 330, po.DT_BF16), (260, 6, 2, 132, po.DT_F32),
         (512, 8, 2, 512, po.DT_F32), (2048, 64, 8, 1024, po.DT_F32)]


@pytest.mark.parametrize("shape", LINES, ids=["D%dE%dK%dH%ddt%d" % s for s in LINES])
def test_full_grouped_is_taken_by_size(shape):
    """A handle whose options nobody set: on either side of the line the call's bits are those of the form it is
    expected to take, and not the other's; setting "prefill_min_tokens" changes nothing of it, and
    "full_min_tokens" 0 brings the size back."""
    from rabbitm2_amd.hip import Device
    D, E, K, H, dt = shape
    esz = po.ELEM[dt]
    fast = (D * esz) % 1024 == 0 and (H * esz) % 1024 == 0  # the specialised GEMVs' rows, in whole wave-steps

    def takes_grouped(T):
        p, sel = T * K, E * (1.0 - (1.0 - K / E) ** T)
        once = p <= 128 and D * esz <= 1024 * (4 if dt == po.DT_BF16 else 8) and (p - sel) * 2.0 * H * D * esz >= 60e6
        return (p - sel) * 3.0 * H * D * esz >= (100e6 if not fast else 1000e6 if once else 450e6)

    edge = next(T for T in range(2, 2000) if takes_grouped(T))
    with Device(0) as dev:
        layer = SynthLayer(dev, D, E, K, H, dt, 1, seed=45, w_scale=1.0, fan_in=True)
        try:
            dev.set_router_order(po.ORDER_AVX2)
            for T in (edge - 1, edge):
                xb = layer.make_x(T, seed=46, bf16=False)
                got = layer.run_gpu(xb)["moe"].tobytes()
                dev.set_option("prefill_min_tokens", 12)
                dev.set_option("full_min_tokens", 65536)
                gemvs = layer.run_gpu(xb)["moe"].tobytes()
                dev.set_option("full_min_tokens", 2)
                grouped = layer.run_gpu(xb)["moe"].tobytes()
                dev.set_option("full_min_tokens", 0)
                assert layer.run_gpu(xb)["moe"].tobytes() == got
                assert gemvs != grouped
                assert got == (grouped if T == edge else gemvs), T
            for bad in (-1, 65537):
                with pytest.raises(Exception):
                    dev.set_option("full_min_tokens", bad)
        finally:
            layer.close()


def test_full_grouped_under_capture():
    """A captured call allocates nothing: where the workspace was not reserved for the grouped form, the per-pair
    GEMVs are captured, and after an eager call the grouped form is. Each replay gives the eager call's bits."""
    import ctypes as C

    from rabbitm2_amd.hip import Device
    hip = C.CDLL("libamdhip64.so")
    hip.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    hip.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    hip.hipGraphInstantiate.argtypes = [C.POINTER(C.c_void_p), C.c_void_p, C.c_void_p, C.c_void_p, C.c_size_t]
    hip.hipGraphLaunch.argtypes = [C.c_void_p, C.c_void_p]
    hip.hipGraphExecDestroy.argtypes = hip.hipGraphDestroy.argtypes = [C.c_void_p]
    D, T = 100, 40
    with Device(0) as dev:
        layer = SynthLayer(dev, D, 7, 3, 33, po.DT_BF16, 1, seed=47, w_scale=1.0, fan_in=True)
        xb = layer.make_x(T, seed=48, bf16=False)
        xd, moe = dev.upload_array(xb), dev.malloc(4 * T * D)
        dev.set_router_order(po.ORDER_AVX2)
        dev.moe_dev(layer.desc(), xd, T, moe=moe)  # by size: the GEMVs
        dev.synchronize()
        gemvs = dev.d2h(moe, (T, D), np.float32).tobytes()
        dev.set_option("full_min_tokens", 2)
        grouped = None
        for reserved in (False, True):
            if reserved:
                dev.moe_dev(layer.desc(), xd, T, moe=moe)
                dev.synchronize()
                grouped = dev.d2h(moe, (T, D), np.float32).tobytes()
                assert grouped != gemvs
            graph, gexec = C.c_void_p(), C.c_void_p()
            assert hip.hipStreamBeginCapture(dev.stream, 2) == 0
            dev.moe_dev(layer.desc(), xd, T, moe=moe)
            assert hip.hipStreamEndCapture(dev.stream, C.byref(graph)) == 0
            assert hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, 0) == 0
            for _ in range(3):
                dev.memset(moe, 0)
                assert hip.hipGraphLaunch(gexec, dev.stream) == 0
                dev.synchronize()
                assert dev.d2h(moe, (T, D), np.float32).tobytes() == (grouped if reserved else gemvs)
            hip.hipGraphExecDestroy(gexec)
            hip.hipGraphDestroy(graph)
        layer.close()
