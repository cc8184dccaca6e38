"""A prompt read in as blocks of positions (rabbitm2_amd/csrc/prompt.hip, the dense form of
grouped_full.hip) by rbt_hip_generate, against the engine's outputs and against the per-token path.

The golden fixtures hold the reference engine's logits and routing at every position; behind a prompt of n
tokens, the forward of its last token must give the logits of that position, and the routing history the
routing of the ones before it. Bars as for the per-token path (tests/test_gpu_forward.py): routing
identical, logits within a normwise 1e-3 of the engine's.

Against the per-token path on the same device: both sum the same f32 products in other orders. A sum of n
terms is off by at most about sqrt(n) * 2^-24 of its scale in either order; with at most 640 terms, six
products and two norms per layer and two layers that is below 640^0.5 * 16 * 2 * 2^-24 = 5e-5 for each.
"""
import os

import numpy as np
import pytest

from oracle import pyoracle as po
from tests.common import normwise_err
from tests.test_gpu_forward import LOGIT_RTOL, MANIFEST, ORDERS, build

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


@pytest.fixture
def history(dev):
    dev.set_option("routing_history", 1)
    yield dev
    dev.set_option("routing_history", 0)
    dev.set_option("full_min_tokens", 0)


@pytest.mark.parametrize("tag", sorted(ORDERS))
@pytest.mark.parametrize("case", [c for c in sorted(MANIFEST["cases"]) if MANIFEST["cases"][c]["n_prompt"] > 5])
def test_block_prompt_matches_reference(history, case, tag):
    dev = history
    spec, cfg, model = build(case)
    fx = np.load(os.path.join(GOLDEN, case + ".npz"))
    dev.upload(model)
    dev.set_router_order(ORDERS[tag])
    tokens = np.asarray(fx["tokens"], np.int32)
    for n in sorted({5, 6, len(tokens)}):  # 4 positions and more before the last are run as a block
        dev.state_init(0)
        dev.generate(tokens[:n], 0)
        logits, routing = dev.forward(int(tokens[n - 1]), n - 1, cfg.vocab, cfg.n_layers, cfg.top_k)
        assert np.array_equal(routing, fx[f"routing_{tag}"][n - 1])
        assert normwise_err(logits, fx[f"logits_{tag}"][n - 1]) <= LOGIT_RTOL
        hist = dev.routing_history(0, 0, n - 1, cfg.n_layers, cfg.top_k)
        assert np.array_equal(hist, fx[f"routing_{tag}"][:n - 1])


# (head_dim, heads, kv heads, dtype, n): blocks around the 16-query and 32-key groups, grouped heads, more
# than one block (512 positions), other head dims, a dim that is no whole k-step
BLOCKS = [
    (128, 2, 1, po.DT_BF16, 17), (128, 2, 2, po.DT_BF16, 18), (128, 4, 2, po.DT_F32, 34), (128, 2, 1, po.DT_BF16, 66),
    (128, 1, 1, po.DT_BF16, 130), (128, 2, 1, po.DT_BF16, 640), (64, 3, 1, po.DT_BF16, 300), (256, 1, 1, po.DT_F32, 40),
    (20, 5, 5, po.DT_BF16, 33),
]


@pytest.mark.parametrize("form", ["gemvs", "grouped"])
@pytest.mark.parametrize("shape", BLOCKS, ids=["hd%dh%dkv%ddt%dn%d" % b for b in BLOCKS])
def test_block_prompt_matches_steps(history, shape, form):
    dev = history
    dev.set_option("full_min_tokens", 2 if form == "grouped" else 65536)  # the blocks' MoE form
    hd, heads, kv, dt, n = shape
    cfg = po.Config(vocab=96, dim=132, n_layers=2, n_heads=heads, n_kv_heads=kv, head_dim=hd, n_experts=8, top_k=2,
                    expert_hidden=72, max_seq=700, dtype=dt, qk_norm=1, norm_topk=1, rope_theta=10000.0, rms_eps=1e-5)
    model = po.build_model(cfg, po.GenParams(seed=41, w_scale=1.0, fan_in_scale=1, emb_scale=0.5, norm_jitter=0.1))
    tokens = np.random.default_rng(42).integers(0, cfg.vocab, n).astype(np.int32)
    dev.upload(model)
    dev.set_router_order(po.ORDER_AVX2)
    dev.state_init(700)
    for pos, tok in enumerate(tokens):
        want_l, want_r = dev.forward(int(tok), pos, cfg.vocab, cfg.n_layers, cfg.top_k)
    want_h = dev.routing_history(0, 0, n - 1, cfg.n_layers, cfg.top_k)
    dev.state_init(700)
    dev.generate(tokens, 0)
    got_l, got_r = dev.forward(int(tokens[-1]), n - 1, cfg.vocab, cfg.n_layers, cfg.top_k)
    got_h = dev.routing_history(0, 0, n - 1, cfg.n_layers, cfg.top_k)
    rel = np.linalg.norm(got_l - want_l) / np.linalg.norm(want_l)
    print(f"hd{hd} n{n}: logits {rel:.2e} from the steps'", flush=True)
    assert np.array_equal(got_h, want_h) and np.array_equal(got_r, want_r)
    assert rel <= 1e-4


@pytest.mark.parametrize("hd", [128, 64])
@pytest.mark.parametrize("bad", [0, 5, 21, 31, 32, 38])
def test_block_prompt_keeps_positions_before_a_nonfinite_one(history, hd, bad):
    """A token whose embedding holds an infinity makes its own and every later position NaN, and none before it:
    routing and logits of the earlier ones are the per-token path's, within its own bar above, and so is all
    routing (NaN logits select experts 0 .. K - 1)."""
    dev, n = history, 40
    cfg = po.Config(vocab=96, dim=132, n_layers=2, n_heads=2, n_kv_heads=1, head_dim=hd, n_experts=8, top_k=2,
                    expert_hidden=72, max_seq=64, dtype=po.DT_BF16, qk_norm=1, norm_topk=1, rope_theta=10000.0,
                    rms_eps=1e-5)
    model = po.build_model(cfg, po.GenParams(seed=43, w_scale=1.0, fan_in_scale=1, emb_scale=0.5, norm_jitter=0.1))
    dev.upload(model)
    emb, _ = dev.tensor("tok_emb")
    model[emb + 95 * 2 * cfg.dim:][:2] = (0x80, 0x7F)  # token 95's first element: infinity
    dev.upload(model)
    dev.set_router_order(po.ORDER_AVX2)
    tokens = np.random.default_rng(44).integers(0, 95, n).astype(np.int32)
    tokens[bad] = 95
    dev.state_init(64)
    want = [dev.forward(int(tok), pos, cfg.vocab, cfg.n_layers, cfg.top_k)[0] for pos, tok in enumerate(tokens)]
    want_h = dev.routing_history(0, 0, n, cfg.n_layers, cfg.top_k)
    dev.state_init(64)
    dev.generate(tokens, 0)
    assert np.array_equal(dev.routing_history(0, 0, n - 1, cfg.n_layers, cfg.top_k), want_h[:n - 1])
    for pos in sorted({max(bad - 1, 0), max(bad - 15, 0), bad, n - 1}):  # steps back over the block's cache rows
        got, _ = dev.forward(int(tokens[pos]), pos, cfg.vocab, cfg.n_layers, cfg.top_k)
        assert np.isnan(want[pos]).all() == (pos >= bad)
        if pos >= bad:
            assert np.isnan(got).all()
        else:
            assert np.linalg.norm(got - want[pos]) <= 1e-4 * np.linalg.norm(want[pos])
