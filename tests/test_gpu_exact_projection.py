"""The batched prefill's exact projections on the matrix cores (k_bgemm)
against the CPU restatement, bit for bit, where the kernel's tiling can go
wrong: token counts around its 16- and 48-token tiles and the count at which
it takes over, widths that leave a partial visit pair, a partial line group or
a single visit, and row counts that end inside a tile. And the products that a
fused multiply-add would round differently: value weights and inputs so small
that the lowest bits of their products lie below the F32 subnormals,
recomputed by k_bgemm_fix (with 300 tokens of 512 value channels some outputs
differ where the fused sums are kept)."""
import numpy as np
import pytest

import cq35
import cq35.config as cc

pytestmark = pytest.mark.gpu


def config(hidden, intermediate, value_heads=4):
    cfg = cc.preset("mini")
    cfg.update(vocab=512, hidden=hidden, intermediate=intermediate, value_heads=value_heads)
    return cfg


def compare(oracle, cfg, weights, prompt):
    gm, om = cq35.Model.from_arrays(cfg, weights), oracle.Model(cfg, weights)
    gs, os_ = gm.session(len(prompt)), om.session(len(prompt))
    gl, gt = gs.step_raw(prompt)
    ot, ol = os_.step(prompt, 0)
    assert gt == ot
    assert np.array_equal(gl, ol), "logits"
    assert np.array_equal(gs.export_state(0), os_.cache()), "state"
    gm.close()


# hidden 576: nine lines (visits of one and two); 1024: one visit pair; 320:
# less than one visit. intermediate 1344: 21 lines, 84 tiles; 1416: 22.125
# lines (not whole ones: the vector kernel) with gate rows ending inside a
# tile; 200: rows ending inside a tile.
@pytest.mark.parametrize("hidden, intermediate, tokens", [
    (576, 1344, 7), (576, 1344, 8), (576, 1344, 17), (1024, 3584, 48), (576, 1416, 49), (320, 200, 257), (576, 1344, 289),
])
def test_tiles_match_restatement(oracle, hidden, intermediate, tokens):
    cfg = config(hidden, intermediate)
    print("exact projection", hidden, intermediate, tokens, flush=True)
    prompt = np.random.default_rng(tokens).integers(0, cfg["vocab"], tokens).tolist()
    compare(oracle, cfg, oracle.synthetic_weights(cfg, 29), prompt)


@pytest.mark.parametrize("tokens", [20, 300])
def test_products_below_the_exact_range(oracle, tokens):
    cfg = config(512, 1408)
    weights = oracle.synthetic_weights(cfg, 30)
    full = cfg["full_interval"] - 1
    base = 1 + 14 * full  # first attention layer: its input norm, and three tensors on attn_v
    specs = oracle.weight_specs(cfg)
    assert specs[base + 3][1] == cfg["kv_heads"] * cfg["head_dim"] and specs[base + 3][2] == cfg["hidden"]
    # inputs of about 2^-16 and weights of about 2^-120: products of 16 bits
    # around 2^-136, the lowest below 2^-149
    weights[base] = weights[base] * np.float32(2.0 ** -16)
    w = weights[base + 3]
    exponent = (w.astype(np.int32) >> 7) & 0xff
    assert exponent.max() < 127
    scaled = np.where(exponent > 114, (w & 0x807f) | ((exponent - 114) << 7).astype(np.uint16), 0)
    assert (scaled != 0).mean() > 0.8
    weights[base + 3] = scaled.astype(np.uint16)
    print("exact projection, tiny weights", tokens, flush=True)
    prompt = np.random.default_rng(tokens).integers(0, cfg["vocab"], tokens).tolist()
    compare(oracle, cfg, weights, prompt)
