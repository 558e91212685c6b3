"""The forms of the prefill attention at their edges: passes that end below position 64 and passes of few tokens (a
workgroup per head and token each), then the tiled kernel with few heads (a head's coordinates over several workgroups)
and many (a workgroup per head), every head dimension, passes that start and end inside a 16-token tile, and a max_ctx
that caps the padded length at 603, so that the four chunks start at multiples of 151 (inside a group of 8 positions).
The KV cache (the second layer's depends on the first layer's attention) and each pass' last logits equal single decode
steps, or the oracle's loop, bit for bit."""
import ctypes

import numpy as np
import pytest

from test_decode_gpu import assert_same_bits, load_decoder
from test_prefill_gpu import kv_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_heads", [2, 8])
@pytest.mark.parametrize("head_dim", [32, 64, 128, 256])
def test_prefill_attention_forms(oracle, head_dim, n_heads):
    model = oracle.Model(oracle.ModelConfig(2, 256, n_heads, n_heads // 2, head_dim, 384, 500, 603, 1e-5, 10000.0), 7)
    pre, ref = load_decoder(oracle, model), load_decoder(oracle, model)
    try:
        tokens = np.random.default_rng(head_dim).integers(0, 500, 603)
        for p0, p1 in ((0, 5), (5, 64), (64, 65), (65, 300), (300, 603)):
            got, _ = pre.prefill(tokens[p0:p1], pos0=p0)
            for pos in range(p0, p1):
                want, _ = ref.step(int(tokens[pos]), pos)
            assert_same_bits(got, want, f"prefill {p0}..{p1}")
        kv_equal(pre, ref, model.cfg, range(603))
    finally:
        pre.close()
        ref.close()
        model.close()


# Passes by their form with 8 heads on 256 CUs: (a) below position 64, (b) a workgroup per head and token (at most 512 of
# them), (c) tiles of one chunk, (d) tiles of four chunks; head_dim 256 takes (b) in place of (d) below 512 tiles.
EVERY_FORM = ((0, 30), (30, 64), (64, 65), (65, 200), (200, 256), (256, 257), (257, 320), (320, 400), (400, 417), (417, 603))


@pytest.mark.parametrize("n_heads,head_dim,passes", [(8, 32, EVERY_FORM), (8, 64, EVERY_FORM), (8, 128, EVERY_FORM),
                                                     (8, 256, EVERY_FORM), (32, 64, ((0, 256), (256, 272), (272, 289)))])
def test_prefill_attention_every_form(oracle, n_heads, head_dim, passes):
    """Every form over one cache, whole and split contexts. 32 heads: (0, 256) one chunk with a workgroup per head, then 512
    and 544 heads times tokens on both sides of form (b)'s limit."""
    model = oracle.Model(oracle.ModelConfig(2, 256, n_heads, n_heads // 2, head_dim, 384, 500, 603, 1e-5, 10000.0), 11)
    check_passes(oracle, model, passes, head_dim)


@pytest.mark.parametrize("head_dim,exponent", [(32, 14.4), (64, 14.3), (128, 14.25), (256, 14.25)])
def test_prefill_attention_infinities(oracle, head_dim, exponent):
    """Infinities in q, K and V, and the NaN that they make of scores and outputs: the first layer's attention norm is
    scaled until a few of its f16 values overflow, first in the middle of the context (outputs of layer 0 are then finite,
    NaN or infinite, between a few and most of them NaN). Without sub-norms a NaN output quantizes to 0 and the others to
    their codes, so the second layer's cache shows which outputs were NaN, and stays finite."""
    cfg = oracle.ModelConfig(2, 256, 8, 4, head_dim, 384, 500, 603, 1e-5, 10000.0, oracle.ACT_RELU2, oracle.ROPE_NORMAL, 1, 1, 0)
    model = oracle.Model(cfg, 7)
    gamma = (ctypes.c_float * cfg.hidden).from_address(oracle.lib().vxo_model_norm(model._h, 0, 0))
    np.ctypeslib.as_array(gamma)[:] *= np.float32(2.0 ** exponent)
    infinite = check_passes(oracle, model, EVERY_FORM, head_dim)
    assert 5 <= infinite <= 300, infinite


def check_passes(oracle, model, passes, seed):
    """Prefills the passes and compares with the oracle; returns how many (position, KV head) hold an infinity."""
    pre = load_decoder(oracle, model)
    try:
        n = passes[-1][1]
        tokens = np.random.default_rng(seed).integers(0, 500, n)
        for p0, p1 in passes:
            print(f"[prefill attention] head_dim {model.cfg.head_dim} {p0}..{p1}", flush=True)
            got, _ = pre.prefill(tokens[p0:p1], pos0=p0)
            for pos in range(p0, p1):
                _, want = model.forward(int(tokens[pos]), pos)
            assert_same_bits(got, want, f"prefill {p0}..{p1}")
        kv_equal(pre, model, model.cfg, range(n))
        return sum(bool(np.isinf(np.concatenate(model.kv(0, pos, h)).view(np.float16)).any())
                   for pos in range(n) for h in range(model.cfg.n_kv_heads))
    finally:
        pre.close()
        model.close()
