"""The forms of the prefill attention at their edges: passes that end below position 64 and passes of few tokens (a
workgroup per head and token each), then the tiled kernel with few heads (a head's coordinates over several workgroups)
and many (a workgroup per head), every head dimension, passes that start and end inside a 16-token tile, and a max_ctx
that caps the padded length at 603, so that the four chunks start at multiples of 151 (inside a group of 8 positions).
The KV cache (the second layer's depends on the first layer's attention) and each pass' last logits equal single decode
steps, or the oracle's loop, bit for bit."""
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


def check_passes(oracle, model, passes, seed):
    """Prefills the passes and compares with the oracle."""
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
    finally:
        pre.close()
        model.close()
