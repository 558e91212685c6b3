"""The forms of the prefill attention at their edges: passes that end below position 64 (a workgroup per head and token),
then the tiled kernel with few heads (a head's coordinates over several workgroups) and many (a workgroup per head), every head dimension, passes that start and end inside a 16-token tile, and a max_ctx
that caps the padded length at 603, so that the four chunks start at multiples of 151 (inside a group of 8 positions).
The KV cache after every pass (the second layer's depends on the first layer's attention) and the last logits equal
single decode steps bit for bit."""
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
