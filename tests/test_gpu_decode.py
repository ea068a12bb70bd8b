"""The few-row products of the cached path (decode.hip) at their edges: 1, 15
and 16 rows beside the tiled path's 17, contractions that are not multiples
of 32 or of 512, a vocabulary that is not a multiple of 16."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv,ffn,experts", [(3, 1, 1000, 0), (1, 1, 8, 0), (16, 4, 2760, 0), (2, 2, 72, 4)])
def test_chunks_around_the_row_limit_equal_the_full_forward(heads, kv, ffn, experts):
    from sejong_amd.benchmark import full_logits
    from sejong_amd.model import ExpertConfig, Model, ModelConfig, TrainConfig, init_params
    T = 192
    mc = ModelConfig(width=64 * heads, layers=2, heads=heads, kv_heads=kv, ffn_width=ffn, context=T, precision="bf16",
                     experts=ExpertConfig(count=experts, top_k=2, ffn_width=ffn) if experts else None)
    m = Model(mc, TrainConfig(sequence=T, batch=1))
    try:
        m.set_params(init_params(mc, std=0.05))
        tokens = np.random.default_rng(heads).integers(0, 257, T).astype(np.int32)
        full = full_logits(m, tokens)
        cache = m.new_cache()
        at = 0
        for n in (1, 15, 16, 17, 2, 1, 16, 60, 1, 13, 1, 1):
            got = m.forward_cached(tokens[at:at + n], cache)
            at += n
            # the same operations in the same order: the full forward's bits
            np.testing.assert_array_equal(got, full[at - 1], err_msg=f"chunk of {n} ending at {at}")
        cache.close()
    finally:
        m.close()
