"""The few-row products of the cached path (decode.hip) at their edges: 1, 7
and 8 rows beside the tiled path's 9 and more, contractions that are not
multiples of 32 or of 512, a vocabulary that is not a multiple of 16."""
import time

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
        for n in (1, 15, 16, 17, 2, 1, 7, 8, 9, 16, 60, 1, 13, 1, 1):
            got = m.forward_cached(tokens[at:at + n], cache)
            at += n
            # the same operations in the same order: the full forward's bits
            np.testing.assert_array_equal(got, full[at - 1], err_msg=f"chunk of {n} ending at {at}")
        cache.close()
    finally:
        m.close()


def test_a_longer_chunk_is_not_the_faster_call():
    """The few-row products serve only as many rows as they are the faster
    path for: a chunk of 16 tokens against one of 20 (6 layers, d 384; on the
    few-row products 16 took 1.18 times the tiled path's time)."""
    from sejong_amd.model import Model, ModelConfig, TrainConfig, init_params
    mc = ModelConfig(width=384, layers=6, heads=6, kv_heads=2, ffn_width=1024, context=512, precision="bf16")
    m = Model(mc, TrainConfig(sequence=64, batch=1))
    try:
        m.set_params(init_params(mc, std=0.02))
        tokens, cache = np.arange(20, dtype=np.int32), m.new_cache()

        def us(n):
            cache.reset()
            m.synchronize()
            t0 = time.perf_counter()
            for _ in range(20):
                m.forward_cached(tokens[:n], cache, read=False)
            m.synchronize()
            return time.perf_counter() - t0
        us(16), us(20)
        chunk, longer = (min(x) for x in zip(*[(us(16), us(20)) for _ in range(16)]))
        cache.close()
    finally:
        m.close()
    assert chunk < 1.1 * longer, (chunk, longer)
