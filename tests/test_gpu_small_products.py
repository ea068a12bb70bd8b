"""sj_gemm with several k-steps in flight (1 to 5 steps of 32, odd row strides,
every operand kind) and the embedding gradient's batches of 64 rows."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_util import dev, empty, rel, rnd, sync

pytestmark = pytest.mark.gpu
DT = {"f32": 0, "bf16": 4}


@pytest.fixture(scope="module")
def api():
    from sejong_amd import _native as N
    N.load()
    return N.api


@pytest.mark.parametrize("K", [1, 31, 32, 33, 96, 128, 129, 257])
@pytest.mark.parametrize("ta,tb,ad,bd", [(0, 0, "bf16", "f32"), (0, 1, "f32", "f32"), (1, 0, "bf16", "f32"),
                                         (1, 1, "f32", "bf16"), (0, 0, "f32", "bf16")])
def test_gemm_steps_in_flight(api, K, ta, tb, ad, bd):
    M, N = 70, 133
    rng = np.random.default_rng(K + 2 * ta + tb)
    a, b = rnd((M, K), ad, rng), rnd((K, N), bd, rng)
    pad = lambda x: np.concatenate([x, np.full((x.shape[0], 3), 9.0)], 1)   # row strides of any residue
    A, B = pad(a.T if ta else a), pad(b.T if tb else b)
    C = empty(M * (N + 1))
    api.sj_gemm(None, ta, tb, M, N, K, dev(A, ad).p, DT[ad], A.shape[1], dev(B, bd).p, DT[bd], B.shape[1], C.p, 0,
                N + 1, 0, None, 0)
    sync()
    got = C.host().reshape(M, N + 1)[:, :N]
    # hi/lo bf16 products, the lo * lo one left out: 2^-16 of the terms' size
    e = np.linalg.norm(got - a @ b) / np.linalg.norm(np.abs(a) @ np.abs(b))
    assert e < 2.0 ** -16, e


@pytest.mark.parametrize("n,d,same,offset", [(1, 4, 1, 0), (64, 128, 64, 0), (65, 132, 65, 1), (4097, 64, 4000, 0),
                                             (9000, 384, 200, 1), (5000, 2048, 130, 3)])
def test_embedding_gradient_batches(api, n, d, same, offset):
    """Rows summed in token order, bit for bit: batches of exactly 64 and one
    more, matches over several scan windows, ids at any alignment."""
    rng = np.random.default_rng(n + d)
    V = 11
    ids = rng.integers(1, V, n).astype(np.int32)
    ids[rng.permutation(n)[:same]] = 3
    dy = rng.normal(0, 1, (n, d)).astype(np.float32)
    I = dev(np.concatenate([np.zeros(offset, np.int32), ids]), "i32")
    W = empty(V * d)
    api.sj_embedding_bwd(None, dev(dy).p, I.at(offset), W.p, n, d, V, None, 0)
    sync()
    want = np.zeros((V, d), np.float32)
    for i in range(n):
        want[ids[i]] += dy[i]
    np.testing.assert_array_equal(W.host().reshape(V, d).astype(np.float32), want)
