"""sj_gemm with several k-steps in flight (1 to 5 steps of 32, odd row strides,
every operand kind) and the embedding gradient's batches of 64 rows."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_util import best_us, dev, empty, rel, rnd, sync

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


@pytest.mark.parametrize("n,d,same,offset,V", [
    (1, 4, 1, 0, 11), (64, 128, 64, 0, 11), (65, 132, 65, 1, 11), (4097, 64, 4000, 0, 11), (9000, 384, 200, 1, 11),
    (5000, 2048, 130, 3, 11),
    # two chunks of 128 columns a workgroup (batches of 32), and four (16); a
    # window without a match; the last chunk of a workgroup partly or wholly past d
    (9000, 388, 33, 0, 2000), (600, 260, 32, 1, 512), (600, 384, 17, 0, 3000), (9000, 516, 16, 2, 12000),
    (3, 2048, 1, 0, 5000),
])
def test_embedding_gradient_batches(api, n, d, same, offset, V):
    """Rows summed in token order, bit for bit: batches exactly full and one
    more, matches over several scan windows, ids at any alignment."""
    rng = np.random.default_rng(n + d)
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


def test_embedding_gradient_of_a_large_vocabulary(api):
    """A row's columns are split over workgroups, and the ids scanned once for
    each, only while the rows are few: with 8192 rows of 16 column chunks each
    the call stays within a few passes over its output (50 us; 279 with every
    chunk its own workgroup)."""
    V, n, d = 8192, 4096, 2048
    ids = (np.random.default_rng(1).random(n) ** 2 * V).astype(np.int32)
    dy, I, W = empty(n * d), dev(ids, "i32"), empty(V * d)
    fill, grad = best_us(lambda: api.sj_fill(None, W.p, 0, V * d, 0.0),
                         lambda: api.sj_embedding_bwd(None, dy.p, I.p, W.p, n, d, V, None, 0))
    assert grad < 6 * fill, (grad, fill)
