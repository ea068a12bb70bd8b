"""The parameter VJP's kernels at the edges of their ranges: ranks 1, 16, 17,
32, 33 and 64, ragged rows, more than 64 selected blocks (the serial draws),
and the coefficient product's tiles (64 x 64, and each taller one)."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from oracle import pvjp as P
from tests.test_gemm_plan_host import COEFFICIENTS, plan
from tests.gpu_util import best_us, dev, empty, rel, rnd, sync, zeros

pytestmark = pytest.mark.gpu
cf = ctypes.c_float


@pytest.fixture(scope="module")
def N():
    from sejong_amd import _native as N
    N.load()
    return N


@pytest.mark.parametrize("A,B,block,S,R,seed", [
    (1024, 2752, 32, 4, 16, 7), (1000, 300, 32, 32, 64, 1 << 40), (37, 5, 8, 5, 5, 3), (64, 64, 1, 64, 64, 11),
    (260, 70, 2, 100, 16, 5),   # more than 64 blocks
    (64, 200, 16, 2, 100, 9),   # more than 64 columns
    (64, 1, 64, 1, 1, 2 ** 64 - 1),
])
def test_indices_match_the_reference_draws(N, A, B, block, S, R, seed):
    NB = -(-A // block)
    scr, cols, rows, fmap = zeros(B + NB, "i32"), zeros(R, "i32"), zeros(S * block, "i32"), zeros(A, "i32")
    N.api.sj_pvjp_indices(None, ctypes.c_uint64(seed), A, B, NB, S, R, block, scr.p, cols.p, rows.p, fmap.p)
    sync()
    c, r, m = P.indices(seed, A, B, NB, S, R, block)
    np.testing.assert_array_equal(cols.host(), c)
    np.testing.assert_array_equal(rows.host(), r)
    np.testing.assert_array_equal(fmap.host(), m)


def test_indices_of_many_blocks_in_one_pass(N):
    """The map is one pass over its rows whatever the blocks (60 of them once
    took 10 times as long as one; the draws themselves are a few us)."""
    A, B, block, R = 65536, 60000, 32, 8
    NB = A // block
    scr, cols, fmap = zeros(B + NB, "i32"), zeros(R, "i32"), zeros(A, "i32")

    rows = zeros(60 * block, "i32")

    def draw(S):
        return lambda: N.api.sj_pvjp_indices(None, ctypes.c_uint64(3), A, B, NB, S, R, block, scr.p, cols.p, rows.p, fmap.p)
    many, one = best_us(draw(60), draw(1))
    assert many < 3 * one, (many, one)


@pytest.mark.parametrize("n,R,dt,dup", [(64, 1, "f32", False), (65, 16, "bf16", False), (1000, 17, "f32", False),
                                        (16400, 32, "bf16", False), (777, 33, "f32", True), (2048, 64, "bf16", True)])
def test_basis_orthonormal_span_and_drop(N, n, R, dt, dup):
    """Q^T Q = I on the kept columns, Q spans the picked columns, a duplicated
    column becomes zero (n x R sums of fp32-rounded Q: 1e-6)."""
    rng = np.random.default_rng(n + R)
    B = R + 9
    y = rnd((n, B), dt, rng)
    cols = rng.permutation(B)[:R].astype(np.int32)
    if dup:
        cols[R - 1] = cols[0]
    q = empty(n * R)
    lib = N.load()
    wb = lib.sj_pvjp_basis_workspace_bytes(n, R)
    ws = empty(wb, "u8")
    N.api.sj_pvjp_basis(None, dev(y, dt).p, 4 if dt == "bf16" else 0, B, n, dev(cols, "i32").p, R,
                        cf(lib.sj_pvjp_basis_tolerance(n, R)), q.p, ws.p, wb)
    sync()
    Q = q.host().reshape(n, R)
    keep = R - 1 if dup else R
    if dup:
        assert np.all(Q[:, R - 1] == 0)
    assert np.max(np.abs(Q[:, :keep].T @ Q[:, :keep] - np.eye(keep))) < 2e-6
    V = y[:, cols[:keep]]
    Qr, _ = np.linalg.qr(V)
    assert rel(Q[:, :keep] @ (Q[:, :keep].T @ V), Qr @ (Qr.T @ V)) < 2e-6


@pytest.mark.parametrize("R,bad", [(5, 0), (16, 7), (20, 19), (64, 33)])
def test_basis_value_out_of_range_stays_in_its_row(N, R, bad):
    """A column with an infinite value is dropped (its pivot is not finite):
    the other rows of Q stay finite whatever the column's place."""
    n = 300
    y = rnd((n, R), "f32", np.random.default_rng(R))
    y[41, bad] = np.inf
    cols, q = np.arange(R, dtype=np.int32), empty(n * R)
    lib = N.load()
    wb = lib.sj_pvjp_basis_workspace_bytes(n, R)
    ws = empty(wb, "u8")
    N.api.sj_pvjp_basis(None, dev(y, "f32").p, 0, R, n, dev(cols, "i32").p, R, cf(lib.sj_pvjp_basis_tolerance(n, R)),
                        q.p, ws.p, wb)
    sync()
    assert np.isfinite(np.delete(q.host().reshape(n, R), 41, axis=0)).all()


@pytest.mark.parametrize("rows,b,n,tile", [
    (48, 200, 8192, (64, 64)), (80, 136, 8200, (64, 64)), (112, 64, 8192, (64, 64)), (144, 264, 8256, (64, 64)),
    (176, 72, 16384, (64, 64)), (272, 320, 8192, (64, 64)), (145, 8, 9000, (64, 64)),
    (66, 1504, 8456, (96, 64)), (129, 976, 8288, (160, 64)), (100, 2056, 8208, (128, 128)), (129, 3344, 8648, (160, 128)),
    (162, 3296, 8312, (192, 128))])
def test_coefficient_tiles(N, rows, b, n, tile):
    """E dY with both operands as hi/lo planes, dY in row layout: against FP64
    (three bf16 products of four: 2^-16 per term, random signs)."""
    assert plan(COEFFICIENTS, rows, b, n)[1:3] == tile
    rng = np.random.default_rng(rows + b)
    split = lambda x: (O.round_to(x, "bf16"), O.round_to(x - O.round_to(x, "bf16"), "bf16"))
    e = rng.normal(0, 1, (rows, n)).astype(np.float32).astype(np.float64)
    dy = rng.normal(0, 1, (n, b)).astype(np.float32).astype(np.float64)
    eh, el = split(e)
    dh, dl = split(dy)
    lib = N.load()
    wb = lib.sj_pvjp_vjp_workspace_bytes(rows, b, n)
    E = [dev(x, "bf16") for x in (eh, el)]
    D = [dev(x, "bf16") for x in (dh, dl)]
    for ws_bytes in (wb, 0):   # with and without room for K slices
        C, ws = zeros(rows * b), empty(max(wb, 256), "u8")
        N.api.sj_pvjp_vjp_rows(None, E[0].p, E[1].p, n, rows, n, D[0].p, D[1].p, b, b, C.p, b,
                               ws.p if ws_bytes else None, ws_bytes)
        sync()
        assert rel(C.host(), (eh + el) @ (dh + dl)) < 3e-5


@pytest.mark.parametrize("a,b,R", [(16383, 40, 5), (16400, 40, 5), (16401, 37, 9)])
def test_factored_apply_table_sizes(N, a, b, R):
    """1024 tiles (the latency form's last table) and more (the wide form's), ragged rows, columns and rank."""
    rng = np.random.default_rng(a + b)
    f = lambda *s: rng.normal(0, 1, s).astype(np.float32)
    left, right, tail, w = f(a, R), f(R, b), f(3, b), f(a, b)
    fmap = np.full(a, -1, np.int32)
    fmap[[0, 17, a - 1]] = [2, 0, 1]
    L, RT, TL, MP, W = dev(left), dev(right), dev(tail), dev(fmap, "i32"), dev(w)
    TA = (N.FactoredTerm * 1)(N.FactoredTerm(L.ptr, RT.ptr, TL.ptr, MP.ptr, R, 0.5, b))
    PA = (N.FactoredParam * 1)(N.FactoredParam(W.ptr, None, a, b, 1, 0, 1, b, None))
    nb = N.load().sj_factored_meta_bytes(PA, 1, 1)
    host, tiles = np.zeros(nb, np.uint8), ctypes.c_long()
    N.api.sj_factored_pack(PA, 1, TA, 1, ctypes.c_void_p(host.ctypes.data), nb, ctypes.byref(tiles))
    assert tiles.value == -(-a // 16)
    meta, part = dev(host, "u8"), empty(tiles.value, "f64")
    N.api.sj_factored_apply(None, meta.p, tiles.value, 2, cf(0), cf(0), part.p)
    N.api.sj_factored_apply(None, meta.p, tiles.value, 1, cf(0.25), cf(0.125), None)
    sync()
    g = 0.5 * left.astype(np.float64) @ right
    g[[0, 17, a - 1]] += 0.5 * tail[[2, 0, 1]].astype(np.float64)
    assert rel(part.host().sum(), (g ** 2).sum()) < 1e-6  # fp32 sums of R terms
    assert rel(W.host().reshape(a, b), w * 0.875 - 0.25 * g) < 1e-6


def test_factored_materialize_of_a_narrow_parameter(N):
    """Half of a tile's threads have no column: the ones that do must not wait
    for them over the tails (2048 tiles of 256 columns; materializing took
    0.88 of the norm's time with two barriers and an LDS copy of the places
    per term, 0.69 without)."""
    a, b, R = 32768, 256, 16
    L, RT, TL, W = (empty(n) for n in (a * R, R * b, 3 * b, a * b))
    for t, n in ((L, a * R), (RT, R * b), (TL, 3 * b), (W, a * b)):
        N.api.sj_fill(None, t.p, 0, n, 0.5)
    MP = dev(np.full(a, -1, np.int32), "i32")
    TA = (N.FactoredTerm * 1)(N.FactoredTerm(L.ptr, RT.ptr, TL.ptr, MP.ptr, R, 0.5, b))
    PA = (N.FactoredParam * 1)(N.FactoredParam(W.ptr, None, a, b, 1, 0, 1, b, None))
    nb = N.load().sj_factored_meta_bytes(PA, 1, 1)
    host, tiles = np.zeros(nb, np.uint8), ctypes.c_long()
    N.api.sj_factored_pack(PA, 1, TA, 1, ctypes.c_void_p(host.ctypes.data), nb, ctypes.byref(tiles))
    meta, part = dev(host, "u8"), empty(tiles.value, "f64")
    write, norm = best_us(*[lambda act=act: N.api.sj_factored_apply(None, meta.p, tiles.value, act, cf(0), cf(0), part.p)
                            for act in (0, 2)])
    assert write < 0.8 * norm, (write, norm)
