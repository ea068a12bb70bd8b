"""The attention row kernels (fp32, and bf16 shapes outside the MFMA layout)
at the edges of their tiles: 64 streamed rows, 4 or 16 fixed rows per
workgroup, column counts that are not powers of two or exceed 64."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_util import assert_stored_close, best_us, dev, empty, rel, rnd, sync

pytestmark = pytest.mark.gpu
DT = {"f32": 0, "bf16": 4}


@pytest.fixture(scope="module")
def api():
    from sejong_amd import _native as N
    N.load()
    return N.api


# B, T, HQ, HK, Dh, dt, window, padding of the row strides
CASES = [
    (1, 1, 2, 1, 2, "f32", 0, 0),        # one key; the smallest head
    (2, 63, 2, 2, 10, "f32", 0, 1),      # below a tile, odd strides (scalar loads)
    (1, 64, 3, 1, 16, "f32", 0, 0),      # exactly a tile
    (2, 65, 4, 2, 40, "f32", 0, 4),      # one row past a tile, columns not a power of two
    (1, 130, 2, 1, 80, "f32", 64, 0),    # more than 64 columns, a window of one tile
    (1, 70, 2, 2, 128, "f32", 1, 0),     # the widest head, every query sees itself only
    (3, 131, 2, 1, 64, "bf16", 65, 8),   # bf16, ragged T, window
    (4, 520, 4, 2, 24, "f32", 200, 0),   # 16 rows per workgroup
    (2, 1100, 4, 4, 72, "bf16", 0, 0),   # 16 rows per workgroup, bf16, two column halves
    (4, 519, 8, 4, 64, "f32", 0, 0),     # 16 rows per workgroup in all three kernels at one 64-column group
    (5, 450, 4, 4, 48, "f32", 77, 4),    # the same, columns not a power of two, a window
    # the short walks (one key at a time) at their lines, and one past them
    (2, 70, 2, 1, 16, "f32", 2, 0), (2, 70, 2, 1, 16, "f32", 3, 0), (3, 4, 2, 1, 10, "bf16", 0, 0),
    (2, 70, 4, 2, 32, "f32", 4, 1), (2, 70, 4, 2, 32, "bf16", 5, 0), (7, 8, 3, 1, 64, "f32", 0, 0),
    (2, 70, 2, 2, 64, "bf16", 9, 8), (2, 70, 2, 1, 128, "f32", 12, 0), (2, 70, 2, 2, 100, "f32", 13, 0),
    (4, 1030, 4, 2, 96, "f32", 24, 0), (4, 1030, 4, 2, 96, "f32", 25, 0),
]


@pytest.mark.parametrize("B,T,HQ,HK,Dh,dt,window,pad", CASES)
def test_row_kernels_against_oracle(api, B, T, HQ, HK, Dh, dt, window, pad):
    rng = np.random.default_rng(B * T + Dh)
    M, ldq, ldk = B * T, HQ * Dh + pad, HK * Dh + pad

    def padded(x, ld):
        return np.concatenate([x, np.full((x.shape[0], ld - x.shape[1]), 7.0)], 1)
    q, k, v = (rnd((M, n * Dh), dt, rng) for n in (HQ, HK, HK))
    do = rng.normal(0, 1e-3, (M, HQ * Dh)).astype(np.float32).astype(np.float64)
    Q, K, V, DO = dev(padded(q, ldq), dt), dev(padded(k, ldk), dt), dev(padded(v, ldk), dt), dev(padded(do, ldq))
    Ot, L = empty(M * HQ * Dh, dt), empty(M * HQ)
    api.sj_attention_fwd(None, Q.p, ldq, K.p, ldk, V.p, ldk, Ot.p, HQ * Dh, L.p, DT[dt], B, T, HQ, HK, Dh, window)
    sync()
    o_ref, lse_ref = O.attention_fwd(q, k, v, B, T, HQ, HK, Dh, window)
    o_abs, _ = O.attention_fwd(q, k, np.abs(v), B, T, HQ, HK, Dh, window)
    assert_stored_close(Ot.host(), o_ref, dt, "O", terms=2 * o_abs)
    assert rel(L.host(), lse_ref) < 1e-5
    o_st, lse_st = Ot.host().reshape(M, HQ * Dh), L.host()
    dQ, dK, dV, De = empty(M * HQ * Dh), empty(M * HK * Dh), empty(M * HK * Dh), empty(M * HQ)
    tab = empty(T * Dh)
    import ctypes
    api.sj_rope_table(None, tab.p, T, Dh, ctypes.c_float(10000.0))
    api.sj_attention_bwd(None, Q.p, ldq, K.p, ldk, V.p, ldk, Ot.p, HQ * Dh, L.p, DO.p, ldq, dQ.p, HQ * Dh, dK.p,
                         HK * Dh, dV.p, HK * Dh, De.p, DT[dt], B, T, HQ, HK, Dh, window, tab.p)
    sync()
    dq, dk, dv, delta = O.attention_bwd(q, k, v, o_st, lse_st, do, B, T, HQ, HK, Dh, window)
    dq = O.rope(dq, T, HQ, Dh, inverse=True)
    dk = O.rope(dk, T, HK, Dh, inverse=True)
    # fp32 products and sums of at most 1100 terms: 1100 * 2^-24 = 7e-5 at the
    # worst.  ds = p (do.v - Delta) may cancel (exactly to 0 with one visible
    # key), so the two dot products' own rounding is allowed beside it: four
    # partial sums of Dh / 4 terms each, (Dh / 4 + 2) 2^-24 |do| |v|, times
    # |k| Dh^-0.5, with |v| and |k| about sqrt(Dh) for unit normal rows
    slack = 2 * (Dh / 4 + 2) * 2.0 ** -24 * np.linalg.norm(do) * Dh ** 0.5
    for name, got, ref in (("delta", De, delta), ("dq", dQ, dq), ("dk", dK, dk), ("dv", dV, dv)):
        e = np.linalg.norm(got.host() - np.asarray(ref, np.float64).ravel())
        assert e < 1e-4 * np.linalg.norm(ref) + slack, (name, e)


def test_cached_rows_of_both_row_counts_have_the_same_bits(api):
    """One 64-column group: the full forward takes 16 rows per workgroup, the
    few cached rows 4; and a window short enough for the walk kernels against
    the same rows of a cache whose length alone differs."""
    T, HQ, HK, Dh = 2112, 4, 2, 64
    d, J = HQ * Dh, HK * Dh
    rng = np.random.default_rng(64)
    Q, K, V = (dev(rnd((T, n), "f32", rng)) for n in (d, J, J))
    for window in (0, 8, 9):
        O1, LSE, O2 = empty(T * d), empty(T * HQ), empty(5 * d)
        api.sj_attention_fwd(None, Q.p, d, K.p, J, V.p, J, O1.p, d, LSE.p, 0, 1, T, HQ, HK, Dh, window)
        for L in (T - 5, 0, 3):
            api.sj_attention_fwd_cached(None, Q.at(L * d), d, K.p, V.p, J, T, 0, 5, L, HQ, HK, Dh, window, O2.p, d)
            sync()
            np.testing.assert_array_equal(O2.host().reshape(5, d), O1.host().reshape(T, d)[L:L + 5])


def test_short_windows_cost_less_than_long_ones(api):
    """A window of 2 walks its few keys: no staged tile of 64 (4 x 1024 tokens,
    head_dim 128: staged, 2 and 64 took the same time and 4.5 times as long)."""
    B, T, H, Dh = 4, 1024, 4, 128
    n = B * T * H * Dh
    Q, K, V, DO, O1 = (empty(n) for _ in range(5))
    L, dQ, dK, dV, De = empty(B * T * H), empty(n), empty(n), empty(n), empty(B * T * H)
    for b in (Q, K, V, DO):
        api.sj_fill(None, b.p, 0, n, 0.25)

    def both(window):
        api.sj_attention_fwd(None, Q.p, H * Dh, K.p, H * Dh, V.p, H * Dh, O1.p, H * Dh, L.p, 0, B, T, H, H, Dh, window)
        api.sj_attention_bwd(None, Q.p, H * Dh, K.p, H * Dh, V.p, H * Dh, O1.p, H * Dh, L.p, DO.p, H * Dh, dQ.p, H * Dh,
                             dK.p, H * Dh, dV.p, H * Dh, De.p, 0, B, T, H, H, Dh, window, None)
    short, long = best_us(lambda: both(2), lambda: both(64))
    assert short < 0.5 * long, (short, long)


@pytest.mark.parametrize("L,window", [(2111, 0), (2107, 100), (2047, 64), (0, 0)])
def test_cached_rows_have_the_full_forwards_bits(api, L, window):
    """Rows L.. through the cached call (4 rows per workgroup for few rows)
    against the full forward's (16): the same operations per row."""
    T, HQ, HK, Dh = 2112, 4, 2, 32
    d, J = HQ * Dh, HK * Dh
    rng = np.random.default_rng(L + window)
    q, k, v = rnd((T, d), "f32", rng), rnd((T, J), "f32", rng), rnd((T, J), "f32", rng)
    Q, K, V = dev(q), dev(k), dev(v)
    O1, LSE = empty(T * d), empty(T * HQ)
    api.sj_attention_fwd(None, Q.p, d, K.p, J, V.p, J, O1.p, d, LSE.p, 0, 1, T, HQ, HK, Dh, window)
    O2 = empty((T - L) * d)
    api.sj_attention_fwd_cached(None, Q.at(L * d), d, K.p, V.p, J, T, 0, T - L, L, HQ, HK, Dh, window, O2.p, d)
    sync()
    np.testing.assert_array_equal(O2.host().reshape(T - L, d), O1.host().reshape(T, d)[L:])
