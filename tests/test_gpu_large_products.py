"""The ping-pong products (k_gemm_pp) at shapes their rule takes: ragged rows
and columns, a contraction that ends inside a stage of 32, padded strides,
every epilogue, K slices.  References in FP64 on rows at the tiles' edges."""
import hashlib
import json
import os
import subprocess
import sys

import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gemm_plan_host import DW, DX, GATE_UP, PP, RESIDUAL, ROOT, SPLIT_OUT, plan
from tests.gpu_util import dev, empty, rel, sync, zeros

pytestmark = pytest.mark.gpu
BF, F32 = 4, 0


@pytest.fixture(scope="module")
def N_():
    from sejong_amd import _native as N
    N.load()
    return N


def bf(x):
    return O.round_to(np.asarray(x, np.float32), "bf16")


def split(x):
    h = bf(x)
    return h, bf(np.asarray(x, np.float32) - h)


def edge_rows(M):
    return np.unique(np.concatenate([np.arange(20), np.arange(120, 136), np.arange(250, 262), np.arange(M - 270, M)]))


def close_bf(got, ref, terms):
    # one bf16 rounding (half an ulp, 2^-8 of the value) of an fp32 sum whose
    # own error is under 2^-16 of its terms; a second rounding's half ulp
    tol = 2.0 ** -7 * np.abs(ref) + 2.0 ** -15 * terms
    assert (np.abs(got - ref) <= tol).all(), np.max(np.abs(got - ref) - tol)


def wide(x, pad):
    return np.pad(x, ((0, 0), (0, pad)), constant_values=np.float32(3.0))  # the row stride's padding: never read


@pytest.mark.parametrize("M,N,K,pad", [(8192, 768, 1032, 0), (16300, 504, 2056, 8), (16384, 1024, 1024, 24)])
@pytest.mark.parametrize("cdt", ["f32", "bf16"])
def test_planes(N_, M, N, K, pad, cdt):
    assert plan(DX, M, N, K)[0] == PP
    rng = np.random.default_rng(M + N + K)
    ah, al = split(rng.normal(0, 1, (M, K)).astype(np.float32))
    b = bf(rng.normal(0, 1, (N, K)))
    A, B = [dev(wide(t, pad), "bf16") for t in (ah, al)], dev(wide(b, pad), "bf16")
    C = zeros(M * (N + pad), cdt)
    dt = BF if cdt == "bf16" else F32
    for acc in ((0, 1) if cdt == "f32" else (0,)):  # stored, then accumulated
        N_.api.sj_gemm_planes(None, M, N, K, A[0].p, A[1].p, K + pad, B.p, None, K + pad, C.p, dt, N + pad, acc, None, 0)
    sync()
    r = edge_rows(M)
    full = (ah[r].astype(np.float64) + al[r]) @ b.T
    C = C.host().reshape(M, N + pad)
    assert not C[:, N:].any()
    if cdt == "bf16":
        close_bf(C[r, :N], full, np.abs(ah[r]) @ np.abs(b.T))
    else:
        assert rel(C[r, :N], 2 * full) < 2e-5


@pytest.mark.parametrize("M,N,K,pad", [(1024, 5504, 4096, 0), (1000, 5000, 5000, 8), (2040, 760, 8008, 16),
                                       (1024, 1536, 16384, 0)])
def test_row_layout(N_, M, N, K, pad):
    assert plan(DW, M, N, K)[0] == PP
    rng = np.random.default_rng(M + N + K)
    x = bf(rng.normal(0, 1, (K, M)))
    yh, yl = split(rng.normal(0, 1, (K, N)).astype(np.float32))
    X, Y = dev(wide(x, pad), "bf16"), [dev(wide(t, pad), "bf16") for t in (yh, yl)]
    wb = N_.load().sj_gemm_planes_workspace_bytes(M, N, K)
    r = np.concatenate([np.arange(10), np.arange(M - 10, M)])
    full = x[:, r].astype(np.float64).T @ (yh.astype(np.float64) + yl)
    for nbytes in (wb, 0):
        C, ws = zeros(M * N), empty(max(wb, 256), "u8")
        N_.api.sj_gemm_planes_tn(None, M, N, K, X.p, None, M + pad, Y[0].p, Y[1].p, N + pad, C.p, F32, N, 0,
                                 ws.p if nbytes else None, nbytes)
        sync()
        assert rel(C.host().reshape(M, N)[r], full) < 2e-5


@pytest.mark.parametrize("M,D,HQ,pad", [(8192, 1024, 16, 0), (16300, 520, 8, 8)])
def test_attention_output(N_, M, D, HQ, pad):
    """The output projection's input gradient as planes, with Delta."""
    assert plan(SPLIT_OUT, M, 64 * HQ, D)[0] == PP
    rng = np.random.default_rng(M + D)
    N, ld = 64 * HQ, 64 * HQ + pad
    dh, dl = split(rng.normal(0, 1, (M, D)).astype(np.float32))
    wo, o = bf(rng.normal(0, D ** -0.5, (N, D))), bf(rng.normal(0, 1, (M, N)))
    ch, cl, delta = empty(M * ld, "bf16"), empty(M * ld, "bf16"), zeros(HQ * M)
    A, B, Og = [dev(wide(t, pad), "bf16") for t in (dh, dl)], dev(wide(wo, pad), "bf16"), dev(wide(o, pad), "bf16")
    N_.api.sj_gemm_planes_split_out(None, M, N, D, A[0].p, A[1].p, D + pad, B.p, D + pad, ch.p, cl.p, ld, None, None, 0,
                                    Og.p, ld, delta.p, M)
    sync()
    r = edge_rows(M)
    got = (ch.host() + cl.host()).reshape(M, ld)[r, :N]
    assert rel(got, (dh[r].astype(np.float64) + dl[r]) @ wo.T) < 3e-5
    dref = (got * o[r]).reshape(len(r), HQ, 64).sum(2)
    assert rel(delta.host().reshape(HQ, M)[:, r].T, dref) < 1e-6


@pytest.mark.parametrize("M,K,N,pad", [(16384, 1024, 1024, 0), (16300, 520, 1000, 8)])
def test_residual(N_, M, K, N, pad):
    assert plan(RESIDUAL, M, N, K)[0] == PP
    rng = np.random.default_rng(M + N)
    x, w, res = bf(rng.normal(0, 1, (M, K))), bf(rng.normal(0, K ** -0.5, (N, K))), bf(rng.normal(0, 1, (M, N)))
    X, W, R, y = dev(wide(x, pad), "bf16"), dev(wide(w, pad), "bf16"), dev(wide(res, pad), "bf16"), empty(M * N, "bf16")
    N_.api.sj_linear_residual_fwd_t(None, X.p, K + pad, M, K, W.p, K + pad, N, R.p, N + pad, y.p, N)
    sync()
    r = edge_rows(M)
    close_bf(y.host().reshape(M, N)[r], res[r] + bf(x[r].astype(np.float64) @ w.T),
             np.abs(x[r]) @ np.abs(w.T) + 2.0 ** 8 * np.abs(res[r]))  # the product's own rounding may flip


@pytest.mark.parametrize("M,D,F,pad", [(8192, 1024, 2752, 0), (16384, 520, 1000, 8)])
def test_gate_up(N_, M, D, F, pad):
    assert plan(GATE_UP, M, F, D)[0] == PP
    rng = np.random.default_rng(M + D)
    x, wg, wu = (bf(rng.normal(0, s, sh)) for s, sh in ((1, (M, D)), (D ** -0.5, (F, D)), (D ** -0.5, (F, D))))
    X, WG, WU = (dev(wide(t, pad), "bf16") for t in (x, wg, wu))
    ld = F + pad
    g, u, h = (empty(M * ld, "bf16") for _ in range(3))
    N_.api.sj_gate_up_fwd_t(None, X.p, D + pad, M, D, WG.p, WU.p, D + pad, F, g.p, u.p, h.p, ld, None, 0)
    sync()
    r = edge_rows(M)
    G, U, H = (t.host().reshape(M, ld)[r, :F] for t in (g, u, h))
    close_bf(G, x[r].astype(np.float64) @ wg.T, np.abs(x[r]) @ np.abs(wg.T))
    close_bf(U, x[r].astype(np.float64) @ wu.T, np.abs(x[r]) @ np.abs(wu.T))
    close_bf(H, G / (1 + np.exp(-G)) * U, np.zeros_like(H))


def digests():
    """sha256 of each product's output at one shape (one K slice on both sides)."""
    from sejong_amd import _native as N
    N.load()
    M, K, C = 16300, 1032, 1000
    rng = np.random.default_rng(5)
    ah, al = split(rng.normal(0, 1, (M, K)).astype(np.float32))
    b, b2 = bf(rng.normal(0, 1, (C, K))), bf(rng.normal(0, 1, (C, K)))
    res = bf(rng.normal(0, 1, (M, C)))
    A, L, B, B2, R = (dev(t, "bf16") for t in (ah, al, b, b2, res))
    Mw, Nw, Kw = 1936, 4016, 1637
    yh, yl = split(rng.normal(0, 1, (Kw, Nw)).astype(np.float32))
    X, YH, YL = (dev(t, "bf16") for t in (bf(rng.normal(0, 1, (Kw, Mw))), yh, yl))
    kinds = [plan(DX, M, C, K), plan(RESIDUAL, M, C, K), plan(GATE_UP, M, C, K), plan(SPLIT_OUT, M, C, K),
             plan(DW, Mw, Nw, Kw)]
    dx, r, dw = empty(M * C), empty(M * C, "bf16"), empty(Mw * Nw)
    g, u, h, ch, cl = (empty(M * C, "bf16") for _ in range(5))
    N.api.sj_gemm_planes(None, M, C, K, A.p, L.p, K, B.p, None, K, dx.p, F32, C, 0, None, 0)
    N.api.sj_linear_residual_fwd_t(None, A.p, K, M, K, B.p, K, C, R.p, C, r.p, C)
    N.api.sj_gate_up_fwd_t(None, A.p, K, M, K, B.p, B2.p, K, C, g.p, u.p, h.p, C, None, 0)
    N.api.sj_gemm_planes_split_out(None, M, C, K, A.p, L.p, K, B.p, K, ch.p, cl.p, C, None, None, 0, None, 0, None, 0)
    N.api.sj_gemm_planes_tn(None, Mw, Nw, Kw, X.p, None, Mw, YH.p, YL.p, Nw, dw.p, F32, Nw, 0, None, 0)
    sync()
    return dict(kernels=[k[0] for k in kinds], slices=kinds[-1][3],
                **{n: hashlib.sha256(t.host().tobytes()).hexdigest()
                   for n, t in dict(dx=dx, r=r, g=g, u=u, h=h, ch=ch, cl=cl, dw=dw).items()})


def test_the_tiled_kernels_bits(N_):
    """k_gemm_pp against the kernels it replaces (SJ_GEMM_PP=0 in a child
    process): the same sums in the same order."""
    here = digests()
    env = {**os.environ, "SJ_GEMM_PP": "0"}
    out = subprocess.run([sys.executable, "-c", "import json; from tests.test_gpu_large_products import digests; "
                          "print(json.dumps(digests()))"], cwd=ROOT, env=env, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr[-2000:]
    there = json.loads(out.stdout.splitlines()[-1])
    assert here.pop("kernels") == [PP] * 5 and PP not in there.pop("kernels")
    assert here == there
