"""RMSNorm's row kernels at the edges of their forms: widths around the
column-pair steps, row counts around a workgroup's 16 and the reduction's
128 groups, mixed types, and the gradient accumulated in place."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_util import assert_stored_close, dev, empty, rel, sync

pytestmark = pytest.mark.gpu
DT = {"f32": 0, "bf16": 4}


@pytest.mark.parametrize("R,D", [(1, 2), (15, 126), (17, 128), (16, 130), (2100, 258), (70, 512), (33, 514), (2048, 770),
                                 (19, 1024), (35, 1026), (5, 2048)])
@pytest.mark.parametrize("xd,wd", [("f32", "f32"), ("bf16", "bf16"), ("f32", "bf16"), ("bf16", "f32")])
def test_rmsnorm_shapes(R, D, xd, wd):
    from sejong_amd import _native as N
    lib, eps, cf = N.load(), 1e-6, ctypes.c_float
    rng = np.random.default_rng(R + D)
    x, w = O.round_to(rng.normal(0, 1, (R, D)), xd), O.round_to(rng.normal(1, 0.1, D), wd)
    dy, acc = (rng.normal(0, 1e-3, (R, D)).astype(np.float32).astype(np.float64) for _ in range(2))
    X, W, DY, A, Y = dev(x, xd), dev(w, wd), dev(dy), dev(acc), empty(R * D, xd)
    N.api.sj_rmsnorm_fwd(None, X.p, DT[xd], W.p, DT[wd], Y.p, R, D, cf(eps))
    wb = lib.sj_rmsnorm_bwd_workspace_bytes(R, D)
    ws, DX, DW = empty(max(wb, 256), "u8"), empty(R * D), empty(D)
    N.api.sj_rmsnorm_bwd(None, X.p, DT[xd], W.p, DT[wd], DY.p, None, DX.p, DW.p, R, D, cf(eps), ws.p, ws.nbytes)
    sync()
    assert_stored_close(Y.host(), O.rmsnorm_fwd(x, w, eps), xd, "rmsnorm y")
    dx, dw = O.rmsnorm_bwd(x, w, dy, eps)
    # a row's dx is a difference of terms of the size of dy; fp32 sums of d and of R terms
    assert np.linalg.norm(DX.host() - dx.ravel()) < 1e-5 * np.linalg.norm(dy) * max(1.0, np.abs(w).max())
    assert rel(DW.host(), dw) < 1e-5
    N.api.sj_rmsnorm_bwd(None, X.p, DT[xd], W.p, DT[wd], DY.p, A.p, A.p, DW.p, R, D, cf(eps), ws.p, ws.nbytes)
    sync()
    # acc + inv * (...) may be one fma: the product's rounding (2^-24 of dx) is
    # left out, and each side rounds its sum once
    dxh, a0 = DX.host().ravel().astype(np.float64), acc.ravel()
    assert (np.abs(A.host().ravel() - (a0 + dxh)) <= 2.0 ** -23 * (np.abs(a0) + np.abs(dxh))).all()
    assert rel(DW.host(), dw) < 1e-5
