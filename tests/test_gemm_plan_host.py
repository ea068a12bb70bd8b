"""The products' dispatch rules through sj_gemm_planes_plan (no GPU: the rules
are host arithmetic, with 256 CUs assumed)."""
import ctypes
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DX, DW, GATE_UP, RESIDUAL, SPLIT_OUT, COEFFICIENTS = range(6)
FAST, KW, PP = range(3)


def plan(op, M, N, K):
    """(kernel, tile rows, tile columns, K slices)"""
    from sejong_amd import _native as N_
    v = [ctypes.c_int() for _ in range(3)]
    k = N_.load().sj_gemm_planes_plan(op, M, N, K, *map(ctypes.byref, v))
    assert k >= 0
    return (k,) + tuple(x.value for x in v)


# one product of each kind that k_gemm_pp (or a tall coefficient tile) takes by itself
LARGE = [(DX, 16384, 1024, 5504), (DW, 1024, 5504, 16384), (GATE_UP, 16384, 2752, 1024), (RESIDUAL, 16384, 1024, 2752),
         (SPLIT_OUT, 8192, 1024, 1024), (COEFFICIENTS, 144, 5504, 16384), (DW, 504, 1440, 11264)]


def plans_under(**env):
    code = ("import json; from tests.test_gemm_plan_host import LARGE, plan; "
            "print(json.dumps([plan(*x) for x in LARGE]))")
    clean = {k: v for k, v in os.environ.items() if not k.startswith("SJ_GEMM_")}
    out = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env={**clean, **env}, check=True, capture_output=True,
                         text=True, timeout=300).stdout
    return [tuple(x) for x in json.loads(out.splitlines()[-1])]


def test_sweep_overrides_reach_the_large_products():
    free = plans_under()
    assert [p[0] for p in free] == [PP, PP, PP, PP, PP, FAST, PP]
    assert free[5][1:3] != (64, 64)
    assert all(p[0] != PP for p in plans_under(SJ_GEMM_PP="0"))
    assert plans_under(SJ_GEMM_PP="0")[5] == free[5]
    tile = plans_under(SJ_GEMM_TILE="128x64")
    assert [p[:3] for p in tile] == [(FAST, 128, 64)] + [(FAST, 128, 64)] * 5 + [(KW, 64, 64)]
    splits = plans_under(SJ_GEMM_SPLITS="3")
    assert all(p[0] != PP for p in splits) and splits[0][3] == splits[5][3] == 3
    assert plans_under(SJ_GEMM_LK_TILE="64x128", SJ_GEMM_LK_SPLITS="5")[5] == (FAST, 64, 128, 5)
    for env in (dict(SJ_GEMM_KW="0"), dict(SJ_GEMM_DW_SPLITS="3"), dict(SJ_GEMM_DW_TILE="64x64")):
        got = plans_under(**env)
        assert got[1][0] != PP and got[6][0] != PP and got[0] == free[0]
    assert plans_under(SJ_GEMM_KW="0")[6][0] == FAST
    assert plans_under(SJ_GEMM_KW_SPLITS="2")[6] == (KW, 64, 64, 2)
    assert all(p[0] != PP for p in plans_under(SJ_GEMM_STAGES="2"))
