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


# measured on an MI355X, us: the kernels before k_gemm_pp, k_gemm_pp
@pytest.mark.parametrize("M,N,K,old,pp", [
    (112, 88, 2447, 22, 35), (904, 312, 2769, 25, 42), (648, 416, 2912, 26, 45), (120, 80, 7947, 22, 35),
    (664, 264, 21918, 51, 73), (1912, 80, 38089, 84, 119), (3040, 128, 35146, 92, 114), (104, 5672, 3337, 29, 35),
    (320, 5600, 7001, 85, 95), (656, 72, 25112, 54, 85), (1024, 1024, 4096, 29, 42), (2752, 1024, 2048, 31, 43),
    (1024, 5504, 16384, 655, 399), (2752, 1024, 16384, 219, 212), (1024, 1536, 16384, 181, 101),
    (232, 3408, 30458, 238, 116), (4320, 144, 18282, 134, 80), (2056, 552, 37632, 551, 200), (504, 1440, 11264, 71, 49),
    (5288, 816, 768, 40, 27), (5936, 4840, 12544, 2056, 1308)])
def test_dw_products_take_the_faster_kernel(M, N, K, old, pp):
    assert (plan(DW, M, N, K)[0] == PP) == (pp < old)


@pytest.mark.parametrize("M,N,K,old,pp", [
    (11537, 864, 3368, 177, 190), (12699, 5720, 400, 272, 298), (23308, 456, 3928, 225, 259), (5532, 1816, 3816, 206, 218),
    (16562, 656, 5832, 322, 335), (4096, 1024, 384, 19, 24), (16384, 2752, 1024, 278, 228), (8000, 2048, 768, 97, 74),
    (1206, 4784, 3512, 124, 93), (28568, 176, 5952, 196, 144), (4472, 1040, 4184, 146, 114), (15200, 2584, 400, 156, 115),
    (9079, 848, 720, 44, 34)])
def test_gate_up_products_take_the_faster_kernel(M, N, K, old, pp):
    assert (plan(GATE_UP, M, N, K)[0] == PP) == (pp < old)


@pytest.mark.parametrize("M,N,K,general,tall", [
    (55, 472, 49920, 37, 52), (176, 256, 65536, 46, 66), (48, 1024, 16384, 19, 24), (112, 512, 8192, 15, 18),
    (96, 768, 12000, 19, 22), (115, 104, 68408, 48, 78), (360, 320, 35624, 40, 48), (432, 576, 28104, 63, 71),
    (386, 768, 46400, 108, 127), (144, 5504, 16384, 159, 117), (144, 2752, 16384, 76, 67), (272, 2048, 16384, 84, 65),
    (144, 1536, 16384, 42, 39), (154, 4784, 14832, 157, 101), (122, 2504, 64032, 287, 195), (144, 1024, 16384, 35, 30)])
def test_coefficient_products_take_the_faster_tile(M, N, K, general, tall):
    _, bm, bn, splits = plan(COEFFICIENTS, M, N, K)
    assert ((bm, bn) != (64, 64)) == (tall < general)
    # no slice more than twice the general plan's: its sums' error grows with the length
    t = -(-M // 64) * -(-N // 64)
    assert 2 * splits >= min(max(4 * 256 // t, 8), 16)
