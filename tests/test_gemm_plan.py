"""The dispatch of dense products (inferc_hip_gemm_plan, host only): that the shapes of
the GPU tests run the kernels they are there for, and the grid of the widest products."""
from __future__ import annotations

import ctypes as C
import random

import pytest

from inferc_amd import lib as L
from tests import test_gpu_gemm_tile as T

CUS = 256  # MI355X


def plan(M, N, K, ta=0, tb=0, batch=1, cus=CUS):
    out = (C.c_int64 * 6)()
    aligned = (M if ta else K) % 4 == 0 and (K if tb else N) % 4 == 0
    L.check(L.load_library().inferc_hip_gemm_plan(ta, tb, M, N, K, batch, int(aligned), cus, out))
    return dict(zip(("rows", "cols", "splits", "groups", "x", "z"), out))


def form(*shape, **kw):
    p = plan(*shape, **kw)
    return "small" if p["groups"] == 0 else f"{p['rows']}x{p['groups']}"


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_edge_shapes_run_the_tiles_they_name(ta, tb):
    forms = [form(*s, ta=ta, tb=tb) for s in T.EDGES_64]
    assert set(forms) == {"64x1", "64x2"}
    assert {form(*s, ta=ta, tb=tb) for s in T.EDGES_128} == {"128x1"}
    # K below, at and above the fp16 path's least K, whole and ragged panels
    assert any(s[2] < 64 for s in T.EDGES_128) and any(s[2] > 64 for s in T.EDGES_128)
    assert any(s[2] == 64 for s in T.EDGES_128)


def test_small_m_shapes_run_every_form():
    got = {tuple(list(plan(*s, tb=tb).values())[:4]) for s in T.SMALL for tb in (0, 1)}
    small = {g[:3] for g in got if g[3] == 0}
    assert small == {(16, 16, 1), (16, 32, 1), (16, 48, 2), (32, 48, 1), (32, 64, 1)}
    assert any(g[3] == 2 for g in got)  # the tiles that replace them


def test_value_shapes_reach_every_kernel():
    for shapes in (T.RANGES, T.MEETS):
        got = {form(*s, tb=tb) for s in shapes for tb in (0, 1)}
        assert {"small", "64x2", "128x1"} <= got
    got = {(form(M, N, K, ta=ta, tb=tb), tb) for ta, tb, M, N, K in T.INFINITIES}
    assert got >= {("small", 0), ("small", 1), ("64x2", 0), ("128x1", 0), ("128x1", 1)}
    assert {form(*s) for s in T.EPILOGUES} >= {"64x2", "64x1", "128x1"}
    assert any(form(*s) == "128x1" and s[2] < 64 for s in T.EPILOGUES)


@pytest.mark.parametrize("K", [32, 64, 256, 640, 768, 1024])
def test_small_m_kernel_up_to_one_block_per_cu(K):
    """Blocks of 32 rows by 48 columns, or 64 where N is no multiple of 48; above one a CU
    the 64x64 tiles are faster at every K below 2048."""
    for M, N in [(128, 3072), (160, 2304), (512, 768), (128, 4096), (256, 2048), (168, 768)]:
        assert form(M, N, K) == "small", (M, N)
    for M, N in [(129, 3072), (512, 3072), (192, 2304), (129, 4096), (257, 2048), (300, 2308)]:
        assert form(M, N, K) != "small", (M, N)
        assert form(M, N, K, tb=1) != "small", (M, N)


def test_small_m_kernel_16_row_blocks_transposed():
    """Above one block a CU, tiles for a short K with B transposed alone."""
    for M, N in [(64, 2304), (64, 3072), (256, 768)]:
        assert form(M, N, 256, tb=1) == "64x2" and form(M, N, 32, tb=1) == "64x1"
        assert form(M, N, 260, tb=1) == form(M, N, 256) == form(M, N, 32) == "small"
    assert form(64, 2048, 256, tb=1) == "small"  # 256 blocks


def test_long_k_transposed():
    """Tiles above 128 rows, but up to K = 3072 not where 16x16 blocks take the product."""
    for K in (2048, 3072):
        assert form(200, 64, K, tb=1) == form(132, 4, K, tb=1) == form(200, 768, K) == "small"
        assert form(128, 768, K, tb=1) == "small" and form(132, 256, K, tb=1) == "64x2"
    assert form(200, 64, 3076, tb=1) == "64x2"


def test_one_panel_has_one_group():
    for M, N in [(516, 64), (600, 600), (204, 5903)]:
        assert form(M, N, 32, ta=1) == form(M, N, 24, ta=1) == "64x1"
        assert form(M, N, 33, ta=1) == "64x2"


def test_few_tiles_split_k():
    assert plan(64, 63, 1500)["splits"] == 7 and plan(64, 63, 575)["splits"] == 1
    assert plan(600, 256, 1000)["splits"] == 5  # 40 tiles
    assert plan(700, 700, 768)["splits"] == 1  # 121 tiles: no CU is idle
    assert plan(512, 768, 3072, tb=1)["splits"] == 4


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
def test_partial_sums_fit_the_scratch(ta, tb):
    """A context starts with 16 MiB of workspace, and the allocation-free entry point has no
    more: the partial sums of any product fit, so that none is refused under capture."""
    rng = random.Random(ta + 2 * tb)
    for _ in range(4000):
        M, N, K = (int(round(2 ** rng.uniform(0, top))) for top in (13, 13, 15))
        if rng.random() < 0.5:
            M, N, K = (max(4, x // 4 * 4) for x in (M, N, K))
        p = plan(M, N, K, ta=ta, tb=tb)
        if p["groups"] == 0:  # whole tiles, one for each of the z blocks
            M, N = -(-M // p["rows"]) * p["rows"], -(-N // p["cols"]) * p["cols"]
        if p["splits"] > 1:
            assert 4 * p["splits"] * M * N <= 16 << 20, (M, N, K, p)


@pytest.mark.parametrize("M,N", [(1, 2 ** 31 - 65), (64, 2 ** 30 + 1), (100, 2 ** 31 - 65),
                                 (128, 2 ** 30 + 77), (4096, 3072), (4 * 10 ** 6, 65)])
def test_grid_dimensions_stay_below_2_32_threads(M, N):
    """One K and 2^30 columns and more: accepted, so the grid has to hold the tiles."""
    p = plan(M, N, 1)
    threads = 256 if (p["rows"], p["groups"]) == (64, 1) else 512
    tiles = -(-M // p["rows"]) * -(-N // p["cols"])
    assert p["x"] * threads < 2 ** 32 and p["x"] * p["z"] >= tiles > p["x"] * (p["z"] - 1)
    assert p["z"] < 65536
