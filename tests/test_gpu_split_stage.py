"""The split FP64 stage (hevi_etile + hevi_columns) at the sizes where it can go
wrong: tile, segment and column-block edges, remainders, the fewest levels, and
level counts on both sides of every column-block width, bit for bit against the
oracle; the RK4 combination fused into both kernels; the rule that chooses
between them and the tile kernel on flat grids."""
import numpy as np
import pytest

import helpers as H
import pyoracle as po
from scale_amd import inputs
from test_gpu_parity import OUTS, hip, oracle_stage, run_stage_gpu  # noqa: F401

pytestmark = pytest.mark.gpu

# (kmax, imax, jmax): the fewest levels and columns; one column past a 32-column tile; one row past a tile; the
# column blocks of hevi_columns: 260 rows of 9 to 18 columns take the widest block that fits (32 columns up to 64
# levels, 16 up to 256, 8 beyond, with 102, 131, 66 and 66 KB of LDS at 200, 256, 257 and 258 levels), grids of few
# columns 8 a block up to 512 levels, any grid 4 up to 1024, 2 up to 2048, 1 up to 4096 and the one-launch march
# beyond; 129 tiles of 64 columns (the wide tile)
SIZES = [(4, 2, 2), (5, 33, 9), (9, 31, 17), (6, 33, 130), (64, 18, 260), (65, 18, 130), (129, 9, 4), (200, 17, 130),
         (256, 17, 130), (257, 6, 3), (257, 17, 130), (258, 17, 130), (512, 7, 5), (513, 7, 5), (1024, 5, 3), (1025, 3, 5),
         (2049, 3, 2), (4096, 2, 3), (4097, 2, 2), (5, 65, 520)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("terrain", [False, True], ids=["flat", "terrain"])
@pytest.mark.parametrize("scheme", [3, 4], ids=["UD3", "CD4"])
def test_stage_sizes(hip, size, terrain, scheme, monkeypatch):  # noqa: F811
    monkeypatch.setenv("SCALE_HIP_FLAT_SPLIT", "1")
    print(f"[split stage] {size} terrain={terrain} scheme={scheme}", flush=True)
    case = H.small_case(kmax=size[0], imax=size[1], jmax=size[2], seed=31, dz=min(80.0, 15000.0 / size[0]))
    inp = H.stage_inputs(case, seed=29, coriolis=True)
    inp["wdamp_coef"] = np.linspace(0.0, 0.01, case.grid.KA)
    inp["divdmp_coef"] = 0.1 if size[2] % 2 else 0.0
    inp["DDIV"] = np.asfortranarray(np.random.Generator(np.random.PCG64(4)).standard_normal(case.grid.shape) * 1e-3)
    metric = H.terrain_metrics(case) if terrain else None
    ref = oracle_stage(case, inp, 0.5, metric, scheme)
    got = run_stage_gpu(hip, case, inp, 0.5, metric, scheme)
    for k in OUTS:
        H.compare(ref[k], got[k], k)


@pytest.mark.parametrize("size", [(4, 2, 2), (9, 65, 9), (33, 30, 7), (70, 33, 6), (520, 5, 3)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("terrain", [False, True], ids=["flat", "terrain"])
@pytest.mark.parametrize("forced", [False, True], ids=["plain", "forced"])
def test_fused_combination(hip, size, terrain, forced, monkeypatch):  # noqa: F811
    """Three large steps through the combining fourth stage, without and with
    divergence damping, Coriolis force and sponge layer, within 1e-12 of each
    field's scale (pow() in the preparation)."""
    monkeypatch.setenv("SCALE_HIP_FLAT_SPLIT", "1")
    print(f"[split stage] model {size} terrain={terrain} forced={forced}", flush=True)
    case = H.small_case(kmax=size[0], imax=size[1], jmax=size[2], seed=37, dz=min(100.0, 15000.0 / size[0]))
    divdmp = 0.2 if forced else 0.0
    if forced:
        case.corioli[:] = 1.0e-2
        case.wdamp_coef[:] = np.linspace(0.0, 0.01, case.grid.KA)
    zs = inputs.bell_topography(case.grid, height=60.0, half_width=1500.0) if terrain else None
    ocase = case
    if terrain:
        ocase = inputs.Case(**{**case.__dict__, "metric": {**case.metric, **po.terrain_metrics(case.grid, zs, case.fz, case.metric)}})
    m = po.Model(ocase, divdmp_coef=divdmp)
    m.step(3)
    g = case.grid
    sl = (slice(g.KS, g.KE + 1), slice(g.IS, g.IE + 1), slice(g.JS, g.JE + 1))
    with hip.model_from_case(case, zsfc=zs, divdmp_coef=divdmp) as ctx:
        ctx.model_large_step(3)
        for k in hip.STATE:
            got, ref = ctx.model_get(k), m.state[k]
            assert np.abs(got - ref).max() <= 1e-12 * max(np.abs(ref).max(), 1.0), k  # ghost levels and halos too
        for k in ("mflx_hi", "tflx_hi"):
            got, ref = ctx.model_get(k)[sl], getattr(m, k)[sl]
            assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max(), k


@pytest.mark.parametrize("rows", [1840, 1848, 2049, 3680, 3688])
def test_flat_route(hip, rows, monkeypatch):  # noqa: F811
    """The rule between the tile kernel and the split launches left alone, on
    256 CUs: 230 tiles of 64 x 8 columns | 231 (90 % of a round), 257 and 460 |
    461 (90 % of two).  A stage bit for bit the oracle's, two large steps
    within 1e-12 of each field's scale."""
    monkeypatch.delenv("SCALE_HIP_FLAT_SPLIT")
    print(f"[split stage] flat route, {rows} rows", flush=True)
    case = H.small_case(kmax=5, imax=3, jmax=rows, seed=39, dz=100.0)
    inp = H.stage_inputs(case, seed=29, coriolis=True)
    ref, got = oracle_stage(case, inp, 0.5), run_stage_gpu(hip, case, inp, 0.5)
    for k in OUTS:
        H.compare(ref[k], got[k], k)
    m = po.Model(case)
    m.step(2)
    with hip.model_from_case(case) as ctx:
        ctx.model_large_step(2)
        for k in hip.STATE:
            assert np.abs(ctx.model_get(k) - m.state[k]).max() <= 1e-12 * max(np.abs(m.state[k]).max(), 1.0), k
