"""The tiled tracer kernels over level segments, flat and on general metrics:
segment remainders, tile edges and the fewest levels and columns, bit for bit
against the oracle; and models whose tracer stages take their densities from
the kernels' own RK3 interpolation."""
import numpy as np
import pytest

import helpers as H
import pyoracle as po
from scale_amd import inputs
from test_gpu_parity import hip  # noqa: F401
from test_gpu_tracer_tile import tracer_case

pytestmark = pytest.mark.gpu


# (kmax, imax, jmax): at most (kmax + 3) / 4 segments of at least 4 levels but the last; one column and one row past a tile
@pytest.mark.parametrize("size", [(4, 2, 2), (5, 65, 9), (9, 64, 8), (13, 63, 17), (34, 33, 7)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("terrain", [False, True], ids=["flat", "terrain"])
@pytest.mark.parametrize("mode", [(True, True), (True, False), (False, False)], ids=["fct_along", "fct_7pt", "nofct"])
@pytest.mark.parametrize("scheme", [3, 4, 31, 1], ids=["UD3", "CD4", "UD3KOREN1993", "UD1"])
def test_tracer_segments(hip, size, terrain, mode, scheme):  # noqa: F811
    print(f"[tracer segments] {size} terrain={terrain} {mode} scheme={scheme}", flush=True)
    case, inp = tracer_case(scheme, size[1], size[2], size[0], 4300)
    if terrain:
        case = inputs.Case(**{**case.__dict__, "metric": H.terrain_metrics(case)})
    g, m = case.grid, case.metric
    ref = np.full(g.shape, np.nan, order="F")
    po.tstep_tracer(case, ref, inp["QTRC"], inp["QTRC0"], inp["RHOQ_t"], inp["DENS0"], inp["DENS"], inp["mflx"],
                    inp["nd"], 1.5, *mode, scheme=scheme)
    got = np.full(g.shape, np.nan, order="F")
    with hip.Context(g, case.scheme, scheme) as ctx:
        ctx.tune_set(hip.TUNE_TRACER_TILE, 2)
        ctx.ATMOS_DYN_Tstep_tracer_fvm_heve(got, inp["QTRC"], inp["QTRC0"], inp["RHOQ_t"], inp["DENS0"], inp["DENS"],
                                            inp["mflx"], inp["nd"], m["GSQRT"],
                                            np.asfortranarray(m["MAPF"][:, :, :, 0]), m["CDZ"], m["RCDZ"], m["RCDX"],
                                            m["RCDY"], 1.5, *mode)
    H.compare(ref, got, "QTRCo")


@pytest.mark.parametrize("terrain", [False, True], ids=["flat", "terrain"])
def test_model_tracers(hip, terrain):  # noqa: F811
    """Three large steps of one short step each, tiles and per-point kernels:
    the same tracers, bit for bit."""
    print(f"[tracer segments] model terrain={terrain}", flush=True)
    case = H.small_case(kmax=19, imax=67, jmax=10, seed=43, dz=100.0)
    zs = inputs.bell_topography(case.grid, height=60.0, half_width=1500.0) if terrain else None
    got = []
    for tile in (0, 2):
        with hip.model_from_case(case, zsfc=zs) as ctx:
            ctx.tune_set(hip.TUNE_TRACER_TILE, tile)
            ctx.model_large_step(3)
            got.append([ctx.model_get(hip.QTRC_BASE + n) for n in range(case.qtrc.shape[-1])])
    for a, b in zip(*got):
        assert np.array_equal(a, b)


def ensemble_tracers(hip, sizes, scheme, fct):  # noqa: F811
    """Two large steps of an ensemble: each member's tracers bit-identical to its own model's."""
    cases = [inputs.make_case(kmax=k, imax=i, jmax=j, noise=0.01, ntracer=2, tracer_kind=["blob", "tophat"], fct=fct,
                              momz_noise=0.05, v0=-2.0, scheme_tracer=scheme, halo=3 if scheme == 5 else 2)
             for k, i, j in sizes]
    alone = [hip.model_from_case(c) for c in cases]
    members = [hip.model_from_case(c) for c in cases]
    try:
        with hip.Ensemble(members) as ens:
            ens.large_step(2)
            ens.synchronize()
            for x, y in zip(alone, members):
                x.model_large_step(2)
                for n in range(2):
                    assert np.array_equal(x.model_get(hip.QTRC_BASE + n), y.model_get(hip.QTRC_BASE + n))
    finally:
        for ctx in alone + members:
            ctx.close()


@pytest.mark.parametrize("scheme", [3, 5], ids=["UD3", "UD5"])
def test_ensemble_tracers_without_fct(hip, scheme):  # noqa: F811
    """An ensemble of few columns without FCT: every stage per point."""
    print(f"[tracer segments] ensemble without FCT, scheme {scheme}", flush=True)
    ensemble_tracers(hip, ((9, 12, 10), (14, 67, 6)), scheme, False)


@pytest.mark.parametrize("scheme", [3, 31], ids=["UD3", "Koren"])
@pytest.mark.parametrize("fct", [False, True], ids=["plain", "fct"])
def test_ensemble_tracers_on_tiles(hip, scheme, fct):  # noqa: F811
    """An ensemble of two tiles of 64 x 4 columns per CU and more: the stages
    without FCT on the tiles too."""
    print(f"[tracer segments] ensemble on tiles, scheme {scheme}, fct={fct}", flush=True)
    ensemble_tracers(hip, ((9, 12, 10), (6, 67, 1030)), scheme, fct)
