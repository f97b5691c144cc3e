"""Tendencies given to a model after steps without any, against the oracle, and
settings given to the members of an ensemble after its creation, against the
members' own models."""
import numpy as np
import pytest

import helpers as H
import pyoracle as po
from scale_amd import inputs
from test_gpu_parity import hip  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("split", ["0", "1"], ids=["tile", "split"])
def test_tendencies_given_later(hip, split, monkeypatch):  # noqa: F811
    """Two steps without tendencies, which the stage then does not read, then
    two with them: 1e-12 of the oracle."""
    monkeypatch.setenv("SCALE_HIP_FLAT_SPLIT", split)
    case = H.small_case(kmax=10, imax=9, jmax=6, seed=43)
    g = case.grid
    rng = np.random.Generator(np.random.PCG64(8))
    tp = {}
    for v in hip.STATE:
        a = g.zeros()
        a[:, g.IS:g.IE + 1, g.JS:g.JE + 1] = 1e-3 * rng.standard_normal((g.KA, g.imax, g.jmax))
        tp[v + "_tp"] = inputs.halo_fill(g, a)
    m = po.Model(case)
    m.step(2)
    later = po.Model(inputs.Case(**{**case.__dict__, "zero_tend": {**case.zero_tend, **tp}}))
    later.state = {k: np.array(v, order="F", copy=True) for k, v in m.state.items()}
    later.qtrc = np.array(m.qtrc, order="F", copy=True)
    later.step(2)
    with hip.model_from_case(case) as ctx:
        ctx.model_large_step(2)
        for k, v in tp.items():
            ctx.model_set(k, v)
        ctx.model_large_step(2)
        for k in hip.STATE:
            ref = later.state[k]
            assert np.abs(ctx.model_get(k) - ref).max() <= 1e-12 * np.abs(ref).max(), k


@pytest.mark.parametrize("mixed", [False, True], ids=["fp64", "mixed"])
@pytest.mark.parametrize("nstep", [1, 3])
def test_tendencies_given_to_a_replayed_ensemble(hip, mixed, nstep):  # noqa: F811
    """An ensemble replaying its captured step is given tendencies: each member
    stays bit-identical to its own model, with one short step and with three
    a large step (the mean of the mass fluxes that the tracers take)."""
    cases = [H.small_case(kmax=10, imax=9, jmax=6, seed=44), H.small_case(kmax=12, imax=66, jmax=5, seed=45)]
    kw = dict(mixed_precision=mixed, dtl=nstep * 0.5)
    rng = np.random.Generator(np.random.PCG64(9))
    tps = []
    for case in cases:
        g = case.grid
        a = g.zeros()
        a[:, g.IS:g.IE + 1, g.JS:g.JE + 1] = 1e-3 * rng.standard_normal((g.KA, g.imax, g.jmax))
        tps.append(inputs.halo_fill(g, a))
    alone = [hip.model_from_case(c, **kw) for c in cases]
    members = [hip.model_from_case(c, **kw) for c in cases]
    try:
        with hip.Ensemble(members) as ens:
            ens.set_graph(True)
            for given in (False, True):
                for ctx, tp in zip(alone + members, tps + tps):
                    if given:
                        ctx.model_set("RHOT_tp", tp)
                for ctx in alone:
                    ctx.model_large_step(2)
                ens.large_step(2)
                ens.synchronize()
                for case, x, y in zip(cases, alone, members):
                    for f in hip.STATE + ("mflx_hi",) + tuple(hip.QTRC_BASE + n for n in range(case.qtrc.shape[-1])):
                        assert np.array_equal(x.model_get(f), y.model_get(f)), (given, f)
    finally:
        for ctx in alone + members:
            ctx.close()


@pytest.mark.parametrize("graph", [False, True], ids=["direct", "replayed"])
@pytest.mark.parametrize("fct", [False, True], ids=["plain", "fct"])
@pytest.mark.parametrize("scheme", [3, 6], ids=["UD3", "CD6"])
def test_settings_given_to_an_ensemble(hip, graph, fct, scheme):  # noqa: F811
    """Members are given a tracer tendency (UD3: tracers in batched launches, CD6: on their own) and the Coriolis
    parameter after steps without, and the parameter's zeros again after that: each stays bit-identical to its own
    model."""
    kw = dict(scheme_tracer=scheme, fct=fct, halo=3 if scheme == 6 else 2)
    cases = [H.small_case(kmax=10, imax=9, jmax=6, seed=46, **kw), H.small_case(kmax=12, imax=66, jmax=5, seed=47, **kw)]
    rng = np.random.Generator(np.random.PCG64(10))
    tps = []
    for case in cases:
        g = case.grid
        a = g.zeros()
        a[:, g.IS:g.IE + 1, g.JS:g.JE + 1] = 1e-3 * rng.standard_normal((g.KA, g.imax, g.jmax))
        tps.append(inputs.halo_fill(g, a))
    alone = [hip.model_from_case(c) for c in cases]
    members = [hip.model_from_case(c) for c in cases]
    try:
        with hip.Ensemble(members) as ens:
            ens.set_graph(graph)
            for given in ("nothing", "RHOQ_tp", "CORIOLI", "zeros"):
                for case, ctx, tp in zip(cases + cases, alone + members, tps + tps):
                    if given == "RHOQ_tp":
                        ctx.model_set(hip.RHOQ_TP_BASE + 1, tp)
                    elif given != "nothing":
                        ctx.model_set("CORIOLI", np.full(case.corioli.shape, 1e-2 if given == "CORIOLI" else 0.0, order="F"))
                for ctx in alone:
                    ctx.model_large_step(2)
                ens.large_step(2)
                ens.synchronize()
                for case, x, y in zip(cases, alone, members):
                    for f in hip.STATE + tuple(hip.QTRC_BASE + n for n in range(case.qtrc.shape[-1])):
                        assert np.array_equal(x.model_get(f), y.model_get(f)), (given, f)
    finally:
        for ctx in alone + members:
            ctx.close()
