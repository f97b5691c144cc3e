"""The FP32 stage's tiles of 4 and of 8 rows (more than one 64 x 8 tile per CU)
give one field: a wide periodic state of identical rows of columns comes out
identical on a grid of 4-row tiles and on one of 8-row tiles."""
import numpy as np
import pytest

import helpers as H
from scale_amd import inputs
from test_gpu_parity import hip  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kmax,rows", [(4, 9), (9, 14)])
def test_tile_rows(hip, kmax, rows):  # noqa: F811
    """rows x 70 columns, and the same rows repeated northward until the 64 x 8
    tiles outnumber the CUs: each repeat equals the small grid."""
    print(f"[fp32 tiles] {kmax} levels, {rows} rows", flush=True)
    small = H.small_case(kmax=kmax, imax=70, jmax=rows, seed=61, dz=100.0)
    rep = 8 * 300 // rows
    wide = H.small_case(kmax=kmax, imax=70, jmax=rows * rep, seed=61, dz=100.0)
    gs, gw = small.grid, wide.grid
    src = gs.JS + np.arange(gw.jmax) % rows
    for k in hip.STATE:
        wide.state[k][:, :, gw.JS:gw.JE + 1] = small.state[k][:, :, src]
        inputs.halo_fill(gw, wide.state[k])
    for n in range(wide.qtrc.shape[-1]):
        wide.qtrc[:, :, gw.JS:gw.JE + 1, n] = small.qtrc[:, :, src, n]
        inputs.halo_fill(gw, wide.qtrc[..., n])
    out = []
    for case in (small, wide):
        with hip.model_from_case(case, mixed_precision=True) as ctx:
            ctx.model_short_step(2)
            out.append({k: ctx.model_get(k) for k in hip.STATE})
    for k in hip.STATE:
        a = out[0][k][:, gs.IS:gs.IE + 1, src]
        b = out[1][k][:, gw.IS:gw.IE + 1, gw.JS:gw.JE + 1]
        assert np.array_equal(a, b), k
