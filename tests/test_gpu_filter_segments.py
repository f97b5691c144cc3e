"""The numerical filter's level segments on small grids: segment remainders,
tile edges and the fewest levels and columns, bit for bit against the oracle."""
import pytest

import helpers as H
import pyoracle as po
from test_gpu_parity import hip  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(4, 3, 2), (5, 65, 5), (6, 64, 9), (7, 2, 4), (17, 67, 13), (33, 70, 6)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("tj", [0, 4, 8])
def test_filter_segments(hip, size, tj):  # noqa: F811
    print(f"[filter] {size} TJ={tj}", flush=True)
    case = H.small_case(kmax=size[0], imax=size[1], jmax=size[2], seed=41, stretched=(60.0, 200.0))
    m, st = case.metric, case.state
    ref = po.numfilter_coef(case, st, 1.5)
    got = case.grid.zeros(5, 3)
    with hip.Context(case.grid) as ctx:
        ctx.tune_set(hip.TUNE_NF_TJ, tj)
        ctx.ATMOS_DYN_numfilter_coef(got, st["DENS"], st["MOMZ"], st["MOMX"], st["MOMY"], st["RHOT"], m["CDZ"], m["CDX"],
                                     m["CDY"], m["FDZ"], m["FDX"], m["FDY"], 1.5, case.ref["REF_dens"],
                                     case.ref["REF_pott"], 1.0e-4, 1, 1.0, True)
    H.compare(ref, got, "num_diff")
