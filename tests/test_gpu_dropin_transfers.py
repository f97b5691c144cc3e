"""The drop-in stage's transfers through pinned slots (calls of 32 MB and more:
partial last chunks, arrays of several chunks and of one) and its look at the
metrics (terrain seen before the uploads and after them), bit for bit against the oracle."""
import numpy as np
import pytest

import helpers as H
from test_gpu_parity import OUTS, hip, oracle_stage, run_stage_gpu  # noqa: F401

pytestmark = pytest.mark.gpu


# (kmax, imax, jmax): a call below 32 MB, array by array; arrays of 0.9 MB, num_diff of four chunks; of 4.1 MB, two
# chunks, and more columns than the first look at the metrics takes
@pytest.mark.parametrize("size", [(9, 12, 10), (40, 47, 48), (60, 91, 85)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("metric", ["flat", "terrain", "one element"])
def test_stage_transfers(hip, size, metric):  # noqa: F811
    print(f"[drop-in] {size} {metric}", flush=True)
    case = H.small_case(kmax=size[0], imax=size[1], jmax=size[2], seed=51, dz=80.0)
    g = case.grid
    inp = H.stage_inputs(case, seed=52, coriolis=True)
    m = None
    if metric == "terrain":
        m = H.terrain_metrics(case)
    elif metric == "one element":  # the last interior element of the last array looked over
        m = {k: np.array(v, order="F", copy=True) for k, v in case.metric.items()}
        m["J23G"][g.KE, g.IE, g.JE, :] = 0.01
    ref = oracle_stage(case, inp, 0.5, m)
    got = run_stage_gpu(hip, case, inp, 0.5, m)
    for k in OUTS:
        H.compare(ref[k], got[k], k)
