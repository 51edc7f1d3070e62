"""The bytes bench.py divides a step's time into, against the launches a captured
chain of steps is made of."""
import pytest

import bench


@pytest.mark.parametrize("sf", [8, 4])
@pytest.mark.parametrize("steps,warmup,graph,chained", [(8, 5, True, 7), (20, 5, True, 14), (20, 5, False, 0),
                                                        (7, 1, True, 0), (8, 0, True, 0), (9, 0, True, 7)])
def test_captured_step_bytes(steps, warmup, graph, chained, sf):
    n, t = 64, 22
    kept, xcol, cs = (2 * t - 1) ** 2 * t, n * (2 * t - 1) * t, 2 * sf
    per = {k: bench.kernel_bytes(k, n, 30, 1309, sf) for k in ("x_zeta2u_inv", "z_adv", "x_f_zeta")}
    table = {k: {"bytes_per_launch": b, "launches": steps} for k, b in per.items()}
    # every step has z_adv and x_f_zeta (whose chained form writes three components more), a chained
    # step's successor no x_zeta2u_inv (two zeta components read, three columns' components written)
    want = (steps * (per["z_adv"] + per["x_f_zeta"]) + chained * cs * 3 * xcol
            + (steps - chained) * cs * (2 * kept + 3 * xcol))
    got = steps * bench.pipeline_step_bytes(table, n, sf, steps, warmup, graph)
    assert abs(got - want) < 1e-9 * want
