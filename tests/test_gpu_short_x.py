"""x axes of 8 and 12 points: a line sits whole in one lane of the fused x
passes, whose wavenumbers are constants there. Plain, squirmer and sheared
steps against the oracle (FP64) and against FP64 (mixed), that they are the
fused steps asked for, and served runs of such a grid against the same run
alone."""
import numpy as np
import pytest

from oracle import kref
from kapsel3_amd._abi import FP64, MIXED

from test_gpu_columns import system
from test_gpu_step import cmp_particles, rel

pytestmark = pytest.mark.gpu

GRIDS = [(8, 24, 32), (12, 64, 128), (12, 12, 8), (8, 8, 12)]


def name(n):
    return "x".join(map(str, n))


def radius(n):
    return 2.0 if min(n) > 8 else 1.0


@pytest.mark.parametrize("kind", ["plain", "slip", "sheared"])
@pytest.mark.parametrize("n", GRIDS, ids=name)
def test_steps_against_oracle(gpu, n, kind):
    print(f"short x {n} {kind}", flush=True)
    P, p = system(n, kind == "slip", a=radius(n))
    o, g = kref.Run(P, 3), gpu.Run(P, 3)
    for r in (o, g):
        r.set_particles(p)
        r.init_fluid()
        if kind == "sheared":
            r.set_shear(1e-2)
    # the Euler step and one more singly, one graph of eight, one single replay
    for r in (o, g):
        r.step(2)
    g.step(9)
    o.step(9)
    if kind != "sheared":
        g.timing(True)
    g.step(1)
    o.step(1)
    if kind != "sheared":
        assert {"x_ns_u", "x_f_zeta", "x_zeta2u_inv"} <= set(g.timing_stats())
    cmp_particles(g.get_particles(), o.get_particles(), 1e-10,
                  ["x_nopbc", "v", "omega", "q", "f_hydro_previous", "torque_hydro_previous"], p0=p, a=2.0)
    zo, zg = o.get_fluid(), g.get_fluid()
    assert rel(zg[0], zo[0]) < 1e-10 and rel(zg[1], zo[1]) < 1e-10
    assert np.abs(zg[2] - zo[2]).max() < 1e-10 * max(np.abs(zo[2]).max(), 1.0)
    o.close()
    g.close()


@pytest.mark.parametrize("slip", [False, True], ids=["plain", "slip"])
@pytest.mark.parametrize("n", GRIDS, ids=name)
def test_mixed_follows_fp64(gpu, n, slip):
    """The bounds of the mixed tests at longer axes: 1e-5, squirmers 1e-4."""
    print(f"short x {n} mixed slip {slip}", flush=True)
    out = []
    for precision in (FP64, MIXED):
        P, p = system(n, slip, precision, a=radius(n))
        with gpu.Run(P, 3) as r:
            r.set_particles(p)
            r.init_fluid()
            r.step(12)
            out.append((r.get_particles(), r.get_fluid()))
    (pd, zd), (pm, zm) = out
    tol = 1e-4 if slip else 1e-5
    assert np.abs(pm["v"] - pd["v"]).max() < tol * np.abs(pd["v"]).max()
    assert rel(zm[0], zd[0]) < tol and rel(zm[1], zd[1]) < tol
    assert np.abs(zm[2] - zd[2]).max() < tol * np.abs(zd[2]).max()


@pytest.mark.parametrize("n", [(8, 24, 32), (12, 16, 24)], ids=name)
def test_served_batch(gpu, n):
    print(f"short x {n} served", flush=True)
    P, p = system(n, a=radius(n))
    with gpu.Server(max_active=4, chunk_steps=8, batch_slots=4) as srv:
        out = [srv.submit(P, p, 40) for _ in range(4)]
        for rid, _ in out:
            srv.wait(rid)
    with gpu.Run(P, 3) as r:
        r.set_particles(p)
        r.init_fluid()
        r.set_trajectory(40)
        r.set_graph(False)
        r.step(40)
        alone = r.get_trajectory()
    for _, got in out:
        d = got - alone
        d[..., :3] -= np.rint(d[..., :3] / n) * n
        assert np.abs(d[..., 3:]).max() < 1e-10 * np.abs(alone[..., 3:]).max()
        assert np.abs(d[..., :3]).max() < 1e-10 * max(n)
