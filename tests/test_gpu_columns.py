"""The column passes at every kind of length (one stage, radix 8 with and
without a shorter last stage, 12 points per lane; tiles that hold more columns
than there are kept modes) along x and along y, through the whole plain step
and the squirmers' slip loop, FP64 against the oracle and mixed against FP64; and
captured steps of plain, squirmer and rigid runs, which go from one step's zeta
straight to the next one's u_hat, against the same steps taken one by one."""
import numpy as np
import pytest

from oracle import kref
from kapsel3_amd import workloads
from kapsel3_amd._abi import FP64, JAX_Z, JP_SLIP, MIXED, Params, make_species

from test_gpu_step import cmp_particles, rel

pytestmark = pytest.mark.gpu


def system(n, slip=False, precision=FP64, a=2.0, slip_tol=0.005):
    sp = [make_species(mass_ratio=1.0, propulsion=JP_SLIP, janus_axis=JAX_Z, slip_vel=0.01, slip_mode=1.3)
          if slip else make_species(mass_ratio=2.0)]
    # (the reference's link cells are 16 points: no pair forces on a shorter axis)
    P = Params(n, a=a, a_xi=2.0, dt=0.05, species=sp, rotation=1, g=0.0 if slip else 1e-3, fix_cell=(0, 1, 1),
               lj_truncate=1 if min(n) >= 16 else -1, precision=precision, slip_tol=slip_tol)
    box = np.array(n, float)
    x = np.mod(np.array([[0.2, 0.3, 0.9], [0.2, 0.3, 0.9], [0.7, 0.8, 0.4]]) * box + [[0, 0, 0], [3.1, 1.2, 2.2], [0, 0, 0]],
               box)
    p = workloads.particles_at(x, spec=np.zeros(3, int), q=workloads.random_quaternions(3, 3))
    rng = np.random.default_rng(4)
    p["v"], p["omega"] = rng.normal(0, 1e-2, (3, 3)), rng.normal(0, 1e-3, (3, 3))
    return P, p


@pytest.mark.parametrize("slip", [False, True], ids=["plain", "slip"])
@pytest.mark.parametrize("n", [(512, 16, 16), (16, 512, 24), (384, 24, 16), (24, 384, 16), (256, 12, 32), (16, 192, 12),
                               (128, 96, 16), (64, 48, 24), (12, 64, 128), (8, 24, 32)],
                         ids=lambda n: "x".join(map(str, n)))
def test_steps_against_oracle(gpu, n, slip):
    import kapsel3_amd
    print(f"columns {n} slip {slip}", flush=True)
    P, p = system(n, slip, a=2.0 if min(n) > 8 else 1.0)
    o, g = kref.Run(P, 3), kapsel3_amd.Run(P, 3)
    for r in (o, g):
        r.set_particles(p)
        r.init_fluid()
        r.step(10)
    cmp_particles(g.get_particles(), o.get_particles(), 1e-10,
                  ["x_nopbc", "v", "omega", "q", "f_hydro_previous", "torque_hydro_previous"], p0=p, a=2.0)
    zo, zg = o.get_fluid(), g.get_fluid()
    assert rel(zg[0], zo[0]) < 1e-10 and rel(zg[1], zo[1]) < 1e-10
    # FIX_CELL leaves x free: its mean velocity is carried from step to step
    assert np.abs(zg[2] - zo[2]).max() < 1e-10 * max(np.abs(zo[2]).max(), 1.0)


@pytest.mark.parametrize("n", [(96, 24, 16), (128, 16, 24), (192, 16, 16), (384, 12, 16), (512, 16, 12), (24, 192, 16)],
                         ids=lambda n: "x".join(map(str, n)))
def test_mixed_follows_fp64(gpu, n):
    """The same passes in FP32 against FP64 at the lengths along x and y that
    the other mixed tests do not reach; the bounds are theirs."""
    import kapsel3_amd
    print(f"columns {n} mixed", flush=True)
    out = []
    for precision in (FP64, MIXED):
        P, p = system(n, precision=precision)
        with kapsel3_amd.Run(P, 3) as r:
            r.set_particles(p)
            r.init_fluid()
            r.step(12)
            out.append((r.get_particles(), r.get_fluid()))
    (pd, zd), (pm, zm) = out
    assert np.abs(pm["v"] - pd["v"]).max() < 1e-5 * np.abs(pd["v"]).max()
    assert rel(zm[0], zd[0]) < 1e-5 and rel(zm[1], zd[1]) < 1e-5
    assert np.abs(zm[2] - zd[2]).max() < 1e-5 * np.abs(zd[2]).max()


def test_fp64_x_192(gpu):
    print("columns (192, 16, 16)", flush=True)
    test_steps_against_oracle(gpu, (192, 16, 16), False)
    test_steps_against_oracle(gpu, (192, 16, 16), True)


@pytest.mark.parametrize("precision", [FP64, MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("n", [(32, 32, 32), (24, 48, 96), (64, 64, 64), (12, 24, 32)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("kind", ["plain", "slip", "rigid"])
def test_captured_chain_is_the_steps_one_by_one(gpu, n, precision, kind):
    """Steps replayed as graphs of eight against steps launched singly: the
    same formulas in other kernels, whose multiply-adds the compiler contracts
    differently, so equal to rounding over the 33 steps (FP64 1e-12, some
    thousand ulps; FP32 fields 1e-5). Squirmers take as many iterations either
    way (no convergence test near a tie: the tolerance is out of reach)."""
    import kapsel3_amd
    print(f"chain {n} precision {precision} {kind}", flush=True)
    out = []
    for graph in (True, False):
        P, p = system(n, kind == "slip", precision=precision, slip_tol=0.0)
        with kapsel3_amd.Run(P, 3) as r:
            r.set_particles(p)
            if kind == "rigid":
                r.set_rigid([0, 2, 3], v0=p["v"][[0, 2]], w0=p["omega"][[0, 2]])
            r.init_fluid()
            r.set_graph(graph)
            r.step(1)
            r.step(16)
            r.step(16)
            out.append((r.get_particles(), r.get_fluid()))
    (pa, za), (pb, zb) = out
    tol = 1e-12 if precision == FP64 else 1e-5
    for k in ("x", "v", "omega", "q"):
        assert rel(pa[k], pb[k]) < tol, k
    assert rel(za[0], zb[0]) < tol and rel(za[1], zb[1]) < tol
    assert np.abs(za[2] - zb[2]).max() < tol * np.abs(zb[2]).max()
