"""The z passes at lengths three times a power of two (12 points per lane,
radices 12, 6 and 4) through everything that runs them: the full transforms
of odd numbers of rows, the plain step (masked inverse, advection, force, the
cleared fields), the squirmers' slip loop and the sheared step, against numpy and
the oracle."""
import numpy as np
import pytest

from oracle import kref
from kapsel3_amd import workloads
from kapsel3_amd._abi import FP64, JAX_Z, JP_SLIP, MIXED, Params, make_species

from test_gpu_step import cmp_particles, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [(FP64, 1e-13), (MIXED, 2e-6)], ids=["fp64", "fp32"])
@pytest.mark.parametrize("nz", [12, 24, 48, 96, 192, 384])
def test_transforms(gpu, nz, precision, tol):
    print(f"z length {nz} precision {precision}", flush=True)
    shape = (8, 24, nz)
    a = np.zeros((8, 24, nz + 2))
    a[:, :, :nz] = np.random.default_rng(nz).standard_normal(shape)
    with gpu.Run(Params(shape, precision=precision, a=1.0, a_xi=1.0), 0) as run:
        g = run.A2a_k(a)
        ref = np.fft.rfftn(a[:, :, :nz])
        assert np.abs(g[:, :, 0::2] + 1j * g[:, :, 1::2] - ref).max() / np.abs(ref).max() < tol
        assert np.abs(run.A_k2a(g)[:, :, :nz] - a[:, :, :nz]).max() < 10 * tol


def system(n, slip, shear, precision=FP64):
    sp = [make_species(mass_ratio=1.0, propulsion=JP_SLIP, janus_axis=JAX_Z, slip_vel=0.01, slip_mode=1.3)
          if slip else make_species(mass_ratio=2.0)]
    P = Params(n, a=4.0, a_xi=2.0, dt=0.05, species=sp, rotation=1, g=0.0 if slip else 1e-3, fix_cell=(1, 1, 1),
               precision=precision)
    # two spheres with overlapping interfaces across the z boundary, one alone
    p = workloads.particles_at(np.array([[8.2, 9.1, n[2] - 3.4], [8.9, 10.0, 5.3], [21.6, 22.3, 10.7]]),
                               spec=np.zeros(3, int), q=workloads.random_quaternions(3, 3))
    rng = np.random.default_rng(4)
    p["v"], p["omega"] = rng.normal(0, 1e-2, (3, 3)), rng.normal(0, 1e-3, (3, 3))
    return P, p


@pytest.mark.parametrize("kind", ["plain", "slip", "sheared"])
@pytest.mark.parametrize("n", [(32, 32, 24), (24, 32, 48), (32, 24, 96)])
def test_steps_against_oracle(gpu, n, kind):
    import kapsel3_amd
    print(f"steps {n} {kind}", flush=True)
    P, p = system(n, kind == "slip", kind == "sheared")
    o, g = kref.Run(P, 3), kapsel3_amd.Run(P, 3)
    for r in (o, g):
        r.set_particles(p)
        r.init_fluid()
        if kind == "sheared":
            r.set_shear(1e-2)
        r.step(12)  # the Euler step, captured steps one at a time and eight at once
    po, pg = o.get_particles(), g.get_particles()
    cmp_particles(pg, po, 1e-10, ["x_nopbc", "v", "omega", "q", "f_hydro_previous", "torque_hydro_previous"], p0=p,
                  a=4.0)
    zo, zg = o.get_fluid(), g.get_fluid()
    assert rel(zg[0], zo[0]) < 1e-10 and rel(zg[1], zo[1]) < 1e-10


def test_mixed_steps_follow_fp64(gpu):
    import kapsel3_amd
    print("steps (32, 24, 96) mixed", flush=True)
    out = []
    for precision in (FP64, MIXED):
        P, p = system((32, 24, 96), False, False, precision)
        with kapsel3_amd.Run(P, 3) as r:
            r.set_particles(p)
            r.init_fluid()
            r.step(12)
            out.append((r.get_particles(), r.get_fluid()))
    (pd, zd), (pm, zm) = out
    assert np.abs(pm["v"] - pd["v"]).max() < 1e-5 * np.abs(pd["v"]).max()
    assert rel(zm[0], zd[0]) < 1e-5 and rel(zm[1], zd[1]) < 1e-5
