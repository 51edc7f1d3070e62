"""The rigidity force's z pass on either side of the size from which its
three components share a workgroup no more, with each of its masks: the
occupancy bits (plain spheres), phi_sum (rigid bodies, squirmers' u* + slip
field) and none (the slip force field). FP64 steps against the oracle."""
import numpy as np
import pytest

from oracle import kref
from kapsel3_amd import workloads
from kapsel3_amd._abi import FP64, JAX_Z, JP_SLIP, Params, make_species, new_particles

from test_gpu_rigid import BEADS, CUM, V0, W0
from test_gpu_step import cmp_particles, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["plain", "rigid", "slip"])
@pytest.mark.parametrize("n", [(64, 64, 128), (64, 96, 128), (64, 48, 192)], ids=lambda n: "x".join(map(str, n)))
def test_steps_against_oracle(gpu, n, kind):
    print(f"force mask {n} {kind}", flush=True)
    sp = [make_species(mass_ratio=1.0, propulsion=JP_SLIP, janus_axis=JAX_Z, slip_vel=0.01, slip_mode=1.3)
          if kind == "slip" else make_species(mass_ratio=1.5), make_species(mass_ratio=2.0)]
    P = Params(n, a=4.0, a_xi=2.0, dt=0.05, kbt=0.0, g=0.0 if kind == "slip" else 1e-3, g_dir=2, rotation=1,
               fix_cell=(1, 1, 1), lj_truncate=1, species=sp, precision=FP64)
    np_ = len(BEADS)
    p = new_particles(np_)
    p["x_nopbc"], p["x"], p["spec"] = BEADS, np.mod(BEADS, n), [0, 0, 0, 1, 1, 0]
    p["q"] = p["q_old"] = workloads.random_quaternions(np_, 3)
    o, g = kref.Run(P, np_), gpu.Run(P, np_)
    for r in (o, g):
        r.set_particles(p)
        if kind == "rigid":
            r.set_rigid(CUM, free=[1, 1, 1], v0=V0, w0=W0)
        r.init_fluid()
        r.step(4)
    cmp_particles(g.get_particles(), o.get_particles(), 1e-10,
                  ["x_nopbc", "v", "omega", "f_hydro_previous", "torque_hydro_previous"], p0=p, a=4.0)
    zo, zg = o.get_fluid(), g.get_fluid()
    assert rel(zg[0], zo[0]) < 1e-10 and rel(zg[1], zo[1]) < 1e-10
    o.close()
    g.close()
