"""Lees-Edwards sheared step (Time_evolution_hydro_OBL, sp_3d_ns.cxx:328-433)
on the GPU against the oracle, through the C ABI.

FP64: whole-step trajectories and the final zeta within 1e-10 of the
oracle's (relative to each quantity's scale), across a remap of the grid
and for AC shear. Mixed precision: within 1e-4 of FP64 over 200 steps."""
import numpy as np
import pytest

from oracle import kref
from kapsel3_amd import workloads
from kapsel3_amd._abi import FP64, MIXED, Params, make_species

import interposed
from test_gpu_step import cmp_particles, kept_mask, rel

pytestmark = pytest.mark.gpu

KEYS = ["x", "x_nopbc", "v", "v_old", "omega", "omega_old", "q", "q_old", "f_hydro_previous",
        "torque_hydro_previous", "fr_previous"]


def sheared_system(n=32, precision=FP64, kbt=1e-4):
    """Four spheres: one straddling the sheared boundary, a pair in LJ
    range across it, one near the centre; gravity, rotation, FIX_CELL on z,
    thermal noise, a random initial flow."""
    sp = [make_species(mass_ratio=1.5), make_species(mass_ratio=2.0)]
    P = Params(n, a=4.0, a_xi=2.0, dt=0.05, eta=0.8, species=sp, rotation=1, g=1e-3, g_dir=2, kbt=kbt,
               fix_cell=(0, 0, 1), lj_truncate=1, epsilon=1.0, precision=precision, seed=9)
    g0 = 0.995
    pos = np.array([[10.2, 30.6, 16.1], [3.0, 29.5, 8.0], [(3.0 - g0 * n + 2.0) % n, 5.2, 8.5],
                    [17.3, 15.1, 24.2]])
    p = workloads.particles_at(pos, spec=np.array([0, 1, 0, 1]))
    rng = np.random.default_rng(21)
    p["v"] = rng.normal(0, 1e-3, (4, 3))
    p["v_old"] = p["v"] + rng.normal(0, 1e-4, (4, 3))
    p["omega"] = rng.normal(0, 1e-4, (4, 3))
    p["omega_old"] = rng.normal(0, 1e-4, (4, 3))
    p["q"] = workloads.random_quaternions(4, 2)
    p["q_old"] = workloads.random_quaternions(4, 3)
    return P, p, g0


def initial_fluid(P, n, g0, rate):
    """A random flow through the oracle's own u -> zeta at strain g0."""
    o = kref.Run(P, 0)
    o.set_shear(rate)
    o.set_shear_state(g0, rate)
    rng = np.random.default_rng(5)
    k = np.fft.fftfreq(n) * n
    kz = np.arange(n // 2 + 1)
    m = (np.abs(k)[:, None, None] < 6) & (np.abs(k)[None, :, None] < 6) & (kz[None, None, :] < 6)
    for d in range(3):
        u = np.fft.irfftn(np.fft.rfftn(rng.normal(size=(n, n, n))) * m, s=(n, n, n), axes=(0, 1, 2)) * 2e-3
        a = np.zeros((n, n, n + 2))
        a[:, :, :n] = u
        o.set_field("u%d" % d, a)
    o.le_apply("solenoidal_u")
    o.le_apply("u2zeta_k")
    z0, z1, uk = o.get_fluid()
    o.close()
    return z0, z1, uk


def _pair(P, p, z, rate, g0, ac=False, freq=0.0, ts0=0):
    from kapsel3_amd import Run
    gr = Run(P, len(p))
    orc = kref.Run(P, len(p))
    t = orc.get_time()
    t.ts = ts0
    t.time = ts0 * t.dt_fluid
    for r in (gr, orc):
        r.set_particles(p)
        r.set_fluid(*z)
        r.set_time(t)
        r.set_shear(rate, ac=ac, frequency=freq)
        r.set_shear_state(g0, rate)
    return gr, orc


@pytest.mark.parametrize("ac", [False, True])
def test_sheared_step_fp64_matches_oracle(gpu, ac):
    n, rate = 32, 0.4 if not ac else 0.3
    P, p, g0 = sheared_system(n)
    z = initial_fluid(P, n, g0, rate)
    gr, orc = _pair(P, p, z, rate, g0, ac=ac, freq=0.5, ts0=0 if not ac else 3)
    seen_remap = seen_lj = False
    gr.set_shear_history(12)
    for chunk in range(4):
        gr.step(3)
        orc.step(3)
        gg, sg = gr.shear_state()
        go, so = orc.shear_state()
        assert abs(gg - go) < 1e-14 and abs(sg - so) < 1e-14 * max(abs(so), 1)
        seen_remap |= gg < g0
        cmp_particles(gr.get_particles(), orc.get_particles(), 1e-10, keys=KEYS, p0=p, a=4.0)
        # the stress record (Mean_shear_stress) of the step just taken
        rg, ro = gr.shear_record(), orc.shear_record()
        for k in ("time", "shear_rate", "degree_oblique", "strain", "fluid_stress"):
            assert abs(rg[k] - ro[k]) <= 1e-13 * max(abs(ro[k]), 1.0), (k, rg[k], ro[k])
        for k in ("lj_dev_stress", "shear_stress_old", "shear_stress_new", "reynolds_stress", "apparent_stress"):
            assert abs(rg[k] - ro[k]) <= 1e-9 * max(abs(ro[k]), 1e-12), (k, rg[k], ro[k])
        seen_lj |= abs(ro["lj_dev_stress"]) > 0
        assert abs(ro["shear_stress_new"]) > 0
        if chunk == 1:  # zeta read mid-run (its modes beyond 2/3 formed on demand), then the run goes on
            zg, zo = gr.get_fluid(), orc.get_fluid()
            assert rel(zg[0], zo[0]) < 1e-10 and rel(zg[1], zo[1]) < 1e-10
    assert seen_lj                              # the LJ pair across the boundary contributes
    hist = gr.get_shear_history()
    assert np.array_equal(hist[-1], np.array(list(gr.shear_record().values())))
    assert np.allclose(np.diff(hist[:, 0]), P.c.dt)
    zg, zo = gr.get_fluid(), orc.get_fluid()
    for a, b in zip(zg[:2], zo[:2]):
        assert rel(a, b) < 1e-10
    assert np.abs(zg[2] - zo[2]).max() < 1e-10 * max(np.abs(zo[2]).max(), 1e-30) + 1e-18
    assert seen_remap or ac                  # the DC case crosses strain 1 and is remapped
    gr.close()


def test_sheared_mixed_tracks_fp64(gpu):
    from kapsel3_amd import Run
    n, rate = 32, 0.05
    out = {}
    for prec in (FP64, MIXED):
        P, p, g0 = sheared_system(n, precision=prec, kbt=0.0)
        r = Run(P, len(p))
        r.set_particles(p)
        r.init_fluid()
        r.set_shear(rate)
        r.step(200)
        out[prec] = r.get_particles()
        r.close()
    a, b = out[MIXED], out[FP64]
    vs = np.abs(b["v"]).max()
    assert np.abs(a["v"] - b["v"]).max() < 1e-4 * vs
    assert np.abs(a["omega"] - b["omega"]).max() < 1e-4 * vs / 4.0
    assert np.abs(a["x_nopbc"] - b["x_nopbc"]).max() < 1e-4 * np.abs(b["x_nopbc"] - p["x_nopbc"]).max()


def test_shear_entry_points_reject_bad_input(gpu):
    from kapsel3_amd import KhError, Run
    P, p, g0 = sheared_system(16 * 2)
    r = Run(P, len(p))
    with pytest.raises(KhError):
        r.set_shear_state(0.1, 0.0)          # not sheared yet
    r.set_shear(0.1)
    with pytest.raises(KhError):
        r.set_shear_state(1.5, 0.1)          # outside (-NX/NY, NX/NY)
    with pytest.raises(KhError):
        r.set_shear(float("nan"))
    r.close()


@pytest.mark.parametrize("n,np_,steps", [(128, 60, 4), (256, 40, 2)])
def test_sheared_production_grid_fp64(gpu, n, np_, steps):
    """The sedimentation geometry (a = 5, LJ, gravity, noise) under shear at
    128^3 and 256^3 (the production z-pass engines), started just below
    unit strain so the grid is remapped during the run."""
    from kapsel3_amd import Run
    print(f"sheared {n}^3 x {np_}, {steps} steps", flush=True)
    P, parts = workloads.sedimentation(n, np_, gap=0.4, seed=5, kbt=1e-3)
    rate = 0.02
    g0 = 1.0 - 1.5 * rate * P.c.dt
    gr, orc = Run(P, np_), kref.Run(P, np_)
    for r in (gr, orc):
        r.set_particles(parts)
        r.init_fluid()
        r.set_shear(rate)
        r.set_shear_state(g0, rate)
        r.step(steps)
    assert gr.shear_state()[0] < g0 and abs(gr.shear_state()[0] - orc.shear_state()[0]) < 1e-14
    cmp_particles(gr.get_particles(), orc.get_particles(), 1e-10, keys=KEYS, p0=parts, a=5.0)
    zo, zg = orc.get_fluid(), gr.get_fluid()
    assert rel(zg[0], zo[0]) < 1e-10 and rel(zg[1], zo[1]) < 1e-10
    gr.close()


@pytest.mark.parametrize("n", [32, 16])
def test_sheared_fluid_without_particles(gpu, n):
    """Lees-Edwards with no particles: the flow of a random initial field
    against the oracle; the stress record has no particle terms. At 16^3 u x
    omega is a separate pass (the fused inverse z pass needs z >= 32)."""
    from kapsel3_amd import Run
    rate = 0.3
    P, _, g0 = sheared_system(n)
    z = initial_fluid(P, n, g0, rate)
    gr, orc = Run(P, 0), kref.Run(P, 0)
    for r in (gr, orc):
        r.set_fluid(*z)
        r.set_shear(rate)
        r.set_shear_state(g0, rate)
        r.step(5)
    zg, zo = gr.get_fluid(), orc.get_fluid()
    assert rel(zg[0], zo[0]) < 1e-10 and rel(zg[1], zo[1]) < 1e-10
    rg, ro = gr.shear_record(), orc.shear_record()
    assert rg["shear_stress_old"] == 0.0 and rg["shear_stress_new"] == 0.0 and ro["shear_stress_new"] == 0.0
    assert abs(rg["reynolds_stress"] - ro["reynolds_stress"]) <= 1e-9 * abs(ro["reynolds_stress"])
    gr.close()


def test_sheared_functions_fp64(gpu):
    """Single functions of Time_evolution_hydro_OBL through kh_apply at
    strain 0.37 against the oracle's: Zeta_k2u_k_OBL, U_oblique2u, the
    particle functions in the Lees-Edwards geometry (phi, F_H on the
    Cartesian u, u_p, position with PBC_OBL), the projection + curl, the
    sheared NS solver."""
    n, rate, g = 32, 0.07, 0.37
    P, p, _ = sheared_system(n)
    p["x"][2] = [(3.0 - g * n + 2.0) % n, 5.2, 8.5]
    z = initial_fluid(P, n, g, rate)
    gr, orc = _pair(P, p, z, rate, g)

    def fields(names):
        return [(gr.get_field(k), orc.get_field(k)) for k in names]

    def close(pairs, tol):
        for a, b in pairs:
            assert rel(a[..., :n], b[..., :n]) < tol

    gr.apply("obl_zeta_k2u")
    orc.le_apply("zeta_k2u")
    close(fields(["u0", "u1", "u2"]), 1e-12)
    gr.apply("obl_oblique2u")
    orc.le_apply("oblique2u")
    close(fields(["u0", "u1", "u2"]), 1e-12)
    gr.apply("make_phi")
    orc.le_apply("make_phi")
    close(fields(["phi_sum"]), 1e-13)
    gr.apply("f_hydro")
    orc.le_apply("f_hydro")
    pg, po = gr.get_particles(), orc.get_particles()
    assert rel(pg["f_hydro"], po["f_hydro"]) < 1e-12 and rel(pg["torque_hydro"], po["torque_hydro"]) < 1e-12
    gr.apply("make_up")
    orc.le_apply("make_up")
    close(fields(["up0", "up1", "up2"]), 1e-12)
    gr.apply("position_euler")
    orc.le_apply("position_euler")
    pg, po = gr.get_particles(), orc.get_particles()
    assert np.abs(pg["x"] - po["x"]).max() < 1e-12 and rel(pg["v"], po["v"]) < 1e-13
    # the closing projection + curl, on a random field
    rng = np.random.default_rng(9)
    for d in range(3):
        a = np.zeros((n, n, n + 2))
        a[:, :, :n] = rng.normal(0, 1e-3, (n, n, n))
        gr.set_field("u%d" % d, a)
        orc.set_field("u%d" % d, a)
    gr.apply("obl_u2zeta_k")
    orc.le_apply("solenoidal_u")
    orc.le_apply("u2zeta_k")
    zg, zo = gr.get_fluid(), orc.get_fluid()
    # the oracle projects through one extra real-space round trip, which does
    # not keep the Nyquist planes of a projected random field (kx or ky = N/2
    # at kz = 0, kz = N/2: not Hermitian after the projection); compared on
    # the 2/3-kept modes (the whole-step tests compare every mode)
    m = kept_mask(zg[0].shape)
    assert rel(zg[0][m], zo[0][m]) < 1e-11 and rel(zg[1][m], zo[1][m]) < 1e-11
    # the sheared NS solver from the flow of initial_fluid
    for r in (gr, orc):
        r.set_fluid(*z)
    gr.apply("obl_ns_solver")
    orc.le_apply("ns_solver")
    zg, zo = gr.get_fluid(), orc.get_fluid()
    assert rel(zg[0], zo[0]) < 1e-12 and rel(zg[1], zo[1]) < 1e-12
    gr.close()


def test_ns_solver_leaves_u(gpu):
    """kh_apply of the sheared NS solver leaves the velocity it was given
    (zeta_k2u of the truncated zeta) in u."""
    n, rate = 32, 0.05
    P, p, g0 = sheared_system(n)
    z = initial_fluid(P, n, g0, rate)
    gr, orc = _pair(P, p, z, rate, g0)
    print("u after the sheared NS solver", flush=True)
    for d in range(3):  # something else in the field
        gr.set_field("u%d" % d, np.full((n, n, n + 2), 7.0))
    gr.apply("obl_ns_solver")
    orc.le_apply("zeta_k2u")
    for d in range(3):
        assert rel(gr.get_field(f"u{d}")[..., :n], orc.get_field(f"u{d}")[..., :n]) < 1e-12, d
    gr.close()


REFUSED = """
calls, live, fail_at = (ctypes.c_int.in_dll(fake, k) for k in ("calls", "live", "fail_at"))
import numpy as np
import kapsel3_amd
from kapsel3_amd._abi import Params
out = []
for refuse in (0, 1, 2, 3, 4):
    with kapsel3_amd.Run(Params((16, 16, 16), a=1.0, a_xi=1.0, dt=0.05), 0) as r:
        z = np.random.default_rng(3).standard_normal(r.shape)
        r.set_fluid(z, z[::-1], [1.0, 2.0, 3.0])
        if refuse:
            fail_at.value = calls.value + refuse
            try:
                r.set_shear(0.1)
                raise SystemExit("accepted")
            except kapsel3_amd.KhError:
                pass
        r.step(2)  # still the plain step
        r.set_shear(0.1)
        r.step(2)
        out.append(r.get_fluid())
    print("live after the run", live.value)
for f in out[1:]:
    assert all(np.array_equal(a, b) for a, b in zip(f, out[0]))
"""


def test_refused_buffers_leave_the_run(gpu, tmp_path):
    """kh_set_shear that cannot allocate one of its buffers says so, the run
    goes on as it was, a later call is accepted, and the run gives back all
    that was allocated."""
    print("set_shear without memory", flush=True)
    out = interposed.run(tmp_path, interposed.COUNTED, REFUSED)
    assert out.splitlines() == 5 * ["live after the run 0"], out


def test_deferred_modes_after_remap_and_transitions(gpu):
    """zeta's modes beyond the 2/3 rule, which sheared steps leave to be
    formed when the state is read, against the oracle (1e-10, uk_dc
    included): right after a step that remaps the grid, and after each entry
    point that completes them before it acts -- kh_set_shear_state,
    kh_apply of the oblique zeta -> u, kh_set_step_path -- taken right after
    sheared steps."""
    n, rate = 32, 0.4
    P, p, g0 = sheared_system(n)  # strain 0.995 + 0.02 per step: the first step remaps (to 0.015)
    z = initial_fluid(P, n, g0, rate)
    gr, orc = _pair(P, p, z, rate, g0)
    print("deferred zeta modes after a remap step and entry points", flush=True)

    def same(tag):
        zg, zo = gr.get_fluid(), orc.get_fluid()
        assert rel(zg[0], zo[0]) < 1e-10 and rel(zg[1], zo[1]) < 1e-10, tag
        assert np.abs(zg[2] - zo[2]).max() <= 1e-10 * max(np.abs(zo[2]).max(), 1e-30) + 1e-18, tag

    def both_step(k):
        gr.step(k)
        orc.step(k)

    both_step(1)
    assert 0 <= gr.shear_state()[0] < g0 and abs(gr.shear_state()[0] - orc.shear_state()[0]) < 1e-14
    same("right after the remap step")
    both_step(2)
    for r in (gr, orc):
        r.set_shear_state(0.3, rate)
    same("set_shear_state after sheared steps")
    both_step(2)
    same("steps after set_shear_state")
    gr.apply("obl_zeta_k2u")  # reads every mode of zeta the steps left
    orc.le_apply("zeta_k2u")
    for d in range(3):
        assert rel(gr.get_field(f"u{d}")[..., :n], orc.get_field(f"u{d}")[..., :n]) < 1e-10, d
    same("zeta -> u after sheared steps")
    both_step(2)
    same("steps after zeta -> u")
    gr.set_step_path("reference")
    same("set_step_path after sheared steps")
    both_step(2)
    same("sheared steps after the path switch")
    cmp_particles(gr.get_particles(), orc.get_particles(), 1e-10, keys=KEYS, p0=p, a=4.0)
    gr.close()
