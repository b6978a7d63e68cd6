"""The device integrators against closed forms and equilibrium statistics
(MI355X, through the C-ABI).

Independent spins in a static field B along z:
- at T = 0 every spin follows damped precession in closed form, so SIB and
  Depondt are checked against it directly (second order in dt);
- at finite T the in-kernel thermal field (Philox normals, amplitude formed on
  the device) gives <m_z> = L(c x), x = mu_s mu_B B / kT, with c = 1 for SIB
  and Depondt (fluctuation-dissipation amplitude) and c = 2 / 4 for the
  reference's integration 1 / 2 (sigma^2 = alpha kT hbar / dt_stage in the
  last stage only, spindynamics.f90:266-269).
"""
import numpy as np
import pytest

from matjes_amd import lattice as L

pytestmark = pytest.mark.gpu


def _paramagnet_case(n, B, m0):
    lat = L.Lattice(np.eye(3), (1.0, 1.0, 1.0), (n, n, 1), (True, True, False), [("Fe", (0, 0, 0), 1.0)])
    H = L.Hamiltonian(lat)
    H.add_zeeman(B)
    return {"lat": lat, "H": H, "m0": m0}


def _langevin(x):
    return 1.0 / np.tanh(x) - 1.0 / x


@pytest.mark.parametrize("alpha", [0.1, 0.5])
@pytest.mark.parametrize("integ", [5, 6])
def test_damped_precession_closed_form_on_device(integ, alpha):
    from matjes_amd import llg
    n, Bz, t_total = 64, 10.0, 4000.0
    rng = np.random.default_rng(3)
    th0 = rng.uniform(0.2, 2.9, n * n)
    ph0 = rng.uniform(0.0, 2 * np.pi, n * n)
    m0 = np.stack([np.sin(th0) * np.cos(ph0), np.sin(th0) * np.sin(ph0), np.cos(th0)], axis=1)
    w = L.MU_B * Bz / L.HBAR
    th = 2.0 * np.arctan(np.tan(th0 / 2.0) * np.exp(-alpha * w * t_total / (1.0 + alpha * alpha)))
    ph = ph0 + w * t_total / (1.0 + alpha * alpha)
    want = np.stack([np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th)], axis=1)
    err = []
    for dt in (8.0, 4.0):
        with llg.from_case(_paramagnet_case(n, [0.0, 0.0, Bz], m0)) as h:
            h.steps(int(round(t_total / dt)), integ, dt, alpha)
            err.append(np.max(np.abs(h.get_state() - want)))
    assert err[1] < 1e-4, err
    assert 3.5 < err[0] / err[1] < 4.5, err


@pytest.mark.parametrize("integ,c", [(1, 2.0), (2, 4.0), (5, 1.0), (6, 1.0)])
def test_paramagnet_equilibrium_on_device(integ, c):
    """In-kernel thermal field: x = 0.168 (B = 50 T, T = 200 K), 256x256 spins;
    L(x) = 0.056, L(2x) = 0.111, L(4x) = 0.217: a sqrt 2 in sigma moves <m_z>
    by more than 0.04."""
    from matjes_amd import llg
    from oracle import oracle as orc
    n, Bz, T, alpha, dt = 256, 50.0, 200.0, 1.0, 1.0
    kT = T * orc.K_B
    x = L.MU_B * Bz / kT
    with llg.from_case(_paramagnet_case(n, [0.0, 0.0, Bz], np.tile([0.0, 0.0, 1.0], (n * n, 1)))) as h:
        h.steps(2000, integ, dt, alpha, kT=kT, seed=11, step0=0)
        acc = []
        for k in range(20):
            h.steps(200, integ, dt, alpha, kT=kT, seed=11, step0=2000 + 200 * k)
            acc.append(h.get_state()[:, 2].mean())
    assert abs(np.mean(acc) - _langevin(c * x)) < 0.01, (np.mean(acc), _langevin(c * x))


def test_order_of_integration_4_between_calls():
    """The same call of integration 4 after another order was set (both calls long
    enough to replay a captured chunk of steps), against a context of that order."""
    from matjes_amd import llg, workloads
    c = workloads.build_case(dict(workloads.SQUARE_JDKB, size=[24, 20, 1], seed=6))
    out = []
    for orders in ((4, 2), (2,)):
        with llg.from_case(c) as h:
            for n in orders:
                h.set_rk_order(n)
                h.set_state(c["m0"])
                E = h.steps(70, 4, 2.0, 0.2, energies=True)
            out.append((h.get_state(), E))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("n", [5, 8, 24])
def test_a_field_without_bonds(n):
    """No entry in the stencil, on lattices below the compiled kernels: the effective
    field is the external one, and two calls agree."""
    from matjes_amd import llg
    m0 = np.tile([0.6, 0.0, 0.8], (n * n, 1))
    c = _paramagnet_case(n, [0.0, 0.0, 2.5], m0)
    with llg.from_case(c) as h:
        B = h.get_eff_field()
        h.steps(3, 2, 1.0, 0.1)
        assert np.max(np.abs(B - np.array([0.0, 0.0, L.MU_B * 2.5]))) <= 4 * 2.0 ** -53 * L.MU_B * 2.5
        assert np.array_equal(h.get_eff_field(), B)
