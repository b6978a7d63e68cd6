"""The Monte Carlo passes and replica energies compiled per Hamiltonian against
the ahead-of-time ones, bit for bit, where the neighbours' slots can go wrong:
rows that do not fill their slots, open and mixed edges, lattices as small as
the stencil's reach, several planes, a per-site field, more than one group of
neighbours, both samplers, T = 0, replicas."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = {
    "tri": dict(w="tri", size=[64, 48, 1]),
    "tri_open": dict(w="tri", size=[37, 21, 1], periodic=[False, False, False]),
    "tri_mixed": dict(w="tri", size=[64, 29, 1], periodic=[True, False, False], bmap_sigma=0.3),
    "tri_small": dict(w="tri", size=[8, 8, 1]),
    "sq": dict(w="sq", size=[70, 66, 1]),
    "sq_open_y_odd": dict(w="sq", size=[31, 64, 1], periodic=[False, True, False]),
    "sq_reach3": dict(w="sq", size=[128, 64, 1], periodic=[False, False, False],
                      J=[1e-3, -0.2e-3, 0.1e-3, 0.05e-3, -0.04e-3, 0.03e-3]),
    "planes": dict(w="film", size=[34, 40, 6], periodic=[True, True, True]),
    "planes_open": dict(w="film", size=[20, 12, 5]),
}


def _run(c, jit, sampler, kT, reps):
    from matjes_amd import llg
    old = os.environ.get("MJ_JIT")
    os.environ["MJ_JIT"] = jit
    try:
        with llg.Hamiltonian(c["lat"].dim_lat, c["lat"].periodic) as h:
            h.load_terms(c["H"], form="stencil")
            h.set_state(c["m0"])
            h.mc_set_cone(0.4)
            if reps:
                h.mc_pt_setup([kT * (1.0 + 0.2 * q) for q in range(reps)], cone=0.4)
                E, M = h.mc_pt_sweeps(6, sampler, seed=9, exchange_every=2, measure_every=3)
                return [np.asarray(E), np.asarray(M)] + [h.mc_pt_get_state(q) for q in range(reps)]
            E, M = h.mc_sweeps(5, sampler, kT, seed=9, measure_every=2)
            return [np.asarray(E), np.asarray(M), h.get_state(), np.asarray(h.mc_stats()["rate"])]
    finally:
        if old is None:
            os.environ.pop("MJ_JIT", None)
        else:
            os.environ["MJ_JIT"] = old


@pytest.mark.parametrize("sampler,kT,reps", [(0, 1e-3, 0), (1, 1e-3, 0), (0, 0.0, 0), (0, 1e-3, 3)])
@pytest.mark.parametrize("name", sorted(CASES))
def test_compiled_equals_ahead_of_time(name, sampler, kT, reps):
    from matjes_amd import workloads
    s = dict(CASES[name])
    base = {"tri": workloads.TRIANGULAR_J3DKB, "sq": workloads.SQUARE_JDKB,
            "film": dict(workloads.FILM_DIP, dipolar=False)}[s.pop("w")]
    c = workloads.build_case(dict(base, seed=11, **s))
    for a, b in zip(_run(c, "0", sampler, kT, reps), _run(c, "1", sampler, kT, reps)):
        assert np.array_equal(a, b), name


@pytest.mark.parametrize("jit", ["0", "1"])
def test_stencil_that_grows_between_sweeps(jit, monkeypatch):
    """A term that enlarges the stencil of a context that has already swept, against
    a context that had it from the start."""
    from matjes_amd import llg, workloads
    monkeypatch.setenv("MJ_JIT", jit)
    c = workloads.build_case(dict(workloads.SQUARE_JDKB, size=[64, 64, 1], seed=4))
    blk = -0.1e-3 * np.eye(3)
    more = {(2, 0, 0): blk, (-2, 0, 0): blk, (0, 2, 0): blk, (0, -2, 0): blk, (1, 1, 0): 2.0 * blk, (-1, -1, 0): 2.0 * blk}
    out = []
    for early in (False, True):
        with llg.Hamiltonian(c["lat"].dim_lat, c["lat"].periodic) as h:
            h.load_terms(c["H"], form="stencil")
            if early:
                h.add_stencil(more)
            else:
                h.set_state(c["m0"])
                h.mc_sweeps(2, 0, 1e-3, seed=8)
                h.add_stencil(more)
            h.set_state(c["m0"])
            h.mc_set_cone(0.4)
            h.mc_sweeps(4, 1, 1e-3, seed=9)
            out.append(h.get_state())
    assert np.array_equal(out[0], out[1])


def test_scan_over_a_coupling_compiles_once(monkeypatch):
    """Sweeps of Hamiltonians that differ in their couplings' values: one module for
    all, each with its own values (against the ahead-of-time passes)."""
    import ctypes
    from matjes_amd import _lib, llg, workloads

    def made():
        v = ctypes.c_int64()
        _lib.check(_lib.load().mj_jit_stats(ctypes.addressof(v), None), "mj_jit_stats")
        return v.value

    def sweep(c, jit):
        monkeypatch.delenv("MJ_JIT", raising=False)
        if jit is not None:
            monkeypatch.setenv("MJ_JIT", jit)
        with llg.from_case(c, form="stencil") as h:
            n = made()
            h.mc_set_cone(0.4)
            h.mc_sweeps(4, 0, 1e-3, seed=9)
            return h.get_state(), made() - n
    base = workloads.TRIANGULAR_J3DKB
    for k, scale in enumerate((1.0, 0.7, -1.3)):
        c = workloads.build_case(dict(base, size=[136, 64, 1], seed=11, J=[scale * j for j in base["J"]],
                                      D=scale * base["D"]))
        (ref, _), (got, n) = sweep(c, "0"), sweep(c, None)
        assert np.array_equal(ref, got) and n == (1 if k == 0 else 0)
