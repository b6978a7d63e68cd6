"""Lattices of several planes coupled to each other on their default tiles (16x4x4,
16x8x2, fewer where an axis is short) against one launch per stage on 32x8x1,
bit for bit: planes that do not fill a tile, one axis shorter than a tile, open
and periodic across the planes."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = {
    "whole": dict(size=[32, 32, 8]),
    "past": dict(size=[33, 37, 5]),
    "two": dict(size=[65, 34, 2]),
    "three_open": dict(size=[47, 40, 3], periodic=[False, False, False]),
    "periodic_z": dict(size=[24, 18, 10], periodic=[True, True, True]),
    "narrow": dict(size=[6, 130, 6]),
    "flat": dict(size=[200, 3, 8]),
}


def _run(c, tile, fuse, integ, T):
    from matjes_amd import llg
    env = {"MJ_FUSE": fuse, "MJ_JIT": "1"}
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        with llg.Hamiltonian(c["lat"].dim_lat, c["lat"].periodic, tile=tile) as h:
            h.load_terms(c["H"], form="stencil")
            h.set_state(c["m0"])
            h.steps(6, integ, 0.5, 0.05, kT=T * 0.000086173324, seed=3)
            return h.get_state()
    finally:
        for k, v in old.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v


@pytest.mark.parametrize("integ,T", [(2, 10.0), (5, 10.0), (6, 0.0)])
@pytest.mark.parametrize("name", sorted(CASES))
def test_default_tile_equals_the_stage_kernels(name, integ, T):
    from matjes_amd import workloads
    c = workloads.build_case(dict(workloads.FILM_DIP, dipolar=False, D=0.3e-3, mediator_dz=-0.5, seed=2, **CASES[name]))
    assert np.array_equal(_run(c, None, "1", integ, T), _run(c, (32, 8, 1), "0", integ, T))


@pytest.mark.parametrize("size,reach", [([16, 16, 16], 6), ([16, 16, 8], 4), ([64, 64, 1], 31), ([70, 66, 1], 33)])
@pytest.mark.parametrize("jit", ["0", "1"])
def test_long_reach_fits_the_lds(size, reach, jit, monkeypatch):
    """Bonds so long that the usual tile's region passes the LDS: the field of
    -J m_(i +- reach) along every axis, each value a sum of at most six products
    and their doubling."""
    from matjes_amd import llg, workloads
    monkeypatch.setenv("MJ_JIT", jit)
    axes = [a for a in range(3) if size[a] > 1]
    ofs = [tuple(s * reach * (a == b) for b in range(3)) for a in axes for s in (1, -1)
           if not (s < 0 and 2 * reach == size[a])]
    m = workloads.random_sphere(int(np.prod(size)), 9)
    with llg.Hamiltonian(size, [True, True, size[2] > 1]) as h:
        h.add_stencil({o: -1e-3 * np.eye(3) for o in ofs})
        h.set_state(m)
        B = h.get_eff_field()
        h.steps(2, 2, 0.1, 0.1)
    g = m.reshape(size[2], size[1], size[0], 3)
    want = sum(2e-3 * 0.5 * (np.roll(g, (-o[2], -o[1], -o[0]), (0, 1, 2)) + np.roll(g, (o[2], o[1], o[0]), (0, 1, 2)))
               for o in ofs).reshape(-1, 3)
    assert np.max(np.abs(B - want)) <= 8 * 2.0 ** -53 * 1e-3 * 2 * len(ofs)


@pytest.mark.parametrize("jit", ["0", "1"])
def test_refused_launch_stays_with_its_call(jit, monkeypatch):
    """A reach for which no tile fits (nothing is launched): the call that asks for it
    fails, and the next one, of another context, does not."""
    from matjes_amd import _lib, llg, workloads
    monkeypatch.setenv("MJ_JIT", jit)
    m = workloads.random_sphere(20 ** 3, 9)
    with llg.Hamiltonian([20, 20, 20], [True, True, True]) as bad, llg.Hamiltonian([20, 20, 20], [True] * 3) as good:
        bad.add_stencil({(9, 0, 0): np.eye(3), (0, 9, 0): np.eye(3), (0, 0, 9): np.eye(3)})
        good.add_stencil({(1, 0, 0): np.eye(3)})
        bad.set_state(m)
        with pytest.raises(_lib.MatjesError, match="invalid argument"):
            bad.get_eff_field()
        good.set_state(m)
        assert np.array_equal(good.get_state(), m)
