"""The film's dipolar field with the transformed tensor as one real number a
value (open in the plane: K_n is even under in-plane inversion bit for bit)
against both parts kept, and against the direct sum over the tensor: one layer
pair up to 32, odd and even grids, an axis of one cell, and the lattices that
must keep both parts (periodic in the plane).

Both forms sum the same products but for the parts that are zero up to the
transform's rounding, so they differ by the rounding of a transform of n points
and lz layers: below 1e-13 of the largest field."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = {
    "open": dict(size=[20, 16, 6], periodic=[False, False, False]),
    "open_odd": dict(size=[13, 9, 3], periodic=[False, False, False]),
    "two_layers": dict(size=[16, 12, 2], periodic=[False, False, False]),
    "thick": dict(size=[6, 5, 32], periodic=[False, False, False]),
    "chain": dict(size=[24, 2, 4], periodic=[False, False, False]),
    "mixed": dict(size=[14, 10, 4], periodic=[True, False, False]),
    "periodic": dict(size=[12, 10, 4], periodic=[True, True, False]),
}


def _field(c, half):
    from matjes_amd import llg
    old = os.environ.get("MJ_DIP_HALF")
    os.environ["MJ_DIP_HALF"] = half
    try:
        with llg.from_case(c, form="stencil") as h:
            return h.get_eff_field()
    finally:
        if old is None:
            os.environ.pop("MJ_DIP_HALF", None)
        else:
            os.environ["MJ_DIP_HALF"] = old


def _direct(c):
    """-2 sum_j K(i - j) m_j of the padded circular convolution, in float64."""
    d = c["H"].dipolar
    K, N = d["K"], d["N_rep"]
    nx, ny, nz = c["lat"].dim_lat
    pos = np.array([(x, y, z) for z in range(nz) for y in range(ny) for x in range(nx)])
    B = np.zeros((len(pos), 3))
    for i, p in enumerate(pos):
        r = (p[None, :] - pos) % np.array(N)[None, :]
        k = r[:, 0] + N[0] * (r[:, 1] + N[1] * r[:, 2])
        B[i] = -2.0 * np.einsum("jab,ja->b", K[k], c["m0"])
    return B


@pytest.mark.parametrize("name", sorted(CASES))
def test_one_part_equals_both(name):
    from matjes_amd import workloads
    c = workloads.build_case(dict(workloads.FILM_DIP, seed=5, **CASES[name]))
    both, one = _field(c, "0"), _field(c, "1")
    scale = np.max(np.abs(both))
    assert np.max(np.abs(one - both)) <= 1e-13 * scale
    plain = workloads.build_case(dict(workloads.FILM_DIP, seed=5, **dict(CASES[name], dipolar=False)))
    want = _direct(c) + _field(plain, "1")
    assert np.max(np.abs(one - want)) <= 1e-12 * scale
    if name in ("mixed", "periodic"):
        assert np.array_equal(one, both)
