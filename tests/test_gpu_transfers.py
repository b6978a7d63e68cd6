"""States and fields to and from host arrays through pinned memory, where its
chunks can go wrong: a few sites, one chunk (21824 sites) and a site either side of
it, two chunks and one site more, whole and odd row lengths; every value arrives
as it was (values below 1e-50 leave as zero, the reference's truncation)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(3, 3, 1), (7, 5, 1), (21823, 1, 1), (21824, 1, 1), (21825, 1, 1), (21824, 2, 1),
                                  (43649, 1, 1), (300, 291, 1)])
def test_state_round_trip(size):
    from matjes_amd import batch, llg, workloads
    c = workloads.build_case(dict(workloads.SQUARE_JDKB, size=list(size), periodic=[False, False, False], seed=3))
    m = np.random.default_rng(4).normal(size=(int(np.prod(size)), 3))
    m[0] = [1e-60, -2.0, 0.0]
    want = m.copy()
    want[0, 0] = 0.0
    with llg.Hamiltonian(c["lat"].dim_lat, c["lat"].periodic) as h:
        h.load_terms(c["H"], form="stencil")
        h.set_state(m)
        assert np.array_equal(h.get_state(), want)
        h.keep_last_field(True)
        B = h.get_eff_field()
        h.steps(1, llg.EULER, 0.1, 0.1)
        assert np.max(np.abs(h.last_field() - B)) <= 1e-12 * np.max(np.abs(B))
        h.set_state(want)
        with batch.Batch() as b:
            b.add(h, 0.1)
            b.energies()
            assert np.array_equal(b.state(0), want)
