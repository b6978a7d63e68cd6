"""The fused batch step compiled per stencil against the ahead-of-time one, bit
for bit, where it can go wrong: one group of systems and several (a launch
each), more groups than it takes or a later group of too many coefficients (the
ahead-of-time kernel runs), coefficients
that differ, change sign or vanish between systems, odd rows (no paired loads),
tiles from one site a row (rows of the region that do not pair up) to one row, inside the lattice,
lattices smaller than a tile and its halo, open edges, several planes, a
per-site field."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SQ = [
    dict(size=[64, 64, 1], D=0.2e-3),
    dict(size=[33, 20, 1], D=-0.2e-3, J=[0.7e-3], B=[0.0, 0.3, 1.5]),
    dict(size=[40, 9, 1], D=0.2e-3, periodic=[False, True, False], J=[-0.7e-3]),
    dict(size=[66, 47, 1], bmap_sigma=0.3, K=0.0),
]
BATCHES = {
    "one_stencil": [("sq", s) for s in SQ],
    "two_stencils": [("sq", SQ[0]), ("tri", dict(size=[24, 24, 1])), ("sq", SQ[1]), ("tri", dict(size=[65, 34, 1]))],
    "reach3": [("sq", dict(size=[64, 66, 1], J=[1e-3, -0.2e-3, 0.1e-3, 0.05e-3, -0.04e-3, 0.03e-3]))] * 2,
    "five_stencils": [("sq", dict(size=[32, 32, 1], J=[1e-3, 0.2e-3, 0.1e-3, 0.05e-3, 0.04e-3][:k])) for k in range(1, 5)]
    + [("tri", dict(size=[24, 24, 1]))],
    "long": [("sq", dict(size=[8, 1030, 1])), ("sq", dict(size=[1030, 8, 1], D=0.1e-3))],
    # the second stencil has more coefficients than the compiled step takes
    "second_too_rich": [("sq", SQ[0]), ("sq", dict(size=[40, 36, 1], rich=True)), ("sq", SQ[1])],
    "planes": [("film", dict(size=[20, 17, 4])), ("film", dict(size=[34, 12, 3], periodic=[False, False, False]))],
    "vanishing": [("sq", dict(size=[48, 40, 1], J=[0.0], B=[0.0, 0.0, 0.0])), ("sq", SQ[0])],
}


def _run(specs, jit, integ, tiles):
    from matjes_amd import batch, lattice, llg, workloads
    base = {"sq": workloads.SQUARE_JDKB, "tri": workloads.TRIANGULAR_J3DKB,
            "film": dict(workloads.FILM_DIP, dipolar=False)}
    old = os.environ.get("MJ_JIT")
    os.environ["MJ_JIT"] = jit
    hs = []
    try:
        with batch.Batch() as b:
            for k, (w, s) in enumerate(specs):
                s = dict(s)
                rich = s.pop("rich", False)
                h = llg.from_case(workloads.build_case(dict(base[w], seed=5 + k, **s)), form="stencil")
                if rich:   # 36 values more: a block of its own for each of four further neighbours
                    rng = np.random.default_rng(1)
                    h.add_stencil({o: 1e-4 * rng.normal(size=(3, 3)) for o in [(1, 1, 0), (2, 0, 0), (0, 2, 0), (2, 1, 0)]})
                b.add(h, 0.05 + 0.1 * (k % 2), kT=(4.0 * k) * lattice.K_B, seed=40 + k)
                hs.append(h)
            if tiles:
                b.set_tiles([tiles] * len(specs))
            b.steps(110, 0.5, integrator=integ)
            return [b.state(k) for k in range(len(specs))], b.energies()
    finally:
        for h in hs:
            h.close()
        if old is None:
            os.environ.pop("MJ_JIT", None)
        else:
            os.environ["MJ_JIT"] = old


@pytest.mark.parametrize("name,integ,tiles", [(n, i, t) for n in sorted(BATCHES)
                                              for i, t in [(2, None), (2, (16, 16)), (5, None), (6, None)]]
                         + [("long", i, t) for i, t in [(2, (1, 256)), (5, (1, 256)), (2, (2, 128)), (2, (256, 1))]])
def test_compiled_equals_ahead_of_time(name, integ, tiles):
    ref, e0 = _run(BATCHES[name], "0", integ, tiles)
    got, e1 = _run(BATCHES[name], "1", integ, tiles)
    for k, (a, b) in enumerate(zip(ref, got)):
        assert np.isfinite(a).all() and np.array_equal(a, b), (name, k)
    assert np.array_equal(e0, e1)
