"""The differentiable SIB trajectory's kernels compiled per parameter set against
the ahead-of-time ones, bit for bit, where they can go wrong: lattices that do
not fill their tiles, smaller than a tile and its halo, open and mixed edges,
several planes, a reach of 2, one parameter, a parameter at zero, two kernels a
step, a last segment shorter than the checkpoints' spacing."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = {
    "whole": dict(size=[64, 64, 1]),
    "past": dict(size=[65, 33, 1]),
    "open": dict(size=[37, 21, 1], periodic=[False, False, False]),
    "mixed": dict(size=[24, 50, 1], periodic=[True, False, False]),
    "small": dict(size=[6, 5, 1]),
    "planes": dict(size=[18, 10, 3]),
    "reach2": dict(size=[40, 36, 1], names=["J1", "J3", "D", "K"], theta=[1e-3, 0.2e-3, 0.3e-3, -0.05e-3]),
    "one": dict(size=[33, 40, 1], names=["J1"], theta=[1e-3]),
    "zero": dict(size=[40, 40, 1], theta=[1e-3, 0.0, -0.05e-3]),
    "two_kernels": dict(size=[40, 33, 1], env={"MJ_ADJ_FUSE": "0"}),
}


def _run(c, jit, before=()):
    import torch
    from matjes_amd import adjoint, workloads
    env = dict({"MJ_JIT": jit}, **c.get("env", {}))
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        lat = workloads.make_lattice(dict(workloads.SQUARE_JDKB, size=c["size"],
                                          periodic=c.get("periodic", [True, True, False])))
        rng = np.random.default_rng(7)

        def dev(a):
            return torch.tensor(a, dtype=torch.float64, device="cuda")
        h, m0 = dev(0.3 * rng.normal(size=(lat.ncell, 3))), dev(workloads.random_sphere(lat.ncell, 7))
        tgt = dev(workloads.random_sphere(lat.ncell, 8))
        r = adjoint.SIBRunner(lat, c.get("names", ["J1", "D", "K"]), nsteps=13, timestep=1.0, damping=0.2, ckpt_every=5)
        try:
            out, gh, gm = torch.empty_like(m0), torch.empty_like(m0), torch.empty_like(m0)
            for th in before:
                r.forward(np.array(th), np.array([0.0, 0.1, 0.5]), h, m0, out)
            r.forward(np.array(c.get("theta", [1e-3, 0.3e-3, -0.05e-3])), np.array([0.0, 0.1, 0.5]), h, m0, out)
            gt, gb = r.backward((2 * (out - tgt)).contiguous(), gh, gm)
            torch.cuda.synchronize()
            return [out.cpu().numpy(), np.asarray(gt), np.asarray(gb), gh.cpu().numpy(), gm.cpu().numpy()]
        finally:
            r.close()
    finally:
        for k, v in old.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v


@pytest.mark.parametrize("name", sorted(CASES))
def test_compiled_equals_ahead_of_time(name):
    ref, got = _run(CASES[name], "0"), _run(CASES[name], "1")
    for a, b in zip(ref, got):
        assert np.isfinite(a).all() and np.array_equal(a, b), name


def test_other_parameters_in_the_same_runner():
    """Passes with other values, zero and of the other sign, before the one compared
    (the kernels stay, their values change; sums that round apart leave them)."""
    c = CASES["reach2"]
    before = ([2e-3, -0.1e-3, 0.0, 0.05e-3], [1e-3, 0.0, 0.0, 0.0], [-1e-3, 0.3e-3, 0.1e-3, 0.0])
    for a, b in zip(_run(c, "0"), _run(c, "1", before)):
        assert np.array_equal(a, b)
