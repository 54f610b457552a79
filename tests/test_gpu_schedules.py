"""GPU: the default schedule of a handle beside others: kernel attributes and
memory that several handles share, and which sweeps ran."""
import ctypes

import numpy as np
import pytest

from helpers import agents_for, gpu_env, load_pkg, make_problem, oracle_for, relmax

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "fp32": 1e-5}


@pytest.fixture(scope="module")
def pkg():
    return load_pkg()


# pairs of grids that run the same kernel with different needs of LDS above
# 64 KiB (whole planes; bricks of 25 FP32 rows)
@pytest.mark.parametrize("precision,large,small", [("fp64", (340, 44, 40), (418, 19, 40)), ("fp64", (340, 24, 3), (328, 19, 3)),
                                                   ("fp32", (203, 157, 121), (325, 44, 3)),
                                                   ("fp32", (832, 51, 74), (680, 51, 74))])
def test_lds_of_one_handle_does_not_limit_another(pkg, precision, large, small):
    """The dynamic LDS limit belongs to the kernel, not to the handle: a handle
    that needs more still launches after one that needs less was made, and
    after the separate sweeps' shapes were set and given back."""
    ps = [make_problem(*sh, 1, seed=61 + k, dirichlet="all") for k, sh in enumerate((large, small))]
    envs = [gpu_env(pkg, p, precision) for p in ps]
    try:
        envs[1].set_tiles(*envs[1].tiles()[:3])
        envs[1].set_tiles(0, 0, 0)
        for e, p in zip(envs, ps):
            u = p.u0.copy()
            orc = oracle_for(p)
            for _ in range(2):
                orc.diffusion_step(u, p.dt)
            e.step(p.dt, 2)
            assert relmax(e.download(), u) <= TOL[precision]
    finally:
        for e in envs:
            e.close()


def test_memory_of_the_fused_sweep_is_held_while_it_runs(pkg):
    """A bricked FP32 field needs a second field; a handle holds it from the
    first step on the default schedule, and not while kernel shapes or
    per-voxel planes are set.  The values are those of a handle that always
    had the setting."""
    n, ns = 250, 1
    field = n ** 3 * 4
    slack = field // 4  # streams, tables and the allocator's rounding
    p = make_problem(n, n, n, ns, seed=71, dirichlet="all")
    v = np.random.default_rng(72).uniform(0, 40, (n, n, n, ns))
    planes = [v[0], v[-1], v[:, 0], v[:, -1], v[:, :, 0], v[:, :, -1]]

    def free_bytes():
        room, card = ctypes.c_size_t(), ctypes.c_size_t()
        assert pkg.lib().hipMemGetInfo(ctypes.byref(room), ctypes.byref(card)) == 0
        return room.value

    def make():
        e = pkg.Microenvironment(p.nx, p.ny, p.nz, p.ns, p.dx, "fp32")
        e.set_coefficients(p.D, p.decay)
        e.set_dirichlet(p.active, p.reg, p.fv)
        e.set_fp32_basis(p.fv[0], np.full(ns, 8.0))
        return e

    def run(e, steps=2):
        e.upload(p.u0)
        e.step(p.dt, steps)
        return e.download()

    warm = make()  # code objects, transfer buffers
    run(warm)
    warm.set_tiles(8, 8, 8)
    run(warm)
    warm.close()
    free = free_bytes()
    used = lambda: free - free_bytes()  # noqa: E731
    e, sep, pv = make(), make(), make()
    try:
        held = used()
        assert held < 4 * field
        sep.set_tiles(8, 8, 8)
        pv.set_dirichlet_planes(planes)
        want = [run(x) for x in (sep, pv)]
        assert used() <= held + slack
        first = run(e)
        assert held + field <= used() <= held + field + slack
        e.set_tiles(8, 8, 8)
        assert used() <= held + slack
        assert np.array_equal(run(e), want[0])
        e.set_tiles(0, 0, 0)
        assert np.array_equal(run(e), first)
        assert used() >= held + field
        e.set_dirichlet_planes(planes)
        assert used() <= held + slack
        assert np.array_equal(run(e), want[1])
        e.set_dirichlet_planes(None)
        # coefficients kept from the first dt are those of the fused sweep too
        e.set_dt_caching(True)
        assert np.array_equal(run(e), first)
        e.set_tiles(8, 8, 8)
        e.set_tiles(0, 0, 0)
        e.step(2 * p.dt, 1)
        pv.set_dirichlet_planes(None)
        assert np.array_equal(e.download(), run(pv, 3))
    finally:
        for x in (e, sep, pv):
            x.close()
    assert used() < field
