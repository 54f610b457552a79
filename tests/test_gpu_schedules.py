"""GPU: the default schedule of a handle beside others: kernel attributes and
memory that several handles share, and which sweeps ran."""
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
