"""GPU: what the field holds at the voxels of a held face before a step.  The
first Dirichlet pass sets these voxels, so a NaN or an infinity there must not
reach any other voxel: bit for bit the result of the same field with finite
values on the faces."""
import numpy as np
import pytest

from helpers import gpu_env, load_pkg, make_problem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pkg():
    return load_pkg()


def fields(p):
    """u0 with NaN and infinities, and with the face values, at the boundary."""
    out = []
    for bad in (True, False):
        u = p.u0.reshape(p.nx, p.ny, p.nz, p.ns).copy()
        edge = np.ones(u.shape[:3], bool)
        edge[1:-1, 1:-1, 1:-1] = False
        u[edge] = p.fv[0]
        if bad:
            u[edge] = np.nan
            u[0, 0], u[-1, :, 0] = np.inf, -np.inf
        out.append(u.ravel())
    return out


# whole planes with several rows per wavefront and with one, bricks in both precisions
@pytest.mark.parametrize("shape,precision", [((31, 17, 9, 2), "fp64"), ((31, 17, 9, 2), "fp32"), ((300, 24, 8, 1), "fp64"),
                                             ((64, 3, 5, 2), "fp64"), ((64, 3, 5, 2), "fp32"), ((180, 171, 26, 1), "fp32"),
                                             ((259, 151, 51, 1), "fp32"), ((400, 300, 290, 1), "fp64")])
def test_values_under_held_faces_do_not_spread(pkg, shape, precision):
    p = make_problem(*shape, seed=21, n_agents=20, dirichlet="all", collide=3)
    got = []
    for u in fields(p):
        e = gpu_env(pkg, p, precision)
        e.set_fp32_basis(p.fv[0], np.full(p.ns, 8.0))
        e.upload(u)
        e.step(p.dt, 2)
        got.append(e.download())
        e.close()
    assert np.isfinite(got[1]).all()
    assert np.array_equal(*got)


@pytest.mark.parametrize("shape", [(31, 17, 9, 2), (64, 63, 5, 1), (12, 300, 5, 1)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_values_under_per_voxel_planes_do_not_spread(pkg, shape, precision):
    p = make_problem(*shape, seed=22, dirichlet="all")
    v = np.random.default_rng(3).uniform(0, 40, (p.nx, p.ny, p.nz, p.ns))
    planes = [v[0], v[-1], v[:, 0], v[:, -1], v[:, :, 0], v[:, :, -1]]
    got = []
    for u in fields(p):
        e = gpu_env(pkg, p, precision)
        e.set_dirichlet_planes(planes)
        e.set_fp32_basis(p.fv[0], np.full(p.ns, 8.0))
        e.upload(u)
        e.step(p.dt, 2)
        got.append(e.download())
        e.close()
    assert np.isfinite(got[1]).all()
    assert np.array_equal(*got)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_values_under_held_faces_of_batch_members_do_not_spread(pkg, precision):
    ps = [make_problem(*sh, seed=31 + k, dirichlet="all") for k, sh in
          enumerate([(7, 16, 9, 2), (33, 17, 5, 3), (65, 131, 5, 2), (160, 160, 3, 1)])]
    got = []
    for q in range(2):
        with pkg.Batch(precision) as b:
            ids = []
            for p in ps:
                ids.append(b.add(p.nx, p.ny, p.nz, p.ns, p.dx, p.D, p.decay, p.active, p.reg, p.fv))
                u = fields(p)[q]
                # the batch chooses its FP32 scale from the finite values
                b.upload(ids[-1], np.where(np.isinf(u), np.nan, u))
            b.step(ps[0].dt, 2)
            got.append([b.download(i) for i in ids])
    for x, y in zip(*got):
        assert np.isfinite(y).all()
        assert np.array_equal(x, y)
