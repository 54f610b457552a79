"""GPU: the fused x + y sweep of the default schedule against the CPU oracle and
against the separate sweeps, which run when kernel shapes are set explicitly.

Bars: relative max-norm 1e-12 (FP64) and 1e-5 (FP32) against the oracle after
every step, as for the separate sweeps; between the two schedules, which run
the same recurrences and differ in the length of the x chunks, 1e-13 and 2e-6
(the batched solver's bar for its two schedules).
"""
import numpy as np
import pytest

import oracle
from helpers import agents_for, gpu_env, load_pkg, make_problem, oracle_for, relmax

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "fp32": 1e-5}
SAME = {"fp64": 1e-13, "fp32": 2e-6}


@pytest.fixture(scope="module")
def pkg():
    return load_pkg()


def compare(pkg, shape, precision, dirichlet, solver, steps=3):
    p = make_problem(*shape, seed=sum(shape) + 3, n_agents=40, dirichlet=dirichlet, collide=4)
    orc = oracle.Oracle(p.nx, p.ny, p.nz, p.ns, p.dx, p.D, p.decay, p.active, p.reg, p.fv, solver=solver)
    ag = agents_for(p)
    u = p.u0.copy()
    fused, sep = gpu_env(pkg, p, precision), gpu_env(pkg, p, precision)
    try:
        sep.set_tiles(*sep.tiles()[:3])
        for e in (fused, sep):
            e.set_solver(solver)
        for _ in range(steps):
            orc.diffusion_step(u, p.dt)
            orc.secretion_uptake(u, ag)
            fused.step(p.dt, 1)
            sep.step(p.dt, 1)
            f, s = (e.download().reshape(-1, p.ns) for e in (fused, sep))
            ref = u.reshape(-1, p.ns)
            for d in range(p.ns):
                assert relmax(f[:, d], ref[:, d]) <= TOL[precision], d
                assert relmax(f[:, d], s[:, d]) <= SAME[precision], d
    finally:
        fused.close()
        sep.close()


# bricks of FP32 rows: 25 rows and one more or less per plane, two bricks and
# many, whole and ragged 16-byte rows, z lines of two chunks and of several with
# every kind of remainder, more and fewer columns than a block has threads
BRICKS32 = [(180, 171, 26, 1), (187, 200, 50, 2), (259, 151, 51, 1), (513, 80, 33, 1), (832, 51, 74, 2), (190, 176, 75, 3),
            (120, 400, 30, 2)]


@pytest.mark.parametrize("shape", BRICKS32)
def test_bricks_match_the_oracle_and_the_separate_sweeps(pkg, shape):
    for dirichlet, solver in (("all", "blocking"), ("mixed", "avx256d"), ("mixed", "blocking"), ("off", "blocking")):
        compare(pkg, shape, "fp32", dirichlet, solver, 2)


@pytest.mark.parametrize("shape,precision", [((64, 801, 701), "fp64"), ((511, 270, 251), "fp64"), ((333, 401, 260), "fp64"),
                                             ((810, 541, 77), "fp64"), ((331, 512, 501), "fp32")])
def test_bricks_of_large_fields(pkg, shape, precision):
    """Fields larger than the last-level cache, against the oracle: FP64 bricks
    of 16 and 20 rows with a z block per few rows."""
    compare(pkg, shape + (1,), precision, "all", "blocking", 1)


# one row, one column, one plane; rows of whole chunks (7, 13, 17, 25 nodes) and
# one node either side of them; rows that are and are not whole 16-byte vectors;
# one and several rows per wavefront; y chunks of 8 and 16 with every kind of
# remainder; columns in one and in several passes; planes near the LDS limit
PLANES = [(1, 5, 3, 2), (5, 1, 7, 1), (31, 17, 1, 2), (28, 16, 9, 1), (27, 33, 5, 2), (29, 32, 6, 1), (64, 63, 5, 1),
          (100, 100, 6, 2), (101, 97, 4, 3), (257, 41, 12, 2), (453, 15, 3, 1), (12, 300, 5, 1), (203, 157, 200, 1),
          (150, 129, 150, 1)]


@pytest.mark.parametrize("shape", PLANES)
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_planes_match_the_oracle_and_the_separate_sweeps(pkg, shape, precision):
    steps = 1 if np.prod(shape) > 10 ** 6 else 3
    for dirichlet, solver in (("all", "blocking"), ("mixed", "avx256d"), ("off", "blocking")):
        compare(pkg, shape, precision, dirichlet, solver, steps)


@pytest.mark.parametrize("shape,precision", [((45, 38, 23, 3), "fp64"), ((45, 38, 23, 3), "fp32"),
                                             ((190, 176, 40, 3), "fp32")])
def test_windows_of_planes_are_bit_identical(pkg, shape, precision):
    """The slab and substrate-stream schedules sweep windows of planes and of
    substrates; the values do not depend on the window.  Shapes that are set
    and given back leave the default schedule as it was."""
    p = make_problem(*shape, seed=5, n_agents=30, dirichlet="mixed", collide=4)
    out = []
    for slab, streams, tiles in ((0, 1, False), (7, 1, False), (23, 1, False), (0, 2, False), (0, 1, True)):
        e = gpu_env(pkg, p, precision)
        if tiles:
            e.set_tiles(8, 8, 8)
            e.step(p.dt, 0)
            e.set_tiles(0, 0, 0)
        e.set_slab(slab)
        e.set_substrate_streams(streams)
        e.step(p.dt, 3)
        out.append(e.download())
        e.close()
    for o in out[1:]:
        assert np.array_equal(o, out[0])


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_batch_planes_of_every_block_class(pkg, precision):
    """Members on both sides of the limits of the batch's fused sweep: planes
    for blocks of 256, 512 and 1024 threads, one past the plane buffer and one
    past its column chunks, against the oracle and the separate sweeps."""
    shapes = [(1, 1, 4, 1), (7, 16, 9, 2), (33, 17, 5, 3), (64, 75, 6, 1), (65, 131, 5, 2), (128, 128, 4, 1),
              (160, 160, 3, 1), (181, 181, 3, 1), (16, 321, 4, 1), (18, 320, 4, 2), (512, 31, 3, 1)]
    ps = [make_problem(*sh, seed=900 + k, n_agents=20, dirichlet=("all", "mixed", "off")[k % 3], collide=3)
          for k, sh in enumerate(shapes)]
    out = {}
    for fuse in (True, False):
        with pkg.Batch(precision) as b:
            if not fuse:
                b.set_fusion(False)
            ids = []
            for p in ps:
                ids.append(b.add(p.nx, p.ny, p.nz, p.ns, p.dx, p.D, p.decay, p.active, p.reg, p.fv))
                b.upload(ids[-1], p.u0)
                b.set_agents(ids[-1], p.voxel, p.c1, p.c2, p.e2, p.agent_active)
            b.step(ps[0].dt, 2)
            out[fuse] = [b.download(i) for i in ids]
    for p, f, s in zip(ps, out[True], out[False]):
        orc, ag, u = oracle_for(p), agents_for(p), p.u0.copy()
        for _ in range(2):
            orc.diffusion_step(u, p.dt)
            orc.secretion_uptake(u, ag)
        f, s, ref = (x.reshape(-1, p.ns) for x in (f, s, u))
        for d in range(p.ns):
            assert relmax(f[:, d], ref[:, d]) <= TOL[precision], (p.nx, p.ny, d)
            assert relmax(f[:, d], s[:, d]) <= SAME[precision], (p.nx, p.ny, d)


@pytest.mark.parametrize("shape", [(1, 5, 3, 2), (5, 1, 7, 1), (31, 17, 1, 2), (29, 33, 6, 3), (64, 63, 5, 1), (257, 41, 12, 2),
                                   (12, 300, 5, 1), (128, 96, 20, 1)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_per_voxel_dirichlet_planes(pkg, shape, precision):
    """Values that vary along the faces, on both schedules and both solvers."""
    nx, ny, nz, ns = shape
    for dirichlet, solver in (("all", "blocking"), ("mixed", "avx256d")):
        p = make_problem(*shape, seed=sum(shape) + 11, n_agents=20, dirichlet=dirichlet, collide=3)
        v = np.random.default_rng(sum(shape)).uniform(0, 40, (nx, ny, nz, ns))
        planes = [v[0], v[-1], v[:, 0], v[:, -1], v[:, :, 0], v[:, :, -1]]
        out = []
        for separate in (False, True):
            e = gpu_env(pkg, p, precision)
            if separate:
                e.set_tiles(*e.tiles()[:3])
            e.set_solver(solver)
            e.set_dirichlet_planes(planes)
            e.step(p.dt, 3)
            out.append(e.download().reshape(-1, ns))
            e.close()
        for d in range(ns):
            assert relmax(out[0][:, d], out[1][:, d]) <= SAME[precision], (solver, d)
