"""GPU: the default schedule of a handle beside others: kernel attributes and
memory that several handles share, and which sweeps ran."""
import ctypes

import numpy as np
import pytest

from helpers import gpu_env, load_pkg, make_problem, oracle_for, relmax
from test_gpu_fused import SAME, compare

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


def planned(pkg, shape, precision):
    e = pkg.Microenvironment(*shape, 20.0, precision)
    try:
        return e.schedule()
    finally:
        e.close()


# whole planes: every kernel (x chunk, y chunk) that the plan can choose, with
# columns in one pass and, third entry set, in several; the last of each
# precision near the LDS limit
PLANES = [("fp64", (33, 17, 7, 2), (7, 8), 0), ("fp64", (257, 1, 267, 2), (7, 8), 1), ("fp64", (1, 73, 1, 1), (7, 16), 0),
          ("fp64", (24, 74, 9, 2), (7, 16), 0), ("fp64", (146, 127, 78, 2), (7, 16), 1), ("fp64", (328, 19, 3, 1), (13, 8), 0),
          ("fp64", (518, 1, 260, 1), (13, 8), 1), ("fp64", (551, 9, 1, 1), (13, 16), 0), ("fp64", (128, 96, 112, 1), (13, 16), 0),
          ("fp64", (262, 9, 549, 1), (13, 16), 1), ("fp64", (522, 18, 54, 1), (17, 8), 1), ("fp64", (425, 17, 7, 2), (17, 16), 0),
          ("fp64", (515, 26, 40, 2), (17, 16), 1), ("fp64", (501, 28, 12, 3), (17, 16), 0),
          ("fp32", (33, 17, 7, 2), (7, 8), 0), ("fp32", (266, 1, 526, 1), (7, 8), 1), ("fp32", (24, 74, 9, 2), (7, 16), 0),
          ("fp32", (450, 2, 3, 1), (13, 8), 0), ("fp32", (519, 1, 260, 1), (13, 8), 1), ("fp32", (520, 9, 1, 1), (13, 16), 0),
          ("fp32", (128, 96, 112, 1), (13, 16), 0), ("fp32", (257, 9, 275, 2), (13, 16), 1), ("fp32", (533, 17, 8, 3), (17, 8), 1),
          ("fp32", (421, 17, 1, 1), (17, 16), 0), ("fp32", (535, 25, 60, 1), (17, 16), 1), ("fp32", (569, 17, 15, 3), (25, 8), 1),
          ("fp32", (88, 163, 50, 1), (25, 16), 0), ("fp32", (775, 19, 36, 2), (25, 16), 1), ("fp32", (507, 62, 35, 3), (17, 16), 1)]


@pytest.mark.parametrize("precision,shape,kernel,passes", PLANES)
def test_planes_of_every_kernel(pkg, precision, shape, kernel, passes):
    s = planned(pkg, shape, precision)
    assert s[0] == "planes" and s[1:3] == kernel and (s[3] < shape[0]) == bool(passes), s
    for dirichlet, solver in (("all", "blocking"), ("mixed", "avx256d")):
        compare(pkg, shape, precision, dirichlet, solver, 1 if np.prod(shape) > 10 ** 6 else 2)


def test_the_plane_cases_reach_the_lds_limit(pkg):
    for precision in ("fp64", "fp32"):
        assert max(planned(pkg, sh, p)[5] for p, sh, *_ in PLANES if p == precision) > 128 << 10


@pytest.mark.parametrize("precision,shape,kernel,passes", PLANES)
def test_per_voxel_planes_of_every_kernel(pkg, precision, shape, kernel, passes):
    """Against the separate sweeps with their face passes."""
    nx, ny, nz, ns = shape
    p = make_problem(*shape, seed=sum(shape) + 17, dirichlet="mixed")
    v = np.random.default_rng(sum(shape)).uniform(0, 40, (nx, ny, nz, ns))
    planes = [v[0], v[-1], v[:, 0], v[:, -1], v[:, :, 0], v[:, :, -1]]
    out = []
    for separate in (False, True):
        e = gpu_env(pkg, p, precision)
        if separate:
            e.set_tiles(*e.tiles()[:3])
        e.set_dirichlet_planes(planes)
        assert e.schedule()[0] == ("separate" if separate else "planes")
        e.step(p.dt, 2)
        out.append(e.download().reshape(-1, ns))
        e.close()
    for d in range(ns):
        assert relmax(out[0][:, d], out[1][:, d]) <= SAME[precision], d


# 17 to 32 bricks per plane and more, and few of long rows; a middle field swept by plane
@pytest.mark.parametrize("shape,bricks", [((121, 426, 30, 1), 18), ((120, 830, 27, 1), 34), ((820, 51, 74, 2), 3),
                                          ((203, 157, 121, 3), 0)])
def test_fp32_bricks_and_planes_of_middle_fields(pkg, shape, bricks):
    s = planned(pkg, shape, "fp32")
    assert s[0] == ("bricks" if bricks else "planes") and (not bricks or s[3] == bricks), s
    compare(pkg, shape, "fp32", "mixed", "avx256d", 1)


# FP64 bricks of 20 and 16 rows, one block of 256, 512 and 1024 threads
@pytest.mark.parametrize("shape,rows,threads", [((150, 130, 450, 4), 20, 256), ((333, 90, 300, 4), 20, 512),
                                                ((500, 110, 170, 4), 16, 512), ((600, 70, 210, 4), 20, 1024)])
@pytest.mark.parametrize("dirichlet,solver", [("mixed", "avx256d"), ("mixed", "blocking"), ("off", "blocking")])
def test_fp64_bricks_with_free_faces_and_windows(pkg, shape, rows, threads, dirichlet, solver):
    """Against the separate sweeps; k-slabs, substrate streams and z tile runs
    give the same values bit for bit."""
    p = make_problem(*shape, seed=sum(shape), n_agents=50, dirichlet=dirichlet, collide=4)

    def run(setting):
        e = gpu_env(pkg, p, "fp64")
        e.set_solver(solver)
        setting(e)
        s = e.schedule()
        e.step(p.dt, 2)
        u = e.download().reshape(-1, p.ns)
        e.close()
        return s, u

    s, u = run(lambda e: None)
    assert s[0] == "bricks" and s[2] == rows and s[4] == threads, s
    assert np.isfinite(u).all()
    s, v = run(lambda e: e.set_tiles(*e.tiles()[:3]))
    assert s == ("separate",)
    for d in range(p.ns):
        assert relmax(u[:, d], v[:, d]) <= SAME["fp64"], d
    if solver == "avx256d":
        for setting in (lambda e: e.set_slab(71), lambda e: e.set_substrate_streams(2), lambda e: e.set_col_runs(1, 5)):
            s, v = run(setting)
            assert s[0] == "bricks"
            assert np.array_equal(u, v)


# fields from HBM on both sides of the lines of bricks_lose
@pytest.mark.parametrize("precision,shape,form", [
    ("fp32", (544, 505, 427, 3), "separate"), ("fp32", (545, 505, 427, 3), "bricks"), ("fp32", (628, 303, 256, 3), "separate"),
    ("fp32", (676, 303, 256, 3), "bricks"), ("fp32", (464, 464, 464, 1), "separate"), ("fp32", (464, 464, 400, 1), "bricks"),
    ("fp32", (464, 464, 551, 1), "bricks"), ("fp32", (416, 464, 464, 1), "bricks"), ("fp32", (400, 400, 400, 4), "bricks"),
    ("fp64", (353, 353, 353, 4), "separate"), ("fp64", (353, 353, 353, 2), "bricks"), ("fp64", (352, 353, 353, 4), "bricks"),
    ("fp64", (354, 353, 353, 4), "bricks"), ("fp64", (353, 353, 385, 4), "bricks"), ("fp64", (514, 353, 353, 1), "bricks"),
    ("fp64", (514, 353, 353, 3), "separate"), ("fp64", (400, 400, 400, 4), "bricks")])
def test_bricks_only_where_they_pay(pkg, precision, shape, form):
    assert planned(pkg, shape, precision)[0] == form


@pytest.mark.parametrize("shape,precision", [((180, 171, 60, 1), "fp32"), ((150, 130, 450, 4), "fp64")])
def test_bricks_keep_the_bars_up_to_their_largest_k(pkg, shape, precision):
    """k = D*dt/dx^2 up to 1000 against the oracle; from there on the separate
    sweeps, bit for bit, and bricks again for a smaller dt."""
    p = make_problem(*shape, seed=81, dirichlet="off")
    p.decay[:] = 0.1
    p.D[:] = 1000.0 * p.dx ** 2 / p.dt
    e, sep = gpu_env(pkg, p, precision), gpu_env(pkg, p, precision)
    try:
        sep.set_tiles(*sep.tiles()[:3])
        u = p.u0.copy()
        oracle_for(p).diffusion_step(u, p.dt)
        e.simulate_diffusion_decay(p.dt)
        assert e.schedule()[0] == "bricks"
        assert relmax(e.download(), u) <= TOL[precision]
        for x in (e, sep):
            x.upload(p.u0)
            x.step(100 * p.dt, 2)
        assert e.schedule() == ("separate",)
        assert np.array_equal(e.download(), sep.download())
        e.upload(p.u0)
        e.step(p.dt, 1)
        assert e.schedule()[0] == "bricks"
        assert relmax(e.download(), u) <= TOL[precision]
    finally:
        e.close()
        sep.close()


def test_memory_of_bricks_is_given_up_before_an_allocation_fails(pkg):
    """800^3 x 20 FP64: the gradients of the field (246 GB) do not fit beside it
    (82 GB).  The call fails as it did, and the handle has given its bricks up
    (8 GB) first; it goes on with the separate sweeps."""
    n, ns = 800, 20
    room, card = ctypes.c_size_t(), ctypes.c_size_t()
    L = pkg.lib()
    assert L.hipMemGetInfo(ctypes.byref(room), ctypes.byref(card)) == 0
    if room.value < 1.2e11 or card.value > 3.2e11:
        pytest.skip("sized for a card of 288 GiB")
    e = pkg.Microenvironment(n, n, n, ns, 20.0, "fp64")
    try:
        # zero decay and free faces: a uniform field stays as it is
        e.set_coefficients(np.linspace(1e3, 1e5, ns), np.zeros(ns))
        e.fill(np.arange(1.0, ns + 1))
        e.step(0.01, 1)
        assert e.schedule()[0] == "bricks"
        before = e.total_mass()
        one = np.zeros(1)
        assert L.bfa_gradients(e._h, one.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), 1) == 4  # no memory
        assert e.schedule() == ("separate",)
        e.step(0.01, 1)
        np.testing.assert_allclose(e.total_mass(), before, rtol=1e-12)
    finally:
        e.close()
