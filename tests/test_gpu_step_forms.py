"""GPU: the forms that a step takes besides the default ones of small grids.
Fields above 40 MiB replay a captured graph, kernel shapes that are set run the
separate sweeps, and a batch may be kept from the fused sweep."""
import numpy as np
import pytest

from helpers import agents_for, gpu_env, load_pkg, make_problem, oracle_for, relmax

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "fp32": 1e-5}

# above 40 MiB: whole planes, separate sweeps, FP32 bricks, FP64 bricks
LARGE = [((203, 157, 121, 3), "fp32", "planes"), ((131, 257, 170, 1), "fp64", "separate"), ((250, 250, 200, 1), "fp32", "bricks"),
         ((150, 130, 450, 4), "fp64", "bricks")]


@pytest.fixture(scope="module")
def pkg():
    return load_pkg()


@pytest.mark.parametrize("shape,precision,form", LARGE)
def test_replayed_steps_equal_eager_calls(pkg, shape, precision, form):
    """Several replays per call and several calls, with the handle's own eager
    work and downloads between them."""
    p = make_problem(*shape, seed=401, n_agents=300, dirichlet="mixed", export=5.0, collide=4)
    a, b = gpu_env(pkg, p, precision), gpu_env(pkg, p, precision)
    try:
        assert a.schedule()[0] == form
        for n in (1, 4, 3):
            a.step(p.dt, n)
            a.simulate_cell_sources_and_sinks()
            for _ in range(n):
                b.simulate_diffusion_decay(p.dt)
                b.simulate_cell_sources_and_sinks()
            b.simulate_cell_sources_and_sinks()
            assert np.array_equal(a.download(), b.download()), n
        assert a.schedule()[0] == form
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("shape,precision,form", LARGE)
def test_setters_right_after_replayed_steps(pkg, shape, precision, form):
    """Calls that replace what a queued graph reads: the result equals a run
    that is synchronised before every call."""
    p = make_problem(*shape, seed=402, n_agents=300, dirichlet="mixed", collide=3)

    def run(sync):
        env = gpu_env(pkg, p, precision)
        try:
            assert env.schedule()[0] == form
            for call in (lambda: env.set_coefficients(p.D * 1.5, p.decay), lambda: env.step(p.dt * 2, 1),
                         lambda: env.set_tiles(8, 8, 8, 0, 16, 16), lambda: env.set_tiles(0, 0, 0),
                         lambda: env.set_col_runs(3, 2), lambda: env.set_substrate_streams(2),
                         lambda: env.set_slab(7), lambda: env.set_slab(0),
                         lambda: env.set_agents(p.voxel[::-1].copy(), p.c1[::-1], p.c2[::-1], p.e2[::-1])):
                env.step(p.dt, 4)
                if sync:
                    env.synchronize()
                call()
            env.step(p.dt, 2)
            return env.download()
        finally:
            env.close()

    assert np.array_equal(run(False), run(True))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("lx", [8, 16])
def test_x_grid_of_the_wave_sweep_is_bit_identical(pkg, precision, lx):
    p = make_problem(57, 33, 29, 3, seed=403, n_agents=120, dirichlet="mixed")
    out = []
    for g in (0, 1, 2, 3, 9):
        env = gpu_env(pkg, p, precision)
        env.set_tiles(lx, 0, 0, 0, 0, 0)
        env.set_x_grid(g)
        assert env.schedule() == ("separate",)
        env.step(p.dt, 2)
        out.append(env.download())
        env.close()
    for o in out[1:]:
        assert np.array_equal(o, out[0])


SHAPES = {"fp64": [(8, 16, 8, 32, 16), (16, 8, 16, 16, 32), (32, 32, 32, 16, 16)],
          "fp32": [(8, 32, 32, 64, 64), (16, 8, 4, 16, 32), (32, 16, 16, 32, 128)]}


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_batch_shapes_of_the_separate_sweeps(pkg, precision):
    """Every x chunk and column shape family, and every column block size, on
    members that would otherwise take the fused sweep."""
    ps = [make_problem(*sh, seed=410 + k, n_agents=30, dirichlet=("all", "mixed", "off")[k % 3], collide=3)
          for k, sh in enumerate([(40, 37, 100, 2), (64, 160, 20, 1), (9, 16, 33, 3), (100, 64, 31, 1)])]

    def add(b, p):
        mid = b.add(p.nx, p.ny, p.nz, p.ns, p.dx, p.D, p.decay, p.active, p.reg, p.fv)
        b.upload(mid, p.u0)
        b.set_agents(mid, p.voxel, p.c1, p.c2, p.e2, p.agent_active)
        return mid

    with pkg.Batch(precision) as b:
        ids = [add(b, p) for p in ps]
        assert b.fused_members() == len(ps)
        b.set_fusion(False)
        assert b.fused_members() == 0
        for shape in SHAPES[precision]:
            b.set_tiles(*shape)
            b.step(ps[0].dt, 1)
        got = [b.download(i) for i in ids]
    for p, g in zip(ps, got):
        orc, ag, u = oracle_for(p), agents_for(p), p.u0.copy()
        for _ in SHAPES[precision]:
            orc.diffusion_step(u, p.dt)
            orc.secretion_uptake(u, ag)
        g, u = g.reshape(-1, p.ns), u.reshape(-1, p.ns)
        for d in range(p.ns):
            assert relmax(g[:, d], u[:, d]) <= TOL[precision], (p.nx, d)
    ref = None
    for thr in (0, 512, 768, 1024):
        with pkg.Batch(precision) as b:
            b.set_fusion(False)
            ids = [add(b, p) for p in ps]
            b.set_tiles(*((8, 16, 16, 32, 32) if precision == "fp32" else (8, 8, 8, 32, 32)))
            b.set_col_threads(thr)
            b.step(ps[0].dt, 2)
            out = [b.download(i) for i in ids]
        if ref is not None:
            assert all(np.array_equal(x, y) for x, y in zip(out, ref)), thr
        ref = out


@pytest.mark.parametrize("shape,precision", [((64, 48, 40, 2), "fp64"), ((180, 171, 26, 1), "fp32")])
def test_autotuned_settings_apply_and_keep_the_bars(pkg, shape, precision):
    import importlib

    at = importlib.import_module("physicellx_amd.autotune")
    res = at.autotune(pkg, *shape, precision, reps=2)
    assert [t for t in res["trials"] if t.get("default") and t["axis"] == "schedule"]
    p = make_problem(*shape, seed=420, n_agents=50, dirichlet="mixed", collide=3)
    orc, ag, u = oracle_for(p), agents_for(p), p.u0.copy()
    env = gpu_env(pkg, p, precision)
    try:
        at.apply(env, res)
        env.step(p.dt, 2)
        for _ in range(2):
            orc.diffusion_step(u, p.dt)
            orc.secretion_uptake(u, ag)
        g, u = env.download().reshape(-1, p.ns), u.reshape(-1, p.ns)
        for d in range(p.ns):
            assert relmax(g[:, d], u[:, d]) <= TOL[precision], d
    finally:
        env.close()
