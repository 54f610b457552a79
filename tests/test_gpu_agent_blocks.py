"""GPU: the device blocks that a handle keeps between agent-state and gradient
calls.  Agent counts that change from call to call (none, one, more and fewer
than before, past the largest kept block) give bit for bit what a new handle
gives, whichever blocks the earlier calls left."""
import numpy as np
import pytest

from helpers import load_pkg, make_problem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pkg():
    return load_pkg()


def agents(p, n, seed):
    rng = np.random.default_rng(seed)
    half = 0.5 * p.dx * np.array([p.nx, p.ny, p.nz])
    return (rng.uniform(-half, half, (n, 3)), np.concatenate([-half, half]), rng.uniform(1000, 4000, n),
            rng.uniform(0, 10, (n, p.ns)), rng.uniform(0, 10, (n, p.ns)), rng.uniform(0, 20, (n, p.ns)),
            rng.uniform(0, 40, (n, p.ns)))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_changing_agent_counts_equal_a_new_handle(pkg, precision):
    p = make_problem(25, 18, 14, 3, seed=77, dirichlet="mixed")

    def env():
        e = pkg.Microenvironment(p.nx, p.ny, p.nz, p.ns, p.dx, precision)
        e.set_coefficients(p.D, p.decay)
        e.set_dirichlet(p.active, p.reg, p.fv)
        e.upload(p.u0)
        return e

    kept = env()
    try:
        for k, n in enumerate((500, 0, 1, 513, 40, 3000000, 499, 500)):
            st = agents(p, n, 100 + k)
            vox = np.arange(0, p.nx * p.ny * p.nz, 7 + k, dtype=np.int32)
            got = []
            for e in (kept, env()):
                e.upload(p.u0)
                e.set_agents_state(*st, p.dt)
                e.step(p.dt, 2)
                # agents given as constants in between leave blocks behind
                e.set_agents(np.zeros(1, np.int32), np.zeros((1, p.ns)), np.ones((1, p.ns)), np.zeros((1, p.ns)))
                e.set_agents_state(*st, p.dt)
                e.step(p.dt, 1)
                got.append((e.gradients_at(vox), e.download()))
                if e is not kept:
                    e.close()
            assert np.array_equal(got[0][0], got[1][0]), n
            assert np.array_equal(got[0][1], got[1][1]), n
    finally:
        kept.close()
