"""CPU tests of the autotuner's comparison with the default schedule, on the
stand-in and the fake clock of the other searches: it is timed with its own
best z tile runs and substrate streams where it sweeps x and y together."""
import time

import pytest

from test_autotune import Clock, FakeEnv, load_autotune


class FakeFusedEnv(FakeEnv):
    """FakeEnv whose default schedule (all shapes 0) sweeps x and y in `xy` ms
    and z in 0.44 ms, 0.03 less with 5 tile runs, 3 % less with two streams."""

    xy = 0.6
    form = ("bricks", 13, 25, 16, 512, 54720)
    made = []

    def __init__(self, *a):
        super().__init__(*a)
        self.default = True
        FakeFusedEnv.made.append(self)

    def schedule(self):
        return self.form if self.default else ("separate",)

    def set_tiles(self, *shape):
        self.default = not any(shape)
        super().set_tiles(*(shape if any(shape) else (16, 16, 16, 0, 32, 32)))

    def kernel_ms(self):
        if not self.default:
            return super().kernel_ms()
        return [self.xy, 0.0, 0.44 - 0.03 * (self.runs[1] == 5), 0.03]

    def step(self, dt, n):
        t = sum(self.kernel_ms()) * ((0.97 if self.default else 0.98) if self.split == 2 else 1.0)
        self.clock.t += t * n * 1e-3


def search(monkeypatch, env, ns=4):
    at = load_autotune()
    clock = Clock()
    monkeypatch.setattr(time, "perf_counter", clock)
    FakeEnv.clock = clock

    class Pkg:
        Microenvironment = env

    return at, at.autotune(Pkg, 400, 400, 400, ns, "fp32", 0.01)


SHAPES = ("Lx", "rows_x", "Ly", "cols_y", "Lz", "cols_z", "x_grid")


@pytest.mark.parametrize("ns", [1, 4])
def test_default_schedule_wins_with_its_own_runs_and_streams(monkeypatch, ns):
    at, res = search(monkeypatch, FakeFusedEnv, ns)
    assert [res[k] for k in SHAPES] == [0] * 7
    assert (res["runs_y"], res["runs_z"], res["slab"], res["substrate_streams"]) == (1, 5, 0, 2 if ns > 1 else 1)
    assert res["ms"]["step"] == pytest.approx((0.6 + 0.41 + 0.03) * (0.97 if ns > 1 else 1.0))
    env = FakeFusedEnv("", "", "", ns, 20.0, "fp32")
    at.apply(env, res)
    assert env.default and env.runs == (1, 5) and env.split == res["substrate_streams"]


def test_slower_default_schedule_is_timed_and_not_kept(monkeypatch):
    class Slow(FakeFusedEnv):
        xy = 0.8  # 1.24 ms x 0.97 against 1.22 x 0.98

    at, res = search(monkeypatch, Slow)
    assert res["Lx"] == 8 and res["runs_z"] == 3 and res["substrate_streams"] == 2
    timed = [t for t in res["trials"] if t.get("default") and t["axis"] == "schedule"]
    assert [t["substrate_streams"] for t in timed] == [1, 2]
    assert min(t["ms_step"] for t in timed) > res["ms"]["step"]


def test_separate_default_schedule_is_not_timed_again(monkeypatch):
    class Separate(FakeFusedEnv):
        form = ("separate",)

    at, res = search(monkeypatch, Separate)
    assert not [t for t in res["trials"] if t.get("default")]


def test_errors_of_the_default_schedule_are_not_swallowed(monkeypatch):
    class Broken(FakeFusedEnv):
        def set_tiles(self, *shape):
            super().set_tiles(*shape)
            if not any(shape):
                raise RuntimeError("device lost")

    with pytest.raises(RuntimeError, match="device lost"):
        search(monkeypatch, Broken)
