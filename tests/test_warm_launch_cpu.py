"""Warm launches of autotuned, callable-grid and deuteron kernels on the CPU,
with stand-in kernels: the short path passes what the first launch passes and
gives way to the full one whenever a fact it rests on changes."""

import re

import pytest
import torch

import newt_amd as newt
import newt_amd.deuteron as dt
import newt_amd.language as nl
from newt_amd import testing
from newt_amd.runtime.autotuner import Autotuner


class _Recorder:
    param_names = ["x", "n", "scale"]
    defaults = {"scale": 2.0}

    def __init__(self):
        self.calls = []

    def __getitem__(self, grid):
        return lambda *args, **kw: self.calls.append((grid, args, kw))


@pytest.fixture
def tuner(monkeypatch):
    monkeypatch.setattr(testing, "do_bench", lambda fn, warmup, rep: (fn(), 1.0)[1])
    return Autotuner(_Recorder(), [newt.Config({"BLOCK": b}, num_warps=4) for b in (1, 2)],
                     key=["n", "x"])


def test_warm_call_launches_the_tuned_config(tuner):
    x = torch.zeros(4)
    tuner[(3,)](x, 7, 1.0)
    n = len(tuner.jitfn.calls)
    first = tuner.jitfn.calls[-1]
    tuner[(3,)](x, 7, 1.0)
    assert len(tuner.jitfn.calls) == n + 1 and tuner.jitfn.calls[-1] == first


@pytest.mark.parametrize("args,kwargs", [
    ((torch.zeros(4), 8, 1.0), {}),                       # key value
    ((torch.zeros(5), 7, 1.0), {}),                       # key tensor's shape
    ((torch.zeros(4).half(), 7, 1.0), {}),                # dtype
])
def test_another_key_is_tuned_again(tuner, args, kwargs):
    tuner[(3,)](torch.zeros(4), 7, 1.0)
    n = len(tuner.timings)
    tuner[(3,)](*args, **kwargs)
    assert len(tuner.timings) == n + 1


def test_calls_the_short_path_does_not_take(tuner):
    """Keyword arguments and defaults bind by name, an emptied cache tunes."""
    x = torch.zeros(4)
    tuner[(3,)](x, 7, 1.0)
    n = len(tuner.timings)
    tuner[(3,)](x, n=7, scale=1.0)
    tuner[(3,)](x, 7)
    assert len(tuner.timings) == n
    tuner.cache.clear()
    m = len(tuner.jitfn.calls)
    tuner[(3,)](x, 7, 1.0)
    assert len(tuner.jitfn.calls) > m + 2


def test_default_key_argument_keeps_the_full_path(monkeypatch):
    monkeypatch.setattr(testing, "do_bench", lambda fn, warmup, rep: 1.0)
    t = Autotuner(_Recorder(), [newt.Config({"BLOCK": 1})], key=["scale"])
    for _ in range(2):
        t[(1,)](torch.zeros(1), 1)
    assert list(t.timings) == [(2.0, "torch.float32")]


@newt.jit
def k(x_ptr, n, BLOCK: nl.constexpr = 64):
    nl.store(x_ptr + nl.arange(0, BLOCK), 1.0)


def test_callable_grid_sees_meta():
    seen = []
    grid = k._grid_of(lambda m: (seen.append(m), (m["n"] // m["BLOCK"],))[1], ("x", 640),
                      {"num_stages": 2, "waves_per_eu": 1})
    assert grid == (10,) and seen == [{"x_ptr": "x", "n": 640, "BLOCK": 64, "num_warps": 4}]
    assert k._grid_of(lambda m: m["num_warps"], ("x", 1), {"num_warps": 8, "BLOCK": 1}) == 8


@dt.kernel(config={"BLOCK_TILE_M": 8, "num_warps": 2})
def scaled_rows(x, y, out, s):
    for tile_m in dt.tile(x.shape[0]):
        out[tile_m, :] = x[tile_m, :] * y[:] + s


def test_deuteron_launch_arguments():
    """Pointers, sizes and strides in the traced order, grid and spans from the
    call's own extents."""
    x, y = torch.zeros(20, 50).t().contiguous().t(), torch.zeros(50)
    out = torch.zeros(20, 50)
    spec = scaled_rows._specialize((x, y, out, 2.0))
    rec = _Recorder()
    spec.jit = rec
    for rows in (20, 17):
        a = (x[:rows], y, out[:rows], 2.0)
        spec.launch(a, scaled_rows.fixed_config)
        grid, args, kw = rec.calls[-1]
        assert grid == (-(-rows // 8),)
        want = []
        for e in spec.traced.args:
            v = a[spec.index[e[1]]]
            want.append(v)
            if e[0] == "tensor":
                want += list(v.shape) + list(v.stride())
        assert len(args) == len(want)
        assert all(p is q or p == q for p, q in zip(args, want))
        assert kw["num_warps"] == 2 and kw["BLOCK_TILE_M"] == 8 and 64 in kw.values()


@dt.kernel(autotune=False)
def doubled(x, out):
    for t in dt.tile(x.shape[0]):
        out[t] = x[t] * 2.0


def test_varying_lengths_keep_a_bounded_table():
    """One length after another: the classes' configurations stay, the table
    of exact shapes does not grow for the life of the kernel."""
    from newt_amd.deuteron import runtime
    spec, classes = None, {}
    x = torch.zeros(5000)
    for n in (*range(1, 5000), 3, 4999):
        a = (x[:n], x[:n])
        spec = doubled._specialize(a)
        cfg = doubled._choose(spec, a)
        assert classes.setdefault(doubled.tuning_key(spec, a), cfg) is cfg
        assert len(doubled._keys) <= runtime._MAX_KEYS
    assert len(doubled._chosen) == len(classes) == 14


@pytest.mark.parametrize("args,kw,error", [
    ((1,), {}, "missing kernel arguments: ['n']"), ((), {"n": 1}, "missing kernel arguments: ['x_ptr']"),
    ((1, 2, 3, 4), {}, "takes 3 arguments but 4 were given"),
    ((1, 2), {"BLOK": 64}, "unknown kernel arguments: ['BLOK']")])
def test_wrong_arguments_are_named_before_the_grid_reads_them(monkeypatch, args, kw, error):
    from newt_amd.runtime import jit as J
    monkeypatch.setattr(J, "_C_LAUNCH", type("C", (), {"run": staticmethod(lambda *a: False)}))
    monkeypatch.setattr(J._Dev, "ready", True)
    monkeypatch.setattr(J._Dev, "device", staticmethod(lambda: 0))
    with pytest.raises(TypeError, match=re.escape(error)):
        k[lambda m: (m["n"] // m["BLOK"] if "BLOK" in m else m["x_ptr"] + m["n"],)](*args, **kw)


def test_a_grids_own_error_reaches_the_caller(monkeypatch):
    from newt_amd.runtime import jit as J
    monkeypatch.setattr(J, "_C_LAUNCH", type("C", (), {"run": staticmethod(lambda *a: False)}))
    monkeypatch.setattr(J._Dev, "ready", True)
    monkeypatch.setattr(J._Dev, "device", staticmethod(lambda: 0))
    monkeypatch.setattr(J.JITFunction, "_slow_path", lambda *a: (None, None))
    with pytest.raises(KeyError, match="ROWS"):
        k[lambda m: (m["ROWS"],)](1, 640)
