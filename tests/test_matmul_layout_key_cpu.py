"""matmul tunes per operand layout, with stand-in kernels: a shape used in
another storage order, or in rows that lose their 16-byte alignment, is tuned
again; the same layout at another row stride is not."""

import pytest
import torch

import newt_amd as newt
from newt_amd import testing
from newt_amd import workloads as W
from newt_amd.runtime.autotuner import Autotuner


class _Recorder:
    param_names = W.matmul_kernel.param_names
    defaults = {}

    def __init__(self):
        self.calls = []

    def __getitem__(self, grid):
        return lambda *args, **kw: self.calls.append((args, kw))


@pytest.fixture
def tuner(monkeypatch):
    monkeypatch.setattr(testing, "do_bench", lambda fn, warmup, rep: (fn(), 1.0)[1])
    t = Autotuner(_Recorder(), [newt.Config({"BLOCK_M": 16, "BLOCK_N": 16, "BLOCK_K": 32})],
                  key=W.matmul_tuned_small.key)
    monkeypatch.setattr(W, "matmul_tuned_small", t)
    return t


def rows(n, m, ld=None, dtype=torch.bfloat16):
    ld = ld or m
    return torch.zeros(n * ld, dtype=dtype).as_strided((n, m), (ld, 1))


LAYOUTS = [("row-major", lambda: (rows(64, 64), rows(64, 64))),
           ("w.t()", lambda: (rows(64, 64), rows(64, 64).t())),
           ("x.t()", lambda: (rows(64, 64).t(), rows(64, 64))),
           ("odd rows of x", lambda: (rows(64, 64, 65), rows(64, 64))),
           ("odd rows of w", lambda: (rows(64, 64), rows(64, 64, 67))),
           ("no unit stride", lambda: (rows(64, 128)[:, ::2], rows(64, 64)))]


def test_every_layout_of_a_shape_is_tuned(tuner):
    for i, (name, make) in enumerate(LAYOUTS):
        for _ in range(2):       # the second call finds the first's entry
            W.matmul(*make())
            assert len(tuner.timings) == i + 1, name
    for name, make in LAYOUTS:   # and so does every later one
        W.matmul(*make())
    assert len(tuner.timings) == len(LAYOUTS)
    assert all(key[:3] == (64, 64, 64) for key in tuner.timings)


def test_warm_call_takes_its_own_layouts_config(tuner):
    small, wide = (newt.Config({"BLOCK_M": 16, "BLOCK_N": n, "BLOCK_K": 32}) for n in (16, 32))
    nn, nt = LAYOUTS[0][1](), LAYOUTS[1][1]()
    for ops, cfg in ((nn, wide), (nt, small)):
        tuner.configs = [cfg]
        W.matmul(*ops)
    for ops, cfg in ((nn, wide), (nt, small), (nn, wide)):
        W.matmul(*ops)
        assert tuner.jitfn.calls[-1][1] == cfg.all_kwargs()


def test_row_strides_of_one_class_share_an_entry(tuner):
    W.matmul(rows(64, 64, 72), rows(64, 64))
    W.matmul(rows(64, 64, 80), rows(64, 64, 128))
    assert len(tuner.timings) == 1


def test_function_in_the_key_of_a_keyword_call(monkeypatch):
    monkeypatch.setattr(testing, "do_bench", lambda fn, warmup, rep: 1.0)
    rec = _Recorder()
    rec.param_names = ["x", "n", "scale"]
    rec.defaults = {"scale": 2.0}
    t = Autotuner(rec, [newt.Config({"BLOCK": 1})], key=["n", lambda scale: scale > 1])
    t[(1,)](0, 1)
    t[(1,)](0, 1, 3.0)
    t[(1,)](0, n=1, scale=3.0)
    assert list(t.timings) == [(1, True)]
    t[(1,)](0, 1, 0.5)
    assert len(t.timings) == 2
