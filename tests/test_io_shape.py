"""Which programs run their edges as transfers and in slices (the planner's
io_shape, printed with the plan): on the host by the plan text, and on the GPU
by their outputs against the same program run without either."""
import os
import re

import numpy as np
import pytest

from pdefa_amd import native, yolo_synth as ys


def _graph(build, in_shape, out_shape):
    b = ys.GraphBuilder()
    y = ys._Yolo(b, np.random.default_rng(3), 0.0)
    return b.model(list(in_shape), list(out_shape), [build(b, y)])


def _conv_slice(cin, cout, k, hw, axis, lo, hi):
    def build(b, y):
        return y.slice(y.conv(-1, cin, cout, k, 1, "c"), lo, hi, axis, "/s")

    out = [1, cout, hw, hw]
    out[axis] = hi - lo
    return _graph(build, (1, cin, hw, hw), out), (1, cin, hw, hw)


def _slice_conv(cin, cout, hw, axis, lo, hi):
    shape = [1, cin, hw, hw]

    def build(b, y):
        return y.conv(y.slice(-1, lo, hi, axis, "/s"), hi - lo if axis == 1 else cin, cout, 3, 1, "c")

    out = list(shape)
    out[axis] = hi - lo
    out[1] = cout
    return _graph(build, shape, out), tuple(shape)


def _conv_conv(c, hw, rows):
    """Two convs, the second's rows cut off: never sliced by rows."""
    def build(b, y):
        h = y.conv(-1, c, c, 3, 1, "a")
        return y.slice(y.conv(h, c, c, 1, 1, "b"), 0, rows, 2, "/s")

    return _graph(build, (1, c, hw, hw), (1, c, rows, hw)), (1, c, hw, hw)


def _one_conv(cin, cout, k, s, hw):
    return ys.build_single_conv(cin, cout, k, s, hw, seed=3)[0], (1, cin, hw, hw)


# name: (model and input shape, slices)
CASES = {
    "conv": (lambda: _one_conv(64, 64, 3, 1, 48), "rows"),
    "conv 1x1": (lambda: _one_conv(32, 24, 1, 1, 40), "rows"),
    # the last copy reads a part of the conv's rows, columns or channels
    "conv rows 4..48": (lambda: _conv_slice(64, 64, 3, 48, 2, 4, 48), "none"),
    "conv rows 0..24": (lambda: _conv_slice(64, 64, 3, 48, 2, 0, 24), "none"),
    "conv cols 0..24": (lambda: _conv_slice(64, 64, 3, 48, 3, 0, 24), "none"),
    "conv channels 4..60": (lambda: _conv_slice(64, 64, 3, 48, 1, 4, 60), "none"),
    "1x1 conv rows 0..20": (lambda: _conv_slice(32, 24, 1, 40, 2, 0, 20), "none"),
    # the conv reads a part of the input
    "rows 4..48 conv": (lambda: _slice_conv(32, 24, 48, 2, 4, 48), "none"),
    "channels 8..32 conv": (lambda: _slice_conv(32, 24, 48, 1, 8, 32), "none"),
    "two convs rows 0..20": (lambda: _conv_conv(32, 40, 20), "none"),
}


def transfers(text):
    """(pull, push, slices) of a plan text."""
    line = next(l for l in text.splitlines() if l.startswith("transfers"))
    pull, push, slices = re.match(r"transfers pull=(\d) push=(\d) slices=(\w+)", line).groups()
    return int(pull), int(push), slices


@pytest.mark.parametrize("name", CASES)
def test_slices(name, tmp_path):
    (model, shape), slices = CASES[name][0](), CASES[name][1]
    path = os.path.join(tmp_path, "m.engine")
    ys.save(model, path)
    assert transfers(native.plan_text(path, list(shape)))[2] == slices


def _run(path, xs, env, monkeypatch):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    try:
        eng = native.Engine(path)
        try:
            return [eng.run(x)[0].copy() for x in xs]
        finally:
            eng.close()
    finally:
        for k in env:
            monkeypatch.delenv(k)


@pytest.mark.gpu
@pytest.mark.parametrize("name", CASES)
def test_outputs(name, tmp_path, monkeypatch):
    model, shape = CASES[name][0]()
    path = os.path.join(tmp_path, "m.engine")
    ys.save(model, path)
    rng = np.random.default_rng(5)
    xs = [rng.standard_normal(shape, dtype=np.float32) for _ in range(2)]
    want = _run(path, xs, {"PDEFA_HIP_GRAPH": "0"}, monkeypatch)
    for n in (0, 1, 2, 3):
        print(f"[case] {name} slices {n}", flush=True)
        got = _run(path, xs + xs[:1], {"PDEFA_IO_SLICES": str(n)} if n else {}, monkeypatch)
        for g, w in zip(got, want + want[:1]):
            np.testing.assert_array_equal(g, w)
