"""Which programs run their edges as transfers and in slices (the planner's
io_shape, printed with the plan): on the host by the plan text, and on the GPU
by their outputs against the same program run without either."""
import os
import random
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


def _one_conv(cin, cout, k, s, hw, groups=1):
    return ys.build_single_conv(cin, cout, k, s, hw, seed=3, groups=groups)[0], (1, cin, hw, hw)


def _batch(build, n, c, h, w, out_shape):
    return _graph(build, (n, c, h, w), out_shape), (n, c, h, w)


def _transpose(b, x, perm):
    return b.node("Transpose", "/t", [x, b.const("/t::perm", np.array(perm, np.float32))])


def _pool(b, x):
    return b.node("MaxPool", "/p", [x], kernel_h=3, kernel_w=3, stride_h=1, stride_w=1, pad_h=1, pad_w=1)


def _block(kind, c, h, w, n):
    def build(b, y):
        if kind == "c2f":
            return y.c2f(-1, c, c, 1, True, "block")
        if kind == "sppf":
            return y.sppf(-1, c, c, "block")
        return y.conv(_pool(b, y.conv(-1, c, c, 1, 1, "a")), c, c, 3, 1, "b")

    return _batch(build, n, c, h, w, (n, c, h, w))


def _transposed(n, cin, mid, h, w, perm, cout, k, pool=False):
    """A conv to `mid` channels, a Transpose, optionally a pool, a conv."""
    dims = [(n, mid, h, w)[i] for i in perm]

    def build(b, y):
        t = _transpose(b, y.conv(-1, cin, mid, 1, 1, "a"), perm)
        return y.conv(_pool(b, t) if pool else t, dims[1], cout, k, 1, "b")

    return _batch(build, n, cin, h, w, (dims[0], cout, dims[2], dims[3]))


def _half_images(n, c, h, w, first):
    """N of the 2N half images that a Reshape makes of N images."""
    def build(b, y):
        half = b.node("Reshape", "/r", [y.conv(-1, c, c, 1, 1, "a"), b.const("/r::shape", [2 * n, c // 2, h, w])])
        return y.conv(y.slice(half, first, first + n, 0, "/s"), c // 2, 16, 3, 1, "b")

    return _batch(build, n, c, h, w, (n, 16, h, w))


def _view_concat(n, c, h, w, view):
    """The input, sliced or reshaped, beside a constant in a concat's
    channels-last buffer, and a conv of both."""
    dims = {"image 0": (1, c, h, w), "halves": (2 * n, c // 2, h, w), "whole": (n, c, h, w)}[view]

    def build(b, y):
        x = -1
        if view == "image 0":
            x = y.slice(-1, 0, 1, 0, "/s")
        elif view == "halves":
            x = b.node("Reshape", "/r", [-1, b.const("/r::shape", list(dims))])
        const = np.random.default_rng(4).standard_normal((dims[0], 16, h, w)).astype(np.float32)
        cat = b.node("Concat", "/c", [x, b.const("/c::const", const)], axis=1)
        return y.conv(cat, dims[1] + 16, 24, 3, 1, "a")

    return _batch(build, n, c, h, w, (dims[0], 24, h, w))


# name: (model and input shape, slices)
CASES = {
    "conv": (lambda: _one_conv(64, 64, 3, 1, 48), "rows"),
    "conv 1x1": (lambda: _one_conv(32, 24, 1, 1, 40), "rows"),
    "conv 5x5": (lambda: _one_conv(32, 40, 5, 1, 57), "rows"),
    "conv 5x5 s2": (lambda: _one_conv(32, 40, 5, 2, 57), "rows"),
    "conv in groups": (lambda: _one_conv(64, 64, 3, 1, 47, groups=4), "rows"),
    "depthwise conv": (lambda: _one_conv(64, 64, 3, 1, 47, groups=64), "none"),
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
    # batches, whose every step keeps the images apart
    "c2f batch": (lambda: _block("c2f", 64, 20, 24, 4), "batch"),
    "sppf batch": (lambda: _block("sppf", 64, 12, 20, 3), "batch"),
    "pool batch": (lambda: _block("pool", 32, 12, 20, 32), "batch"),
    # an outer dimension of the batch's size that is channels or rows
    "channels as images": (lambda: _transposed(16, 32, 16, 20, 20, (1, 0, 2, 3), 24, 3), "none"),
    "channels as images, pool": (lambda: _transposed(16, 32, 16, 20, 20, (1, 0, 2, 3), 24, 3, True), "none"),
    "channels as images, 1x1": (lambda: _transposed(16, 32, 16, 20, 20, (1, 0, 2, 3), 24, 1), "none"),
    "rows as images": (lambda: _transposed(20, 32, 48, 20, 16, (2, 1, 0, 3), 24, 3), "none"),
    "rows and columns swapped": (lambda: _transposed(4, 32, 48, 12, 20, (0, 1, 3, 2), 24, 3), "batch"),
    # parts of images
    "first half images": (lambda: _half_images(4, 32, 12, 12, 0), "none"),
    "last half images": (lambda: _half_images(4, 32, 12, 12, 4), "none"),
    # the first copy reads a part of the input, or it in another shape
    "image 0 of 2": (lambda: _view_concat(2, 16, 20, 20, "image 0"), "none"),
    "halves of an image": (lambda: _view_concat(1, 32, 20, 20, "halves"), "none"),
    "halves of images": (lambda: _view_concat(2, 32, 20, 20, "halves"), "none"),
    "input beside a constant": (lambda: _view_concat(1, 16, 20, 20, "whole"), "none"),
    "inputs beside a constant": (lambda: _view_concat(2, 16, 20, 20, "whole"), "none"),
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


@pytest.mark.parametrize("name,pull", [
    ("conv", 1), ("image 0 of 2", 0), ("halves of an image", 0), ("halves of images", 0), ("input beside a constant", 1),
    ("inputs beside a constant", 1), ("rows 4..48 conv", 0), ("conv rows 4..48", 1),
])
def test_pull(name, pull, tmp_path):
    """The upload takes the first layout copy's place only where that copy
    reads the whole input in its own shape."""
    model, shape = CASES[name][0]()
    path = os.path.join(tmp_path, "m.engine")
    ys.save(model, path)
    assert transfers(native.plan_text(path, list(shape)))[0] == pull


# steps that run on chunks of the batch as the input arrives (of CASES' steps:
# the layout copy, the convs and pools, the layout copy)
@pytest.mark.parametrize("name,early", [
    ("c2f batch", 6), ("channels as images", 2), ("channels as images, 1x1", 2), ("rows as images", 2),
    ("rows and columns swapped", 4), ("first half images", 3), ("last half images", 3),
])
def test_early_steps(name, early, tmp_path, monkeypatch):
    monkeypatch.setenv("PDEFA_EARLY_HW", "1")
    model, shape = CASES[name][0]()
    path = os.path.join(tmp_path, "m.engine")
    ys.save(model, path)
    assert int(re.search(r"early_steps=(\d+)", native.plan_text(path, list(shape))).group(1)) == early


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
    envs = [{}] + [{"PDEFA_IO_SLICES": str(n)} for n in (1, 2, 3)]
    if shape[0] % 2 == 0:
        envs.append({"PDEFA_EARLY_HW": "1"})  # chunks of the batch
    for env in envs:
        print(f"[case] {name} {env}", flush=True)
        for g, w in zip(_run(path, xs + xs[:1], env, monkeypatch), want + want[:1]):
            np.testing.assert_array_equal(g, w)


# ---- the rules against what the steps do: random graphs, sliced on paper

_VIEW = re.compile(r" (out|a|b|c|res|up)=b(-?\d+)\+(\d+)\[([\d,]*)\]s\[([-\d,]*)\]")


def _views(line):
    """(views read, views written) of a plan's step line: (buffer, offset, dims, strides)."""
    writes = ("out", "b", "c") if " maxpool_chain " in line else ("out", "up")
    rd, wr = [], []
    for key, buf, off, dims, strides in _VIEW.findall(line):
        v = (int(buf), int(off), [int(d) for d in dims.split(",")], [int(s) for s in strides.split(",")])
        if v[0] >= 0:  # not a constant
            (wr if key in writes else rd).append(v)
    return rd, wr


def _item(v, i):
    """Elements of item i of a view's outer dimension."""
    _, off, dims, strides = v
    e = np.array([off + i * strides[0]])
    for d, s in zip(dims[1:], strides[1:]):
        e = (e[:, None] + np.arange(d) * s).reshape(-1)
    return e


def _run_sliced(steps, n, slices, inputs, elems):
    """Runs steps slice by slice on tags: which image's data an element holds."""
    mem = {inputs: np.full(elems, -1)}

    def tags(v, e):
        if v[0] not in mem or len(mem[v[0]]) <= e.max():
            mem[v[0]] = np.concatenate([mem.get(v[0], np.empty(0, int)), np.full(int(e.max()) + 1, -1)])
        return mem[v[0]]

    for lo, hi in slices:
        mem[inputs][lo * elems // n:hi * elems // n] = np.repeat(np.arange(lo, hi), elems // n)
        for line in steps:
            rd, wr = _views(line)
            for i in range(lo, hi):
                for v in rd:
                    e = _item(v, i)
                    assert (tags(v, e)[e] == i).all(), (line, i)
            for i in range(lo, hi):
                for v in wr:
                    e = _item(v, i)
                    tags(v, e)[e] = i


def _random_graph(rng):
    """A chain of convs, pools, views, concats and upsamples whose dimensions
    often have the batch's size."""
    n = rng.choice([2, 2, 4])
    d = shape = [n, rng.choice([n, 4, 8, 16]), rng.choice([n, 4, 6]), rng.choice([n, 4, 5])]
    b = ys.GraphBuilder()
    y = ys._Yolo(b, np.random.default_rng(1), 0.0)
    x, old = -1, []
    for i, op in enumerate(["conv"] * (rng.random() < 0.7) + rng.choices(
            ["conv", "conv s2", "pool", "slice", "reshape", "transpose", "concat", "resize"], k=rng.randint(1, 4))):
        d = list(d)
        if op.startswith("conv"):
            c, s = rng.choice([8, 16, 8 * n]), 2 if op == "conv s2" else 1
            x = y.conv(x, d[1], c, rng.choice([1, 3]) if s == 1 else 3, s, f"c{i}")
            d = [d[0], c, (d[2] - 1) // s + 1, (d[3] - 1) // s + 1]
        elif op == "pool":
            x = b.node("MaxPool", f"/p{i}", [x], kernel_h=3, kernel_w=3, stride_h=1, stride_w=1, pad_h=1, pad_w=1)
        elif op == "slice":
            ax = rng.randrange(4)
            size = n if d[ax] > n and rng.random() < 0.5 else rng.randint(1, d[ax])
            lo = rng.randint(0, d[ax] - size)
            x, d[ax] = y.slice(x, lo, lo + size, ax, f"/s{i}"), size
        elif op == "reshape":
            p, q = rng.sample(range(4), 2)
            if d[p] % 2 == 0:
                d[p], d[q] = d[p] // 2, d[q] * 2
                x = b.node("Reshape", f"/r{i}", [x, b.const(f"/r{i}::shape", d)])
        elif op == "transpose":
            perm = rng.sample(range(4), 4)
            x, d = b.node("Transpose", f"/t{i}", [x, b.const(f"/t{i}::perm", np.array(perm, np.float32))]), [d[p] for p in perm]
        elif op == "concat":
            other = [o for o in old if o[1][0] == d[0] and o[1][2:] == d[2:]]
            k, c = rng.choice(other) if other else (b.const(f"/k{i}", np.ones((d[0], 4, d[2], d[3]))), [0, 4])
            x, d[1] = b.node("Concat", f"/cat{i}", [x, k], axis=1), d[1] + c[1]
        else:
            x, d = y.upsample(x, f"u{i}"), [d[0], d[1], 2 * d[2], 2 * d[3]]
        old.append((x, d))
    return b.model(shape, d, [x]), shape


def test_random_graphs(tmp_path, monkeypatch):
    """Every step of a program that runs in slices of the batch, or early on
    chunks of it, reads only what its own slice has written."""
    monkeypatch.setenv("PDEFA_EARLY_HW", "1")
    path = os.path.join(tmp_path, "m.engine")
    batch = early = 0
    for seed in range(600):
        model, shape = _random_graph(random.Random(seed))
        if not model.nodes:
            continue
        ys.save(model, path)
        try:
            text = native.plan_text(path, shape)
        except native.NativeError:
            continue  # a form that the device program does not take
        steps = text.split("\narena")[0].splitlines()[1:]
        if not steps:
            continue
        n, elems = shape[0], int(np.prod(shape))
        written = {v[0] for line in steps for v in _views(line)[1]}
        inputs = {v[0] for line in steps for v in _views(line)[0]} - written
        if len(inputs) != 1:
            continue
        inputs = inputs.pop()
        if transfers(text)[2] == "batch":
            batch += 1
            for s in {2, n}:
                _run_sliced(steps, n, [(n * i // s, n * (i + 1) // s) for i in range(s)], inputs, elems)
        e = int(re.search(r"early_steps=(\d+)", text).group(1))
        if e:
            early += 1
            _run_sliced(steps[:e], n, [(0, n // 2), (n // 2, n)], inputs, elems)
    assert batch > 60 and early > 200
