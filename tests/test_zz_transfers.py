"""Programs whose edges are layout copies: the transfers by kernels and the
sliced runs (PDEFA_IO_SLICES) give the bits of the same program run without
either (PDEFA_HIP_GRAPH=0: upload, every step, download).  The products here
grow ops_matmul's scratch, so this file runs after test_zz_no_alloc, which
watches it grow."""
import os
import re

import numpy as np
import pytest

from pdefa_amd import native, yolo_synth as ys

pytestmark = pytest.mark.gpu


def _block(kind, c, h, w, batch):
    if kind == "scdown":
        return ys.build_scdown(c, c, h, n=batch, seed=3)[0]
    b = ys.GraphBuilder()
    y = ys._Yolo(b, np.random.default_rng(3), 0.0)
    out = y.c2f(-1, c, c, 1, True, "block") if kind == "c2f" else y.sppf(-1, c, c, "block")
    return b.model([batch, c, h, w], [batch, c, h, w], [out])


def _run(path, xs, env, monkeypatch):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    try:
        eng = native.Engine(path)
        try:
            return [eng.run(x)[0].copy() for x in xs], eng.plan()
        finally:
            eng.close()
    finally:
        for k in env:
            monkeypatch.delenv(k)


def _check(model, shape, tmp_path, monkeypatch, slices, kind, most, direct):
    """kind: the slices of the plan, `most` of them at the most; direct: whether
    kernels move the unsliced program's input and output on host memory."""
    path = os.path.join(tmp_path, "m.engine")
    ys.save(model, path)
    rng = np.random.default_rng(5)
    xs = [rng.standard_normal(shape, dtype=np.float32) for _ in range(2)]
    want, plan = _run(path, xs, {"PDEFA_HIP_GRAPH": "0"}, monkeypatch)
    assert not np.array_equal(want[0], want[1])
    assert " last_run=0" in plan
    for s in slices:
        print(f"[case] {shape} slices {s}", flush=True)
        got, plan = _run(path, xs + xs[:1], {"PDEFA_IO_SLICES": str(s)} if s else {}, monkeypatch)
        if kind == "rows" and not re.search(r"conv_mfma\(\S*,splits=1,", plan):
            kind = "none"  # the launch shape timed for it splits K
        assert f"transfers pull=1 push=1 slices={kind}\n" in plan
        ran, pull, push, last = map(int, re.search(
            r"io slices=(\d+) pull_direct=(\d) push_direct=(\d) last_run=(\d+)", plan).groups())
        # slices of rows take page-locked inputs
        assert last == (ran if ran == 1 or kind == "batch" or xs[0].nbytes >= 256 * 1024 else 0)
        if s:
            assert ran == (1 if kind == "none" else max(1, min(s, most)))
        assert (pull, push) == (int(direct and ran == 1),) * 2
        for g, w in zip(got, want + want[:1]):
            np.testing.assert_array_equal(g, w)


# Output rows that do not divide by the slice count, odd widths (4-byte
# accesses), one and two channels past a 64-wide tile, strides and kernel
# sizes whose slices share input rows, tensors below and above the size from
# which host tensors are page-locked.
@pytest.mark.parametrize("cin,cout,k,s,hw", [
    (64, 64, 3, 1, 40), (32, 66, 3, 1, 37), (16, 24, 3, 2, 65), (96, 144, 3, 2, 33), (64, 65, 1, 1, 50),
    (128, 64, 1, 1, 31), (16, 16, 3, 1, 16), (24, 40, 3, 2, 18), (32, 66, 3, 1, 61), (64, 30, 3, 2, 43),
])
def test_single_conv_transfers(cin, cout, k, s, hw, tmp_path, monkeypatch):
    model = ys.build_single_conv(cin, cout, k, s, hw, seed=3)[0]
    _check(model, (1, cin, hw, hw), tmp_path, monkeypatch, [0, 1, 2, 3, 8], "rows", ((hw - 1) // s + 1) // 8, True)


@pytest.mark.parametrize("kind,c,h,w,batch", [
    ("c2f", 64, 20, 24, 5), ("c2f", 96, 13, 11, 2), ("c2f", 96, 37, 31, 3), ("sppf", 64, 21, 20, 3), ("scdown", 64, 22, 22, 4),
])
def test_block_transfers(kind, c, h, w, batch, tmp_path, monkeypatch):
    _check(_block(kind, c, h, w, batch), (batch, c, h, w), tmp_path, monkeypatch, [0, 1, 2, 3, 8], "batch", batch, True)


@pytest.mark.parametrize("name,pinned", [("pageable", False), ("page-locked", True)])
def test_row_slices_need_page_locked_inputs(name, pinned, tmp_path):
    """A pageable input (under the size from which tensors are page-locked
    here) goes up whole, whatever the slices asked for."""
    model = ys.build_single_conv(16, 64, 3, 1, 80 if pinned else 60, seed=3)[0]
    hw = 80 if pinned else 60
    assert (16 * hw * hw * 4 >= 256 * 1024) == pinned
    path = os.path.join(tmp_path, "m.engine")
    ys.save(model, path)
    x = np.random.default_rng(5).standard_normal((1, 16, hw, hw), dtype=np.float32)
    want = _run(path, [x], {"PDEFA_HIP_GRAPH": "0"}, pytest.MonkeyPatch())[0]
    got, plan = _run(path, [x], {"PDEFA_IO_SLICES": "3"}, pytest.MonkeyPatch())
    print(f"[case] {name}", flush=True)
    assert "io slices=3 " in plan and f" last_run={3 if pinned else 0}\n" in plan
    np.testing.assert_array_equal(got[0], want[0])


# Row counts around the slice rule's smallest slice, a remainder row per slice,
# K % 4 != 0 (4-byte operand loads), products below and above the sizes from
# which operands are page-locked (each of A, B and C alone too) and sliced, and
# C in A's memory (never sliced).
@pytest.mark.parametrize("m,k,n", [(1, 5, 7), (300, 260, 300), (512, 512, 512), (2049, 1023, 1030), (3001, 2047, 601),
                                   (371, 201, 55), (32, 1251, 211), (300, 100, 300), (64, 300, 2000), (1659, 69, 518)])
def test_matmul_transfers(m, k, n):
    from pdefa_amd import pdefa as api

    print(f"[case] matmul {m}x{k}x{n}", flush=True)
    rng = np.random.default_rng(7)
    for _ in range(2):
        a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
        ta, tb = (api.Tensor(native.tensor_from_numpy(v)) for v in (a, b))
        out = api.empty(m, n)
        api.ops_matmul(ta, tb, out)
        want = a.astype(np.float64) @ b.astype(np.float64)
        # k products of unit variance, each partial sum rounded to 2^-24 of
        # itself: an error of about sqrt(k) * sqrt(k) * 2^-24 at the most
        np.testing.assert_allclose(out.numpy(), want, rtol=0, atol=k * 2.0**-24 * 4 + 1e-6)


@pytest.mark.parametrize("m,k,n", [(258, 260, 300), (513, 512, 512), (2049, 1023, 1030)])
def test_matmul_slices(m, k, n, monkeypatch):
    """Every number of row slices (operands that are page-locked, in memory of
    their own: the count asked for is the one that runs) gives the whole
    product's bits."""
    print(f"[case] matmul slices {m}x{k}x{n}", flush=True)
    assert min(m * k, k * n, m * n) * 4 >= 256 * 1024  # page-locked
    rng = np.random.default_rng(7)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    outs = []
    for slices in (1, 2, 3, 4):
        monkeypatch.setenv("PDEFA_IO_SLICES", str(slices))
        outs.append(native.matmul(a, b))
    for out in outs[1:]:
        np.testing.assert_array_equal(out, outs[0])


def test_matmul_of_many_rows():
    """2^24 rows and more in one piece (B is too small to be page-locked, so
    the product is never sliced)."""
    m, k, n = (1 << 24) + 5, 4, 4
    print(f"[case] matmul {m}x{k}x{n}", flush=True)
    rng = np.random.default_rng(9)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    got = native.matmul(a, b)
    for rows in (slice(0, 1000), slice(m - 1000, m)):
        np.testing.assert_allclose(got[rows], a[rows].astype(np.float64) @ b.astype(np.float64), rtol=0, atol=k * 2.0**-24 * 16)


def test_matmul_into_its_own_operand():
    from pdefa_amd import pdefa as api

    print("[case] matmul 1024 into A", flush=True)
    rng = np.random.default_rng(8)
    a, b = (rng.standard_normal((1024, 1024), dtype=np.float32) for _ in range(2))
    ta, tb = (api.Tensor(native.tensor_from_numpy(v)) for v in (a, b))
    apart = api.empty(1024, 1024)
    api.ops_matmul(ta, tb, apart)
    api.ops_matmul(ta, tb, ta)
    np.testing.assert_allclose(ta.numpy(), apart.numpy(), rtol=0, atol=1024 * 2.0**-24 * 4)
    np.testing.assert_array_equal(tb.numpy(), b)


def test_images_twice_before_a_run_and_one_after(tmp_path, monkeypatch):
    """Images go up while set_images copies them: a second set_images before
    the run replaces the first one's, a larger one grows the staging, and a
    run after them reads the last."""
    from pdefa_amd import pdefa as api

    print("[case] images staged twice", flush=True)
    path = os.path.join(tmp_path, "n.engine")
    ys.save(ys.build_yolov8("n", seed=0, imgsz=(96, 160)), path)
    rng = np.random.default_rng(6)
    small = [rng.integers(0, 256, (90, 150, 3), dtype=np.uint8) for _ in range(4)]
    large = [rng.integers(0, 256, (480, 333, 3), dtype=np.uint8) for _ in range(4)]

    def session():
        ctx = api.Context()
        return api.Session(ctx, api.Model(ctx, path))

    def stage(sess, images):
        sess.set_images(0, [api.Image.from_array(i) for i in images], 160, 96, 1.0 / 255.0, 114.0 / 255.0)

    def out(sess):
        sess.run()
        return sess.output(0).numpy().copy()

    want = []
    for images in (small, large):
        sess = session()
        stage(sess, images)
        want.append(out(sess))
    assert not np.array_equal(*want)
    sess = session()
    for images in (small, large):
        stage(sess, images)
    np.testing.assert_array_equal(out(sess), want[1])
    np.testing.assert_array_equal(out(sess), want[1])
    stage(sess, small)
    np.testing.assert_array_equal(out(sess), want[0])
    stage(sess, large)  # and no run
