"""The split implicit-GEMM tile (f32 operands as three bf16 terms) against
the float64 oracle and the f32 tile of the same shape."""
import os

import numpy as np
import pytest

from oracle import graph_ref
from pdefa_amd import native, yolo_synth as ys

pytestmark = pytest.mark.gpu


def _run(path, x, tile, monkeypatch):
    monkeypatch.setenv("PDEFA_CONV_TILE", tile)
    try:
        eng = native.Engine(path)
        try:
            y = eng.run(x)[0].copy()
            assert f"tile={tile}" in eng.plan()
            return y
        finally:
            eng.close()
    finally:
        monkeypatch.delenv("PDEFA_CONV_TILE")


# Remainders of the 128 x 128 tile in both directions, one row or channel
# past it, less than one tile, K that is no multiple of 32 or 16, padding,
# strides, a 1x1 layer and one with a single K step.
@pytest.mark.parametrize("cin,cout,k,s,hw", [
    (64, 128, 3, 2, 32), (36, 130, 3, 2, 45), (128, 384, 1, 1, 23), (32, 129, 1, 1, 8), (20, 40, 1, 1, 5),
    (200, 257, 3, 2, 19),
])
@pytest.mark.parametrize("scale", [1.0, 1e-12, 1e12])
def test_split_tile(cin, cout, k, s, hw, scale, tmp_path, monkeypatch):
    print(f"[case] split {cin}->{cout} k{k} s{s} {hw} x{scale}", flush=True)
    model = ys.build_single_conv(cin, cout, k, s, hw, seed=3)[0]
    path = os.path.join(tmp_path, "c.engine")
    ys.save(model, path)
    x = (np.random.default_rng(1).standard_normal((1, cin, hw, hw)) * scale).astype(np.float32)
    want = graph_ref.run_graph(model, [x])[0].astype(np.float64)
    got, f32 = (_run(path, x, t, monkeypatch).astype(np.float64) for t in ("split128x128w8", "128x128w8"))

    def err(y):
        return np.linalg.norm(y - want) / np.linalg.norm(want)

    # terms: the dropped products are below 2^-23 of each product, and the
    # K / 16 additions of the leading ones round by 2^-24 of the running sum
    K = cin * k * k
    assert err(got) <= 2.0**-23 + np.sqrt(K / 16 + 1) * 2.0**-24 * 2
    # and no further off than the f32 tile's K / 2 additions, where those
    # are enough to show
    if K >= 256:
        assert err(got) <= err(f32)


def test_split_tile_infinities(tmp_path, monkeypatch):
    """Infinite and NaN inputs reach the outputs that the f32 tile's reach,
    as the same infinities and NaNs, and no others."""
    print("[case] split infinities", flush=True)
    model = ys.build_single_conv(64, 128, 3, 2, 33, seed=3)[0]
    path = os.path.join(tmp_path, "c.engine")
    ys.save(model, path)
    x = np.random.default_rng(2).standard_normal((1, 64, 33, 33)).astype(np.float32)
    x[0, 3, 4, 4], x[0, 7, 20, 9], x[0, 60, 12, 28], x[0, 1, 30, 30] = np.inf, -np.inf, np.nan, 3e38
    got, f32 = (_run(path, x, t, monkeypatch) for t in ("split128x128w8", "128x128w8"))
    assert np.isinf(f32).any() and np.isnan(f32).any()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(f32))
    np.testing.assert_array_equal(np.where(np.isinf(got), got, 0), np.where(np.isinf(f32), f32, 0))
    fin = np.isfinite(f32)
    np.testing.assert_allclose(got[fin], f32[fin], rtol=1e-4, atol=1e-4)


def test_split_rule(tmp_path, monkeypatch):
    """Long wide layers take the split tile, without it when a weight is not
    finite or PDEFA_SPLIT_TERMS=0."""
    print("[case] split rule", flush=True)
    model = ys.build_single_conv(768, 256, 1, 1, 96, seed=3)[0]
    x = np.random.default_rng(4).standard_normal((1, 768, 96, 96)).astype(np.float32)
    path = os.path.join(tmp_path, "c.engine")

    def plan():
        ys.save(model, path)
        eng = native.Engine(path)
        try:
            eng.run(x)
            return eng.plan()
        finally:
            eng.close()

    assert "tile=split128x128w8" in plan()
    monkeypatch.setenv("PDEFA_SPLIT_TERMS", "0")
    assert "split128x128w8" not in plan()
    monkeypatch.delenv("PDEFA_SPLIT_TERMS")
    w = next(v for v in model.weights if v.size == 768 * 256)
    w.reshape(-1)[77] = np.inf
    assert "split128x128w8" not in plan()
