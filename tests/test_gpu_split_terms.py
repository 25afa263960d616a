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

    # terms: the dropped products are at most 2^-24 of each product, and the
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


def _engine(model, path):
    ys.save(model, path)
    return path


@pytest.mark.parametrize("bits", [0x7F800001, 0x7F80FFFF, 0xFF800001, 0xFF80FFFF, 0x7FC00000, 0xFFFFFFFF, 0x7F800000,
                                  0xFF800000, 0x7F7FFFFF, 0xFF7F8000])
def test_split_tile_special_values(bits, tmp_path, monkeypatch):
    """NaNs of every payload, infinities and the largest finite values give
    the f32 tile's bits in the tile that they reach (here all of it)."""
    print(f"[case] split {bits:#x}", flush=True)
    path = _engine(ys.build_single_conv(64, 128, 1, 1, 8, seed=3, silu=False)[0], os.path.join(tmp_path, "c.engine"))
    x = np.random.default_rng(2).standard_normal((1, 64, 8, 8)).astype(np.float32)
    x.view(np.uint32)[0, 5, 3, 3] = bits
    got, f32 = (_run(path, x, t, monkeypatch) for t in ("split128x128w8", "128x128w8"))
    np.testing.assert_array_equal(np.isnan(got), np.isnan(f32))
    np.testing.assert_array_equal(got[~np.isnan(got)], f32[~np.isnan(f32)])
    if bits & 0x7FFFFFFF > 0x7F800000:
        assert np.isnan(got[0, :, 3, 3]).all()


@pytest.mark.parametrize("scale", [1e-27, 1e-30, 1e-33, 1e-36, 1e-39])
@pytest.mark.parametrize("rows", ["all", "one"])
def test_split_tile_tiny_rows(scale, rows, tmp_path, monkeypatch):
    """An input whose values are all tiny (or those of one pixel), where the
    terms run out of exponents, is no further off than with the f32 tile."""
    print(f"[case] split tiny {scale} {rows}", flush=True)
    model = ys.build_single_conv(256, 128, 1, 1, 16, seed=3, silu=False)[0]
    model.weights[1][:] = 0  # no bias: the products alone
    path = _engine(model, os.path.join(tmp_path, "c.engine"))
    x = np.random.default_rng(1).standard_normal((1, 256, 16, 16)).astype(np.float32)
    part = (0, slice(None), 9, 3) if rows == "one" else (0,)
    x[part] *= np.float32(scale)
    want = np.einsum("oi,ihw->ohw", model.weights[0][:, :, 0, 0].astype(np.float64), x[0].astype(np.float64))
    got, f32 = (_run(path, x, t, monkeypatch)[0].astype(np.float64) for t in ("split128x128w8", "128x128w8"))

    def err(y):
        d, r = (y - want)[part[1:]], want[part[1:]]
        return np.linalg.norm(d / scale) / np.linalg.norm(r / scale)

    assert err(got) <= err(f32)


@pytest.mark.parametrize("splits", [2, 3])
def test_split_tile_in_k_parts(splits, tmp_path, monkeypatch):
    """PDEFA_CONV_SPLITS with the split tile: the K parts' sums."""
    print(f"[case] split {splits} parts", flush=True)
    path = _engine(ys.build_single_conv(200, 140, 3, 2, 33, seed=3)[0], os.path.join(tmp_path, "c.engine"))
    x = np.random.default_rng(2).standard_normal((2, 200, 33, 33)).astype(np.float32)
    whole = _run(path, x, "split128x128w8", monkeypatch)
    x[1, 3, 4, 4] = np.nan  # one part of one tile goes to the f32 kernel
    monkeypatch.setenv("PDEFA_CONV_SPLITS", str(splits))
    got = _run(path, x, "split128x128w8", monkeypatch)
    # K = 1800 products of magnitude about 0.1, rounded to 2^-24 of the sum
    # some K / 16 times in either order
    np.testing.assert_allclose(got[0], whole[0], rtol=2e-5, atol=2e-5)
    assert np.isnan(got[1]).any() and np.isfinite(got[1]).any()


def test_split_rule_weights(tmp_path, monkeypatch):
    """An output channel of tiny weights, or a huge one, keeps the layer on
    the f32 tiles; channels of zeros and a tiny weight beside others do not."""
    print("[case] split rule weights", flush=True)
    x = np.random.default_rng(4).standard_normal((1, 768, 96, 96)).astype(np.float32)
    path = os.path.join(tmp_path, "c.engine")

    def split(change):
        model = ys.build_single_conv(768, 256, 1, 1, 96, seed=3)[0]
        change(model.weights[0])
        eng = native.Engine(_engine(model, path))
        try:
            eng.run(x)
            return "tile=split128x128w8" in eng.plan()
        finally:
            eng.close()

    def set_to(at, value):
        def change(w):
            w[at] = value
        return change

    assert split(set_to(7, 0.0))
    assert split(set_to((7, 5), 1e-40))
    assert not split(set_to(7, 1e-30))
    assert not split(set_to((7, 5), 3e38))
    assert not split(set_to((7, 5), np.nan))


@pytest.mark.parametrize("x_bits", [0x3F80FFFF, 0x3F80FF7F, 0x3F808080, 0x3F80807F, 0x3FFFFFFF, None])
def test_split_tile_single_products(x_bits, tmp_path, monkeypatch):
    """Pixels of one channel, so that every output is one product, with the
    significands whose terms leave the most out (truncated terms: 2^-21 of the
    product, always towards zero)."""
    print(f"[case] split single {x_bits}", flush=True)
    model = ys.build_single_conv(256, 256, 1, 1, 16, seed=3, silu=False)[0]
    w = model.weights[0]
    model.weights[1][:] = 0
    rng = np.random.default_rng(1)
    x = np.zeros((1, 256, 16, 16), np.float32)
    if x_bits is None:
        x[0, np.arange(256), np.arange(256) // 16, np.arange(256) % 16] = rng.standard_normal(256)
    else:
        v = np.uint32(x_bits).view(np.float32)
        x[0, np.arange(256), np.arange(256) // 16, np.arange(256) % 16] = v
        w[:] = np.where(rng.random(w.shape) < 0.5, v, -v)
        w[::2] *= (rng.integers(1 << 23, 1 << 24, w[::2].shape) / (1 << 23)).astype(np.float32)
    path = _engine(model, os.path.join(tmp_path, "c.engine"))
    want = np.einsum("oi,ihw->ohw", w[:, :, 0, 0].astype(np.float64), x[0].astype(np.float64))
    got = _run(path, x, "split128x128w8", monkeypatch)[0].astype(np.float64)
    rel = (got - want) / np.abs(want)
    # two dropped products of 2^-25 each, the sum's last rounding, and the
    # low sum's (six of 2^-24 of 2^-7)
    assert np.abs(rel).max() <= 2.0**-24 * (1 + 1 + 6 / 128)
    # centred: over random significands the mean error is far below the largest
    if x_bits is None:
        assert abs((rel * np.sign(want)).mean()) <= 2.0**-29


def test_split_tile_compat_silu(tmp_path, monkeypatch):
    """A 3x3 stride-1 layer (the SiLU form with the float64 second pass) on
    the split tile: an infinity and a pixel of tiny values in one tile each
    give the f32 tile's bits there, other tiles the split sums."""
    print("[case] split compat SiLU", flush=True)
    path = _engine(ys.build_single_conv(64, 128, 3, 1, 24, seed=3)[0], os.path.join(tmp_path, "c.engine"))
    x = np.random.default_rng(2).standard_normal((1, 64, 24, 24)).astype(np.float32)
    plain = [_run(path, x, t, monkeypatch) for t in ("split128x128w8", "128x128w8")]
    # a SiLU jump of 2% lies between the two sums at a few outputs at most
    off = np.abs(plain[0] - plain[1]) > 1e-4 * (1 + np.abs(plain[1]))
    assert off.sum() <= 3
    x[0, 5, 1, 1] = np.inf
    got, f32 = (_run(path, x, t, monkeypatch) for t in ("split128x128w8", "128x128w8"))
    # the first tile: output rows 0 to 4 and 8 pixels of row 5
    np.testing.assert_array_equal(got[:, :, :5], f32[:, :, :5])
    assert not np.array_equal(got[:, :, 6:], f32[:, :, 6:])


def test_split_tile_upsampled_copy(tmp_path, monkeypatch):
    """A layer that the rule takes and whose epilogue writes an upsampled copy,
    with a NaN in one tile."""
    print("[case] split upsampled copy", flush=True)
    b = ys.GraphBuilder()
    y = ys._Yolo(b, np.random.default_rng(3), 0.0)
    out = y.conv(y.upsample(y.conv(-1, 768, 128, 1, 1, "c"), "u"), 128, 16, 1, 1, "d")
    path = _engine(b.model([1, 768, 128, 128], [1, 16, 256, 256], [out]), os.path.join(tmp_path, "c.engine"))
    x = np.random.default_rng(2).standard_normal((1, 768, 128, 128)).astype(np.float32)
    x[0, 700, 3, 77] = np.nan
    outs = []
    for terms in ("1", "0"):
        monkeypatch.setenv("PDEFA_SPLIT_TERMS", terms)
        eng = native.Engine(path)
        try:
            outs.append(eng.run(x)[0].copy())
            conv = next(l for l in eng.plan().splitlines() if " conv_mfma(" in l)
        finally:
            eng.close()
        assert ("tile=split128x128w8" in conv) == (terms == "1") and " up=b" in conv
    got, f32 = outs
    nan = np.zeros((256, 256), bool)
    nan[6:8, 154:156] = True
    np.testing.assert_array_equal(np.isnan(got[0]), np.broadcast_to(nan, got[0].shape))
    np.testing.assert_array_equal(np.isnan(f32), np.isnan(got))
    # 768 and 128 products of about unit size, in sums of either order, each
    # addition rounded to 2^-24 of a few units
    np.testing.assert_allclose(got[~np.isnan(got)], f32[~np.isnan(f32)], rtol=1e-5, atol=(768 + 128) * 2.0**-24)
