"""Matmuls too small to fill the GPU with their best-scored tile: the tiles and
splits ``select_filled`` picks, every tile size and number of parts forced, and
the unaligned 128-bit loaders, on the GPU against float64."""

from __future__ import annotations

import numpy as np
import pytest

from metellus_amd.api import compile_program, run, run_batch
from metellus_amd.compute.matmul import config
from metellus_amd.orchestrator import Operations
from metellus_amd.orchestrator.assembly import matmul as mm

pytestmark = pytest.mark.gpu


def _program(shape, a_view=False, b_view=False, seed=13, divisor=False):
    M, K, N = shape
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((M, K)).astype(np.float32)
    b = rng.standard_normal((K, N)).astype(np.float32)
    bias = rng.standard_normal((1, N)).astype(np.float32)
    ops = Operations()
    ops.from_numpy(np.ascontiguousarray(a.T) if a_view else a, "A")
    ops.from_numpy(np.ascontiguousarray(b.T) if b_view else b, "B")
    ops.from_numpy(bias, "bias")
    left, right, ref_a = "A", "B", a.astype(np.float64)
    if a_view:
        ops.transpose("A", out="At")
        left = "At"
    if b_view:
        ops.transpose("B", out="Bt")
        right = "Bt"
    if divisor:
        s = (rng.random((M, 1)) + 1.0).astype(np.float32)
        ops.from_numpy(s, "s")
        ops.elementwise("div", out="P", operands=(left, "s"), y_broadcast="col")
        left, ref_a = "P", ref_a / s
    ops.matmul(a=left, b=right, out="C")
    ops.elementwise("add", out="Y", operands=("C", "bias"), y_broadcast="row")
    ref = ref_a @ b.astype(np.float64) + bias
    bound = (np.abs(ref_a) @ np.abs(b.astype(np.float64)) + np.abs(bias)) * (K + 8) * 2.0**-24
    return ops, ref, bound


def _check(ops, ref, bound, repeats=2):
    got = run(ops).env["Y"]
    assert np.all(np.abs(got - ref) <= bound)
    for _ in range(repeats - 1):  # the counters are left at zero; parts add in order
        assert np.array_equal(run(ops).env["Y"], got)


@pytest.mark.parametrize("views", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("shape", [(256, 256, 256), (129, 331, 195), (1000, 130, 77), (70, 2048, 1030)], ids=str)
def test_picked(shape, views):
    print(f"filled {shape} {views}", flush=True)
    ops, ref, bound = _program(shape, *views)
    _check(ops, ref, bound)


@pytest.mark.parametrize("parts", [1, 2, 3, 16])
@pytest.mark.parametrize("index", range(len(config.FILL_TILES)))
def test_every_tile_and_split(index, parts, monkeypatch):
    tile = config.FILL_TILES[index].tile
    monkeypatch.setattr(mm, "select_filled", lambda *a, **k: (tile, parts))
    monkeypatch.setattr(mm, "fills", lambda *a, **k: False)
    for shape in ((256, 1024, 512), (300, 1027, 259)):
        print(f"filled {shape} {tile.tile_M}x{tile.tile_N} parts={parts}", flush=True)
        ops, ref, bound = _program(shape)
        (g,) = compile_program(ops)
        assert g.grid[0] == -(-shape[2] // tile.tile_N) * parts and (g.kernel.workspace_bytes > 0) == (parts > 1)
        _check(ops, ref, bound)
        batched = g.kernel.batched()  # without a workspace the first part walks the whole K
        assert batched.workspace_bytes == 0 and "mt_ws" not in batched.source.split('extern "C"')[-1]


def test_divisors_and_batches():
    for shape in ((200, 515, 131), (512, 512, 256)):
        print(f"filled divisor {shape}", flush=True)
        _check(*_program(shape, divisor=True))
    made = [_program((130, 300, 90), seed=30 + i) for i in range(3)]
    for (_, ref, bound), res in zip(made, run_batch([m[0] for m in made])):
        assert np.all(np.abs(res.env["Y"] - ref) <= bound)


@pytest.mark.parametrize("parts", [1, 2, 16])
def test_pair_sharing_a(parts, monkeypatch):
    """Two products of one A merged in a kernel split like the single ones: their
    sums come in the same order, so the values are the same bits."""
    monkeypatch.setattr(config, "filled_parts", lambda *a: parts)
    rng = np.random.default_rng(17)
    M, K, N = 130, 1040, 200
    x, w1, w2 = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (K, N), (K, N)))
    ops, one, two = Operations(), Operations(), Operations()
    for o, ws in ((ops, ("W1", "W2")), (one, ("W1",)), (two, ("W2",))):
        o.from_numpy(x, "X")
        for w in ws:
            o.from_numpy(w1 if w == "W1" else w2, w)
            o.matmul(a="X", b=w, out="h" + w)
    ops.elementwise("mul", out="z", operands=("hW1", "hW2"))
    config.select_filled.cache_clear()
    print(f"pair parts={parts}", flush=True)
    try:
        (g,) = compile_program(ops)
        assert g.kernel.function_name.startswith("multi_anchor") and (g.kernel.workspace_bytes > 0) == (parts > 1)
        z = run(ops).env["z"]
        h1, h2 = run(one).env["hW1"], run(two).env["hW2"]
        again = run(ops).env["z"]
    finally:
        config.select_filled.cache_clear()
    assert np.array_equal(z, h1 * h2) and np.array_equal(z, again)
    ref = (x.astype(np.float64) @ w1) * (x.astype(np.float64) @ w2)
    np.testing.assert_allclose(z, ref, rtol=1e-4, atol=1e-2)


def test_pair_of_few_rows():
    """Alone, a product of up to 64 rows takes the skinny kernel (fp32 MFMAs, k's in
    other groups); in a pair the tiles: both within an fp32 sum's rounding."""
    rng = np.random.default_rng(18)
    M, K, N = 48, 1040, 200
    x, w1, w2 = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (K, N), (K, N)))
    pair, one = Operations(), Operations()
    for o in (pair, one):
        o.from_numpy(x, "X")
        o.from_numpy(w1, "W1")
        o.matmul(a="X", b="W1", out="h1")
    pair.from_numpy(w2, "W2")
    pair.matmul(a="X", b="W2", out="h2")
    pair.elementwise("add", out="z", operands=("h1", "h2"))
    print("pair of few rows", flush=True)
    (g,), (s,) = compile_program(pair), compile_program(one)
    assert "mt_mfma_tile" in g.kernel.source.split('extern "C"')[-1]
    assert "mt_sn_mainloop<" in s.kernel.source.split('extern "C"')[-1]
    x64, a64 = x.astype(np.float64), np.abs(x.astype(np.float64))
    unit = (K + 8) * 2.0**-24
    assert np.all(np.abs(run(one).env["h1"] - x64 @ w1) <= unit * (a64 @ np.abs(w1)))
    assert np.all(np.abs(run(pair).env["z"] - x64 @ (w1.astype(np.float64) + w2)) <= unit * (a64 @ (np.abs(w1) + np.abs(w2))))


@pytest.mark.parametrize("a_view", [False, True])
@pytest.mark.parametrize("kind", ["recip", "none", "row", "col"])
def test_odd_prologues(kind, a_view):
    """Bounds inside a 128-bit slot: nothing outside the matrix is loaded for a
    prologue's operands or reaches the product (1 / 0 would)."""
    rng = np.random.default_rng(19)
    for M, K, N in ((201, 131, 77), (67, 258, 130), (130, 1030, 35)):
        print(f"odd prologue {kind} {(M, K, N)} a_view={a_view}", flush=True)
        a = (rng.random((M, K)) + 0.5).astype(np.float32)
        b = rng.standard_normal((K, N)).astype(np.float32)
        ops = Operations()
        ops.from_numpy(np.ascontiguousarray(a.T) if a_view else a, "A")
        ops.from_numpy(b, "B")
        left, ref_a = "A", a.astype(np.float64)
        if a_view:
            ops.transpose("A", out="At")
            left = "At"
        if kind == "recip":
            ops.elementwise("recip", out="P", operands=(left,))
            ref_a = 1.0 / ref_a
        else:
            v = (rng.random({"none": (M, K), "row": (1, K), "col": (M, 1)}[kind]) + 0.5).astype(np.float32)
            ops.from_numpy(v, "v")
            ops.elementwise("div", out="P", operands=(left, "v"), y_broadcast=kind)
            ref_a = ref_a / v
        ops.matmul(a="P", b="B", out="C")
        got = run(ops).env["C"]
        ref = ref_a @ b.astype(np.float64)
        # the quotients are within 2 ulp, the sum as above
        assert np.all(np.abs(got - ref) <= (K + 12) * 2.0**-24 * (np.abs(ref_a) @ np.abs(b.astype(np.float64))))


@pytest.mark.parametrize("divisor", [False, True])
@pytest.mark.parametrize("index", range(len(config.FILL_TILES)))
def test_a_along_its_rows(index, divisor, monkeypatch):
    """A transposed view of A: its loader stores 4, 2 or 1 columns of a row at a
    time, by the tile and its lanes; whole and ragged rows and k's."""
    tile = config.FILL_TILES[index].tile
    monkeypatch.setattr(mm, "select_filled", lambda *a, **k: (tile, 1))
    monkeypatch.setattr(mm, "fills", lambda *a, **k: False)
    for shape in ((256, 256, 256), (300, 517, 259)):
        print(f"filled A^T {shape} {tile.tile_M}x{tile.tile_N} divisor={divisor}", flush=True)
        ops, ref, bound = _program(shape, a_view=True, divisor=divisor)
        # the quotient rounds once more and its divisor's reciprocal twice
        _check(ops, ref, bound + 4 * 2.0**-24 * bound / ((shape[1] + 8) * 2.0**-24))
