"""Skinny matmuls (``mt_sn_*``) on the GPU against float64, within the rounding
of an fp32 sum: every row-block count, ragged edges of tiles, groups and
128-bit loads, both readings of B, views of A, prologues of every broadcast,
epilogues, splits over workgroups (and the counters they leave), batches."""

from __future__ import annotations

import numpy as np
import pytest

from metellus_amd.api import compile_program, run, run_batch
from metellus_amd.orchestrator import Operations
from metellus_amd.orchestrator.assembly import matmul as mm

pytestmark = pytest.mark.gpu

SHAPES = [(1, 129, 64), (1, 4096, 65), (3, 128, 128), (16, 1000, 331), (17, 77, 1001), (33, 1027, 258), (64, 2048, 67),
          (8, 4096, 1024)]


def _program(shape, a_view=False, b_view=False, prologue=None, epilogue=False, seed=11):
    M, K, N = shape
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((M, K)).astype(np.float32)
    b = rng.standard_normal((K, N)).astype(np.float32)
    ops = Operations()
    ops.from_numpy(np.ascontiguousarray(a.T) if a_view else a, "A")
    ops.from_numpy(np.ascontiguousarray(b.T) if b_view else b, "B")
    left, right = "A", "B"
    if a_view:
        ops.transpose("A", out="At")
        left = "At"
    if b_view:
        ops.transpose("B", out="Bt")
        right = "Bt"
    ref_a = a.astype(np.float64)
    if prologue is not None:
        sizes = {"none": (M, K), "row": (1, K), "col": (M, 1), "scalar": (1, 1)}
        for name, kind in (("p", prologue), ("q", "none")):
            v = (rng.random(sizes[kind]) + 0.5).astype(np.float32)
            ops.from_numpy(v, name)
            ops.elementwise("mul", out=name + "m", operands=(left, name), y_broadcast=kind)
            left = name + "m"
            ref_a = ref_a * v
    ops.matmul(a=left, b=right, out="C")
    ref = ref_a @ b.astype(np.float64)
    bound = np.abs(ref_a) @ np.abs(b.astype(np.float64))
    out = "C"
    if epilogue:
        bias = rng.standard_normal((1, N)).astype(np.float32)
        ops.from_numpy(bias, "bias")
        ops.elementwise("add", out="Cb", operands=("C", "bias"), y_broadcast="row")
        ops.elementwise("max", out="Y", operands=("Cb", 0.0))
        ref, out = np.maximum(ref + bias, 0.0), "Y"
        bound = bound + np.abs(bias)
    return ops, out, ref, bound


def _check(got, ref, bound, K):
    # K products and sums, each rounded by at most 2^-24 of the sum of magnitudes
    assert np.all(np.abs(got - ref) <= (K + 8) * 2.0**-24 * bound + 1e-37)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("a_view,b_view", [(False, False), (False, True), (True, False)])
def test_shapes_and_views(shape, a_view, b_view):
    print(f"skinny {shape} a_view={a_view} b_view={b_view}", flush=True)
    ops, out, ref, bound = _program(shape, a_view, b_view, epilogue=True)
    (g,) = compile_program(ops)
    assert "mt_sn_mainloop<" in g.kernel.source.split('extern "C"')[-1]
    for _ in range(2):  # a split's counters are left at zero
        _check(run(ops).env[out], ref, bound, shape[1])


@pytest.mark.parametrize("prologue", ["none", "row", "col", "scalar"])
@pytest.mark.parametrize("a_view", [False, True])
def test_prologues(prologue, a_view):
    for shape in ((8, 1000, 331), (40, 1031, 131)):
        print(f"skinny prologue {prologue} {shape} a_view={a_view}", flush=True)
        ops, out, ref, bound = _program(shape, a_view=a_view, prologue=prologue)
        assert "mt_sn_mainloop<" in compile_program(ops)[-1].kernel.source.split('extern "C"')[-1]
        _check(run(ops).env[out], ref, bound, shape[1])


@pytest.mark.parametrize("splits", [1, 2, 5, 16])
def test_splits_and_repeats(splits, monkeypatch):
    """Any split adds in split order: repeated runs are bit-identical."""
    monkeypatch.setattr(mm, "skinny_shape", lambda M, K, N, batch=1: (1, 8, splits))
    ops, out, ref, bound = _program((7, 2100, 200))
    (g,) = compile_program(ops)
    assert g.grid == (4 * splits, 1, 1) and (g.kernel.workspace_bytes > 0) == (splits > 1)
    first = run(ops).env[out]
    _check(first, ref, bound, 2100)
    for _ in range(3):
        assert np.array_equal(run(ops).env[out], first)
    # the batched variant of a kernel built for one program walks whole tiles
    assert g.kernel.batched().workspace_bytes == 0 and "mt_ws" not in g.kernel.batched().source.split('extern "C"')[-1]


@pytest.mark.parametrize("b_view", [False, True])
def test_batch(b_view):
    made = [_program((2, 300, 140), b_view=b_view, seed=20 + i) for i in range(3)]
    for (ops, out, ref, bound), res in zip(made, run_batch([m[0] for m in made])):
        _check(res.env[out], ref, bound, 300)
