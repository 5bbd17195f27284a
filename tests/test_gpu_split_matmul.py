"""Split matmuls on the GPU: fp32 operands as three bf16 parts, six bf16 MFMAs
per step (``mt_mfma_split``), with the fp32 retry for what a split cannot hold.

Precision: each of the six partial products is exact, so the result differs
from the float64 one by the accumulator's roundings, fewer than the fp32 MFMA
makes: the existing bar of an fp32 matmul (``matmul_tolerance``) holds.
Special values: NaNs and infinities come out where float32 arithmetic has
them, and operands below bf16's range keep their relative precision."""

from __future__ import annotations

import numpy as np
import pytest

from metellus_amd.api import compile_program, run
from metellus_amd.orchestrator import Operations
from oracle.ir_eval import matmul_tolerance

pytestmark = pytest.mark.gpu

SHAPES = [(256, 256, 256), (33, 47, 65), (300, 777, 1000), (512, 4096, 512)]


def _matmul(a: np.ndarray, b: np.ndarray, divisor: np.ndarray | None = None) -> np.ndarray:
    ops = Operations()
    ops.from_numpy(a, "A")
    ops.from_numpy(b, "B")
    left = "A"
    if divisor is not None:
        ops.from_numpy(divisor, "s")
        ops.reshape("s", (a.shape[0], 1), out="sv")
        ops.elementwise("div", out="P", operands=("A", "sv"), y_broadcast="col")
        left = "P"
    ops.matmul(a=left, b="B", out="C")
    assert "mt_mfma_retry<" in compile_program(ops)[-1].kernel.source.split('extern "C"')[-1]
    return run(ops).env["C"]


def _positive(shape, seed):
    rng = np.random.default_rng(seed)
    m, k, n = shape
    return (rng.random((m, k), dtype=np.float32) + 0.1, rng.random((k, n), dtype=np.float32) + 0.1)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("kind", ["normal", "positive", "wide exponents"])
def test_precision(shape, kind):
    print(f"split matmul {shape} {kind}", flush=True)
    rng = np.random.default_rng(3)
    a, b = _positive(shape, 3)
    if kind == "normal":
        a, b = (rng.standard_normal(x.shape).astype(np.float32) for x in (a, b))
    elif kind == "wide exponents":
        a *= np.exp2(rng.integers(-40, 40, a.shape)).astype(np.float32)
    c = _matmul(a, b)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    assert np.all(np.abs(c - ref) <= matmul_tolerance(a, b))
    # fp32 accumulation: at most one rounding of at most 2^-24 sum |a||b| for each
    # of the 6 products a step of 16 k's adds, and the dropped products' 2^-23
    k = shape[1]
    bound = (6 * -(-k // 16) + 2) * 2.0**-24 * (np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64)))
    assert np.all(np.abs(c - ref) <= bound)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("divided", [False, True])
def test_special_values(shape, divided):
    print(f"split matmul specials {shape} divided={divided}", flush=True)
    a, b = _positive(shape, 5)
    a[1, 2], a[2, 3], a[3, 4] = np.inf, -np.inf, np.nan
    a[5, 1] = np.float32(3.4e38)  # rounds to an infinite bf16
    a[7, :] = 0.0
    b[6, 9] = np.inf  # meets the zeros of row 7
    divisor = np.full(a.shape[0], 2.0, np.float32) if divided else None
    c = _matmul(a, b, divisor)
    with np.errstate(all="ignore"):
        left = (a / divisor[:, None] if divided else a).astype(np.float64)
        # NumPy's matmul may block infinities differently: sum term by term over k
        ref = np.zeros((a.shape[0], b.shape[1]))
        for k in range(a.shape[1]):
            ref += left[:, k, None] * b[None, k].astype(np.float64)
        ref32 = ref.astype(np.float32)
    assert np.array_equal(np.isnan(c), np.isnan(ref32))
    assert np.array_equal(np.isposinf(c), np.isposinf(ref32)) and np.array_equal(np.isneginf(c), np.isneginf(ref32))
    ok = np.isfinite(ref32)
    assert np.all(np.abs(c - ref)[ok] <= (1e-4 * np.sqrt(a.shape[1]) * np.abs(ref) + 1e-6)[ok])


@pytest.mark.parametrize("scale", [1e-30, 1e-36, 1e-39])
def test_small_operands(scale):
    """Below 2^-110 a split's lower parts vanish: the retry's fp32 MFMAs keep
    the precision (the rows of ordinary size share its tiles)."""
    for shape in SHAPES[:2]:
        print(f"split matmul small operands {shape} {scale}", flush=True)
        a, b = _positive(shape, 7)
        a[:16] = (a[:16].astype(np.float64) * scale).astype(np.float32)
        c = _matmul(a, b)
        ref = a.astype(np.float64) @ b.astype(np.float64)
        assert np.all(np.abs(c - ref) <= 1e-5 * np.abs(ref) + 2.0**-148)
