"""Data-moving kernels at odd sizes on the GPU: strided row reductions
(``StridedReductionFragment``, bit for bit the order of the wave-per-row kernel,
replayed on the CPU), elementwise chains and transposing copies whose rows end
inside a 128-bit slot."""

from __future__ import annotations

import numpy as np
import pytest

from metellus_amd.api import compile_program, run
from metellus_amd.orchestrator import Operations
from metellus_amd.orchestrator.assembly.reduction import reduction_order
from oracle.ir_eval import evaluate, ordered_row_reduce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("op", ["sum", "max", "min", "product"])
@pytest.mark.parametrize("shape", [(32, 64), (33, 65), (4096, 300), (70, 5000), (1000, 16384)], ids=str)
def test_strided_reduction_keeps_the_order(op, shape):
    M, K = shape
    print(f"strided reduction {op} {shape}", flush=True)
    rng = np.random.default_rng(3)
    x = rng.standard_normal((K, M)).astype(np.float32)
    if op == "product":
        x = (1.0 + 0.01 * x).astype(np.float32)
    if op in ("max", "min"):
        x[K // 2, 5] = np.nan
        x[K - 1, 7] = -np.inf
    ops = Operations()
    ops.from_numpy(x, "X")
    ops.transpose("X", out="Xt")
    ops.reduction(op, out="r", x="Xt")
    (g,) = compile_program(ops)
    assert "mt_acc[" in g.kernel.source.split('extern "C"')[-1] and g.threads == (512, 1, 1)
    order = reduction_order(g)
    ref = ordered_row_reduce(np.ascontiguousarray(x.T), **{k: v for k, v in order.items() if k != "unroll"})
    np.testing.assert_array_equal(run(ops).env["r"], ref)


def test_strided_reduction_with_prologue_and_epilogue():
    rng = np.random.default_rng(4)
    for M, K in ((129, 300), (40, 4100)):
        x = rng.standard_normal((K, M)).astype(np.float32)
        y = rng.standard_normal((M, K)).astype(np.float32)
        ops = Operations()
        ops.from_numpy(x, "X")
        ops.from_numpy(y, "y")
        ops.transpose("X", out="Xt")
        ops.elementwise("mul", out="p", operands=("Xt", "y"))
        ops.reduction("sum", out="s", x="p")
        ops.elementwise("mul", out="m", operands=("s", 1.0 / K))
        print(f"strided reduction with prologue {(M, K)}", flush=True)
        got = run(ops).env["m"]
        ref = (x.T.astype(np.float64) * y).sum(1) / K
        bound = (K + 4) * 2.0**-24 * np.abs(x.T.astype(np.float64) * y).sum(1) / K
        assert np.all(np.abs(got - ref) <= bound)


@pytest.mark.parametrize("n", [63, 64, 65, 255, 257, 1023, 4098])
def test_odd_chains(n):
    """IEEE-exact ops over every broadcast and a transposed view: the same bits
    as NumPy, and nothing outside the rows is written."""
    m = 37
    rng = np.random.default_rng(n)
    x, y, t = (rng.standard_normal(s).astype(np.float32) for s in ((m, n), (m, n), (n, m)))
    c, r = rng.standard_normal((m, 1)).astype(np.float32), rng.standard_normal((1, n)).astype(np.float32)
    ops = Operations()
    for name, v in (("x", x), ("y", y), ("t", t), ("c", c), ("r", r)):
        ops.from_numpy(v, name)
    ops.transpose("t", out="tt")
    ops.elementwise("subtract", out="a1", operands=("x", "c"), y_broadcast="col")
    ops.elementwise("mul", out="a2", operands=("a1", "r"), y_broadcast="row")
    ops.elementwise("add", out="a3", operands=("a2", "y"))
    ops.elementwise("div", out="z", operands=("a3", "tt"))
    print(f"odd chain {(m, n)}", flush=True)
    np.testing.assert_array_equal(run(ops).env["z"], evaluate(ops)["z"])


@pytest.mark.parametrize("shape", [(257, 256), (1023, 129), (300, 501), (4099, 17), (130, 515), (2, 40000)], ids=str)
def test_odd_transposes(shape):
    x = np.arange(shape[0] * shape[1], dtype=np.float32).reshape(shape)
    ops = Operations()
    ops.from_numpy(x, "x")
    ops.transpose("x", out="xt")
    ops.reshape("xt", (x.size,), out="y")
    print(f"odd transpose {shape}", flush=True)
    np.testing.assert_array_equal(run(ops).env["y"], x.T.reshape(-1))
