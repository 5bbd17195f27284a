"""Split matmuls at the ends of float32's range, in every kernel that splits
its operands (``mt_split``): operands too small for three bf16 parts against
ones large enough that the products are of ordinary size, and accumulators
that pass the largest float inside a step although no sum of products does."""

from __future__ import annotations

import numpy as np
import pytest

from metellus_amd.api import compile_program, run
from metellus_amd.compute.matmul import config
from metellus_amd.orchestrator import Operations
from metellus_amd.orchestrator.assembly import matmul as mm

pytestmark = pytest.mark.gpu

# kernel form: sizes, what picks it, its text
FORMS = {
    "short": ((129, 8, 195), {}, "mt_mfma_tile<"),
    "ragged tile": ((129, 331, 195), {}, "mt_mfma_tile<"),
    "long k loop": ((512, 1024, 256), {"FILL": False}, "mt_mfma_tile_held<"),
    "looking together": ((256, 512, 512), {"FILL": False}, "mt_k_loop(mt_cut<true>"),
    "summed in parts": ((256, 1024, 256), {}, "mt_part_i"),
    "in parts, looking together": ((1024, 1024, 1024), {}, "mt_k_loop(mt_cut<true>"),
    "stream-K": ((384, 512, 640), {"FILL": False}, "mt_sk_wait("),
    "row waves": ((256, 1024, 128), {}, "mt_rw_chunk("),
    "divided row waves": ((256, 1024, 128), {}, "mt_rw_chunk("),
    "divided tile": ((129, 331, 195), {}, "mt_mfma_tile<"),
    "transposed operands": ((129, 331, 195), {}, "mt_mfma_tile<"),
    "pair": ((130, 333, 200), {}, "acc_1"),
    "pair of two left operands": ((130, 333, 200), {}, "acc_1"),
    "pair, looking together": ((512, 512, 512), {"FILL": False}, "mt_k_loop(mt_cut<true>"),
}


def _form(name, monkeypatch):
    shape, flags, text = FORMS[name]
    for flag, value in flags.items():
        monkeypatch.setattr(mm, flag, value)
    if name == "stream-K":
        monkeypatch.setattr(config, "FORCE_TILE", config.TileConfig(128, 128, 32, 2, 2))
        monkeypatch.setattr(config, "PERSISTENT_CAPACITY", 8)
    return shape, text


def _product(name, a, b, text):
    """The product through the form's kernel; a pair's as the sum of two equal ones."""
    ops = Operations()
    left, right = "A", "B"
    if name.startswith("transposed"):
        ops.from_numpy(np.ascontiguousarray(a.T), "At")
        ops.from_numpy(np.ascontiguousarray(b.T), "Bt")
        ops.transpose("At", out="A")
        ops.transpose("Bt", out="B")
    else:
        ops.from_numpy(a, "A")
        ops.from_numpy(b, "B")
    if name.startswith("divided"):
        ops.from_numpy(np.full((a.shape[0], 1), 2.0, np.float32), "s")
        ops.elementwise("div", out="P", operands=("A", "s"), y_broadcast="col")
        left = "P"
    ops.matmul(a=left, b=right, out="C")
    out = "C"
    if name.startswith("pair"):
        ops.from_numpy(b, "B2")
        if "two" in name:
            ops.from_numpy(a, "A2")
        ops.matmul(a="A2" if "two" in name else "A", b="B2", out="C2")
        ops.elementwise("add", out="Y", operands=("C", "C2"))
        out = "Y"
    (g,) = compile_program(ops)
    assert text in g.kernel.source.split('extern "C"')[-1]
    got = run(ops).env[out]
    return got, {"d": 0.5, "p": 2.0}.get(name[0], 1.0) if name.startswith(("divided", "pair")) else 1.0


def _spread(rng, shape, low, high):
    return (rng.uniform(1.0, 2.0, shape) * rng.choice((-1.0, 1.0), shape)
            * np.exp2(rng.integers(low, high, shape, endpoint=True))).astype(np.float32)


@pytest.mark.parametrize("large", ["right", "left"])
@pytest.mark.parametrize("rows", ["every", "some"])
@pytest.mark.parametrize("low,high", [(-140, -112), (-117, -116), (-140, -140)])
@pytest.mark.parametrize("name", list(FORMS))
def test_small_against_large(name, low, high, rows, large, monkeypatch):
    """Below 2^-110 a float is no sum of three bf16 numbers; products with 2^40
    .. 2^100 are of ordinary size, so only the operands show it."""
    (M, K, N), text = _form(name, monkeypatch)
    print(f"split range {name} 2^{low}..2^{high} {rows} large={large}", flush=True)
    rng = np.random.default_rng(31)
    a, b = _spread(rng, (M, K), low, high), _spread(rng, (K, N), 40, 100)
    if rows == "some":  # the others share their waves and tiles
        a[np.arange(M) % 37 != 5] = 0.0
    if large == "left":
        flip = _spread(rng, (M, K), 40, 100), _spread(rng, (K, N), low, high)
        a, b = flip
        if rows == "some":
            b[:, np.arange(N) % 41 != 7] = 0.0
    if name.startswith("divided"):
        a = (a * np.float32(0.5)) * np.float32(2.0)  # exact quotients, subnormal ones too
    got, scale = _product(name, a, b, text)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    # K products and as many sums, each rounded by at most 2^-24 of the sum of
    # magnitudes (a part, a merge and an underflow are within the 8)
    bound = scale * (K + 8) * 2.0**-24 * (np.abs(a64) @ np.abs(b64)) + K * 2.0**-149
    assert np.all(np.abs(got - scale * (a64 @ b64)) <= bound)


@pytest.mark.parametrize("name", list(FORMS))
def test_small_values_of_a_softmax(name, monkeypatch):
    """Weights from 1 down to the smallest subnormal, as a row of exponentials has them."""
    (M, K, N), text = _form(name, monkeypatch)
    print(f"split range {name} softmax", flush=True)
    rng = np.random.default_rng(32)
    a = np.exp(-rng.uniform(0, 103, (M, K))).astype(np.float32)
    a[:, 0] = 1.0
    b = rng.standard_normal((K, N)).astype(np.float32)
    got, scale = _product(name, a, b, text)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    bound = scale * (K + 8) * 2.0**-24 * (np.abs(a64) @ np.abs(b64)) + K * 2.0**-149
    assert np.all(np.abs(got - scale * (a64 @ b64)) <= bound)


@pytest.mark.parametrize("name", [f for f in FORMS if not f.startswith("pair")])  # (twice the sum is infinite)
def test_largest_accumulators(name, monkeypatch):
    """-1.00586 is -1.0078 + 0.00195 in bf16 parts: added to 0.9995 of the largest
    float, the second part alone passes it, the product does not."""
    (M, K, N), text = _form(name, monkeypatch)
    print(f"split range {name} largest", flush=True)
    half = 0.5 if name.startswith("divided") else 1.0
    a, b = np.zeros((M, K), np.float32), np.zeros((K, N), np.float32)
    a[:, 0], b[0] = np.float32(0.9995 * 2.0**64 / half), np.float32(2.0**64)
    a[:, K - 1], b[K - 1] = np.float32(-1.005859375 * 2.0**63 / half), np.float32(2.0**64)
    a[0], b[:, 0] = 1.0, 1.0
    got, _ = _product(name, a, b, text)
    ref = half * (a.astype(np.float64) @ b.astype(np.float64))
    assert np.all(np.isfinite(got))
    assert np.all(np.abs(got - ref) <= (K + 8) * 2.0**-24 * half * (np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64))))
