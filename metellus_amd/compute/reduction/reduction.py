"""Last-axis reduction fragments for gfx950 (sum / max / min / product).

Replaces the reference's one-threadgroup-per-row simdgroup reduction
(reference: src/compute/reduction/reduction.py:23-205) with a wave64 design:

* ``W`` waves cooperate on a row (``T = 64*W`` lanes) and a 256-lane
  workgroup holds ``R = 4/W`` rows.  W = 1 (one wave per row, no LDS) when
  there are enough rows to fill the GPU; W = 2 or 4 for few, long rows.
* Each lane walks its row in chunks.  Vector path (unit column stride,
  K % 4 == 0, row stride % 4 == 0): lane t reads float4 chunks
  q = t, t+T, t+2T, ... (elements 4q..4q+3) into four accumulators a0..a3
  (a_j sees element 4q+j), then its value is (a0 op a1) op (a2 op a3).
  Scalar path: lane t reads elements t, t+T, ... into a0; its value is a0.
  Up to U chunks are loaded before they are combined, in chunk order.
* The 64 lane values of a wave are combined by the butterfly
  ``v = v op shfl_xor(v, off)`` for off = 32, 16, 8, 4, 2, 1.
* With W > 1 each wave's result goes to LDS ``scratch``; the row's first
  wave folds them left to right: ((w0 op w1) op w2) op w3.
* The optional epilogue is applied to the final value, which lane 0 stores.

This order is fixed and documented so the CPU oracle
(``oracle/ir_eval.py: ordered_row_reduce``) replays it exactly: sums and
products are then bit-identical to the oracle's, not merely close.
"""

from __future__ import annotations

from dataclasses import dataclass
from typing import Callable

from metellus_amd.compute.fragments import CodegenContext, TgmemAccess

REDUCTION_OPS = ("sum", "max", "min", "product")

ValueTransform = Callable[[str], str]

# Measured on MI355X with the caches flushed by a read pass before each
# launch: nontemporal loads take an 8192^2 row reduction from ~48 us to
# ~42.5 us (6.3 TB/s) and the 32-head 2048^2 attention reductions from
# ~89 us to ~81 us (6.6 TB/s); unroll 4..32 and 1..4 waves per row move
# either by less than run-to-run noise.
UNROLL = 16  # float4 chunks (or elements) in flight per lane
NT_LOAD = True  # nontemporal (streaming) row loads


def _identity(op: str) -> str:
    return {"sum": "0.0f", "product": "1.0f", "max": "(-INFINITY)", "min": "INFINITY"}[op]


def _combine(op: str, a: str, b: str) -> str:
    if op == "sum":
        return f"{a} + {b}"
    if op == "product":
        return f"{a} * {b}"
    if op == "max":
        return f"fmaxf({a}, {b})"
    if op == "min":
        return f"fminf({a}, {b})"
    raise ValueError(f"unsupported reduction op: {op}")


def _mult4(v: str) -> bool:
    try:
        return int(v) % 4 == 0
    except (TypeError, ValueError):
        return False


def _uint(v: str) -> str:
    """An unsigned operand: integer literals get the ``u`` suffix, anything
    else (a dim name or expression) is parenthesised."""
    try:
        return f"{int(v)}u"
    except (TypeError, ValueError):
        return f"({v})"


def _check_op(op: str) -> None:
    if op not in REDUCTION_OPS:
        raise ValueError(f"unsupported reduction op: {op}")


def scratch_floats(waves_per_row: int, rows_per_group: int) -> int:
    return waves_per_row * rows_per_group if waves_per_row > 1 else 0


@dataclass(frozen=True)
class LastAxisReductionSetupFragment:
    """Declares ``lane``, ``wave``, ``row`` (this lane's row), ``t`` (lane
    index within the row's T lanes) and ``row_ok``."""

    rows_dim: str
    name: str
    waves_per_row: int | None = None
    rows_per_group: int = 1
    kind: str = "setup"

    @property
    def tgmem_accesses(self) -> tuple[TgmemAccess, ...]:
        return ()

    def render(self, ctx: CodegenContext) -> str:
        W = self.waves_per_row or max(1, ctx.tg_x // 64)
        R = self.rows_per_group
        return "\n".join(
            [
                "const unsigned lane = mt_lane();",
                "const unsigned wave = mt_wave();",
                f"const unsigned row = blockIdx.x * {R}u + wave / {W}u;",
                f"const unsigned t = (wave % {W}u) * 64u + lane;",
                f"const bool row_ok = row < {self.rows_dim};",
            ]
        )


@dataclass(frozen=True)
class LastAxisReductionComputeFragment:
    """Per-row reduction of ``input_name[row*row_stride + idx*col_stride]``
    over ``idx < reduce_dim``; ``value_transform`` wraps each element (it may
    use ``row`` and ``idx``).  Leaves the lane's wave-reduced value in ``r``
    (valid in the row's first wave)."""

    op: str
    input_name: str
    scratch_name: str
    reduce_dim: str
    row_stride: str
    name: str
    tg_x: int
    col_stride: str = "1"
    value_transform: ValueTransform | None = None
    waves_per_row: int | None = None
    rows_per_group: int = 1
    vectorized: bool | None = None
    unroll: int = UNROLL
    nt_load: bool = NT_LOAD
    kind: str = "compute"

    @property
    def W(self) -> int:
        return self.waves_per_row or max(1, self.tg_x // 64)

    @property
    def tgmem_accesses(self) -> tuple[TgmemAccess, ...]:
        n = scratch_floats(self.W, self.rows_per_group)
        if n == 0:
            return ()
        return (TgmemAccess(self.scratch_name, "readwrite", n, (n,)),)

    def _vec(self) -> bool:
        """128-bit loads need contiguous rows whose length and stride are
        known multiples of 4 (the vector loop covers ``reduce_dim / 4``
        quads and nothing else); symbolic sizes take the per-element loop."""
        if self.vectorized is not None:
            return self.vectorized
        return self.col_stride == "1" and _mult4(self.reduce_dim) and _mult4(self.row_stride)

    def render(self, ctx: CodegenContext) -> str:
        _check_op(self.op)
        W, T = self.W, 64 * self.W
        U = self.unroll
        ld4 = "mt_ld4_nt" if self.nt_load else "mt_ld4"
        ident = _identity(self.op)
        tf = self.value_transform or (lambda raw: raw)
        src = f"{self.input_name} + (size_t)row * {_uint(self.row_stride)}"
        L = [f"float a0 = {ident}, a1 = {ident}, a2 = {ident}, a3 = {ident};", "if (row_ok) {",
             f"    const float* __restrict__ src = {src};"]
        if self._vec():
            L += [
                f"    const unsigned nq = {self.reduce_dim} / 4u;",
                "    unsigned q = t;",
                f"    for (; q + {(U - 1) * T}u < nq; q += {U * T}u) {{",
                f"        mt_f32x4 x[{U}];",
                "#pragma unroll",
                f"        for (int u = 0; u < {U}; ++u) x[u] = {ld4}(src + 4u * (q + (unsigned)u * {T}u));",
                "#pragma unroll",
                f"        for (int u = 0; u < {U}; ++u) {{",
            ]
            for j in range(4):
                L += [
                    f"            {{ const unsigned idx = 4u * (q + (unsigned)u * {T}u) + {j}u; (void)idx;",
                    f"              a{j} = {_combine(self.op, f'a{j}', tf(f'x[u][{j}]'))}; }}",
                ]
            L += [
                "        }",
                "    }",
                f"    for (; q < nq; q += {T}u) {{",
                f"        const mt_f32x4 xv = {ld4}(src + 4u * q);",
            ]
            for j in range(4):
                L += [
                    f"        {{ const unsigned idx = 4u * q + {j}u; (void)idx;",
                    f"          a{j} = {_combine(self.op, f'a{j}', tf(f'xv[{j}]'))}; }}",
                ]
            L += ["    }"]
        else:
            cs = self.col_stride
            load = "src[idx]" if cs == "1" else f"src[(size_t)idx * {_uint(cs)}]"
            L += [
                "    unsigned e = t;",
                f"    for (; e + {(U - 1) * T}u < {self.reduce_dim}; e += {U * T}u) {{",
                f"        float x[{U}];",
                "#pragma unroll",
                f"        for (int u = 0; u < {U}; ++u) {{ const unsigned idx = e + (unsigned)u * {T}u; x[u] = {load}; }}",
                "#pragma unroll",
                f"        for (int u = 0; u < {U}; ++u) {{",
                f"            const unsigned idx = e + (unsigned)u * {T}u; (void)idx;",
                f"            a0 = {_combine(self.op, 'a0', tf('x[u]'))};",
                "        }",
                "    }",
                f"    for (; e < {self.reduce_dim}; e += {T}u) {{",
                f"        const unsigned idx = e; const float xv = {load};",
                f"        a0 = {_combine(self.op, 'a0', tf('xv'))};",
                "    }",
            ]
        L += ["}"]
        if self._vec():
            lo = "(" + _combine(self.op, "a0", "a1") + ")"
            hi = "(" + _combine(self.op, "a2", "a3") + ")"
            L.append(f"float r = {_combine(self.op, lo, hi)};")
        else:
            L.append("float r = a0;")
        L.append(f"r = mt_wave_{self.op}(r);")
        if W > 1:
            sc = self.scratch_name
            L += [
                f"if (lane == 0u) {sc}[wave] = r;",
                "__syncthreads();",
                f"if (wave % {W}u == 0u) {{",
                f"    r = {sc}[wave];",
            ]
            for w in range(1, W):
                L.append(f"    r = {_combine(self.op, 'r', f'{sc}[wave + {w}u]')};")
            L.append("}")
        return "\n".join(L)


STRIDED_LANES = 512
STRIDED_LOADS = 32  # elements in flight per lane (16: 8192 rows of 8192 61 instead of 49 us, 64: 53)


@dataclass(frozen=True)
class StridedReductionFragment(LastAxisReductionComputeFragment):
    """The same reduction of rows that are contiguous across each other (row
    stride 1: the columns of a row-major matrix, e.g. a bias gradient), in the
    same order.  One wave per row would load one element per cache line; here a
    workgroup takes ``rows`` rows, as many lanes load one element of each at a
    time, and lane group G keeps the partial values of lanes t = J G .. J G + J - 1
    of the wave-per-row order (J = T rows / STRIDED_LANES).  They meet in LDS, where one lane per
    row folds them along the butterfly's tree.  Bound by what the workgroups keep in
    flight; measured on MI355X against a wave per row: 4096 rows of 4096 (64 MiB,
    128 workgroups) 103 -> 15 us, 1000 rows of 16384 141 -> 31 us.  Includes the store (``out_name``, ``epilogue``)."""

    rows_dim: str = "M"
    rows: int = 32
    out_name: str = ""
    epilogue: ValueTransform | None = None
    kind: str = "compute"

    @property
    def tgmem_accesses(self) -> tuple[TgmemAccess, ...]:
        shape = strided_scratch_shape(self.W, self.rows)
        return (TgmemAccess(self.scratch_name, "readwrite", shape[0] * shape[1], shape),)

    def render(self, ctx: CodegenContext) -> str:
        _check_op(self.op)
        W, R = self.W, self.rows
        T = 64 * W
        J = T * R // STRIDED_LANES
        U = max(1, STRIDED_LOADS // J)  # chunks of T elements in flight
        ident = _identity(self.op)
        tf = self.value_transform or (lambda raw: raw)
        ep = self.epilogue or (lambda raw: raw)
        sc = self.scratch_name
        at = f"src[(size_t)idx * {_uint(self.col_stride)}]"
        lines = [
            f"const unsigned mt_r = threadIdx.x % {R}u, mt_g = threadIdx.x / {R}u;",
            f"const unsigned row = blockIdx.x * {R}u + mt_r;",
            f"const bool row_ok = row < {self.rows_dim};",
            f"float mt_acc[{J}];",
            "#pragma unroll",
            f"for (int j = 0; j < {J}; ++j) mt_acc[j] = {ident};",
            "if (row_ok) {",
            f"    const float* __restrict__ src = {self.input_name} + row;",
            f"    unsigned e = mt_g * {J}u;  // this lane's first element of the chunk",
            f"    for (; e + {(U - 1) * T + J - 1}u < {self.reduce_dim}; e += {U * T}u) {{",
            f"        float x[{U}][{J}];",
            "#pragma unroll",
            f"        for (int u = 0; u < {U}; ++u)",
            "#pragma unroll",
            f"            for (int j = 0; j < {J}; ++j) {{",
            f"                const unsigned idx = e + (unsigned)(u * {T} + j);",
            f"                x[u][j] = {at};",
            "            }",
            "#pragma unroll",
            f"        for (int u = 0; u < {U}; ++u)",
            "#pragma unroll",
            f"            for (int j = 0; j < {J}; ++j) {{",
            f"                const unsigned idx = e + (unsigned)(u * {T} + j);",
            "                (void)idx;",
            f"                mt_acc[j] = {_combine(self.op, 'mt_acc[j]', tf('x[u][j]'))};",
            "            }",
            "    }",
            f"    for (; e < {self.reduce_dim}; e += {T}u) {{  // the rest: all loads of a chunk, then its sums",
            f"        float x[{J}];",
            "#pragma unroll",
            f"        for (int j = 0; j < {J}; ++j) {{",
            "            const unsigned idx = e + (unsigned)j;",
            f"            x[j] = idx < {self.reduce_dim} ? {at} : 0.0f;",
            "        }",
            "#pragma unroll",
            f"        for (int j = 0; j < {J}; ++j) {{",
            "            const unsigned idx = e + (unsigned)j;",
            f"            if (idx < {self.reduce_dim}) mt_acc[j] = {_combine(self.op, 'mt_acc[j]', tf('x[j]'))};",
            "        }",
            "    }",
            "}",
            "#pragma unroll",
            f"for (int j = 0; j < {J}; ++j) {sc}[mt_g * {J}u + (unsigned)j][mt_r] = mt_acc[j];",
            "__syncthreads();",
            f"if (threadIdx.x < {R}u && row_ok) {{",
            "    float r = 0.0f;",
            f"    for (unsigned w = 0; w < {W}u; ++w) {{  // a wave's 64 lanes, then the waves left to right",
            "        float mt_v[64];",
            "#pragma unroll",
            f"        for (int t = 0; t < 64; ++t) mt_v[t] = {sc}[64u * w + (unsigned)t][mt_r];",
            "#pragma unroll",
            "        for (int off = 32; off > 0; off >>= 1)",
            "#pragma unroll",
            f"            for (int t = 0; t < off; ++t) mt_v[t] = {_combine(self.op, 'mt_v[t]', 'mt_v[t + off]')};",
            f"        r = w == 0u ? mt_v[0] : {_combine(self.op, 'r', 'mt_v[0]')};",
            "    }",
            f"    {self.out_name}[row] = {ep('r')};",
            "}",
        ]
        return "\n".join(lines)


def strided_scratch_shape(waves_per_row: int, rows: int) -> tuple[int, int]:
    return (64 * waves_per_row, rows)


@dataclass(frozen=True)
class StoreReductionResultFragment:
    """Lane 0 of the row's first wave stores ``r`` (optionally transformed)."""

    output_name: str
    scratch_name: str
    name: str
    tg_x: int
    value_transform: ValueTransform | None = None
    setup: tuple[str, ...] = ()
    waves_per_row: int | None = None
    kind: str = "store"

    @property
    def tgmem_accesses(self) -> tuple[TgmemAccess, ...]:
        return ()

    def render(self, ctx: CodegenContext) -> str:
        W = self.waves_per_row or max(1, self.tg_x // 64)
        lines = ["float v = r;", *self.setup]
        if self.value_transform is not None:
            lines.append(f"v = {self.value_transform('v')};")
        lines.append(f"{self.output_name}[row] = v;")
        body = "\n    ".join(lines)
        return f"if (row_ok && lane == 0u && wave % {W}u == 0u) {{\n    {body}\n}}"
