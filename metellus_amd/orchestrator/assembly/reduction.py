"""Reduction strategy: standalone, prologue-fused or epilogue-fused
last-axis reduction (reference: src/orchestrator/assembly/reduction.py:24-109).

Bindings ``(src, out, *extras)`` and dims ``(M, K)`` follow the reference.
The launch differs: 256-lane workgroups holding ``4/W`` rows with ``W``
waves per row (see ``compute.reduction.reduction``); grid ``(ceil(M/R), 1, 1)``.
"""

from __future__ import annotations

from metellus_amd.compute.fragments import CodegenContext, lds_decl
from metellus_amd.compute.reduction import reduction as _red
from metellus_amd.compute.reduction.reduction import (
    LastAxisReductionComputeFragment,
    LastAxisReductionSetupFragment,
    StoreReductionResultFragment,
    StridedReductionFragment,
    scratch_floats,
    strided_scratch_shape,
)
from metellus_amd.orchestrator.assembly.decision import DecisionView
from metellus_amd.orchestrator.assembly.expressions import (
    build_reduction_epilogue_transform,
    chain_value_transform,
)
from metellus_amd.orchestrator.assembly.extras import Extras, input_param, output_param, param_name
from metellus_amd.orchestrator.ir import ReductionOp, Tensor
from metellus_amd.orchestrator.kernel_group import KernelGroup
from metellus_amd.runtime.program import Kernel

WG_LANES = 256
FORCE_WAVES_PER_ROW: int | None = None  # tuning override


def reduction_waves_per_row(M: int, K: int) -> int:
    """Waves cooperating on one row: 1 when M rows already give >= 2048
    waves; otherwise up to 4, as long as each lane still gets >= 16 elements."""
    if FORCE_WAVES_PER_ROW is not None:
        return FORCE_WAVES_PER_ROW
    W = 1
    while W < 4 and M * W < 2048 and K >= 64 * (2 * W) * 16:
        W *= 2
    return W


# A reduction of side-by-side rows from so many of them on, or of rows up to so
# long: fewer and longer ones are a few workgroups, and a wave per row keeps more
# loads in flight.  Measured on MI355X, this way against a wave per row: 256 rows of
# 4096 6 against 9 us, 70 of 4096 6.8 against 6.2, 64 of 8192 8 against 10.5, 192 of
# 16384 24 against 22, 32 of 65536 70 against 52, 320 of 65536 156 against 186.
STRIDED_MIN_ROWS = 320
STRIDED_MAX_LENGTH = 5120


def strided_rows(src: Tensor) -> bool:
    """Rows lying side by side in memory (the columns of a row-major matrix), at
    least 32 of them and a wave's 64 elements each: the lanes of a workgroup then
    load contiguous bytes where a wave per row loads 64 cache lines."""
    M, K = src.shape
    if src.row_stride != 1 or src.col_stride == 1 or M < 32 or K < 64:
        return False
    return M >= STRIDED_MIN_ROWS or K <= STRIDED_MAX_LENGTH


def strided_rows_per_group(M: int) -> int:
    """32 rows fill a 128-byte line; fewer where that leaves compute units without a
    workgroup (1000 rows of 16384: 40 us with 32 rows, 31 with 16, 38 with 8; 3001
    of 3000: 15, 18, 27; 70 of 5000: 15, 12, 9.6)."""
    return 8 if M < 128 else 16 if M < 2560 else 32


def _assemble_strided(decision: DecisionView, function_name: str | None, src: Tensor, final_out: Tensor,
                      extras: Extras, helpers: list[str], prologue, epilogue, M: int, K: int, W: int) -> KernelGroup:
    anchor = decision.anchor
    rows = strided_rows_per_group(M)
    frag = StridedReductionFragment(
        op=anchor.op,
        input_name=param_name(src.buffer_key),
        scratch_name="scratch",
        reduce_dim="K",
        row_stride=str(src.row_stride),
        col_stride=str(src.col_stride),
        name="reduction_compute",
        tg_x=_red.STRIDED_LANES,
        value_transform=prologue,
        waves_per_row=W,
        vectorized=False,
        rows=rows,
        out_name=param_name(final_out.buffer_key),
        epilogue=epilogue,
    )
    ctx = CodegenContext(
        function_name=function_name or f"reduce_{anchor.out.name}_fused",
        buffers=(input_param(src.buffer_key), output_param(final_out.buffer_key), *extras.buffers),
        dims=("M", "K"),
        tg_x=_red.STRIDED_LANES,
        tg_y=1,
        threadgroup_decls=(lds_decl("scratch", strided_scratch_shape(W, rows)),),
        helpers=tuple(helpers),
    )
    return KernelGroup(
        kernel=Kernel(fragments=(frag,), ctx=ctx),
        bindings=(src.buffer_key, final_out.buffer_key, *extras.bindings),
        dims=(M, K),
        grid=((M + rows - 1) // rows, 1, 1),
        threads=(_red.STRIDED_LANES, 1, 1),
        ops=decision.ops,
        strategy=decision.strategy,
    )


def assemble_reduction(decision: DecisionView, function_name: str | None) -> KernelGroup:
    anchor = decision.anchor
    assert isinstance(anchor, ReductionOp)
    src = decision.prologue_a[0].operands[0] if decision.prologue_a else anchor.input
    assert isinstance(src, Tensor)
    M, K = src.shape
    final_out = decision.epilogue[-1].out if decision.epilogue else anchor.out
    extras = Extras(base_slots_by_key={src.buffer_key: 0, final_out.buffer_key: 1})
    helpers: list[str] = []
    prologue = None
    if decision.prologue_a:
        prologue = chain_value_transform(
            decision.prologue_a, row_var="row", col_var="idx", extras=extras, base_slot=2, name="prologue"
        )
        helpers.append(prologue.helper)
    epilogue = None
    if decision.epilogue:
        epilogue = build_reduction_epilogue_transform(decision.epilogue, name="epilogue")
        helpers.append(epilogue.helper)

    W = reduction_waves_per_row(M, K)
    if strided_rows(src):
        return _assemble_strided(decision, function_name, src, final_out, extras, helpers, prologue, epilogue, M, K, W)
    R = WG_LANES // (64 * W)
    vec = src.col_stride == 1 and K % 4 == 0 and src.row_stride % 4 == 0
    setup = LastAxisReductionSetupFragment(rows_dim="M", name="reduction_setup", waves_per_row=W, rows_per_group=R)
    compute = LastAxisReductionComputeFragment(
        op=anchor.op,
        input_name=param_name(src.buffer_key),
        scratch_name="scratch",
        reduce_dim="K",
        row_stride=str(src.row_stride),
        col_stride=str(src.col_stride),
        name="reduction_compute",
        tg_x=WG_LANES,
        value_transform=prologue,
        waves_per_row=W,
        rows_per_group=R,
        vectorized=vec,
        unroll=_red.UNROLL,
        nt_load=_red.NT_LOAD,
    )
    store = StoreReductionResultFragment(
        output_name=param_name(final_out.buffer_key),
        scratch_name="scratch",
        name="reduction_store",
        tg_x=WG_LANES,
        value_transform=epilogue,
        waves_per_row=W,
    )
    n_scratch = scratch_floats(W, R)
    ctx = CodegenContext(
        function_name=function_name or f"reduce_{anchor.out.name}_fused",
        buffers=(input_param(src.buffer_key), output_param(final_out.buffer_key), *extras.buffers),
        dims=("M", "K"),
        tg_x=WG_LANES,
        tg_y=1,
        threadgroup_decls=(lds_decl("scratch", (n_scratch,)),) if n_scratch else (),
        helpers=tuple(helpers),
    )
    return KernelGroup(
        kernel=Kernel(fragments=(setup, compute, store), ctx=ctx),
        bindings=(src.buffer_key, final_out.buffer_key, *extras.bindings),
        dims=(M, K),
        grid=((M + R - 1) // R, 1, 1),
        threads=(WG_LANES, 1, 1),
        ops=decision.ops,
        strategy=decision.strategy,
    )


def reduction_order(group: KernelGroup) -> dict:
    """The combine-order parameters of a reduction kernel (for the CPU
    replay of its exact order): op, waves per row, vector path."""
    frag = next(f for f in group.kernel.fragments if isinstance(f, LastAxisReductionComputeFragment))
    return {"op": frag.op, "waves_per_row": frag.W, "vectorized": frag._vec(), "unroll": frag.unroll}
