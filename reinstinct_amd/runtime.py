"""Launch sites of the path, as thin wrappers over the C ABI.  Arguments are
device pointers (ints or DeviceBuf) exactly as the C functions take them.

The calls that launch are compiled (csrc/python/native.cpp), or ctypes' where that extension is not built for this interpreter
(_calls.py); what follows here asks, sizes or places something.  Importing needs nothing built; a call without librein.so raises."""
import ctypes as C

from ._lib import MoeShape, check, lib

try:
    from ._native import (  # noqa: F401
        quantize_q8, rmsnorm_q8, add_rmsnorm_q8, swiglu_q8, sigmoid_mul_q8, rmsnorm_gated_q8, moe_geglu_q8, matvec_xq8,
        matvec_batched_xq8, matvec_multi_xq8, matvec_ondisk_xq8, matvec_q8_0_splitk, mmq_xq8, mmq_xq8_ws,
        mmq_xq8_noalloc, matmul, matmul_ws, moe_topk, moe_sort, moe_gather_xq, moe_quantize_scatter, moe_scatter_rows,
        moe_grouped_gemm, moe_grouped_swiglu_q8, moe_expert_matvec, moe_down, moe_gate_up_swiglu, moe_gate_up_swiglu_q8,
        moe_down_combine, swiglu_mul, moe_combine, moe_ffn)
except ImportError:
    from ._calls import (  # noqa: F401
        quantize_q8, rmsnorm_q8, add_rmsnorm_q8, swiglu_q8, sigmoid_mul_q8, rmsnorm_gated_q8, moe_geglu_q8, matvec_xq8,
        matvec_batched_xq8, matvec_multi_xq8, matvec_ondisk_xq8, matvec_q8_0_splitk, mmq_xq8, mmq_xq8_ws,
        mmq_xq8_noalloc, matmul, matmul_ws, moe_topk, moe_sort, moe_gather_xq, moe_quantize_scatter, moe_scatter_rows,
        moe_grouped_gemm, moe_grouped_swiglu_q8, moe_expert_matvec, moe_down, moe_gate_up_swiglu, moe_gate_up_swiglu_q8,
        moe_down_combine, swiglu_mul, moe_combine, moe_ffn)


def matvec_kernel_name(fmt, in_dim, out_dim, n_rows):
    """the kernel a product of 1..32 activation rows launches for this shape ('' where rein_mmq_xq8 launches token tiles)"""
    buf = C.create_string_buffer(64)
    check(lib.rein_matvec_kernel_name(fmt, in_dim, out_dim, n_rows, buf, len(buf)))
    return buf.value.decode()


def mmq_workspace_bytes(fmt, in_dim, p_rows):
    """bytes of workspace mmq_xq8_ws wants for this shape (0: none)"""
    return int(lib.rein_mmq_workspace_bytes(fmt, in_dim, p_rows))


def mmq_form_ws(fmt, in_dim, out_dim, p_rows, workspace_bytes):
    """0: int8 launch, 1: fp6 with one token group per workgroup, 2: fp6 split-tail, 3: int8 split-tail,
    4: fp16 with superblocks summed in the matrix unit (REIN_MMQ16=1)"""
    return int(lib.rein_mmq_form_ws(fmt, in_dim, out_dim, p_rows, workspace_bytes))


def mmq_workspace_min_bytes(fmt, in_dim, p_rows):
    """the smallest workspace rein_mmq_xq8_ws accepts: the activation image alone (no split-tail launch)"""
    return int(lib.rein_mmq_workspace_min_bytes(fmt, in_dim, p_rows))


def noalloc_prepare():
    """rein_noalloc_prepare: place the fixed scratch array on the current device; outside any capture."""
    check(lib.rein_noalloc_prepare())


def mmq_tile_plan_ws(fmt, out_dim, p_rows):
    """(n4, n2): token groups of four and of two 32-token tiles per 128-row block in mmq_xq8_ws"""
    n4, n2 = C.c_uint(0), C.c_uint(0)
    check(lib.rein_mmq_tile_plan_ws(fmt, out_dim, p_rows, C.byref(n4), C.byref(n2)))
    return n4.value, n2.value


def mmq_block_dots_ws(fmt, w, xq, out, in_dim, out_dim, n_rows, workspace, workspace_bytes, stream=None):
    check(lib.rein_mmq_block_dots_ws(fmt, w, xq, out, in_dim, out_dim, n_rows, workspace, workspace_bytes,
                                     stream.raw if stream is not None else None))


def matmul_scratch_bytes(fmt, in_dim, n_rows):
    return int(lib.rein_matmul_scratch_bytes(fmt, in_dim, n_rows))


def matmul_path(fmt, n_rows):
    rc = lib.rein_matmul_path(fmt, n_rows)
    if rc < 0:
        check(rc)
    return ("matvec", "batched_matvec", "mmq")[rc]


def mmq_tile_plan(fmt, in_dim, out_dim, p_rows):
    """64-token tiles per 128-row block that mmq_xq8 launches for this shape (0: 32-token tiles only)"""
    rc = lib.rein_mmq_tile_plan(fmt, in_dim, out_dim, p_rows)
    if rc < 0:
        check(rc)
    return rc


def block_dots(fmt, w, xq, out, in_dim, out_dim, n_rows, via_mfma=False, stream=None):
    check(lib.rein_block_dots(fmt, w, xq, out, in_dim, out_dim, n_rows, int(via_mfma),
                              stream.raw if stream is not None else None))


def moe_gemm_bn():
    return lib.rein_moe_gemm_bn()


def moe_shape(n_tok, hidden, n_expert, n_used, expert_ff, gate_up_fmt, down_fmt):
    return MoeShape(n_tok, hidden, n_expert, n_used, expert_ff, gate_up_fmt, down_fmt)


def moe_workspace_bytes(shape):
    return lib.rein_moe_workspace_bytes(C.byref(shape))
