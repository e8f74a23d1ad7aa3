"""Launch sites of the path, as thin wrappers over the C ABI.  Arguments are
device pointers (ints or DeviceBuf) exactly as the C functions take them."""
import ctypes as C

from ._lib import MoeShape, check, lib
from .hip import DeviceBuf

# A decode step makes hundreds of these calls of a few microseconds each, so a wrapper does nothing but the call: ctypes takes
# the pointer out of a DeviceBuf or Stream by itself (their `_as_parameter_`), and `check` is entered for an error only.


def _p(x):
    """for the elements of a table of pointers"""
    return x.ptr if isinstance(x, DeviceBuf) else x


def _table_types(n):
    return C.c_int * n, C.c_void_p * n, C.c_uint * n


_TABLES = [_table_types(n) for n in range(5)]         # matvec_multi_xq8 takes up to four matrices


def quantize_q8(x, xq, in_dim, n_vec=1, stream=None):
    """launch_quantize_q8 (src/runtime/qwen35.rs:3202-3211)"""
    rc = lib.rein_quantize_q8(x, xq, in_dim, n_vec, stream)
    if rc:
        check(rc)


def rmsnorm_q8(x, w, xq, n, n_vec=1, eps=1e-6, stream=None):
    """rmsnorm_q8_f32 (kernels/rmsnorm_q8.cpp:38-103): xq = q8(rmsnorm(x) * w)"""
    rc = lib.rein_rmsnorm_q8(x, w, xq, n, n_vec, eps, stream)
    if rc:
        check(rc)


def add_rmsnorm_q8(hidden, add, w, y, xq, n, n_vec=1, eps=1e-6, stream=None):
    """add_rmsnorm_q8_f32 (kernels/qwen35_fused.cpp:66-121): hidden += add; y, xq = rmsnorm(hidden) * w"""
    rc = lib.rein_add_rmsnorm_q8(hidden, add, w, y, xq, n, n_vec, eps, stream)
    if rc:
        check(rc)


def swiglu_q8(gate, up, out, xq, n, stream=None):
    """swiglu_q8_f32 (kernels/qwen35_fused.cpp:132-146): out, xq = silu(gate) * up"""
    rc = lib.rein_swiglu_q8(gate, up, out, xq, n, stream)
    if rc:
        check(rc)


def sigmoid_mul_q8(x, gate, xq, n, stream=None):
    """sigmoid_mul_q8_f32 (kernels/qwen35_fused.cpp:149-162): x *= sigmoid(gate); xq = q8(x)"""
    rc = lib.rein_sigmoid_mul_q8(x, gate, xq, n, stream)
    if rc:
        check(rc)


def rmsnorm_gated_q8(x, z, w, y, xq, n_heads, head_dim, eps=1e-6, stream=None):
    """rmsnorm_gated_q8_f32 (kernels/qwen35_fused.cpp:195-217)"""
    rc = lib.rein_rmsnorm_gated_q8(x, z, w, y, xq, n_heads, head_dim, eps, stream)
    if rc:
        check(rc)


def moe_geglu_q8(gu, xq, ff_exp, n_slot, stream=None):
    """moe_geglu_q8_f32 (kernels/moe_geglu_q8.cpp:31-66): xq = q8(gelu(gate) * up)"""
    rc = lib.rein_moe_geglu_q8(gu, xq, ff_exp, n_slot, stream)
    if rc:
        check(rc)


def matvec_xq8(fmt, w, xq, y, in_dim, out_dim, stream=None):
    """launch_matvec_repacked_xq8 (src/runtime/qwen35.rs:2232-2280)"""
    rc = lib.rein_matvec_xq8(fmt, w, xq, y, in_dim, out_dim, stream)
    if rc:
        check(rc)


def matvec_batched_xq8(fmt, w, xq, y, in_dim, out_dim, n_rows, stream=None):
    """matmul_kquant_batched_into minus its quantize (src/runtime/prefill.rs:448-508)"""
    rc = lib.rein_matvec_batched_xq8(fmt, w, xq, y, in_dim, out_dim, n_rows, stream)
    if rc:
        check(rc)


def matvec_multi_xq8(fmts, ws, ys, out_dims, xq, in_dim, n_rows=1, stream=None):
    """the decode step's consecutive matvecs on the same activations (Q / K / V, gate / up; src/runtime/qwen35.rs:2670-2672,
    2702-2703) as one launch: ys[i][n_rows][out_dims[i]] = xq . ws[i]^T, up to four matrices and four rows"""
    n = len(fmts)
    ints, pointers, unsigneds = _TABLES[n] if n < 5 else _table_types(n)
    rc = lib.rein_matvec_multi_xq8(n, ints(*fmts), pointers(*map(_p, ws)), pointers(*map(_p, ys)), unsigneds(*out_dims),
                                   xq, in_dim, n_rows, stream)
    if rc:
        check(rc)


def matvec_kernel_name(fmt, in_dim, out_dim, n_rows):
    """the kernel a product of 1..32 activation rows launches for this shape ('' where rein_mmq_xq8 launches token tiles)"""
    buf = C.create_string_buffer(64)
    rc = lib.rein_matvec_kernel_name(fmt, in_dim, out_dim, n_rows, buf, len(buf))
    if rc:
        check(rc)
    return buf.value.decode()


def matvec_ondisk_xq8(fmt, w_blocks, xq, y, in_dim, out_dim, stream=None):
    """the on-disk-layout dp4a matvec (src/runtime/qwen35.rs:2209-2229)"""
    rc = lib.rein_matvec_ondisk_xq8(fmt, w_blocks, xq, y, in_dim, out_dim, stream)
    if rc:
        check(rc)


def matvec_q8_0_splitk(w, xq, y_partials, in_dim, out_dim, n_split, stream=None):
    """matvec_q8_0_repacked_splitk_f32 (kernels/matvec_q8_0_repacked.cpp:117-176)"""
    rc = lib.rein_matvec_q8_0_splitk(w, xq, y_partials, in_dim, out_dim, n_split, stream)
    if rc:
        check(rc)


def mmq_xq8(fmt, w, xq, y, in_dim, out_dim, p_rows, stream=None):
    """matmul_mmq_into minus its quantize (src/runtime/prefill.rs:512-567)"""
    rc = lib.rein_mmq_xq8(fmt, w, xq, y, in_dim, out_dim, p_rows, stream)
    if rc:
        check(rc)


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


def mmq_xq8_ws(fmt, w, xq, y, in_dim, out_dim, p_rows, workspace, workspace_bytes, stream=None):
    """mmq_xq8 with the caller's workspace (the scratch PrefillGemm keeps, prefill.rs:479-495)"""
    rc = lib.rein_mmq_xq8_ws(fmt, w, xq, y, in_dim, out_dim, p_rows, workspace, workspace_bytes,
                             stream)
    if rc:
        check(rc)


def noalloc_prepare():
    """rein_noalloc_prepare: place the fixed scratch array on the current device; outside any capture."""
    rc = lib.rein_noalloc_prepare()
    if rc:
        check(rc)


def mmq_xq8_noalloc(fmt, w, xq, y, in_dim, out_dim, p_rows, stream=None):
    """mmq_xq8_ws on the library's fixed 48 MiB device array: allocates nothing"""
    rc = lib.rein_mmq_xq8_noalloc(fmt, w, xq, y, in_dim, out_dim, p_rows, stream)
    if rc:
        check(rc)


def mmq_tile_plan_ws(fmt, out_dim, p_rows):
    """(n4, n2): token groups of four and of two 32-token tiles per 128-row block in mmq_xq8_ws"""
    n4, n2 = C.c_uint(0), C.c_uint(0)
    rc = lib.rein_mmq_tile_plan_ws(fmt, out_dim, p_rows, C.byref(n4), C.byref(n2))
    if rc:
        check(rc)
    return n4.value, n2.value


def mmq_block_dots_ws(fmt, w, xq, out, in_dim, out_dim, n_rows, workspace, workspace_bytes, stream=None):
    rc = lib.rein_mmq_block_dots_ws(fmt, w, xq, out, in_dim, out_dim, n_rows, workspace,
                                    workspace_bytes, stream)
    if rc:
        check(rc)


def matmul_scratch_bytes(fmt, in_dim, n_rows):
    return int(lib.rein_matmul_scratch_bytes(fmt, in_dim, n_rows))


def matmul_ws(fmt, w, x, y, in_dim, out_dim, n_rows, scratch, scratch_bytes, stream=None):
    """matmul with one scratch buffer for the quantized activations and the MMQ workspace"""
    rc = lib.rein_matmul_ws(fmt, w, x, y, in_dim, out_dim, n_rows, scratch, scratch_bytes, stream)
    if rc:
        check(rc)


def matmul(fmt, w, x, y, in_dim, out_dim, n_rows, xq_scratch, stream=None):
    """PrefillGemm::matmul_into_raw (src/runtime/prefill.rs:343-384)"""
    rc = lib.rein_matmul(fmt, w, x, y, in_dim, out_dim, n_rows, xq_scratch, stream)
    if rc:
        check(rc)


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
    rc = lib.rein_block_dots(fmt, w, xq, out, in_dim, out_dim, n_rows, int(via_mfma), stream)
    if rc:
        check(rc)


def moe_topk(logits, n_tok, n_expert, n_used, out_ids, out_weights, stream=None):
    rc = lib.rein_moe_topk(logits, n_tok, n_expert, n_used, out_ids, out_weights, stream)
    if rc:
        check(rc)


def moe_sort(ids, n_entries, n_expert, bn, count, cursor, perm, expert_off, tile_off, stream=None):
    rc = lib.rein_moe_sort(ids, n_entries, n_expert, bn, count, cursor, perm,
                           expert_off, tile_off, stream)
    if rc:
        check(rc)


def moe_gather_xq(xq_src, perm, xq_dst, nsub, n_used, n_entries, stream=None):
    rc = lib.rein_moe_gather_xq(xq_src, perm, xq_dst, nsub, n_used, n_entries, stream)
    if rc:
        check(rc)


def moe_quantize_scatter(x, inv, xq_dst, in_dim, n_used, n_tok, stream=None):
    """quantize_q8 + moe_gather_xq in one launch (inv = inverse of the sort's perm)"""
    rc = lib.rein_moe_quantize_scatter(x, inv, xq_dst, in_dim, n_used, n_tok, stream)
    if rc:
        check(rc)


def moe_scatter_rows(src, perm, dst, dim, n_entries, stream=None):
    rc = lib.rein_moe_scatter_rows(src, perm, dst, dim, n_entries, stream)
    if rc:
        check(rc)


def moe_grouped_gemm(fmt, slab, bytes_per_expert, expert_off, tile_off, n_expert, xq, y, in_dim, out_dim,
                     n_entries, stream=None):
    rc = lib.rein_moe_grouped_gemm(fmt, slab, bytes_per_expert, expert_off, tile_off, n_expert,
                                   xq, y, in_dim, out_dim, n_entries, stream)
    if rc:
        check(rc)


def moe_grouped_swiglu_q8(fmt, gate_slab, up_slab, bytes_per_expert, expert_off, tile_off, n_expert, xq, xq_out,
                          in_dim, out_dim, n_entries, stream=None):
    """gate + up grouped GEMM with SwiGLU and the BlockQ8 quantizer in the epilogue"""
    rc = lib.rein_moe_grouped_swiglu_q8(fmt, gate_slab, up_slab, bytes_per_expert, expert_off,
                                        tile_off, n_expert, xq, xq_out, in_dim, out_dim, n_entries,
                                        stream)
    if rc:
        check(rc)


def moe_expert_matvec(fmt, slab, ids, xq, y, in_dim, out_dim, bytes_per_expert, xq_tok_stride, xq_slot_stride,
                      n_used, n_tok=1, stream=None):
    """launch_moe_expert_matvec (src/runtime/qwen35.rs:3071-3100)"""
    rc = lib.rein_moe_expert_matvec(fmt, slab, ids, xq, y, in_dim, out_dim, bytes_per_expert,
                                    xq_tok_stride, xq_slot_stride, n_used, n_tok, stream)
    if rc:
        check(rc)


def moe_down(fmt, slab, ids, xq, y, in_dim, out_dim, bytes_per_expert, xq_tok_stride, xq_slot_stride, n_used,
             n_tok=1, stream=None):
    """launch_moe_down (src/runtime/qwen35.rs:3102-3139)"""
    rc = lib.rein_moe_down(fmt, slab, ids, xq, y, in_dim, out_dim, bytes_per_expert,
                           xq_tok_stride, xq_slot_stride, n_used, n_tok, stream)
    if rc:
        check(rc)


def moe_gate_up_swiglu(fmt, gate_slab, up_slab, ids, xq, y, in_dim, out_dim, bytes_per_expert, xq_tok_stride,
                       xq_slot_stride, n_used, n_tok=1, stream=None):
    """launch_moe_gate_up_swiglu (src/runtime/qwen35.rs:3141-3167)"""
    rc = lib.rein_moe_gate_up_swiglu(fmt, gate_slab, up_slab, ids, xq, y, in_dim, out_dim,
                                     bytes_per_expert, xq_tok_stride, xq_slot_stride, n_used, n_tok, stream)
    if rc:
        check(rc)


def moe_gate_up_swiglu_q8(fmt, gate_slab, up_slab, ids, xq, xq_out, in_dim, out_dim, bytes_per_expert, xq_tok_stride,
                          xq_slot_stride, n_used, n_tok=1, stream=None):
    """moe_gate_up_swiglu followed by quantize_q8 in one launch (BlockQ8 rows of the down projection's input)"""
    rc = lib.rein_moe_gate_up_swiglu_q8(fmt, gate_slab, up_slab, ids, xq, xq_out, in_dim, out_dim,
                                        bytes_per_expert, xq_tok_stride, xq_slot_stride, n_used, n_tok, stream)
    if rc:
        check(rc)


def moe_down_combine(fmt, slab, ids, weights, down_exps_s, xq, out, in_dim, out_dim, bytes_per_expert, xq_tok_stride,
                     xq_slot_stride, n_used, n_tok=1, stream=None):
    """moe_down followed by moe_combine in one launch"""
    rc = lib.rein_moe_down_combine(fmt, slab, ids, weights, down_exps_s, xq, out, in_dim,
                                   out_dim, bytes_per_expert, xq_tok_stride, xq_slot_stride, n_used, n_tok,
                                   stream)
    if rc:
        check(rc)


def swiglu_mul(gate, up, out, n, stream=None):
    rc = lib.rein_swiglu_mul(gate, up, out, n, stream)
    if rc:
        check(rc)


def moe_combine(experts, ids, weights, down_exps_s, out, n_tok, hidden, n_used, stream=None):
    rc = lib.rein_moe_combine(experts, ids, weights, down_exps_s, out, n_tok, hidden,
                              n_used, stream)
    if rc:
        check(rc)


def moe_gemm_bn():
    return lib.rein_moe_gemm_bn()


def moe_shape(n_tok, hidden, n_expert, n_used, expert_ff, gate_up_fmt, down_fmt):
    return MoeShape(n_tok, hidden, n_expert, n_used, expert_ff, gate_up_fmt, down_fmt)


def moe_workspace_bytes(shape):
    return lib.rein_moe_workspace_bytes(C.byref(shape))


def moe_ffn(shape, x, logits, gate_exps, up_exps, down_exps, down_exps_s, workspace, out, stream=None):
    """routed-expert part of step_moe_ffn_batched (src/runtime/qwen35.rs:2788-2870)"""
    rc = lib.rein_moe_ffn(C.byref(shape), x, logits, gate_exps, up_exps, down_exps,
                          down_exps_s, workspace, out, stream)
    if rc:
        check(rc)
