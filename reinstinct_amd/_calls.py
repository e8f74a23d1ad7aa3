"""The launch calls of reinstinct_amd.runtime by ctypes: what csrc/python/native.cpp compiles, for a build without Python's headers.
The same functions, parameters and defaults; a call takes 1-2 us longer."""
import ctypes as C

from ._lib import check, lib

# parameters in the order of the C function; `stream` is a hip.Stream or None
_SIGNATURES = """
quantize_q8(x, xq, in_dim, n_vec=1, stream=None)
rmsnorm_q8(x, w, xq, n, n_vec=1, eps=1e-06, stream=None)
add_rmsnorm_q8(hidden, add, w, y, xq, n, n_vec=1, eps=1e-06, stream=None)
swiglu_q8(gate, up, out, xq, n, stream=None)
sigmoid_mul_q8(x, gate, xq, n, stream=None)
rmsnorm_gated_q8(x, z, w, y, xq, n_heads, head_dim, eps=1e-06, stream=None)
moe_geglu_q8(gu, xq, ff_exp, n_slot, stream=None)
matvec_xq8(fmt, w, xq, y, in_dim, out_dim, stream=None)
matvec_batched_xq8(fmt, w, xq, y, in_dim, out_dim, n_rows, stream=None)
matvec_ondisk_xq8(fmt, w_blocks, xq, y, in_dim, out_dim, stream=None)
matvec_q8_0_splitk(w, xq, y_partials, in_dim, out_dim, n_split, stream=None)
mmq_xq8(fmt, w, xq, y, in_dim, out_dim, p_rows, stream=None)
mmq_xq8_ws(fmt, w, xq, y, in_dim, out_dim, p_rows, workspace, workspace_bytes, stream=None)
mmq_xq8_noalloc(fmt, w, xq, y, in_dim, out_dim, p_rows, stream=None)
matmul(fmt, w, x, y, in_dim, out_dim, n_rows, xq_scratch, stream=None)
matmul_ws(fmt, w, x, y, in_dim, out_dim, n_rows, scratch, scratch_bytes, stream=None)
moe_topk(logits, n_tok, n_expert, n_used, out_ids, out_weights, stream=None)
moe_sort(ids, n_entries, n_expert, bn, count, cursor, perm, expert_off, tile_off, stream=None)
moe_gather_xq(xq_src, perm, xq_dst, nsub, n_used, n_entries, stream=None)
moe_quantize_scatter(x, inv, xq_dst, in_dim, n_used, n_tok, stream=None)
moe_scatter_rows(src, perm, dst, dim, n_entries, stream=None)
moe_grouped_gemm(fmt, slab, bytes_per_expert, expert_off, tile_off, n_expert, xq, y, in_dim, out_dim, n_entries, stream=None)
moe_grouped_swiglu_q8(fmt, gate_slab, up_slab, bytes_per_expert, expert_off, tile_off, n_expert, xq, xq_out, in_dim, out_dim, n_entries, stream=None)
moe_expert_matvec(fmt, slab, ids, xq, y, in_dim, out_dim, bytes_per_expert, xq_tok_stride, xq_slot_stride, n_used, n_tok=1, stream=None)
moe_down(fmt, slab, ids, xq, y, in_dim, out_dim, bytes_per_expert, xq_tok_stride, xq_slot_stride, n_used, n_tok=1, stream=None)
moe_gate_up_swiglu(fmt, gate_slab, up_slab, ids, xq, y, in_dim, out_dim, bytes_per_expert, xq_tok_stride, xq_slot_stride, n_used, n_tok=1, stream=None)
moe_gate_up_swiglu_q8(fmt, gate_slab, up_slab, ids, xq, xq_out, in_dim, out_dim, bytes_per_expert, xq_tok_stride, xq_slot_stride, n_used, n_tok=1, stream=None)
moe_down_combine(fmt, slab, ids, weights, down_exps_s, xq, out, in_dim, out_dim, bytes_per_expert, xq_tok_stride, xq_slot_stride, n_used, n_tok=1, stream=None)
swiglu_mul(gate, up, out, n, stream=None)
moe_combine(experts, ids, weights, down_exps_s, out, n_tok, hidden, n_used, stream=None)
"""


def _s(stream):
    return None if stream is None else stream.raw


for _line in _SIGNATURES.split("\n")[1:-1]:
    _name, _params = _line[:-1].split("(")
    _args = ", ".join(p.split("=")[0] for p in _params.split(", "))
    exec(f"def {_line}:\n    check(lib.rein_{_name}({_args.replace('stream', '_s(stream)')}))")


def matvec_multi_xq8(fmts, ws, ys, out_dims, xq, in_dim, n_rows=1, stream=None):
    n = len(fmts)
    for what, table in (("ws", ws), ("ys", ys), ("out_dims", out_dims)):
        if len(table) != n:
            raise ValueError(f"matvec_multi_xq8: {what} holds {len(table)} elements, fmts {n}")
    pointers = [(C.c_void_p * n)(*[getattr(p, "_as_parameter_", p) for p in table]) for table in (ws, ys)]
    check(lib.rein_matvec_multi_xq8(n, (C.c_int * n)(*fmts), *pointers, (C.c_uint * n)(*out_dims), xq, in_dim, n_rows, _s(stream)))


def moe_ffn(shape, x, logits, gate_exps, up_exps, down_exps, down_exps_s, workspace, out, stream=None):
    check(lib.rein_moe_ffn(C.byref(shape), x, logits, gate_exps, up_exps, down_exps, down_exps_s, workspace, out, _s(stream)))
