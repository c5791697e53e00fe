"""The C-ABI library loads without a GPU, exports every symbol include/distca_ca.h declares,
and rejects bad arguments on the host before anything is launched."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

from distca_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "distca_ca.h")


def _declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    text = re.sub(r"//[^\n]*", "", text)
    return sorted(set(re.findall(r"\b(distca_[a-z0-9_]+)\s*\(", text)))


def test_header_compiles_as_plain_c(tmp_path):
    src = tmp_path / "t.c"
    src.write_text('#include "distca_ca.h"\nint main(void) { distca_ca_params p; (void)p; return 0; }\n')
    subprocess.run(["gcc", "-std=c99", "-Wall", "-Werror", "-I", os.path.join(ROOT, "include"), "-c", str(src),
                    "-o", str(tmp_path / "t.o")], check=True)


def test_every_declared_symbol_is_exported_and_bound():
    names = _declared_functions()
    assert len(names) >= 12
    lib = ctypes.CDLL(_lib.LIB_PATH)
    for n in names:
        assert hasattr(lib, n), f"{n} declared in distca_ca.h but not exported"
    assert set(names) == set(_lib.SYMBOLS), "ctypes table and header disagree"


def test_params_struct_layout_matches_header():
    text = open(HEADER).read()
    body = re.search(r"typedef struct distca_ca_params \{(.*?)\} distca_ca_params;", text, re.S).group(1)
    body = re.sub(r"/\*.*?\*/", "", body, flags=re.S)
    body = re.sub(r"//[^\n]*", "", body)
    fields = re.findall(r"(int32_t|float)\s+([a-z_]+)\s*;", body)
    assert [f for _, f in fields] == [f for f, _ in _lib.CaParams._fields_]
    assert ctypes.sizeof(_lib.CaParams) == 4 * len(fields)


def test_abi_version_and_error_string():
    lib = _lib.load()
    assert lib.distca_abi_version() == _lib.ABI_VERSION
    assert isinstance(lib.distca_last_error(), bytes)


def _p(**kw):
    base = dict(num_tasks=1, total_q=16, total_k=16, num_heads_q=32, num_heads_kv=8, head_dim=128,
                max_seqlen_q=16, max_seqlen_k=16, softmax_scale=0.088, causal=1, deterministic=0, dtype=0)
    base.update(kw)
    return _lib.CaParams(*[base[f] for f, _ in _lib.CaParams._fields_])


@pytest.mark.parametrize("bad", [dict(head_dim=64), dict(num_heads_q=30), dict(num_heads_kv=0), dict(num_tasks=-1),
                                 dict(total_q=-5), dict(dtype=3), dict(dtype=-1)])
def test_unsupported_shapes_are_rejected_on_the_host(bad):
    lib = _lib.load()
    p = _p(**bad)
    assert lib.distca_ca_fwd_workspace_bytes(ctypes.byref(p)) < 0
    # validation precedes any device call: with null pointers the call must return an error code
    rc = lib.distca_ca_fwd(None, None, None, None, None, None, None, None, ctypes.byref(p), None, 0, None)
    assert rc in (-1, -2)
    assert lib.distca_last_error()


def test_workspace_sizes_are_positive_and_monotone():
    lib = _lib.load()
    # element type: 0 (callers from before the field existed) and DISTCA_DTYPE_BF16 = 2 mean bf16, 1 is fp16; same sizes
    sizes = {lib.distca_ca_bwd_workspace_bytes(ctypes.byref(_p(dtype=t))) for t in (0, 1, 2)}
    assert len(sizes) == 1 and min(sizes) > 0
    small = lib.distca_ca_bwd_workspace_bytes(ctypes.byref(_p()))
    big = lib.distca_ca_bwd_workspace_bytes(ctypes.byref(_p(total_q=131072, total_k=131072, num_tasks=27,
                                                              max_seqlen_q=65536, max_seqlen_k=65536)))
    assert 0 < small < big
    assert lib.distca_ca_fwd_workspace_bytes(ctypes.byref(_p())) > 0


def test_pack_argument_checks_need_no_gpu():
    lib = _lib.load()
    # token size not a multiple of 16 bytes: rejected as the reference rejects it (memcpy.cu:246)
    dummy = ctypes.create_string_buffer(64)        # host memory, never dereferenced: the size check comes first
    a = ctypes.addressof(dummy)
    assert lib.distca_memcpy_non_cp(a, a, a, a, None, 1, 24, 8, 1, None) < 0
    assert b"16" in lib.distca_last_error()
    assert lib.distca_memcpy_cp(a, a, a, a, a, 24, 8, 2, 1, 1, None) < 0
    assert b"16" in lib.distca_last_error()
    assert lib.distca_memcpy_non_cp(None, None, None, None, None, 1, 32, 8, 1, None) < 0
    assert b"null" in lib.distca_last_error()
    assert lib.distca_grad_sum(None, 99, None, None, None, 8, 128, 1, 1, None) < 0   # unknown dtype code
    # zero-sized problems are no-ops that never touch the device
    assert lib.distca_memcpy_non_cp(None, None, None, None, None, 0, 32, 0, 1, None) == 0


def test_timing_api_without_launches():
    lib = _lib.load()
    ms, n = ctypes.c_double(-1), ctypes.c_int64(-1)
    assert lib.distca_timing_read(99, ctypes.byref(ms), ctypes.byref(n)) < 0
    lib.distca_timing_enable(0)
    assert lib.distca_timing_read(0, ctypes.byref(ms), ctypes.byref(n)) == 0 and n.value == 0


def test_schedule_host_reports_needed_capacity():
    lib = _lib.load()
    cu = np.array([0, 1000], dtype=np.int32)
    p = _p(total_q=1000, total_k=1000, max_seqlen_q=1000, max_seqlen_k=1000)
    n = lib.distca_ca_schedule_host(0, cu.ctypes.data, cu.ctypes.data, ctypes.byref(p), None, 0)
    assert n > 0
    small = np.full((2, 4), -7, dtype=np.int32)
    # a short array receives the first max_items items; the full count is still returned
    assert lib.distca_ca_schedule_host(0, cu.ctypes.data, cu.ctypes.data, ctypes.byref(p), small.ctypes.data, 1) == n
    assert small[0, 0] == 0 and (small[1] == -7).all()


def test_attention_argument_errors_are_reported_before_any_launch():
    """Null, misaligned and undersized arguments come back as error codes with a message; the
    pointers are fake host addresses, so reaching a kernel launch would fail differently."""
    lib = _lib.load()
    buf = ctypes.create_string_buffer(4096)
    base = (ctypes.addressof(buf) + 255) // 256 * 256
    ptr = ctypes.c_void_p(base)
    odd = ctypes.c_void_p(base + 2)
    p = _p()
    need = lib.distca_ca_fwd_workspace_bytes(ctypes.byref(p))
    args = lambda **kw: [kw.get("q", ptr), ptr, ptr, ptr, ptr, ptr, ptr, None, ctypes.byref(p), kw.get("ws", ptr), kw.get("ws_bytes", need), None]
    assert lib.distca_ca_fwd(*args(ws_bytes=need - 1)) == -3
    assert b"workspace" in lib.distca_last_error()
    assert lib.distca_ca_fwd(*args(ws=None)) == -3
    assert lib.distca_ca_fwd(*args(q=odd)) == -1
    assert b"aligned" in lib.distca_last_error()
    assert lib.distca_ca_fwd(*args(q=None)) == -1
    # backward: deterministic together with shared KV rows is served (one work item owns a key block on behalf of every
    # task that reads it), so the call passes validation up to the workspace check, like the form without kv_task_offsets
    pd = _p(deterministic=1)
    needb = lib.distca_ca_bwd_workspace_bytes(ctypes.byref(pd))
    bargs = [ptr] * 9 + [ptr, ptr, ptr, ctypes.byref(pd), ptr, 64, None]
    assert lib.distca_ca_bwd(*bargs) == -3
    assert b"workspace" in lib.distca_last_error()
    bargs[11] = None
    assert lib.distca_ca_bwd(*bargs) == -3
    bargs[14] = needb
    bargs[0] = odd
    assert lib.distca_ca_bwd(*bargs) == -1
    assert b"aligned" in lib.distca_last_error()
    # a batch without tasks or rows is a no-op that touches nothing
    assert lib.distca_ca_fwd(None, None, None, None, None, None, None, None, ctypes.byref(_p(num_tasks=0, total_q=0, total_k=0)), None, 0, None) == 0


def test_backward_workspace_is_sized_for_what_the_call_needs():
    """The work lists and the two row statistics, and nothing else, for a batch large enough to occupy the device or a
    deterministic one: 131072 tokens with 32 query heads need 34 MB.  Only a small batch with deterministic == 0 also
    brings room for a few pieces of key blocks: 8 bytes per stored element of K."""
    lib = _lib.load()
    big = _p(num_tasks=27, total_q=131072, total_k=131072, num_heads_q=32, num_heads_kv=8, max_seqlen_q=65536, max_seqlen_k=65536)
    n = lib.distca_ca_bwd_workspace_bytes(ctypes.byref(big))
    stats = 2 * 32 * 131072 * 4
    assert stats < n <= 40e6
    big.deterministic = 1
    assert lib.distca_ca_bwd_workspace_bytes(ctypes.byref(big)) == n
    cfg5 = _p(num_tasks=40, total_q=524288, total_k=524288, num_heads_q=64, num_heads_kv=8, max_seqlen_q=262144, max_seqlen_k=262144)
    assert lib.distca_ca_bwd_workspace_bytes(ctypes.byref(cfg5)) <= 2 * 64 * 524288 * 4 + 8e6
    small = _p(num_tasks=3, total_q=4096, total_k=4096, num_heads_q=32, num_heads_kv=8, max_seqlen_q=2560, max_seqlen_k=2560)
    pieces = lib.distca_ca_bwd_workspace_bytes(ctypes.byref(small))
    small.deterministic = 1
    whole = lib.distca_ca_bwd_workspace_bytes(ctypes.byref(small))
    assert pieces - whole >= 2 * 4096 * 8 * 128 * 4          # 8 bytes per element
    assert whole < 2 * 32 * 4096 * 4 + 1e6


@pytest.mark.parametrize("deterministic", [0, 1])
def test_smallest_workspace_stays_what_fixed_buffers_were_sized_for(deterministic):
    """Over sizes of every magnitude: lists (16 bytes an item, a few words a task), 8 bytes per query row and head, and with
    deterministic == 0 at most 8 bytes per stored element of K.  A batch of 4096 tokens: 8.7 MB at 8/2 heads, 34.6 at 32/8, 4.3 at 4/1.
    The preferred size is never less, and beyond that at most 1024 slots (130 KB forward, 256 KB backward) with their tables."""
    lib = _lib.load()
    rng = np.random.default_rng(deterministic)
    for _ in range(5000):
        hq, hkv = [(4, 1), (8, 2), (32, 8), (64, 8), (8, 8), (128, 8), (16, 16), (1, 1), (6, 2), (256, 256)][rng.integers(10)]
        n, tq, tk, mq, mk = (int(2 ** rng.uniform(0, top)) for top in (8, 20, 20, 18, 18))
        p = _p(num_tasks=n, total_q=tq, total_k=tk, num_heads_q=hq, num_heads_kv=hkv, max_seqlen_q=mq, max_seqlen_k=mk, deterministic=deterministic)
        fwd, bwd, fwd_more, bwd_more = (int(getattr(lib, f"distca_ca_{d}_workspace_{s}bytes")(ctypes.byref(p))) for s in ("", "preferred_") for d in ("fwd", "bwd"))
        rows = tq * (hq // hkv) // 256 + n + 1
        keys = max(tk // 256 + n + 1, (mk // 256 + 1) * n + 1) if not deterministic and (tk // 256 + n + 1) * hkv < 512 else tk // 256 + n + 1
        per_task, fixed = 8 * 4, 4096
        assert 0 < fwd <= 16 * rows + per_task * n + fixed
        more = 8 * tk * hkv * 128 + 16 * 512 if not deterministic and (tk // 256 + n + 1) * hkv < 512 else 0
        assert 0 < bwd <= 16 * (rows + keys) + 2 * (per_task + 32) * n + 8 * hq * tq + more + 2 * fixed
        tables = 64 * (rows + keys + 512) + 2 * fixed
        assert fwd <= fwd_more <= fwd + 1024 * (256 * 128 * 4 + 256 * 8) + tables
        assert bwd <= bwd_more <= bwd + 1024 * 2 * 256 * 128 * 4 + tables
    for hq, hkv, mb in ((8, 2, 8.7), (32, 8, 34.6), (4, 1, 4.3)):
        p = _p(num_tasks=3, total_q=4096, total_k=4096, num_heads_q=hq, num_heads_kv=hkv, max_seqlen_q=2560, max_seqlen_k=2560)
        assert int(lib.distca_ca_bwd_workspace_bytes(ctypes.byref(p))) <= mb * 1e6 + 1e5


def test_preferred_sizes_that_the_header_names():
    """The sizes quoted for one document of 4096 tokens are those that the functions return."""
    lib = _lib.load()
    text = re.sub(r"\s*\n \* ", " ", open(HEADER).read())
    quoted = re.search(r"one document of 4096 tokens: (\d+) and (\d+) MB at 4/1 heads, (\d+) and (\d+) MB at 32/8", text)
    sizes = []
    for hq, hkv in ((4, 1), (32, 8)):
        p = _p(total_q=4096, total_k=4096, num_heads_q=hq, num_heads_kv=hkv, max_seqlen_q=4096, max_seqlen_k=4096)
        sizes += [int(getattr(lib, f"distca_ca_{d}_workspace_preferred_bytes")(ctypes.byref(p))) for d in ("fwd", "bwd")]
    assert [int(mb) for mb in quoted.groups()] == [round(b / 1e6) for b in sizes]


def test_python_wrappers_reject_wrong_inputs():
    """The host layer raises RuntimeError for what the reference's C++ wrappers check
    (all_to_all.cpp:18-21, 47-99): device, rank, dtype of metadata."""
    import torch
    from distca_amd import ops
    from distca_amd.fused_comm_attn import ca_varlen_fwd
    t = torch.zeros((4, 8), dtype=torch.bfloat16)
    off = torch.zeros(1, dtype=torch.int64)
    with pytest.raises(AssertionError, match="DispatcherWrapper not initialized"):   # ops.py:112-115 of the reference
        ops.a2a_memcpy_non_cp(t, off, off, True)
    with pytest.raises(NotImplementedError):
        ops.DispatcherWrapper.init(0, 0, 2, 1024, device="cpu")
    ops.DispatcherWrapper.init(0, 0, 1, 1024, device="cpu")
    try:
        with pytest.raises(AssertionError, match="no all-to-all has filled"):
            ops.a2a_memcpy_non_cp(t, off, off, False, instance_id=0)
        ops.DispatcherWrapper.acquire(0)
        with pytest.raises(AssertionError, match="not released"):
            ops.a2a_memcpy_non_cp(t, off, off, True, instance_id=0)
        ops.DispatcherWrapper.release(0)
        ops.DispatcherWrapper.get_instance(0).send_buffer[:8] = torch.arange(8, dtype=torch.uint8)
        one = torch.ones((1, 1), dtype=torch.int64)
        ops.fast_a2a(one, one, one, one, 0, 16, 8, instance_id=0)
        assert ops.DispatcherWrapper.is_acquired[0]
        assert ops.DispatcherWrapper.get_instance(0).recv_buffer[16:24].tolist() == list(range(8))
        with pytest.raises(RuntimeError, match="do not fit"):
            ops.fast_a2a(one, one, one, one, 0, 1020, 8)
        assert ops.DispatcherWrapper.get_instance() is ops.DispatcherWrapper.instance[0]
        ops.DispatcherWrapper.switch_buffer()
        assert ops.DispatcherWrapper.get_instance() is ops.DispatcherWrapper.instance[1]
    finally:
        ops.DispatcherWrapper.instance = None
        ops.DispatcherWrapper.is_acquired = [False, False]
        ops.DispatcherWrapper.cur_instance = 0
    with pytest.raises(RuntimeError):
        ops.a2a_memcpy_non_cp(t, off.to(torch.int32), off, True, buffer=torch.zeros(64, dtype=torch.uint8))
    with pytest.raises(RuntimeError):
        ops.pre_a2a_grad_acc(t.to(torch.float64), off.to(torch.int32), off.reshape(1, 1), off)
    q = torch.zeros((4, 2, 128), dtype=torch.bfloat16)
    cu = torch.tensor([0, 4], dtype=torch.int32)
    with pytest.raises(RuntimeError, match="CUDA"):
        ca_varlen_fwd(q, q, q, cu, cu, 4, 4)


def test_token_layout_entry_points_check_their_layouts():
    """distca_ca_fwd_tokens / distca_ca_bwd_tokens refuse token sizes that cannot hold their parts, a
    missing lse destination, and (backward) head counts that put q off 16-byte alignment; all before
    any launch."""
    lib = _lib.load()
    ptr = ctypes.c_void_p(0x1000)
    p = _lib.CaParams(2, 64, 64, 8, 2, 128, 32, 32, 0.088, 1, 0, 0)
    need = lib.distca_ca_fwd_workspace_bytes(ctypes.byref(p))
    row = 8 * 128 * 2
    fwd = lambda **kw: lib.distca_ca_fwd_tokens(*[kw.get(n, d) for n, d in (
        ("q", ptr), ("q_off", ptr), ("q_tok", row), ("k", ptr), ("v", ptr), ("out", ptr), ("out_off", ptr), ("out_tok", row + 32),
        ("lse", None), ("cu_q", ptr), ("cu_k", ptr), ("kv_off", None), ("p", ctypes.byref(p)), ("ws", ptr), ("ws_bytes", 16), ("stream", None))])
    assert fwd() == -3 and b"workspace" in lib.distca_last_error()          # everything else is in order
    assert fwd(q_tok=row - 16) == -1 and b"query token" in lib.distca_last_error()
    assert fwd(out_tok=row) == -1 and b"output token" in lib.distca_last_error()   # no room for the lse
    assert fwd(out_tok=row + 8) == -1
    assert fwd(out_off=None, out_tok=0) == -1 and b"lse is null" in lib.distca_last_error()
    assert fwd(q=None) == -1
    assert need > 16
    needb = lib.distca_ca_bwd_workspace_bytes(ctypes.byref(p))
    bwd = lambda **kw: lib.distca_ca_bwd_tokens(*[kw.get(n, d) for n, d in (
        ("req", ptr), ("req_off", ptr), ("req_tok", 3 * row + 32), ("k", ptr), ("v", ptr), ("dq", ptr), ("dq_off", ptr), ("dq_tok", row),
        ("dk", ptr), ("dv", ptr), ("cu_q", ptr), ("cu_k", ptr), ("kv_off", None), ("p", ctypes.byref(kw.get("params", p))), ("ws", ptr),
        ("ws_bytes", 64), ("stream", None))])
    assert bwd() == -3 and needb > 64
    assert bwd(req_tok=3 * row) == -1 and b"request token" in lib.distca_last_error()
    assert bwd(dq_tok=row - 16) == -1 and b"dq token" in lib.distca_last_error()
    assert bwd(req_off=None) == -1 and b"offset" in lib.distca_last_error()
    p6 = _lib.CaParams(2, 64, 64, 6, 2, 128, 32, 32, 0.088, 1, 0, 0)
    assert bwd(params=p6) == -2 and b"alignment" in lib.distca_last_error()
    # a server without a task this tick: empty (null) arrays everywhere, nothing to do, no error
    idle = _lib.CaParams(0, 0, 0, 8, 2, 128, 0, 0, 0.088, 1, 0, 0)
    nothing = dict(req=None, req_off=None, k=None, v=None, dq=None, dq_off=None, dk=None, dv=None, cu_q=None, cu_k=None, ws=None, ws_bytes=0)
    assert bwd(params=idle, **nothing) == 0
    p_save = p
    p = idle
    assert fwd(q=None, q_off=None, k=None, v=None, out=None, out_off=None, cu_q=None, cu_k=None, ws=None, ws_bytes=0) == 0
    p = p_save


def test_torch_ops_are_registered_for_device_tensors_only():
    """`torch.ops.distca_amd.*` carry the reference's op names and schemas
    (csrc/bindings/all_to_all.cpp:102-113,182-254) and have no host implementation."""
    import torch
    from distca_amd import torch_ops
    for name, schema in torch_ops.SCHEMAS.items():
        op = getattr(torch.ops.distca_amd, name)
        got = str(op.default._schema)
        assert got == f"distca_amd::{name}{schema}", got
    t = torch.zeros((4, 8), dtype=torch.bfloat16)
    i64 = torch.zeros(1, dtype=torch.int64)
    with pytest.raises(NotImplementedError):
        torch.ops.distca_amd.fast_a2a_memcpy_non_cp_debug(t, i64, i64, None, True, torch.zeros(64, dtype=torch.uint8))
    with pytest.raises(NotImplementedError):
        torch.ops.distca_amd.fast_a2a_grad_acc(t, torch.zeros(1, dtype=torch.int32), torch.zeros((1, 1), dtype=torch.int64), i64)


def test_parts_of_a_request_token_are_rows_the_launch_can_read():
    """What goes into a request as it is has a pitch of whole vectors, at least a row long, and a 16-byte aligned start (the launch
    refuses anything else); every other form a caller may bring is copied, the gradient of a sum over tokens (a pitch of 0) among them."""
    import torch
    from distca_amd.ops import token_part
    T, h = 5, 32
    base = torch.arange(2 * T * h + 64, dtype=torch.float32).to(torch.bfloat16)
    rows = base[:T * h].view(T, h)
    assert token_part(rows) is rows
    wide = base[:2 * T * h].view(T, 2 * h)[:, h:]
    assert token_part(wide) is wide
    forms = [rows[:1].expand(T, h), rows[:, :1].expand(T, h), base[:h * T].view(h, T).t(), base.as_strided((T, h), (8, 1)), base.as_strided((T, h), (h + 1, 1)),
             base[1:1 + T * h].view(T, h), base.as_strided((T, h), (2 * h, 2)), rows[:1].expand(T, h)[:1], rows[:0]]
    for t in forms:
        p = token_part(t)
        assert torch.equal(p, t) and p.stride(1) == 1 and p.data_ptr() % 16 == 0
        assert p.size(0) <= 1 or (p.stride(0) >= h and p.stride(0) * 2 % 16 == 0)


def test_request_parts_that_are_no_matrices_are_named():
    """A part of a backward request that is no [tokens, hidden] matrix is an AssertionError that says so, whichever way the token goes."""
    import torch
    from distca_amd.dispatch import pre_a2a_attn_out_grad_resend_qkv, send_attn_out_grad_resend_qkv
    t, lse, none = torch.zeros((3, 64), dtype=torch.bfloat16), torch.zeros((3, 16), dtype=torch.uint8), [None] * 8
    for bad in (lse.reshape(-1), lse[:2], lse[:, None]):
        for send in (pre_a2a_attn_out_grad_resend_qkv, send_attn_out_grad_resend_qkv):
            with pytest.raises(AssertionError, match="every part must be"):
                send(t, t, bad, t, *none)


def test_exchange_steps_take_a_length_for_every_shard_they_place():
    """The gradients' way out and the request's way in refuse lengths that are not one per shard placed, as the launch of several
    tensors did."""
    import torch
    from distca_amd.dispatch import post_a2a_attn_out_grad_resend_qkv, pre_a2a_qkv
    t, off, long = torch.zeros((4, 8), dtype=torch.bfloat16), torch.zeros(2, dtype=torch.int64), torch.tensor([2, 2, 0])
    right, mask, buf = long[:2], torch.ones(2, dtype=torch.int8), torch.zeros(64, dtype=torch.uint8)
    for q_lens, k_lens in ((long, right), (right, long), (right[:1], right), (right, right[:, None])):
        with pytest.raises(RuntimeError, match="seq_tokens must be of shape"):
            pre_a2a_qkv(t, t, t, None, q_lens, k_lens, off, off, off, is_fwd=False, kv_grad_copy_shard_mask=mask, buffer=buf)
        with pytest.raises(RuntimeError, match="seq_tokens must be of shape"):
            post_a2a_attn_out_grad_resend_qkv([4, 8], [4, 4], [4, 8], torch.float32, t, t, None, q_lens, k_lens, off, off, off, False, buffer=buf)


@pytest.mark.parametrize("parts", ["generator", "dict", "tensor", "number", "set", "none"])
def test_parts_of_a_job_are_a_list_or_a_tuple(parts):
    """Anything else that a caller may take for a sequence of tensors is a TypeError, whatever lies in its memory."""
    import torch
    from distca_amd.ops import exchange, plain_job
    t, lens = torch.zeros((2, 8), dtype=torch.bfloat16), torch.tensor([2])
    given = dict(generator=(x for x in [t]), dict={0: t}, tensor=t, number=3, set={1}, none=None)[parts]
    with pytest.raises(TypeError, match="list or a tuple"):
        exchange([plain_job(given, torch.zeros(1, dtype=torch.int64), lens)], torch.zeros(64, dtype=torch.uint8), True)


def test_the_package_names_nothing_private_of_torch():
    """No underscored attribute of torch's modules in the package's Python files: they come and go between releases."""
    import pathlib
    for f in pathlib.Path(ROOT, "distca_amd").rglob("*.py"):
        assert not re.findall(r"\btorch(?:\.\w+)*\._\w+", f.read_text()), f


def test_numbers_of_an_attention_call_are_what_int_and_float_take():
    """Sequence lengths and the scale in any form int() and float() take, truncated as int() does; anything else is a TypeError or ValueError."""
    import torch
    from distca_amd.fused_comm_attn import ca_varlen_fwd
    q = torch.zeros((4, 2, 128), dtype=torch.bfloat16)
    cu = torch.tensor([0, 4], dtype=torch.int32)
    for n, scale in ((4, None), (4.7, 0.1), ("4", "0.1"), (np.int64(4), np.float32(0.1)), (torch.tensor(4), torch.tensor(0.1)), (True, 1)):
        with pytest.raises(RuntimeError, match="CUDA"):   # (the first thing that is wrong here)
            ca_varlen_fwd(q, q, q, cu, cu, n, n, scale)
    for n, scale in ((None, 0.1), (4, [0.1]), ("x", 0.1), (4, "x"), (float("nan"), 0.1)):
        with pytest.raises((TypeError, ValueError)):
            ca_varlen_fwd(q, q, q, cu, cu, n, n, scale)
