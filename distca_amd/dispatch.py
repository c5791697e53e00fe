"""The pack / unpack steps on either side of the all-to-all, by their reference names.

Call surface (names, positional order, returned tuples) and byte layouts follow
distca/runtime/attn_kernels/dispatch.py:13-221.  The transport buffer is either handed over as
`buffer=` (a uint8 device tensor) or, as in the reference, found through the `DispatcherWrapper`:
then `instance_id` / `dispatcher_id` select the instance (None: the current one), and the unpacking
steps switch the current instance and release the receive buffer the way the reference's do.

How the steps are carried out is this library's own: the q, k and v of a step go through one launch (`ops.exchange`) where the
reference makes three and more, and the parts of a composite transport token ([out | lse | pad], [dO | O | lse | q | pad])
are copied straight between their own tensors and the buffer where their rows are whole 16-byte vectors and the token holds at most
512 KiB.  Where not, or where the caller gets the token matrix itself, a `TokenLayout` writes every part into its byte range of one
preallocated matrix, instead of concatenating and then padding.
"""
from __future__ import annotations

from typing import List, Sequence, Tuple

import torch
from torch import Tensor

from . import _lib
from .ops import (TOKEN_OF_PARTS_MAX_BYTES, DispatcherWrapper, _transport_buffer, a2a_memcpy_cp, a2a_memcpy_non_cp, a2a_memcpy_non_cp_multi,
                  copy_sum_job, exchange, plain_job, pre_a2a_grad_acc, replicas_job, token_part, whole_vectors)
from .utils import round_up


class TokenLayout:
    """Byte layout of a transport token that carries several per-token rows side by side, rounded up to
    a whole number of 128-bit vectors with zero bytes (dispatch.py:129-135 of the reference builds the
    same bytes with a concat followed by a pad)."""

    def __init__(self, parts: Sequence[Tuple[int, torch.dtype]]):
        self.dtypes = [dt for _, dt in parts]
        self.sizes = [n * dt.itemsize for n, dt in parts]
        self.starts = [sum(self.sizes[:i]) for i in range(len(parts))]
        self.payload = sum(self.sizes)
        self.token_bytes = round_up(self.payload)

    @property
    def in_parts(self) -> bool:
        """Whether one launch can copy the parts straight between their tensors and the buffer."""
        return whole_vectors(*self.sizes) and self.token_bytes <= TOKEN_OF_PARTS_MAX_BYTES

    @classmethod
    def of(cls, tensors: Sequence[Tensor]) -> "TokenLayout":
        return cls([(t.shape[1], t.dtype) for t in tensors])

    def merge(self, tensors: Sequence[Tensor]) -> Tensor:
        """[T, token_bytes] uint8 with part i of every token at bytes starts[i].."""
        rows = tensors[0].shape[0]
        out = torch.empty((rows, self.token_bytes), dtype=torch.uint8, device=tensors[0].device)
        for t, a, n in zip(tensors, self.starts, self.sizes):
            if t.shape[0] != rows:
                raise RuntimeError(f"token parts disagree on the token count: {t.shape[0]} against {rows}")
            out[:, a:a + n] = t.contiguous().view(torch.uint8).view(rows, n)
        if self.token_bytes > self.payload:
            out[:, self.payload:] = 0
        return out

    def split(self, merged: Tensor) -> List[Tensor]:
        """The parts of `merged` [T, token_bytes] as contiguous tensors of their own dtypes."""
        return [merged[:, a:a + n].contiguous().view(dt) for a, n, dt in zip(self.starts, self.sizes, self.dtypes)]


def _unpacked(buffer, switch_buffer: bool, instance_id) -> None:
    """What the reference does once a receive buffer has been read (dispatch.py:90-93, 119-122): the next
    call without an instance id finds the other instance, and a named instance is released for the next
    all-to-all.  An explicit buffer belongs to the caller and has neither."""
    if buffer is not None:
        return
    if switch_buffer:
        DispatcherWrapper.switch_buffer()
    if instance_id is not None:
        DispatcherWrapper.release(instance_id)


def _lengths_of(tokens: Tensor, offset: Tensor) -> Tensor:
    """The lengths of exactly the shards `offset` places (a plain job alone takes longer arrays, as a2a_memcpy_non_cp does)."""
    if tokens.shape != offset.shape:
        raise RuntimeError("seq_tokens must be of shape (num_sequence,)")
    return tokens


def pre_a2a_qkv(
    q: Tensor, k: Tensor, v: Tensor, kv_dispatch_mask: Tensor,
    q_seq_tokens: Tensor, k_seq_tokens: Tensor,
    q_send_buffer_offset: Tensor, k_send_buffer_offset: Tensor, v_send_buffer_offset: Tensor,
    is_fwd: bool, instance_id: int = None,
    kv_grad_copy_shard_mask: Tensor = None,
    pre_a2a_grad_acc_args=None, *, buffer: Tensor = None,
):
    """Sender side.  Forward (dispatch.py:30-38): q shards as they are, every k / v shard once per destination
    that needs it.  Backward (:39-56): the gradients of duplicate k / v copies are first summed into their main
    copy, then q and only the main copies go out."""
    buffer = _transport_buffer(buffer, instance_id, True)
    if is_fwd:
        return _lib.host().pack_qkv(q, k, v, kv_dispatch_mask, q_seq_tokens, k_seq_tokens, q_send_buffer_offset, k_send_buffer_offset,
                                    v_send_buffer_offset, buffer)
    q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    if kv_grad_copy_shard_mask is None:
        raise AssertionError("kv grad copy requires a dedup mask.")
    jobs = [plain_job([q], q_send_buffer_offset, _lengths_of(q_seq_tokens, q_send_buffer_offset))]
    for t, off in ((k, k_send_buffer_offset), (v, v_send_buffer_offset)):
        _lengths_of(k_seq_tokens, off)
        if pre_a2a_grad_acc_args is None:
            jobs.append(plain_job([t], off, k_seq_tokens, kv_grad_copy_shard_mask))
        else:
            num_copies, copy_start_id, lens = pre_a2a_grad_acc_args
            if lens.data_ptr() == k_seq_tokens.data_ptr() and lens.shape == k_seq_tokens.shape and lens.stride() == k_seq_tokens.stride():
                jobs.append(copy_sum_job(t, off, k_seq_tokens, kv_grad_copy_shard_mask, num_copies, copy_start_id))
            else:   # the shards that are summed are not those that are sent
                pre_a2a_grad_acc(t, num_copies, copy_start_id, lens)
                jobs.append(plain_job([t], off, k_seq_tokens, kv_grad_copy_shard_mask))
    exchange(jobs, buffer, True)
    return q, k, v


def post_a2a_qkv(
    recv_q: Tensor, recv_k: Tensor, recv_v: Tensor, kv_dispatch_mask: Tensor,
    q_recv_seq_tokens: Tensor, k_recv_seq_tokens: Tensor,
    q_recv_buffer_offset: Tensor, k_recv_buffer_offset: Tensor, v_recv_buffer_offset: Tensor,
    is_fwd: bool, switch_buffer: bool = True, instance_id: int = None, *, buffer: Tensor = None,
):
    """Receiver side (dispatch.py:60-94).  Forward: three plain unpacks (a k / v shard that several tasks need
    arrives once and is copied out once per task, the entries' offsets being equal).  Backward: k / v gradients
    land in replica planes [max_cp, T, hidden] for the caller to sum."""
    if is_fwd:
        a2a_memcpy_non_cp_multi(
            [recv_q, recv_k, recv_v], [q_recv_buffer_offset, k_recv_buffer_offset, v_recv_buffer_offset],
            [q_recv_seq_tokens, k_recv_seq_tokens, k_recv_seq_tokens], False, buffer=buffer, instance_id=instance_id)
    else:
        a2a_memcpy_non_cp(recv_q, q_recv_buffer_offset, q_recv_seq_tokens, False, buffer=buffer, instance_id=instance_id)
        for t, off in ((recv_k, k_recv_buffer_offset), (recv_v, v_recv_buffer_offset)):
            a2a_memcpy_cp(t, kv_dispatch_mask, off, k_recv_seq_tokens, False, buffer=buffer, instance_id=instance_id)
    _unpacked(buffer, switch_buffer, instance_id)
    return recv_q, recv_k, recv_v


def pre_a2a_attn_out(q: Tensor, q_seq_tokens: Tensor, q_send_buffer_offset: Tensor,
                     instance_id: int = None, *, buffer: Tensor = None):
    """Packs the attention output shards (dispatch.py:97-106)."""
    q = q.contiguous()
    a2a_memcpy_non_cp(q, q_send_buffer_offset, q_seq_tokens, True, buffer=buffer, instance_id=instance_id)
    return q


def post_a2a_attn_out(recv_q: Tensor, q_recv_seq_tokens: Tensor, q_recv_buffer_offset: Tensor,
                      switch_buffer: bool = True, instance_id: int = None, *, buffer: Tensor = None):
    """Unpacks the attention output shards (dispatch.py:109-126)."""
    a2a_memcpy_non_cp(recv_q, q_recv_buffer_offset, q_recv_seq_tokens, False, buffer=buffer, instance_id=instance_id)
    _unpacked(buffer, switch_buffer, instance_id)
    return recv_q


def _concat_with_uint8_and_pad(tensors: List[Tensor], dim: int):
    """The reference's helper (dispatch.py:129-135), kept by name: tokens of `tensors` side by side as bytes,
    zero-padded to a multiple of 16."""
    if dim not in (1, -1) or any(t.dim() != 2 for t in tensors):
        raise RuntimeError("token parts are [tokens, hidden] matrices joined along the hidden dimension")
    return TokenLayout.of(tensors).merge(tensors)


def _same_tokens(what: str, *tensors: Tensor) -> int:
    rows = tensors[0].shape[0]
    for t in tensors:
        if t.dim() != 2 or t.shape[0] != rows:
            raise AssertionError(f"{what}: every part must be [tokens, hidden] with {rows} tokens, got {tuple(t.shape)}")
    return rows


def pre_a2a_attn_out_grad_resend_qkv(
    attn_out_grad: Tensor, attn_out: Tensor, lse_norm: Tensor,
    q: Tensor, k: Tensor, v: Tensor, kv_dispatch_mask: Tensor,
    q_seq_tokens: Tensor, k_seq_tokens: Tensor,
    q_send_buffer_offset: Tensor, k_send_buffer_offset: Tensor, v_send_buffer_offset: Tensor,
    instance_id: int = None, *, buffer: Tensor = None,
):
    """Backward request of the linear side (dispatch.py:138-158): every query token travels as
    [dO | O | lse | q | pad], k and v as in the forward."""
    _same_tokens("backward request", attn_out_grad, attn_out, lse_norm, q)
    if q.dtype != attn_out.dtype or attn_out_grad.shape != attn_out.shape:
        raise AssertionError("dO, O and q of a backward request share one dtype, and dO has the shape of O")
    request = TokenLayout.of([attn_out_grad, attn_out, lse_norm, q]).merge([attn_out_grad, attn_out, lse_norm, q])
    return pre_a2a_qkv(request, k, v, kv_dispatch_mask, q_seq_tokens, k_seq_tokens,
                       q_send_buffer_offset, k_send_buffer_offset, v_send_buffer_offset,
                       is_fwd=True, buffer=buffer, instance_id=instance_id)


def send_attn_out_grad_resend_qkv(attn_out_grad: Tensor, attn_out: Tensor, lse_norm: Tensor, q: Tensor, k: Tensor, v: Tensor,
                                  kv_dispatch_mask: Tensor, q_seq_tokens: Tensor, k_seq_tokens: Tensor, q_send_buffer_offset: Tensor,
                                  k_send_buffer_offset: Tensor, v_send_buffer_offset: Tensor, instance_id: int = None, *, buffer: Tensor = None) -> None:
    """pre_a2a_attn_out_grad_resend_qkv for a caller that does not want the request tokens themselves: the four parts go
    straight into the buffer, where the merged matrix is written and read once more on the way (half the launch's bytes)."""
    parts = [attn_out_grad, attn_out, lse_norm, q]
    _same_tokens("backward request", *parts)
    if not TokenLayout.of(parts).in_parts:
        pre_a2a_attn_out_grad_resend_qkv(attn_out_grad, attn_out, lse_norm, q, k, v, kv_dispatch_mask, q_seq_tokens, k_seq_tokens,
                                         q_send_buffer_offset, k_send_buffer_offset, v_send_buffer_offset, instance_id, buffer=buffer)
        return
    if q.dtype != attn_out.dtype or attn_out_grad.shape != attn_out.shape:
        raise AssertionError("dO, O and q of a backward request share one dtype, and dO has the shape of O")
    buffer = _transport_buffer(buffer, instance_id, True)
    k, v = k.contiguous(), v.contiguous()
    exchange([plain_job([token_part(t) for t in parts], q_send_buffer_offset, q_seq_tokens), replicas_job(k, kv_dispatch_mask, k_send_buffer_offset, k_seq_tokens),
              replicas_job(v, kv_dispatch_mask, v_send_buffer_offset, k_seq_tokens)], buffer, True)


def post_a2a_attn_out_grad_resend_qkv(
    recv_attn_out_shape: List[int], recv_lse_shape: List[int], recv_q_shape: List[int],
    recv_lse_dtype: torch.dtype,
    recv_k: Tensor, recv_v: Tensor,
    kv_dispatch_mask: Tensor, q_recv_seq_tokens: Tensor, k_recv_seq_tokens: Tensor,
    q_recv_buffer_offset: Tensor, k_recv_buffer_offset: Tensor, v_recv_buffer_offset: Tensor,
    is_fwd: bool, switch_buffer: bool = True, instance_id: int = None, *, buffer: Tensor = None,
):
    """Server side of the backward request (dispatch.py:161-206): unpack the [dO | O | lse | q | pad] tokens and
    k, v, then cut the token matrix into its four parts.  Like the reference, always unpacks k / v the forward
    way, whatever `is_fwd` says."""
    rows = recv_attn_out_shape[0]
    if not (len(recv_attn_out_shape) == len(recv_lse_shape) == len(recv_q_shape) == 2) or recv_lse_shape[0] != rows \
            or recv_q_shape[0] != rows:
        raise AssertionError("the parts of a backward request are [tokens, hidden] shapes with one token count")
    act = recv_k.dtype
    layout = TokenLayout([(recv_attn_out_shape[1], act), (recv_attn_out_shape[1], act),
                          (recv_lse_shape[1], recv_lse_dtype), (recv_q_shape[1], act)])
    if layout.in_parts and recv_k.dim() == recv_v.dim() == 2:
        dev = recv_k.device
        parts = [torch.empty(tuple(shape), dtype=dt, device=dev)
                 for shape, dt in zip((recv_attn_out_shape, recv_attn_out_shape, recv_lse_shape, recv_q_shape), layout.dtypes)]
        source = _transport_buffer(buffer, instance_id, False)
        exchange([plain_job(t, off, _lengths_of(tokens, off))
                  for t, off, tokens in ((parts, q_recv_buffer_offset, q_recv_seq_tokens), ([recv_k], k_recv_buffer_offset, k_recv_seq_tokens),
                                         ([recv_v], v_recv_buffer_offset, k_recv_seq_tokens))], source, False)
        _unpacked(buffer, switch_buffer, instance_id)
        d_out, out, lse, q = parts
        return d_out, out, lse, q, recv_k, recv_v
    request = torch.empty((rows, layout.token_bytes), dtype=torch.uint8, device=recv_k.device)
    post_a2a_qkv(request, recv_k, recv_v, kv_dispatch_mask, q_recv_seq_tokens, k_recv_seq_tokens,
                 q_recv_buffer_offset, k_recv_buffer_offset, v_recv_buffer_offset,
                 True, switch_buffer=switch_buffer, instance_id=instance_id, buffer=buffer)
    d_out, out, lse, q = layout.split(request)
    return d_out, out, lse, q, recv_k, recv_v


def pre_a2a_attn_out_with_lse(attn_out: Tensor, softmax_lse: Tensor, send_seqlens: Tensor,
                              send_memcpy_metadata: Tensor, dispatcher_id: int = None, *, buffer: Tensor = None):
    """Forward reply of the server (dispatch.py:209-221): every token travels as [out | lse | pad], lse given
    token-major [T, Hq]."""
    if softmax_lse.shape[0] != attn_out.shape[0]:
        raise AssertionError(f"softmax_lse has {softmax_lse.shape[0]} tokens, attn_out {attn_out.shape[0]}")
    reply = TokenLayout.of([attn_out, softmax_lse]).merge([attn_out, softmax_lse])
    return pre_a2a_attn_out(reply, send_seqlens, send_memcpy_metadata, dispatcher_id, buffer=buffer)
