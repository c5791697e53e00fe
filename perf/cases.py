"""The work a user of this package has it do, as cases that can be timed and compared.

Four kinds of case, each one pass through public entry points:

  attention   varlen causal core attention over whole packed documents: the forward alone (`ca_varlen_fwd`), or forward
              and backward through autograd (`core_attention`)
  tick        one tick of a CA server that holds its tasks' shards in a receive buffer: `fused_comm_attn_forward`, and with
              the backward direction `fused_comm_attn_backward` on the request that follows it
  linear      the linear-layer rank's side of a layer: packs q, k, v for the servers and takes the [out | lse] reply apart,
              and in the backward direction packs the request [dO | O | lse | q], k, v and takes the gradients apart
  copies      a server that keeps attention apart from the exchange: unpacks q and one copy of every K/V prefix per task,
              and packs dq and the copies' summed dk, dv

Documents are packed token after token, their lengths lognormal(8, 1.5) cut to a range, all equal, or one document for
everything.  For the kinds with an exchange the documents lie on `world` ranks of `tokens` tokens each, the planner
balances them over as many servers, and the case is what rank 0 does.  The layout (lengths, plan) belongs to the case;
the tensors are drawn from the seed.
"""
import math

import numpy as np
import torch

from distca_amd.compute_metadata import from_planner_output, step_params
from distca_amd.dispatch_fn import (post_all2all_layout_transfer, post_all2all_layout_transfer_backward, pre_all2all_layout_transfer,
                                    pre_all2all_layout_transfer_backward)
from distca_amd.fused_comm_attn import (FlashAttnArgs, ca_varlen_fwd, core_attention, fused_comm_attn_backward, fused_comm_attn_forward,
                                        post_a2a_attn_out_with_lse, post_a2a_attn_out_with_lse_backward)
from distca_amd.ops import a2a_memcpy_non_cp
from distca_amd.planner import Planner, batch_to_items_general

D = 128          # head dimension of every model configuration here
DEV = "cuda"
LARGEST_FLOPS = 2.4e14   # of a drawn case: that of the largest listed one


def _case(kind, tokens, heads, kv_heads, backward, lengths, lo, hi, dtype="bf16", deterministic=False, world=1, layout=0, **name):
    return dict(kind=kind, tokens=tokens, heads=heads, kv_heads=kv_heads, backward=backward, lengths=lengths, lo=lo, hi=hi,
                dtype=dtype, deterministic=deterministic, world=world, layout=layout, **name)


def listed():
    return [
        # one short sample on a rank that holds an eighth of the heads: launches and the host path are what it costs
        _case("attention", 389, 4, 1, True, "one", 389, 389, name="one_389_token_sample"),
        # three short documents, forward only (evaluation of a few samples)
        _case("attention", 4096, 32, 8, False, "three", 512, 2560, name="three_documents_forward"),
        # a micro-batch of 8192 tokens with the deterministic backward
        _case("attention", 8192, 32, 8, True, "lognormal", 128, 8192, deterministic=True, layout=11, name="micro_batch_8192"),
        # many short documents (instruction tuning data packed to 64k tokens), no two of one length
        _case("attention", 65536, 32, 8, True, "uniform", 128, 2048, layout=12, name="short_documents_65536"),
        # fp16, 70B-model heads, a token count that is no multiple of anything
        _case("attention", 30011, 64, 8, True, "lognormal", 256, 16384, dtype="fp16", layout=13, name="fp16_30011_64_heads"),
        # the benchmark's workload: 131072 packed tokens, documents of 128 to 65536 tokens
        _case("attention", 131072, 32, 8, True, "lognormal", 128, 65536, layout=5002, name="packed_131072"),
        # a lightly loaded server: a few query shards over prefixes of a document that lies on eight ranks, a quarter of the heads
        _case("tick", 4096, 8, 2, False, "one", 32768, 32768, world=8, name="tick_light_forward"),
        # a server in the middle of a training step: documents of all lengths over four ranks
        _case("tick", 16384, 32, 8, True, "lognormal", 128, 32768, world=4, layout=14, name="tick_16384"),
        # long-context training: one document of 131072 tokens over four ranks
        _case("tick", 32768, 32, 8, True, "one", 131072, 131072, world=4, name="tick_long_document"),
        # the linear side of a small step, a quarter of the heads
        _case("linear", 1021, 8, 2, False, "lognormal", 64, 2048, world=4, layout=15, name="linear_1021_forward"),
        # the linear side of a large step, both directions
        _case("linear", 65536, 32, 8, True, "lognormal", 128, 65536, world=4, layout=16, name="linear_65536"),
        # a server with one copy of the prefix per task, both directions
        _case("copies", 32768, 32, 8, True, "lognormal", 128, 65536, world=4, layout=17, name="copies_32768"),
    ]


def draw(rng):
    spread = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    kind = rng.choice(["attention"] * 4 + ["tick"] * 3 + ["linear"] * 2 + ["copies"])
    heads, kv_heads = rng.choice([(4, 1), (8, 2), (32, 8), (32, 8), (64, 8)])
    backward = rng.random() < 0.6
    layout = rng.randrange(1, 1 << 20)
    dtype = "fp16" if rng.random() < 0.2 else "bf16"
    if kind == "attention":
        tokens = spread(256, 131072)
        lengths = rng.choice(["one", "lognormal", "lognormal", "uniform"])
        lo, hi = (64, spread(256, 4096)) if lengths == "uniform" else (128, 65536)
        world, deterministic = 1, rng.random() < 0.5
    else:
        tokens = spread(1024, 32768 if kind == "tick" else 65536 if kind == "linear" else 16384)
        lengths = rng.choice(["one", "lognormal", "lognormal"])
        lo, hi, world, deterministic = 64, 131072, rng.choice([2, 4, 8]), True
    make = lambda n: _case(kind, n, heads, kv_heads, backward, lengths, lo, hi, dtype, deterministic, world, layout)
    while tokens > 1024 and (work(make(tokens))["flops"] > LARGEST_FLOPS or work(make(tokens))["bytes"] > 6e9):
        tokens = tokens * 2 // 3
    return make(tokens)


def _documents(case):
    """Document lengths that add up to the case's tokens (over all ranks)."""
    total = case["tokens"] * case["world"]
    if case["lengths"] == "one":
        return [total]
    if case["lengths"] == "three":
        return [total // 8, total // 4, total - total // 8 - total // 4]
    rng = np.random.default_rng(case["layout"])
    lens, left = [], total
    while left > 0:
        if case["lengths"] == "uniform":
            n = int(rng.integers(case["lo"], case["hi"] + 1))
        else:
            n = int(np.clip(round(math.exp(rng.normal(8.0, 1.5))), case["lo"], case["hi"]))
        lens.append(min(n, left))
        left -= lens[-1]
    if len(lens) > 1 and lens[-1] < case["lo"]:   # a short remainder joins the document before it
        last = lens.pop()
        lens[-1] += last
    return lens


def _plan(case):
    """Per document its shards (owner rank, server rank, place in the document, tokens), balanced by the planner."""
    world, hq, hkv = case["world"], case["heads"] * D, case["kv_heads"] * D
    planner = Planner.from_individual_params(1, 1, world, world, hq, hkv)
    items = batch_to_items_general([_documents(case)], case["tokens"], world, planner.model_config)
    return planner.items_to_shardinfo(items)


def _rank0(case):
    """What rank 0 has of the plan: (tokens it owns, copies of its tokens that go out for k and for v, query tokens and
    stored K/V tokens it serves, K/V tokens with one copy per task, causal pairs it computes)."""
    owned = sent = served_q = served_kv = copied_kv = pairs = 0
    for doc in _plan(case):
        end = 0
        reach = {}   # server -> last shard of the document it needs
        for i, s in enumerate(doc):
            end += s.shard_len
            reach[s.dispatch_rid] = i
            if s.dispatch_rid == 0:
                served_q += s.shard_len
                copied_kv += end
                pairs += s.shard_len * end - s.shard_len * (s.shard_len - 1) // 2
        for i, s in enumerate(doc):
            if s.rid == 0:
                owned += s.shard_len
                sent += s.shard_len * sum(1 for last in reach.values() if last >= i)
            if 0 in reach and i <= reach[0]:
                served_kv += s.shard_len
    return owned, sent, served_q, served_kv, copied_kv, pairs


def _element(case):
    return torch.float16 if case["dtype"] == "fp16" else torch.bfloat16


def _steps(case):
    lse = math.ceil(case["heads"] * 4 / 16) * 16 // 2
    md = from_planner_output(case["world"], _plan(case), case["heads"] * D, case["kv_heads"] * D, lse, 2, is_pipeline_tick=False,
                             is_resend_qkv=True)
    step = step_params(0, md, DEV)
    names = ("qkv", "grad", "out", "request")
    sizes = {n: (int(m.fa2a_metadata[1][0].sum()), int(m.fa2a_metadata[3][0].sum())) for n, m in zip(names, md)}   # rank 0: bytes out, bytes in
    return step, sizes


def _buffer(n):
    return torch.zeros(n, dtype=torch.uint8, device=DEV)


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    dtype = _element(case)
    hq, hkv = case["heads"], case["kv_heads"]
    rand = lambda *shape: torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32).to(dtype)
    rand_bytes = lambda n: rand(n // 2).view(torch.uint8)
    if case["kind"] == "attention":
        lens = _documents(case)
        t = case["tokens"]
        s = dict(q=rand(t, hq, D), k=rand(t, hkv, D), v=rand(t, hkv, D), longest=max(lens),
                 cu=torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).to(DEV))
        if case["backward"]:
            s["dout"] = rand(t, hq, D)
            for name in "qkv":
                s[name].requires_grad_(True)
        return dict(s, case=case)

    step, sizes = _steps(case)
    s = dict(case=case, step=step, dtype=dtype, args=FlashAttnArgs(hq, hkv, D, deterministic=case["deterministic"]))
    out_tok = (hq * D * 2 + hq * 4 + 15) // 16 * 16
    if case["kind"] == "linear":
        t = int(step.qkv_fwd_metadata.seq_lens[0].send_seqlens.sum())
        s.update(q=rand(t, hq * D), k=rand(t, hkv * D), v=rand(t, hkv * D), send=_buffer(sizes["qkv"][0]), reply=rand_bytes(sizes["out"][1]))
        if case["backward"]:
            s.update(dout=rand(t, hq * D), request=_buffer(sizes["request"][0]), grads=rand_bytes(sizes["grad"][1]))
        return s

    s["recv"] = rand_bytes(sizes["qkv"][1])   # q, k and v tokens fill the receive buffer
    if case["kind"] == "copies":
        if case["backward"]:
            tq, tk = step.qkv_fwd_metadata.tensor_shape[0].recv_shape, step.qkv_fwd_metadata.tensor_shape[1].recv_shape
            s.update(dq=rand(*tq), dk=rand(*tk), dv=rand(*tk), send=_buffer(sizes["grad"][0]))
        return s

    s["reply"] = _buffer(sizes["out"][0])
    s["out_tok"] = out_tok
    if case["backward"]:
        # the request that follows this forward: its own out and lse beside dO and q, and the same K/V shards
        fused_comm_attn_forward(s["recv"], s["reply"], step, s["args"], dtype)
        qkv, out, req = step.qkv_fwd_metadata, step.attn_out_fwd_metadata, step.attn_out_bwd_metadata
        tq, row = int(qkv.tensor_shape[0].recv_shape[0]), hq * D * 2
        q = torch.empty((tq, hq * D), dtype=dtype, device=DEV)
        a2a_memcpy_non_cp(q, qkv.recv_memcpy_metadata[0], qkv.seq_lens[0].recv_seqlens, False, buffer=s["recv"])
        token = torch.empty((tq, out_tok), dtype=torch.uint8, device=DEV)
        a2a_memcpy_non_cp(token, out.send_memcpy_metadata[0], out.seq_lens[0].send_seqlens, False, buffer=s["reply"])
        tok = (3 * row + hq * 4 + 15) // 16 * 16
        request = torch.zeros((tq, tok), dtype=torch.uint8, device=DEV)
        request[:, :row] = rand(tq, hq * D).view(torch.uint8)
        request[:, row:2 * row + 4 * hq] = token[:, :row + 4 * hq]
        request[:, 2 * row + 4 * hq:3 * row + 4 * hq] = q.view(torch.uint8)
        s["request"] = _buffer(sizes["request"][1])
        a2a_memcpy_non_cp(request, req.recv_memcpy_metadata[0], req.seq_lens[0].recv_seqlens, True, buffer=s["request"])
        for i in (1, 2):
            entries = zip(qkv.recv_memcpy_metadata[i].tolist(), req.recv_memcpy_metadata[i].tolist(), qkv.seq_lens[1].recv_seqlens.tolist())
            for a, b, n in set(entries):   # an entry per task and shard: aliases of a shard share their place
                s["request"][b:b + n * hkv * D * 2] = s["recv"][a:a + n * hkv * D * 2]
        s["send"] = _buffer(sizes["grad"][0])
        s["reply"].zero_()
    return s


def run(s):
    case = s["case"]
    if case["kind"] == "attention":
        q, k, v, cu, n = s["q"], s["k"], s["v"], s["cu"], s["longest"]
        if not case["backward"]:
            return ca_varlen_fwd(q, k, v, cu, cu, n, n)
        out = core_attention(q, k, v, cu, cu, n, n, deterministic=case["deterministic"])
        return (out,) + torch.autograd.grad(out, (q, k, v), s["dout"])

    step, dtype = s["step"], s["dtype"]
    if case["kind"] == "linear":
        pre_all2all_layout_transfer(s["q"], s["k"], s["v"], step.qkv_fwd_metadata, buffer=s["send"])
        out, lse = post_a2a_attn_out_with_lse(s["reply"], s["q"], case["heads"], step.attn_out_fwd_metadata, dtype)
        if not case["backward"]:
            return s["send"].view(torch.int64), out, lse
        post_a2a_attn_out_with_lse_backward(s["request"], s["dout"], out, lse, s["q"], s["k"], s["v"], step.attn_out_bwd_metadata)
        grads = pre_all2all_layout_transfer_backward(step.qkv_bwd_metadata, dtype, buffer=s["grads"])
        return s["send"].view(torch.int64), out, lse, s["request"].view(torch.int64), grads

    if case["kind"] == "copies":
        qkv = post_all2all_layout_transfer(step.qkv_fwd_metadata, dtype, buffer=s["recv"])
        if not case["backward"]:
            return qkv
        post_all2all_layout_transfer_backward((s["dq"], s["dk"], s["dv"]), step.qkv_bwd_metadata, buffer=s["send"])
        return qkv, s["send"].view(dtype)

    fused_comm_attn_forward(s["recv"], s["reply"], step, s["args"], dtype)
    row, lse = case["heads"] * D * 2, case["heads"] * 4
    token = s["reply"].view(-1, s["out_tok"])   # views of the reply: out and lse of every query token
    reply = token[:, :row].view(dtype), token[:, row:row + lse].view(torch.float32)
    if not case["backward"]:
        return reply
    fused_comm_attn_backward(s["request"], s["send"], step, s["args"], dtype)
    return reply, s["send"].view(dtype)   # dq tokens and the shards' dk, dv


def work(case):
    """Causal pairs at 4 FLOP per pair, head and dimension forward and 10 backward; every input read and every output written once."""
    hq, hkv = case["heads"], case["kv_heads"]
    row, kv, lse = hq * D * 2, hkv * D * 2, hq * 4
    if case["kind"] == "attention":
        tq = tk = case["tokens"]
        pairs = sum(n * (n + 1) // 2 for n in _documents(case))
    else:
        owned, sent, tq, tk, copied, pairs = _rank0(case)
        if case["kind"] == "linear":
            # q, k, v in and their copies out; the reply's tokens in, out and lse out
            nbytes = owned * (2 * row + 2 * kv) + sent * 2 * kv + owned * 2 * (row + lse)
            if case["backward"]:   # dO, O, lse, q, k, v in, request out; dq and every replica's dk, dv in, dq, dk, dv out
                nbytes += owned * 2 * (3 * row + lse) + (owned + sent) * 2 * kv + owned * 2 * row + (sent + owned) * 2 * kv
            return {"bytes": nbytes, "flops": 0}
        if case["kind"] == "copies":
            nbytes = tq * 2 * row + tk * 2 * kv + copied * 2 * kv
            if case["backward"]:
                nbytes += tq * 2 * row + copied * 2 * kv + tk * 2 * kv
            return {"bytes": nbytes, "flops": 0}
    nbytes = tq * (2 * row + lse) + tk * 2 * kv
    if case["backward"]:
        nbytes += tq * (4 * row + lse) + tk * 4 * kv
    return {"bytes": nbytes, "flops": (14 if case["backward"] else 4) * hq * D * pairs}


def tolerance(case):
    """P and dS enter the matrix products in the element type and results are rounded to it: 2 to 3e-3 of a tensor's norm in bf16
    against exact arithmetic, an eighth of that in fp16.  Copies are exact; where copies of a gradient are added up, the sum
    is rounded once or once per copy."""
    if case["kind"] in ("attention", "tick"):
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}
    if not case["backward"]:
        return "exact"
    return {"rel": 5e-3 if case["dtype"] == "bf16" else 7e-4}
