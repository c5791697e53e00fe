"""GPU parity of the HIP attention kernels (through the C ABI) against the CPU oracle."""
import numpy as np
import pytest
import torch

from helpers import assert_close_bf16, cu, make_qkv
from oracle.attention import ca_reference_bwd, ca_reference_fwd

pytestmark = pytest.mark.gpu


def _run(q_lens, k_lens, hq, hkv, seed, cuda, causal=True, kv_offsets=None, total_k=None, bwd=True, d=128, kv_grad_tol=None,
         dtype=torch.bfloat16, deterministic=False):
    from distca_amd.fused_comm_attn import ca_varlen_bwd, ca_varlen_fwd
    cu_q, cu_k = cu(q_lens), cu(k_lens)
    tq = int(cu_q[-1])
    tk = int(total_k if total_k is not None else cu_k[-1])
    q, k, v, do = (t.to(dtype) for t in make_qkv(tq, tk, hq, hkv, d, seed))   # bf16 values are exact in fp16 at this scale
    ref_out, ref_lse = ca_reference_fwd(q, k, v, cu_q, cu_k, causal=causal, kv_task_offsets=kv_offsets)
    dcu_q = torch.tensor(cu_q, device=cuda)
    dcu_k = torch.tensor(cu_k, device=cuda)
    dkv = torch.tensor(np.asarray(kv_offsets, dtype=np.int32), device=cuda) if kv_offsets is not None else None
    qd, kd, vd, dod = q.to(cuda), k.to(cuda), v.to(cuda), do.to(cuda)
    print(f"case q_lens={list(q_lens)[:6]} k_lens={list(k_lens)[:6]} hq={hq} hkv={hkv} causal={causal} alias={kv_offsets is not None}", flush=True)
    out, lse = ca_varlen_fwd(qd, kd, vd, dcu_q, dcu_k, int(max(q_lens)), int(max(k_lens)), None, causal, dkv)
    torch.cuda.synchronize()
    assert out.dtype == dtype and out.shape == qd.shape
    assert_close_bf16(out, ref_out, "out")
    finite = torch.isfinite(ref_lse)
    lse_c = lse.cpu()
    assert torch.equal(torch.isfinite(lse_c), finite)
    assert (lse_c[finite] - ref_lse[finite]).abs().max().item() <= 2e-3, "lse"
    if not bwd:
        return
    # the oracle consumes the same (out, lse) the kernel is handed, as the reference's backward does
    ref_dq, ref_dk, ref_dv = ca_reference_bwd(do, q, k, v, cu_q, cu_k, causal=causal, kv_task_offsets=kv_offsets,
                                              out=out.cpu(), softmax_lse=lse.cpu())
    dq, dk, dv = ca_varlen_bwd(dod, qd, kd, vd, out, lse, dcu_q, dcu_k, int(max(q_lens)), int(max(k_lens)), None, causal,
                               deterministic, dkv)
    torch.cuda.synchronize()
    assert dq.dtype == dk.dtype == dv.dtype == dtype and dq.shape == qd.shape and dk.shape == kd.shape
    if deterministic:
        again = ca_varlen_bwd(dod, qd, kd, vd, out, lse, dcu_q, dcu_k, int(max(q_lens)), int(max(k_lens)), None, causal, True, dkv)
        torch.cuda.synchronize()
        for name, x, y in zip(("dq", "dk", "dv"), (dq, dk, dv), again):
            assert torch.equal(x, y), f"{name} differs between two deterministic runs"
    assert_close_bf16(dq, ref_dq, "dq")
    tol = dict(max_abs=kv_grad_tol[0], mean_rel=kv_grad_tol[1]) if kv_grad_tol else {}
    assert_close_bf16(dk, ref_dk, "dk", **tol)
    assert_close_bf16(dv, ref_dv, "dv", **tol)


def test_config1_tiny_forward(cuda):
    """docs [512, 1024, 2560], 32q/8kv, d128, causal, forward."""
    _run([512, 1024, 2560], [512, 1024, 2560], 32, 8, 1, cuda, bwd=False)


@pytest.mark.parametrize("lens", [[64], [1], [33, 1, 130], [257, 255, 256, 3]])
def test_whole_docs_fwd_bwd_small(cuda, lens):
    _run(lens, lens, 8, 2, 7, cuda)


def test_whole_docs_fwd_bwd_medium(cuda):
    _run([512, 1024, 700], [512, 1024, 700], 32, 8, 2, cuda)


@pytest.mark.parametrize("hq,hkv", [(4, 4), (8, 1), (6, 2), (16, 2), (64, 1), (24, 8), (32, 1), (16, 16), (3, 3), (80, 80)])
def test_head_groupings(cuda, hq, hkv):
    """MHA (also with 16, 3 and 80 kv heads: more lists of work items than XCDs, a count that does not divide
    their number, and more lists than a wave has lanes to look at them), MQA, a non-power-of-two group, the Llama-3-70B group of 8; groups of 64 (more heads per token than a
    backward row block holds), of 3 (a row block does not start at a token boundary) and of 32 (exactly one)."""
    # dK and dV of a kv head sum the bf16-rounded P and dS of all its query heads: with 32 or 64 of them the
    # rounding noise of the sum (growing as the square root of the count) is allowed twice the bar
    _run([300, 45], [300, 45], hq, hkv, 3, cuda, kv_grad_tol=(4e-2, 2e-3) if hq // hkv >= 32 else None)


def test_prefix_tasks_lk_gt_lq(cuda):
    """CA tasks: query shard shorter than its KV prefix (bottom-right causal)."""
    _run([128, 200, 64], [384, 200, 1000], 8, 2, 4, cuda)


@pytest.mark.parametrize("hq,hkv", [(8, 2), (4, 4), (16, 2)])
def test_prefix_lengths_around_tile_and_ring_boundaries(cuda, hq, hkv):
    """Tasks whose K/V prefixes end one key before, on and one key after multiples of 32 (a K/V tile of the dQ
    kernel), of 64 (a tile of the forward) and of 128 (one round of the dQ kernel's four ring stages), with query
    shards of 1 to 100 tokens: workgroups with one to a dozen tiles, with and without unmasked tiles, whose last
    waves own no row or only a few."""
    k_lens = [1, 31, 32, 33, 63, 64, 65, 95, 97, 127, 128, 129, 159, 161, 191, 193, 255, 256, 257, 289, 383, 385]
    q_lens = [1, 31, 17, 33, 5, 64, 65, 16, 97, 100, 3, 1, 64, 33, 100, 17, 8, 100, 65, 1, 100, 49]
    assert all(q <= k for q, k in zip(q_lens, k_lens))
    _run(q_lens, k_lens, hq, hkv, 21, cuda)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("hq,hkv", [(8, 8), (16, 8), (32, 8)])
def test_runs_of_whole_tiles_and_blocks(cuda, hq, hkv, causal):
    """Documents long enough for the runs of whole tiles (dQ) and whole blocks (dK/dV) whose requests stand between the MFMAs, of lengths that end
    a key, a row and a block either side of where the runs end, and enough of them that dK/dV items of both walk directions are among them
    (more key blocks than compute units serve a kv head).  At most four query heads per kv head: a bf16-rounded P of about 1 per head (a
    document's first rows) puts a deviation of 2^-9 / sqrt(3) * sqrt(1.5 heads) on an entry of dV there, and five of them, the largest of the
    eighty thousand such entries here, are 1.4e-2 for four heads and, at the bar of 2e-2, 2.0e-2 for eight."""
    lens = [1031, 769, 770, 768, 767, 991, 1024, 1023, 1025, 640, 832]
    _run(lens, lens, hq, hkv, 23, cuda, causal=causal)


def test_runs_of_whole_tiles_in_merged_blocks_non_causal(cuda):
    """Without a diagonal every tile of a document but the last is whole, also for the blocks that one work item takes after another:
    documents short enough to be merged (below 768 tokens on average, more than 12 blocks of rows per compute unit)."""
    lens = [577, 640, 575, 576, 704, 321] * 8
    _run(lens, lens, 32, 8, 25, cuda, causal=False)


@pytest.mark.parametrize("causal,prefix", [(True, 0), (True, 37), (False, 0)])
def test_rounds_of_one_block_per_ring_stage(cuda, causal, prefix):
    """Runs of whole blocks (dK/dV) and whole tiles (dQ) that begin and end at every stage of the ring of four: at four heads per kv head a
    block of query rows is 8 tokens, so lengths 8 apart (and off by up to 7, with ends of tiles between) leave each remainder, from the first stage on
    and, in dK/dV items that walk upwards, from wherever the diagonal ends; more key blocks than compute units serve a kv head, for both directions."""
    q_lens = [600 + 8 * i + (5 * i) % 8 for i in range(16)]
    _run(q_lens, [n + prefix for n in q_lens], 32, 8, 27, cuda, causal=causal)


@pytest.mark.parametrize("hq,hkv,lens", [(4, 1, [1020]), (4, 1, [1030]), (4, 1, [1540]), (4, 1, [1600]), (32, 8, [2048]), (64, 16, [2050]), (16, 4, [1800, 250])])
def test_either_side_of_the_lines_from_which_blocks_are_cut(cuda, hq, hkv, lens):
    """Tiles that cutting could take off the longest block, where dQ's line is 16 and the forward's 24: 15.5, 16.5, 23.8, 24.7, 16.5 (half of a longer
    block's), none (two blocks of the task a unit), 22.6 (with a short task beside)."""
    _run(lens, lens, hq, hkv, 29, cuda, deterministic=True)


@pytest.mark.parametrize("q_lens,k_lens", [([2048, 40], [2048, 6000]), ([100, 2050], [5003, 2050])])
def test_new_document_beside_a_short_shard_of_a_long_one(cuda, q_lens, k_lens):
    """Two blocks of query rows a unit of one task, whose blocks stay whole, beside a block of another over a long prefix, which is cut."""
    _run(q_lens, k_lens, 64, 16, 37, cuda, deterministic=True)


def test_shared_kv_prefix(cuda):
    """Three shards of one 600-token document reading one stored KV copy."""
    _run([200, 150, 250], [200, 350, 600], 8, 2, 5, cuda, kv_offsets=[0, 0, 0], total_k=600)


@pytest.mark.parametrize("hq,hkv", [(8, 2), (4, 4), (12, 4)])
@pytest.mark.parametrize("causal", [True, False])
def test_shared_kv_documents_deterministic(cuda, hq, hkv, causal):
    """Three stored documents read by tasks that are prefixes of them, with the deterministic switch the reference's
    server has by default: one work item per (document, key block) walks the query rows of every task that sees the
    block and writes dK/dV once.  The documents lie in the store out of order and with unread rows before, between
    and behind them (those come back as zeros); prefixes end around key-block (256) and tile (32, 64) edges, one task
    has no queries, one document is read by a single task, two tasks of a document have the same prefix length."""
    #          document at row 40 (700 rows)      at row 1000 (513 rows)   at row 800 (130 rows)
    k_lens = [255, 256, 257, 700, 700, 33,        512, 513, 300,            130]
    q_lens = [255, 1, 1, 443, 100, 33,            212, 1, 0,                64]
    offs = [40, 40, 40, 40, 40, 40,               1000, 1000, 1000,         800]
    _run(q_lens, k_lens, hq, hkv, 31, cuda, causal=causal, kv_offsets=offs, total_k=1600, deterministic=True)


def test_queries_that_see_no_key(cuda):
    """A task with more queries than keys under the bottom-right aligned mask: its first Lq - Lk rows see nothing.
    Their output and dq are zero and their lse is -inf, and they add nothing to dk / dv (the backward kernels meet
    exp2(+inf) for such rows and must mask it away)."""
    from distca_amd.fused_comm_attn import ca_varlen_bwd, ca_varlen_fwd
    _run([300, 64], [100, 64], 8, 2, 41, cuda)
    q, k, v, do = (t.to(cuda) for t in make_qkv(364, 164, 8, 2, 128, 41))
    cq, ck = torch.tensor(cu([300, 64]), device=cuda), torch.tensor(cu([100, 64]), device=cuda)
    out, lse = ca_varlen_fwd(q, k, v, cq, ck, 300, 100)
    dq, dk, dv = ca_varlen_bwd(do, q, k, v, out, lse, cq, ck, 300, 100)
    torch.cuda.synchronize()
    assert (out[:200] == 0).all() and (dq[:200] == 0).all() and torch.isinf(lse[:, :200]).all() and (lse[:, :200] < 0).all()
    assert torch.isfinite(dk.float()).all() and torch.isfinite(dv.float()).all() and torch.isfinite(dq.float()).all()


@pytest.mark.parametrize("hq,hkv", [(8, 2), (4, 4)])
def test_short_tasks_as_merged_work_items(cuda, hq, hkv):
    """A batch whose tasks average fewer than 2048 query tokens has the forward and dQ kernels work off several
    consecutive blocks of a task per work item (eight for the 1024-token document here, whose sixteen blocks at four
    heads per kv head make two items; the last item of a task is usually shorter), the next block's Q rows and first K
    tile requested while the present one is normalised and stored.  Whole documents and tasks with prefixes, lengths
    on and off the block edges."""
    _run([1024, 1000, 513, 1, 2047, 64], [1024, 1000, 513, 1, 2047, 64], hq, hkv, 51, cuda)
    _run([1024, 300, 700], [1024, 1324, 764], hq, hkv, 52, cuda)


@pytest.mark.parametrize("q_lens,k_lens,hq,hkv", [
    ([64, 1, 300, 0, 37], [5000, 4097, 2348, 300, 2600], 8, 2),     # few query rows over long prefixes, none of a tile's length
    ([33, 70], [4100, 70], 6, 2),                                   # three heads per kv head: blocks end inside a token
    ([3000, 129], [3000, 129], 4, 4),                               # one document longer than the rest together
    ([200], [9000], 16, 1)])
@pytest.mark.parametrize("causal", [True, False])
def test_blocks_cut_into_pieces(cuda, q_lens, k_lens, hq, hkv, causal):
    """Batches of so few blocks that the longest are cut into pieces, whose fp32 results a second kernel adds up: forward (pieces of
    KV tiles, some of which no row of a wave sees), dQ, and dK/dV (pieces of query blocks), with the workspace that has room
    for them, the same bits in a second run, and within rounding of whole blocks (the smallest workspace)."""
    import ctypes
    from distca_amd._lib import CaParams, load
    from distca_amd.fused_comm_attn import ca_varlen_bwd, ca_varlen_fwd
    lib = load()
    tq, tk = sum(q_lens), sum(k_lens)
    p = CaParams(len(q_lens), tq, tk, hq, hkv, 128, max(q_lens), max(k_lens), 128 ** -0.5, int(causal), 1, 0)
    assert lib.distca_ca_fwd_workspace_preferred_bytes(ctypes.byref(p)) > lib.distca_ca_fwd_workspace_bytes(ctypes.byref(p))
    small = int(lib.distca_ca_bwd_workspace_bytes(ctypes.byref(p)))
    assert lib.distca_ca_bwd_workspace_preferred_bytes(ctypes.byref(p)) > small
    _run(q_lens, k_lens, hq, hkv, 71, cuda, causal=causal, deterministic=True)
    q, k, v, do = (t.to(cuda) for t in make_qkv(tq, tk, hq, hkv, 128, 72))
    cq, ck = torch.tensor(cu(q_lens), device=cuda), torch.tensor(cu(k_lens), device=cuda)
    fwd = lambda x, ws=None: ca_varlen_fwd(q, k, x, cq, ck, max(q_lens), max(k_lens), None, causal, None, ws)
    bwd = lambda ws=None: ca_varlen_bwd(do, q, k, v, *first, cq, ck, max(q_lens), max(k_lens), None, causal, True, workspace=ws)
    first, again = fwd(v), fwd(v)
    whole = fwd(v, torch.empty(int(lib.distca_ca_fwd_workspace_bytes(ctypes.byref(p))), dtype=torch.uint8, device=cuda))
    sizes = fwd(v.abs())[0].float()
    grads, grads_again, grads_whole = bwd(), bwd(), bwd(torch.empty(small, dtype=torch.uint8, device=cuda))
    torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in zip(first + grads, again + grads_again))
    # Forward: each P is rounded to bf16 under another running maximum, at most 2^-9 of it on either side, so that the sums differ by at
    # most 2^-8 sum P |V|, which the call with |V| gives (itself to 2^-8); then both results are rounded, 2^-9 each.
    x, y = first[0].float(), whole[0].float()
    assert ((x - y).abs() <= 2.0 ** -8 * (1.01 * sizes + torch.maximum(x.abs(), y.abs()))).all()
    # the sums of the unrounded P: fp32 roundings of some hundred additions and of the exponents
    live = torch.isfinite(whole[1])
    assert torch.equal(torch.isfinite(first[1]), live)
    assert ((first[1] - whole[1])[live].abs() <= 256 * 2.0 ** -24 * whole[1][live].abs().clamp(min=1)).all()
    # Backward, from the same out and lse: the same P and dS, added up in fp32 in another order, then rounded to bf16: one unit in the last
    # place (2^-7 at most), and for what nearly cancels, n / 16 additions of 2^-24 of terms that sum to no more than sqrt(n) times the largest result
    for x, y in zip(grads, grads_whole):
        x, y = x.float(), y.float()
        assert ((x - y).abs() <= 2.0 ** -7 * y.abs() + max(k_lens) ** 1.5 / 16 * 2.0 ** -24 * y.abs().max()).all()


@pytest.mark.parametrize("n", [8, 7, 16, 15])
def test_very_short_tasks_either_side_of_their_merging_rule(cuda, n):
    """Tasks of fewer than 768 tokens in the mean are merged from 8 blocks of query rows per compute unit on, and into items twice
    as long from 16 on: n of them here, on 256 units."""
    lens = [1000, 17, 512, 519] * (n // 2) + [700, 324] * (n % 2)      # n * 1024 tokens x 64 heads = n blocks per unit
    _run(lens, lens, 64, 16, 56, cuda, bwd=n < 9)


@pytest.mark.parametrize("n", [12, 11])
def test_short_tasks_either_side_of_the_merging_rule(cuda, n):
    """Blocks of short tasks are merged into larger work items from 12 blocks of query rows per compute unit on (n of them
    here, on 256 units), and not below that: the first and the last document of a batch on either side against the oracle."""
    from distca_amd.fused_comm_attn import ca_varlen_bwd, ca_varlen_fwd
    lens = [1000, 1048] * (n // 2) + [1024] * (n % 2)      # n * 1024 tokens x 64 heads = n blocks per unit
    q, k, v, do = make_qkv(sum(lens), sum(lens), 64, 16, 128, 53)
    c = cu(lens)
    dev = [t.to(cuda) for t in (q, k, v, do)]
    dc = torch.tensor(c, device=cuda)
    out, lse = ca_varlen_fwd(*dev[:3], dc, dc, max(lens), max(lens))
    grads = ca_varlen_bwd(dev[3], *dev[:3], out, lse, dc, dc, max(lens), max(lens))
    torch.cuda.synchronize()
    for b in (0, len(lens) - 1):
        r = slice(int(c[b]), int(c[b + 1]))
        one = cu([lens[b]])
        ref_out, ref_lse = ca_reference_fwd(q[r], k[r], v[r], one, one)
        assert_close_bf16(out[r], ref_out, "out")
        assert (lse[:, r].cpu() - ref_lse).abs().max().item() < 2e-3
        ref = ca_reference_bwd(do[r], q[r], k[r], v[r], one, one, out=out[r].cpu(), softmax_lse=lse[:, r].cpu())
        for name, got, want in zip(("dq", "dk", "dv"), grads, ref):
            assert_close_bf16(got[r], want, name)


@pytest.mark.parametrize("hq,hkv", [(64, 16), (64, 64)])
def test_merged_items_whose_blocks_start_alike_and_not(cuda, hq, hkv):
    """A merged item requests the first tiles of its next block before it stores the present one: blocks of no tile, one tile and
    several after one another (prefixes shorter than, equal to and longer than the queries, ends on either side of a tile), items of
    one block, a last block that is not full; enough of them for the merging rule (12 blocks of query rows per compute unit)."""
    q_lens = [1, 63, 64, 65, 100, 128, 129, 200, 257, 300, 31]
    k_lens = [1, 63, 64, 70, 100, 128, 193, 100, 257, 40, 95]
    n = -(-12 * 256 * 256 // (hq * sum(q_lens)))
    _run(q_lens * n, k_lens * n, hq, hkv, 54, cuda)


@pytest.mark.parametrize("lens", [[255], [300], [1023], [1024, 65], [2048], [40, 1500, 8]])
@pytest.mark.parametrize("hq,hkv", [(4, 1), (8, 2)])
def test_small_batches_either_side_of_the_cutting_rules(cuda, lens, hq, hkv):
    """Blocks left whole, key blocks in pieces of eight query blocks and more, blocks of query rows from 1024 keys on; the same bits twice."""
    _run(lens, lens, hq, hkv, 55, cuda, deterministic=True)


@pytest.mark.parametrize("hq,hkv,lens", [(4, 1, [1]), (4, 1, [389]), (8, 2, [0, 65, 0, 0, 129, 64, 0]), (4, 4, [1, 257, 3] * 5), (32, 8, [1000]),
                                         (8, 1, [2, 0] * 70 + [33, 31]), (2, 2, [3] * 127), (2, 2, [3] * 128), (32, 8, [1300])])
def test_few_blocks_without_a_list(cuda, hq, hkv, lens):
    """Forward batches whose blocks all run at once are taken by a scan of the task bounds: empty tasks, more tasks than a wave has
    lanes, as many blocks as compute units and more, a longer prefix; the lists of the backward beside them."""
    _run(lens, lens, hq, hkv, 57, cuda, bwd=len(lens) < 20)
    _run(lens, [n + 70 if n else 0 for n in lens], hq, hkv, 58, cuda, bwd=False)


def test_non_causal(cuda):
    _run([100, 260], [100, 260], 4, 2, 6, cuda, causal=False)


def test_long_document_in_pieces(cuda):
    """One document of 4096 tokens: too few key blocks to occupy the device, so the backward cuts every key
    block into pieces of consecutive query blocks (the first block into about thirty) and adds their dK/dV in
    fp32; also a deterministic run of the same, whole blocks, bit for bit equal to a second one."""
    from distca_amd.fused_comm_attn import ca_varlen_bwd, ca_varlen_fwd
    _run([4096], [4096], 8, 2, 11, cuda)
    q, k, v, do = (t.to(cuda) for t in make_qkv(4096, 4096, 8, 2, 128, 11))
    c = torch.tensor(cu([4096]), device=cuda)
    out, lse = ca_varlen_fwd(q, k, v, c, c, 4096, 4096, None, True, None)
    a = ca_varlen_bwd(do, q, k, v, out, lse, c, c, 4096, 4096, None, True, True, None)
    b = ca_varlen_bwd(do, q, k, v, out, lse, c, c, 4096, 4096, None, True, True, None)
    torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in zip(a, b))
    n = ca_varlen_bwd(do, q, k, v, out, lse, c, c, 4096, 4096, None, True, False, None)
    torch.cuda.synchronize()
    for x, y, name in zip(n, a, ("dq", "dk", "dv")):
        # same products, summed per piece and then across pieces in fp32: a bf16 unit in the last place apart at most
        err = ((x.float() - y.float()).abs() / y.float().abs().clamp_min(2.0 ** -6)).max().item()
        assert err <= 2.0 ** -7, f"{name}: pieces against whole blocks {err:.2e}"


@pytest.mark.parametrize("hq,hkv,n", [(128, 8, 989), (64, 8, 1345), (64, 8, 1364), (32, 8, 2999), (4, 1, 3000), (8, 2, 1500),
                                      (16, 16, 7600), (16, 16, 7700)])
def test_single_documents_around_the_piece_cutting_threshold(cuda, hq, hkv, n):
    """One document per call, backward with key blocks cut into pieces: lengths at which the piece count comes
    closest to the room the work list has (989 tokens at 128/8 heads and 1345 at 64/8 made one piece too many when
    the piece size was rounded down), and a pair of lengths either side of the size from which blocks stay whole
    (7680 tokens at 16 kv heads).  Gradients against the oracle, and the builder's count of entries it had no
    room for must be zero."""
    from distca_amd._lib import CaParams, load
    from distca_amd.fused_comm_attn import ca_varlen_bwd, ca_varlen_fwd
    import ctypes
    q, k, v, do = make_qkv(n, n, hq, hkv, 128, 31)
    c = cu([n])
    dc = torch.tensor(c, device=cuda)
    qd, kd, vd, dod = q.to(cuda), k.to(cuda), v.to(cuda), do.to(cuda)
    p = CaParams(1, n, n, hq, hkv, 128, n, n, 128 ** -0.5, 1, 0, 0)
    ws = torch.zeros(load().distca_ca_bwd_workspace_bytes(ctypes.byref(p)), dtype=torch.uint8, device=cuda)
    print(f"case single document n={n} hq={hq} hkv={hkv}", flush=True)
    out, lse = ca_varlen_fwd(qd, kd, vd, dc, dc, n, n)
    dq, dk, dv = ca_varlen_bwd(dod, qd, kd, vd, out, lse, dc, dc, n, n, None, True, False, None, workspace=ws)
    torch.cuda.synchronize()
    head = ws[:16].view(torch.int32).cpu()
    assert int(head[2]) == 0, f"the key-block list dropped {int(head[2])} entries"
    from distca_amd import scheduler
    assert int(head[0]) == len(scheduler.build_schedule(scheduler.BWD, c, c, hq, hkv))
    ref_dq, ref_dk, ref_dv = ca_reference_bwd(do, q, k, v, c, c, out=out.cpu(), softmax_lse=lse.cpu())
    tol = dict(max_abs=4e-2, mean_rel=2e-3) if hq // hkv >= 16 else {}
    assert_close_bf16(dq, ref_dq, "dq")
    assert_close_bf16(dk, ref_dk, "dk", **tol)
    assert_close_bf16(dv, ref_dv, "dv", **tol)


def test_key_blocks_walked_in_both_directions(cuda):
    """The dK/dV list marks alternate rounds of items (as many as compute units serve a kv head: 16 here) to be
    walked upwards from the diagonal instead of downwards from the end.  Whole key blocks (deterministic), prefix
    tasks among them: both directions occur, the gradients match the oracle and a second run bit for bit."""
    from distca_amd import scheduler
    from distca_amd.fused_comm_attn import ca_varlen_bwd, ca_varlen_fwd
    q_lens, k_lens, hq, hkv = [2600, 900, 1800, 37], [2600, 2100, 1800, 300], 16, 16
    items = scheduler.build_schedule(scheduler.BWD, cu(q_lens), cu(k_lens), hq, hkv, deterministic=True)
    up = items[:, 3] < 0
    assert up.any() and (~up).any() and (scheduler.item_pieces(items[:, 3]) == 1).all()
    cu_q, cu_k = cu(q_lens), cu(k_lens)
    q, k, v, do = make_qkv(int(cu_q[-1]), int(cu_k[-1]), hq, hkv, 128, 77)
    dq_, dk_ = torch.tensor(cu_q, device=cuda), torch.tensor(cu_k, device=cuda)
    qd, kd, vd, dod = q.to(cuda), k.to(cuda), v.to(cuda), do.to(cuda)
    out, lse = ca_varlen_fwd(qd, kd, vd, dq_, dk_, max(q_lens), max(k_lens))
    a = ca_varlen_bwd(dod, qd, kd, vd, out, lse, dq_, dk_, max(q_lens), max(k_lens), None, True, True, None)
    b = ca_varlen_bwd(dod, qd, kd, vd, out, lse, dq_, dk_, max(q_lens), max(k_lens), None, True, True, None)
    torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in zip(a, b))
    ref = ca_reference_bwd(do, q, k, v, cu_q, cu_k, out=out.cpu(), softmax_lse=lse.cpu())
    for x, r, name in zip(a, ref, ("dq", "dk", "dv")):
        assert_close_bf16(x, r, name)


def test_empty_task(cuda):
    _run([128, 0, 70], [128, 0, 70], 4, 2, 8, cuda)


@pytest.mark.parametrize("span", [6.0, 40.0, 400.0, -400.0])
def test_scores_that_drift_along_the_keys(cuda, span):
    """The forward keeps a running reference per row that trails the row maximum by up to 2^8 and
    is only corrected when a tile overshoots it.  Scores here carry a trend of `span` (natural-log
    units) from the first key to the last: a reference that is seldom, sometimes, or in every tile
    overtaken, and one that is never overtaken after the first tile."""
    from distca_amd.fused_comm_attn import ca_varlen_bwd, ca_varlen_fwd
    n, hq, hkv, d = 2048, 4, 2, 128
    q, k, v, do = make_qkv(n, n, hq, hkv, d, 21)
    q, k = q.float(), k.float()
    q[:, :, 0] = 16.0
    k[:, :, 0] = (span * (d ** 0.5) / 16.0) * torch.arange(n, dtype=torch.float32)[:, None] / n
    q, k = q.to(torch.bfloat16), k.to(torch.bfloat16)
    cu_q = cu([n])
    ref_out, ref_lse = ca_reference_fwd(q, k, v, cu_q, cu_q)
    dcu = torch.tensor(cu_q, device=cuda)
    qd, kd, vd, dod = q.to(cuda), k.to(cuda), v.to(cuda), do.to(cuda)
    print(f"case drift span={span}", flush=True)
    out, lse = ca_varlen_fwd(qd, kd, vd, dcu, dcu, n, n, None, True, None)
    torch.cuda.synchronize()
    assert_close_bf16(out, ref_out, "out")
    assert (lse.cpu() - ref_lse).abs().max().item() <= 2e-3 * max(1.0, abs(span) / 40), "lse"
    if abs(span) > 10:
        return  # the backward keeps no running reference, and K entries of tens amplify the bf16 rounding of dS beyond the bar
    ref_dq, ref_dk, ref_dv = ca_reference_bwd(do, q, k, v, cu_q, cu_q, out=out.cpu(), softmax_lse=lse.cpu())
    dq, dk, dv = ca_varlen_bwd(dod, qd, kd, vd, out, lse, dcu, dcu, n, n, None, True, False, None)
    torch.cuda.synchronize()
    assert_close_bf16(dq, ref_dq, "dq")
    assert_close_bf16(dk, ref_dk, "dk")
    assert_close_bf16(dv, ref_dv, "dv")


@pytest.mark.parametrize("case", ["one block", "two blocks", "group of 3", "many blocks", "shared", "non-causal"])
@pytest.mark.parametrize("dtype,level", [(torch.float16, -24.0), (torch.bfloat16, -120.0)])
def test_missing_rows_of_a_task_whose_scores_are_far_below_zero(cuda, dtype, level, case):
    """The last block of 32 query rows of a task that is no multiple of it: where every key is seen the dK/dV kernel compares nothing, so that its
    missing rows have to add nothing by themselves.  With the statistics of the task's last row their P was exp(-lse): infinite in the element type
    below lse = -11.1 (fp16) and -88.7 (bf16), and 0 * inf put NaN into dV and dK of every key seen.  Scores are shifted by `level`: dimension 0 of q
    and k holds constants whose product it is.  Gradients of those constants are left out of the comparison (dS rounded to the element type times a
    constant of tens, in sums whose exact value is near zero), but not of the check for NaN."""
    from distca_amd.fused_comm_attn import ca_varlen_bwd, ca_varlen_fwd
    hq, hkv, offs = 32, 8, None
    k_lens = {"one block": [150], "two blocks": [300, 129, 159], "group of 3": [139, 270], "many blocks": [289, 300, 383, 141, 258] * 16, "shared": [150, 281, 300],
              "non-causal": [150, 301]}[case]
    q_lens = [70, 90, 19] if case == "shared" else k_lens
    if case == "group of 3":
        hq, hkv = 12, 4
    if case == "many blocks":   # enough for the kernel of batches that are not cut
        hq, hkv = 32, 16
    causal = case != "non-causal"
    if case == "shared":
        offs = [0, 0, 0]
    cu_q, cu_k = cu(q_lens), cu(k_lens)
    tk = max(k_lens) if offs else int(cu_k[-1])
    q, k, v, do = (t.to(dtype) for t in make_qkv(int(cu_q[-1]), tk, hq, hkv, 128, 28))
    a = 16.0 if dtype == torch.float16 else 32.0
    q[:, :, 0], k[:, :, 0] = a, round(level * 128 ** 0.5 / a * 4) / 4   # (exact in both types)
    c = (torch.tensor(cu_q, device=cuda), torch.tensor(cu_k, device=cuda), max(q_lens), max(k_lens))
    dkv = torch.tensor(offs, dtype=torch.int32, device=cuda) if offs else None
    qd, kd, vd, dod = (t.to(cuda) for t in (q, k, v, do))
    print(f"case {case} {dtype} level={level}", flush=True)
    out, lse = ca_varlen_fwd(qd, kd, vd, *c, None, causal, dkv)
    torch.cuda.synchronize()
    assert lse.max().item() < (-11.2 if dtype == torch.float16 else -88.8)
    got = ca_varlen_bwd(dod, qd, kd, vd, out, lse, *c, None, causal, False, dkv)
    torch.cuda.synchronize()
    ref = ca_reference_bwd(do, q, k, v, cu_q, cu_k, causal=causal, kv_task_offsets=offs, out=out.cpu(), softmax_lse=lse.cpu())
    for name, x, r in zip(("dq", "dk", "dv"), got, ref):
        bad = int((~torch.isfinite(x.float())).sum())
        assert bad == 0, f"{name}: {bad} values are not finite"
        assert_close_bf16(x if name == "dv" else x[..., 1:], r if name == "dv" else r[..., 1:], name)


@pytest.mark.parametrize("seed", range(12))
def test_random_task_batches(cuda, seed):
    """Seeded random batches of CA tasks: lengths around the tile edges (32, 64, 128, 256 +- 1), prefixes
    longer than the query shard, every head grouping the kernels accept, causal or not, with and
    without tasks that share one stored K/V copy."""
    rng = np.random.default_rng(1000 + seed)
    edges = [1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 383, 511, 513]
    n = int(rng.integers(1, 7))
    q_lens = [int(rng.choice(edges)) if rng.random() < 0.7 else int(rng.integers(1, 700)) for _ in range(n)]
    if rng.random() < 0.25:
        q_lens[int(rng.integers(n))] = 0
    hq, hkv = [(4, 4), (8, 2), (8, 1), (12, 4), (16, 2), (2, 1)][int(rng.integers(6))]
    causal = bool(rng.random() < 0.8)
    if rng.random() < 0.3 and all(q_lens):
        # shards of one document over one stored copy of its K/V
        ends = np.cumsum(q_lens)
        _run(q_lens, [int(e) for e in ends], hq, hkv, seed, cuda, causal=causal, kv_offsets=[0] * n, total_k=int(ends[-1]))
        return
    k_lens = [q + (int(rng.choice(edges)) if (q and rng.random() < 0.5) else 0) for q in q_lens]
    _run(q_lens, k_lens, hq, hkv, seed, cuda, causal=causal)


@pytest.mark.parametrize("case", ["whole", "prefix", "shared", "groups", "pieces"])
def test_fp16_inputs(cuda, case):
    """The same kernels compiled for IEEE half precision (the reference's own tests run fp16,
    tests/test_megatron_layer.py of the reference): whole documents, prefix tasks, tasks that share one stored K/V
    copy (float atomics in dK/dV), a group of 8 query heads, and a batch small enough for key blocks to be cut into
    pieces.  Same bar as bf16, with the rounding floor taken in fp16 (its rounding error is an eighth of bf16's, so the
    bar is the looser of the two here)."""
    f16 = torch.float16
    if case == "whole":
        _run([257, 255, 256, 3, 700], [257, 255, 256, 3, 700], 8, 2, 61, cuda, dtype=f16)
    elif case == "prefix":
        _run([128, 200, 64], [384, 200, 1000], 8, 2, 62, cuda, dtype=f16)
    elif case == "shared":
        _run([200, 150, 250], [200, 350, 600], 8, 2, 63, cuda, kv_offsets=[0, 0, 0], total_k=600, dtype=f16)
    elif case == "groups":
        _run([300, 45], [300, 45], 16, 2, 64, cuda, dtype=f16)
    else:
        _run([4096], [4096], 8, 2, 65, cuda, dtype=f16)


@pytest.mark.parametrize("form", ["own", "shared", "whole"])
@pytest.mark.parametrize("group", [(4, 4), (12, 4), (8, 2)])
def test_key_blocks_that_end_anywhere(cuda, form, group):
    """Tasks that end at every edge of the 32-key halves that the dK/dV kernel's waves own in a block of 256 keys, seen whole or
    through a prefix, own or shared, causal (some halves are never seen by a query block) and not."""
    ends = [1, 32, 33, 96, 97, 128, 129, 160, 223, 225, 256 + 31, 512 + 127]
    if form == "shared":
        _run([32] * 5, [32, 96, 128, 160, 287], *group, 71, cuda, kv_offsets=[0] * 5, total_k=287)
    elif form == "whole":
        _run(ends, ends, *group, 72, cuda, causal=False)
    else:
        _run(ends, ends, *group, 73, cuda)
        _run([e - e // 3 for e in ends], ends, *group, 74, cuda)


def test_fp16_and_bf16_agree_on_the_same_values(cuda):
    """Inputs that are exact in both types give outputs that differ by the types' rounding only: the fp16 build is
    the bf16 build with another element type, not another algorithm."""
    from distca_amd.fused_comm_attn import ca_varlen_fwd
    lens = [513, 64, 300]
    q, k, v, _ = make_qkv(sum(lens), sum(lens), 8, 2, 128, 66)
    c = torch.tensor(cu(lens), device=cuda)
    outs, lses = [], []
    for dt in (torch.bfloat16, torch.float16):
        o, l = ca_varlen_fwd(q.to(cuda).to(dt), k.to(cuda).to(dt), v.to(cuda).to(dt), c, c, max(lens), max(lens))
        outs.append(o.float().cpu()); lses.append(l.cpu())
    assert (lses[0] - lses[1]).abs().max().item() <= 2e-3
    assert (outs[0] - outs[1]).abs().max().item() <= 2e-2


@pytest.mark.parametrize("seed", range(6))
def test_blocks_by_rank_and_from_a_list(cuda, seed):
    """A forward of few blocks over at most 64 tasks has no list: workgroups find the block of their rank.  With a 65th task there is one.  Tasks of all
    sizes, without tokens or keys among them, more queries than keys or fewer, over their own or over shared rows, causal or not: every block is
    computed exactly once, to the same bits."""
    from distca_amd.fused_comm_attn import ca_varlen_fwd
    rng = np.random.default_rng(900 + seed)
    hq, hkv = [(32, 8), (16, 4), (8, 8), (12, 4), (64, 8), (4, 1)][seed]
    n = [64, 64, 63, 64, 8, 64][seed]
    top = [200, 800, 400, 500, 1400, 1400][seed]   # (no blocks long enough to be cut)
    q_lens = [int(x) for x in rng.integers(0, top, n)]
    k_lens = [int(q) if rng.random() < 0.5 else int(rng.integers(0, top + 100)) for q in q_lens]
    if seed == 1:
        q_lens[:40] = [0] * 40   # ranks past the last task with blocks
    causal, shared = seed != 3, seed == 2
    fill = 65 - n
    tq = sum(q_lens) + fill
    tk = max(k_lens) if shared else sum(k_lens) + fill
    assert tq * hq > 256 * torch.cuda.get_device_properties(0).multi_processor_count, "one round of workgroups: blocks as they come"
    q, k, v, _ = (t.to(cuda) for t in make_qkv(tq, max(tk, 1), hq, hkv, 128, 90 + seed))
    res = []
    for ql, kl in ((q_lens, k_lens), (q_lens + [1] * fill, k_lens + [1] * fill)):
        off = torch.zeros(len(ql), dtype=torch.int32, device=cuda) if shared else None
        rows = sum(kl) if not shared else tk
        res.append(ca_varlen_fwd(q[:sum(ql)].contiguous(), k[:rows].contiguous(), v[:rows].contiguous(), torch.tensor(cu(ql), device=cuda),
                                 torch.tensor(cu(kl), device=cuda), max(ql), max(kl), None, causal, off))
    tokens = sum(q_lens)
    assert torch.equal(res[0][0], res[1][0][:tokens])
    assert torch.equal(res[0][1], res[1][1][:, :tokens])
    assert bool(torch.isfinite(res[0][0].float()).all())
    # prefixes longer than they were said to be: every block all the same (a bound on the same side of the line between the forward's kernels)
    low = max(k_lens) // 2 if max(k_lens) <= 1280 else 1300
    ql, kl, off = q_lens, k_lens, torch.zeros(n, dtype=torch.int32, device=cuda) if shared else None
    rows = sum(kl) if not shared else tk
    short = ca_varlen_fwd(q[:sum(ql)].contiguous(), k[:rows].contiguous(), v[:rows].contiguous(), torch.tensor(cu(ql), device=cuda),
                          torch.tensor(cu(kl), device=cuda), max(ql), low, None, causal, off)
    assert torch.equal(short[0], res[0][0]) and torch.equal(short[1], res[0][1])


@pytest.mark.parametrize("q_lens,k_lens,hq,hkv,causal", [
    ([5000], [5000], 8, 2, True), ([5100], [5100], 8, 2, True),               # pieces of one document
    ([300, 150], [12000, 2500], 16, 2, True), ([500, 60], [12000, 2500], 16, 2, True),   # pieces of a few rows over long prefixes
    ([2400], [2400], 32, 8, True), ([2600], [2600], 32, 8, True),             # blocks by rank
    ([1700], [1700], 32, 8, False), ([1800], [1800], 32, 8, False),
    ([1280] * 5, [1280] * 5, 32, 8, True), ([1281] * 5, [1281] * 5, 32, 8, True),
    ([4096] * 2, [4096] * 2, 8, 2, True), ([4097, 4000], [4097, 4000], 8, 2, True)])   # a block a unit
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_either_side_of_the_lines_between_the_forwards_mfmas(cuda, q_lens, k_lens, hq, hkv, causal, dtype):
    """Batches of few blocks have 32x32x16 MFMAs up to 24 tiles a compute unit (as far as the bounds tell) or prefixes of 1280 keys, or, where no unit has two blocks, 33
    tiles and prefixes of 4096, 16x16x32 beyond.  The smallest workspace, without room for pieces, leaves blocks whole: 32x32x16 MFMAs wherever no unit has two, and
    results within rounding of the others."""
    keys = max(k_lens) - min(max(q_lens), max(k_lens)) // 2 if causal else max(k_lens)
    load = sum(q_lens) * hq * keys / (256 * 64 * torch.cuda.get_device_properties(0).multi_processor_count)
    assert 20 < load < 34, "sizes near the line"
    _run(q_lens, k_lens, hq, hkv, 84, cuda, causal=causal, bwd=False, dtype=dtype)
    import ctypes
    from distca_amd._lib import CaParams, load
    from distca_amd.fused_comm_attn import ca_varlen_fwd
    q, k, v, _ = (t.to(dtype).to(cuda) for t in make_qkv(sum(q_lens), sum(k_lens), hq, hkv, 128, 84))
    p = CaParams(len(q_lens), sum(q_lens), sum(k_lens), hq, hkv, 128, max(q_lens), max(k_lens), 128 ** -0.5, int(causal), 0, 0)
    ws = torch.empty(int(load().distca_ca_fwd_workspace_bytes(ctypes.byref(p))), dtype=torch.uint8, device=cuda)
    args = (torch.tensor(cu(q_lens), device=cuda), torch.tensor(cu(k_lens), device=cuda), max(q_lens), max(k_lens), None, causal, None)
    few, sizes, (out, lse) = ca_varlen_fwd(q, k, v, *args, ws), ca_varlen_fwd(q, k, v.abs(), *args)[0].float(), ca_varlen_fwd(q, k, v, *args)
    x, y = few[0].float(), out.float()   # (the bounds of test_blocks_cut_into_pieces)
    assert ((x - y).abs() <= 2.0 ** -8 * (1.01 * sizes + torch.maximum(x.abs(), y.abs()))).all()
    assert ((few[1] - lse).abs() <= 256 * 2.0 ** -24 * lse.abs().clamp(min=1)).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gradients_side_by_side_and_one_after_the_other(cuda, dtype):
    """40 documents of 256 tokens at 32/8 heads are the most blocks of query rows (five a compute unit) whose dQ and dK/dV share a launch, with the row
    statistics made ahead of both; with a document of one token more the dQ kernel makes them and runs first.  Documents that are one
    key block each are never cut, so that every one of their gradients comes from the same sums in the same order: the same bits."""
    from distca_amd.fused_comm_attn import ca_varlen_bwd, ca_varlen_fwd
    n = 5 * 256 * torch.cuda.get_device_properties(0).multi_processor_count // 32 // 256
    lens = [256] * n + [1]
    tokens = 256 * n
    q, k, v, do = (t.to(dtype).to(cuda) for t in make_qkv(tokens + 1, tokens + 1, 32, 8, 128, 81))
    res = []
    for part, docs in ((slice(0, tokens), lens[:-1]), (slice(0, tokens + 1), lens)):
        c = torch.tensor(cu(docs), device=cuda)
        x = [t[part].contiguous() for t in (q, k, v, do)]
        out, lse = ca_varlen_fwd(*x[:3], c, c, 256, 256)
        res.append(ca_varlen_bwd(x[3], *x[:3], out, lse, c, c, 256, 256, None, True, True))
    for name, a, b in zip(("dq", "dk", "dv"), *res):
        assert torch.equal(a, b[:tokens]), name
    ref = ca_reference_bwd(*(t[:256].cpu() for t in (do, q, k, v)), cu([256]), cu([256]))
    for name, a, b in zip(("dq", "dk", "dv"), res[0], ref):
        assert_close_bf16(a[:256], b, name)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,rows,prefixes", [(4, 1, 256, [2048 * (i + 1) for i in range(8)]), (8, 2, 200, [900, 4000, 4100]), (32, 8, 512, [512, 4096])])
def test_gradients_of_queries_over_shared_rows_and_over_copies(cuda, hq, hkv, rows, prefixes, dtype):
    """Tasks over prefixes of one stored document, and over a copy of the prefix each: dq has the same bits, whether its kernel shares a launch with
    dK/dV (which the number of stored rows decides) or not."""
    import ctypes
    from distca_amd import _lib
    from distca_amd.fused_comm_attn import ca_varlen_bwd, ca_varlen_fwd
    n = len(prefixes)
    q, k, v, do = (t.to(dtype).to(cuda) for t in make_qkv(n * rows, max(prefixes), hq, hkv, 128, 83))
    cq, ck = (torch.tensor(cu(x), device=cuda) for x in ([rows] * n, prefixes))
    res = []
    for copies in (False, True):
        kk, vv = (torch.cat([t[:p] for p in prefixes]) if copies else t for t in (k, v))
        off = None if copies else torch.zeros(n, dtype=torch.int32, device=cuda)
        p = _lib.CaParams(n, n * rows, kk.shape[0], hq, hkv, 128, rows, max(prefixes), 128 ** -0.5, 1, 1, 1 if dtype == torch.float16 else 2)
        ws = torch.empty(_lib.load().distca_ca_bwd_workspace_preferred_bytes(ctypes.byref(p)), dtype=torch.uint8, device=cuda)
        out, lse = ca_varlen_fwd(q, kk, vv, cq, ck, rows, max(prefixes), None, True, off)
        res.append((out, lse, ca_varlen_bwd(do, q, kk, vv, out, lse, cq, ck, rows, max(prefixes), None, True, True, off, workspace=ws)[0]))
    for name, a, b in zip(("out", "lse", "dq"), *res):
        assert torch.equal(a, b), name


@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("lens", [[256, 31, 200, 130], [2048], [1500, 257, 300]])
def test_gradients_in_the_place_of_their_inputs(cuda, lens, shared):
    """dk and dv written over k and v: dQ, which reads all keys, is then not made beside them.  Small batches, whose gradients otherwise share a launch,
    whole and in pieces, which may have other ends then: the order of a few fp32 sums, 2^-24 each of their size, ahead of one rounding to 2^-9, which
    moves about one result in some thousand by a unit."""
    from distca_amd.fused_comm_attn import ca_varlen_bwd, ca_varlen_fwd
    hq, hkv = 8, 2
    q_lens, k_lens = (lens, lens) if not shared else ([n // 2 for n in lens], lens)
    off = torch.zeros(len(lens), dtype=torch.int32, device=cuda) if shared else None
    tq, tk = sum(q_lens), max(lens) if shared else sum(lens)
    cq, ck = torch.tensor(cu(q_lens), device=cuda), torch.tensor(cu(k_lens), device=cuda)
    q, k, v, do = (t.to(cuda) for t in make_qkv(tq, tk, hq, hkv, 128, 82))
    out, lse = ca_varlen_fwd(q, k, v, cq, ck, max(q_lens), max(k_lens), None, True, off)
    args = (cq, ck, max(q_lens), max(k_lens), None, True, False, off)
    want = ca_varlen_bwd(do, q, k, v, out, lse, *args)
    ki, vi = k.clone(), v.clone()
    got = ca_varlen_bwd(do, q, ki, vi, out, lse, *args, dk=ki, dv=vi)
    assert got[1].data_ptr() == ki.data_ptr()
    for name, a, b in zip(("dq", "dk", "dv"), got, want):
        assert (a.float() - b.float()).norm() <= 1e-3 * b.float().norm(), name


@pytest.mark.parametrize("d,dtype", [(64, torch.bfloat16), (96, torch.float16), (40, torch.bfloat16), (8, torch.bfloat16)])
def test_head_dims_below_128(cuda, d, dtype):
    """Head dimensions that are multiples of 8 below 128 (the reference pads to a multiple of 8 and lets flash-attn
    handle the rest, fused_comm_attn.py:125-129): zero-padded to 128 on the way in, outputs and gradients cut back.
    The softmax scale is that of the true head dimension."""
    _run([130, 257, 64], [130, 300, 64], 4, 2, 67 + d, cuda, d=d, dtype=dtype)


def test_head_dims_that_are_refused(cuda):
    from distca_amd.fused_comm_attn import ca_varlen_fwd
    c = torch.tensor([0, 16], dtype=torch.int32, device=cuda)
    for d in (136, 256, 100):
        x = torch.zeros((16, 2, d), dtype=torch.bfloat16, device=cuda)
        with pytest.raises(RuntimeError, match="head_dim"):
            ca_varlen_fwd(x, x, x, c, c, 16, 16)
    q = torch.zeros((16, 2, 128), dtype=torch.float16, device=cuda)
    with pytest.raises(RuntimeError, match="same for q, k and v"):
        ca_varlen_fwd(q, q.to(torch.bfloat16), q, c, c, 16, 16)
    with pytest.raises(RuntimeError, match="bfloat16 or float16"):
        ca_varlen_fwd(q.float(), q.float(), q.float(), c, c, 16, 16)


@pytest.mark.parametrize("q_lens,hq,hkv", [([3000, 129, 40, 33], 8, 2), ([2000] + [64] * 20, 4, 1), ([2600, 900, 600], 32, 8), ([512], 8, 2), ([4100, 17], 2, 2)])
@pytest.mark.parametrize("shared", [False, True])
def test_pieces_within_the_smallest_workspace(cuda, q_lens, hq, hkv, shared):
    """Without the deterministic switch the smallest workspace has room for a few pieces of key blocks (of the longest document; none
    where all blocks are alike or too few): nothing is written behind it, nothing is dropped, and dK / dV are the preferred workspace's
    but for the order of their fp32 sums."""
    import ctypes
    from distca_amd._lib import CaParams, load
    from distca_amd.fused_comm_attn import ca_varlen_bwd, ca_varlen_fwd
    tq = sum(q_lens)
    q, k, v, do = (t.to(cuda) for t in make_qkv(tq, tq, hq, hkv, 128, 61))
    c, off = torch.tensor(cu(q_lens), device=cuda), torch.tensor(cu(q_lens)[:-1], device=cuda) if shared else None
    n = max(q_lens)
    out, lse = ca_varlen_fwd(q, k, v, c, c, n, n, kv_task_offsets=off)
    p = CaParams(len(q_lens), tq, tq, hq, hkv, 128, n, n, 128 ** -0.5, 1, 0, 0)
    need = int(load().distca_ca_bwd_workspace_bytes(ctypes.byref(p)))
    ws = torch.full((need + 65536,), 0x5A, dtype=torch.uint8, device=cuda)
    print(f"smallest workspace {need} B, tasks {q_lens} heads {hq}/{hkv} shared={shared}", flush=True)
    few = ca_varlen_bwd(do, q, k, v, out, lse, c, c, n, n, kv_task_offsets=off, workspace=ws[:need])
    many = ca_varlen_bwd(do, q, k, v, out, lse, c, c, n, n, kv_task_offsets=off)
    torch.cuda.synchronize()
    assert (ws[need:] == 0x5A).all()
    assert int(ws[:16].view(torch.int32)[2]) == 0
    for x, y, name in zip(few, many, ("dq", "dk", "dv")):
        # the bound of test_blocks_cut_into_pieces: the same P and dS, added up in fp32 in another order, then rounded to bf16
        x, y = x.float(), y.float()
        assert ((x - y).abs() <= 2.0 ** -7 * y.abs() + n ** 1.5 / 16 * 2.0 ** -24 * y.abs().max()).all(), name


@pytest.mark.parametrize("tokens,hq,hkv,mb", [(4096, 4, 1, 139.3), (4096, 8, 2, 144.0), (2048, 4, 1, 89.3)])
@pytest.mark.parametrize("shared", [False, True])
def test_workspace_with_one_place_for_pieces(cuda, tokens, hq, hkv, mb, shared):
    """Workspaces of what the preferred size was when the pieces of dQ and of dK/dV had their slots in one place (the test's figures): blocks are cut as with
    the present size, the kernels run one after the other, and nothing is written behind the workspace."""
    import ctypes
    from distca_amd._lib import CaParams, load
    from distca_amd.fused_comm_attn import ca_varlen_bwd, ca_varlen_fwd
    q, k, v, do = (t.to(cuda) for t in make_qkv(tokens, tokens, hq, hkv, 128, 65))
    c, off = torch.tensor(cu([tokens]), device=cuda), torch.zeros(1, dtype=torch.int32, device=cuda) if shared else None
    p = CaParams(1, tokens, tokens, hq, hkv, 128, tokens, tokens, 128 ** -0.5, 1, 1, 0)
    need, room = int(load().distca_ca_bwd_workspace_preferred_bytes(ctypes.byref(p))), int(mb * 1e6)
    assert int(load().distca_ca_bwd_workspace_bytes(ctypes.byref(p))) < room < need
    ws = torch.full((room + 65536,), 0x5A, dtype=torch.uint8, device=cuda)
    out, lse = ca_varlen_fwd(q, k, v, c, c, tokens, tokens, kv_task_offsets=off)
    args = (do, q, k, v, out, lse, c, c, tokens, tokens, None, True, True, off)
    res = [ca_varlen_bwd(*args, workspace=ws[:room]), ca_varlen_bwd(*args, workspace=ws[:room]),
           ca_varlen_bwd(*args, workspace=torch.empty(need, dtype=torch.uint8, device=cuda))]
    assert int(ws[:4].view(torch.int32)) > tokens // 256, "no key block was cut"
    assert (ws[room:] == 0x5A).all()
    for name, x, again, y in zip(("dq", "dk", "dv"), *res):
        assert torch.equal(x, again), name
        x, y = x.float(), y.float()   # (the bound of test_pieces_within_the_smallest_workspace; dq's pieces are the same)
        assert torch.equal(x, y) if name == "dq" else ((x - y).abs() <= 2.0 ** -7 * y.abs() + tokens ** 1.5 / 16 * 2.0 ** -24 * y.abs().max()).all(), name


def test_small_batches_where_memory_is_short(cuda):
    """A batch whose preferred workspace does not fit any more: the smallest is taken, and the results are those of calls that bring it."""
    import ctypes
    from distca_amd._lib import CaParams, load
    from distca_amd.fused_comm_attn import _workspace, ca_varlen_bwd, ca_varlen_fwd, core_attention
    n, hq, hkv = 4096, 8, 2
    q, k, v, do = (t.to(cuda) for t in make_qkv(n, n, hq, hkv, 128, 63))
    c = torch.tensor(cu([n]), device=cuda)
    p = CaParams(1, n, n, hq, hkv, 128, n, n, 128 ** -0.5, 1, 1, 0)
    size = lambda name: int(getattr(load(), name)(ctypes.byref(p)))
    least = [size(f"distca_ca_{d}_workspace_bytes") for d in ("fwd", "bwd")]
    assert min(size(f"distca_ca_{d}_workspace_preferred_bytes") for d in ("fwd", "bwd")) > 80e6
    small = [torch.empty(b, dtype=torch.uint8, device=cuda) for b in least]
    out, lse = ca_varlen_fwd(q, k, v, c, c, n, n, workspace=small[0])
    want = (out,) + tuple(ca_varlen_bwd(do, q, k, v, out, lse, c, c, n, n, deterministic=True, workspace=small[1]))
    for t in (q, k, v):
        t.requires_grad_(True)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    print("memory capped at 64 MB beyond what is held", flush=True)
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / torch.cuda.mem_get_info()[1])
    try:
        ticks = [_workspace(d, p, cuda, "tick").numel() for d in ("fwd", "bwd")]
        got = core_attention(q, k, v, c, c, n, n, deterministic=True)
        got = (got,) + torch.autograd.grad(got, (q, k, v), do)
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert ticks == least
    assert all(torch.equal(x, y) for x, y in zip(got, want))


def test_offsets_may_be_written_again_before_the_backward(cuda):
    """The first rows of the tasks, in a buffer that every layer's call fills anew with the same values."""
    from distca_amd.fused_comm_attn import core_attention
    lens = [100, 200]
    q, k, v, do = (t.to(cuda) for t in make_qkv(300, 300, 4, 1, 128, 64))
    c, off = torch.tensor(cu(lens), device=cuda), torch.tensor(cu(lens)[:-1], device=cuda)
    buf, res = off.clone(), []
    for again in (False, True):
        leaf = [t.clone().requires_grad_(True) for t in (q, k, v)]
        out = core_attention(*leaf, c, c, 200, 200, deterministic=True, kv_task_offsets=buf)
        if again:
            buf.copy_(off)
        res.append(torch.autograd.grad(out, leaf, do))
    assert all(torch.equal(x, y) for x, y in zip(*res))
