"""GPU parity (bit-exact) of the shard pack / unpack / grad-sum kernels against the oracle."""
import numpy as np
import pytest
import torch

from oracle import fa2a

pytestmark = pytest.mark.gpu


def _layout(rng, lens, token_bytes, slack=64):
    perm = rng.permutation(len(lens))
    off = np.zeros(len(lens), dtype=np.int64)
    cur = 16 * int(rng.integers(0, 4))
    for s in perm:
        off[s] = cur
        cur += int(lens[s]) * token_bytes + 16 * int(rng.integers(0, slack))
    return off, cur


@pytest.mark.parametrize("hidden,dtype", [(128, torch.bfloat16), (1024, torch.bfloat16), (4096, torch.bfloat16), (24, torch.float32), (8320, torch.uint8)])
@pytest.mark.parametrize("nshard", [1, 7, 300])
def test_non_cp_pack_unpack(cuda, hidden, dtype, nshard):
    from distca_amd.ops import a2a_memcpy_non_cp
    rng = np.random.default_rng(hidden * 1000 + nshard)
    lens = rng.integers(0, 40, size=nshard).astype(np.int64)
    lens[rng.integers(0, nshard)] += 5
    T = int(lens.sum())
    esz = torch.empty((), dtype=dtype).element_size()
    tb = hidden * esz
    off, nbuf = _layout(rng, lens, tb)
    src = torch.from_numpy(rng.integers(0, 256, size=(T, tb), dtype=np.uint8)).view(dtype).reshape(T, hidden)
    mask = (rng.random(nshard) < 0.7).astype(np.int8)
    for use_mask in (False, True):
        buf0 = rng.integers(0, 256, size=nbuf, dtype=np.uint8)
        exp = buf0.copy()
        fa2a.copy_non_cp(src.view(torch.uint8).numpy().reshape(T, tb), exp, off, lens, mask if use_mask else None, True)
        dbuf = torch.from_numpy(buf0.copy()).to(cuda)
        print(f"pack hidden={hidden} {dtype} nshard={nshard} mask={use_mask}", flush=True)
        a2a_memcpy_non_cp(src.to(cuda), torch.from_numpy(off).to(cuda), torch.from_numpy(lens).to(cuda), True,
                          torch.from_numpy(mask).to(cuda) if use_mask else None, buffer=dbuf)
        torch.cuda.synchronize()
        assert np.array_equal(dbuf.cpu().numpy(), exp)
    # unpack the unmasked pack into a poisoned tensor: identity
    dst = torch.full((T, tb), 0xA5, dtype=torch.uint8, device=cuda).view(dtype).reshape(T, hidden)
    a2a_memcpy_non_cp(dst, torch.from_numpy(off).to(cuda), torch.from_numpy(lens).to(cuda), False, None, buffer=dbuf if not use_mask else torch.from_numpy(exp).to(cuda))
    exp_t = np.full((T, tb), 0xA5, dtype=np.uint8)
    fa2a.copy_non_cp(exp_t, exp, off, lens, None, False)
    torch.cuda.synchronize()
    assert np.array_equal(dst.view(torch.uint8).reshape(T, tb).cpu().numpy(), exp_t)


@pytest.mark.parametrize("scale", [1, 60])
def test_several_tensors_in_one_launch(cuda, scale):
    """a2a_memcpy_non_cp_multi (q, k, v of a tick against one buffer in one launch) leaves the bytes the oracle leaves
    after three separate copies: packing with and without per-shard masks, then unpacking into poisoned tensors.
    `scale` 60 makes shards of up to 2 400 tokens (19 MB): slices of several loop rounds that cross shard ends."""
    from distca_amd.ops import a2a_memcpy_non_cp_multi
    rng = np.random.default_rng(500 + scale)
    hiddens = [4096, 1024, 1024, 520]                      # bf16 q, k, v and an odd fourth tensor (1040-byte tokens)
    shard_counts = [11, 17, 17, 3]
    lens = [(rng.integers(0, 40, size=n) * scale).astype(np.int64) for n in shard_counts]
    for l in lens:
        l[rng.integers(0, len(l))] += 5
    lens[2] = lens[1].copy()
    tbs = [h * 2 for h in hiddens]
    offs, base = [], 0
    for l, tb in zip(lens, tbs):
        o, n = _layout(rng, l, tb)
        offs.append(o + base)
        base += n
    srcs = [rng.integers(0, 256, size=(int(l.sum()), tb), dtype=np.uint8) for l, tb in zip(lens, tbs)]
    masks = [(rng.random(len(l)) < 0.6).astype(np.int8) for l in lens]
    dev = lambda a: torch.from_numpy(a).to(cuda)
    d_srcs = [dev(a).view(torch.bfloat16) for a in srcs]
    d_offs, d_lens, d_masks = [dev(o) for o in offs], [dev(l) for l in lens], [dev(m) for m in masks]
    for use_mask in (True, False):
        buf0 = rng.integers(0, 256, size=base, dtype=np.uint8)
        exp = buf0.copy()
        for a, o, l, m, tb in zip(srcs, offs, lens, masks, tbs):
            fa2a.copy_non_cp(a, exp, o, l, m if use_mask else None, True)
        dbuf = dev(buf0.copy())
        print(f"multi pack scale={scale} mask={use_mask} buffer {base} B", flush=True)
        a2a_memcpy_non_cp_multi(d_srcs, d_offs, d_lens, True, d_masks if use_mask else None, buffer=dbuf)
        torch.cuda.synchronize()
        assert np.array_equal(dbuf.cpu().numpy(), exp)
    dsts = [torch.full(a.shape, 0x5A, dtype=torch.uint8, device=cuda).view(torch.bfloat16) for a in srcs]
    print(f"multi unpack scale={scale}", flush=True)
    a2a_memcpy_non_cp_multi(dsts, d_offs, d_lens, False, d_masks, buffer=dbuf)     # masks are ignored when unpacking
    torch.cuda.synchronize()
    for a, d in zip(srcs, dsts):
        assert np.array_equal(d.view(torch.uint8).cpu().numpy(), a)
    # fewer jobs, one of them empty
    empty = torch.empty((0, 1024), dtype=torch.bfloat16, device=cuda)
    z = torch.zeros(0, dtype=torch.int64, device=cuda)
    dbuf2 = dev(np.zeros(base, dtype=np.uint8))
    a2a_memcpy_non_cp_multi([d_srcs[0], empty], [d_offs[0], z], [d_lens[0], z], True, buffer=dbuf2)
    torch.cuda.synchronize()
    exp2 = np.zeros(base, dtype=np.uint8)
    fa2a.copy_non_cp(srcs[0], exp2, offs[0], lens[0], None, True)
    assert np.array_equal(dbuf2.cpu().numpy(), exp2)


@pytest.mark.parametrize("max_cp", [1, 3])
def test_cp_pack_unpack(cuda, max_cp):
    from distca_amd.ops import a2a_memcpy_cp
    rng = np.random.default_rng(77 + max_cp)
    nshard, hidden = 9, 1024
    lens = rng.integers(1, 50, size=nshard).astype(np.int64)
    T = int(lens.sum())
    tb = hidden * 2
    do_shard = (rng.random((nshard, max_cp)) < 0.6).astype(np.int8)
    do_shard[:, 0] = 1
    off = np.zeros((max_cp, nshard), dtype=np.int64)
    cur = 0
    for c in range(max_cp):
        for s in rng.permutation(nshard):
            off[c, s] = cur
            cur += int(lens[s]) * tb
    src = torch.from_numpy(rng.integers(0, 256, size=(T, tb), dtype=np.uint8))
    exp = np.zeros(cur, dtype=np.uint8)
    fa2a.copy_cp(src.numpy(), exp, do_shard, off, lens, True)
    dbuf = torch.zeros(cur, dtype=torch.uint8, device=cuda)
    d_do, d_off, d_len = (torch.from_numpy(x).to(cuda) for x in (do_shard, off, lens))
    print(f"cp pack max_cp={max_cp}", flush=True)
    a2a_memcpy_cp(src.view(torch.bfloat16).to(cuda), d_do, d_off, d_len, True, buffer=dbuf)
    torch.cuda.synchronize()
    assert np.array_equal(dbuf.cpu().numpy(), exp)
    planes = torch.zeros((max_cp, T, hidden), dtype=torch.bfloat16, device=cuda)
    a2a_memcpy_cp(planes, d_do, d_off, d_len, False, buffer=dbuf)
    exp_p = np.zeros((max_cp, T, tb), dtype=np.uint8)
    fa2a.copy_cp(exp_p, exp, do_shard, off, lens, False)
    torch.cuda.synchronize()
    assert np.array_equal(planes.view(torch.uint8).reshape(max_cp, T, tb).cpu().numpy(), exp_p)


@pytest.mark.parametrize("max_cp,nshard,hidden,longest", [
    (1, 4, 8, 1), (64, 4, 8, 3), (65, 5, 8, 40), (130, 4, 24, 5), (2, 256, 8, 2), (3, 40, 2048, 140),   # a vector a thread: at most 256 shards
    (2, 257, 8, 2), (3, 520, 16, 9), (2, 300, 1024, 60)])                                              # by slices: more than that
def test_many_replicas_and_shards(cuda, max_cp, nshard, hidden, longest):
    """Replicas and shards are found by lanes of a wave: more of either than a wave has, shards of fewer rows than that, empty ones among
    them.  Packed, unpacked, summed over replicas and over copies (exact: small whole numbers); plain copies of the same shards."""
    from distca_amd.ops import a2a_memcpy_cp, a2a_memcpy_non_cp, copy_sum_job, exchange, replica_sum_job
    rng = np.random.default_rng(max_cp)
    lens = rng.integers(0, longest + 1, size=nshard).astype(np.int64)
    lens[[0, 2, 3]] = longest
    T, tb = int(lens.sum()), hidden * 2
    do_shard = (rng.random((nshard, max_cp)) < 0.5).astype(np.int8)
    do_shard[:, max_cp - 1] = 1
    off = np.zeros((max_cp, nshard), dtype=np.int64)
    cur = 0
    for c in range(max_cp):
        for s in rng.permutation(nshard):
            off[c, s] = cur
            cur += int(lens[s]) * tb
    src = torch.randint(-2, 3, (T, hidden), generator=torch.Generator().manual_seed(nshard)).to(torch.bfloat16)
    raw = src.view(torch.uint8).numpy()
    exp = np.zeros(cur, dtype=np.uint8)
    fa2a.copy_cp(raw, exp, do_shard, off, lens, True)
    d_do, d_off, d_len = (torch.from_numpy(x).to(cuda) for x in (do_shard, off, lens))
    print(f"replicas {max_cp} shards {nshard}", flush=True)
    dbuf = torch.zeros(cur, dtype=torch.uint8, device=cuda)
    a2a_memcpy_cp(src.to(cuda), d_do, d_off, d_len, True, buffer=dbuf)
    planes = torch.zeros((max_cp, T, hidden), dtype=torch.bfloat16, device=cuda)
    a2a_memcpy_cp(planes, d_do, d_off, d_len, False, buffer=dbuf)
    total = torch.empty((T + 3, hidden), dtype=torch.bfloat16, device=cuda)
    exchange([replica_sum_job(total, d_do, d_off, d_len)], dbuf, False)
    torch.cuda.synchronize()
    assert np.array_equal(dbuf.cpu().numpy(), exp)
    exp_p = np.zeros((max_cp, T, tb), dtype=np.uint8)
    fa2a.copy_cp(exp_p, exp, do_shard, off, lens, False)
    assert np.array_equal(planes.view(torch.uint8).reshape(max_cp, T, tb).cpu().numpy(), exp_p)
    want = torch.from_numpy(exp_p).view(torch.bfloat16).reshape(max_cp, T, hidden).float().sum(0).to(torch.bfloat16)
    assert torch.equal(total[:T].cpu(), want) and not total[T:].any()   # (rows behind the last shard: sums of nothing)

    mask = (rng.random(nshard) < 0.7).astype(np.int8)
    nc, cs = np.zeros(nshard, np.int32), np.zeros((nshard, 70), np.int64)
    start = np.concatenate([[0], np.cumsum(lens)])
    nc[0], cs[0, :66] = 66, np.resize(start[[2, 3]], 66)   # (more copies than lanes)
    exp_t, exp1 = src.clone(), np.zeros(cur, dtype=np.uint8)
    fa2a.grad_sum(exp_t, nc, cs, lens)
    fa2a.copy_non_cp(exp_t.view(torch.uint8).numpy(), exp1, off[0], lens, mask, True)
    d, dbuf1, d_mask = src.to(cuda), torch.zeros(cur, dtype=torch.uint8, device=cuda), torch.from_numpy(mask).to(cuda)
    exchange([copy_sum_job(d, d_off[0], d_len, d_mask, torch.from_numpy(nc).to(cuda), torch.from_numpy(cs).to(cuda))], dbuf1, True)
    dbuf2, back = torch.zeros_like(dbuf1), torch.zeros_like(d)
    a2a_memcpy_non_cp(d, d_off[0], d_len, True, d_mask, buffer=dbuf2)
    a2a_memcpy_non_cp(back, d_off[max_cp - 1], d_len, False, None, buffer=dbuf)
    torch.cuda.synchronize()
    assert torch.equal(d.cpu(), exp_t) and np.array_equal(dbuf1.cpu().numpy(), exp1) and np.array_equal(dbuf2.cpu().numpy(), exp1)
    assert torch.equal(back.cpu(), src)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("hidden", [128, 1024, 20])
def test_grad_sum(cuda, dtype, hidden):
    from distca_amd.ops import pre_a2a_grad_acc
    rng = np.random.default_rng(hidden)
    # shards: mains with copies interleaved with plain shards
    lens, num_copies, starts = [], [], []
    spec = [(37, 2), (5, 0), (64, 1), (1, 3), (12, 0)]
    order = []
    for i, (ln, nc) in enumerate(spec):
        order.append((i, ln, nc, True))
        for c in range(nc):
            order.append((i, ln, 0, False))
    perm = rng.permutation(len(order))
    order = [order[i] for i in perm]
    pos, main_idx, copy_pos = 0, {}, {}
    for j, (i, ln, nc, is_main) in enumerate(order):
        if is_main:
            main_idx[i] = j
        else:
            copy_pos.setdefault(i, []).append(pos)
        lens.append(ln)
        pos += ln
    T = pos
    max_copies = 3
    nc_arr = np.zeros(len(order), dtype=np.int32)
    cs = np.zeros((len(order), max_copies), dtype=np.int64)
    for i, (ln, nc) in enumerate(spec):
        nc_arr[main_idx[i]] = nc
        for c, p in enumerate(copy_pos.get(i, [])):
            cs[main_idx[i], c] = p
    g = torch.Generator().manual_seed(hidden)
    data = (torch.randn((T, hidden), generator=g) * 3).to(dtype)
    exp = data.clone()
    fa2a.grad_sum(exp, nc_arr, cs, lens)
    d = data.to(cuda)
    print(f"grad_sum {dtype} hidden={hidden}", flush=True)
    pre_a2a_grad_acc(d, torch.from_numpy(nc_arr).to(cuda), torch.from_numpy(cs).to(cuda), torch.tensor(lens, dtype=torch.int64, device=cuda))
    torch.cuda.synchronize()
    assert torch.equal(d.cpu().view(torch.uint8), exp.view(torch.uint8))


def test_through_torch_ops(cuda):
    """The same kernels called as `torch.ops.distca_amd.*` with the reference's op names and argument
    order (csrc/bindings/all_to_all.cpp:102-113,182-254): pack, replicating pack and duplicate sum."""
    from distca_amd import torch_ops  # noqa: F401  (registers the ops)
    rng = np.random.default_rng(5)
    nshard, hidden = 6, 256
    lens = rng.integers(1, 30, size=nshard).astype(np.int64)
    T, tb = int(lens.sum()), hidden * 2
    off, nbuf = _layout(rng, lens, tb)
    src = torch.from_numpy(rng.integers(0, 256, size=(T, tb), dtype=np.uint8))
    mask = np.array([1, 0, 1, 1, 0, 1], dtype=np.int8)
    exp = np.full(nbuf, 0x33, dtype=np.uint8)
    fa2a.copy_non_cp(src.numpy(), exp, off, lens, mask, True)
    dbuf = torch.full((nbuf,), 0x33, dtype=torch.uint8, device=cuda)
    d_off, d_len = torch.from_numpy(off).to(cuda), torch.from_numpy(lens).to(cuda)
    print("torch.ops non_cp", flush=True)
    torch.ops.distca_amd.fast_a2a_memcpy_non_cp_debug(src.view(torch.bfloat16).to(cuda), d_off, d_len, torch.from_numpy(mask).to(cuda), True, dbuf)
    torch.cuda.synchronize()
    assert np.array_equal(dbuf.cpu().numpy(), exp)

    max_cp = 2
    do_shard = np.ones((nshard, max_cp), dtype=np.int8)
    do_shard[2, 1] = 0
    off2 = np.zeros((max_cp, nshard), dtype=np.int64)
    cur = 0
    for c in range(max_cp):
        for s in rng.permutation(nshard):
            off2[c, s] = cur
            cur += int(lens[s]) * tb
    exp2 = np.zeros(cur, dtype=np.uint8)
    fa2a.copy_cp(src.numpy(), exp2, do_shard, off2, lens, True)
    dbuf2 = torch.zeros(cur, dtype=torch.uint8, device=cuda)
    print("torch.ops cp", flush=True)
    torch.ops.distca_amd.fast_a2a_memcpy_cp_debug(src.view(torch.bfloat16).to(cuda), torch.from_numpy(do_shard).to(cuda),
                                                  torch.from_numpy(off2).to(cuda), d_len, True, dbuf2)
    torch.cuda.synchronize()
    assert np.array_equal(dbuf2.cpu().numpy(), exp2)

    # rows 0..9 are a main shard with one copy in rows 10..19
    g = torch.Generator().manual_seed(9)
    data = torch.randn((20, hidden), generator=g).to(torch.bfloat16)
    nc = np.array([1, 0], dtype=np.int32)
    cs = np.array([[10], [0]], dtype=np.int64)
    ln = [10, 10]
    expd = data.clone()
    fa2a.grad_sum(expd, nc, cs, ln)
    d = data.to(cuda)
    print("torch.ops grad_acc", flush=True)
    torch.ops.distca_amd.fast_a2a_grad_acc(d, torch.from_numpy(nc).to(cuda), torch.from_numpy(cs).to(cuda), torch.tensor(ln, dtype=torch.int64, device=cuda))
    torch.cuda.synchronize()
    assert torch.equal(d.cpu().view(torch.uint8), expd.view(torch.uint8))


@pytest.mark.parametrize("sizes,pad,shards,most", [(*form, *layout) for form in [((8192, 8192, 128, 8192), 0), ((16,), 32), ((1040, 16), 16), ((2048, 24, 2048), None)]
                                                    for layout in [(9, 12), (9, 480), (300, 12)]] + [((262144, 128, 16), 32, 9, 12), ((262144, 128, 16), 32, 300, 3)])
def test_tokens_of_several_parts(cuda, sizes, pad, shards, most):
    """Parts of a transport token copied straight between their tensors and the buffer, next to a replicated tensor in the
    same launch, against the oracle's copy of the joined rows: one-vector parts, padding behind the last part, a part read at a pitch, by vectors
    and (300 shards) by slices, of many tokens and of a part of which one token is several rounds.  Sizes that are no whole vectors are refused on the host."""
    from distca_amd.ops import exchange, plain_job, replicas_job, whole_vectors
    rng = np.random.default_rng(len(sizes) * 100 + shards + most)
    lens = rng.integers(0, most, size=shards).astype(np.int64)
    lens[4] += 3
    T = int(lens.sum())
    parts = [rng.integers(0, 256, size=(T, n), dtype=np.uint8) for n in sizes]
    dev = lambda a: torch.from_numpy(a).to(cuda)
    if pad is None:
        assert not whole_vectors(*sizes)
        with pytest.raises(RuntimeError, match="multiple"):
            exchange([plain_job([dev(p) for p in parts], dev(np.zeros(shards, np.int64)), dev(lens))], torch.zeros(64, dtype=torch.uint8, device=cuda), True)
        return
    tb = sum(sizes) + pad
    off, nbuf = _layout(rng, lens, tb)
    joined = np.concatenate(parts + [np.zeros((T, pad), np.uint8)], axis=1)
    # a second tensor, replicated twice behind the tokens
    do_shard = np.ones((shards, 2), np.int8)
    do_shard[1::2, 1] = 0
    src = rng.integers(0, 256, size=(T, 64), dtype=np.uint8)
    cp_off = np.zeros((2, shards), np.int64)
    for c in range(2):
        cp_off[c] = nbuf + np.concatenate([[0], np.cumsum(lens * 64)[:-1]])
        nbuf += T * 64
    exp = rng.integers(0, 256, size=nbuf, dtype=np.uint8)
    dbuf = dev(exp.copy())
    fa2a.copy_non_cp(joined, exp, off, lens, None, True)
    fa2a.copy_cp(src, exp, do_shard, cp_off, lens, True)
    wide = [np.zeros((T, n + 48), np.uint8) for n in sizes]
    for w, p in zip(wide, parts):
        w[:, 16:16 + p.shape[1]] = p
    d_parts = [dev(p) for p in parts]
    d_parts[-1] = dev(wide[-1])[:, 16:16 + sizes[-1]]
    print(f"parts {sizes} pad {pad} shards {shards} tokens {T}", flush=True)
    exchange([plain_job(d_parts, dev(off), dev(lens), token_bytes=tb), replicas_job(dev(src), dev(do_shard), dev(cp_off), dev(lens))], dbuf, True)
    torch.cuda.synchronize()
    assert np.array_equal(dbuf.cpu().numpy(), exp)
    back = [dev(np.full_like(w, 0x5A)) for w in wide]
    exchange([plain_job([b[:, 16:16 + n] for b, n in zip(back, sizes)], dev(off), dev(lens), token_bytes=tb)], dbuf, False)
    torch.cuda.synchronize()
    for b, p in zip(back, parts):
        want = np.full(b.shape, 0x5A, np.uint8)
        want[:, 16:16 + p.shape[1]] = p
        assert np.array_equal(b.cpu().numpy(), want)


@pytest.mark.parametrize("what,mb", [(w, mb) for w in ("pack", "unpack", "reply", "sum") for mb in (20, 100)] + [("pack", 60)])
def test_either_side_of_the_lines_between_vectors_and_slices(cuda, what, mb):
    """The same shards by either kernel: few and long, so that the lines lie between 30 and 60 MB (and a pack's again above 84)."""
    from distca_amd.ops import exchange, plain_job, replica_sum_job
    rng = np.random.default_rng(mb)
    sizes = [4096, 128] if what == "reply" else [4096]
    tb = sum(sizes)
    T = mb * 10 ** 6 // tb
    lens = np.array([T // 3, 1, 0, T // 2, T - T // 3 - T // 2 - 1], dtype=np.int64)
    off, nbuf = _layout(rng, lens, tb)
    dev = lambda a: torch.from_numpy(a).to(cuda)
    print(f"{what} {T} tokens", flush=True)
    if what == "pack":
        rows, exp, dbuf = rng.integers(0, 256, size=(T, tb), dtype=np.uint8), np.zeros(nbuf, np.uint8), torch.zeros(nbuf, dtype=torch.uint8, device=cuda)
        fa2a.copy_non_cp(rows, exp, off, lens, None, True)
        exchange([plain_job([dev(rows)], dev(off), dev(lens))], dbuf, True)
        torch.cuda.synchronize()
        assert np.array_equal(dbuf.cpu().numpy(), exp)
        return
    buf = torch.randint(-9, 10, (nbuf // 2,), generator=torch.Generator().manual_seed(mb)).to(torch.bfloat16).view(torch.uint8)
    exp = np.zeros((T, tb), np.uint8)
    fa2a.copy_non_cp(exp, buf.numpy(), off, lens, None, False)
    if what == "sum":   # two replicas of every row, the second the first one over again
        got = torch.empty((T, tb // 2), dtype=torch.bfloat16, device=cuda)
        exchange([replica_sum_job(got, torch.ones((5, 2), dtype=torch.int8, device=cuda), dev(np.stack([off, off])), dev(lens))], buf.to(cuda), False)
        torch.cuda.synchronize()
        assert torch.equal(got.cpu(), 2 * torch.from_numpy(exp).view(torch.bfloat16))
        return
    got = [torch.empty((T, n), dtype=torch.uint8, device=cuda) for n in sizes]
    exchange([plain_job(got, dev(off), dev(lens))], buf.to(cuda), False)
    torch.cuda.synchronize()
    assert np.array_equal(np.concatenate([x.cpu().numpy() for x in got], axis=1), exp)


@pytest.mark.parametrize("shards", [20, 300])
def test_parts_beside_sums_in_one_launch(cuda, shards):
    """A token of two parts and a tensor whose copies are added up, in one launch, and the parts taken apart beside a sum over replicas: by vectors,
    and by slices (300 shards)."""
    from distca_amd.ops import copy_sum_job, exchange, plain_job, replica_sum_job
    rng = np.random.default_rng(shards)
    lens = rng.integers(0, 30, size=shards).astype(np.int64)
    lens[7] = lens[3]
    T, start = int(lens.sum()), np.concatenate([[0], np.cumsum(lens)])
    dev = lambda a: torch.from_numpy(a).to(cuda)
    parts = [rng.integers(0, 256, size=(T, n), dtype=np.uint8) for n in (1040, 16)]
    off, at = _layout(rng, lens, 1056)
    main = torch.randint(-2, 3, (T, 72), generator=torch.Generator().manual_seed(shards)).to(torch.bfloat16)
    sum_off, nbuf = _layout(rng, lens, 144)
    sum_off += at
    nbuf += at
    nc, cs = np.zeros(shards, np.int32), np.zeros((shards, 1), np.int64)
    nc[3], cs[3, 0] = 1, start[7]
    mask = (np.arange(shards) != 7).astype(np.int8)
    exp, exp_main = np.zeros(nbuf, np.uint8), main.clone()
    fa2a.copy_non_cp(np.concatenate(parts, axis=1), exp, off, lens, None, True)
    fa2a.grad_sum(exp_main, nc, cs, lens)
    fa2a.copy_non_cp(exp_main.view(torch.uint8).numpy(), exp, sum_off, lens, mask, True)
    d, dbuf = main.to(cuda), torch.zeros(nbuf, dtype=torch.uint8, device=cuda)
    print(f"parts beside sums, {shards} shards", flush=True)
    exchange([plain_job([dev(p) for p in parts], dev(off), dev(lens)), copy_sum_job(d, dev(sum_off), dev(lens), dev(mask), dev(nc), dev(cs))], dbuf, True)
    back = [torch.zeros((T, n), dtype=torch.uint8, device=cuda) for n in (1040, 16)]
    total = torch.empty((T, 72), dtype=torch.bfloat16, device=cuda)
    do_shard = np.stack([mask, np.zeros(shards, np.int8), mask], axis=1)
    exchange([plain_job(back, dev(off), dev(lens)), replica_sum_job(total, dev(np.ascontiguousarray(do_shard)), dev(np.stack([sum_off] * 3)), dev(lens))], dbuf, False)
    torch.cuda.synchronize()
    assert np.array_equal(dbuf.cpu().numpy(), exp) and torch.equal(d.cpu(), exp_main)
    for x, p in zip(back, parts):
        assert np.array_equal(x.cpu().numpy(), p)
    want = 2 * exp_main
    want[int(start[7]):int(start[8])] = 0
    assert torch.equal(total.cpu(), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("scale", [1, 60])
def test_rows_added_up_on_the_way(cuda, dtype, scale):
    """A sum over replicas is the oracle's planes summed in fp32 and rounded once (three replicas: exact in fp32 for two-byte
    elements of this range, one rounding of 2^-24 apart in fp32), shards without replicas give zeros; a sum over copies leaves
    in tensor and buffer what the oracle's sum followed by its masked pack leaves, bit for bit."""
    from distca_amd.ops import copy_sum_job, exchange, replica_sum_job
    rng = np.random.default_rng(scale)
    hidden, S = 72, 7
    esz = torch.empty((), dtype=dtype).element_size()
    tb = hidden * esz
    lens = (rng.integers(1, 20, size=S) * scale).astype(np.int64)
    T = int(lens.sum())
    dev = lambda a: torch.from_numpy(a).to(cuda)
    do_shard = (rng.random((S, 3)) < 0.6).astype(np.int8)
    do_shard[0], do_shard[1] = 1, 0
    off = np.zeros((3, S), np.int64)
    cur = 16
    for c in range(3):
        for s in rng.permutation(S):
            off[c, s] = cur
            cur += int(lens[s]) * tb
    g = torch.Generator().manual_seed(scale)
    buf = torch.randn(cur // esz, generator=g).to(dtype).view(torch.uint8)
    planes = np.zeros((3, T, tb), np.uint8)
    fa2a.copy_cp(planes, buf.numpy(), do_shard, off, lens, False)
    want = torch.from_numpy(planes).view(dtype).reshape(3, T, hidden).double().sum(0)
    got = torch.full((T, hidden), float("nan"), dtype=dtype, device=cuda)
    print(f"replica sum {dtype} tokens {T}", flush=True)
    exchange([replica_sum_job(got, dev(do_shard), dev(off), dev(lens))], buf.to(cuda), False)
    torch.cuda.synchronize()
    if dtype == torch.float32:
        assert (got.cpu().double() - want).abs().max().item() <= 2 ** -22 * want.abs().max().item()
    else:
        assert torch.equal(got.cpu(), want.to(dtype))

    # shards 0 and 2 have copies (2 and 1) in shards 3, 4 and 5 of the same lengths
    lens[[3, 4]] = lens[0]
    lens[5] = lens[2]
    start = np.concatenate([[0], np.cumsum(lens)])
    T = int(start[-1])
    nc = np.array([2, 0, 1, 0, 0, 0, 0], np.int32)
    cs = np.zeros((S, 2), np.int64)
    cs[0], cs[2, 0] = start[[3, 4]], start[5]
    for mask in (np.array([1, 1, 1, 0, 0, 0, 1], np.int8), np.array([0, 1, 1, 0, 0, 0, 0], np.int8)):
        data = torch.randn((T, hidden), generator=g).to(dtype)
        boff, nbuf = _layout(rng, lens, tb)
        exp_t, exp = data.clone(), np.full(nbuf, 0x11, np.uint8)
        fa2a.grad_sum(exp_t, nc, cs, lens)
        fa2a.copy_non_cp(exp_t.view(torch.uint8).numpy(), exp, boff, lens, mask, True)
        d, dbuf = data.to(cuda), torch.full((nbuf,), 0x11, dtype=torch.uint8, device=cuda)
        exchange([copy_sum_job(d, dev(boff), dev(lens), dev(mask), dev(nc), dev(cs))], dbuf, True)
        torch.cuda.synchronize()
        assert torch.equal(d.cpu().view(torch.uint8), exp_t.view(torch.uint8)) and np.array_equal(dbuf.cpu().numpy(), exp)


REQUEST_FORMS = {
    "expanded": lambda t: t[:1].expand_as(t),                                       # what autograd hands on for a sum over tokens
    "one value": lambda t: t[:1, :1].expand_as(t),
    "overlapping": lambda t: t.reshape(-1).as_strided(t.shape, (16, 1)),
    "transposed": lambda t: t.t().contiguous().t(),
    "every other column": lambda t: t.repeat_interleave(2, dim=1)[:, ::2],
    "off alignment": lambda t: torch.cat([t.reshape(-1)[:1], t.reshape(-1)])[1:].view(t.shape),
    "odd pitch": lambda t: torch.cat([t, t[:, :1]], dim=1)[:, :t.shape[1]],
    "wide pitch": lambda t: torch.cat([t, t], dim=1)[:, :t.shape[1]],
}


@pytest.mark.parametrize("form", list(REQUEST_FORMS))
@pytest.mark.parametrize("which", range(4))
def test_request_tokens_from_any_strides(cuda, form, which):
    """The backward request with one of its parts in a form other than packed rows: the bytes of the token matrix, which takes any."""
    from distca_amd.dispatch import pre_a2a_attn_out_grad_resend_qkv, send_attn_out_grad_resend_qkv
    g = torch.Generator().manual_seed(5 + which)
    lens = [3, 0, 9, 1]
    T, hq, hkv, d = sum(lens), 4, 1, 128
    rnd = lambda n, dt=torch.bfloat16: torch.randn((T, n), generator=g).to(dt).to(cuda)
    parts = [rnd(hq * d), rnd(hq * d), rnd(hq, torch.float32).view(torch.uint8), rnd(hq * d)]
    parts[which] = REQUEST_FORMS[form](parts[which])
    k, v = rnd(hkv * d), rnd(hkv * d)
    i64 = lambda x: torch.tensor(x, dtype=torch.int64, device=cuda)
    tb, kb = 3 * hq * d * 2 + hq * 4, hkv * d * 2
    start = np.concatenate([[0], np.cumsum(lens)[:-1]])
    end = T * tb
    args = (k, v, torch.ones((len(lens), 1), dtype=torch.int8, device=cuda), i64(lens), i64(lens), i64(start * tb), i64(end + start * kb)[None],
            i64(end + T * kb + start * kb)[None])
    print(f"request with part {which} {form}: strides {parts[which].stride()}", flush=True)
    got, want = (torch.zeros(end + 2 * T * kb, dtype=torch.uint8, device=cuda) for _ in range(2))
    send_attn_out_grad_resend_qkv(*parts, *args, buffer=got)
    pre_a2a_attn_out_grad_resend_qkv(*parts, *args, buffer=want)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


@pytest.mark.parametrize("hq", [2016, 2020, 676, 680])
def test_tokens_either_side_of_what_a_launch_takes_apart(cuda, hq):
    """A launch puts tokens together from parts, or takes them apart, up to 512 KiB; larger ones pass as whole rows.  A reply holds
    260 bytes a head (2016: 524 160, 2020: 525 200), a request 772 (676: 521 872, 680: 524 960)."""
    from distca_amd.dispatch import post_a2a_attn_out_grad_resend_qkv, send_attn_out_grad_resend_qkv
    from distca_amd.fused_comm_attn import post_a2a_attn_out_with_lse
    from types import SimpleNamespace as NS
    g = torch.Generator().manual_seed(hq)
    lens, row = [1, 0, 2], hq * 256
    T = sum(lens)
    i64 = lambda x: torch.tensor(x, dtype=torch.int64, device=cuda)
    start = np.concatenate([[0], np.cumsum(lens)[:-1]])
    rows = lambda n: torch.randint(0, 256, (T, n), generator=g, dtype=torch.uint8)
    print(f"tokens of {hq} heads", flush=True)
    if hq > 2000:
        tb = (row + 4 * hq + 15) // 16 * 16
        reply = rows(tb)
        md = NS(tensor_shape=[NS(recv_shape=(T, tb // 2))], recv_memcpy_metadata=[i64(start * tb)], seq_lens=[NS(recv_seqlens=i64(lens))])
        out, lse = post_a2a_attn_out_with_lse(reply.reshape(-1).to(cuda), torch.empty((T, hq * 128), dtype=torch.bfloat16, device=cuda), hq, md)
        assert torch.equal(out.reshape(T, -1).view(torch.uint8).cpu(), reply[:, :row]) and torch.equal(lse.cpu(), reply[:, row:row + 4 * hq])
        return
    tb, kb = 3 * row + 4 * hq, 256
    parts = [rows(row), rows(row), rows(4 * hq), rows(row)]
    k, v = rows(kb), rows(kb)
    bf = lambda t: t.to(cuda).view(torch.bfloat16)
    ones = torch.ones((len(lens), 1), dtype=torch.int8, device=cuda)
    offs = [i64(start * tb), i64(T * tb + start * kb), i64(T * (tb + kb) + start * kb)]
    buf = torch.zeros(T * (tb + 2 * kb), dtype=torch.uint8, device=cuda)
    send_attn_out_grad_resend_qkv(bf(parts[0]), bf(parts[1]), parts[2].to(cuda), bf(parts[3]), bf(k), bf(v), ones, i64(lens), i64(lens), offs[0],
                                  offs[1][None], offs[2][None], buffer=buf)
    assert torch.equal(buf.cpu(), torch.cat([torch.cat(parts, dim=1).reshape(-1), k.reshape(-1), v.reshape(-1)]))
    rk, rv = (torch.empty((T, kb // 2), dtype=torch.bfloat16, device=cuda) for _ in range(2))
    got = post_a2a_attn_out_grad_resend_qkv([T, row // 2], [T, hq], [T, row // 2], torch.float32, rk, rv, None, i64(lens), i64(lens), *offs, True,
                                            buffer=buf)
    for t, want in zip(got, parts + [k, v]):
        assert torch.equal(t.view(torch.uint8).cpu(), want)


@pytest.mark.parametrize("max_cp,nshard,behind", [(0, 3, 0), (2, 0, 0), (0, 0, 5), (2, 3, 1), (2, 3, 9000), (1, 1, 700)])
def test_sums_over_no_replicas_are_zeros(cuda, max_cp, nshard, behind):
    """The gradients a rank gets back are sums over replicas: zeros for rows without a replica, with no shard at all, and behind the last
    shard (`behind` rows, in slices of their own and in one with shards), as the zeroed planes of a2a_memcpy_cp summed up."""
    from distca_amd.dispatch_fn import pre_all2all_layout_transfer_backward
    from distca_amd.ops import a2a_memcpy_cp
    from types import SimpleNamespace as NS
    rng = np.random.default_rng(behind + nshard)
    hidden, lens = 512, rng.integers(1, 40, size=nshard).astype(np.int64)
    covered = int(lens.sum()) if max_cp else 8
    T, tb = covered + behind, hidden * 2
    off = np.array([[c * covered * tb + int(lens[:s].sum()) * tb for s in range(nshard)] for c in range(max_cp)], np.int64).reshape(max_cp, nshard)
    mask = np.ones((nshard, max_cp), np.int8)
    mask[1:2] = 0
    dev = lambda a: torch.from_numpy(a).to(cuda)
    buf = torch.randn(max_cp * covered * hidden, device=cuda).to(torch.bfloat16).view(torch.uint8)
    poison = [torch.full((T, hidden), float("nan"), dtype=torch.bfloat16, device=cuda) for _ in range(4)]   # what the allocator hands out next
    torch.cuda.synchronize()
    del poison
    md = NS(tensor_shape=[NS(recv_shape=(0, hidden)), NS(recv_shape=(max_cp, T, hidden))], kv_replica_mask=dev(mask),
            recv_memcpy_metadata=[torch.zeros(0, dtype=torch.int64, device=cuda), dev(off), dev(off)],
            seq_lens=[NS(recv_seqlens=torch.zeros(0, dtype=torch.int64, device=cuda)), NS(recv_seqlens=dev(lens))])
    print(f"replica sums: {max_cp} replicas of {nshard} shards, {behind} rows behind them", flush=True)
    _, dk, dv = pre_all2all_layout_transfer_backward(md, torch.bfloat16, buffer=buf)
    planes = torch.zeros((max_cp, T, hidden), dtype=torch.bfloat16, device=cuda)
    a2a_memcpy_cp(planes, md.kv_replica_mask, dev(off), dev(lens), False, buffer=buf)
    torch.cuda.synchronize()
    assert dk.shape == dv.shape == (T, hidden) and torch.equal(dk, planes.sum(0)) and torch.equal(dv, planes.sum(0))


def test_gradients_without_copies_are_sent_as_they_are(cuda):
    """A table of copies without a column (no shard of the step has any): the main shards go out unchanged."""
    from distca_amd.dispatch import pre_a2a_qkv
    lens, hidden = [3, 2], 64
    T, tb = sum(lens), hidden * 2
    i64 = lambda x: torch.tensor(x, dtype=torch.int64, device=cuda)
    q, k, v = (torch.randn((T, hidden), device=cuda).to(torch.bfloat16) for _ in range(3))
    start = np.concatenate([[0], np.cumsum(lens)[:-1]]) * tb
    offs = [i64(start + i * T * tb) for i in range(3)]
    buf = torch.full((3 * T * tb,), 0x11, dtype=torch.uint8, device=cuda)
    copies = (torch.zeros(2, dtype=torch.int32, device=cuda), torch.zeros((2, 0), dtype=torch.int64, device=cuda))
    lens = i64(lens)
    print("no copies", flush=True)
    pre_a2a_qkv(q, k, v, None, lens, lens, *offs, is_fwd=False, kv_grad_copy_shard_mask=torch.tensor([1, 0], dtype=torch.int8, device=cuda),
                pre_a2a_grad_acc_args=(*copies, lens), buffer=buf)
    for i, (t, rows) in enumerate(((q, T), (k, 3), (v, 3))):
        part = buf[i * T * tb:(i + 1) * T * tb].view(T, tb)
        assert torch.equal(part[:rows], t.view(torch.uint8)[:rows]) and (part[rows:] == 0x11).all()


def test_copies_of_the_first_shards_alone(cuda):
    """Sums over copies for a leading part of the shards that are sent: their lengths are a view of the same memory as the sent shards'
    and must not be taken for them.  Shard 0 has its copy in shard 2; shards 1 and 2 lie behind the summed ones or have no copies."""
    from distca_amd.dispatch import pre_a2a_qkv
    lens, hidden = [3, 2, 3], 64
    T, tb = sum(lens), hidden * 2
    dev = lambda x, dt=torch.int64: torch.tensor(x, dtype=dt, device=cuda)
    g = torch.Generator().manual_seed(2)
    q, k, v = (torch.randn((T, hidden), generator=g).to(torch.bfloat16) for _ in range(3))
    start = np.concatenate([[0], np.cumsum(lens)[:-1]]) * tb
    nc, cs, mask = np.array([1, 0], np.int32), np.array([[5], [0]], np.int64), np.array([1, 1, 0], np.int8)
    want = [q.clone(), k.clone(), v.clone()]
    for t in want[1:]:
        fa2a.grad_sum(t, nc, cs, lens[:2])
    exp = np.full(3 * T * tb, 0x11, np.uint8)
    for i, t in enumerate(want):
        fa2a.copy_non_cp(t.view(torch.uint8).numpy(), exp, start + i * T * tb, lens, mask if i else None, True)
    d_lens, buf = dev(lens), torch.full((3 * T * tb,), 0x11, dtype=torch.uint8, device=cuda)
    print("copies of the first shards", flush=True)
    pre_a2a_qkv(q.to(cuda), k.to(cuda), v.to(cuda), None, d_lens, d_lens, *(dev(start + i * T * tb) for i in range(3)), is_fwd=False,
                kv_grad_copy_shard_mask=dev(mask, torch.int8), pre_a2a_grad_acc_args=(dev(nc, torch.int32), dev(cs), d_lens[:2]), buffer=buf)
    assert np.array_equal(buf.cpu().numpy(), exp)


def test_launches_go_to_the_current_stream(cuda):
    """The raw stream the pack calls are handed is torch's current one, the default stream's handle among them."""
    from distca_amd._lib import host
    from distca_amd.ops import on_stream
    side = torch.cuda.Stream()
    for s in (torch.cuda.current_stream(), side):
        with torch.cuda.stream(s):
            assert host().current_stream(cuda.index) == host().current_stream(-1) == (cuda.index, s.cuda_stream)
            assert on_stream(lambda *a: a, cuda, 1) == (1, s.cuda_stream) == on_stream(lambda *a: a, torch.device("cuda"), 1)


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs a second GPU")
def test_packing_into_the_memory_of_another_device(cuda):
    """A buffer that is another device's memory: the launch is one of the tensors' device and comes behind what made them there."""
    from distca_amd.dispatch import pre_a2a_qkv
    if not torch.cuda.can_device_access_peer(0, 1):
        pytest.skip("no peer access")
    T, hidden = 4096, 512
    tb = hidden * 2
    buf = torch.zeros(3 * T * tb, dtype=torch.uint8, device="cuda:1")
    buf.copy_(torch.zeros_like(buf, device=cuda))   # (makes the two devices peers)
    torch.cuda.synchronize(1)
    i64 = lambda x: torch.tensor(x, dtype=torch.int64, device=cuda)
    lens, ones = i64([T]), torch.ones((1, 1), dtype=torch.int8, device=cuda)
    torch.cuda._sleep(20_000_000)
    q, k, v = (torch.full((T, hidden), x, dtype=torch.bfloat16, device=cuda) for x in (1., 2., 3.))
    pre_a2a_qkv(q, k, v, ones, lens, lens, i64([0]), i64([[T * tb]]), i64([[2 * T * tb]]), is_fwd=True, buffer=buf)
    torch.cuda.current_stream(cuda).synchronize()
    assert torch.equal(buf.view(torch.bfloat16).view(3 * T, hidden).cpu(), torch.cat([q, k, v]).cpu())


@pytest.mark.parametrize("form", ["longer", "matrix"])
def test_lengths_of_a_plain_pack_in_other_shapes(cuda, form):
    """The queries' lengths on the way out may go on behind the shards that are placed, and be a matrix: a2a_memcpy_non_cp's terms."""
    from distca_amd.dispatch import pre_a2a_qkv
    lens, hidden = [3, 2, 4, 1], 64
    T, tb = sum(lens), hidden * 2
    i64 = lambda x: torch.tensor(x, dtype=torch.int64, device=cuda)
    q, k, v = (torch.randn((T, hidden), device=cuda).to(torch.bfloat16) for _ in range(3))
    start = np.concatenate([[0], np.cumsum(lens)[:-1]]) * tb
    q_lens = i64(lens + [7, 9]) if form == "longer" else i64(lens).view(2, 2)
    buf = torch.zeros(3 * T * tb, dtype=torch.uint8, device=cuda)
    print("lengths", form, flush=True)
    pre_a2a_qkv(q, k, v, torch.ones((4, 1), dtype=torch.int8, device=cuda), q_lens, i64(lens), i64(start), i64(start + T * tb)[None],
                i64(start + 2 * T * tb)[None], is_fwd=True, buffer=buf)
    assert torch.equal(buf, torch.cat([q, k, v]).view(torch.uint8).view(-1))
