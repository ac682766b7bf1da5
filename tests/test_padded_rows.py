"""Padded batches where they lie: boundaries as (first row, one past the last) pairs, rows in between that belong to no sequence."""
import pytest
import torch

from tests import emu_util

D = 128
SCALE = D ** -0.5


def reference(q1, k1, v1, q2, k2, v2, pos2, g1, g2):
    """One sequence in float64 with the dense rule: outputs and gradients."""
    x = [t.double().requires_grad_(True) for t in (q1, k1, v1, q2, k2, v2)]
    a, b, c, d, e, f = x
    group = a.shape[1] // b.shape[1]
    at = torch.arange(a.shape[0], device=a.device)
    wide = lambda t: t.repeat_interleave(group, 1)

    def attend(q, k, v, seen):
        s = torch.einsum("qhd,khd->hqk", q, wide(k)) * SCALE
        return torch.einsum("hqk,khd->qhd", torch.softmax(s.masked_fill(~seen, float("-inf")), -1), wide(v))

    outs = [attend(a, b, c, at[None] <= at[:, None])]
    if pos2.numel():
        outs.append(attend(d, torch.cat([b, e]), torch.cat([c, f]), torch.cat([at, pos2])[None] <= pos2[:, None]))
    else:
        outs.append(d * 0.0)
    return [t.detach() for t in outs] + list(torch.autograd.grad(outs, x, (g1.double(), g2.double()), allow_unused=True))


def run_case(dev, hq, hkv, lens, lead, T, hard, paired2, exchange):
    """Rows of B x T blocks, sequence b at lead[b] ... lead[b] + lens[b], NaN everywhere else."""
    from tah_amd import ops
    from tah_amd.attention import duo_attn_varlen

    g = torch.Generator().manual_seed(sum(lens))
    B = len(lens)

    def block(counts, at, heads, width):
        rows = torch.full((B, width, heads, D), float("nan"), dtype=torch.bfloat16)
        for b, n in enumerate(counts):
            rows[b, at[b]:at[b] + n] = (torch.randn(n, heads, D, generator=g) * 0.5).to(torch.bfloat16)
        return rows

    pos = [torch.randperm(n, generator=g)[:max(0, round(hard * n))].sort().values for n in lens]
    n2 = [len(p) for p in pos]
    W = max(n2) + 3
    lead2 = [2] * B if paired2 else [0] * B
    t1 = [block(lens, lead, h, T) for h in (hq, hkv, hkv, hq)]
    t2 = [block(n2, lead2, h, W) for h in (hq, hkv, hkv, hq)]
    pairs1 = torch.tensor([[b * T + lead[b], b * T + lead[b] + n] for b, n in enumerate(lens)], dtype=torch.int32).flatten()
    if paired2:
        pairs2 = torch.tensor([[b * W + 2, b * W + 2 + n] for b, n in enumerate(n2)], dtype=torch.int32).flatten()
        p2 = torch.full((B, W), -7, dtype=torch.int32)
        for b, p in enumerate(pos):
            p2[b, 2:2 + len(p)] = p.int()
        flat2 = [t.view(B * W, -1, D) for t in t2]
        p2 = p2.flatten()
    else:
        pairs2 = torch.tensor([0] + torch.tensor(n2).cumsum(0).tolist(), dtype=torch.int32)
        flat2 = [torch.cat([t[b, :n] for b, n in enumerate(n2)]) for t in t2]
        p2 = torch.cat(pos).int()
    flat1 = [t.view(B * T, -1, D) for t in t1]
    bits = 3 + (12 if paired2 else 0)
    on = lambda t: t.clone().to(dev)
    q1, k1, v1, g1 = map(on, flat1)
    q2, k2, v2, g2 = map(on, flat2)
    pairs1, pairs2, p2 = on(pairs1), on(pairs2), on(p2)
    leaves = [t.requires_grad_(True) for t in (q1, k1, v1, q2, k2, v2)]
    sched = ops.duo_schedule(pairs1, pairs1, pairs2, pairs2, p2, hq, hkv, B * T, B * T, k2.shape[0], bits)
    was, ops.DS_EXCHANGE = ops.DS_EXCHANGE, exchange
    try:
        o = duo_attn_varlen(q1, k1, v1, pairs1, pairs1, q2, k2, v2, p2, p2, pairs2, pairs2, SCALE, schedule=sched, max_seqlen_k1=T,
                            max_seqlen_k2=W, pairs=bits)
        got = list(o) + list(torch.autograd.grad(o, leaves, (g1, g2)))
    finally:
        ops.DS_EXCHANGE = was
    got = [t.detach().cpu() for t in got]
    streams = [0, 1, 0, 0, 0, 1, 1, 1]  # of o1, o2, dq1, dk1, dv1, dq2, dk2, dv2
    wants = [reference(*[t[b, lead[b]:lead[b] + lens[b]].to(dev) for t in t1[:3]], *[t[b, lead2[b]:lead2[b] + n2[b]].to(dev) for t in t2[:3]],
                       pos[b].to(dev), t1[3][b, lead[b]:lead[b] + lens[b]].to(dev), t2[3][b, lead2[b]:lead2[b] + n2[b]].to(dev)) for b in range(B)]
    for i, (t, stream) in enumerate(zip(got, streams)):
        diff = ref = 0.0
        if stream == 0 or paired2:
            rows, at, counts = t.view(B, T if stream == 0 else W, -1, D), (lead if stream == 0 else lead2), (lens if stream == 0 else n2)
            parts = [rows[b, at[b]:at[b] + n] for b, n in enumerate(counts)]
            for b, n in enumerate(counts):  # rows of no sequence: zeros, whatever lies there in the inputs
                assert (rows[b, :at[b]] == 0).all() and (rows[b, at[b] + n:] == 0).all(), i
        else:
            parts = t.split(n2)
        for part, want in zip(parts, wants):
            if part.numel() == 0 or want[i] is None:
                continue
            w = want[i].cpu()
            diff += float((part.double() - w).square().sum())
            ref += float(w.square().sum())
        # bf16 operands, probabilities and results (2^-9 each): the tolerance the other attention tests have
        assert diff <= (0.013 ** 2) * ref + 1e-9, (i, diff, ref)


CASES = [
    # hq, hkv, lens, first row of each, T, hard, depth-1 rows padded too
    (2, 1, [70, 1, 33], [0, 0, 0], 70, 0.2, False),      # right-padded, one row alone
    (2, 2, [65, 40], [5, 30], 70, 0.3, True),            # left-padded, both streams
    (4, 1, [129, 64], [0, 65], 129, 0.1, False),         # one key past a tile, four heads to a group
]


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
@pytest.mark.parametrize("case", CASES[:2])
def test_padded_rows_emu(case):
    with emu_util.emulated():
        run_case("cpu", *case, exchange=True)


@pytest.mark.gpu
@pytest.mark.parametrize("exchange", [True, False])
@pytest.mark.parametrize("case", CASES + [(16, 8, [700, 1300, 5], [0, 0, 11], 1300, 0.1, False), (8, 1, [200, 130], [0, 70], 200, 0.2, True)])
def test_padded_rows_gpu(case, exchange):
    run_case("cuda", *case, exchange=exchange)


def check_attention_blocks(dev):
    """The callable on a padded batch: where the rows lie, against the same rows alone; what lies in the pads, and rows whose
    strides or address the kernels do not take, change nothing."""
    import types

    from tah_amd.attention import _Packed, build_attention_mask, duo_attention_forward
    from tah_amd.cache import TaHDuoCache

    g = torch.Generator().manual_seed(3)
    B, T, hq, hkv, lens = 2, 40, 2, 1, [40, 23]

    def loop(valid, q, k, v):
        valid = valid.to(dev)
        pos = (valid.long().cumsum(-1) - 1).clamp(min=0)
        cache = TaHDuoCache()
        mask = build_attention_mask(pos, valid, cache, 0)
        cache.current_iter_depth, cache.position_ids_to_cache, cache.valid_mask_to_cache = 0, pos, valid
        kk, vv = cache.update(k, v, 0)
        return duo_attention_forward(types.SimpleNamespace(layer_idx=0), q, kk, vv, mask, scaling=SCALE)[0], mask

    valid = torch.arange(T)[None] < torch.tensor(lens)[:, None]
    x = [(torch.randn(B, T, h, D, generator=g) * 0.5).to(torch.bfloat16).to(dev) for h in (hq, hkv, hkv)]
    got, mask = loop(valid, *[t.transpose(1, 2) for t in x])
    assert mask._packed.paired and mask._packed.rows is None
    dirty = [t.clone() for t in x]
    for t in dirty:
        t[1, 23:] = float("inf")
    again, _ = loop(valid, *[t.transpose(1, 2) for t in dirty])
    assert torch.equal(got, again) and (got[1, 23:] == 0).all()
    for b, n in enumerate(lens):
        alone, _ = loop(torch.ones(1, n, dtype=torch.bool), *[t[b:b + 1, :n].transpose(1, 2) for t in x])
        assert torch.equal(got[b, :n], alone[0])
    odd = []
    for t in x:  # rows 4 elements into a buffer, 12 more between heads
        buf = torch.zeros(B * T * t.shape[2] * (D + 12) + 4, dtype=torch.bfloat16, device=dev)[4:].view(B, T, t.shape[2], D + 12)
        buf[..., :D] = t
        odd.append(buf[..., :D].transpose(1, 2))
    again, _ = loop(valid, *odd)
    assert torch.equal(got, again)
    # a hole, or mostly padding: packed as before
    holes = valid.clone()
    holes[0, 7] = False
    assert not _Packed(holes.to(dev), None, B, T, dev).paired
    thin = torch.arange(T)[None] < torch.tensor([9, 20])[:, None]
    assert not _Packed(thin.to(dev), None, B, T, dev).paired


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_attention_blocks_emu(monkeypatch):
    from tah_amd import attention
    monkeypatch.setattr(attention, "NO_SYNC_ROWS", 0)
    with emu_util.emulated():
        check_attention_blocks("cpu")


@pytest.mark.gpu
def test_attention_blocks_gpu(monkeypatch):
    from tah_amd import attention
    monkeypatch.setattr(attention, "NO_SYNC_ROWS", 0)
    check_attention_blocks("cuda")


def check_rows_select(dev):
    """Rows by a table against torch's indexing, for row lengths at the edges of a wave's share (16-byte pieces: 31, 32, 33, 256, 257),
    rows that 16 bytes do not divide, a count on the device, and sources whose rows are apart or not contiguous."""
    from tah_amd import ops

    g = torch.Generator().manual_seed(5)
    n, rows = 37, 75
    index = torch.randint(-1, n, (rows,), generator=g, dtype=torch.int32)
    srcs = [torch.randint(0, 255, (n, w), generator=g, dtype=torch.uint8) for w in (1, 16 * 31, 16 * 32, 16 * 33, 16 * 257, 1000)]
    srcs[2], srcs[3] = [torch.randint(0, 255, shape, generator=g, dtype=torch.uint8) for shape in ((n, 16 * 40), (16 * 33, n))]
    dense = [s.to(dev) for s in srcs]
    dense[2], dense[3] = dense[2][:, :16 * 32], dense[3].t()
    srcs[2], srcs[3] = srcs[2][:, :16 * 32], srcs[3].t()
    want = [torch.where(index[:, None] >= 0, s[index.clamp(min=0).long()], torch.zeros_like(s[:1])) for s in srcs]
    for got, w in zip(ops.rows_select(dense, index.to(dev), rows), want):
        assert torch.equal(got.cpu(), w)
    some = ops.rows_select(dense, index.to(dev), rows, torch.tensor([50], dtype=torch.int32, device=dev))
    for got, w in zip(some, want):
        assert torch.equal(got[:50].cpu(), w[:50])
    nothing = ops.rows_select([dense[0][:0]], torch.full((9,), -1, dtype=torch.int32, device=dev), 9)[0]
    assert nothing.shape == (9, 1) and (nothing == 0).all()


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_rows_select_emu():
    with emu_util.emulated():
        check_rows_select("cpu")


@pytest.mark.gpu
def test_rows_select_gpu():
    check_rows_select("cuda")


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_gathered_tensors_want_gradients_as_before():
    """Of several tensors packed together only those that want a gradient hand one on."""
    from tah_amd.pack import gather_active

    with emu_util.emulated():
        g = torch.Generator().manual_seed(1)
        mask = torch.rand(3, 11, generator=g) < 0.4
        x, y = torch.randn(3, 11, 4, generator=g, requires_grad=True), torch.randn(3, 11, 4, generator=g)
        pad, gx, gy, ids = gather_active(mask, x, y, torch.arange(33).view(3, 11))
        assert gx.requires_grad and not gy.requires_grad and not ids.requires_grad
        w = torch.randn(gx.shape, generator=g)
        (gx * w).sum().backward()
        want = torch.zeros(3, 11, 4)
        for b in range(3):
            want[b, mask[b]] = w[b, :int(mask[b].sum())]
        assert torch.equal(x.grad, want)


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_gathered_tensors_have_gradients_of_their_own():
    """Tensors packed together stay apart for autograd: one backward leaves the others' gradients alone and frees nothing of theirs,
    and forward mode is refused as by any node that has no rule for it."""
    import torch.autograd.forward_ad as fwd

    from tah_amd.pack import gather_active

    with emu_util.emulated():
        g = torch.Generator().manual_seed(2)
        mask = torch.rand(3, 11, generator=g) < 0.4
        x, y = [torch.randn(3, 11, 4, generator=g, requires_grad=True) for _ in range(2)]
        want = mask[..., None].expand(3, 11, 4).float()
        pad, gx, gy, ids = gather_active(mask, x, y, torch.arange(33).view(3, 11))
        gx.sum().backward()
        assert torch.equal(x.grad, want) and y.grad is None
        gy.sum().backward()
        assert torch.equal(y.grad, want) and torch.equal(x.grad, want)
        gx = gather_active(mask, x)[1]
        gx *= 2.0  # (a result of its own, not a view of anything)
        assert torch.equal(torch.autograd.grad(gx.sum(), x)[0], 2.0 * want)
        with fwd.dual_level(), pytest.raises(RuntimeError):
            gather_active(mask, fwd.make_dual(x.detach(), torch.ones_like(x)))


def check_workspace_of_padded_blocks(dev, monkeypatch, lens, left, hq, hkv):
    """dS of a padded block in place: blocks for the rows that exist and no others, none written behind them, and the gradients of the
    same block packed, to the bit."""
    import types

    from tah_amd import attention as A, ops
    from tah_amd.cache import TaHDuoCache

    g = torch.Generator().manual_seed(sum(lens))
    B, T = len(lens), max(lens)
    at, n = torch.arange(T)[None], torch.tensor(lens)[:, None]
    valid = ((at >= T - n) if left else (at < n)).to(dev)
    x = [(torch.randn(B, T, h, D, generator=g) * 0.5).to(torch.bfloat16).to(dev) for h in (hq, hkv, hkv, hq)]
    asked = []

    def buffer(device, nbytes):
        whole = torch.full((nbytes + 65536,), 171, dtype=torch.uint8, device=device)
        asked.append((nbytes, whole))
        return whole[:nbytes]

    monkeypatch.setattr(ops, "_ds_workspace", buffer)
    monkeypatch.setattr(A, "NO_SYNC_ROWS", 0)
    results = []
    for paired in (True, False):
        v = valid.clone()
        pos = (v.long().cumsum(-1) - 1).clamp(min=0)
        if not paired:
            A.HardIndex.of(v).intervals = None
        t = [a.clone().requires_grad_(True) for a in x[:3]]
        cache = TaHDuoCache()
        mask = A.build_attention_mask(pos, v, cache, 0)
        cache.current_iter_depth, cache.position_ids_to_cache, cache.valid_mask_to_cache = 0, pos, v
        kk, vv = cache.update(t[1].transpose(1, 2), t[2].transpose(1, 2), 0)
        o = A.duo_attention_forward(types.SimpleNamespace(layer_idx=0), t[0].transpose(1, 2), kk, vv, mask, scaling=SCALE)[0]
        assert mask._packed.paired == paired
        results.append([o.detach()] + list(torch.autograd.grad(o, t, x[3])))
    assert len(asked) == 2 and asked[0][0] == asked[1][0] > 0
    assert all((whole[nbytes:] == 171).all() for nbytes, whole in asked)
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
@pytest.mark.parametrize("lens,left,hq,hkv", [([130, 70, 66], False, 2, 1), ([65, 33], True, 1, 1)])
def test_workspace_of_padded_blocks_emu(monkeypatch, lens, left, hq, hkv):
    with emu_util.emulated():
        check_workspace_of_padded_blocks("cpu", monkeypatch, lens, left, hq, hkv)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,left,hq,hkv", [([1000, 520, 513, 600], False, 16, 8), ([400] + [210] * 69, True, 4, 1)])
def test_workspace_of_padded_blocks_gpu(monkeypatch, lens, left, hq, hkv):
    check_workspace_of_padded_blocks("cuda", monkeypatch, lens, left, hq, hkv)
