"""Linear layers of a decode step on packed operands (tah_linear_pack_weight / tah_linear_pack_rows / tah_linear_rows).

The packed orders are checked element by element against the layout the header documents; the products against
float64 sums of the same bf16 inputs with the roundings the eager modules make (nn.Linear output in bf16, residual
add in bf16, ``act_fn(gate) * up`` of Qwen3MLP.forward with each step in bf16).  Tolerance: the float32 sums run in a
different order from the float64 ones, so a result may land on the neighbouring bf16 value -- 2^-7 relative, and
most elements have to agree exactly.  The CPU tests run the kernels on the CPU execution shim; the GPU tests call the
library through the extension and through ctypes.
"""
import contextlib
import ctypes

import numpy as np
import pytest
import torch

from tests import emu_util

BF = torch.bfloat16


def _rand(shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(BF)


def weight_row_of_slot(n, gate_up, tile, c):
    """Row of the [n, k] (or [2n, k]) weight that sits in column slot c of tile `tile` of the packed order."""
    if not gate_up:
        return 16 * tile + c
    if n % 24 == 0:  # groups of 24 output columns, three tiles: gate 0-15 | gate 16-23, up 16-23 | up 0-15
        g, t = divmod(tile, 3)
        if t == 0:
            return 24 * g + c
        if t == 2:
            return n + 24 * g + c
        return 24 * g + 16 + c if c < 8 else n + 24 * g + 16 + (c - 8)
    g, t = divmod(tile, 2)  # groups of 16 output columns: gate tile, up tile
    return (n if t else 0) + 16 * g + c


def unpack_weight(packed, n, k, gate_up):
    """Inverse of the packed order, written from its description: [tiles][k / 32][64 lanes][8]."""
    total = 2 * n if gate_up else n
    p = packed.view(total // 16, k // 32, 64, 8)
    w = torch.empty(total, k, dtype=packed.dtype)
    for tile in range(total // 16):
        for c in range(16):
            row = weight_row_of_slot(n, gate_up, tile, c)
            # lanes c, c + 16, c + 32, c + 48 hold k = 0-7, 8-15, 16-23, 24-31 of every step
            w[row] = p[tile, :, c::16, :].reshape(k)
    return w


def unpack_rows(packed, k):
    """[k / 32][2][64][8] -> [32, k]"""
    p = packed.view(k // 32, 2, 64, 8)
    x = torch.empty(32, k, dtype=packed.dtype)
    for half in range(2):
        for r in range(16):
            x[16 * half + r] = p[:, half, r::16, :].reshape(k)
    return x


def reference(x, w, *, residual=None, gate_up=False, norm_eps=None, bias=None, relu=False, gelu=False, layer_norm=False):
    """float64 sums with the eager modules' bf16 roundings.  ``layer_norm``: the rows go through a LayerNorm without
    scale and shift first (those sit in w and bias), written as the library routine, not as the kernel's fold."""
    xd, wd = x.double(), w.double()
    r = torch.rsqrt((xd ** 2).mean(-1, keepdim=True) + norm_eps) if norm_eps is not None and not layer_norm else 1.0
    if layer_norm:
        xd = torch.nn.functional.layer_norm(xd, xd.shape[-1:], eps=norm_eps)
    if not gate_up:
        y = (r * (xd @ wd.t())).to(BF)
        if bias is not None:
            y = (y.double() + bias.double()).to(BF)
        if residual is not None:
            y = (y.double() + residual.double()).to(BF)
        if gelu:
            return torch.nn.functional.gelu(y.double()).to(BF)
        return torch.relu(y) if relu else y
    n = w.shape[0] // 2
    g = (r * (xd @ wd[:n].t())).to(BF).double()
    u = (r * (xd @ wd[n:].t())).to(BF).double()
    act = (g / (1.0 + torch.exp(-g))).to(BF).double()
    return (act * u).to(BF)


def _close(got, want, exact_share=0.97):
    got, want = got.float(), want.float()
    assert torch.allclose(got, want, rtol=2.0 ** -7, atol=2.0 ** -9), (got - want).abs().max()
    assert (got == want).float().mean() >= exact_share


def _pack_checks(dev):
    from tah_amd import ops
    for n, k, gu in ((48, 96, False), (32, 64, True), (48, 64, True)):
        w = _rand(((2 if gu else 1) * n, k), 3 + n)
        packed = ops.linear_pack_weight(w.to(dev), gate_up=gu).cpu()
        assert packed.shape == (w.numel(),)
        assert torch.equal(unpack_weight(packed, n, k, gu), w)
    # a weight that is a view with a row stride of its own
    big = _rand((32, 256), 9)
    assert torch.equal(unpack_weight(ops.linear_pack_weight(big.to(dev)[:, 64:192]).cpu(), 32, 128, False), big[:, 64:192])
    for rows in (32, 17, 1, 0):
        x = _rand((rows, 160), 5 + rows)
        xp = ops.linear_pack_rows(x.to(dev)).cpu()
        full = unpack_rows(xp, 160)
        assert torch.equal(full[:rows], x) and not full[rows:].any()


CASES = [
    # rows, n, k, kind
    (32, 48, 96, "plain"),       # 3 steps over 8 waves: most waves have no step
    (7, 32, 1024, "residual"),   # 4 steps per wave, any-K kernel
    (17, 16, 2048, "residual"),  # K known at compile time (8 steps per wave)
    (32, 16, 6144, "plain"),     # 24 steps per wave, three chunks
    (20, 32, 352, "plain"),      # 11 steps: uneven shares
    (32, 96, 2048, "gate_up_norm"),   # 24-column groups
    (9, 32, 2048, "gate_up_norm"),    # 16-column groups
    (32, 24, 320, "gate_up"),         # 24-column groups, any K, no norm
    (5, 16, 96, "gate_up_norm"),      # 16-column groups, any K
    # more than 128 column groups: a workgroup takes all 32 rows (below, and up to 16 rows, it takes 16)
    (20, 2080, 96, "residual"),
    (32, 3120, 64, "gate_up_norm"),
    (9, 48, 2048, "plain_norm"),      # an RMSNorm of the rows folded in (an output head behind the final norm)
    (32, 32, 160, "plain_norm"),
    (11, 32, 2048, "bias_relu_norm"),  # first layer of a small MLP behind a folded norm (the decider)
    (32, 48, 96, "bias_relu"),
    (32, 64, 256, "bias_gelu_ln"),     # a layer behind a LayerNorm, GELU last (the learned decider's blocks)
    (13, 2048, 512, "bias_gelu_ln"),   # sixteen rows per workgroup
    (32, 2080, 96, "bias_ln"),         # all 32 rows per workgroup
    (5, 16, 1280, "bias_gelu"),
]


def _linear_case(dev, rows, n, k, kind, seed=0):
    from tah_amd import ops
    gu = kind.startswith("gate_up")
    x = _rand((rows, k), 11 + seed, 1.5)
    w = _rand(((2 if gu else 1) * n, k), 12 + seed, k ** -0.5)
    res = _rand((rows, n), 13 + seed) if kind == "residual" else None
    eps = 1e-6 if kind.endswith("_norm") else None
    bias = _rand((n,), 14 + seed) if kind.startswith("bias") else None
    relu, gelu, ln = "relu" in kind, "gelu" in kind, kind.endswith("_ln")
    if ln:  # rows with a mean of their own, so that a fold that forgets it fails
        x = (x.float() * 0.7 + 0.9 * torch.arange(rows).view(-1, 1) / max(rows, 1) - 0.4).to(BF)
        eps = 1e-5
    want = reference(x, w, residual=res, gate_up=gu, norm_eps=eps, bias=bias, relu=relu, gelu=gelu, layer_norm=ln)
    extra = dict(bias=bias.to(dev), relu=relu, gelu=gelu) if bias is not None else {}
    if ln:
        extra["ln_colsum"] = w.float().sum(-1).to(dev)
    wp = ops.linear_pack_weight(w.to(dev), gate_up=gu)
    xp = ops.linear_pack_rows(x.to(dev))
    yp = torch.full((32 * n,), 7.0, dtype=BF, device=dev) if n % 32 == 0 else None  # the packed form holds whole steps of 32
    if res is not None:  # in place on the residual, as the engine calls it
        h = res.clone().to(dev)
        got = ops.linear_rows(wp, xp, rows, n, k, residual=h, out=h, out_packed=yp)
        assert got.data_ptr() == h.data_ptr()
    else:
        got = ops.linear_rows(wp, xp, rows, n, k, gate_up=gu, out_packed=yp, norm_eps=eps, **extra)
        if relu:
            assert (got.float() >= 0).all() and (got == 0).any()
    got = got.cpu()
    _close(got, want)
    if yp is not None:
        full = unpack_rows(yp.cpu(), n)
        assert torch.equal(full[:rows], got) and not full[rows:].any()   # the packed copy, zero past the last row
        # packed result only
        yp2 = torch.empty_like(yp)
        h2 = res.clone().to(dev) if res is not None else None
        assert ops.linear_rows(wp, xp, rows, n, k, gate_up=gu, residual=h2, out_packed=yp2, want_out=False, norm_eps=eps, **extra) is None
        assert torch.equal(yp2, yp)
    # twice the same: sums run in a fixed order
    again = ops.linear_rows(wp, xp, rows, n, k, gate_up=gu, residual=res.to(dev) if res is not None else None, norm_eps=eps, **extra)
    assert torch.equal(again.cpu(), got)


def _error_checks(dev):
    from tah_amd import ops
    from tah_amd._capi import TahDuoError
    w = _rand((32, 64), 1).to(dev)
    wp = ops.linear_pack_weight(w)
    xp = ops.linear_pack_rows(_rand((4, 64), 2).to(dev))
    with pytest.raises((TahDuoError, RuntimeError)):
        ops.linear_pack_weight(_rand((24, 64), 1).to(dev))            # n % 16
    with pytest.raises((TahDuoError, RuntimeError)):
        ops.linear_pack_weight(_rand((32, 48), 1).to(dev))            # k % 32
    with pytest.raises((TahDuoError, RuntimeError)):
        ops.linear_pack_rows(_rand((33, 64), 1).to(dev))              # more than 32 rows
    with pytest.raises((TahDuoError, RuntimeError)):
        ops.linear_rows(wp, xp, 33, 32, 64)
    with pytest.raises((TahDuoError, RuntimeError)):
        ops.linear_rows(wp, xp, 4, 32, 32)                            # sizes the operands were not packed for
    with pytest.raises((TahDuoError, RuntimeError)):
        ops.linear_rows(wp, xp, 4, 32, 64, norm_eps=1e-5, ln_colsum=torch.zeros(16, device=dev))   # one sum per output column
    with pytest.raises((TahDuoError, RuntimeError)):
        ops.linear_rows(wp, xp, 4, 16, 64, gate_up=True, norm_eps=1e-5, ln_colsum=torch.zeros(16, device=dev))  # no LayerNorm with the gate
    with pytest.raises((TahDuoError, RuntimeError)):
        ops.linear_rows(wp, xp, 4, 16, 64, gate_up=True, residual=_rand((4, 16), 3).to(dev))  # no residual with the gate
    w48 = ops.linear_pack_weight(_rand((48, 64), 4).to(dev))
    with pytest.raises((TahDuoError, RuntimeError)):
        ops.linear_rows(w48, xp, 4, 48, 64, out_packed=torch.empty(32 * 48, dtype=BF, device=dev))  # 48 is not whole steps of 32
    assert ops.linear_rows(wp, xp, 0, 32, 64).shape == (0, 32)


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_packed_orders_on_cpu_shim():
    with emu_util.emulated():
        _pack_checks("cpu")
        _error_checks("cpu")


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
@pytest.mark.parametrize("rows,n,k,kind", CASES)
def test_linear_rows_on_cpu_shim(rows, n, k, kind):
    with emu_util.emulated():
        _linear_case("cpu", rows, n, k, kind)


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_c_abi_refuses_bad_arguments():
    from tah_amd import _capi
    with emu_util.emulated() as lib:
        a = _capi.LinearRowsArgs()
        assert lib.tah_linear_rows(None, None) < 0
        buf = (ctypes.c_uint16 * (32 * 64))()
        addr = ctypes.addressof(buf)
        a.w_packed, a.x_packed, a.out, a.out_row_stride = addr, addr, addr, 32
        a.rows, a.n, a.k, a.kind = 4, 32, 64, 0
        a.rows = 33
        assert lib.tah_linear_rows(ctypes.byref(a), None) < 0
        a.rows, a.n = 4, 24
        assert lib.tah_linear_rows(ctypes.byref(a), None) < 0
        a.n, a.k = 32, 40
        assert lib.tah_linear_rows(ctypes.byref(a), None) < 0
        a.k, a.kind = 64, 5
        assert lib.tah_linear_rows(ctypes.byref(a), None) < 0
        a.kind, a.out = 0, None
        assert lib.tah_linear_rows(ctypes.byref(a), None) < 0          # nothing to write
        a.out, a.x_packed = addr, addr + 2
        assert lib.tah_linear_rows(ctypes.byref(a), None) < 0          # alignment


# ── GPU ──────────────────────────────────────────────────────────────────────────────────────────────────────
@pytest.mark.gpu
def test_packed_orders_gpu():
    _pack_checks("cuda")
    _error_checks("cuda")


# Few rows, K known at compile time: eight columns per workgroup (few column groups), rows past the last one read as row 0.
FEW = [(1, 32, 2048, "residual"), (8, 48, 2048, "plain"), (9, 16, 2048, "residual"), (3, 16, 4096, "residual"), (16, 32, 6144, "residual"),
       (8, 2064, 2048, "plain"), (5, 24, 2048, "gate_up_norm"), (8, 16, 2048, "plain_norm"),
       # one, two, four and eight rows' operand folded into a load, a row fewer, and the last load's steps past the end (24 of 32)
       (1, 16, 6144, "residual"), (2, 32, 6144, "residual"), (3, 16, 2048, "plain_norm"), (4, 32, 6144, "residual"), (7, 16, 6144, "residual"),
       (1, 16, 2048, "plain_norm"), (2, 48, 2048, "plain_norm")]


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
@pytest.mark.parametrize("rows,n,k,kind", [c for c in FEW if c[1] < 100])
def test_linear_rows_of_few_rows_on_cpu_shim(rows, n, k, kind):
    with emu_util.emulated():
        _linear_case("cpu", rows, n, k, kind)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,k,kind", FEW + [
    # (without a residual: added to products of up to 4, which the sum's order may move by one bf16 step of 2^-6, it can cancel
    # them to a value whose own step is finer than that move)
    (1, 2048, 2048, "plain"), (16, 2048, 6144, "plain"), (4, 6144, 2048, "gate_up_norm"),
    # more than sixteen rows of an output head: a resident workgroup per compute unit, one, two or three column groups each
    (17, 16384, 2048, "plain"), (32, 16416, 2048, "plain_norm"), (24, 32000, 2048, "plain"), (31, 151936, 2048, "plain_norm")])
def test_linear_rows_of_few_rows_and_output_heads_gpu(rows, n, k, kind):
    _linear_case("cuda", rows, n, k, kind, seed=n % 5)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,k,kind", CASES + [
    (32, 4096, 2048, "plain"), (32, 2048, 2048, "residual"), (32, 6144, 2048, "gate_up_norm"), (32, 2048, 6144, "residual"),
    (13, 1024, 3072, "residual"), (32, 2560, 2560, "plain"), (32, 1600, 1024, "gate_up_norm"),
    (32, 151936, 2048, "plain_norm"), (32, 16384, 512, "plain"), (20, 32000, 1024, "plain_norm"),   # output heads: 32 columns per workgroup
])
def test_linear_rows_gpu(rows, n, k, kind):
    _linear_case("cuda", rows, n, k, kind, seed=n % 7)


@pytest.mark.gpu
def test_linear_rows_through_the_c_abi_gpu():
    """The same call through ctypes, on the library itself."""
    from tah_amd import _capi, _lib, ops
    lib = _capi.bind(ctypes.CDLL(_lib.LIB_PATH))
    rows, n, k = 32, 64, 2048
    x, w, res = _rand((rows, k), 1), _rand((n, k), 2, k ** -0.5), _rand((rows, n), 3)
    dx, dw, h = x.cuda(), w.cuda(), res.clone().cuda()
    wp = torch.empty(n * k, dtype=BF, device="cuda")
    xp = torch.empty(32 * k, dtype=BF, device="cuda")
    yp = torch.empty(32 * n, dtype=BF, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    assert lib.tah_linear_pack_weight(dw.data_ptr(), k, wp.data_ptr(), n, k, _capi.LINEAR_PLAIN, st) == 0
    assert lib.tah_linear_pack_rows(dx.data_ptr(), k, xp.data_ptr(), rows, k, st) == 0
    a = _capi.LinearRowsArgs()
    a.w_packed, a.x_packed, a.residual, a.out, a.out_packed = wp.data_ptr(), xp.data_ptr(), h.data_ptr(), h.data_ptr(), yp.data_ptr()
    a.residual_row_stride = a.out_row_stride = n
    a.rows, a.n, a.k, a.kind = rows, n, k, _capi.LINEAR_PLAIN
    assert lib.tah_linear_rows(ctypes.byref(a), st) == 0
    torch.cuda.synchronize()
    _close(h.cpu(), reference(x, w, residual=res))
    assert torch.equal(unpack_rows(yp.cpu(), n), h.cpu())
    assert torch.equal(ops.linear_pack_weight(dw), wp) and torch.equal(ops.linear_pack_rows(dx), xp)


# ── the linear layers between two attentions in one launch (tah_linear_chain) ──
# rows on both sides of each of its kernels' row counts; q|k|v narrower than the other phases; without q|k|v
CHAIN_CASES = [(1, 4096, False), (2, 4096, True), (3, 16, False), (4, 0, True), (5, 4096, True), (8, 4096, False), (8, 0, False)]


def _chain_case(dev, rows, hidden, o_cols, ff, n_qkv, views, launches=2, polls=0):
    """Against the four ``linear_rows`` launches: the same bits (512 columns, on the CPU only: ``linear_rows`` adds even and odd steps
    up together there, a neighbouring bf16 value).  ``views``: row-major tensors with strides of their own."""
    from tah_amd import ops
    same = torch.equal if hidden == 2048 else lambda a, b: torch.allclose(a.float(), b.float(), rtol=2.0 ** -6, atol=2.0 ** -6)
    pack = lambda n, k, seed, gu=False: ops.linear_pack_weight(_rand(((2 if gu else 1) * n, k), seed, k ** -0.5).to(dev), gate_up=gu)
    wo, wgu, wdown = pack(hidden, o_cols, 21), pack(ff, hidden, 22, True), pack(hidden, ff, 23)
    wqkv = pack(n_qkv, hidden, 24) if n_qkv else None
    empty = lambda: torch.full((rows, hidden + 64), 7.0, dtype=BF, device=dev)[:, 8:hidden + 8] if views else torch.full((rows, hidden), 7.0, dtype=BF, device=dev)
    form = lambda n: torch.full((32 * n,), 7.0, dtype=BF, device=dev)
    words = torch.zeros(2, ops.LINEAR_CHAIN_WORDS, dtype=torch.int32, device=dev)
    words[1] = 5  # what the launch before left there
    for i in range(launches):
        attn, res = ops.linear_pack_rows(_rand((rows, o_cols), 31 + i).to(dev)), empty()
        res.copy_(_rand((rows, hidden), 41 + i))
        before = res.clone()
        mid, out, between, out_p = empty(), empty(), torch.full((8 * (2 * hidden + ff),), 7.0, dtype=BF, device=dev), form(hidden)
        got = ops.linear_chain(wo, wgu, wdown, wqkv, attn, res, mid=mid, out=out, handover=between, out_packed=out_p if i != 1 else None,
                               arrived=words[i % 2], clear=words[1 - i % 2], norm_eps=1e-6, polls=polls)
        x, xp, ap = before.clone(), form(hidden), form(ff)
        ops.linear_rows(wo, attn, rows, hidden, o_cols, residual=x, out=x, out_packed=xp)
        assert same(mid, x)
        ops.linear_rows(wgu, xp, rows, ff, hidden, gate_up=True, out_packed=ap, want_out=False, norm_eps=1e-6)
        ops.linear_rows(wdown, ap, rows, hidden, ff, residual=x, out=x, out_packed=xp)
        assert same(out, x) and (i == 1 or same(out_p, xp)) and torch.equal(res, before)
        if n_qkv:
            assert same(got, ops.linear_rows(wqkv, xp, rows, n_qkv, hidden))
        else:
            assert got is None
        assert not words[1 - i % 2].any()
        assert words[i % 2].view(3, 64, 32)[:2, :hidden // 32, 0].eq(15).all()


def _chain_errors(dev):
    from tah_amd import ops
    from tah_amd._capi import TahDuoError
    z = lambda *s: torch.zeros(*s, dtype=BF, device=dev)
    w = lambda n: torch.zeros(n, dtype=torch.int32, device=dev)
    good = dict(mid=z(2, 2048), out=z(2, 2048), handover=z(8 * (2 * 2048 + 6144)), out_packed=z(32 * 2048),
                arrived=w(ops.LINEAR_CHAIN_WORDS), clear=w(ops.LINEAR_CHAIN_WORDS), norm_eps=1e-6)
    head = (z(2048 * 2048), z(2 * 6144 * 2048), z(2048 * 6144), None, z(32 * 2048))
    res = z(2, 2048)
    for bad in (dict(mid=res), dict(out=res), dict(out=good["mid"]), dict(out_packed=head[4]), dict(handover=head[4]), dict(handover=z(8 * 6144)),
                dict(clear=good["arrived"]), dict(arrived=w(64))):
        with pytest.raises((TahDuoError, RuntimeError)):
            ops.linear_chain(*head, res, **{**good, **bad})
    with pytest.raises((TahDuoError, RuntimeError)):
        ops.linear_chain(*head, z(9, 2048), **{**good, "mid": z(9, 2048), "out": z(9, 2048)})
    assert not ops.linear_chain_supported(9, 2048, 2048, 6144, 0) and not ops.linear_chain_supported(1, 2048, 2048, 6144, 8)
    assert not ops.linear_chain_supported(1, 1024, 2048, 6144, 0) and not ops.linear_chain_supported(1, 2048, 2048, 6144, 16 * 257)


def test_linear_chain_wants_a_compute_unit_for_each_workgroup(monkeypatch):
    import types
    from tah_amd import ops
    sizes = (1, 2048, 2048, 6144, 4096)
    for units, want in ((256, True), (304, True), (255, False), (32, False)):
        monkeypatch.setattr(torch.cuda, "get_device_properties", lambda device: types.SimpleNamespace(multi_processor_count=units))
        assert ops.linear_chain_supported(*sizes, device="cuda:0") is want
    assert ops.linear_chain_supported(*sizes) and ops.linear_chain_supported(*sizes, device="cpu")


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_linear_chain_without_rows_clears_the_next_words_on_the_cpu_shim():
    """The launch behind an empty one finds zeros too."""
    from tah_amd import _capi, ops
    words = torch.full((2, ops.LINEAR_CHAIN_WORDS), 15, dtype=torch.int32)
    with emu_util.emulated() as lib:
        assert lib.tah_linear_chain(ctypes.byref(_capi.LinearChainArgs(arrived=words[0].data_ptr(), clear=words[1].data_ptr())), None) == 0
        assert lib.tah_linear_chain(ctypes.byref(_capi.LinearChainArgs()), None) == 0
    assert bool((words[0] == 15).all()) and not words[1].any()


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
@pytest.mark.parametrize("which", range(4))
def test_linear_chain_refuses_results_on_a_weight_on_the_cpu_shim(which):
    """A late workgroup reads its weights after others' results are stored: on the last rows of any of them."""
    from tah_amd import ops
    from tah_amd._capi import TahDuoError
    z = lambda *s: torch.zeros(*s, dtype=BF)
    weights = (z(512 * 512), z(2 * 1536 * 512), z(512 * 1536), z(16 * 512))
    words = torch.zeros(2, ops.LINEAR_CHAIN_WORDS, dtype=torch.int32)
    with emu_util.emulated():
        with pytest.raises((TahDuoError, RuntimeError)):
            ops.linear_chain(*weights, z(32 * 512), z(1, 512), mid=z(1, 512), out=weights[which][-512:].view(1, 512),
                             handover=z(8 * (2 * 512 + 1536)), arrived=words[0], clear=words[1], norm_eps=1e-6)


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_linear_chain_on_the_cpu_shim():
    """Workgroups run one after another there: the first one's waits all end by computing the others' tiles itself."""
    with emu_util.emulated():
        _chain_errors("cpu")
        _chain_case("cpu", 7, 512, 512, 1536, 16, True, launches=1)


@contextlib.contextmanager
def _only_blocks(lib, first, count):
    lib.tah_emu_run_blocks(first, count)
    try:
        yield
    finally:
        lib.tah_emu_run_blocks(0, 0xffffffff)


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_linear_chain_waiters_take_different_tiles_on_the_cpu_shim():
    """Three workgroups that each see the same three tiles missing begin with a different one; tiles of workgroups that have begun
    are left to them until the polls are used up."""
    from tah_amd import _capi, ops
    z = lambda *s: torch.zeros(*s, dtype=BF)
    weights = (z(512 * 512), z(2 * 1536 * 512), z(512 * 1536))
    missing = [5, 18, 40]
    with emu_util.emulated() as lib:
        def taken(block, begun, polls):
            words = torch.zeros(2, ops.LINEAR_CHAIN_WORDS, dtype=torch.int32)
            lines = words[0].view(3, 64, 32)
            lines[:2, :, 0] = 15
            for t in missing:
                lines[0, t // 4, 0] &= ~(1 << t % 4)
            lines[0, :, 1] = 15 if begun else lines[0, :, 0]
            with _only_blocks(lib, block, 1):
                ops.linear_chain(*weights, None, z(32 * 512), z(1, 512), mid=z(1, 512), out=z(1, 512), handover=z(8 * (2 * 512 + 1536)),
                                 arrived=words[0], clear=words[1], norm_eps=1e-6, polls=polls)
                at = (ctypes.c_void_p * 64)()
                n = lib.tah_emu_ors(at, 64)
            words_at = [(a - words.data_ptr()) // 4 for a in at[:n]]
            line = [w // 32 for w in words_at if w < 64 * 32 and w % 32 == 0]  # phase 0, without the workgroup's own
            assert line[0] == block // 4 and sorted(line[1:]) == sorted(t // 4 for t in missing)
            return line[1]
        assert sorted(taken(b, False, 0) for b in range(3)) == sorted(t // 4 for t in missing)
        assert sorted(taken(b, True, 1) for b in range(3)) == sorted(t // 4 for t in missing)


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
@pytest.mark.parametrize("rows,n_qkv", [(1, 0), (2, 16), (4, 0)])
def test_linear_chain_by_one_workgroup_on_the_cpu_shim(rows, n_qkv):
    """What the first workgroup computes in the others' place, before they run themselves (all tiles but those of q|k|v)."""
    from tah_amd import ops
    dense = [_rand(s, 21 + i, s[1] ** -0.5) for i, s in enumerate([(512, 512), (2 * 1536, 512), (512, 1536), (16, 512)])]
    attn, res = _rand((rows, 512), 31), _rand((rows, 512), 41)
    mid, out = [torch.full((rows, 512), 7.0, dtype=BF) for _ in range(2)]
    words = torch.zeros(2, ops.LINEAR_CHAIN_WORDS, dtype=torch.int32)
    with emu_util.emulated() as lib:
        packed = [ops.linear_pack_weight(w, gate_up=i == 1) for i, w in enumerate(dense)]
        attn_p = ops.linear_pack_rows(attn)
        with _only_blocks(lib, 0, 1):
            got = ops.linear_chain(*packed[:3], packed[3] if n_qkv else None, attn_p, res, mid=mid, out=out,
                                   handover=torch.full((8 * (2 * 512 + 1536),), 7.0, dtype=BF), arrived=words[0], clear=words[1], norm_eps=1e-6)
    close = lambda a, b: torch.allclose(a.float(), b.float(), rtol=2.0 ** -6, atol=2.0 ** -6)
    _close(mid, reference(attn, dense[0], residual=res))
    if n_qkv:  # (without q|k|v nobody waits for down's tiles)
        assert close(out, reference(reference(mid, dense[1], gate_up=True, norm_eps=1e-6), dense[2], residual=mid))
        assert close(got, reference(out, dense[3]))
    else:
        assert close(out[:, :8], reference(reference(mid, dense[1], gate_up=True, norm_eps=1e-6), dense[2], residual=mid)[:, :8])


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("n_qkv", [4096, 0])
def test_linear_chain_tiles_of_others_gpu(rows, n_qkv):
    """A wait that gives up at its first look: whoever finds a tile missing computes it, the same bits."""
    _chain_case("cuda", rows, 2048, 2048, 6144, n_qkv, rows == 3, launches=5, polls=1)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,n_qkv,views", CHAIN_CASES)
def test_linear_chain_gpu(rows, n_qkv, views):
    _chain_case("cuda", rows, 2048, 2048, 6144, n_qkv, views, launches=5)
    _chain_errors("cuda")


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 2, 4, 8])
@pytest.mark.parametrize("n_qkv", [128, 2048, 2064])
def test_linear_chain_narrow_qkv_gpu(rows, n_qkv):
    """Up to 2048 columns of q|k|v and above: ``linear_rows`` sums even and odd steps apart up to there."""
    _chain_case("cuda", rows, 2048, 2048, 6144, n_qkv, False)


@pytest.mark.gpu
def test_linear_chains_side_by_side_gpu():
    """Two streams' launches share the compute units: whichever workgroups are resident, both finish with the same bits."""
    from tah_amd import ops
    pack = lambda n, k, seed, gu=False: ops.linear_pack_weight(_rand(((2 if gu else 1) * n, k), seed, k ** -0.5).cuda(), gate_up=gu)
    weights = pack(2048, 2048, 51), pack(6144, 2048, 52, True), pack(2048, 6144, 53), pack(4096, 2048, 54)
    attn, res = ops.linear_pack_rows(_rand((2, 2048), 55).cuda()), _rand((2, 2048), 56).cuda()
    z = lambda *s: torch.zeros(*s, dtype=BF, device="cuda")
    sets = [dict(mid=z(2, 2048), out=z(2, 2048), handover=z(8 * (2 * 2048 + 6144))) for _ in range(3)]
    words = torch.zeros(3, 2, ops.LINEAR_CHAIN_WORDS, dtype=torch.int32, device="cuda")
    run = lambda s, i: ops.linear_chain(*weights, attn, res, arrived=words[s][i % 2], clear=words[s][1 - i % 2], norm_eps=1e-6, **sets[s])
    want = run(2, 0)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    got = [[], []]
    for i in range(50):
        for s, stream in enumerate(streams):
            with torch.cuda.stream(stream):
                got[s].append(run(s, i))
    torch.cuda.synchronize()
    for one in got:
        assert all(torch.equal(q, want) for q in one)
    assert torch.equal(sets[0]["out"], sets[2]["out"]) and torch.equal(sets[1]["out"], sets[2]["out"])


# ── products chosen by a list shorter than the products (a workgroup per entry) and by a longer one ──
def _select_case(dev, rows, n, k, gate_up, lists):
    from tah_amd import ops
    batch = 8
    w = torch.cat([ops.linear_pack_weight(_rand(((2 if gate_up else 1) * n, k), 61 + b, k ** -0.5).to(dev), gate_up=gate_up) for b in range(batch)])
    xp = ops.linear_pack_rows(_rand((rows, k), 60).to(dev))
    run = lambda **kw: ops.linear_rows(w, xp, rows, n, k, gate_up=gate_up, batch=batch, shared_rows=True, **kw)
    want = run()
    for chosen in lists:
        out = torch.full((batch, rows, n), 5.0, dtype=BF, device=dev)
        run(out=out, select=torch.tensor(chosen, dtype=torch.int32, device=dev))
        for b in range(batch):
            assert torch.equal(out[b], want[b]) if b in chosen else bool((out[b] == 5.0).all())


# one entry, repeats, entries that name no product; as many entries as products and more
SELECT_LISTS = [[7], [5, 0, 5, 2, 0], [-1, 3, 8, 1 << 30], list(range(7)), [4] * 8, [6, 1] * 40]


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_linear_rows_select_on_the_cpu_shim():
    with emu_util.emulated():
        _select_case("cpu", 3, 16, 64, False, SELECT_LISTS[1:3])


@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,k,gate_up", [(1, 768, 2048, True), (9, 48, 2048, True), (20, 96, 320, True), (1, 2048, 768, False), (8, 64, 2048, False), (32, 32, 96, False)])
def test_linear_rows_select_gpu(rows, n, k, gate_up):
    _select_case("cuda", rows, n, k, gate_up, SELECT_LISTS)


def _beside_case(dev, rows, n, n2, k, bias, relu):
    """An output head and a second layer of the same rows in one launch: the bits of the two calls, and nothing behind either result."""
    from tah_amd import ops
    d = lambda t: t.to(dev)
    w, w2, x = d(_rand((n, k), 1, k ** -0.5)), d(_rand((n2, k), 2, k ** -0.5)), d(_rand((rows, k), 3))
    b2 = d(_rand((n2,), 4)) if bias else None
    wp, w2p, xp = ops.linear_pack_weight(w), ops.linear_pack_weight(w2), ops.linear_pack_rows(x)
    assert ops.linear_beside_supported(rows, n, k, n2)
    out = torch.full((rows + 1, n + 16), 3.0, dtype=BF, device=dev)
    y, y2 = ops.linear_beside(wp, w2p, xp, rows, n, n2, k, norm_eps=1e-6, out=out[:rows, :n], bias2=b2, relu2=relu)
    assert torch.equal(y, ops.linear_rows(wp, xp, rows, n, k, norm_eps=1e-6))
    assert torch.equal(y2, ops.linear_rows(w2p, xp, rows, n2, k, norm_eps=1e-6, bias=b2, relu=relu))
    assert (out[rows:] == 3.0).all() and (out[:, n:] == 3.0).all() and y2.any()


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_linear_beside_on_cpu_shim():
    from tah_amd import ops
    from tah_amd._capi import TahDuoError
    with emu_util.emulated():
        _beside_case("cpu", 3, 16384, 64, 32, True, True)
        # no head, widths of half a workgroup's, too many rows
        for rows, n, n2, k in ((1, 16352, 64, 32), (1, 16384 + 16, 64, 32), (1, 16384, 48, 32), (17, 16384, 64, 32)):
            assert not ops.linear_beside_supported(rows, n, k, n2)
            z = torch.zeros(n * k, dtype=BF)
            with pytest.raises(TahDuoError):
                ops.linear_beside(z, z[:n2 * k], torch.zeros(32 * k, dtype=BF), rows, n, n2, k, norm_eps=1e-6)


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_linear_beside_refuses_results_on_each_other_and_on_what_it_reads():
    """Two calls have an order that one launch has not; columns of one array side by side share nothing and are taken (with a bias off
    its alignment: refused by the check behind, before a launch)."""
    import ctypes as C

    from tah_amd import _capi
    rows, n, n2, k = 3, 16384, 32, 32
    w, w2, x = torch.zeros(n * k, dtype=BF), torch.zeros(n2 * k, dtype=BF), torch.zeros(64 * k, dtype=BF)
    buf, b2 = torch.zeros(rows, n + n2 + 32, dtype=BF), torch.zeros(n2 + 8, dtype=BF)[1:]
    with emu_util.emulated() as lib:
        def call(out, out2, x2=x, bias=b2, stride=buf.stride(0), stride2=buf.stride(0)):
            a, b = [_capi.LinearRowsArgs(w_packed=ww.data_ptr(), x_packed=xx.data_ptr(), out=o.data_ptr(), out_row_stride=s, rows=rows, n=nn, k=k, input_norm=1,
                                         norm_eps=1e-6) for ww, xx, o, s, nn in ((w, x, out, stride, n), (w2, x2, out2, stride2, n2))]
            b.bias = bias.data_ptr()
            return lib.tah_linear_beside(C.byref(a), C.byref(b), None)

        other = torch.zeros(rows, n2, dtype=BF)
        shape, taken = _capi.TAH_E_SHAPE, _capi.TAH_E_ALIGN
        assert call(buf, buf[:, n:]) == taken and call(buf[:, n2:], buf) == taken and call(buf, other, stride2=n2) == taken
        assert call(buf, buf[:, n - 16:]) == shape and call(buf[:, 16:], buf) == shape  # half of the narrow result's columns
        assert call(buf, buf[1:, :n2]) == shape                                     # rows of the same array, one further down
        assert call(buf, x, stride2=n2) == shape and call(buf, w2, stride2=n2) == shape and call(buf, w, stride2=n2) == shape
        assert call(buf, other, stride2=n2, bias=other) == shape and call(buf, other, stride2=n2, bias=buf) == shape
        assert call(buf, other, x2=torch.zeros(64 * k, dtype=BF), stride2=n2) == shape


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 8, 9, 16])
@pytest.mark.parametrize("n,n2,k,bias,relu", [(151936, 512, 2048, True, True), (16384, 32, 2048, False, False), (32000, 96, 1024, True, False)])
def test_linear_beside_gpu(rows, n, n2, k, bias, relu):
    _beside_case("cuda", rows, n, n2, k, bias, relu)
