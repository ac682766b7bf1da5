"""A norm of the residual stream and the choice of experts behind it in one launch (tah_norm_route): the bits of tah_residual_norm and
tah_moe_route, for both designs' norms and rules, row lengths at the ends of a thread's unit and expert counts at the edges of a wave's share."""
import pytest
import torch

from tests import emu_util

# rows, cols, norm groups, experts, top, shared gate, sigmoid, expert groups, keep, norm in front of the router, something added
CASES = [
    (1, 2048, 8, 64, 8, False, True, 8, 4, True, True),     # the grouped design, one row
    (8, 2048, 1, 64, 8, True, False, 1, 1, False, True),    # the shared expert's gate is the 65th
    (3, 2040, 1, 71, 2, True, False, 1, 1, True, True),     # as many as fit, columns a thread short
    (2, 520, 1, 40, 4, False, False, 1, 1, False, False),   # five to a wave, one column block and a unit, nothing added
    (32, 256, 4, 16, 3, False, True, 4, 2, True, True),     # two to a wave
    (5, 8, 1, 1, 1, False, False, 1, 1, True, True),
]


def route_case(dev, rows, cols, norm_groups, experts, top, gate, sigmoid, groups, keep, normed, added):
    from tah_amd import ops

    call = lambda name, *a: ops._call(name, *a)
    g = torch.Generator().manual_seed(rows * 1000 + cols)
    r = lambda *s, dt=torch.float32: torch.randn(*s, generator=g).to(dt).to(dev)
    bf = torch.bfloat16
    x, y, scale = r(rows, cols), (r(rows, cols, dt=bf) if added else None), (r(rows) if added else None)
    coef, nxt = (r(cols) if added else None), (r(cols) if normed else None)
    router, gate_w = r(experts, cols, dt=bf) * 0.1, (r(1, cols, dt=bf) if gate else None)
    got = []
    for fused in (False, True):
        xe, xp = torch.zeros(rows, cols, dtype=bf, device=dev), torch.zeros(32 * cols, dtype=bf, device=dev)
        rows_form = xp if cols % 32 == 0 else None
        index = torch.full((rows, top), -1, dtype=torch.int32, device=dev)
        weight, sg = torch.zeros(rows, top, device=dev), (torch.zeros(rows, device=dev) if gate else None)
        tail = (norm_groups, cols // norm_groups)
        x_packed, normed_packed = (None, rows_form) if normed else (rows_form, None)
        if not normed and rows_form is None:
            x_packed = None
        if fused:
            assert call("norm_route_supported", rows, cols, experts, gate)
            out = torch.full_like(x, float("nan"))
            call("norm_route", x, out, coef, cols, 1e-6, y, scale, x_packed, nxt, xe if normed else None, normed_packed, *tail, router, gate_w, index, weight,
                 sg, int(sigmoid), groups, keep)
        else:
            out = x.clone()
            call("residual_norm", out, coef, cols, 1e-6, y, scale, None, None, None, None if normed else xe, x_packed, nxt, xe if normed else None,
                 normed_packed, 1, 0, *tail, None, None, None)
            xe_kept = xe.clone()
            call("moe_route", xe if normed else out, router, gate_w, index, weight, sg, int(sigmoid), groups, keep)
        got.append([t.cpu() for t in (out, xe if normed else out, xp, index, weight) + ((sg,) if gate else ())])
    for a, b in zip(*got):
        assert torch.equal(a, b)
    assert (got[1][3] >= 0).all()


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
@pytest.mark.parametrize("case", [CASES[2], CASES[3], CASES[4], CASES[5]])
def test_norm_route_on_cpu_shim(case):
    with emu_util.emulated():
        rows, cols, *rest = case
        route_case("cpu", min(rows, 3), cols, *rest)


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_norm_route_refuses_what_it_is_not_built_for():
    from tah_amd import ops

    with emu_util.emulated():
        for rows, cols, experts, gate in ((33, 2048, 64, False), (1, 2056, 64, False), (1, 2048, 72, True), (1, 2044, 8, False)):
            assert not ops._call("norm_route_supported", rows, cols, experts, gate)
        x = torch.zeros(2, 64)
        bf = torch.bfloat16
        i, w = torch.zeros(2, 2, dtype=torch.int32), torch.zeros(2, 2)
        args = lambda out: (x, out, torch.zeros(64), 64, 1e-6, torch.zeros(2, 64, dtype=bf), None, None, None, None, None, 1, 64, torch.zeros(4, 64, dtype=bf),
                            None, i, w, None, 0, 1, 1)
        ops._call("norm_route", *args(torch.zeros(2, 64)))
        with pytest.raises(ops._capi.TahDuoError):
            ops._call("norm_route", *args(x))  # results on what is read


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_norm_route_refuses_a_choice_on_what_other_rows_read_or_leave():
    """Two calls have an order, one launch has none: a row's experts may be stored before another row's norm has read its own."""
    from tah_amd import ops

    bf = torch.bfloat16
    with emu_util.emulated():
        def call(**kw):
            t = dict(x=torch.randn(4, 64), out=torch.zeros(4, 64), coef=torch.ones(64), y=torch.randn(4, 64).to(bf), y_scale=torch.ones(4), nxt=torch.ones(64),
                     normed=torch.zeros(4, 64, dtype=bf), packed=torch.zeros(32 * 64, dtype=bf), router=torch.randn(8, 64).to(bf),
                     gate_w=torch.randn(1, 64).to(bf), index=torch.zeros(4, 2, dtype=torch.int32), weight=torch.zeros(4, 2), sg=torch.zeros(4))
            for name, on in kw.items():  # (the result `name` at the start of tensor `on`)
                t[name] = t[on].view(-1).view(t[name].dtype)[:t[name].numel()].view(t[name].shape)
            ops._call("norm_route", t["x"], t["out"], t["coef"], 64, 1e-6, t["y"], t["y_scale"], None, t["nxt"], t["normed"], t["packed"], 1, 64, t["router"],
                      t["gate_w"], t["index"], t["weight"], t["sg"], 0, 1, 1)

        call()
        call(normed="y")  # (row by row, as the norm alone takes it)
        for name in ("index", "weight", "sg"):
            for on in ("x", "y", "coef", "nxt", "out", "normed", "packed", "router") + (("y_scale", "gate_w") if name == "sg" else ()):
                with pytest.raises(ops._capi.TahDuoError):
                    call(**{name: on})
        with pytest.raises(ops._capi.TahDuoError):
            call(normed="router")


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_norm_route_gpu(case):
    print("case norm_route", case, flush=True)
    route_case("cuda", *case)
