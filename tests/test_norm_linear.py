"""A norm of the residual stream and the linear layer behind it in one launch (tah_norm_linear): the bits of tah_residual_norm and
tah_linear_rows, what both leave behind included.  (Three and four rows, and the widest layer: two launches.)"""
import pytest
import torch

from tests import emu_util

COLS = 2048
needs_clang = pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
# rows, columns of the layer, (groups, true width), experts' top, (taps, slots of the rows), sublayer result, its scale, norm in front, activation
CASES = [
    (1, 3616, (8, 2048), 0, (4, [2]), True, False, True, {}),
    (1, 2048, (1, 2048), 8, None, True, True, False, {}),
    (2, 6144, (8, 2048), 0, None, True, False, True, {"xielu": (0.7, 1.1)}),
    (2, 2064, (1, 2000), 3, (3, [0, -1]), False, False, True, {}),
    (3, 2048, (5, 2040), 11, (6, [1, 4, 0]), True, False, True, {"gelu_tanh": True}),
    (4, 1024, (16, 2048), 8, (4, [3, 0, 2, 1]), True, True, True, {}),
    (1, 2080, (8, 2048), 0, (4, [1]), False, False, True, {}),
    (2, 2048, (5, 2040), 11, (6, [1, 4]), True, False, True, {"gelu_tanh": True}),
    (1, 8192, (16, 2048), 8, (4, [0]), True, True, True, {}),
    (1, 12352, (1, 2048), 0, None, True, False, False, {}),
]
# neither experts nor convolution: wide layers and narrow ones, groups and none
CASES += [(rows, n, groups, 0, None, True, False, normed, act) for rows in (1, 2) for n, act in ((6144, {"xielu": (0.7, 1.1)}), (2048, {}))
          for groups, normed in (((8, 2048), True), ((1, 2048), False))]


def norm_linear_case(dev, rows, n, geometry, top, conv, with_y, scaled, normed, act, seed=3):
    from tah_amd import ops
    from tah_amd.mixers import Activation, Linear, Norm, Step
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g)
    groups, width = geometry
    group_cols = width // groups if groups > 1 else COLS
    true = torch.zeros(COLS, dtype=torch.bool)
    true[:width] = True
    bf = lambda t: t.to(torch.bfloat16).to(dev)
    x = (r(rows, COLS) * true).to(dev)
    y = bf(r(rows, COLS) * true) if with_y else None
    experts = index = weight = None
    if top:
        experts, index = bf(r(20 * rows, COLS) * true), torch.randint(0, 20, (rows, top), generator=g, dtype=torch.int32).to(dev)
        weight = torch.rand(rows, top, generator=g).to(dev)
    coef, norm = [(torch.rand(COLS, generator=g) * true).to(dev) for _ in range(2)]
    layer = Linear(bf(r(n, COLS) * COLS ** -0.5))
    pos = torch.tensor([9, 2, 0, 41][:rows], dtype=torch.int32).to(dev)
    a = Activation(0, rows=act)

    def run(fused):
        st = Step(x.clone(), torch.zeros(rows, COLS, dtype=torch.bfloat16, device=dev), pos, torch.zeros(32 * COLS, dtype=torch.bfloat16, device=dev),
                  normed=normed, x_other=torch.full_like(x, 7.0))
        cv = slot = ring = None
        if conv:
            gc = torch.Generator().manual_seed(seed + 1)
            ring = torch.randn(5, conv[0], COLS, generator=gc).to(torch.bfloat16).to(dev)
            cv = ops.lib().InputConv((torch.randn(conv[0], COLS, generator=gc) * true).to(dev), ring)
            slot = torch.tensor(conv[1], dtype=torch.int32).to(dev)
        front = (coef if with_y or top else None, width, 1e-5, y, torch.linspace(0.2, 1.0, rows).to(dev) if scaled else None, experts, index, weight)
        st.pending = Norm(front, norm if normed else None, (rows, 1, groups, group_cols, cv, slot, pos if conv else None))
        if not fused:
            st.settle()
        packed = torch.full((32 * n,), 3.0, dtype=torch.bfloat16, device=dev) if n % 32 == 0 else None
        out = st.linear(layer, out_packed=packed, act=a)
        assert st.pending is None
        return [t for t in (out, packed, st.x, ring) if t is not None]

    got, want = run(True), run(False)
    assert all(torch.isfinite(t.float()).all() for t in want)
    for u, v in zip(got, want):
        assert torch.equal(u, v)


@needs_clang
@pytest.mark.parametrize("case", [0, 6, 10])
def test_norm_and_linear_layer_in_one_launch_on_cpu_shim(case):
    rows, n, *rest = CASES[case]
    with emu_util.emulated():
        norm_linear_case("cpu", rows, min(n, 64), *rest)


@needs_clang
def test_norm_linear_refuses_results_on_operands_on_cpu_shim():
    from tah_amd import TahDuoError
    from tah_amd.mixers import Linear, Norm, Step
    with emu_util.emulated():
        x = torch.randn(1, COLS)
        st = Step(x, None, None, torch.zeros(32 * COLS, dtype=torch.bfloat16), x_other=x)
        st.pending = Norm((None, COLS, 1e-5, None, None, None, None, None), torch.ones(COLS), (1, 0, 1, COLS, None, None, None))
        with pytest.raises(TahDuoError):
            st.linear(Linear(torch.zeros(32, COLS, dtype=torch.bfloat16)))


@needs_clang
def test_norm_linear_refuses_results_on_what_a_row_comes_with_on_cpu_shim():
    """The factor, the experts' choice, slot, position, convolution and its inputs: in the residual rows' place and in the layer's result's."""
    import ctypes as C

    from tah_amd import _capi
    TAPS, SLOTS, N = 3, 2, 32
    mem = torch.zeros(4 << 20, dtype=torch.uint8)
    at = lambda k: mem.data_ptr() + (k << 18)   # places a quarter of a megabyte apart
    names = ["x", "y", "y_scale", "experts", "index", "weight", "coef", "next_coef", "conv", "conv_state", "slot", "pos"]
    place = {name: at(i) for i, name in enumerate(names)}
    ends = {"y_scale": 4, "index": 8, "weight": 8, "slot": 4, "pos": 4, "conv": 4 * TAPS * COLS, "conv_state": 2 * SLOTS * TAPS * COLS, "coef": 4 * COLS}
    with emu_util.emulated() as lib:
        def call(x_out, out):
            n = _capi.ResidualNormArgs(**place, y_row_stride=COLS, experts_row_stride=COLS, rows=1, width=COLS, cols=COLS, top=2, index_scale=1, eps=1e-5,
                                       groups=1, group_cols=COLS, taps=TAPS, nslots=SLOTS, dtype=0)
            a = _capi.LinearRowsArgs(w_packed=at(12), out=out, out_row_stride=N, rows=1, n=N, k=COLS)
            return lib.tah_norm_linear(C.byref(n), x_out, C.byref(a), None)

        assert call(at(13), at(14)) == 0
        for name, size in ends.items():
            for offset in {0, (size - 1) // 16 * 16}:  # (results are 16-byte aligned)
                assert call(place[name] + offset, at(14)) == _capi.TAH_E_SHAPE, name
                assert call(at(13), place[name] + offset) == _capi.TAH_E_SHAPE, name
        assert int(mem[14 << 18:].sum()) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_norm_and_linear_layer_in_one_launch_gpu(case):
    print("case norm_linear", case, flush=True)
    norm_linear_case("cuda", *case)
