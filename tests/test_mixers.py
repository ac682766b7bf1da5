"""Layer mechanisms (tah_amd.mixers, include/tah_mixers.h), each alone, against the plain oracle: on the CPU execution build
at small sizes, on the GPU at those and at larger ones."""
import pytest
import torch

from tests import emu_util
from tests import zedudra_cases as D
from tests import zozosun_cases as Z

needs_clang = pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
BOTH = pytest.mark.parametrize("dtype", ["f32", "bf16"])


def delta(heads, kv, dim, vdim, conv, eps=1e-4):
    return {"heads": heads, "kv_heads": kv, "dim": dim, "vdim": vdim, "conv": conv, "eps": eps}


def latent(heads, dim, rot, vdim, rank, window, base=50.0, scale=0.4):
    return Z.latent_of(heads, dim, rot, vdim, rank, window, base, scale)["mixer"]


# (sizes, lengths, portions per sequence)
DELTA_SMALL = [(delta(2, 1, 6, 5, 3), (5, 3), ((2, 3), (3,))), (delta(2, 2, 12, 8, 4), (7, 2), ((7,), (2,))),
               (delta(2, 1, 16, 32, 3), (5, 4), ((3, 2), (4,))),
               (delta(2, 1, 16, 16, 4), (100, 49), ((50, 50), (49,)))]   # long enough for the chunked form
DELTA_GPU = DELTA_SMALL + [
    (delta(6, 3, 40, 24, 4), (70, 33), ((37, 2, 31), (2, 31))), (delta(4, 4, 64, 64, 2), (130, 5), ((128, 2), (3, 2))),
    (delta(8, 2, 128, 128, 4), (200, 65), ((64, 17, 119), (65,))), (delta(2, 1, 256, 96, 4), (40, 40), ((40,), (17, 23))),
    (delta(3, 1, 17, 130, 1), (30, 9), ((16, 14), (9,))), (delta(2, 2, 100, 256, 5), (21, 2), ((5, 16), (2,))),
    (delta(5, 5, 32, 512, 3), (19, 18), ((19,), (2, 16))), (delta(4, 2, 128, 64, 4), (333, 97), ((96, 64, 173), (97,))),
    (delta(2, 1, 224, 64, 4), (7, 5), ((7,), (5,))),   # a step holds two channels per thread, the last one too
    (delta(2, 1, 256, 32, 2), (161, 70), ((100, 61), (70,))), (delta(6, 3, 32, 48, 4), (520, 520), ((255, 265), (256, 264))),
]
# (sizes, prompt, portions, decoded tokens, ring capacity)
LATENT_SMALL = [(latent(2, 8, 4, 6, 10, 4), 9, (2, 5, 2), 3, None), (latent(1, 32, 6, 16, 40, 3), 6, (6,), 2, 5)]
LATENT_GPU = LATENT_SMALL + [
    (latent(3, 24, 8, 20, 48, 40), 150, (64, 2, 84), 45, None), (latent(16, 128, 64, 128, 512, 100), 300, (300,), 70, 130),
    (latent(20, 64, 32, 64, 96, 65), 129, (1 + 63, 65), 66, 65), (latent(5, 64, 16, 200, 64, 7), 40, (7, 2, 31), 9, None),
    (latent(2, 96, 32, 96, 288, 128), 260, (128, 132), 4, 200), (latent(33, 32, 32, 32, 32, 2), 20, (20,), 3, None),
    (latent(4, 200, 40, 48, 700, 33), 70, (3, 67), 5, None), (latent(2, 400, 6, 300, 64, 9), 21, (21,), 3, None),
    (latent(2, 32, 2, 16, 960, 5), 12, (12,), 2, None),
]
MOE_SMALL = [(5, 40, 12, 4, 2, 9), (3, 32, 32, 3, 1, 0)]
MOE_GPU = MOE_SMALL + [(32, 96, 48, 16, 4, 64), (200, 160, 96, 8, 8, 32), (700, 256, 192, 64, 6, 128), (31, 512, 100, 7, 3, 0), (300, 72, 40, 5, 5, 17)]
# (sizes, prompt, portions, decoded tokens, further arguments): windows inside, at and across the 64-key tiles and the 32-key
# passes, kept tokens that fill tiles of their own, more query heads than a tile or a pass takes, heads of up to 256
WINDOW_SMALL = [(D.window_of(2, 1, 12, 6, 4, 2), 11, (2, 7, 2), 4, {}), (D.window_of(2, 2, 32, 32, 6, 3), 13, (13,), 2, {}),
                (D.window_of(2, 1, 16, 8, 5, 1), 7, (5, 2), 3, dict(own_values=20, adjacent=False, gate=False))]
WINDOW_GPU = WINDOW_SMALL + [
    (D.window_of(16, 8, 128, 64, 64, 4), 200, (64, 2, 63, 71), 70, {}), (D.window_of(10, 2, 128, 48, 33, 3), 150, (150,), 40, {}),
    (D.window_of(20, 1, 64, 32, 65, 1), 140, (1 + 62, 2, 75), 66, {}), (D.window_of(5, 5, 24, 24, 128, 7), 260, (130, 130), 9, {}),
    (D.window_of(33, 1, 96, 2, 31, 5), 90, (33, 57), 34, {}), (D.window_of(4, 2, 160, 40, 40, 70), 180, (90, 90), 45, {}),
    (D.window_of(6, 2, 256, 256, 100, 130), 310, (200, 2, 108), 12, {}), (D.window_of(2, 2, 300, 20, 9, 2), 40, (40,), 12, {}),
    (D.window_of(4, 1, 128, 64, 1, 0), 70, (35, 35), 5, {}), (D.window_of(4, 4, 128, 128, 600, 64), 700, (300, 400), 20, {}),
    (D.window_of(9, 3, 40, 0, 17, 3), 80, (80,), 20, {}), (D.window_of(8, 1, 128, 64, 50, 4), 120, (60, 60), 30, dict(max_len=4000)),
    (D.window_of(8, 2, 64, 64, 40, 2), 130, (65, 65), 45, dict(own_values=64)), (D.window_of(4, 2, 128, 32, 50, 4), 130, (130,), 20, dict(own_values=72, gate=False)),
    (D.window_of(4, 1, 48, 24, 20, 3), 70, (70,), 22, dict(own_values=100, adjacent=False)),
]
GROUPS = [(5, 44, 4), (3, 96, 3), (2, 64, 8)]
GROUPS_GPU = GROUPS + [(32, 2048, 8), (40, 2048, 1), (3, 1920, 16), (7, 5000, 5), (2, 600, 200), (6, 16384, 2), (4, 24, 24), (9, 1000, 8)]
CONVS = [(20, 4, 3), (32, 1, 1), (24, 2, 4), (16, 1, 6)]
CONVS_GPU = CONVS + [(2048, 8, 4), (600, 3, 2), (1000, 8, 9), (72, 1, 33)]
EXPERTS_SMALL = [(5, 40, 12, 6, 2, 3, 2, 0.7), (3, 32, 32, 4, 1, 1, 1, 1.5)]
EXPERTS_GPU = EXPERTS_SMALL + [(32, 96, 48, 16, 4, 4, 2, 1.0), (200, 160, 96, 8, 3, 2, 1, 7.0), (700, 256, 192, 64, 6, 8, 4, 0.5), (300, 72, 40, 130, 5, 65, 20, 1.0),
                               (31, 512, 100, 256, 8, 128, 64, 2.0), (20, 64, 32, 9, 2, 9, 5, 1.0)]


# ── CPU execution build ──────────────────────────────────────────────────────────────────────────────────────────────
@needs_clang
@BOTH
def test_rows_on_cpu_shim(dtype):
    with emu_util.emulated():
        Z.rows_case("cpu", Z.DTYPES[dtype])


@needs_clang
def test_linear_batches_on_cpu_shim():
    with emu_util.emulated():
        Z.linear_batch_case("cpu", 3, 16, 32, 3)


def check_delta_columns(dev, dtype, m, lens):
    """Many sequences' scans hold 32 state columns to a workgroup, one's 16: the same results and states, to the bit."""
    assert m["heads"] * len(lens) * (m["vdim"] // 16) >= 512 > m["heads"] * (m["vdim"] // 16) and min(lens) >= 48
    layer, w, cols, width, S = Z.delta_layer(dev, dtype, m, 2 * len(lens), torch.Generator().manual_seed(5))
    proj = [Z.rnd(torch.Generator().manual_seed(6 + b), n, width).to(dtype) for b, n in enumerate(lens)]
    out_cols = (m["heads"] * m["vdim"] + 31) // 32 * 32

    def run(seqs, first_slot):
        P, _ = Z.portions_of([lens[b] for b in seqs], [0] * len(seqs), [first_slot + b for b in seqs], dev)
        out = torch.zeros((sum(lens[b] for b in seqs), out_cols), dtype=dtype, device=dev)
        layer.portions(torch.cat([proj[b] for b in seqs]).to(dev), P, out)
        return out

    together = run(range(len(lens)), 0)
    alone = torch.cat([run([b], len(lens)) for b in range(len(lens))])
    assert together.any() and torch.equal(together, alone)
    assert torch.equal(S[:len(lens)], S[len(lens):])


@needs_clang
def test_delta_scan_columns_on_cpu_shim():
    with emu_util.emulated():
        check_delta_columns("cpu", torch.bfloat16, delta(64, 32, 16, 32, 4), (64, 49, 97, 48))


@pytest.mark.gpu
@pytest.mark.parametrize("m,lens", [(delta(32, 16, 128, 128, 4), (333, 48, 64, 97)), (delta(8, 8, 64, 96, 2), (65,) * 11), (delta(16, 4, 32, 64, 3), (50,) * 9)])
def test_delta_scan_columns_gpu(m, lens):
    check_delta_columns("cuda", torch.bfloat16, m, lens)


@needs_clang
@BOTH
@pytest.mark.parametrize("case", range(len(DELTA_SMALL)))
def test_delta_rule_on_cpu_shim(dtype, case):
    m, lens, cuts = DELTA_SMALL[case]
    with emu_util.emulated():
        Z.delta_case("cpu", Z.DTYPES[dtype], m, lens, cuts, steps=2)


@needs_clang
@BOTH
@pytest.mark.parametrize("case", range(len(LATENT_SMALL)))
def test_latent_attention_on_cpu_shim(dtype, case):
    m, total, cuts, steps, cap = LATENT_SMALL[case]
    with emu_util.emulated():
        Z.latent_case("cpu", Z.DTYPES[dtype], m, total, cuts, steps, cap)


@needs_clang
@BOTH
@pytest.mark.parametrize("case", range(len(MOE_SMALL)))
def test_mixture_of_experts_on_cpu_shim(dtype, case):
    with emu_util.emulated():
        Z.moe_case("cpu", Z.DTYPES[dtype], *MOE_SMALL[case])


@needs_clang
@BOTH
@pytest.mark.parametrize("case", range(len(WINDOW_SMALL)))
def test_window_attention_on_cpu_shim(dtype, case):
    m, total, cuts, steps, kw = WINDOW_SMALL[case]
    with emu_util.emulated():
        D.window_case("cpu", Z.DTYPES[dtype], m, total, cuts, steps, **kw)


@needs_clang
@BOTH
def test_norms_over_groups_on_cpu_shim(dtype):
    with emu_util.emulated():
        for case in GROUPS:
            D.group_norm_case("cpu", Z.DTYPES[dtype], *case)


@needs_clang
@BOTH
def test_input_convolution_on_cpu_shim(dtype):
    with emu_util.emulated():
        for case in CONVS:
            D.conv_case("cpu", Z.DTYPES[dtype], *case)


@needs_clang
@BOTH
def test_activations_on_cpu_shim(dtype):
    with emu_util.emulated():
        D.activation_case("cpu", Z.DTYPES[dtype], 2, 16, 32)


@needs_clang
@BOTH
@pytest.mark.parametrize("case", range(len(EXPERTS_SMALL)))
def test_grouped_experts_on_cpu_shim(dtype, case):
    with emu_util.emulated():
        D.moe_case("cpu", Z.DTYPES[dtype], *EXPERTS_SMALL[case])


# ── GPU ──────────────────────────────────────────────────────────────────────────────────────────────────────────────
@pytest.mark.gpu
@BOTH
@pytest.mark.parametrize("rows,width,cols", [(5, 72, 96), (32, 2048, 2048), (40, 100, 104), (3, 5000, 5024), (2, 16384, 16384)])
def test_rows_gpu(dtype, rows, width, cols):
    Z.rows_case("cuda", Z.DTYPES[dtype], rows, width, cols)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,k,batch", [(3, 16, 32, 3), (32, 512, 128, 16), (20, 128, 512, 16), (7, 48, 96, 1), (32, 96, 256, 5)])
def test_linear_batches_gpu(rows, n, k, batch):
    Z.linear_batch_case("cuda", rows, n, k, batch)


@pytest.mark.gpu
@BOTH
@pytest.mark.parametrize("case", range(len(DELTA_GPU)))
def test_delta_rule_gpu(dtype, case):
    m, lens, cuts = DELTA_GPU[case]
    Z.delta_case("cuda", Z.DTYPES[dtype], m, lens, cuts, steps=4)


@pytest.mark.gpu
@BOTH
@pytest.mark.parametrize("case", range(len(LATENT_GPU)))
def test_latent_attention_gpu(dtype, case):
    m, total, cuts, steps, cap = LATENT_GPU[case]
    Z.latent_case("cuda", Z.DTYPES[dtype], m, total, cuts, steps, cap)


@pytest.mark.gpu
@BOTH
@pytest.mark.parametrize("case", range(len(MOE_GPU)))
def test_mixture_of_experts_gpu(dtype, case):
    Z.moe_case("cuda", Z.DTYPES[dtype], *MOE_GPU[case])


@pytest.mark.gpu
@BOTH
@pytest.mark.parametrize("case", range(len(WINDOW_GPU)))
def test_window_attention_gpu(dtype, case):
    m, total, cuts, steps, kw = WINDOW_GPU[case]
    D.window_case("cuda", Z.DTYPES[dtype], m, total, cuts, steps, **kw)


@pytest.mark.gpu
@BOTH
@pytest.mark.parametrize("case", range(len(GROUPS_GPU)))
def test_norms_over_groups_gpu(dtype, case):
    D.group_norm_case("cuda", Z.DTYPES[dtype], *GROUPS_GPU[case])


@pytest.mark.gpu
@BOTH
@pytest.mark.parametrize("case", range(len(CONVS_GPU)))
def test_input_convolution_gpu(dtype, case):
    D.conv_case("cuda", Z.DTYPES[dtype], *CONVS_GPU[case], cuts=((50, 2, 33), (1 + 2, 64)))


@pytest.mark.gpu
@BOTH
def test_activations_gpu(dtype):
    D.activation_case("cuda", Z.DTYPES[dtype])
    D.activation_case("cuda", Z.DTYPES[dtype], 32, 480, 256)


@pytest.mark.gpu
@BOTH
@pytest.mark.parametrize("case", range(len(EXPERTS_GPU)))
def test_grouped_experts_gpu(dtype, case):
    D.moe_case("cuda", Z.DTYPES[dtype], *EXPERTS_GPU[case])


def _route_case(dev, rows, experts, top, groups, keep, sigmoid=False):
    """Scores that the inputs are (the router is the identity), many of them equal: the chosen ones against a plain ordering,
    the lower index first among equals, groups by the sum of their two largest."""
    from tah_amd.ops import _call
    cols = (experts + 7) // 8 * 8
    g = torch.Generator().manual_seed(experts + top)
    z = torch.randint(-24, 25, (rows, experts), generator=g).float() / 8
    if rows > 3:
        z[1], z[2, :experts // 2] = 0.5, -1.0
    x = torch.zeros(rows, cols)
    x[:, :experts] = z
    index, weight = torch.full((rows, top), -1, dtype=torch.int32, device=dev), torch.zeros(rows, top, device=dev)
    _call("moe_route", x.to(dev), torch.eye(experts, cols).to(torch.bfloat16).to(dev), None, index, weight, None, int(sigmoid), groups, keep)
    size = experts // groups
    for r, s in enumerate((torch.sigmoid(z) if sigmoid else z).tolist()):
        two = lambda i: sum(sorted(s[i * size:(i + 1) * size])[-2:])
        best = sorted(range(groups), key=lambda i: (-two(i), i))[:keep]
        allowed = [e for i in best for e in range(i * size, (i + 1) * size)]
        want = sorted(allowed, key=lambda e: (-s[e], e))[:top]
        assert index[r].tolist() == want, (r, index[r].tolist(), want)
        v = torch.tensor([s[e] for e in want], dtype=torch.float64)
        assert torch.allclose(weight[r].cpu().double(), v if sigmoid else torch.softmax(v, 0), rtol=1e-5)


ROUTES = [(5, 8, 8, 1, 1), (4, 63, 5, 1, 1), (6, 64, 8, 8, 4), (4, 65, 64, 1, 1), (4, 128, 6, 64, 3), (4, 256, 8, 1, 1), (4, 260, 7, 65, 9), (5, 320, 3, 2, 1)]


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
@pytest.mark.parametrize("rows,experts,top,groups,keep", ROUTES[1:4] + ROUTES[6:7])
def test_router_choice_among_equal_scores_on_cpu_shim(rows, experts, top, groups, keep):
    with emu_util.emulated():
        _route_case("cpu", rows, experts, top, groups, keep)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,experts,top,groups,keep", ROUTES + [(300, 64, 8, 8, 4), (300, 256, 8, 1, 1), (300, 300, 4, 75, 10)])
def test_router_choice_among_equal_scores_gpu(rows, experts, top, groups, keep):
    print(f"route rows={rows} experts={experts} top={top} groups={groups} keep={keep}", flush=True)
    _route_case("cuda", rows, experts, top, groups, keep)
    if groups == 1:
        _route_case("cuda", rows, experts, top, groups, keep, sigmoid=True)


# a shared expert of the experts' padded size is one more product of their launches: fewer, as many and more choices than products
SHARED_AMONG = [(1, 64, 40, 8, 2, 40), (4, 64, 40, 8, 2, 50), (5, 96, 33, 8, 2, 64), (3, 32, 32, 2, 1, 32)]


@needs_clang
@pytest.mark.parametrize("case", range(len(SHARED_AMONG)))
def test_shared_expert_among_the_experts_on_cpu_shim(case):
    with emu_util.emulated():
        Z.moe_case("cpu", Z.BF, *SHARED_AMONG[case])


@pytest.mark.gpu
@pytest.mark.parametrize("case", SHARED_AMONG + [(8, 2048, 768, 64, 8, 768), (1, 2048, 768, 64, 8, 768), (32, 2048, 768, 16, 8, 768)])
def test_shared_expert_among_the_experts_gpu(case):
    Z.moe_case("cuda", Z.BF, *case)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,width,ff,experts,top", [(1, 64, 32, 8, 2), (1, 2048, 768, 64, 8), (8, 2048, 768, 64, 8), (17, 2048, 768, 16, 8), (32, 256, 96, 16, 8)])
def test_shared_expert_among_the_experts_has_the_bits_of_launches_of_its_own_gpu(rows, width, ff, experts, top):
    from tah_amd import ops
    from tah_amd.mixers import GatedMlp, MoeMlp, PackedBatch, Router, Step

    class Engine:
        packed, device = True, torch.device("cuda")
    g = torch.Generator().manual_seed(rows + width)
    w = lambda *s: (torch.randn(*s, generator=g) * s[-1] ** -0.5).to(torch.bfloat16).cuda()
    routed = {"router": 3 * w(experts, width), "gate": w(experts, ff, width), "up": w(experts, ff, width), "down": w(experts, width, ff)}
    shared = {"gate": w(ff, width), "up": w(ff, width), "down": w(width, ff), "sg": 2 * w(1, width)}
    x = torch.randn(rows, width, generator=g).to(torch.bfloat16).cuda()
    zeros = torch.zeros(rows, dtype=torch.int32, device="cuda")
    step = lambda: Step(x.float(), x, zeros, ops.linear_pack_rows(x), slot=zeros)
    m = MoeMlp(Router(top), routed, shared, width)
    assert m.shared_among
    got = m.bind(Engine).rows(step())
    # the same weights, the shared expert in two launches beside the experts'
    m.shared_among, m.shared = False, GatedMlp(shared, width)
    m.gate_up_rows, m.down_rows = PackedBatch(m.gate_up, gate_up=True), PackedBatch(m.down)
    want = m.bind(Engine).rows(step())
    assert torch.equal(got.y, want.y) and torch.equal(got.index, want.index) and torch.equal(got.weight, want.weight) and torch.equal(got.y_scale, want.y_scale)
    assert got.index_scale == want.index_scale and got.index_row == want.index_row
    at = (want.index.long() * want.index_scale + torch.arange(rows, device="cuda")[:, None] * want.index_row).flatten()
    assert torch.equal(got.experts[at], want.experts[at])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cols,width,groups", [(2048, 2048, 1), (2048, 2048, 8), (2048, 2040, 5), (4096, 4096, 8), (8192, 8192, 8), (16384, 16384, 1)])
def test_a_rows_norm_does_not_depend_on_how_many_rows_the_call_has_gpu(dtype, cols, width, groups):
    """Calls of up to 256 rows ask for everything at once, others do not: two kernels, the same bits of a row.  (The residual rows
    in float32: they show the last bit of the norm in front of the sum, and so does the float32 result of the one behind it.)"""
    from tah_amd.ops import _call
    g = torch.Generator().manual_seed(cols + groups)
    r = lambda *s: torch.nn.functional.pad(torch.randn(*s, width, generator=g), (0, cols - width)).cuda()
    x, y, coef, norm = r(300), r(300).to(dtype), r(), r()

    def run(rows):
        out, normed = x[:rows].clone(), torch.zeros(rows, cols, dtype=dtype, device="cuda")
        _call("residual_norm", out, coef, width, 1e-5, y[:rows], None, None, None, None, None, None, norm, normed, None, 1, 0, groups,
              width // groups if groups > 1 else cols, None, None, None)
        return out, normed

    (a, na), (b, nb) = run(300), run(64)
    assert torch.equal(a[:64], b) and torch.equal(na[:64], nb)
