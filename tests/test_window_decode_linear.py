"""A windowed attention's split decode call with the output projection in the merge's launch (tah_window_decode_linear): the bits of
tah_window_decode and tah_linear_rows, for one and two rows, few and many parts, gates and none, heads of two sizes."""
import pytest
import torch

from tests import emu_util

BF = torch.bfloat16
# rows, heads, kv_heads, dim, rotated, window, kept, positions, gate, output columns
CASES = [
    (1, 16, 8, 128, 64, 1024, 4, [1400], True, 2048),           # five parts
    (2, 16, 8, 128, 64, 1024, 4, [1400, 37], True, 2048),       # one row whose later parts saw nothing
    (1, 16, 8, 128, 64, 4096, 0, [3000], False, 8192),          # sixteen parts: two turns; whole tiles of columns
    (2, 32, 4, 64, 32, 512, 8, [511, 0], True, 64),             # a first token; small heads
]


def case_of(dev, rows, heads, kv, dim, rot, window, keep, positions, gate, n):
    from tah_amd import ops
    from tah_amd.kv_cache import WindowCache

    g = torch.Generator().manual_seed(window + rows)
    rnd = lambda *s, dt=BF: (torch.randn(*s, generator=g) * 0.5).to(dt).to(dev)
    row_len, width = dim + rot, heads * dim
    k_col, g_col = heads * dim, heads * dim + kv * row_len
    cols = g_col + (heads if gate else 0)
    cols += -cols % 8
    max_len = max(positions) + 1
    angles = torch.randn(max_len, rot // 2, generator=g)
    cos, sin = angles.cos().to(dev), angles.sin().to(dev)
    weight = rnd(n, width) * 0.1
    packed = ops.linear_pack_weight(weight)
    cached = rnd(3, kv, keep + window, row_len)
    proj = rnd(rows, cols)
    slot = torch.arange(rows, dtype=torch.int32, device=dev)
    pos = torch.tensor(positions, dtype=torch.int32, device=dev)
    got = []
    for fused in (False, True):
        cache = WindowCache(3, kv, keep, window, row_len, device=dev, dtype=BF)
        cache.rows.copy_(cached)
        layer = ops.lib().WindowLayer(cache.rows, cos, sin, heads, dim, dim, rot, rot, 0, keep, window, dim ** -0.5, 0, k_col, g_col if gate else -1)
        ws = torch.zeros(max(int(layer.decode_workspace(rows)), 16), dtype=torch.uint8, device=dev)
        p = proj.clone()
        if fused:
            assert layer.decode_linear_supported(rows, n)
            y = layer.decode_linear(p, slot, pos, packed, n, ws)
        else:
            op = torch.zeros(32 * width, dtype=BF, device=dev)
            layer.decode(p, slot, pos, None, op, ws)
            y = ops.linear_rows(packed, op, rows, n, width)
        got.append((y.cpu(), cache.rows.cpu()))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    assert got[0][0].float().abs().max() > 0
    return layer


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
def test_parts_merged_in_the_projections_launch_on_cpu_shim():
    with emu_util.emulated():
        layer = case_of("cpu", 2, 32, 4, 64, 32, 512, 8, [600, 0], True, 16)
        for rows, n in ((3, 64), (2, 24), (0, 64), (1, 1 << 20)):  # more rows than it is for, columns in no whole tile, too many of them
            assert not layer.decode_linear_supported(rows, n)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_parts_merged_in_the_projections_launch_gpu(case):
    print("case window_decode_linear", case, flush=True)
    case_of("cuda", *case)
