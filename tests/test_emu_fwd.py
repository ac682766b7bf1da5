"""Runs the HIP forward and pack kernels on the CPU execution shim against the oracle.  No GPU."""
import numpy as np
import pytest
import torch

from oracle import duo_ref as R
from tests import emu_util
from tests.cases import add_score_drift, make_varlen_case, varlen_args

pytestmark = pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")

TOL = dict(atol=2e-2, rtol=2e-2)  # bf16 outputs vs float64-accumulated oracle on bf16-rounded inputs


def _to_dev(case):
    out = {}
    for k, v in case.items():
        if isinstance(v, np.ndarray):
            out[k] = torch.from_numpy(v.copy())
        elif torch.is_tensor(v):
            out[k] = v.to(torch.bfloat16)
        else:
            out[k] = v
    return out


def _oracle(dev):
    args = [a.float().numpy() if torch.is_tensor(a) and a.is_floating_point() else
            (a.numpy() if torch.is_tensor(a) else a) for a in varlen_args(dev)]
    return R.fwd(*args)


def _check(dev, got):
    o1, lse1, o2, lse2 = _oracle(dev)
    np.testing.assert_allclose(got[0].float().numpy(), o1, **TOL)
    np.testing.assert_allclose(got[1].numpy(), lse1, atol=2e-3, rtol=1e-3)
    np.testing.assert_allclose(got[2].float().numpy(), o2, **TOL)
    np.testing.assert_allclose(got[3].numpy(), lse2, atol=2e-3, rtol=1e-3)


@pytest.mark.parametrize("hq,hkv,seqlens,p", [
    (2, 1, [70], 0.3),           # G=2, one partial tile, depth-1 rows
    (2, 2, [130, 3], 0.1),       # G=1, 256-row tiles, second tiny sequence
    (4, 1, [65, 64], 0.2),       # G=4, 64-row tiles
    (2, 1, [3, 0, 9, 1] * 17 + [40], 0.3),   # 69 sequences: the tile lookup takes them 64 at a time
])
def test_fwd_kernel_on_cpu_shim(hq, hkv, seqlens, p):
    from tah_amd import ops
    dev = _to_dev(make_varlen_case(100 + hq, seqlens, p, Hq=hq, Hkv=hkv, D=128))
    with emu_util.emulated():
        got = ops.duo_fwd_varlen(*varlen_args(dev))
    _check(dev, got)


@pytest.mark.parametrize("nats_per_key", [0.25, 0.02])
def test_fwd_kernel_moving_softmax_reference(nats_per_key):
    """Scores that keep growing along the keys: per 64-key tile the row maximum rises by 16 nats (the
    exponent reference has to follow in every tile) or by 1.3 nats (it follows only every few tiles)."""
    from tah_amd import ops
    dev = _to_dev(add_score_drift(make_varlen_case(21, [200], 0.2, Hq=2, Hkv=1, D=128), nats_per_key))
    with emu_util.emulated():
        got = ops.duo_fwd_varlen(*varlen_args(dev))
    _check(dev, got)


@pytest.mark.parametrize("rows,p", [(258, 0.1)])
def test_fwd_of_a_head_does_not_depend_on_its_group(rows, p):
    """Eight query heads of one kv head (8-wave workgroups) and the same heads four at a time (4-wave workgroups): the same
    bits.  The probabilities are rounded to bf16 under a reference that moves along the keys, so this holds only if a
    query's keys are always taken one after another from the first."""
    from tah_amd import ops
    eight = _to_dev(make_varlen_case(61, [rows], p, Hq=8, Hkv=1, D=128))
    with emu_util.emulated():
        want = ops.duo_fwd_varlen(*varlen_args(eight))
        for h in (0, 4):
            four = dict(eight, q1=eight["q1"][:, h:h + 4].contiguous(), q2=eight["q2"][:, h:h + 4].contiguous())
            o1, lse1, o2, lse2 = ops.duo_fwd_varlen(*varlen_args(four))
            assert torch.equal(o1, want[0][:, h:h + 4]) and torch.equal(lse1, want[1][h:h + 4])
            assert torch.equal(o2, want[2][:, h:h + 4]) and torch.equal(lse2, want[3][h:h + 4])


def test_fwd_kernel_cache_prefix_and_strided_views():
    from tah_amd import ops
    dev = _to_dev(make_varlen_case(7, [5, 40], 0.5, Hq=2, Hkv=1, D=128, seqlens_k=[90, 40], extra_k2=70))
    # q/k/v as strided views of a fused [rows, Hq+2*Hkv, D] projection buffer
    fused = torch.zeros(dev["q1"].shape[0], 4, 128, dtype=torch.bfloat16)
    fused[:, :2] = dev["q1"]
    dev["q1"] = fused[:, :2]
    with emu_util.emulated():
        got = ops.duo_fwd_varlen(*varlen_args(dev))
    _check(dev, got)


def test_fwd_depth1_only_call():
    """Depth-1 queries alone against cached depth-0 and depth-1 keys (the per-layer call at depth 1)."""
    from tah_amd import ops
    dev = _to_dev(make_varlen_case(9, [33], 0.4, Hq=2, Hkv=1, D=128))
    want = _oracle(dev)
    d1 = dict(dev)
    d1["q1"] = dev["q1"][:0]
    d1["cu_q1"] = torch.zeros(2, dtype=torch.int32)
    with emu_util.emulated():
        got = ops.duo_fwd_varlen(*varlen_args(d1))
    assert got[0].shape[0] == 0
    np.testing.assert_allclose(got[2].float().numpy(), want[2], **TOL)


@pytest.mark.parametrize("B,S,p", [(3, 50, 0.3), (2, 9000, 0.06), (1, 1, 1.0), (4, 16, 0.0)])
def test_hard_index_bit_exact(B, S, p):
    from tah_amd import ops
    g = torch.Generator().manual_seed(B * 1000 + S)
    mask = torch.rand(B, S, generator=g) < p
    with emu_util.emulated():
        pos, flat, seq, cu = ops.hard_index_build(mask)
        n = int(cu[-1])
        pad = ops.pad_rows_build(cu, seq, n, max(int((cu[1:] - cu[:-1]).max()), 1))
    nz = mask.nonzero()
    assert cu.tolist() == [0] + torch.cumsum(mask.sum(1), 0).tolist()
    assert pos[:n].tolist() == nz[:, 1].tolist()
    assert seq[:n].tolist() == nz[:, 0].tolist()
    assert flat[:n].tolist() == (nz[:, 0] * S + nz[:, 1]).tolist()
    ridx, rcu = R.hard_index(mask.numpy())
    assert ridx.tolist() == pos[:n].tolist() and rcu.tolist() == cu.tolist()
    width = max(int(mask.sum(1).max()), 1)
    rank = torch.cat([torch.arange(int(c)) for c in mask.sum(1)]) if n else torch.zeros(0, dtype=torch.long)
    assert pad.tolist() == (nz[:, 0] * width + rank).tolist()


@pytest.mark.parametrize("dtype,inner", [(torch.bfloat16, (8,)), (torch.int64, ()), (torch.uint8, (3,)), (torch.float32, (5, 2))])
def test_rows_copy_bit_exact(dtype, inner):
    from tah_amd import ops
    g = torch.Generator().manual_seed(3)
    src = torch.randint(0, 100, (40,) + inner, generator=g).to(dtype)
    rows = torch.randperm(40, generator=g)[:17].to(torch.int32)
    with emu_util.emulated():
        out = torch.zeros((17,) + inner, dtype=dtype)
        ops.rows_copy(src, rows, out, None, 17)
        back = torch.full_like(src, 7)
        ops.rows_copy(out, None, back, rows, 17)
    assert torch.equal(out, src[rows.long()])
    want = torch.full_like(src, 7)
    want[rows.long()] = src[rows.long()]
    assert torch.equal(back, want)


@pytest.mark.parametrize("hq,hkv,seqlens,p,drift", [(2, 1, [330], 0.3, 0.0), (4, 1, [193, 80], 1.0, 0.25)])
def test_fwd_kernel_chains_of_key_tiles_on_cpu_shim(hq, hkv, seqlens, p, drift):
    """Small launches with at least four key tiles (also where the exponent reference moves far along them)."""
    from tah_amd import ops
    case = make_varlen_case(33, seqlens, p, Hq=hq, Hkv=hkv, D=128)
    dev = _to_dev(add_score_drift(case, drift) if drift else case)
    with emu_util.emulated():
        got = ops.duo_fwd_varlen(*varlen_args(dev))
    _check(dev, got)


@pytest.mark.parametrize("lens,p", [([97], 0.3), ([64, 1, 33], 0.5)])
def test_two_waves_to_the_same_rows_give_the_bits_of_one(lens, p):
    """Few workgroups: two waves share 32 query rows (two heads of a kv head, and one).  The same heads four at a time run with a
    wave to 32 rows: the same bits, outputs and LSE, with a reference that moves (tile edges, idle waves, one-row sequences)."""
    from tah_amd import ops
    four = _to_dev(add_score_drift(make_varlen_case(71, lens, p, Hq=4, Hkv=1, D=128), 0.2))
    with emu_util.emulated():
        want = ops.duo_fwd_varlen(*varlen_args(four))
        for h, n in ((0, 2), (2, 2), (3, 1)):
            part = dict(four, q1=four["q1"][:, h:h + n].contiguous(), q2=four["q2"][:, h:h + n].contiguous())
            o1, lse1, o2, lse2 = ops.duo_fwd_varlen(*varlen_args(part))
            assert torch.equal(o1, want[0][:, h:h + n]) and torch.equal(lse1, want[1][h:h + n])
            assert torch.equal(o2, want[2][:, h:h + n]) and torch.equal(lse2, want[3][h:h + n])


def test_fwd_of_depth0_queries_beside_depth1_keys_without_boundaries():
    """Depth-1 keys that no query looks at, described by their number alone: the outputs of the call without them."""
    import ctypes as C

    from tah_amd import _capi, ops
    dev = _to_dev(make_varlen_case(73, [40], 0.0, Hq=2, Hkv=1, D=128))
    with emu_util.emulated() as lib:
        want = ops.duo_fwd_varlen(*varlen_args(dev))
        o, lse = torch.zeros_like(want[0]), torch.zeros_like(want[1])
        q, k, v = dev["q1"], dev["k1"], dev["v1"]
        s1 = _capi.DuoStream(q=q.data_ptr(), k=k.data_ptr(), v=v.data_ptr(), o=o.data_ptr(), lse=lse.data_ptr(), cu_q=dev["cu_q1"].data_ptr(),
                             cu_k=dev["cu_k1"].data_ptr(), total_q=q.shape[0], total_k=k.shape[0])
        for name, t in (("q", q), ("k", k), ("v", v), ("o", o)):
            setattr(s1, f"{name}_row_stride", t.stride(0))
            setattr(s1, f"{name}_head_stride", t.stride(1))
        a = _capi.DuoFwdArgs(s1=s1, s2=_capi.DuoStream(total_k=7), nseq=1, hq=2, hkv=1, d=128, scale=dev["scale"])
        assert lib.tah_duo_fwd_varlen(C.byref(a), None) == 0
    assert torch.equal(o, want[0]) and torch.equal(lse, want[1])
