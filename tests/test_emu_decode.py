"""Decode and KV-append kernels on the CPU execution shim against the oracle.  No GPU."""
import numpy as np
import pytest
import torch

from oracle import duo_oracle as O
from tests import emu_util
from tests.cases import build_slabs, make_decode_case

pytestmark = pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")


def oracle_decode(c):
    f = lambda x: x.float().numpy()
    nseq = len(c["lens"])
    o0, l0 = O.duo_decode_f64(f(c["q1"]), f(c["k1"]), f(c["v1"]), c["cu_k1"], f(c["k2"]), f(c["v2"]), c["pos_k2"],
                              c["cu_k2"], c["q_pos"], [0] * nseq, c["scale"])
    hr = c["hard_rows"]
    q2full = np.zeros((nseq,) + tuple(c["q2"].shape[1:]))
    q2full[hr] = f(c["q2"])
    o1, l1 = O.duo_decode_f64(q2full, f(c["k1"]), f(c["v1"]), c["cu_k1"], f(c["k2"]), f(c["v2"]), c["pos_k2"],
                              c["cu_k2"], c["q_pos"], [1] * nseq, c["scale"])
    return o0, l0, o1[hr], l1[hr]


# The last case has 16 (query, kv head) pairs: in the CPU execution build such calls run one workgroup per pair over
# both segments (duo_decode_whole_kernel; the MI355X build does from 256 pairs on, see the GPU tests).
@pytest.mark.parametrize("hq,hkv,lens", [(2, 1, [700, 3, 513]), (4, 1, [40]), (2, 2, [1030]), (8, 1, [70, 5]),
                                         (16, 8, [150, 37])])
def test_decode_and_append_on_cpu_shim(hq, hkv, lens):
    from tah_amd import kv_cache
    c = make_decode_case(20 + hq, lens, 0.2, Hq=hq, Hkv=hkv, hard_new=[True] + [False] * (len(lens) - 1))
    with emu_util.emulated():
        s1, s2 = build_slabs(c, 1100, 600)
        assert s1.len.tolist() == lens and s2.len.tolist() == np.diff(c["cu_k2"]).tolist()
        assert int(s1.overflow) == 0
        nseq = len(lens)
        slot = torch.arange(nseq, dtype=torch.int32)
        qpos = torch.from_numpy(c["q_pos"])
        o0, l0 = kv_cache.decode(c["q1"], slot, qpos, s1, None, scale=c["scale"], depth=0, return_lse=True)
        hr = torch.tensor(c["hard_rows"], dtype=torch.int32)
        o1, l1 = kv_cache.decode(c["q2"], hr, qpos[hr.long()], s1, s2, scale=c["scale"], depth=1, return_lse=True)
        # both depths in one launch
        qd = torch.tensor([0] * nseq + [1] * len(hr), dtype=torch.int32)
        packed = torch.full((32 * hq * 128,), 3.0, dtype=torch.bfloat16) if nseq + len(hr) <= 32 else None
        om = kv_cache.decode(torch.cat([c["q1"], c["q2"]]), torch.cat([slot, hr]), torch.cat([qpos, qpos[hr.long()]]),
                             s1, s2, scale=c["scale"], q_depth=qd, out_packed=packed)
        # a query without a sequence (slot -1, as a generation loop marks its finished rows): zeros, -inf, nothing read
        gone = slot.clone()
        gone[0] = -1
        og, lg = kv_cache.decode(c["q1"], gone, qpos, s1, None, scale=c["scale"], depth=0, return_lse=True)
        assert not og[0].any() and torch.isinf(lg[0]).all() and torch.equal(og[1:], o0[1:]) and torch.equal(lg[1:], l0[1:])
    # the same output as the rows operand of the o projection; rows past the last query are left alone
    if packed is not None:
        from tests.test_linear_rows import unpack_rows
        rows = unpack_rows(packed, hq * 128)
        assert torch.equal(rows[:om.shape[0]], om.reshape(om.shape[0], -1)) and (rows[om.shape[0]:] == 3.0).all()
    w0, wl0, w1, wl1 = oracle_decode(c)
    np.testing.assert_allclose(o0.float().numpy(), w0, atol=2e-2, rtol=2e-2)
    np.testing.assert_allclose(l0.numpy(), wl0, atol=2e-3, rtol=1e-3)
    np.testing.assert_allclose(o1.float().numpy(), w1, atol=2e-2, rtol=2e-2)
    np.testing.assert_allclose(l1.numpy(), wl1, atol=2e-3, rtol=1e-3)
    assert torch.equal(om[:nseq], o0)
    if nseq * hkv < 16:
        assert torch.equal(om[nseq:], o1)
    else:  # the depth-1 query alone went through split-K, in the joint call through the one-workgroup kernel: other sum order
        np.testing.assert_allclose(om[nseq:].float().numpy(), o1.float().numpy(), atol=2e-2, rtol=2e-2)


def test_append_is_exact_and_flags_overflow():
    from tah_amd.kv_cache import KvSlabs
    with emu_util.emulated():
        s = KvSlabs(3, 5, 2, with_pos=True, device="cpu")
        g = torch.Generator().manual_seed(0)
        k = torch.randn(6, 2, 128, generator=g).to(torch.bfloat16)
        v = torch.randn(6, 2, 128, generator=g).to(torch.bfloat16)
        pos = torch.arange(6, dtype=torch.int32) * 3
        # rows 0-1 -> slot 2, rows 2-5 -> slot 0
        s.append(k, v, torch.tensor([0, 2, 6], dtype=torch.int32), pos_new=pos, slot_of=torch.tensor([2, 0], dtype=torch.int32))
        assert s.len.tolist() == [4, 0, 2]
        assert torch.equal(s.k[2, :, :2], k[:2].transpose(0, 1)) and torch.equal(s.v[0, :, :4], v[2:].transpose(0, 1))
        assert s.pos[2, :2].tolist() == [0, 3] and s.pos[0, :4].tolist() == [6, 9, 12, 15]
        assert int(s.overflow) == 0
        s.append(k[:3], v[:3], torch.tensor([0, 3], dtype=torch.int32), pos_new=pos[:3], slot_of=torch.tensor([0], dtype=torch.int32))
        assert s.len.tolist() == [5, 0, 2] and int(s.overflow) == 1
        assert torch.equal(s.k[0, :, 4], k[0])


def test_fused_decode_step_equals_prep_then_decode_on_cpu_shim():
    """16 (query, kv head) pairs: the CPU execution build takes such calls in one launch."""
    from tests import decode_step_case
    from tah_amd import kv_cache
    with emu_util.emulated():
        assert kv_cache.decode_step_supported(2, 16, 8, 128) and not kv_cache.decode_step_supported(1, 16, 8, 128)
        assert not kv_cache.decode_step_supported(2, 32, 8, 128)  # four query heads per kv head
        decode_step_case.run("cpu", B=3, hq=16, hkv=8, seed=5)
        decode_step_case.run("cpu", B=2, hq=8, hkv=8, seed=6, full_slab=True)
        decode_step_case.run_mixed("cpu", B=4, hq=8, hkv=8, seed=7)
        decode_step_case.run("cpu", B=3, hq=8, hkv=8, seed=5, slots=[1, -1, 0])  # not row i in slot i; fewer slots than rows


def test_fused_decode_step_with_a_pairs_rows_shared_by_workgroups_on_cpu_shim():
    """Fewer pairs than the one-workgroup kernel wants, slabs of 1500 rows: up to four workgroups per pair, the last one merges.
    Without a workspace such calls are refused; too small a one is refused too."""
    from tests import decode_step_case
    from tah_amd import TahDuoError, kv_cache
    with emu_util.emulated():
        ws = kv_cache.decode_step_workspace(3, 2, 1, 1500, 700, "cpu")  # the largest of three sizes serves all
        decode_step_case.run("cpu", B=2, hq=1, hkv=1, seed=9, max_len=600, cap2=300, full_slab=True, workspace=ws)
        decode_step_case.run("cpu", B=3, hq=2, hkv=1, seed=8, max_len=1400, cap1=1500, cap2=700, workspace=ws)
        decode_step_case.run_mixed("cpu", B=4, hq=2, hkv=1, seed=10, max_len=1400, cap1=1500, cap2=700, workspace=ws)
        decode_step_case.run_mixed("cpu", B=3, hq=2, hkv=1, seed=11, max_len=700, cap1=720, cap2=300, workspace=True, slots=[5, 2, 0])
        decode_step_case.run("cpu", B=2, hq=2, hkv=1, seed=16, max_len=1000, cap1=1024, workspace=True, infinite=True)
        with pytest.raises(TahDuoError):
            decode_step_case.run("cpu", B=3, hq=2, hkv=1, seed=8, workspace=-16)
        with pytest.raises(TahDuoError):
            decode_step_case.run("cpu", B=3, hq=2, hkv=1, seed=8)
        assert kv_cache.decode_step_workspace(3, 4, 1, 1500, 700, "cpu") is None  # four query heads per kv head


def test_fused_decode_step_with_an_empty_segment_without_pointers_on_cpu_shim():
    """A depth-1 segment of no capacity, described by null pointers: beside queries of depth 0, and as the place of a new row that
    does not fit.  And a depth-0 segment of that kind beside a depth-1 segment that takes the rows."""
    import ctypes as C

    from tah_amd import _capi, kv_cache
    from tah_amd.kv_cache import KvSlabs
    B, hq, hkv = 2, 8, 8
    g = torch.Generator().manual_seed(4)
    rn = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32)
    q, k, v, qw, kw = rn(B, hq, 128), rn(B, hkv, 128), rn(B, hkv, 128), rn(128), rn(128)
    ang = torch.randn(B, 128, generator=g)
    cos, sin = ang.cos().to(torch.bfloat16), ang.sin().to(torch.bfloat16)
    rows, cu, pos = i32(0, 1), i32(0, 1, 2), i32(20, 33)
    scale = 128 ** -0.5

    def slabs(with_pos=False):
        s = KvSlabs(B, 48, hkv, 128, with_pos=with_pos, device="cpu")
        gs = torch.Generator().manual_seed(5)
        s.k.copy_(torch.randn(s.k.shape, generator=gs).to(torch.bfloat16))
        s.v.copy_(torch.randn(s.v.shape, generator=gs).to(torch.bfloat16))
        s.len.copy_(pos)
        if with_pos:
            s.pos.copy_(torch.arange(48, dtype=torch.int32))
        return s

    def segment(s):
        if s is None:
            return _capi.KvSegment(nslots=B)
        ptr = lambda t: None if t is None else t.data_ptr()
        return _capi.KvSegment(ptr(s.k), ptr(s.v), ptr(s.pos), ptr(s.start), ptr(s.len), s.k.stride(2), s.k.stride(1), s.v.stride(2), s.v.stride(1),
                               s.capacity, B)

    def step(lib, c1, c2, cache, q_slot, q_depth, append_at, append_depth=None, pos_new=None):
        o = torch.zeros(B, hq, 128, dtype=torch.bfloat16)
        prep = _capi.QkPrepArgs(q=q.data_ptr(), k=k.data_ptr(), v=v.data_ptr(), q_weight=qw.data_ptr(), k_weight=kw.data_ptr(), cos=cos.data_ptr(),
                                sin=sin.data_ptr(), cos_sin_row_stride=128, eps=1e-6, rows=B, hq=hq, hkv=hkv, d=128, append=1, nseq=B,
                                append_one_row_per_seq=1, cu_new=cu.data_ptr(), slot_of=q_slot.data_ptr(), cache=segment(cache),
                                overflow=cache.overflow.data_ptr(), pos_new=None if pos_new is None else pos_new.data_ptr())
        for name in ("q", "k", "v"):
            setattr(prep, f"{name}_row_stride", (hq if name == "q" else hkv) * 128)
            setattr(prep, f"{name}_head_stride", 128)
        dec = _capi.DuoDecodeArgs(o=o.data_ptr(), o_row_stride=hq * 128, o_head_stride=128, q_slot=rows.data_ptr(), q_pos=pos.data_ptr(),
                                  q_depth=q_depth.data_ptr(), c1=segment(c1), c2=segment(c2), nq=B, hq=hq, hkv=hkv, d=128, scale=scale)
        assert lib.tah_duo_decode_step(C.byref(prep), C.byref(dec), append_at.data_ptr(), None if append_depth is None else append_depth.data_ptr(), None) == 0
        return o

    with emu_util.emulated() as lib:
        def whole(c1, q_slot):
            return kv_cache.decode_step(q, k, v, qw, kw, cos, sin, 1e-6, cache=c1, cu_new=cu, append_at=c1.len.clone(), q_slot=rows, q_pos=pos, c1=c1,
                                        c2=None, scale=scale, slot_of=q_slot)
        a, b = slabs(), slabs()
        want = whole(a, rows)
        assert torch.equal(step(lib, b, None, b, rows, i32(0, 0), pos.clone()), want)
        assert torch.equal(a.k, b.k) and torch.equal(a.len, b.len) and int(b.overflow) == 0
        # row 0 appends to the depth-1 segment: no room, so it attends over what is cached
        a, b = slabs(), slabs()
        want = whole(a, i32(-1, 1))
        assert torch.equal(step(lib, b, None, b, rows, i32(1, 0), i32(0, 33), i32(1, 0)), want)
        assert torch.equal(a.k, b.k) and torch.equal(a.len, b.len) and int(b.overflow) == 1
        # no depth-0 rows: what the call gives over a depth-0 segment without any
        a, b, none = slabs(True), slabs(True), slabs()
        none.len.zero_()
        want = step(lib, none, a, a, rows, i32(1, 1), pos.clone(), pos_new=pos)
        assert torch.equal(step(lib, None, b, b, rows, i32(1, 1), pos.clone(), pos_new=pos), want)
        assert torch.equal(a.k, b.k) and torch.equal(a.len, b.len)
