"""Dense layers of a prompt's few rows: its hard tokens, the rows in front of the output head, a short prompt."""
import pytest
import torch

from tests import emu_util

BF = torch.bfloat16


def linear_case(dev, rows, n, k):
    from tah_amd.mixers import Linear

    g = torch.Generator().manual_seed(rows)
    x, w = torch.randn(rows, k, generator=g).to(BF), (torch.randn(n, k, generator=g) * k ** -0.5).to(BF)
    got = Linear(w.to(dev))(x.to(dev)).cpu()
    want = x.double() @ w.double().t()
    # one rounding to bf16 of a float32 sum: half an ulp of the largest result, and the sums' own error
    assert got.shape == (rows, n) and (got.double() - want).abs().max() <= want.abs().max() * 2 ** -8 + 1e-3


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
@pytest.mark.parametrize("rows", [1, 32, 33])
def test_linear_of_few_rows_on_cpu_shim(rows):
    with emu_util.emulated():
        linear_case("cpu", rows, 32, 64)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 2, 31, 32, 33])
def test_linear_of_few_rows_gpu(rows):
    linear_case("cuda", rows, 4128, 2048)


def library_case(dev, rows, n, k):
    from tah_amd.mixers import Linear

    g = torch.Generator().manual_seed(rows)
    x, w = torch.randn(rows, k, generator=g).to(BF).to(dev), (torch.randn(n, k, generator=g) * k ** -0.5).to(BF).to(dev)
    assert torch.equal(Linear(w)(x), x @ w.t())


@pytest.mark.skipif(not emu_util.have_host_clang(), reason="host clang++ not available")
@pytest.mark.parametrize("rows", [1, 32])
def test_linear_of_few_rows_is_the_library_s(rows):
    """Products of a prompt take the library's bits, few rows or many.  (Logits come as float32 numbers that were rounded to bf16: another order of
    the sum moves some of them by a whole bf16 step.)"""
    with emu_util.emulated():
        library_case("cpu", rows, 1024, 2048)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 12, 32, 33])
def test_linear_of_few_rows_is_the_library_s_gpu(rows):
    library_case("cuda", rows, 4128, 2048)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,hard", [([5], 2), ([20, 12], 32), ([20, 13], 33), ([200, 90], 3)])
def test_prompts_of_few_rows_against_library_products_gpu(lens, hard):
    """The same prompts on an engine with packed linear layers and on one without, with few rows and more: logits and both
    iterations' cached keys.  Two bf16 layers apart by what a change of summation order travels through them."""
    from tah_amd.engine import EngineConfig, TaHDecodeEngine, Weights

    dev, B, N = "cuda", len(lens), sum(lens)
    # (the second iteration's input mixes every row of the vocabulary: with random weights a choice among nearly equal logits would
    # hang on the last bit of one)
    cfg = EngineConfig(layers=2, hidden=256, intermediate=480, hq=4, hkv=2, vocab=256, topk=256)
    g = torch.Generator().manual_seed(N)
    ids = torch.randint(0, cfg.vocab, (N,), generator=g).to(dev)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    force = torch.zeros(N, dtype=torch.bool)
    force[torch.randperm(N, generator=g)[:min(hard, N)]] = True
    got = []
    for packed in (False, True):
        eng = TaHDecodeEngine(Weights.random_init(cfg, dev, seed=3), B, max(lens) + 4, packed_linear=packed)
        first, _ = eng.prefill(ids, cu, force_hard=force.to(dev))
        got.append([first.float()] + [s.k.float() for s in (eng.slabs0[-1], eng.slabs1[-1])])
    for a, b in zip(*got):
        assert (a - b).norm() <= 0.02 * a.norm(), float((a - b).norm() / a.norm())


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 12, 32, 33])
def test_mlp_of_few_prompt_rows_is_the_library_s_gpu(rows):
    """Prompts of any length take the library's products, whose float32 sum the residual joins before it is rounded (from a dozen rows
    on; below it the library's own split of the sum rounds between): a layer for few rows that rounds its product first is further from
    64 bits (12 rows of 6144 -> 2048: 2.1e-3 against 1.7e-3)."""
    from tah_amd import ops
    from tah_amd.engine import EngineConfig, TaHDecodeEngine, Weights

    cfg = EngineConfig(layers=1, hidden=2048, intermediate=6144, hq=4, hkv=2, vocab=128, topk=16)
    eng = TaHDecodeEngine(Weights.random_init(cfg, "cuda", seed=3), 2, 64, packed_linear=True)
    L = eng.w.layers[0]
    x = torch.randn(rows, cfg.hidden, generator=torch.Generator().manual_seed(rows)).to(BF).cuda()
    act = ops.silu_mul(x @ L["wgu"].t(), norm_input=x, norm_eps=cfg.rms_eps)
    want = torch.addmm(x, act, L["wdown"].t())
    assert torch.equal(eng._mlp(x.clone(), L), want)
