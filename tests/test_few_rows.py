"""Dense layers of a prompt's few rows (its hard tokens, the rows in front of the output head, a short prompt) on the decode step's kernels."""
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


@pytest.mark.gpu
@pytest.mark.parametrize("lens,hard", [([5], 2), ([20, 12], 32), ([20, 13], 33), ([200, 90], 3)])
def test_prompts_of_few_rows_against_library_products_gpu(lens, hard):
    """The same prompts on an engine with packed linear layers and on one without, up to and past the rows they take: logits and both
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
        assert eng._few(32) == packed and not eng._few(33)
    for a, b in zip(*got):
        assert (a - b).norm() <= 0.02 * a.norm(), float((a - b).norm() / a.norm())
