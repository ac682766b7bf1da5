"""What the speed of this package is measured on: calls as users' programs make them, from the smallest to the largest.

A case is a dict of plain values.  ``kind`` names the path:

  prefill   packed attention, forward only (both latent iterations in one call)
  train     packed attention, forward and backward
  layers    the attention of a model's layers as the reference's forward loop drives it: masks, cache, the packing of hard
            tokens, both iterations, backward
  decode    one attention call of a decode step over the KV slabs
  qwen3     the decode engine on a Think-at-Hard model: prompts in, generated tokens out
  zozosun, zedudra   the engine of layer-by-layer decoders: prompts, generated tokens, then a next turn of the conversation

Sizes: the head shape (16 query and 8 key/value heads of 128) and layer sizes are those of the 1.7B Qwen3 architecture and of
the layer-by-layer models that ``bench.py`` times; of the flagship's 28 layers 8 are kept and of the 12 of the others 4,
since every layer costs alike and the weights are made anew for every state.
"""
from __future__ import annotations

import math
import types

import torch

from tah_amd import kv_cache, ops, zedudra, zozosun
from tah_amd.attention import build_attention_mask, duo_attention_forward, duo_attn_varlen
from tah_amd.cache import TaHDuoCache
from tah_amd.engine import EngineConfig, TaHDecodeEngine, Weights
from tah_amd.pack import gather_active

DEV = "cuda"
D = 128
SCALE = D ** -0.5
VOCAB, WIDTH, FF = 151936, 2048, 6144


# ── the cases ────────────────────────────────────────────────────────────────
def listed():
    attn = dict(hq=16, hkv=8)
    return [
        # one short prompt of an interactive user: a launch or two, latency
        dict(name="prefill_333", kind="prefill", seqs=1, lo=333, hi=333, hard=0.06, **attn),
        # a serving batch of long prompts (the headline prefill)
        dict(name="prefill_4x4096", kind="prefill", seqs=4, lo=4096, hi=4096, hard=0.06, **attn),
        # a training step on one long document (the headline forward and backward)
        dict(name="train_8192", kind="train", seqs=1, lo=8192, hi=8192, hard=0.06, **attn),
        # a training step on a pack of documents of unequal length, many hard tokens
        dict(name="train_docs", kind="train", seqs=5, lo=611, hi=3210, hard=0.10, **attn),
        # fine-tuning through the reference's own loop: padded rows, two layers
        dict(name="layers_4x3210", kind="layers", seqs=4, lo=1024, hi=3210, hard=0.10, layers=2, **attn),
        # a decode step of a loaded server: 64 sequences at all lengths (the headline decode)
        dict(name="decode_64", kind="decode", seqs=64, lo=1024, hi=16384, hard=0.06, **attn),
        # a decode step of a few users
        dict(name="decode_3", kind="decode", seqs=3, lo=200, hi=1500, hard=0.06, **attn),
        # one user, a short question, greedy
        dict(name="generate_1", kind="qwen3", seqs=1, lo=203, hi=203, new=96, layers=8, temperature=0.0),
        # a few users, unequal prompts, sampled as reasoning models are
        dict(name="generate_8", kind="qwen3", seqs=8, lo=100, hi=900, new=96, layers=8, temperature=0.6),
        # the end-to-end workload: 32 prompts of 512
        dict(name="generate_32", kind="qwen3", seqs=32, lo=512, hi=512, new=96, layers=8, temperature=0.0),
        # layer-by-layer decoders: a small batch with long prompts, and one user
        dict(name="zozosun_8", kind="zozosun", seqs=8, lo=500, hi=1500, new=64, turn=33, layers=4),
        dict(name="zedudra_1", kind="zedudra", seqs=1, lo=1337, hi=1337, new=64, turn=33, layers=4),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["prefill", "train", "layers", "decode", "qwen3", "zozosun", "zedudra"])
    hard = rng.choice([0.03, 0.06, 0.1, 0.2])
    hq, hkv = rng.choice([(16, 8), (16, 8), (16, 8), (32, 8), (16, 16)])
    if kind in ("prefill", "train"):
        seqs = spread(1, 8)
        hi = spread(64, (16384 if kind == "prefill" else 8192) // seqs)
        return dict(kind=kind, seqs=seqs, lo=max(16, spread(max(16, hi // 8), hi)), hi=hi, hard=hard, hq=hq, hkv=hkv)
    if kind == "layers":
        seqs = spread(1, 4)
        hi = spread(128, 3210)
        return dict(kind=kind, seqs=seqs, lo=spread(max(32, hi // 4), hi), hi=hi, hard=hard, layers=2, hq=hq, hkv=hkv)
    if kind == "decode":
        hi = spread(64, 16384)
        return dict(kind=kind, seqs=spread(1, 64), lo=max(16, spread(max(16, hi // 16), hi)), hi=hi, hard=hard, hq=hq, hkv=hkv)
    seqs = spread(1, 32)
    hi = spread(16, 8192 // seqs if kind == "qwen3" else 4096 // seqs)
    lo = spread(max(8, hi // 8), hi)
    if kind == "qwen3":
        return dict(kind=kind, seqs=seqs, lo=lo, hi=hi, new=spread(24, 96), layers=8, temperature=rng.choice([0.0, 0.6]))
    return dict(kind=kind, seqs=seqs, lo=lo, hi=hi, new=spread(16, 64), turn=spread(2, 64), layers=4)


def lengths(case):
    """Sequence lengths of a case, spread over [lo, hi], the longest one hi."""
    n, lo, hi = case["seqs"], case["lo"], case["hi"]
    return [hi] + [lo + int((hi - lo) * ((i * 0.6180339887) % 1.0)) for i in range(1, n)]


# ── inputs ───────────────────────────────────────────────────────────────────
def generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def normal(g, *shape, std=1.0, dtype=torch.bfloat16):
    t = torch.randn(*shape, generator=g, device=DEV, dtype=dtype)
    return t if std == 1.0 else t.mul_(std)


def boundaries(lens):
    return torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=DEV)


def hard_rows(g, lens, p):
    """Which tokens are hard: (flat rows, positions, boundaries); a share p of every sequence, its last token among them."""
    pos = []
    for n in lens:
        some = torch.randperm(n - 1, generator=g, device=DEV)[:max(1, round(p * n)) - 1]
        pos.append(torch.cat([some.sort().values, torch.full((1,), n - 1, device=DEV)]))
    starts = torch.tensor([0] + lens[:-1], device=DEV).cumsum(0)
    rows = torch.cat([q + a for q, a in zip(pos, starts)])
    return rows, torch.cat(pos).to(torch.int32), boundaries([q.numel() for q in pos])


def packed_inputs(case, seed):
    g, lens = generator(seed), lengths(case)
    n, hq, hkv = sum(lens), case["hq"], case["hkv"]
    rows, pos2, cu2 = hard_rows(g, lens, case["hard"])
    n2 = rows.numel()
    one = lambda rows, heads, std=0.5: normal(g, rows, heads, D, std=std)
    t = dict(q1=one(n, hq), k1=one(n, hkv), v1=one(n, hkv), q2=one(n2, hq), k2=one(n2, hkv), v2=one(n2, hkv),
             g1=one(n, hq, 1.0), g2=one(n2, hq, 1.0))
    return types.SimpleNamespace(lens=lens, cu=boundaries(lens), pos2=pos2, cu2=cu2, **t)


LEAVES = ("q1", "k1", "v1", "q2", "k2", "v2")


def prepare_packed(case, seed):
    s = packed_inputs(case, seed)
    s.train = case["kind"] == "train"
    if s.train:
        for n in LEAVES:
            getattr(s, n).requires_grad_(True)
    # the launch order of the batch's tiles: one table per batch, for all its layers
    s.schedule = ops.duo_schedule(s.cu, s.cu, s.cu2, s.cu2, s.pos2, case["hq"], case["hkv"], s.q1.shape[0], s.k1.shape[0], s.k2.shape[0])
    s.longest = (max(s.lens), int((s.cu2[1:] - s.cu2[:-1]).max()))
    return s


def run_packed(s):
    o1, o2 = duo_attn_varlen(s.q1, s.k1, s.v1, s.cu, s.cu, s.q2, s.k2, s.v2, s.pos2, s.pos2, s.cu2, s.cu2, SCALE, schedule=s.schedule,
                             max_seqlen_k1=s.longest[0], max_seqlen_k2=s.longest[1])
    if not s.train:
        return [o1, o2]
    return [o1, o2, *torch.autograd.grad((o1, o2), [getattr(s, n) for n in LEAVES], (s.g1, s.g2))]


def prepare_layers(case, seed):
    g, lens, n_layers = generator(seed), lengths(case), case["layers"]
    B, T, hq, hkv = len(lens), max(lens), case["hq"], case["hkv"]
    at = torch.arange(T, device=DEV)[None]
    valid = (at < torch.tensor(lens, device=DEV)[:, None]).long()
    rows, pos2, cu2 = hard_rows(g, lens, case["hard"])
    hard = torch.zeros(B, T, dtype=torch.bool, device=DEV)
    hard[torch.repeat_interleave(torch.arange(B, device=DEV), (cu2[1:] - cu2[:-1]).long()), pos2.long()] = True
    W = int((cu2[1:] - cu2[:-1]).max())
    make = lambda n, h: [normal(g, B, n, h, D, std=0.5).requires_grad_(True) for _ in range(n_layers)]
    s = types.SimpleNamespace(lens=lens, valid=valid, hard=hard, pos=(valid.cumsum(-1) - 1).clamp(min=0), n_layers=n_layers)
    # the projections as every layer's linears leave them: of all tokens, and of the hard ones packed to the left
    s.q1, s.k1, s.v1, s.q2, s.k2, s.v2 = make(T, hq), make(T, hkv), make(T, hkv), make(W, hq), make(W, hkv), make(W, hkv)
    s.hidden = normal(g, B, T, WIDTH, std=0.5).requires_grad_(True)
    s.g1, s.g2 = [[normal(g, B, n, hq, D) for _ in range(n_layers)] for n in (T, W)]
    s.gx = normal(g, B, W, WIDTH)
    s.modules = [types.SimpleNamespace(layer_idx=i, num_key_value_groups=hq // hkv) for i in range(n_layers)]
    return s


def run_layers(s):
    cache = TaHDuoCache()
    outs = []

    def iteration(depth, pos, valid, q, k, v):
        mask = build_attention_mask(pos, valid, cache, depth, dtype=torch.bfloat16)
        cache.current_iter_depth, cache.position_ids_to_cache, cache.valid_mask_to_cache = depth, pos, valid
        for i, module in enumerate(s.modules):
            kk, vv = cache.update(k[i].transpose(1, 2), v[i].transpose(1, 2), i)
            outs.append(duo_attention_forward(module, q[i].transpose(1, 2), kk, vv, mask, scaling=SCALE)[0])

    iteration(0, s.pos, s.valid, s.q1, s.k1, s.v1)
    _, pos2, valid2, x2 = gather_active(s.hard, s.pos, s.valid, s.hidden)
    iteration(1, pos2, valid2, s.q2, s.k2, s.v2)
    leaves = [*s.q1, *s.k1, *s.v1, *s.q2, *s.k2, *s.v2, s.hidden]
    grads = torch.autograd.grad([*outs, x2], leaves, [*s.g1, *s.g2, s.gx])
    return [*outs, x2, *grads]


def decode_inputs(case, seed):
    g, lens, hq, hkv = generator(seed), lengths(case), case["hq"], case["hkv"]
    rows, pos2, cu2 = hard_rows(g, lens, case["hard"])
    n_hard = round(case["hard"] * len(lens))  # sequences whose token takes its second iteration in this call
    again = torch.arange(n_hard, dtype=torch.int32, device=DEV) * (len(lens) // max(n_hard, 1))
    s = types.SimpleNamespace(lens=lens, cu=boundaries(lens), cu2=cu2, pos2=pos2, again=again)
    s.k1, s.v1 = [normal(g, sum(lens), hkv, D) for _ in range(2)]
    s.k2, s.v2 = [normal(g, rows.numel(), hkv, D) for _ in range(2)]
    s.slot = torch.cat([torch.arange(len(lens), dtype=torch.int32, device=DEV), again])
    s.qpos = (torch.tensor(lens, dtype=torch.int32, device=DEV) - 1)[s.slot.long()]
    s.depth = torch.cat([torch.zeros(len(lens), dtype=torch.int32, device=DEV), torch.ones(n_hard, dtype=torch.int32, device=DEV)])
    s.q = normal(g, s.slot.numel(), hq, D)
    return s


def prepare_decode(case, seed):
    s = decode_inputs(case, seed)
    hkv, n = case["hkv"], len(s.lens)
    capacity = max(256, 1 << (max(s.lens) - 1).bit_length())
    s.c1 = kv_cache.KvSlabs(n, capacity, hkv, with_pos=False, device=DEV)
    s.c2 = kv_cache.KvSlabs(n, max(256, capacity // 4), hkv, with_pos=True, device=DEV)
    s.c1.append(s.k1, s.v1, s.cu)
    s.c2.append(s.k2, s.v2, s.cu2, pos_new=s.pos2)
    del s.k1, s.v1, s.k2, s.v2
    return s


def run_decode(s):
    return kv_cache.decode(s.q, s.slot, s.qpos, s.c1, s.c2, scale=SCALE, q_depth=s.depth)


# Language models: random weights, but an output head that knows which token follows which -- one long cycle through the
# vocabulary -- so that the next token's logit stands as clear of the others as a trained model's does, and the tokens of a
# generation do not hang on the last bit of a logit.
def followers(g, hard_ids=None):
    """next[t] over the vocabulary, one cycle.  A token of ``hard_ids`` is followed by one that is not."""
    key = torch.randperm(VOCAB, generator=g, device=DEV).double()
    if hard_ids is not None:
        easy = torch.ones(VOCAB, dtype=torch.bool, device=DEV)
        easy[hard_ids] = False
        easy = torch.nonzero(easy).flatten()
        key[easy] = torch.randperm(easy.numel(), generator=g, device=DEV).double()
        key[hard_ids] = torch.randperm(easy.numel(), generator=g, device=DEV)[:hard_ids.numel()].double() + 0.5
    cycle = torch.argsort(key)
    nxt = torch.empty(VOCAB, dtype=torch.long, device=DEV)
    nxt[cycle] = cycle.roll(-1)
    return nxt


def head_for(g, embed, nxt, gain):
    """Output head [vocab, width]: noise, and for every token its predecessor's embedding times ``gain`` (a number or one per
    predecessor)."""
    head = normal(g, VOCAB, WIDTH, std=0.02)
    head[nxt] += embed * gain
    return head


def prompt_inputs(g, case):
    lens = lengths(case)
    return lens, torch.randint(0, VOCAB, (sum(lens),), generator=g, device=DEV)


def qwen3_inputs(case, seed):
    """Prompts and a Qwen3 checkpoint's tensors.  About 6 % of the tokens are hard: they carry a feature that the decider
    knows, so that its decisions are as clear as a trained decider's."""
    g, n_layers = generator(seed), case["layers"]
    mat = lambda o, i: normal(g, o, i, std=i ** -0.5)
    ones = lambda n: normal(g, n, std=0.05).add_(1.0)
    t = {"model.norm.weight": ones(WIDTH)}
    for i in range(n_layers):
        a, m = f"model.layers.{i}.self_attn.", f"model.layers.{i}.mlp."
        t.update({f"model.layers.{i}.input_layernorm.weight": ones(WIDTH), f"model.layers.{i}.post_attention_layernorm.weight": ones(WIDTH),
                  a + "q_proj.weight": mat(16 * D, WIDTH), a + "k_proj.weight": mat(8 * D, WIDTH), a + "v_proj.weight": mat(8 * D, WIDTH),
                  a + "o_proj.weight": mat(WIDTH, 16 * D), a + "q_norm.weight": ones(D), a + "k_norm.weight": ones(D),
                  m + "gate_proj.weight": mat(FF, WIDTH), m + "up_proj.weight": mat(FF, WIDTH), m + "down_proj.weight": mat(WIDTH, FF)})
    hard_ids = torch.nonzero(torch.rand(VOCAB, generator=g, device=DEV) < 0.06).flatten()
    nxt = followers(g, hard_ids)
    embed = normal(g, VOCAB, WIDTH)
    gain = torch.full((VOCAB, 1), 0.016, dtype=torch.bfloat16, device=DEV)
    gain[hard_ids] = 0.036  # (the second iteration's logits are added: the first one's choice has to stand)
    t["lm_head.weight"] = head_for(g, embed, nxt, gain)
    feature = normal(g, WIDTH)
    feature /= feature.float().norm()
    embed[hard_ids] += 24.0 * feature
    t["model.embed_tokens.weight"] = embed
    decider = (mat(512, WIDTH).add_(feature), torch.zeros(512, dtype=torch.bfloat16, device=DEV),
               torch.full((1, 512), 1 / 512, dtype=torch.bfloat16, device=DEV), torch.full((1,), -6.0, dtype=torch.bfloat16, device=DEV))
    lens, ids = prompt_inputs(g, case)
    return types.SimpleNamespace(tensors=t, decider=decider, lens=lens, ids=ids, next=nxt, hard_ids=hard_ids, new=case["new"])


def prepare_qwen3(case, seed):
    s = qwen3_inputs(case, seed)
    w = Weights.from_tensors(s.tensors, EngineConfig(layers=case["layers"]), DEV)
    w.dec_w1, w.dec_b1, w.dec_w2, w.dec_b2 = s.decider
    w.threshold = 0.5
    s.engine = TaHDecodeEngine(w, len(s.lens), max(s.lens) + s.new)
    s.cu = boundaries(s.lens)
    s.sampling = dict(temperature=case["temperature"], top_p=0.95) if case["temperature"] > 0 else {}
    del s.tensors, s.next
    return s


def run_qwen3(s):
    first, hard = s.engine.prefill(s.ids, s.cu)
    tokens = s.engine.generate(first, s.new, **s.sampling)
    last = s.engine.slabs0[-1]  # what the last layer has cached says what every layer below made of every token
    return dict(first=first, hard=hard, tokens=tokens, k=last.k, v=last.v)


def moe_spec(**more):
    return dict({"kind": "moe", "router": {"experts": 64, "top": 8}, "expert": {"ff": 768}}, **more)


def zozosun_config(n_layers):
    delta = {"heads": 32, "kv_heads": 16, "dim": D, "vdim": D, "conv": 4}
    latent = {"heads": 16, "dim": D, "rot_dim": 64, "vdim": D, "kv_rank": 512, "scale": 192 ** -0.5, "rot": {"base": 1e6, "dims": 64},
              "mask": {"size": 1024}}
    return {"architecture": "Zozosun", "width": WIDTH, "vocab": VOCAB, "norm": {"eps": 1e-6},
            "layers": [{"type": "latent_attention" if i % 4 == 3 else "delta", "mixer": latent if i % 4 == 3 else delta,
                        "mlp": moe_spec(shared={"ff": 768}) if i % 2 else {"kind": "dense", "ff": FF}} for i in range(n_layers)]}


def zedudra_config(n_layers):
    mixer = {"heads": 16, "kv_heads": 8, "dim": D, "vdim": D, "scale": SCALE, "rot": {"base": 1e6, "dims": 64},
             "mask": {"size": 1024, "keep_first": 4}}
    moe = moe_spec(router={"experts": 64, "top": 8, "groups": {"count": 8, "keep": 4}}, expert={"ff": 768, "limit": 7.0})
    return {"architecture": "Zedudra", "width": WIDTH, "vocab": VOCAB, "norm": {"eps": 1e-6, "groups": 8}, "canon": {"taps": 4},
            "embedding": {"scale": WIDTH ** 0.5},
            "layers": [{"type": "attention", "mixer": mixer, "mlp": moe if i % 2 else {"kind": "dense", "ff": FF}} for i in range(n_layers)]}


def expert_features(g, grouped):
    """A direction per expert and, for every token of the vocabulary, the sum of those of its eight experts: a router that
    reads them chooses as clearly as a trained one (``grouped``: two experts in each of four groups)."""
    directions = torch.nn.functional.normalize(normal(g, 64, WIDTH).float(), dim=1).to(torch.bfloat16)
    key = torch.rand(VOCAB, 64, generator=g, device=DEV)
    if grouped:
        key = key.view(VOCAB, 8, 8)
        best = (key >= key.topk(2, -1).values[..., -1:]).view(VOCAB, 64)
        key = torch.rand(VOCAB, 8, generator=g, device=DEV)
        chosen = best & (key >= key.topk(4, -1).values[..., -1:]).repeat_interleave(8, 1)
    else:
        chosen = key >= key.topk(8, -1).values[..., -1:]
    return directions, chosen.to(torch.bfloat16) @ directions


def mlp_tensors(g, t, p, spec, directions):
    mat = lambda o, i: normal(g, o, i, std=i ** -0.5)
    if spec["kind"] == "dense":
        t[p + "up"], t[p + "down"] = mat(FF, WIDTH), mat(WIDTH, FF)
        return
    n, ff = spec["router"]["experts"], spec["expert"]["ff"]
    t[p + "router"] = mat(n, WIDTH) * 0.05 + directions * (0.2 if spec.get("shared") else 0.5)
    for leaf, shape in (("gate", (n, ff, WIDTH)), ("up", (n, ff, WIDTH)), ("down", (n, WIDTH, ff))):
        every = normal(g, *shape, std=shape[2] ** -0.5)
        t.update({f"{p}e{e}.{leaf}": every[e] for e in range(n)})
    if spec.get("shared"):
        t.update({p + "shared.gate": mat(ff, WIDTH), p + "shared.up": mat(ff, WIDTH), p + "shared.down": mat(WIDTH, ff),
                  p + "shared.sg": mat(1, WIDTH)})


def stack_inputs(case, seed):
    g, is_zozosun = generator(seed), case["kind"] == "zozosun"
    config = (zozosun_config if is_zozosun else zedudra_config)(case["layers"])
    mat = lambda o, i: normal(g, o, i, std=i ** -0.5)
    near = lambda n, at, std=0.1: normal(g, n, std=std).add_(at)
    t = {}
    directions, features = expert_features(g, not is_zozosun)
    for i, layer in enumerate(config["layers"]):
        p, m = f"l{i}.", layer["mixer"]
        if is_zozosun:
            t.update({p + k: near(WIDTH, at, std) for k, at, std in (("norm1", 0.0, 0.1), ("norm2", 0.0, 0.1), ("ls1", 0.5, 0.2), ("ls2", 0.5, 0.2))})
        else:
            t.update({p + k: near(WIDTH, 1.0) for k in ("norm1", "norm1b", "norm2", "norm2b")})
            t[p + "canon1"] = normal(g, WIDTH, 4, std=0.25)
        mlp_tensors(g, t, p + "mlp.", layer["mlp"], directions)
        if not is_zozosun and layer["mlp"]["kind"] == "dense":
            t[p + "mlp.act"] = normal(g, 2, std=0.5)
        p += "mix."
        if layer["type"] == "delta":
            H, K = m["heads"], m["kv_heads"]
            for k, n in (("q", K * D), ("k", K * D), ("v", H * D)):
                t[p + k], t[f"{p}{k}.conv"] = mat(n, WIDTH), normal(g, n, m["conv"], std=m["conv"] ** -0.5)
            t.update({p + "b": mat(H, WIDTH), p + "a": mat(H, WIDTH), p + "g": mat(H * D, WIDTH), p + "o": mat(WIDTH, H * D),
                      p + "A_log": torch.rand(H, generator=g, device=DEV).mul_(2).sub_(3).to(torch.bfloat16), p + "dt_bias": normal(g, H, std=0.1),
                      p + "norm": near(D, 1.0)})
        elif layer["type"] == "latent_attention":
            H, R, rank = m["heads"], m["rot_dim"], m["kv_rank"]
            t.update({p + "q": mat(H * (D + R), WIDTH), p + "dkv": mat(rank + R, WIDTH), p + "dkv.norm": near(rank, 1.0),
                      p + "uk": mat(H * D, rank), p + "uv": mat(H * D, rank), p + "o": mat(WIDTH, H * D)})
        else:
            H, K = m["heads"], m["kv_heads"]
            t.update({p + "q": mat(H * D, WIDTH), p + "k": mat(K * D, WIDTH), p + "g": mat(H, WIDTH), p + "o": mat(WIDTH, H * D)})
    t["final.norm"] = near(WIDTH, 0.0 if is_zozosun else 1.0)
    nxt, embed = followers(g), normal(g, VOCAB, WIDTH)
    t["head"] = head_for(g, embed, nxt, 0.025 if is_zozosun else 0.03)
    embed += features * 20.0
    t["embed"] = embed if is_zozosun else embed * WIDTH ** -0.5
    lens, ids = prompt_inputs(g, case)
    turn = torch.randint(0, VOCAB, (len(lens), case["turn"]), generator=g, device=DEV)
    return types.SimpleNamespace(config=config, tensors=t, lens=lens, ids=ids, next=nxt, new=case["new"], turn=turn)


def prepare_stack(case, seed):
    s = stack_inputs(case, seed)
    design = zozosun if case["kind"] == "zozosun" else zedudra
    model = design.load(s.config, s.tensors, DEV)
    s.engine = design.engine(model, len(s.lens), max(s.lens) + s.new + case["turn"])
    s.cu = boundaries(s.lens)
    s.entries = list(enumerate(s.turn.tolist()))
    s.want = [[case["turn"] - 1]] * len(s.lens)
    del s.tensors, s.next
    return s


def run_stack(s):
    first, _ = s.engine.prefill(s.ids, s.cu)
    tokens = s.engine.generate(first, s.new)
    after = s.engine.extend(s.entries, s.want)  # the next turn: the logits after its last token
    return dict(first=first, tokens=tokens, after=after)


KINDS = {"prefill": (prepare_packed, run_packed), "train": (prepare_packed, run_packed), "layers": (prepare_layers, run_layers),
         "decode": (prepare_decode, run_decode), "qwen3": (prepare_qwen3, run_qwen3), "zozosun": (prepare_stack, run_stack),
         "zedudra": (prepare_stack, run_stack)}


def prepare(case, seed):
    s = KINDS[case["kind"]][0](case, seed)
    s.run = KINDS[case["kind"]][1]
    return s


def run(state):
    return state.run(state)


# ── what a pass cannot do without ────────────────────────────────────────────
def pairs(lens, p):
    """Visible (query, key) pairs per head: depth-0 queries, and hard ones over both depths' keys."""
    return sum(n * (n + 1) / 2 * (1 + p) + (p * n) * (p * n + 1) / 2 for n in lens)


def layer_parameters(kind, i):
    """(parameters every token meets, all parameters) of a layer's matrices."""
    expert = 3 * 768 * WIDTH
    if kind == "qwen3":
        n = WIDTH * (32 * D + 16 * D) + 3 * FF * WIDTH
        return n, n
    if kind == "zedudra":
        mix = WIDTH * (16 * D + 8 * D + 16 + 16 * D)
    elif i % 4 == 3:
        mix = WIDTH * (16 * 192 + 576 + 16 * D) + 2 * 16 * D * 512
    else:
        mix = WIDTH * (2 * 16 * D + 3 * 32 * D + 64)
    if i % 2 == 0:
        return mix + 2 * FF * WIDTH, mix + 2 * FF * WIDTH
    shared = expert if kind == "zozosun" else 0
    return mix + 8 * expert + shared + 64 * WIDTH, mix + 64 * expert + shared + 64 * WIDTH


def work(case):
    kind, lens = case["kind"], lengths(case)
    n, p = sum(lens), case.get("hard", 0.06)
    if kind in ("prefill", "train", "layers"):
        hq, hkv, layers = case["hq"], case["hkv"], case.get("layers", 1)
        rows = n * (1 + p) * layers
        flops = 4.0 * D * hq * pairs(lens, p) * layers
        if kind == "prefill":
            return {"bytes": rows * 2 * D * (2 * hq + 2 * hkv), "flops": flops}
        # forward: q, k, v in, o out; backward: the output's gradient in (o and k, v are at hand), three gradients out
        # (of the layers' hidden rows: the hard ones out and their gradient in, the gradient of all of them out)
        extra = 2 * WIDTH * n * (3 * p + 1) if kind == "layers" else 0
        return {"bytes": rows * 2 * D * (4 * hq + 4 * hkv) + extra, "flops": 3.5 * flops}
    if kind == "decode":
        n_hard = round(p * len(lens))
        rows = n + n_hard * (1 + p) * n / len(lens)
        return {"bytes": rows * 2 * case["hkv"] * D * 2, "flops": rows * 4 * case["hq"] * D}
    # generation: the prompt's products, then for every token all weights that some row meets and the cache so far
    new, layers, B = case["new"], case["layers"], len(lens)
    met, held = [sum(x) for x in zip(*(layer_parameters(kind, i) for i in range(layers)))]
    dense = met - sum(8 * 3 * 768 * WIDTH for i in range(layers) if kind != "qwen3" and i % 2)
    moe = held - met + (met - dense)
    used = dense + moe * (1 - (1 - 8 / 64) ** B)
    again = 1.06 if kind == "qwen3" else 1.0  # hard tokens run through the layers twice
    tokens = n * again + B * new * again + B * case.get("turn", 0)
    head = VOCAB * WIDTH
    # a row's cache per layer: keys and values, or one row for both, or in one layer of four the latents ...
    per_row = {"qwen3": 2 * 8 * D, "zedudra": 8 * 192, "zozosun": 576 / 4}[kind]
    cache = sum(min(x + new / 2, math.inf if kind == "qwen3" else 1028) for x in lens) * per_row * 2 * layers
    if kind == "zozosun":  # ... and in the others the float32 states, read and written
        cache += B * 32 * D * D * 4 * 2 * layers * 3 / 4
    attention = {"qwen3": 4 * 16 * D * pairs(lens, p), "zedudra": 4 * 16 * D * sum(min(x, 1028) * x for x in lens),
                 "zozosun": 2 * 16 * 320 * sum(min(x, 1024) * x for x in lens) / 4 + 4 * 32 * D * D * n * 3 / 4}[kind] * layers
    # one pass over the held weights for the prompt (and the next turn), one per generated token over those that are met
    passes = 1 + (1 if case.get("turn") else 0)
    nbytes = passes * 2 * (held + head) + (new - 1) * (2 * (used + head) + cache) + n * 2 * WIDTH + 4 * B * VOCAB
    return {"bytes": float(nbytes), "flops": 2.0 * met * tokens + 2.0 * head * B * (new * again + 1) + attention}


# Largest differences another correct implementation shows: about four times what these paths measure against exact()
# (attention 0.0023 forward and 0.0032 with gradients, layer-by-layer models 0.0048, eight Qwen3 layers 0.012).
def tolerance(case):
    kind = case["kind"]
    if kind in ("prefill", "decode"):
        return {"rel": 0.01, "max": 0.1}
    if kind in ("train", "layers"):
        return {"rel": 0.013, "max": 0.3}
    if kind == "qwen3":
        return {"rel": 0.03, "max": 0.6, "differ": 0.005}
    return {"rel": 0.02, "max": 0.4, "differ": 0.005}


# ── the same in 64 bits, without the package ─────────────────────────────────
def softmax_products(q, k, v, seen, scale, go=None):
    """q [n, D], k, v [m, D], seen [n, m] -> o, and with the output's gradient also dq, dk, dv."""
    p = torch.softmax((q @ k.t()).mul_(scale).masked_fill_(~seen, -math.inf), -1)
    o = p @ v
    if go is None:
        return (o,)
    dv = p.t() @ go
    ds = p * ((go @ v.t()) - (go * o).sum(-1, keepdim=True))
    return o, (ds @ k) * scale, (ds.t() @ q) * scale, dv


def exact_duo(q1, k1, v1, q2, k2, v2, pos2, g1=None, g2=None):
    """One sequence: o1, o2 and, with gradients, dq1, dk1, dv1, dq2, dk2, dv2 (float64)."""
    n, n2, hq, hkv = q1.shape[0], q2.shape[0], q1.shape[1], k1.shape[1]
    x = [t.detach().double() for t in (q1, k1, v1, q2, k2, v2)]
    q1, k1, v1, q2, k2, v2 = x
    at = torch.arange(n, device=DEV)
    seen1 = at[None] <= at[:, None]
    kpos = torch.cat([at, pos2.long()])
    seen2 = kpos[None] <= pos2.long()[:, None]
    o1, o2 = torch.empty_like(q1), torch.empty_like(q2)
    dq1, dk1, dv1, dq2, dk2, dv2 = (torch.zeros_like(t) for t in x)
    for h in range(hq):
        j = h // (hq // hkv)
        k, v = torch.cat([k1[:, j], k2[:, j]]), torch.cat([v1[:, j], v2[:, j]])
        a = softmax_products(q1[:, h], k1[:, j], v1[:, j], seen1, SCALE, None if g1 is None else g1[:, h].double())
        b = softmax_products(q2[:, h], k, v, seen2, SCALE, None if g2 is None else g2[:, h].double())
        o1[:, h], o2[:, h] = a[0], b[0]
        if g1 is None:
            continue
        dq1[:, h], dq2[:, h] = a[1], b[1]
        dk1[:, j] += a[2] + b[2][:n]
        dv1[:, j] += a[3] + b[3][:n]
        dk2[:, j] += b[2][n:]
        dv2[:, j] += b[3][n:]
    return (o1, o2) if g1 is None else (o1, o2, dq1, dk1, dv1, dq2, dk2, dv2)


def exact_packed(case, seed):
    s = packed_inputs(case, seed)
    parts, cu, cu2 = [], s.cu.tolist(), s.cu2.tolist()
    for b in range(len(s.lens)):
        r, r2 = slice(cu[b], cu[b + 1]), slice(cu2[b], cu2[b + 1])
        g = (s.g1[r], s.g2[r2]) if case["kind"] == "train" else ()
        parts.append(exact_duo(s.q1[r], s.k1[r], s.v1[r], s.q2[r2], s.k2[r2], s.v2[r2], s.pos2[r2], *g))
    return [torch.cat(t) for t in zip(*parts)]


def exact_layers(case, seed):
    s = prepare_layers(case, seed)
    outs = [[], []]
    grads = [[] for _ in LEAVES]
    for i in range(s.n_layers):
        o = [torch.zeros_like(t[i], dtype=torch.float64) for t in (s.q1, s.q2)]
        d = [torch.zeros_like(t[i], dtype=torch.float64) for t in (s.q1, s.k1, s.v1, s.q2, s.k2, s.v2)]
        for b, n in enumerate(s.lens):
            rows = torch.nonzero(s.hard[b]).flatten()
            m = rows.numel()
            e = exact_duo(s.q1[i][b, :n], s.k1[i][b, :n], s.v1[i][b, :n], s.q2[i][b, :m], s.k2[i][b, :m], s.v2[i][b, :m], rows,
                          s.g1[i][b, :n], s.g2[i][b, :m])
            o[0][b, :n], o[1][b, :m] = e[0], e[1]
            for t, x, k in zip(d, e[2:], (n, n, n, m, m, m)):
                t[b, :k] = x
        for all_, x in zip((*outs, *grads), (*o, *d)):
            all_.append(x)
    B, W = s.g2[0].shape[:2]
    x2, dx = torch.zeros(B, W, WIDTH, dtype=torch.float64, device=DEV), torch.zeros_like(s.hidden, dtype=torch.float64)
    for b in range(B):
        rows = torch.nonzero(s.hard[b]).flatten()
        x2[b, :rows.numel()] = s.hidden.detach()[b, rows].double()
        dx[b, rows] = s.gx[b, :rows.numel()].double()
    return [*outs[0], *outs[1], x2, *[t for g in grads for t in g], dx]


def exact_decode(case, seed):
    s = decode_inputs(case, seed)
    out = torch.empty(s.q.shape, dtype=torch.float64, device=DEV)
    cu, cu2, slots = s.cu.tolist(), s.cu2.tolist(), s.slot.tolist()
    for i, b in enumerate(slots):
        k, v = s.k1[cu[b]:cu[b + 1]], s.v1[cu[b]:cu[b + 1]]
        if i >= len(s.lens):  # a second iteration: it sees the depth-1 rows too
            k, v = torch.cat([k, s.k2[cu2[b]:cu2[b + 1]]]), torch.cat([v, s.v2[cu2[b]:cu2[b + 1]]])
        group = s.q.shape[1] // k.shape[1]
        q = s.q[i].double().view(k.shape[1], group, D)
        p = torch.softmax(torch.matmul(q, k.double().permute(1, 2, 0).contiguous()) * SCALE, -1)
        out[i] = torch.matmul(p, v.double().transpose(0, 1).contiguous()).view(-1, D)
    return out


def rms(x, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def silu(x):
    return x * torch.sigmoid(x)


def attention_rows(q, k, v, scale, window=None, keep=0, step=512):
    """One sequence: q [n, hq, dk], k [n, hkv, dk], v [n, hkv, dv], causal, in a window that keeps the first tokens."""
    n, group = q.shape[0], q.shape[1] // k.shape[1]
    k, v = [t.repeat_interleave(group, 1).transpose(0, 1).contiguous() for t in (k, v)]
    at, out = torch.arange(n, device=DEV), []
    for a in range(0, n, step):
        i = at[a:a + step, None]
        seen = at[None] <= i
        if window is not None:
            seen &= (i - at[None] < window) | (at[None] < keep)
        s = torch.matmul(q[a:a + step].transpose(0, 1), k.transpose(1, 2).contiguous()).mul_(scale).masked_fill_(~seen, -math.inf)
        out.append(torch.matmul(torch.softmax(s, -1), v).transpose(0, 1))
    return torch.cat(out)


def rotated(x, angles, pairs_apart):
    """Rotary positions on the last axis: entry i with i + half, or entries 2 i and 2 i + 1; angles (cos, sin) [n, 1, half]."""
    c, s = angles
    half = c.shape[-1]
    u, v = (x[..., :half], x[..., half:2 * half]) if pairs_apart else (x[..., 0:2 * half:2], x[..., 1:2 * half:2])
    a, b = u * c - v * s, v * c + u * s
    turned = torch.cat([a, b], -1) if pairs_apart else torch.stack([a, b], -1).flatten(-2)
    return torch.cat([turned, x[..., 2 * half:]], -1)


def angles(n, base, dims, dtype=None):
    f = base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device=DEV) / dims)
    a = torch.arange(n, dtype=torch.float64, device=DEV)[:, None, None] * f
    c, s = a.cos(), a.sin()
    return (c, s) if dtype is None else (c.to(dtype).double(), s.to(dtype).double())


def whole_rows(s, turn=None):
    """Every sequence's tokens as the path sees them: prompt, generated tokens but the last (it is not fed back), next turn."""
    at, out = 0, []
    for b, n in enumerate(s.lens):
        row = s.ids[at:at + n].tolist()
        at += n
        t = row[-1]
        follow = s.next_list
        for _ in range(s.new - 1):
            t = follow[t]
            row.append(t)
        out.append(row + (turn[b] if turn is not None else []))
    return out


def exact_qwen3(case, seed):
    s = qwen3_inputs(case, seed)
    s.next_list = s.next.tolist()
    rows = whole_rows(s)
    lens = [len(r) for r in rows]
    cu = boundaries(lens).tolist()
    ids = torch.tensor([t for r in rows for t in r], device=DEV)
    t = s.tensors
    w = lambda name: t[name].double()
    x = t["model.embed_tokens.weight"][ids].double()
    cos_sin = angles(max(lens), 1e6, D, torch.bfloat16)  # (the architecture keeps its tables in the model's type)
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        h = rms(x) * w(p + "input_layernorm.weight")
        q, k, v = [(h @ w(f"{p}self_attn.{c}_proj.weight").t()).view(len(ids), -1, D) for c in "qkv"]
        q, k = rms(q) * w(p + "self_attn.q_norm.weight"), rms(k) * w(p + "self_attn.k_norm.weight")
        o = torch.empty_like(q)
        for b, n in enumerate(lens):
            r = slice(cu[b], cu[b + 1])
            a = (cos_sin[0][:n], cos_sin[1][:n])
            q[r], k[r] = rotated(q[r], a, True), rotated(k[r], a, True)
            o[r] = attention_rows(q[r], k[r], v[r], SCALE)
        x = x + o.flatten(1) @ w(p + "self_attn.o_proj.weight").t()
        h = rms(x) * w(p + "post_attention_layernorm.weight")
        x = x + (silu(h @ w(p + "mlp.gate_proj.weight").t()) * (h @ w(p + "mlp.up_proj.weight").t())) @ w(p + "mlp.down_proj.weight").t()
    last = torch.tensor([cu[b] + n - 1 for b, n in enumerate(s.lens)], device=DEV)
    first = (rms(x[last]) * w("model.norm.weight")) @ w("lm_head.weight").t()
    if bool(torch.isin(ids[last], s.hard_ids).any()):
        first = None  # a prompt that ends in a hard token returns both iterations' sum
    slabs = torch.zeros(2, len(lens), 8, max(s.lens) + s.new, D, dtype=torch.float64, device=DEV)
    for b, n in enumerate(lens):
        slabs[0, b, :, :n], slabs[1, b, :, :n] = k[cu[b]:cu[b + 1]].transpose(0, 1), v[cu[b]:cu[b + 1]].transpose(0, 1)
    return dict(first=first, hard=None, tokens=None, k=slabs[0], v=slabs[1])


def exact_mlp(h, w, spec, gate):
    """Mixture of experts on rows h; ``w`` gives a tensor by name, ``gate`` joins an expert's two products."""
    z = h @ w("router").t()
    top, groups = spec["router"]["top"], spec["router"].get("groups")
    if groups is None:
        vals, idx = torch.topk(z, top, -1)
        weight = torch.softmax(vals, -1)
    else:
        z = torch.sigmoid(z)
        best = z.view(len(z), groups["count"], -1).topk(2, -1).values.sum(-1).topk(groups["keep"], -1).indices
        open_ = torch.zeros(len(z), groups["count"], dtype=torch.bool, device=DEV).scatter_(1, best, True)
        open_ = open_.repeat_interleave(z.shape[1] // groups["count"], 1)
        idx = z.masked_fill(~open_, -1.0).topk(top, -1).indices
        weight = z.gather(1, idx)
    out = torch.zeros_like(h)
    for e in range(spec["router"]["experts"]):
        row, place = torch.nonzero(idx == e, as_tuple=True)
        y = gate(h[row] @ w(f"e{e}.gate").t(), h[row] @ w(f"e{e}.up").t()) @ w(f"e{e}.down").t()
        out.index_add_(0, row, y * weight[row, place][:, None])
    if spec.get("shared"):
        y = gate(h @ w("shared.gate").t(), h @ w("shared.up").t()) @ w("shared.down").t()
        out += torch.sigmoid(h @ w("shared.sg").t()) * y
    return out


def causal_conv(x, w):
    """x [..., n, channels] and the taps w [channels, taps], the last one the current token's."""
    taps, n = w.shape[1], x.shape[-2]
    y = torch.zeros_like(x)
    for j in range(min(taps, n)):
        y[..., j:, :] += w[:, taps - 1 - j] * x[..., :n - j, :]
    return y


def delta_rule(x, lens, cu, w, m):
    """The gated delta rule of all sequences side by side, token by token."""
    B, T, H, K = len(lens), max(lens), m["heads"], m["kv_heads"]

    def grid(t):
        out = torch.zeros(B, T, t.shape[-1], dtype=torch.float64, device=DEV)
        for b, n in enumerate(lens):
            out[b, :n] = t[cu[b]:cu[b + 1]]
        return out

    q, k, v = [silu(causal_conv(grid(x @ w(c).t()), w(c + ".conv"))) for c in "qkv"]
    unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)
    q, k = [unit(t.view(B, T, K, D)).repeat_interleave(H // K, 2) for t in (q, k)]
    q, v = q * D ** -0.5, v.view(B, T, H, D)
    beta = torch.sigmoid(grid(x @ w("b").t()))
    decay = torch.exp(-torch.exp(w("A_log")) * torch.nn.functional.softplus(grid(x @ w("a").t()) + w("dt_bias")))
    state, out = torch.zeros(B, H, D, D, dtype=torch.float64, device=DEV), torch.empty(B, T, H, D, dtype=torch.float64, device=DEV)
    for i in range(T):
        state = state * decay[:, i, :, None, None]
        u = beta[:, i, :, None] * (v[:, i] - (state * k[:, i, :, :, None]).sum(2))
        state = state + k[:, i, :, :, None] * u[:, :, None]
        out[:, i] = (state * q[:, i, :, :, None]).sum(2)
    out = torch.cat([out[b, :n] for b, n in enumerate(lens)])
    gate = silu(x @ w("g").t()).view(-1, H, D)
    return (rms(out) * w("norm") * gate).flatten(1) @ w("o").t()


def exact_zozosun_layer(x, lens, cu, w, layer):
    m = layer["mixer"]
    mix = lambda name: w("mix." + name)
    if layer["type"] == "delta":
        y = delta_rule(x, lens, cu, mix, m)
    else:
        H, R, rank = m["heads"], m["rot_dim"], m["kv_rank"]
        q, c = (x @ mix("q").t()).view(-1, H, D + R), x @ mix("dkv").t()
        latent = rms(c[:, :rank]) * mix("dkv.norm")
        kn, v = [(latent @ mix(n).t()).view(-1, H, D) for n in ("uk", "uv")]
        o = torch.empty_like(v)
        cos_sin = angles(max(lens), m["rot"]["base"], R)
        for b, n in enumerate(lens):
            r, a = slice(cu[b], cu[b + 1]), (cos_sin[0][:n], cos_sin[1][:n])
            kr = rotated(c[r, None, rank:], a, True).expand(-1, H, -1)
            qr = rotated(q[r][..., D:], a, True)
            o[r] = attention_rows(torch.cat([q[r][..., :D], qr], -1), torch.cat([kn[r], kr], -1), v[r], m["scale"], m["mask"]["size"])
        y = o.flatten(1) @ mix("o").t()
    x = x + rms(y) * (1.0 + w("norm1")) * w("ls1")
    ff = lambda name: w("mlp." + name)
    if layer["mlp"]["kind"] == "dense":
        y = torch.nn.functional.gelu(x @ ff("up").t(), approximate="tanh") @ ff("down").t()
    else:
        y = exact_mlp(x, ff, layer["mlp"], lambda a, b: silu(a) * b)
    return x + rms(y) * (1.0 + w("norm2")) * w("ls2")


def group_norm(x, weight, groups=8):
    return rms(x.view(len(x), groups, -1)).flatten(1) * weight


def exact_zedudra_layer(x, lens, cu, w, layer):
    m = layer["mixer"]
    h = group_norm(x, w("norm1"))
    h = torch.cat([h[cu[b]:cu[b + 1]] + causal_conv(h[cu[b]:cu[b + 1]], w("canon1")) for b in range(len(lens))])
    q, k = [(h @ w("mix." + c).t()).view(len(x), -1, D) for c in "qk"]
    o = torch.empty_like(q)
    cos_sin = angles(max(lens), m["rot"]["base"], m["rot"]["dims"])
    for b, n in enumerate(lens):
        r, a = slice(cu[b], cu[b + 1]), (cos_sin[0][:n], cos_sin[1][:n])
        o[r] = attention_rows(rotated(q[r], a, False), rotated(k[r], a, False), k[r], m["scale"], m["mask"]["size"], m["mask"]["keep_first"])
    o = o * torch.sigmoid(h @ w("mix.g").t())[:, :, None]
    x = x + group_norm(o.flatten(1) @ w("mix.o").t(), w("norm1b"))
    h = group_norm(x, w("norm2"))
    ff = lambda name: w("mlp." + name)
    if layer["mlp"]["kind"] == "dense":
        z, (a, c) = h @ ff("up").t(), torch.nn.functional.softplus(ff("act"))
        low = z.clamp(max=0)
        y = (torch.where(z > 0, a * z * z, (0.5 + c) * (torch.expm1(low) - low)) + z / 2) @ ff("down").t()
    else:
        limit = layer["mlp"]["expert"]["limit"]
        gated = lambda g, u: (lambda g: g * torch.sigmoid(1.702 * g))(g.clamp(max=limit)) * (u.clamp(-limit, limit) + 1)
        y = exact_mlp(h, ff, layer["mlp"], gated)
    return x + group_norm(y, w("norm2b"))


def exact_stack(case, seed):
    s = stack_inputs(case, seed)
    s.next_list = s.next.tolist()
    rows = whole_rows(s, s.turn.tolist())
    lens = [len(r) for r in rows]
    cu = boundaries(lens).tolist()
    ids = torch.tensor([t for r in rows for t in r], device=DEV)
    is_zozosun = case["kind"] == "zozosun"
    x = s.tensors["embed"][ids].double() * s.config.get("embedding", {"scale": 1.0})["scale"]
    for i, layer in enumerate(s.config["layers"]):
        w = lambda name: s.tensors[f"l{i}.{name}"].double()
        x = (exact_zozosun_layer if is_zozosun else exact_zedudra_layer)(x, lens, cu, w, layer)
    at = torch.tensor([cu[b] + n - 1 for b, n in enumerate(s.lens)] + [c - 1 for c in cu[1:]], device=DEV)
    norm = s.tensors["final.norm"].double()
    h = rms(x[at]) * (1.0 + norm) if is_zozosun else group_norm(x[at], norm)
    logits = h @ s.tensors["head"].double().t()
    B = len(lens)
    return dict(first=logits[:B], tokens=None, after=logits[B:])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "train"):
        return exact_packed(case, seed)
    return {"layers": exact_layers, "decode": exact_decode, "qwen3": exact_qwen3, "zozosun": exact_stack, "zedudra": exact_stack}[kind](case, seed)
