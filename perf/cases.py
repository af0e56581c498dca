"""What a speculative-decoding engine has this framework do, as timed cases.

A case is a dict of plain values; ``kind`` says which entry points it calls:

* ``attention``     one forward's decode/verify attention, layer after layer, over the paged cache
                    (``paged_attention``, or with ``fused`` the prologue inside it);
* ``prefill``       causal attention of a packed batch of prompts (``flash_attn_varlen_func``);
* ``prefill_layer`` what a layer does with its prompts' q/k/v: QK-norm, RoPE, KV store, attention;
* ``ffn``           a decode/verify layer's FFN (``up_gate_silu_and_mul``, ``linear``);
* ``lm_head``       the greedy next token of each row (``lm_head_argmax``);
* ``stack``         a whole decode/verify forward short of the head: its metadata, then the native
                    decoder stack, which leaves the hidden state.

Lengths come from the case alone (so a case is the same work for every seed), in an order that the seed
gives; tensors and block tables come from the seed.  Layer counts are chosen so that a pass streams
more than the last-level cache holds, as a model's layers do, wherever the path is bound by memory.
"""

import itertools
import math
import random

import torch

from nebulasd_amd.config import QWEN3_0_6B, QWEN3_8B, EngineConfig, ModelConfig
from nebulasd_amd.decoder import DecoderStack
from nebulasd_amd.infer_state import build_infer_state, model_rope_cache
from nebulasd_amd.kernels import (flash_attn_varlen_func, linear, lm_head_argmax, paged_attention,
                                  paged_attention_fused, rmsnorm_inplace, rotary_embedding_inplace, store_kvcache,
                                  up_gate_silu_and_mul)

BLOCK = 16
D = 128
DEV = "cuda"


def listed():
    draft = dict(hq=16, hkv=8)
    target = dict(hq=32, hkv=8)
    return [
        # A draft step for four requests with short contexts: the smallest forward, where latency and the
        # number of launches count.
        dict(name="stack_draft_4", kind="stack", hidden=1024, inter=3072, layers=28, batch=4, q_len=1, lo=64, hi=256,
             log=False, **draft),
        # A draft step at the serving batch (Qwen3-0.6B shape, 64 requests): what runs `depth` times a round.
        dict(name="stack_draft_64", kind="stack", hidden=1024, inter=3072, layers=28, batch=64, q_len=1, lo=128,
             hi=1152, log=False, **draft),
        # A verify of 16 requests x 5 rows through four Qwen3-8B layers: what runs once a round.
        dict(name="stack_target_16x5", kind="stack", hidden=4096, inter=12288, layers=4, batch=16, q_len=5, lo=128,
             hi=1152, log=False, **target),
        # Draft decode attention with the prologue in its launch, 64 requests.
        dict(name="decode_draft_64", kind="attention", batch=64, q_len=1, lo=512, hi=2048, log=False, layers=4,
             fused=True, lse=False, **draft),
        # One long request, decoded alone: a chip to fill from eight kv heads.
        dict(name="decode_long_1", kind="attention", batch=1, q_len=1, lo=32000, hi=32000, log=False, layers=8,
             fused=False, lse=False, **target),
        # Target verify at the headline shape: 16 requests, 5 rows each, with the LSE.
        dict(name="verify_target_16x5", kind="attention", batch=16, q_len=5, lo=256, hi=4096, log=False, layers=8,
             fused=False, lse=True, **target),
        # Ragged long-context verify, 9 rows each.
        dict(name="verify_ragged_16x9", kind="attention", batch=16, q_len=9, lo=1024, hi=32768, log=True, layers=2,
             fused=False, lse=True, **target),
        # One prefill chunk of the target: 16 prompts of ordinary lengths.
        dict(name="prefill_target_16", kind="prefill", batch=16, lo=128, hi=1024, log=False, lse=False, **target),
        # Two long prompts of the target.
        dict(name="prefill_long_2", kind="prefill", batch=2, lo=7000, hi=8192, log=False, lse=False, **target),
        # The draft's prefill chunk with the calls that surround its attention.
        dict(name="prefill_layer_draft", kind="prefill_layer", batch=16, lo=128, hi=1024, log=False, layers=4,
             **draft),
        # The target's FFN at 80 verify rows, three layers.
        dict(name="ffn_target_80", kind="ffn", rows=80, hidden=4096, inter=12288, layers=3),
        # The target's next tokens of 80 verify rows.
        dict(name="lm_head_target_80", kind="lm_head", rows=80, hidden=4096, vocab=151936),
    ]


def _between(rng, lo, hi):
    """A whole number in [lo, hi], spread over its logarithm where the range is wide."""
    if hi > 10 * lo:
        return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))
    return rng.randint(lo, hi)


def draw(rng):
    kind = rng.choice(["stack", "attention", "attention", "prefill", "prefill_layer", "ffn", "lm_head"])
    hq, hkv = rng.choice([(16, 8), (32, 8), (16, 8), (32, 8), (8, 8), (64, 8)])
    if kind == "stack":
        big = rng.random() < 0.5
        q_len = rng.randint(2, 8) if big else rng.choice([1, 1, 2])
        batch = _between(rng, 1, 128 // q_len)
        lo = _between(rng, 32, 512)
        return dict(kind=kind, batch=batch, q_len=q_len, lo=lo, hi=lo + _between(rng, 16, 1024), log=False,
                    **(dict(hidden=4096, inter=12288, layers=4, hq=32, hkv=8) if big else
                       dict(hidden=1024, inter=3072, layers=28, hq=16, hkv=8)))
    if kind == "attention":
        q_len = rng.choice([1, 1, 2, 3, 5, 7, 9])
        batch = _between(rng, 1, 128)
        top = min(32768, 160000 // batch)  # cached tokens of one call, as in the largest listed case
        lo = _between(rng, 64, max(65, top // 4))
        hi = _between(rng, lo + 1, max(lo + 1, top))
        log = rng.random() < 0.5
        layers = 2 if batch * (lo + hi) > 160000 else 4
        return dict(kind=kind, hq=hq, hkv=hkv, batch=batch, q_len=q_len, lo=lo, hi=hi, log=log, layers=layers,
                    fused=hq // hkv * q_len <= 48 and rng.random() < 0.5, lse=rng.random() < 0.5)
    if kind in ("prefill", "prefill_layer"):
        hq = min(hq, 32)
        lo = _between(rng, 16, 4096)
        hi = min(8192, rng.randint(lo, 3 * lo))
        batch = _between(rng, 1, max(1, min(32, 12000 // hi)))
        case = dict(kind=kind, hq=hq, hkv=hkv, batch=batch, lo=lo, hi=hi, log=False)
        return dict(case, lse=rng.random() < 0.5) if kind == "prefill" else dict(case, layers=2)
    rows = _between(rng, 1, 128)
    if kind == "ffn":
        hidden, inter = rng.choice([(4096, 12288), (1024, 3072), (2048, 6144)])
        return dict(kind=kind, rows=rows, hidden=hidden, inter=inter, layers=3 if hidden == 4096 else 8)
    return dict(kind=kind, rows=rows, hidden=rng.choice([1024, 2048, 4096]), vocab=rng.choice([151936, 128256, 32000]))


# ---------------------------------------------------------------- inputs


def _lengths(case):
    """One length per request, from the case alone."""
    rng = random.Random("%s %s %s %s" % (case["batch"], case["lo"], case["hi"], case["log"]))
    lo, hi = case["lo"], case["hi"]
    if case["log"]:
        return [round(math.exp(rng.uniform(math.log(lo), math.log(hi)))) for _ in range(case["batch"])]
    return [rng.randint(lo, hi) for _ in range(case["batch"])]


def _model(case):
    base = QWEN3_8B if case.get("hidden", 0) == 4096 or case["hq"] > 16 else QWEN3_0_6B
    return ModelConfig(dict(base, num_hidden_layers=case["layers"], num_attention_heads=case["hq"],
                            num_key_value_heads=case["hkv"],
                            hidden_size=case.get("hidden", base["hidden_size"]),
                            intermediate_size=case.get("inter", base["intermediate_size"])))


class _Maker:
    """Tensors from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)
        self.rng = random.Random(seed)

    def normal(self, *shape, std=1.0):
        t = torch.empty(shape, dtype=torch.float16, device=DEV)
        t.normal_(0.0, std, generator=self.g)
        return t

    def gamma(self, n):
        return (torch.rand(n, device=DEV, generator=self.g) + 0.5).half()


def _cache(make, case, tokens):
    """KV caches filled with values, and a block table of shuffled blocks for these token counts."""
    need = [-(-n // BLOCK) for n in tokens]
    total, width = sum(need) + 1, max(need)
    ids = list(range(total))
    make.rng.shuffle(ids)
    table = torch.full((len(tokens), width), ids[-1], dtype=torch.int32)  # unused entries: a block nobody owns
    at = 0
    for r, n in enumerate(need):
        table[r, :n] = torch.tensor(ids[at:at + n], dtype=torch.int32)
        at += n
    shape = (total, case["layers"], case["hkv"], BLOCK, D)
    return make.normal(*shape), make.normal(*shape), table.to(DEV), EngineConfig(BLOCK, width, len(tokens), total)


def prepare(case, seed):
    make = _Maker(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "lm_head":
        s["w"] = make.normal(case["vocab"], case["hidden"], std=0.02)
        # hidden states that point at a token, as a trained model's do: its logit stands clear of the others
        s["want"] = torch.randint(0, case["vocab"], (case["rows"],), device=DEV, generator=make.g)
        s["x"] = (make.normal(case["rows"], case["hidden"]).float()
                  + 14.0 / (case["hidden"] * 0.02 ** 2) * s["w"][s["want"]].float()).half()
        return s
    if kind == "ffn":
        h, i = case["hidden"], case["inter"]
        s["layers"] = [(make.normal(case["rows"], h), make.normal(2 * i, h, std=h ** -0.5),
                        make.normal(h, i, std=i ** -0.5)) for _ in range(case["layers"])]
        return s
    lengths = _lengths(case)
    make.rng.shuffle(lengths)
    s["lengths"] = lengths
    hq, hkv = case["hq"], case["hkv"]
    if kind == "prefill":
        t = sum(lengths)
        s["cu"] = torch.tensor([0] + list(itertools.accumulate(lengths)), dtype=torch.int32, device=DEV)
        s["q"], s["k"], s["v"] = make.normal(t, hq, D), make.normal(t, hkv, D), make.normal(t, hkv, D)
        return s
    mc = s["mc"] = _model(case)
    if kind == "prefill_layer":
        s["cos"], s["sin"] = model_rope_cache(mc, max(lengths) + 1, DEV)
        s["k_cache"], s["v_cache"], s["table"], s["ec"] = _cache(make, case, lengths)
        s["ids"] = list(range(len(lengths)))
        s["st"] = build_infer_state(s["ids"], [], lengths, mc, s["cos"], s["sin"], DEV)
        s["layers"] = [(make.normal(sum(lengths), (hq + 2 * hkv) * D), make.gamma(D), make.gamma(D))
                       for _ in range(case["layers"])]
        return s
    q_len = case["q_len"]
    s["seq_ids"] = [r for r in range(len(lengths)) for _ in range(q_len)]
    s["seq_lens"] = [n + j + 1 for n in lengths for j in range(q_len)]
    rows = len(s["seq_ids"])
    s["cos"], s["sin"] = model_rope_cache(mc, max(s["seq_lens"]) + 1, DEV)
    s["k_cache"], s["v_cache"], s["table"], s["ec"] = _cache(make, case, [n + q_len for n in lengths])
    if kind == "stack":
        h, i = case["hidden"], case["inter"]
        s["embedded"] = make.normal(rows, h)
        s["layers"] = [dict(wqkv=make.normal((hq + 2 * hkv) * D, h, std=0.02), wo=make.normal(h, hq * D, std=0.02),
                            wug=make.normal(2 * i, h, std=0.02), wd=make.normal(h, i, std=0.02), n_in=make.gamma(h),
                            n_post=make.gamma(h), q_norm=make.gamma(D), k_norm=make.gamma(D))
                       for _ in range(case["layers"])]
        s["stack"] = DecoderStack(mc, s["layers"])
        return s
    s["st"] = build_infer_state(s["seq_ids"], s["seq_lens"], [], mc, s["cos"], s["sin"], DEV)
    if case["fused"]:
        s["layers"] = [(make.normal(rows, (hq + 2 * hkv) * D), make.gamma(D), make.gamma(D))
                       for _ in range(case["layers"])]
    else:
        s["layers"] = [make.normal(rows, hq, D) for _ in range(case["layers"])]
    return s


def _heads(case, qkv):
    hq, hkv = case["hq"], case["hkv"]
    return (qkv[:, :hq * D].view(-1, hq, D), qkv[:, hq * D:(hq + hkv) * D].view(-1, hkv, D),
            qkv[:, (hq + hkv) * D:].view(-1, hkv, D))


# ---------------------------------------------------------------- one pass


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "lm_head":
        return lm_head_argmax(s["x"], s["w"])
    if kind == "ffn":
        out = []
        for x, wug, wd in s["layers"]:
            h = up_gate_silu_and_mul(x, wug)
            out.append((h, linear(h, wd)))
        return out
    if kind == "prefill":
        top = max(s["lengths"])
        lse = torch.empty(s["q"].shape[:2], dtype=torch.float32, device=DEV) if case["lse"] else None
        o = flash_attn_varlen_func(s["q"], s["k"], s["v"], s["cu"], s["cu"], top, top, softmax_scale=D ** -0.5, lse=lse)
        return (o, lse) if case["lse"] else o
    mc, ec, table, kc, vc = s["mc"], s["ec"], s["table"], s["k_cache"], s["v_cache"]
    if kind == "stack":
        st = build_infer_state(s["seq_ids"], s["seq_lens"], [], mc, s["cos"], s["sin"], DEV)
        x = s["embedded"].clone()  # the embedding lookup's output, which the stack overwrites
        residual = torch.zeros_like(x)
        s["stack"].forward(x, residual, kc, vc, table, ec, st, s["cos"], s["sin"])
        x += residual
        return x, kc, vc
    st = s["st"]
    if kind == "prefill_layer":
        cu, top, out = st.prefill_seq_start_locs_with_end, st.max_prefill_len, []
        for li, (qkv, q_norm, k_norm) in enumerate(s["layers"]):
            q, k, v = (t.contiguous() for t in _heads(case, qkv))
            rmsnorm_inplace(q.view(-1, D), q_norm, mc.rms_norm_eps)
            rmsnorm_inplace(k.view(-1, D), k_norm, mc.rms_norm_eps)
            rotary_embedding_inplace(q, k, st)
            store_kvcache(k, v, kc, vc, table, mc, ec, st, li)
            out.append(flash_attn_varlen_func(q, k, v, cu, cu, top, top, softmax_scale=st.softmax_scale))
        return out, kc, vc
    out, rows = [], len(s["seq_ids"])
    for li, layer in enumerate(s["layers"]):
        o = torch.empty((rows, case["hq"], D), dtype=torch.float16, device=DEV)
        lse = torch.empty((rows, case["hq"]), dtype=torch.float32, device=DEV) if case["lse"] else None
        if case["fused"]:
            qkv, q_norm, k_norm = layer
            paged_attention_fused(*_heads(case, qkv), kc, vc, table, q_norm, k_norm, mc, ec, st, li, s["cos"],
                                  s["sin"], o, lse)
        else:
            paged_attention(layer, kc, vc, table, mc, ec, st, li, o, lse)
        out.append((o, lse) if case["lse"] else o)
    return (out, kc, vc) if case["fused"] else out


# ---------------------------------------------------------------- what a pass cannot do without


def work(case):
    kind = case["kind"]
    if kind == "lm_head":
        r, h, v = case["rows"], case["hidden"], case["vocab"]
        return {"bytes": 2 * h * (v + r) + 8 * r, "flops": 2 * r * h * v}
    if kind == "ffn":
        r, h, i, n = case["rows"], case["hidden"], case["inter"], case["layers"]
        return {"bytes": n * 2 * (3 * h * i + 2 * r * h + r * i), "flops": n * 6 * r * h * i}
    hq, hkv = case["hq"], case["hkv"]
    lengths = _lengths(case)
    if kind in ("prefill", "prefill_layer"):
        t, n = sum(lengths), case.get("layers", 1)
        flops = sum(2 * hq * D * m * (m + 1) for m in lengths)
        heads = 2 * hq + 2 * hkv + (2 * hkv if kind == "prefill_layer" else 0)  # q k v in, o out, the cache rows
        lse = 4 * t * hq if case.get("lse") else 0
        return {"bytes": n * (2 * t * heads * D + lse), "flops": n * flops}
    q_len, n = case["q_len"], case["layers"]
    rows = case["batch"] * q_len
    kv = 4 * D * hkv * sum(m + q_len for m in lengths) + 4 * sum(-(-(m + q_len) // BLOCK) for m in lengths)
    flops = sum(4 * hq * D * (m + j + 1) for m in lengths for j in range(q_len))
    if kind == "stack":
        h, i = case["hidden"], case["inter"]
        weights = (hq + 2 * hkv) * D * h + h * hq * D + 3 * h * i
        return {"bytes": n * (2 * weights + kv) + 4 * rows * h, "flops": n * (2 * rows * weights + flops)}
    io = 4 * rows * hq * D + (4 * rows * hq if case["lse"] else 0)
    if case["fused"]:
        io += 2 * rows * 2 * hkv * D  # the new tokens' k and v (their place in the cache is counted with it)
    return {"bytes": n * (kv + io), "flops": n * flops}


# About four times the largest error against 64 bits that the path showed over the listed cases and drawn
# ones (fp16 inputs and outputs, fp32 sums): 4.4e-4, 2.6e-4, 4.9e-4, 4.9e-4 and 2.2e-3.
TOLERANCE = {
    "attention": {"rel": 2e-3},
    "prefill": {"rel": 1e-3},
    "prefill_layer": {"rel": 2e-3},
    "ffn": {"rel": 2e-3},
    "stack": {"rel": 9e-3},
}


def tolerance(case):
    return TOLERANCE.get(case["kind"], "exact")


# ---------------------------------------------------------------- the same in 64 bits


def _norm(x, gamma, eps):
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)
    return x * gamma.double()


def _rotate(x, cos, sin):
    """[rows, heads, D] rotated by each row's angles."""
    lo, hi = x[..., :D // 2], x[..., D // 2:]
    c, n = cos.double()[:, None], sin.double()[:, None]
    return torch.cat((lo * c - hi * n, lo * n + hi * c), -1)


def _causal(q, k, v):
    """q [m, hq, D] over k, v [n, hkv, D]; the last query sees all n tokens.  Returns o and the LSE."""
    m, hq, _ = q.shape
    n, hkv, _ = k.shape
    g = hq // hkv
    hide = torch.arange(n, device=DEV)[None] > torch.arange(n - m, n, device=DEV)[:, None]
    o, lse = torch.empty_like(q), torch.empty((m, hq), dtype=torch.float64, device=DEV)
    for h in range(hkv):
        kt, vh = k[:, h].t().contiguous(), v[:, h].contiguous()
        for j in range(h * g, (h + 1) * g):
            p = (q[:, j].contiguous() @ kt).mul_(D ** -0.5).masked_fill_(hide, -math.inf)
            lse[:, j] = torch.logsumexp(p, 1)
            o[:, j] = p.sub_(lse[:, j:j + 1]).exp_() @ vh
    return o, lse


def _paged(s, li, q, k_cache, v_cache):
    """The decode/verify rows' attention at layer `li` over caches [blocks, layers, hkv, 16, D]."""
    case, q_len = s["case"], s["case"]["q_len"]
    hq, hkv = case["hq"], case["hkv"]
    g = hq // hkv
    o, lse = torch.empty_like(q), torch.empty(q.shape[:2], dtype=torch.float64, device=DEV)
    for r, n in enumerate(s["lengths"]):
        n += q_len
        at = s["table"][r, :-(-n // BLOCK)].long()
        k, v = (c[at, li].double().transpose(0, 1).reshape(hkv, -1, D)[:, :n].contiguous() for c in (k_cache, v_cache))
        rows = slice(r * q_len, (r + 1) * q_len)
        qr = q[rows].view(q_len, hkv, g, D).permute(1, 0, 2, 3).reshape(hkv, q_len * g, D).contiguous()
        p = torch.bmm(qr, k.transpose(1, 2).contiguous()).mul_(D ** -0.5).view(hkv, q_len, g, n)
        hide = torch.arange(n, device=DEV)[None] > torch.arange(n - q_len, n, device=DEV)[:, None]
        p.masked_fill_(hide[None, :, None], -math.inf)
        l = torch.logsumexp(p, -1)
        p = p.sub_(l[..., None]).exp_().view(hkv, q_len * g, n)
        o[rows] = torch.bmm(p, v).view(hkv, q_len, g, D).permute(1, 0, 2, 3).reshape(q_len, hq, D)
        lse[rows] = l.permute(1, 0, 2).reshape(q_len, hq)
    return o, lse


def _slots(s, seq_ids, positions):
    """Block and offset of each token."""
    pos = torch.tensor(positions, device=DEV)
    return s["table"][torch.tensor(seq_ids, device=DEV), pos // BLOCK].long(), pos % BLOCK


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind == "lm_head":
        x = s["x"].double()
        return torch.cat([x @ w.double().t().contiguous() for w in s["w"].split(16384)], 1).argmax(1)
    if kind == "ffn":
        out = []
        for x, wug, wd in s["layers"]:
            up, gate = (x.double() @ wug.double().t().contiguous()).chunk(2, 1)
            h = up * torch.nn.functional.silu(gate)
            out.append((h, h @ wd.double().t().contiguous()))
        return out
    if kind == "prefill":
        got = [_causal(*(s[n][a:b].double() for n in "qkv")) for a, b in itertools.pairwise(s["cu"].tolist())]
        o, lse = (torch.cat(t) for t in zip(*got))
        return (o, lse) if case["lse"] else o
    mc, hq, hkv = s["mc"], case["hq"], case["hkv"]
    eps = mc.rms_norm_eps
    if kind == "prefill_layer":
        kc, vc = s["k_cache"].double(), s["v_cache"].double()
        positions = [p for n in s["lengths"] for p in range(n)]
        blk, off = _slots(s, [r for r, n in enumerate(s["lengths"]) for _ in range(n)], positions)
        cos, sin = s["cos"][torch.tensor(positions)], s["sin"][torch.tensor(positions)]
        cu, out = [0] + list(itertools.accumulate(s["lengths"])), []
        for li, (qkv, q_norm, k_norm) in enumerate(s["layers"]):
            q, k, v = (t.double() for t in _heads(case, qkv))
            q, k = _rotate(_norm(q, q_norm, eps), cos, sin), _rotate(_norm(k, k_norm, eps), cos, sin)
            kc[blk, li, :, off], vc[blk, li, :, off] = k, v
            out.append(torch.cat([_causal(q[a:b], k[a:b], v[a:b])[0] for a, b in itertools.pairwise(cu)]))
        return out, kc, vc
    if kind == "attention" and not case["fused"]:
        out = [_paged(s, li, q.double(), s["k_cache"], s["v_cache"]) for li, q in enumerate(s["layers"])]
        return out if case["lse"] else [o for o, _ in out]
    kc, vc = s["k_cache"].double(), s["v_cache"].double()
    positions = [n - 1 for n in s["seq_lens"]]
    blk, off = _slots(s, s["seq_ids"], positions)
    cos, sin = s["cos"][torch.tensor(positions)], s["sin"][torch.tensor(positions)]

    def attend(li, qkv, q_norm, k_norm):
        q, k, v = _heads(case, qkv)
        q, k = _rotate(_norm(q, q_norm, eps), cos, sin), _rotate(_norm(k, k_norm, eps), cos, sin)
        kc[blk, li, :, off], vc[blk, li, :, off] = k, v
        return _paged(s, li, q, kc, vc)

    if kind == "attention":
        out = [attend(li, qkv.double(), a, b) for li, (qkv, a, b) in enumerate(s["layers"])]
        return (out if case["lse"] else [o for o, _ in out]), kc, vc
    x = s["embedded"].double()
    residual = torch.zeros_like(x)
    for li, w in enumerate(s["layers"]):
        residual = residual + x
        qkv = _norm(residual, w["n_in"], eps) @ w["wqkv"].double().t().contiguous()
        o = attend(li, qkv, w["q_norm"], w["k_norm"])[0].reshape(len(x), -1)
        residual = residual + o @ w["wo"].double().t().contiguous()
        up, gate = (_norm(residual, w["n_post"], eps) @ w["wug"].double().t().contiguous()).chunk(2, 1)
        x = (up * torch.nn.functional.silu(gate)) @ w["wd"].double().t().contiguous()
    return x + residual, kc, vc
