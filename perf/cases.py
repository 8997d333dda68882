"""Performance cases of the KVM framework on one MI355X.

Each case is a call that a user's program makes through the public entry
points, at sizes between the smallest prompt and a full 128K-context batch:

  prefill   ``SequenceMixer.prefill_raw``: one layer at the post-QKV boundary
            (memory updates, window + memory attention), as a prompt is read
  decode    ``SequenceMixer._decode_one_token`` on a ``KVMDecodeCache``: one
            token of every sequence, a state update every ``C`` tokens
  train     ``training.prefill_with_grad`` and its backward, as in a training
            step of one layer
  layer     ``SequenceMixer.forward_inference``: a decoder layer's whole mixer
            (projections, value residual, token shift, RoPE, prefill, output
            projection) on an empty cache
  model     ``DecodeGraph.step``: one token of a whole decoder, logits out

Inputs are synthetic and made from a seed on the GPU: queries and keys with
unit-variance features (what the mixer's ln_q / ln_k produce), a tenth of the
keys correlated with one of eight shared directions (topics), merge gates
1 + elu(N(0, 1)), all bfloat16.
"""

import math
import os
import sys
from types import SimpleNamespace

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "kvm-paper_amd"))

from kvm_amd import DecodeCacheSnapshot, SequenceMixer  # noqa: E402
from kvm_amd.backbone import (DecodeGraph, MixerConfig, RotaryEmbedding, RWKV7BackboneForCausalLM,  # noqa: E402
                              StatesDictCache, init_random_)
from kvm_amd.training import prefill_with_grad  # noqa: E402

DEV = "cuda"
N_CENTRES, CLUSTERED = 8, 0.1

# Memory budgets: (mode, growth factor, n_max_d_chunks * C as a slot cap).
#   fixed       the first chunk's slots, never more (the 120M paper runs)
#   sqrt        floor(16 sqrt(t)) slots (the 16-sqrt(T) runs)
#   saturation  1024 t / (1024 + t) slots (the saturating runs)


def _case(kind, B, Hq, Hkv, D, C, T, budget="fixed", **kw):
    return dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, D=D, C=C, T=T, budget=budget, **kw)


def listed():
    return [
        # A chat turn's prompt read by one GQA layer: a few chunks, launch latency counts.
        dict(name="prefill_chat", **_case("prefill", 1, 32, 8, 128, 256, 999)),
        # The batch-8, 32-head layer of the reference's own prefill benchmark, 8K tokens, fixed 256 slots.
        dict(name="prefill_b8_8k", **_case("prefill", 8, 32, 32, 128, 256, 8192)),
        # One long document: 32K tokens, 32 heads, 512-token chunks and slots (bench.py's headline workload).
        dict(name="prefill_32k", **_case("prefill", 1, 32, 32, 128, 512, 32768)),
        # A growing memory: 16 sqrt(t) slots, up to about 2000, ragged length.
        dict(name="prefill_sqrt", **_case("prefill", 2, 16, 16, 128, 256, 16001, "sqrt")),
        # 64-wide heads, four query heads per key head, short chunks, saturating memory, ragged length.
        dict(name="prefill_gqa_d64", **_case("prefill", 4, 16, 4, 64, 128, 5003, "saturation")),
        # Serving at 128K context: 64 sequences, 32 heads, 1024 slots and a 512-token window.
        dict(name="decode_128k", **_case("decode", 64, 32, 32, 128, 256, 131072, S=1024)),
        # One sequence decoding alone with grouped heads: a call of a few microseconds of GPU work.
        dict(name="decode_one", **_case("decode", 1, 32, 8, 128, 256, 4096, S=256)),
        # A training step of the 120M decoder's layer: 6 heads, 8192-token sequences, batch 8, 256-token chunks.
        dict(name="train_8k", **_case("train", 8, 6, 6, 128, 256, 8192)),
        # Training with grouped 64-wide heads and a growing memory, ragged length.
        dict(name="train_gqa_sqrt", **_case("train", 2, 16, 4, 64, 128, 4099, "sqrt")),
        # A long-document training step: 32K tokens, 32 heads, 512-token chunks.
        dict(name="train_32k", **_case("train", 1, 32, 32, 128, 512, 32768)),
        # The whole mixer of a d_model 2048 decoder layer (value residual, token shift) reading 2 x 4096 tokens.
        dict(name="layer_d2048", **_case("layer", 2, 16, 16, 128, 512, 4096)),
        # Token-by-token serving of a 12-layer, d_model 768 decoder (vocabulary 50304), 4 sequences.
        dict(name="model_decode", **_case("model", 4, 6, 6, 128, 256, 700, L=12, V=50304)),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(["prefill", "prefill", "prefill", "train", "train", "decode", "decode", "layer", "model"])
        if kind in ("prefill", "train"):
            D = rng.choice([64, 128, 128])
            Hkv = rng.choice([4, 6, 8, 16, 32])
            Hq = Hkv * rng.choice([1, 1, 2, 4])
            C = rng.choice([64, 128, 256, 256, 512])
            c = _case(kind, rng.choice([1, 1, 2, 3, 4, 8]), Hq, Hkv, D, C, _log_int(rng, 300, 32768),
                      rng.choice(["fixed", "fixed", "sqrt", "saturation"]))
            top = work(listed()[9])["flops"] if kind == "train" else work(listed()[2])["flops"]
            if Hq > 32 or c["T"] > 250 * C or work(c)["flops"] > top:
                continue
        elif kind == "decode":
            Hkv = rng.choice([4, 6, 8, 16, 32])
            C = rng.choice([128, 256, 512])
            c = _case(kind, _log_int(rng, 1, 64), Hkv * rng.choice([1, 1, 2, 4]), Hkv, rng.choice([64, 128, 128]), C,
                      C * rng.randint(3, 400), S=rng.choice([C, 2 * C, 1000, 1024]))
            if c["Hq"] > 32 or c["S"] < C or work(c)["bytes"] > work(listed()[5])["bytes"]:
                continue
        elif kind == "layer":
            H = rng.choice([6, 8, 16])
            c = _case(kind, rng.choice([1, 2, 3]), H, H, 128, rng.choice([256, 512]), _log_int(rng, 600, 8192))
        else:
            H = rng.choice([6, 8])
            c = _case(kind, rng.randint(1, 8), H, H, 128, 256, rng.randint(520, 760), L=rng.choice([6, 12]), V=50304)
        return c


# ---------------------------------------------------------------- inputs

def _config(c):
    mode = {"fixed": "fixed", "sqrt": "power_law", "saturation": "kvm_saturation"}[c["budget"]]
    cap = {"fixed": c["C"], "sqrt": 4096, "saturation": 1024}[c["budget"]]
    full = c["kind"] in ("layer", "model")
    S = c.get("S", c["C"])
    return MixerConfig(
        vocab_size=c.get("V", 1024), num_hidden_layers=c.get("L", 12), num_attention_heads=c["Hq"],
        num_key_value_heads=c["Hkv"], hidden_size=c["Hq"] * c["D"], mup_base_dim=c["Hq"] * c["D"],
        d_qk_head=c["D"], d_v_head=c["D"], use_tokenshift_att=int(full), use_tokenshift_ffn=int(full),
        use_value_residual=int(full), residual_scale=0.5, rope_partial_dim=64 if c["D"] == 128 else 32, sink_len=1,
        chunk_len=c["C"], n_bswa_chunks=2, n_max_d_chunks=-(-max(cap, S) // c["C"]), state_budget_mode=mode,
        state_growth_factor=16.0, state_growth_exponent=0.5, state_round_down=1, state_min_len=1,
        state_saturation_n=1024 if c["budget"] == "saturation" else None)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _mixer(c, g, layer_idx=0):
    with torch.device(DEV):
        mixer = SequenceMixer(_config(c), layer_idx).to(torch.bfloat16).eval()
    init_random_(mixer, int(torch.randint(0, 1 << 30, (1,), generator=g, device=DEV)))
    return mixer


def _qkvg(c, g, T):
    B, Hq, Hkv, D = c["B"], c["Hq"], c["Hkv"], c["D"]
    q = _randn(g, B, Hq, T, D).bfloat16()
    k = _randn(g, B, Hkv, T, D)
    centre = _randn(g, N_CENTRES, D)[torch.randint(0, N_CENTRES, (B, Hkv, T), generator=g, device=DEV)]
    near = torch.rand(B, Hkv, T, 1, generator=g, device=DEV) < CLUSTERED
    k = torch.where(near, 0.7 * centre + 0.7 * k, k).bfloat16()
    v = _randn(g, B, Hkv, T, D).bfloat16()
    gate = (1 + F.elu(_randn(g, B, Hkv, T, 1))).bfloat16()
    return q, k, v, gate


def prepare(case, seed):
    c = dict(case)
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    s = SimpleNamespace(case=c)
    if c["kind"] in ("prefill", "train"):
        s.mixer = _mixer(c, g)
        s.q, s.k, s.v, s.gate = _qkvg(c, g, c["T"])
        if c["kind"] == "prefill":
            s.plan = s.mixer.make_plan(c["T"])
        else:
            s.dout = (0.05 * _randn(g, c["B"], c["T"], c["Hq"], c["D"])).bfloat16()
            m = s.mixer
            s.leaves = [t.requires_grad_(True) for t in (s.q, s.k, s.v, s.gate)]
            s.leaves += [m.ln_s_k.weight, m.ln_s_k.bias, m.state_head_temp, m.front_head_temp]
    elif c["kind"] == "decode":
        s.mixer = _mixer(c, g)
        B, Hkv, D, S, W = c["B"], c["Hkv"], c["D"], c["S"], 2 * c["C"]
        n = torch.randint(1, 65, (B, Hkv, S, 1), generator=g, device=DEV).float()
        _, rk, rv, rg = _qkvg(c, g, W)
        mean_v = _randn(g, B, Hkv, S, D)
        s.snapshot = DecodeCacheSnapshot(
            state_k=(_randn(g, B, Hkv, S, D) * n).bfloat16(), state_v=(mean_v * n).bfloat16(),
            state_vlen=mean_v.norm(dim=-1, keepdim=True), recent_k=rk, recent_v=rv, recent_gate=rg,
            total_len=c["T"], state_coverage_len=c["T"] - W, recent_begin=c["T"] - W)
        s.cache = s.mixer.make_decode_cache(s.snapshot)
        s.tokens = [_qkvg(c, g, 1) for _ in range(8)]
        s.step = 0
    elif c["kind"] == "layer":
        s.mixer = _mixer(c, g, layer_idx=3)
        d = c["Hq"] * c["D"]
        s.x = _randn(g, c["B"], c["T"], d).bfloat16()
        s.v_first = _randn(g, c["B"], c["T"], d).bfloat16()
        s.rope = RotaryEmbedding(c["D"], 64)(torch.arange(c["T"], device=DEV).unsqueeze(0))
    else:
        with torch.device("meta"):
            model = RWKV7BackboneForCausalLM(_config(c))
        s.model = init_random_(model.to_empty(device=DEV).to(torch.bfloat16), int(seed)).eval()
        s.ids = torch.randint(0, c["V"], (c["B"], c["T"] + 64), generator=g, device=DEV)
        cache = StatesDictCache()
        with torch.no_grad():
            s.model(input_ids=s.ids[:, :c["T"]], past_key_values=cache, use_cache=True,
                    cache_position=torch.arange(c["T"], device=DEV), logits_to_keep=1)
        s.runner = DecodeGraph(s.model, cache)
        s.step = 0
        for _ in range(2):  # the first step packs the weights, the second captures the graph
            _model_step(s)
    return s


# ---------------------------------------------------------------- one pass

def _model_step(s):
    tok = s.ids[:, s.case["T"] + s.step % 64]
    s.step += 1
    return s.runner.step(tok)


def run(s):
    kind = s.case["kind"]
    if kind == "prefill":
        with torch.no_grad():
            r = s.mixer.prefill_raw(s.q, s.k, s.v, s.gate, plan=s.plan, check_status=False)
        return {key: r[key] for key in ("out", "state_k", "state_v", "state_vlen", "state_k_attn", "state_v_attn")}
    if kind == "train":
        for t in s.leaves:
            t.grad = None
        y = prefill_with_grad(s.mixer, s.q, s.k, s.v, s.gate)
        y.backward(s.dout)
        return [y.detach()] + [t.grad for t in s.leaves]
    if kind == "decode":
        q, k, v, gate = s.tokens[s.step % len(s.tokens)]
        s.step += 1
        with torch.no_grad():
            out = s.mixer._decode_one_token(q, k, v, gate, s.cache)
        c = s.cache
        return {"out": out, "state_k": c.state_k, "state_v": c.state_v, "state_k_attn": c.state_k_attn,
                "state_v_attn": c.state_v_attn, "state_vlen": c.state_vlen, "recent_k": c.recent_k,
                "recent_v": c.recent_v, "recent_gate": c.recent_gate}
    if kind == "layer":
        cache = StatesDictCache()
        with torch.no_grad():
            y = s.mixer.forward_inference(s.x, s.v_first, s.rope, None, cache)
        dc = cache.get_states(s.mixer.layer_idx)[s.mixer._CACHE_TRITON_DECODE]
        return {"y": y, "state_k": dc.state_k, "state_v": dc.state_v, "state_vlen": dc.state_vlen}
    logits = _model_step(s)
    carried = [s.runner.cache.get_states(i) for i in range(s.case["L"])]
    return {"logits": logits, "k": [st[SequenceMixer._CACHE_K_FINAL] for st in carried],
            "v": [st[SequenceMixer._CACHE_V_FINAL] for st in carried]}


# ---------------------------------------------------------------- what a pass cannot do without

def _schedule(c):
    """(chunks [(qb, qe, slots or 0)], updates [(token, slots before, appended)], final slots)."""
    T, C = c["T"], c["C"]

    def begin(t):
        return max(0, -(-t // C) * C - 2 * C)

    cap = -(-{"fixed": C, "sqrt": 4096, "saturation": 1024}[c["budget"]] // C) * C
    slots = min(T, C)
    chunks, updates = [], []
    for qb in range(0, T, C):
        qe = min(T, qb + C)
        if qb < 2 * C:
            chunks.append((qb, qe, 0))
            continue
        chunks.append((qb, qe, slots))
        now, nxt = begin(qe), begin(min(T, qe + C))
        if nxt > now:
            want = {"fixed": 1, "sqrt": math.floor(16.0 * qe ** 0.5),
                    "saturation": math.floor(1024.0 * qe / (1024.0 + qe))}[c["budget"]]
            grow = min(max(min(max(want, 1), nxt, cap) - slots, 0), C)
            updates.append((now, slots, grow))
            slots += grow
    return chunks, updates, slots


def _prefill_flops(c):
    """(attention pairs, routing flops): a query sees its snapshot's slots and the window up to itself."""
    chunks, updates, _ = _schedule(c)
    pairs = 0
    for qb, qe, slots in chunks:
        wb = max(0, qb - c["C"]) if qb >= 2 * c["C"] else 0
        n = qe - qb
        pairs += n * slots + n * (qb - wb) + n * (n + 1) // 2
    rows = c["B"] * c["Hkv"]
    route = sum(c["C"] * (before + grow) + (c["C"] * before if grow else 0) for _, before, grow in updates)
    return c["B"] * c["Hq"] * pairs, 2 * c["D"] * rows * route


def work(case):
    c = case
    B, Hq, Hkv, D, C, T = (c[k] for k in ("B", "Hq", "Hkv", "D", "C", "T"))
    d, rows = Hq * D, B * Hkv
    if c["kind"] == "decode":
        keys = c["S"] + 1.5 * C  # slots, and the window's rows averaged over a cycle
        return {"bytes": 2.0 * (rows * keys * 2 * D + 2 * B * d + 2 * rows * (2 * D + 1)),
                "flops": 4.0 * D * B * Hq * keys}
    if c["kind"] == "model":
        L, V = c["L"], c["V"]
        per_layer = d * d * 4 + 2 * 4 * d * d
        keys = C + 1.5 * C
        return {"bytes": 2.0 * (L * (per_layer + rows * keys * 2 * D) + V * d) + 4.0 * B * V,
                "flops": 2.0 * B * (L * per_layer + V * d) + 4.0 * D * B * Hq * keys * L}
    pairs, route = _prefill_flops(c)
    slots = _schedule(c)[2]
    io = 2.0 * (2 * B * T * d + rows * T * (2 * D + 1))
    state = rows * slots * (4.0 * 2 * D + 4)
    if c["kind"] == "prefill":
        return {"bytes": io + state, "flops": 4.0 * D * pairs + route}
    if c["kind"] == "train":  # forward, then scores again, dP, dV, dQ, dK
        return {"bytes": io + 2.0 * (2 * B * T * d + rows * T * (2 * D + 1)), "flops": 14.0 * D * pairs + route}
    weights = 4 * d * d + d * Hkv
    return {"bytes": 2.0 * (3 * B * T * d + weights) + state, "flops": 4.0 * D * pairs + route + 2.0 * B * T * weights}


def tolerance(case):
    # About four times the distance from ``exact`` that was measured where no
    # near tie of a routing score falls the other way: 2e-3 for bf16 outputs
    # of one attention, 3e-3 to 5e-3 for gradients (sums of bf16 products),
    # 3e-3 for a mixer with its projections, 9e-3 to 1.2e-2 for logits behind
    # 6 to 12 layers.
    rel = {"prefill": 0.01, "decode": 0.01, "train": 0.02, "layer": 0.015, "model": 0.03}[case["kind"]]
    return {"rel": rel, "max": 0.9}


# ---------------------------------------------------------------- 64 bits

class _Bf16(torch.autograd.Function):
    """bf16(x), the identity in the backward."""

    @staticmethod
    def forward(ctx, x):
        return x.bfloat16().double()

    @staticmethod
    def backward(ctx, g):
        return g


_bf16 = _Bf16.apply


def _ln(x, w, b):
    return F.layer_norm(x, (x.size(-1),), w, b, 1e-5)


def _take(x, idx):
    return x.gather(2, idx.unsqueeze(-1).expand(-1, -1, -1, x.size(-1)))


def _unit_rows(s_v, vlen):
    return _bf16(s_v / s_v.norm(dim=-1, keepdim=True).clamp_min(1e-12) * vlen)


def _exact_update(k, v, gate, s_k, s_v, vlen, grow, p, rope):
    """One memory update: the least similar ``grow`` tokens become slots, the
    others are added to their best non-sink slot.  State rows are bf16."""
    kp = torch.cat([torch.zeros_like(k[..., :rope]), k[..., rope:]], -1)
    kp = _bf16(_ln(kp, p.w, p.b))
    kg, vg = _bf16(kp * gate), _bf16(v * gate)
    B, H, n, D = k.shape
    merge = torch.arange(n, device=k.device).expand(B, H, n)
    if grow:
        with torch.no_grad():
            score = (kp @ _bf16(_ln(s_k, p.w, p.b)).mT).bfloat16().float().amax(-1)
            order = torch.argsort(score, dim=-1, stable=True)
        new, merge = order[..., :grow].sort(-1).values, order[..., grow:].sort(-1).values
        s_k, s_v = torch.cat([s_k, _take(kp, new)], 2), torch.cat([s_v, _take(v, new)], 2)
        vlen = torch.cat([vlen, _take(v, new).norm(dim=-1, keepdim=True)], 2)
        kg, vg = _take(kg, merge), _take(vg, merge)
    with torch.no_grad():
        score = kg @ _bf16(_ln(s_k, p.w, p.b)).mT
        score[..., :1] = -math.inf
        best = score.argmax(-1).unsqueeze(-1).expand(-1, -1, -1, D)
    s_k = _bf16(s_k + _bf16(torch.zeros_like(s_k).scatter_add(2, best, kg)))
    s_v = _bf16(s_v + _bf16(torch.zeros_like(s_v).scatter_add(2, best, vg)))
    return s_k, s_v, vlen


def _exact_attention(q, s_k, s_v, k, v, causal_from, p):
    """softmax over [slots ; window]; ``causal_from``: window keys before the first query."""
    B, Hq, n, D = q.shape
    g = Hq // k.size(1)

    def heads(x):
        return x.repeat_interleave(g, 1) if g > 1 else x

    score = (q @ heads(k).mT) * (p.tf.view(1, -1, 1, 1) / math.sqrt(D))
    hidden = torch.ones(n, k.size(2), dtype=torch.bool, device=q.device).triu(1 + causal_from)
    score = score.masked_fill(hidden, -math.inf)
    if s_k is None:
        return score.softmax(-1) @ heads(v)
    score = torch.cat([(q @ heads(s_k).mT) * (p.ts.view(1, -1, 1, 1) / math.sqrt(D)), score], -1).softmax(-1)
    return score[..., :s_k.size(2)] @ heads(s_v) + score[..., s_k.size(2):] @ heads(v)


def _exact_prefill(c, q, k, v, gate, p):
    chunks, updates, _ = _schedule(c)
    C, rope = c["C"], 64 if c["D"] == 128 else 32
    n0 = min(c["T"], C)
    s_k = _bf16(_ln(torch.cat([torch.zeros_like(k[:, :, :n0, :rope]), k[:, :, :n0, rope:]], -1), p.w, p.b))
    s_v, vlen = v[:, :, :n0], v[:, :, :n0].norm(dim=-1, keepdim=True)
    out, todo = [], list(updates)
    for qb, qe, slots in chunks:
        wb = max(0, qb - C) if slots else 0
        rows = (_bf16(_ln(s_k, p.w, p.b)), _unit_rows(s_v, vlen)) if slots else (None, None)
        out.append(_exact_attention(q[:, :, qb:qe], *rows, k[:, :, wb:qe], v[:, :, wb:qe], qb - wb, p))
        if slots and todo:
            t, _, grow = todo.pop(0)
            s_k, s_v, vlen = _exact_update(k[:, :, t:t + C], v[:, :, t:t + C], gate[:, :, t:t + C], s_k, s_v, vlen,
                                           grow, p, rope)
    rows = (_bf16(_ln(s_k, p.w, p.b)), _unit_rows(s_v, vlen))
    return torch.cat(out, 2).transpose(1, 2), s_k, s_v, vlen, *rows


def _params(mixer, grad=False):
    f = lambda t: t.detach().double().requires_grad_(grad)  # noqa: E731
    return SimpleNamespace(w=f(mixer.ln_s_k.weight), b=f(mixer.ln_s_k.bias), ts=f(mixer.state_head_temp),
                           tf=f(mixer.front_head_temp))


def _exact_mixer(m, c, x, v_first, rope):
    """The mixer on an empty cache: y, and the final state rows.  Every
    operation's result is bf16, as in the modules it restates: the routes of
    the memory are decided by those values."""
    R = _bf16
    P = lambda t: t.detach().double()  # noqa: E731
    W = lambda lin, t: R(t @ P(lin.weight).t())  # noqa: E731

    def shift(t, mix):
        return R(t + R(P(mix) * R(torch.cat([t[:, :1], t[:, :-1]], 1) - t)))

    B, T, _ = x.shape
    q, k, v = W(m.c_q, x), W(m.c_k, x), W(m.c_v, x)
    v = R(v + R(R(v_first - v) * R(torch.sigmoid(R(P(m.v_gate0) + W(m.v_gate2, W(m.v_gate1, x)))))))
    q, k, v = shift(q, m.x_q), shift(k, m.x_k), shift(v, m.x_v)
    cos, sin = (t.double() for t in rope)

    def rotate(t, ln):
        t = R(_ln(t.view(B, T, -1, c["D"]), P(ln.weight), P(ln.bias)))
        return R(R(cos * t) + R(sin * t.view(B, T, -1, c["D"] // 2, 2).flip(-1).view(t.shape))).transpose(1, 2)

    gate = R(1 + R(F.elu(W(m.key_weighting, x)))).transpose(1, 2).unsqueeze(-1)
    out, s_k, s_v, vlen, _, _ = _exact_prefill(c, rotate(q, m.ln_q), rotate(k, m.ln_k),
                                               v.view(B, T, -1, c["D"]).transpose(1, 2), gate, _params(m))
    return W(m.c_proj, R(out.reshape(B, T, -1))), s_k, s_v, vlen


def _rows(t):
    return t.reshape(-1, *t.shape[2:])


# Every update routes its tokens by an argmax over the slots that the updates
# before it made, so a near tie decided the other way changes all that follow.
# Up to this many updates the 64-bit result stays within a few percent of any
# correct one; past it there is no single value to compare with.
EXACT_UPDATES = 40


def exact(case, seed):
    c = dict(case)
    if c["kind"] != "decode" and len(_schedule(c)[1]) > EXACT_UPDATES:
        return None
    s = prepare(case, seed)
    with torch.enable_grad() if c["kind"] == "train" else torch.no_grad():
        if c["kind"] == "prefill":
            out, s_k, s_v, vlen, ka, va = _exact_prefill(c, *(t.double() for t in (s.q, s.k, s.v, s.gate)),
                                                         _params(s.mixer))
            return {"out": out, "state_k": _rows(s_k), "state_v": _rows(s_v), "state_vlen": _rows(vlen).squeeze(-1),
                    "state_k_attn": _rows(ka), "state_v_attn": _rows(va)}
        if c["kind"] == "train":
            x = [t.detach().double().requires_grad_(True) for t in (s.q, s.k, s.v, s.gate)]
            p = _params(s.mixer, grad=True)
            y = _exact_prefill(c, *x, p)[0]
            grads = torch.autograd.grad(y, x + [p.w, p.b, p.ts, p.tf], s.dout.double(), allow_unused=True)
            return [y.detach()] + list(grads)
        if c["kind"] == "decode":
            q, k, v, gate = (t.double() for t in s.tokens[0])
            sn, C, p = s.snapshot, c["C"], _params(s.mixer)
            rk, rv, rg = (t.double() for t in (sn.recent_k, sn.recent_v, sn.recent_gate))
            s_k, s_v, vlen = _exact_update(rk[:, :, :C], rv[:, :, :C], rg[:, :, :C], sn.state_k.double(),
                                           sn.state_v.double(), sn.state_vlen.double(), 0, p,
                                           64 if c["D"] == 128 else 32)
            ka, va = _bf16(_ln(s_k, p.w, p.b)), _unit_rows(s_v, vlen)
            out = _exact_attention(q, ka, va, torch.cat([rk[:, :, C:], k], 2), torch.cat([rv[:, :, C:], v], 2), C, p)
            for ring, new in ((rk, k), (rv, v), (rg, gate)):  # the token takes the oldest row's place
                ring[:, :, :1] = new
            return {"out": out, "state_k": _rows(s_k), "state_v": _rows(s_v), "state_k_attn": _rows(ka),
                    "state_v_attn": _rows(va), "state_vlen": _rows(vlen).squeeze(-1), "recent_k": _rows(rk),
                    "recent_v": _rows(rv), "recent_gate": _rows(rg).squeeze(-1)}
        if c["kind"] == "layer":
            y, s_k, s_v, vlen = _exact_mixer(s.mixer, c, s.x.double(), s.v_first.double(), s.rope)
            return {"y": y, "state_k": _rows(s_k), "state_v": _rows(s_v), "state_vlen": _rows(vlen).squeeze(-1)}
        # The token after the prompt and prepare's two steps, as the last position of one long prompt.
        tr, T, R = s.model.transformer, c["T"] + 3, _bf16
        norm = lambda ln, t: R(_ln(t, ln.weight.double(), ln.bias.double()))  # noqa: E731
        W = lambda lin, t: R(t @ lin.weight.double().t())  # noqa: E731
        rope = tr.rotary(torch.arange(T, device=DEV).unsqueeze(0))
        x = norm(tr.ln_emb, tr.wte.weight.double()[s.ids[:, :T]])
        v_first = W(tr.h[0].attn.c_v, norm(tr.h[0].ln_attn, x))
        for blk in tr.h:
            x = R(x + 0.5 * _exact_mixer(blk.attn, dict(c, T=T), norm(blk.ln_attn, x), v_first, rope)[0])
            h = norm(blk.ln_mlp, x)
            h = R(h + R(blk.mlp.x_k.double() * R(F.pad(h, (0, 0, 1, 0))[:, :-1] - h)))
            x = R(x + 0.5 * W(blk.mlp.c_proj, R(R(F.relu(W(blk.mlp.c_fc, h))).square())))
        return {"logits": W(s.model.lm_head, norm(tr.ln_head, x[:, -1])), "k": None, "v": None}
