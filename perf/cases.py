"""The work this library is measured on: decode steps as a serving program issues them.

A decode step calls each operator once per decoder layer, on that layer's own weights and KV cache. A program allocates
its buffers once, runs the step once eagerly and captures it into a HIP graph, then replays it for every token, so most
cases here are one replay of such a graph ("layers" calls, each on its own tensors); the transformers attention function
is called eagerly, as generate() calls it. Kinds:

  attn    one attention call per layer: form "plain" (gqa_decode, ranges from seq_lens), "fused" (gqa_decode_fused: q/k
          norm, RoPE, cache write, attention) or "masked" (attn_decode_fused: the same, ranges from the additive mask)
  depth   a depth-transformer frame: 16 steps over a 17-slot cache, the first with two query tokens, 12 layers each
  eager   mi355_decode_attention called eagerly once per layer with the additive mask (transformers' attention hook)
  proj    the projections around the attention of one layer: RMSNorm + q | k | v, and the output projection + residual
  mlp     the MLP of one layer: RMSNorm + gate / up + SiLU * up, and down + residual
  step    the whole backbone decode step: embedding, layers, final norm, logits, classifier-free guidance

Values are N(0, 1) activations and caches, weights N(0, 1 / k), norm weights around 1, as after a norm in a trained model.
"""
import math
import random
import types

import torch

import __graft_entry__

pkg = __graft_entry__.package()

DEV = "cuda:0"
BF16 = torch.bfloat16
EPS = 1e-6
DEPTH_STEPS = 16
VOCAB = 2048


def listed():
    return [
        # one depth-transformer frame of a CFG pair: 192 launches over at most 17 positions, latency only
        dict(name="depth_frame", kind="depth", batch=2, kv_heads=2, group=4, head_dim=128, layers=12),
        # the smallest call: one eager attention of a CFG pair early in an utterance, one row left-padded
        dict(name="eager_call", kind="eager", batch=2, kv_heads=8, group=2, head_dim=128, capacity=2048, lo=301, hi=301,
             layers=1),
        # the backbone's attention at serving shape: a CFG pair, 1024 positions of a 2048-slot cache
        dict(name="pair_1k_fused", kind="attn", form="fused", batch=2, kv_heads=8, group=2, head_dim=128, capacity=2048,
             lo=1024, hi=1024, layers=28),
        # the same through the reference's argument order: the range of each row comes from the interval mask
        dict(name="pair_masked", kind="attn", form="masked", batch=2, kv_heads=8, group=2, head_dim=128, capacity=2048,
             lo=1377, hi=1377, layers=28),
        # a CFG pair late in a long utterance
        dict(name="pair_4k", kind="attn", form="plain", batch=2, kv_heads=8, group=2, head_dim=128, capacity=4096,
             lo=4096, hi=4096, layers=28),
        # a server's ragged batch: eight CFG pairs, each pair at its own length
        dict(name="ragged_b16", kind="attn", form="plain", batch=16, kv_heads=8, group=2, head_dim=128, capacity=2048,
             lo=128, hi=2048, layers=28),
        # a larger group over a long context (32 q / 4 KV heads)
        dict(name="long_32k_g8", kind="attn", form="plain", batch=2, kv_heads=4, group=8, head_dim=128, capacity=32768,
             lo=20001, hi=32768, layers=8),
        # a wide ragged batch with head_dim 64 (32 q / 8 KV heads)
        dict(name="batch32_d64_g4", kind="attn", form="plain", batch=32, kv_heads=8, group=4, head_dim=64, capacity=4096,
             lo=64, hi=4096, layers=8),
        # a single stream's attention projections (no guidance: one row)
        dict(name="proj_m1", kind="proj", batch=1, hidden=2048, kv_heads=8, group=2, layers=28),
        # the MLP of two CFG pairs
        dict(name="mlp_m4", kind="mlp", batch=4, hidden=2048, inter=6144, layers=28),
        # the MLP of a CFG pair in a backbone of twice the width
        dict(name="mlp_m2_wide", kind="mlp", batch=2, hidden=4096, inter=12288, layers=8),
        # the whole backbone decode step of a CFG pair at serving shape
        dict(name="step_pair", kind="step", batch=2, hidden=2048, inter=6144, kv_heads=8, group=2, capacity=2048,
             position=1023, layers=28),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["attn", "mlp", "proj", "eager", "depth", "step"], [9, 4, 2, 2, 1, 1])[0]
    kv_heads, group = rng.choice([(8, 2), (8, 2), (8, 1), (4, 2), (2, 4), (8, 4), (4, 8), (2, 8), (1, 8)])
    head_dim = rng.choice([64, 128, 128])
    if kind == "depth":
        return dict(kind=kind, batch=rng.randint(1, 8), kv_heads=rng.choice([2, 4, 8]), group=rng.choice([1, 2, 4]),
                    head_dim=head_dim, layers=rng.randint(3, 12))
    if kind in ("attn", "eager"):
        form = rng.choice(["plain", "plain", "fused", "masked"])
        case = dict(kind=kind, batch=_log_int(rng, 1, 32), kv_heads=kv_heads, group=group)
        if kind == "attn":
            case["form"] = form
        case["head_dim"] = 128 if kind == "attn" and form != "plain" else head_dim
        case["capacity"] = _log_int(rng, 64, 32768)
        case["hi"] = rng.randint(max(1, case["capacity"] // 2), case["capacity"])
        case["lo"] = case["hi"] if rng.random() < 0.5 else rng.randint(1, case["hi"])
        case["layers"] = rng.randint(4, 28)
        slot = case["batch"] * case["capacity"] * case["kv_heads"] * case["head_dim"] * 4
        while case["batch"] > 1 and slot > 600_000_000:  # a call reads no more than the largest listed one's
            case["batch"] //= 2
            slot = case["batch"] * case["capacity"] * case["kv_heads"] * case["head_dim"] * 4
        case["layers"] = max(1, min(case["layers"], 1_000_000_000 // slot))
        return case
    batch = rng.randint(1, 4)
    widest = 32768 // batch // 1024 * 1024  # the GEMVs take rows of at most 64 KiB of x
    hidden = 8 * _log_int(rng, 64, 512)
    layers = rng.randint(4, 28)
    if kind == "proj":
        heads = group * kv_heads if group * kv_heads <= 32 else 32
        return dict(kind=kind, batch=batch, hidden=hidden, kv_heads=heads // group, group=group, layers=layers)
    inter = min(widest, 8 * int(hidden * rng.uniform(1.5, 4.0) / 8))
    if kind == "mlp":
        return dict(kind=kind, batch=batch, hidden=hidden, inter=inter, layers=max(1, min(layers, 1_200_000_000 // (6 * hidden * inter))))
    hidden, inter = min(hidden, 2048), min(inter, 6144)  # a step stays within the listed one
    capacity = _log_int(rng, 256, 4096)
    return dict(kind="step", batch=rng.choice([1, 2, 4]), hidden=hidden, inter=inter, kv_heads=rng.choice([2, 4, 8]), group=rng.choice([1, 2, 4]),
                capacity=capacity, position=rng.randint(capacity // 4, capacity - 1), layers=rng.randint(2, 12))


# ---------------------------------------------------------------------------------------------- what a case implies


def _lengths(case):
    """Length of each row, shared by each CFG pair: the case's hi, or spread over [lo, hi] by its own sizes."""
    B, lo, hi = case["batch"], case["lo"], case["hi"]
    r = random.Random("%d %d %d" % (B, lo, hi))
    pair = [r.randint(lo, hi) for _ in range((B + 1) // 2)]
    return [hi if b < 2 else pair[b // 2] for b in range(B)]


def _starts(case):
    """Left padding of each row, where the form carries one: the second row of a pair starts a few positions in."""
    if case.get("form") == "plain":
        return [0] * case["batch"]
    return [min(7, n - 1) if b % 2 else 0 for b, n in enumerate(_lengths(case))]


def _cache_pos(case):
    """The slot a fused step writes: the last position of the longest row."""
    return max(_lengths(case)) - 1


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, scale=1.0):
    return torch.empty(shape, dtype=BF16, device=DEV).normal_(0.0, scale, generator=g)


def _norm_weight(g, *shape):
    return torch.empty(shape, dtype=BF16, device=DEV).normal_(1.0, 0.1, generator=g)


def _rope(g, batch, dim, longest):
    """cos / sin rows of one position per row, [B, 1, dim]."""
    pos = torch.randint(0, max(1, longest), (batch, 1), generator=g, device=DEV)
    freq = 10000.0 ** (-torch.arange(0, dim, 2, device=DEV, dtype=torch.float64) / dim)
    a = (pos.double() * freq).repeat(1, 2)[:, None, :]
    return a.cos().to(BF16), a.sin().to(BF16)


def _mask(case):
    """The additive interval mask [B, 1, 1, capacity]: 0 on a row's positions, the lowest bf16 elsewhere."""
    lens = torch.tensor(_lengths(case), device=DEV)[:, None]
    starts = torch.tensor(_starts(case), device=DEV)[:, None]
    pos = torch.arange(case["capacity"], device=DEV)[None]
    m = torch.full((case["batch"], case["capacity"]), torch.finfo(BF16).min, dtype=BF16, device=DEV)
    return m.masked_fill_((pos >= starts) & (pos < lens), 0.0)[:, None, None, :]


def _inputs(case, seed):
    """The tensors of a case, a pure function of the seed (prepare and exact share them)."""
    g, kind, B, L = _gen(seed), case["kind"], case["batch"], case["layers"]
    s = types.SimpleNamespace()
    if kind in ("attn", "eager", "depth"):
        NKV, D = case["kv_heads"], case["head_dim"]
        NH = NKV * case["group"]
        s.scale = D ** -0.5
        cap = DEPTH_STEPS + 1 if kind == "depth" else case["capacity"]
        s.k, s.v = _randn(g, L, B, NKV, cap, D), _randn(g, L, B, NKV, cap, D)
        if kind == "depth":
            s.q0 = _randn(g, L, B, NH, 2, D)
            s.q = _randn(g, DEPTH_STEPS - 1, L, B, NH, D)
        elif kind == "eager":
            s.q = _randn(g, L, B, NH, 1, D)
        elif case["form"] == "plain":
            s.q = _randn(g, L, B, NH, D)
        else:
            s.qkv = _randn(g, L, B, (NH + 2 * NKV) * D)
            s.qn, s.kn = _norm_weight(g, L, D), _norm_weight(g, L, D)
            s.cos, s.sin = _rope(g, B, D, case["capacity"])
        return s
    H = case["hidden"]
    if kind == "proj":
        nk = case["kv_heads"] * 128
        nq = nk * case["group"]
        s.x, s.res = _randn(g, L, B, H), _randn(g, L, B, H)
        s.ln = _norm_weight(g, L, H)
        s.wq, s.wk, s.wv = (_randn(g, L, n, H, scale=H ** -0.5) for n in (nq, nk, nk))
        s.ao = _randn(g, L, B, nq)
        s.wo = _randn(g, L, H, nq, scale=nq ** -0.5)
        return s
    I = case["inter"]
    if kind == "mlp":
        s.x = _randn(g, L, B, H)
        s.ln = _norm_weight(g, L, H)
        s.wg, s.wu = _randn(g, L, I, H, scale=H ** -0.5), _randn(g, L, I, H, scale=H ** -0.5)
        s.wd = _randn(g, L, H, I, scale=I ** -0.5)
        return s
    NKV, D = case["kv_heads"], 128
    nk = NKV * D
    nq = nk * case["group"]
    s.ids = torch.randint(0, VOCAB, (B, 1), generator=g, device=DEV)
    s.emb = _randn(g, VOCAB, H)
    s.ln1, s.ln2 = _norm_weight(g, L, H), _norm_weight(g, L, H)
    s.qn, s.kn = _norm_weight(g, L, D), _norm_weight(g, L, D)
    s.wq, s.wk, s.wv = (_randn(g, L, n, H, scale=H ** -0.5) for n in (nq, nk, nk))
    s.wo = _randn(g, L, H, nq, scale=nq ** -0.5)
    s.wg, s.wu = _randn(g, L, I, H, scale=H ** -0.5), _randn(g, L, I, H, scale=H ** -0.5)
    s.wd = _randn(g, L, H, I, scale=I ** -0.5)
    s.norm = _norm_weight(g, H)
    s.head = torch.empty(VOCAB, H, device=DEV).normal_(0.0, H ** -0.5, generator=g)
    s.k, s.v = _randn(g, L, B, NKV, case["capacity"], D), _randn(g, L, B, NKV, case["capacity"], D)
    s.pads = [min(7, case["position"]) if b % 2 else 0 for b in range(B)]
    return s


# ---------------------------------------------------------------------------------------------- prepare and run


def _capture(step):
    """The step, run once eagerly and then captured into a HIP graph."""
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    torch.cuda.synchronize()
    return graph


def _workspace(batch, heads, kv_heads, head_dim, capacity):
    n = pkg.workspace_bytes(batch, heads, kv_heads, head_dim, capacity)
    return torch.zeros((n + 255) // 256 * 256, dtype=torch.uint8, device=DEV)


def _prepare_attn(case, s):
    B, L, NKV, D, cap = case["batch"], case["layers"], case["kv_heads"], case["head_dim"], case["capacity"]
    NH = NKV * case["group"]
    s.out = torch.zeros(L, B, 1, NH, D, dtype=BF16, device=DEV)
    s.lens = torch.tensor(_lengths(case), dtype=torch.int32, device=DEV)
    s.starts = torch.tensor(_starts(case), dtype=torch.int32, device=DEV)
    if case["form"] == "plain":
        s.ws = _workspace(B, NH, NKV, D, cap)
        s.outputs = {"out": s.out}

        def step():
            for i in range(L):
                pkg.gqa_decode(s.q[i], s.k[i], s.v[i], s.lens, s.scale, s.out[i], workspace=s.ws)
    else:
        s.pos = torch.tensor([_cache_pos(case)], dtype=torch.int64, device=DEV)
        s.outputs = {"out": s.out, "k": s.k, "v": s.v}
        if case["form"] == "fused":
            s.ws = _workspace(B, NH, NKV, D, cap)

            def step():
                for i in range(L):
                    pkg.gqa_decode_fused(s.qkv[i], s.qn[i], s.kn[i], EPS, s.cos, s.sin, s.k[i], s.v[i], s.pos, s.scale,
                                         s.out[i], seq_lens=s.lens, kv_start=s.starts, workspace=s.ws)
        else:
            s.mask = _mask(case)
            s.counters = torch.zeros(B * NKV, dtype=torch.int32, device=DEV)

            def step():
                for i in range(L):
                    pkg.attn_decode_fused(s.qkv[i], s.qn[i], s.kn[i], EPS, s.cos, s.sin, s.k[i], s.v[i], s.mask, s.pos,
                                          s.scale, None, None, None, s.counters, s.out[i])
    s.graph = _capture(step)


def _prepare_depth(case, s):
    B, L, NKV, D = case["batch"], case["layers"], case["kv_heads"], case["head_dim"]
    NH = NKV * case["group"]
    cap = DEPTH_STEPS + 1
    s.lens = torch.arange(2, cap + 1, dtype=torch.int32, device=DEV)[:, None].expand(DEPTH_STEPS, B).contiguous()
    s.out0 = torch.zeros(L, B, 2, NH, D, dtype=BF16, device=DEV)
    s.out = torch.zeros(DEPTH_STEPS - 1, L, B, NH, D, dtype=BF16, device=DEV)
    s.ws0, s.ws = _workspace(2 * B, NH, NKV, D, cap), _workspace(B, NH, NKV, D, cap)
    s.outputs = {"out0": s.out0, "out": s.out}

    def step():
        for i in range(L):
            pkg.gqa_decode(s.q0[i], s.k[i], s.v[i], s.lens[0], s.scale, s.out0[i], workspace=s.ws0)
        for t in range(1, DEPTH_STEPS):
            for i in range(L):
                pkg.gqa_decode(s.q[t - 1, i], s.k[i], s.v[i], s.lens[t], s.scale, s.out[t - 1, i], workspace=s.ws)
    s.graph = _capture(step)


def _prepare_proj(case, s):
    L, B = case["layers"], case["batch"]
    s.qkv = torch.zeros(L, B, s.wq.size(1) + 2 * s.wk.size(1), dtype=BF16, device=DEV)
    s.y = torch.zeros_like(s.res)
    s.outputs = {"qkv": s.qkv, "y": s.y}

    def step():
        for i in range(L):
            pkg.gemv_seg(s.x[i], s.ln[i], EPS, s.wq[i], s.wk[i], s.wv[i], s.qkv[i])
            pkg.gemv_resid(s.ao[i], s.wo[i], s.res[i], s.y[i])
    s.graph = _capture(step)


def _prepare_mlp(case, s):
    L, B = case["layers"], case["batch"]
    s.act = torch.zeros(L, B, case["inter"], dtype=BF16, device=DEV)
    s.y = torch.zeros_like(s.x)
    s.outputs = {"act": s.act, "y": s.y}

    def step():
        for i in range(L):
            pkg.gemv_gateup(s.x[i], s.ln[i], EPS, s.wg[i], s.wu[i], s.act[i])
            pkg.gemv_resid(s.act[i], s.wd[i], s.x[i], s.y[i])
    s.graph = _capture(step)


def _rope_tables(position_ids, dim):
    freq = 10000.0 ** (-torch.arange(0, dim, 2, device=position_ids.device, dtype=torch.float32) / dim)
    a = (position_ids.float()[:, :, None] * freq).repeat(1, 1, 2)
    return a.cos().to(BF16), a.sin().to(BF16)


def _prepare_step(case, s):
    """A graph object with the attributes that backbone.fused_decode_step reads."""
    N = types.SimpleNamespace
    B, L, cap, pos = case["batch"], case["layers"], case["capacity"], case["position"]

    def norm(w):
        return N(weight=w, variance_epsilon=EPS)

    def linear(w):
        return N(weight=w, bias=None)

    layers = []
    for i in range(L):
        attn = N(q_proj=linear(s.wq[i]), k_proj=linear(s.wk[i]), v_proj=linear(s.wv[i]), o_proj=linear(s.wo[i]),
                 q_norm=norm(s.qn[i]), k_norm=norm(s.kn[i]), scaling=128 ** -0.5, head_dim=128,
                 num_key_value_groups=case["group"], sliding_window=None)
        mlp = N(gate_proj=linear(s.wg[i]), up_proj=linear(s.wu[i]), down_proj=linear(s.wd[i]), act_fn=torch.nn.SiLU())
        layers.append(N(self_attn=attn, mlp=mlp, input_layernorm=norm(s.ln1[i]), post_attention_layernorm=norm(s.ln2[i])))
    pads = torch.tensor(s.pads, device=DEV)
    valid = torch.arange(cap, device=DEV)[None]
    valid = (valid >= pads[:, None]) & (valid <= pos)
    mask = torch.full((B, cap), torch.finfo(BF16).min, dtype=BF16, device=DEV).masked_fill_(valid, 0.0)
    half = max(1, B // 2)
    g = N(model=N(layers=layers, norm=norm(s.norm), rotary_emb=lambda x, p: _rope_tables(p, 128)),
          embed_tokens=lambda ids: torch.nn.functional.embedding(ids, s.emb),
          lm_head=lambda x: torch.nn.functional.linear(x, s.head), batch_size=B, half=half, hidden_size=case["hidden"],
          max_seq_len=cap, static_cache=N(layers=[N(keys=s.k[i], values=s.v[i]) for i in range(L)]),
          cache_position=torch.tensor([pos], dtype=torch.int64, device=DEV), position_ids=(pos - pads)[:, None],
          guidance_scale=torch.tensor(3.0, device=DEV), input_ids_buf=s.ids, attn_mask=mask[:, None, None, :],
          hidden_buf=torch.zeros(B, 1, case["hidden"], dtype=BF16, device=DEV),
          logits_buf=torch.zeros(B, VOCAB, device=DEV), cfg_logits_buf=torch.zeros(half, VOCAB, device=DEV))
    s.decode = g
    s.outputs = {"hidden": g.hidden_buf, "logits": g.logits_buf, "cfg": g.cfg_logits_buf, "k": s.k, "v": s.v}
    s.graph = _capture(lambda: pkg.backbone.fused_decode_step(g))


def prepare(case, seed):
    s = _inputs(case, seed)
    if case["kind"] == "eager":
        s.module = types.SimpleNamespace(training=False)
        s.mask = _mask(case)
        return s
    {"attn": _prepare_attn, "depth": _prepare_depth, "proj": _prepare_proj, "mlp": _prepare_mlp,
     "step": _prepare_step}[case["kind"]](case, s)
    return s


def run(state):
    if hasattr(state, "graph"):
        state.graph.replay()
        return state.outputs
    return [pkg.hf_attention.mi355_decode_attention(state.module, state.q[i], state.k[i], state.v[i], state.mask,
                                                    scaling=state.scale)[0] for i in range(state.q.size(0))]


# ---------------------------------------------------------------------------------------------- work and tolerance


def work(case):
    kind, B, L = case["kind"], case["batch"], case["layers"]
    if kind in ("attn", "eager", "depth"):
        NKV, D, G = case["kv_heads"], case["head_dim"], case["group"]
        if kind == "depth":  # the cache positions of a frame stay on the chip: each is read once
            lens, calls = [DEPTH_STEPS + 1] * B, DEPTH_STEPS
            pairs = B * (2 + sum(range(2, DEPTH_STEPS + 2)))
        else:
            lens, calls = [n - a for n, a in zip(_lengths(case), _starts(case))], 1
            pairs = sum(lens)
        kv = sum(lens) * NKV * D * 2 * 2
        qo = 2 * B * NKV * G * D * 2 * calls
        new = 4 * B * NKV * D * 2 if case.get("form", "plain") != "plain" else 0
        mask = B * case["capacity"] * 2 if kind == "eager" or case.get("form") == "masked" else 0
        return {"bytes": L * (kv + qo + new) + mask, "flops": L * 4 * pairs * NKV * G * D}
    if kind == "proj":
        nk = case["kv_heads"] * 128
        weights = case["hidden"] * (2 * nk * case["group"] + 2 * nk)
    else:
        weights = 3 * case["hidden"] * case["inter"]
    bytes_, flops = 2 * L * weights, 2 * L * B * weights
    if kind == "step":
        nk = case["kv_heads"] * 128
        proj = case["hidden"] * (2 * nk * case["group"] + 2 * nk)
        kv = B * (case["position"] + 1) * nk * 2 * 2
        bytes_ += L * (2 * proj + kv) + VOCAB * case["hidden"] * 4
        flops += L * (2 * B * proj + 4 * B * (case["position"] + 1) * nk * case["group"]) + 2 * B * VOCAB * case["hidden"]
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    # fp32 sums rounded to bf16 at the end: another order of the sums moves a few results to the neighbouring bf16 value
    # (other split counts: rel up to 7e-6, one value in a thousand by 2^-8 at most)
    if case["kind"] == "step":  # a change of rounding in one layer travels through all that follow
        return {"rel": 0.01, "max": 0.25}
    return {"rel": 1e-3, "max": 0.03}


# ---------------------------------------------------------------------------------------------- the same in 64 bits


def _attend(q, k, v, start, end, scale):
    """q [NH, D] of one row over positions [start, end) of k, v [NKV, cap, D], in float64: [NH, D]."""
    NKV, D = k.size(0), k.size(2)
    kk, vv = k[:, start:end].double(), v[:, start:end].double()
    qq = q.double().reshape(NKV, -1, D)
    p = torch.softmax(torch.matmul(kk, qq.transpose(1, 2).contiguous()) * scale, dim=1)  # [NKV, len, G]
    return torch.matmul(p.transpose(1, 2).contiguous(), vv).reshape(-1, D)


def _rms(x, w):
    x = x.double()
    return w.double() * x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)


def _rotate(x, cos, sin):
    d = x.size(-1) // 2
    return x * cos + torch.cat([-x[..., d:], x[..., :d]], -1) * sin


def _exact_fused(qkv, qn, kn, cos, sin, k, v, pos, starts, lens, scale):
    """One fused attention layer in float64: (out [B, 1, NH, D], k, v with the new position written)."""
    B, NKV, _, D = k.shape
    rows = qkv.double().reshape(B, -1, D)
    NH = rows.size(1) - 2 * NKV
    c, s = cos.double().reshape(B, 1, D), sin.double().reshape(B, 1, D)
    q = _rotate(_rms(rows[:, :NH], qn), c, s)
    k, v = k.double(), v.double()
    k[:, :, pos] = _rotate(_rms(rows[:, NH:NH + NKV], kn), c, s)
    v[:, :, pos] = rows[:, NH + NKV:]
    out = torch.stack([_attend(q[b], k[b], v[b], starts[b], lens[b], scale) for b in range(B)])
    return out[:, None], k, v


def exact(case, seed):
    s = _inputs(case, seed)
    kind, B, L = case["kind"], case["batch"], case["layers"]
    if kind == "depth":
        out0, out = [], [[] for _ in range(DEPTH_STEPS - 1)]
        for i in range(L):
            out0.append(torch.stack([torch.stack([_attend(s.q0[i, b, :, t], s.k[i, b], s.v[i, b], 0, t + 1, s.scale)
                                                  for t in range(2)]) for b in range(B)]))
            for t in range(1, DEPTH_STEPS):
                out[t - 1].append(torch.stack([_attend(s.q[t - 1, i, b], s.k[i, b], s.v[i, b], 0, t + 2, s.scale)
                                               for b in range(B)]))
        return {"out0": torch.stack(out0), "out": torch.stack([torch.stack(o) for o in out])}
    if kind in ("attn", "eager"):
        lens, starts = _lengths(case), _starts(case)
        if kind == "eager" or case["form"] == "plain":
            q = s.q.reshape(L, B, -1, case["head_dim"])
            out = [torch.stack([_attend(q[i, b], s.k[i, b], s.v[i, b], starts[b], lens[b], s.scale) for b in range(B)])[:, None]
                   for i in range(L)]
            return out if kind == "eager" else {"out": torch.stack(out)}
        pos = _cache_pos(case)
        out, slots = [], []
        for i in range(L):
            o, k, v = _exact_fused(s.qkv[i], s.qn[i], s.kn[i], s.cos, s.sin, s.k[i], s.v[i], pos, starts, lens, s.scale)
            out.append(o)
            slots.append((k[:, :, pos].clone(), v[:, :, pos].clone()))
        k, v = s.k.double(), s.v.double()
        for i, (a, b) in enumerate(slots):
            k[i, :, :, pos], v[i, :, :, pos] = a, b
        return {"out": torch.stack(out), "k": k, "v": v}
    if kind == "proj":
        qkv, y = [], []
        for i in range(L):
            n = _rms(s.x[i], s.ln[i])
            qkv.append(torch.cat([n @ w.double().t() for w in (s.wq[i], s.wk[i], s.wv[i])], -1))
            y.append(s.res[i].double() + s.ao[i].double() @ s.wo[i].double().t())
        return {"qkv": torch.stack(qkv), "y": torch.stack(y)}
    if kind == "mlp":
        act, y = [], []
        for i in range(L):
            n = _rms(s.x[i], s.ln[i])
            a = torch.nn.functional.silu(n @ s.wg[i].double().t()) * (n @ s.wu[i].double().t())
            act.append(a)
            y.append(s.x[i].double() + a @ s.wd[i].double().t())
        return {"act": torch.stack(act), "y": torch.stack(y)}
    pos = case["position"]
    ids = torch.tensor([[pos - p] for p in s.pads], device=DEV)
    cos, sin = _rope_tables(ids, 128)
    x = s.emb[s.ids[:, 0]].double()
    k, v = s.k.double(), s.v.double()
    for i in range(L):
        n = _rms(x, s.ln1[i])
        qkv = torch.cat([n @ w.double().t() for w in (s.wq[i], s.wk[i], s.wv[i])], -1)
        o, ki, vi = _exact_fused(qkv, s.qn[i], s.kn[i], cos, sin, s.k[i], s.v[i], pos, s.pads, [pos + 1] * B, 128 ** -0.5)
        k[i, :, :, pos], v[i, :, :, pos] = ki[:, :, pos], vi[:, :, pos]
        h = x + o.reshape(B, -1) @ s.wo[i].double().t()
        n = _rms(h, s.ln2[i])
        x = h + (torch.nn.functional.silu(n @ s.wg[i].double().t()) * (n @ s.wu[i].double().t())) @ s.wd[i].double().t()
    hidden = _rms(x, s.norm)
    logits = hidden @ s.head.double().t()
    cfg = logits
    if B >= 2:
        half = B // 2
        cond, uncond = logits[:half], logits[half:]
        cfg = uncond + 3.0 * (cond - uncond)
    return {"hidden": hidden[:, None], "logits": logits, "cfg": cfg, "k": k, "v": v}
