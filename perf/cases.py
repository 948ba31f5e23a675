"""Workloads of the serving engine: what a deployment has it do, step by step.

Every case is one step (or the few steps of one long prompt) of an
`LLMEngine` with random weights of a catalog architecture. "prefill" cases
hand prompts to the engine and take the next-token logits of each;
"decode" cases advance every running request by one token from the decode
graph, as the engine does between two samplings.

Architectures: the layers of llama-3.1-8b, eight of its 32 deep (a pass costs
about a quarter of the model's, and the engine's preparation stays quick), in
bf16, with 4-bit weights, and with an fp8 K/V cache; and three stacks of the
hybrid benchmark at its middle size, w2048: the sliding-window MoE
transformer, the latent-attention MoE transformer and the Gurapel hybrid.

Weights: layer inputs of unit scale, queries and keys large enough that
attention is decided, sub-layer outputs smaller than the residual stream, and
routers that read a component that tokens of a kind share, as trained ones do.
"""
from __future__ import annotations

import dataclasses
import math
import random

import torch

F64 = torch.float64
DEV = "cuda"
LLAMA_LAYERS = 8
SIZE = "w2048"
KINDS = 16              # kinds of tokens that the routers tell apart
BUDGET = 8192           # tokens of one prompt step (the engine's default)


# ------------------------------------------------------------------ the cases

def _case(name, model, phase, batch, tokens, ragged=0.5, weights="bf16",
          kv="bf16"):
    return {"name": name, "model": model, "phase": phase, "batch": batch,
            "tokens": tokens, "ragged": ragged, "weights": weights, "kv": kv}


def listed():
    return [
        # one user in a chat, the answer being written: the smallest call
        _case("llama-decode-1", "llama", "decode", 1, 217),
        # the same from 4-bit weights, two users on a small replica
        _case("llama-w4a16-decode-2", "llama", "decode", 2, 340,
              weights="w4a16"),
        # a busy replica at the headline benchmark's 200 in / 200 out
        _case("llama-decode-250", "llama", "decode", 250, 400),
        # long documents under discussion, K/V cache in fp8
        _case("llama-fp8kv-decode-16", "llama", "decode", 16, 4100, kv="fp8"),
        # a burst of the headline benchmark's prompts fills one step
        _case("llama-prefill-short", "llama", "prefill", 40, 230, 0.3),
        # one long document, cut by the step's token budget
        _case("llama-prefill-long", "llama", "prefill", 1, 20011, 0.0),
        # the hybrid benchmark's two phases (prompts of 2048, batch 32)
        _case("swa-moe-prefill", "swa-moe", "prefill", 4, 2048, 0.0),
        _case("swa-moe-decode-32", "swa-moe", "decode", 32, 2048),
        _case("mla-moe-prefill", "mla-moe", "prefill", 4, 2048, 0.0),
        _case("mla-moe-decode-32", "mla-moe", "decode", 32, 2048),
        _case("gurapel-prefill", "gurapel", "prefill", 4, 2048, 0.0),
        _case("gurapel-decode-32", "gurapel", "decode", 32, 2048),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    model = rng.choice(("llama", "llama", "swa-moe", "mla-moe", "gurapel"))
    phase = rng.choice(("prefill", "decode"))
    ragged = round(rng.uniform(0.0, 0.6), 2)
    weights = kv = "bf16"
    if phase == "decode":
        batch = spread(1, 250 if model == "llama" else 96)
        tokens = spread(64, min(4100, 98000 // batch))
        if model == "llama":
            weights, kv = rng.choice((("bf16", "bf16"), ("bf16", "bf16"),
                                      ("bf16", "fp8"), ("w4a16", "bf16")))
            if weights == "w4a16":
                batch = spread(1, 8)
    else:
        # whole prompts of one step, or one prompt of several
        if model == "llama" and rng.random() < 0.3:
            batch, tokens = 1, spread(BUDGET, 20000)
        else:
            tokens = spread(100, 4096)
            batch = spread(1, max(1, BUDGET // tokens))
    c = _case("", model, phase, batch, tokens, ragged, weights, kv)
    del c["name"]
    return c


def _lengths(case):
    """Prompt (decode: context) lengths; a property of the case."""
    r = random.Random(case["batch"] * 1000003 + case["tokens"])
    lo = max(1, int(case["tokens"] * (1 - case["ragged"])))
    return [case["tokens"]] + [r.randint(lo, case["tokens"])
                               for _ in range(case["batch"] - 1)]


def _tokens(case, seed, vocab):
    """Known tokens per request; decode: the last one is the step's own."""
    more = 1 if case["phase"] == "decode" else 0
    g = torch.Generator().manual_seed(seed)
    return [torch.randint(10, vocab - 10, (n + more,), generator=g).tolist()
            for n in _lengths(case)]


def _steps(case, known):
    """Prompt steps as (request, tokens) portions under the token budget."""
    out, room = [[]], BUDGET
    for i, toks in enumerate(known):
        left = len(toks) - (1 if case["phase"] == "decode" else 0)
        # prompts that fit a step stay whole
        if left > room and left <= BUDGET and out[-1]:
            out.append([])
            room = BUDGET
        while left:
            n = min(left, room)
            out[-1].append((i, n))
            left -= n
            room -= n
            if room == 0:
                out.append([])
                room = BUDGET
    return [s for s in out if s]


# ------------------------------------------------------------------ weights

def _sizes(case):
    if case["model"] == "llama":
        return dict(width=4096, layers=LLAMA_LAYERS, heads=32, kv_heads=8,
                    dim=128, vocab=128256, ff=14336, theta=500000.0, window=0,
                    experts=0)
    z = dict(width=2048, layers=6, heads=16, kv_heads=4, dim=128, window=1024,
             experts=8, top=2, ff=2048, vocab=32000, lru_blocks=16,
             theta=10000.0 if case["model"] != "swa-moe" else 500000.0,
             nope=128, rope=64, rank=512, groups=4, keep=2)
    if case["model"] == "mla-moe":
        z["theta"] = 500000.0
    return z


def _shapes(case):
    """(name, shape, f32?, how to draw it) of every weight, by the
    parameters' names in the model."""
    z = _sizes(case)
    h, L = z["width"], z["layers"]
    inp, out = h ** -0.5, (2 * L) ** -0.5
    m = case["model"]
    rows = [("embed_tokens.weight", (z["vocab"], h), 0, "embed")]

    def moe(p, f32):
        e, ff = z["experts"], z["ff"]
        rows.append((p + "gate", (e, h), f32, "router"))
        rows.append((p + "w_gate_up", (e, 2 * ff, h), 0, inp))
        rows.append((p + "w_down", (e, h, ff), 0, 1.5 * out * ff ** -0.5))

    def dense(p, ff):
        rows.append((p + "gate_up_proj.weight", (2 * ff, h), 0, inp))
        rows.append((p + "down_proj.weight", (h, ff), 0,
                     1.5 * out * ff ** -0.5))

    if m == "gurapel":
        rows.append(("pos_embed", (_max_len(case), h), 0, 0.3))
    for i in range(L):
        p = "layers.%d." % i
        if m == "gurapel":
            n = z["heads"] * z["dim"]
            g = z["kv_heads"] * z["dim"]
            if i % 3 == 0:
                q = p + "mixer."
                rows += [
                    (q + "in_proj", (2 * g + 2 * n + 2 * z["heads"], h), 0,
                     inp),
                    (q + "conv_weight", (2 * g + n, 4), 1, 0.5),
                    (q + "a_log", (z["heads"],), 1, (-2.5, 0.5)),
                    (q + "dt_bias", (z["heads"],), 1, 0.3),
                    (q + "out_norm", (z["dim"],), 1, (0.8, 1.2)),
                    (q + "o_proj", (h, n), 0, n ** -0.5)]
            else:
                q = p + "attn."
                rows += [
                    (q + "qkv_proj", (n + 2 * g, h), 0, inp),
                    (q + "q_norm", (z["dim"],), 1, (1.0, 1.8)),
                    (q + "k_norm", (z["dim"],), 1, (1.0, 1.8)),
                    (q + "r1", (z["heads"],), 1, (0.05, 0.6)),
                    (q + "r2", (z["heads"],), 1, (0.1, 1.0)),
                    (q + "o_proj", (h, n), 0, n ** -0.5)]
                q, nb = p + "rglru.", z["lru_blocks"]
                bw = h // nb
                rows += [
                    (q + "in_proj", (2 * h, h), 0, inp),
                    (q + "in_bias", (2 * h,), 0, 0.1),
                    (q + "conv_weight", (h, 4), 1, 0.5),
                    (q + "conv_bias", (h,), 1, 0.1),
                    (q + "gate_w", (nb, bw, 2 * bw), 1, bw ** -0.5),
                    (q + "gate_b", (nb, 1, 2 * bw), 1, 0.3),
                    (q + "decay_rate", (h,), 1, (0.02, 1.0)),
                    (q + "o_proj", (h, h), 0, inp)]
                rows += [(p + "attn_out_norm", (h,), 1, (0.8, 1.2)),
                         (p + "rglru_out_norm", (h,), 1, (0.8, 1.2))]
            rows.append((p + "norm1", (h,), 1, (0.1, 0.3)))
            moe(p + "mlp.", 1)
            rows.append((p + "norm2", (h,), 1, (0.1, 0.3)))
            continue
        q = p + "self_attn."
        if m == "mla-moe":
            H, d = z["heads"], z["nope"] + z["rope"]
            rows += [
                (q + "q_proj.weight", (H * d, h), 0, 1.5 * inp),
                (q + "kv_a_proj_with_mqa", (z["rank"] + z["rope"], h), 0,
                 inp),
                (q + "kv_a_layernorm", (z["rank"],), 0, (0.8, 1.2)),
                (q + "w_kc", (H, z["nope"], z["rank"]), 0,
                 z["rank"] ** -0.5),
                (q + "w_vc", (H, z["rank"], z["nope"]), 0,
                 z["rank"] ** -0.5),
                (q + "o_proj.weight", (h, H * z["nope"]), 0,
                 out * (H * z["nope"]) ** -0.5)]
            if i == 0:
                dense(p + "mlp.", z["ff"] * (z["top"] + 1))
            else:
                moe(p + "mlp.", 0)
                rows += [
                    (p + "mlp.e_score_correction_bias", (z["experts"],), 1,
                     0.02),
                    (p + "mlp.w_shared_gate_up", (2 * z["ff"], h), 0, inp),
                    (p + "mlp.w_shared_down", (h, z["ff"]), 0,
                     1.5 * out * z["ff"] ** -0.5)]
        else:
            n = z["heads"] * z["dim"]
            g = z["kv_heads"] * z["dim"]
            rows += [(q + "qkv_proj.weight", (n + 2 * g, h), 0, 1.3 * inp),
                     (q + "o_proj.weight", (h, n), 0, out * n ** -0.5)]
            if z["experts"]:
                moe(p + "mlp.", 0)
            else:
                dense(p + "mlp.", z["ff"])
        rows += [(p + "input_layernorm", (h,), 0, (0.8, 1.2)),
                 (p + "post_attention_layernorm", (h,), 0, (0.8, 1.2))]
    rows.append(("norm", (h,), m == "gurapel", (0.8, 1.2)))
    rows.append(("lm_head" if m == "gurapel" else "lm_head.weight",
                 (z["vocab"], h), 0, inp))
    return rows


def _preferences(case, z, order):
    """[experts, KINDS] router logits of the kinds: evenly spaced, in an
    order per kind; with groups, an order that decides between them too."""
    e = z["experts"]
    steps = torch.linspace(-2.5, 2.5, e)

    def margin(t):
        if case["model"] != "mla-moe":
            return 1.0
        s = torch.sigmoid(t).view(z["groups"], -1)
        best = s.topk(2, -1)[0].sum(-1)
        b = best.sort(descending=True)[0]
        inside = s[best.topk(z["keep"])[1]].flatten().sort(
            descending=True)[0]
        return min(b[z["keep"] - 1] - b[z["keep"]],
                   inside[z["top"] - 1] - inside[z["top"]]).item()
    cols = []
    for _ in range(KINDS):
        tries = [steps[torch.tensor(order.sample(range(e), e))]
                 for _ in range(16)]
        cols.append(max(tries, key=margin))
    return torch.stack(cols, 1)


def _weights(case, seed):
    """Yields (name, tensor as the model holds it)."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    z = _sizes(case)
    h = z["width"]

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=DEV)

    order = random.Random(seed)
    centers = normal(KINDS, h)
    for name, shape, f32, how in _shapes(case):
        if how == "embed":
            t = torch.empty(shape, dtype=torch.bfloat16, device=DEV)
            t.normal_(0, 0.6, generator=g)
            t += (0.8 * centers)[torch.arange(shape[0], device=DEV)
                                 % KINDS].to(t.dtype)
        elif how == "router":
            t = _preferences(case, z, order).to(DEV) @ centers / h
        elif isinstance(how, tuple):
            t = torch.empty(shape, device=DEV).uniform_(*how, generator=g)
        else:
            t = torch.empty(shape, dtype=torch.float32 if f32
                            else torch.bfloat16, device=DEV)
            t.normal_(0, how, generator=g)
        yield name, t.to(torch.float32 if f32 else torch.bfloat16)


def _max_len(case):
    return max(_lengths(case)) + 16


# ------------------------------------------------------------------ the engine

def _config(case):
    from kaito_amd.engine import hybrid_bench
    from kaito_amd.models import get_model_config
    n = _max_len(case)
    if case["model"] == "llama":
        return dataclasses.replace(get_model_config("llama-3.1-8b"),
                                   num_layers=LLAMA_LAYERS)
    make = {"swa-moe": hybrid_bench.transformer_config,
            "mla-moe": hybrid_bench.latent_transformer_config,
            "gurapel": hybrid_bench.hybrid_config}[case["model"]]
    return make(SIZE, hybrid_bench.SIZES[SIZE], n)


@torch.no_grad()
def prepare(case, seed):
    from kaito_amd.engine import EngineConfig, LLMEngine
    from kaito_amd.engine.scheduler import ScheduledBatch
    from kaito_amd.models.quant import quantize_parallel_linears
    from kaito_amd.parallel import state as ps
    ps.init_parallel(1)
    mc = _config(case)
    known = _tokens(case, seed, mc.vocab_size)
    n = _max_len(case)
    slots = case["batch"]
    if case["phase"] == "decode":   # the engine pads to the next graph
        slots = min(b for b in EngineConfig().graph_batch_sizes
                    if b >= case["batch"])
    eng = LLMEngine(EngineConfig(
        model=mc, device=DEV, max_num_seqs=slots, max_model_len=n,
        max_num_batched_tokens=BUDGET, graph_batch_sizes=(slots,),
        num_gpu_blocks=sum(-(-len(t) // 16) + 1 for t in known) + 1,
        kv_cache_dtype="fp8" if case["kv"] == "fp8" else "auto",
        enable_prefix_caching=False))
    params = dict(eng.runner.model.named_parameters())
    for name, t in _weights(case, seed):
        p = params.pop(name)
        assert p.shape == t.shape and p.dtype == t.dtype, name
        p.copy_(t)
    assert not params, list(params)
    if case["weights"] == "w4a16":
        quantize_parallel_linears(eng.runner.model)
    state = {"eng": eng, "known": known, "steps": _steps(case, known),
             "batch": None}
    if case["phase"] == "decode":
        eng.capture_graphs()
        for i, toks in enumerate(known):
            eng.extend_request(i, toks[:-1])
        for step in state["steps"]:
            eng.step_explicit(step, [])
        for i, toks in enumerate(known):
            eng.extend_request(i, toks[-1:])
        # pages for the step's own tokens
        seqs = eng.scheduler.schedule_explicit(
            [(eng.seqs[i], 1) for i in range(len(known))]).seqs
        state["batch"] = ScheduledBatch(is_prefill=False, seqs=seqs)
    return state


def run(state):
    eng = state["eng"]
    if state["batch"] is not None:
        return eng.runner.execute(state["batch"])
    known = state["known"]
    for i, toks in enumerate(known):
        eng.extend_request(i, toks)
    left = [len(t) for t in known]
    logits = []
    for step in state["steps"]:
        want = []
        for j, (i, n) in enumerate(step):
            left[i] -= n
            if left[i] == 0:
                want.append((j, n - 1))
        out = eng.step_explicit(step, want)
        if out is not None:
            logits.append(out)
    for i in range(len(known)):
        eng.release(i)
    return logits


# ------------------------------------------------------------------ costs

def work(case):
    z = _sizes(case)
    lens = _lengths(case)
    decode = case["phase"] == "decode"
    T = len(lens) if decode else sum(lens)
    heads, dim = z["heads"], z["dim"]
    total = active = 0.0            # weight bytes read, weights per token
    for name, shape, f32, how in _shapes(case):
        n = math.prod(shape)
        size = 4 if f32 else 2
        if name in ("embed_tokens.weight", "pos_embed"):
            total += T * shape[1] * size
        elif name.startswith("lm_head"):
            total += n * size
        elif name.endswith(("w_gate_up", "w_down")):
            hit = min(z["experts"], T * z["top"])
            total += n * size * hit / z["experts"]
            active += n * z["top"] / z["experts"]
        else:
            if case["weights"] == "w4a16" and len(shape) == 2:
                size = 0.5 + 8 / 128
            total += n * size
            active += n if len(shape) > 1 else 0
    # keys that each of the step's queries sees, summed
    def seen(n):
        w = z["window"] or n
        if decode:
            return min(n + 1, w)
        return n * (n + 1) / 2 - max(0, n - w) * (n - w + 1) / 2
    keys = sum(seen(n) for n in lens)
    kv_el = 1 if case["kv"] == "fp8" else 2
    flops = 2 * active * T
    if case["model"] == "mla-moe":
        row = (z["rank"] + z["rope"]) * 2
        per_key = 2 * heads * (z["rank"] * 2 + z["rope"]) if decode else \
            2 * heads * (2 * z["nope"] + z["rope"])
        layers = z["layers"]
    else:
        row = 2 * z["kv_heads"] * dim * kv_el
        per_key = 4 * heads * dim
        layers = z["layers"]
        if case["model"] == "gurapel":
            layers = z["layers"] * 2 // 3
            recur = z["layers"] - layers
            flops += recur * T * heads * dim * dim * 6
            states = len(lens) * (recur * heads * dim * dim * 4
                                  + layers * z["width"] * 4)
            total += states * (2 if decode else 1)
    flops += layers * keys * per_key
    # decode reads every visible row; a prompt's rows are written once
    total += layers * row * ((keys + T) if decode else T)
    flops += 2 * z["vocab"] * z["width"] * len(lens)
    total += len(lens) * z["vocab"] * 4
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """Relative error of logits: bf16 activations through 6 or 8 layers are
    0.008 to 0.01 off their value in 64 bits, two implementations of them
    a little more off each other."""
    return {"rel": 0.04}


# ------------------------------------------------------------------ in 64 bits

def _lin(x, w):
    """x [T, in] @ w [out, in] transposed, in row blocks."""
    w = w.to(F64)
    return torch.cat([b @ w.T for b in x.split(16384)])


def _rms(x, w, eps=1e-5):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.to(F64)


def _silu(x):
    return x * torch.sigmoid(x)


def _swiglu(x, gate_up, down):
    out = []
    for b in x.split(8192):
        g, u = _lin(b, gate_up).chunk(2, -1)
        out.append(_lin(_silu(g) * u, down))
    return torch.cat(out)


def _rope(x, pos, theta):
    """x [T, heads, dim]: halves rotated against each other."""
    half = x.shape[-1] // 2
    inv = theta ** (-torch.arange(half, dtype=F64, device=x.device) / half)
    a = pos.to(F64)[:, None] * inv
    c, s = a.cos()[:, None], a.sin()[:, None]
    p, q = x[..., :half], x[..., half:]
    return torch.cat([p * c - q * s, q * c + p * s], -1)


def _attend(q, k, v, scale, window=0, scores=None, first=0):
    """q [n, H, d] at positions first.., k/v [m, G, d] from position 0."""
    n, H, _ = q.shape
    rep = H // k.shape[1]
    k = k.repeat_interleave(rep, 1).permute(1, 2, 0)
    v = v.repeat_interleave(rep, 1).transpose(0, 1)
    at = torch.arange(k.shape[2], device=q.device)
    out = []
    for a in range(0, n, 512):
        pos = torch.arange(first + a, first + min(n, a + 512),
                           device=q.device)[:, None]
        s = torch.matmul(q[a:a + 512].transpose(0, 1), k) * scale
        dist = pos - at
        if scores is not None:
            s = scores(s, dist)
        dead = dist < 0
        if window:
            dead = dead | (dist >= window)
        s = s.masked_fill_(dead, float("-inf")).softmax(-1)
        out.append(torch.matmul(s, v).transpose(0, 1))
    return torch.cat(out)


def _mix(x, W, p, idx, wts):
    """Routed experts: idx, wts [T, k]."""
    out = torch.zeros_like(x)
    for e in range(W[p + "w_gate_up"].shape[0]):
        t, j = torch.nonzero(idx == e, as_tuple=True)
        if len(t):
            y = _swiglu(x[t], W[p + "w_gate_up"][e], W[p + "w_down"][e])
            out.index_add_(0, t, y * wts[t, j, None])
    return out


def _top_softmax(x, W, p, top):
    z, idx = _lin(x, W[p + "gate"]).topk(top, -1)
    return _mix(x, W, p, idx, z.softmax(-1))


def _corrected(x, W, p, z):
    """Sigmoid scores; the choice adds a correction and is limited to the
    groups with the largest sum of their two best."""
    s = torch.sigmoid(_lin(x, W[p + "gate"]))
    c = (s + W[p + "e_score_correction_bias"].to(F64)).view(
        len(x), z["groups"], -1)
    best = c.topk(2, -1)[0].sum(-1).topk(z["keep"], -1)[1]
    keep = torch.zeros(c.shape[:2], dtype=torch.bool, device=x.device)
    keep.scatter_(1, best, True)
    c = c.masked_fill(~keep[..., None], float("-inf")).view(len(x), -1)
    idx = c.topk(z["top"], -1)[1]
    return _mix(x, W, p, idx, s.gather(1, idx)) + _swiglu(
        x, W[p + "w_shared_gate_up"], W[p + "w_shared_down"])


def _conv(x, w, lens, bias=None):
    """Causal, per sequence; the last column weighs the token itself."""
    taps, out = w.shape[1], []
    for s in x.split(lens):
        y = torch.zeros_like(s)
        for j in range(taps):
            back = taps - 1 - j
            y[back:] += w[:, j].to(F64) * s[:len(s) - back]
        out.append(y)
    y = torch.cat(out)
    return y if bias is None else y + bias.to(F64)


def _padded(x, lens):
    return torch.nn.utils.rnn.pad_sequence(list(x.split(lens)))   # [T, B, ..]


def _unpadded(y, lens):
    return torch.cat([y[:n, b] for b, n in enumerate(lens)])


def _delta(x, W, p, z, lens):
    H, G, D = z["heads"], z["kv_heads"], z["dim"]
    y = _lin(x, W[p + "in_proj"])
    c = (2 * G + H) * D
    qkv = _silu(_conv(y[:, :c], W[p + "conv_weight"], lens))
    gate = _silu(y[:, c:c + H * D]).view(-1, H, D)
    a, b = y[:, c + H * D:].chunk(2, -1)
    q, k, v = qkv.split([G * D, G * D, H * D], -1)

    def unit(t):
        t = t.reshape(-1, G, D)
        t = t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)
        return _padded(t.repeat_interleave(H // G, 1), lens)
    q, k = unit(q) / math.sqrt(D), unit(k)
    v = _padded(v.reshape(-1, H, D), lens)
    beta = _padded(torch.sigmoid(b), lens)[..., None]
    step = torch.nn.functional.softplus(a + W[p + "dt_bias"].to(F64))
    decay = _padded(torch.exp(-torch.exp(W[p + "a_log"].to(F64)) * step),
                    lens)[..., None, None]
    S = torch.zeros(len(lens), H, D, D, dtype=F64, device=x.device)
    o = torch.empty_like(v)
    for t in range(len(v)):
        S = S * decay[t]
        u = beta[t] * (v[t] - (k[t][:, :, None] @ S)[:, :, 0])
        S = S + k[t][..., None] * u[:, :, None]
        o[t] = (q[t][:, :, None] @ S)[:, :, 0]
    o = _rms(_unpadded(o, lens), W[p + "out_norm"]) * gate
    return _lin(o.reshape(len(x), -1), W[p + "o_proj"])


def _recurrent(x, W, p, z, lens):
    h, nb = z["width"], z["lru_blocks"]
    y, u = (_lin(x, W[p + "in_proj"]) + W[p + "in_bias"].to(F64)).chunk(2, -1)
    y = torch.nn.functional.gelu(y, approximate="tanh")
    u = _conv(u, W[p + "conv_weight"], lens, W[p + "conv_bias"])
    ub = u.view(-1, nb, h // nb).transpose(0, 1)
    g = torch.sigmoid(ub.contiguous() @ W[p + "gate_w"].to(F64)
                      + W[p + "gate_b"].to(F64))
    r, i = (t.transpose(0, 1).reshape(-1, h) for t in g.chunk(2, -1))
    log_a = -r * W[p + "decay_rate"].to(F64)
    a = _padded(torch.exp(log_a), lens)
    b = _padded(torch.sqrt(-torch.expm1(2 * log_a)) * i * u, lens)
    S = torch.zeros_like(b[0])
    o = torch.empty_like(b)
    for t in range(len(b)):
        S = a[t] * S + b[t]
        o[t] = S
    return _lin(_unpadded(o, lens) * y, W[p + "o_proj"])


def _windowed(x, W, p, z, lens):
    H, G, D = z["heads"], z["kv_heads"], z["dim"]
    q, k, v = _lin(x, W[p + "qkv_proj"]).split([H * D, G * D, G * D], -1)
    q = _rms(q.reshape(-1, H, D), W[p + "q_norm"])
    k = _rms(k.reshape(-1, G, D), W[p + "k_norm"])
    r1 = W[p + "r1"].to(F64)[:, None, None]
    r2 = W[p + "r2"].to(F64)[:, None, None]

    def scores(s, dist):
        return 30 * torch.tanh(s / 30) - r1 * torch.log1p(
            r2 * dist.clamp(min=0).to(F64))
    o = torch.cat([_attend(a, b, c, D ** -0.5, z["window"], scores)
                   for a, b, c in zip(q.split(lens), k.split(lens),
                                      v.reshape(-1, G, D).split(lens))])
    return _lin(o.reshape(len(x), -1), W[p + "o_proj"])


def _rotary(x, W, p, z, lens, pos, fp8):
    H, G, D = z["heads"], z["kv_heads"], z["dim"]
    q, k, v = _lin(x, W[p + "qkv_proj.weight"]).split(
        [H * D, G * D, G * D], -1)
    q = _rope(q.reshape(-1, H, D), pos, z["theta"])
    k = _rope(k.reshape(-1, G, D), pos, z["theta"])
    out = []
    for a, b, c in zip(q.split(lens), k.split(lens),
                       v.reshape(-1, G, D).split(lens)):
        o = _attend(a, b, c, D ** -0.5, z["window"])
        if fp8:     # the step's query reads the cache, prompts did not
            b, c = (t.to(torch.bfloat16).to(torch.float8_e4m3fn).to(F64)
                    for t in (b, c))
            o[-1:] = _attend(a[-1:], b, c, D ** -0.5, first=len(a) - 1)
        out.append(o)
    return _lin(torch.cat(out).reshape(len(x), -1), W[p + "o_proj.weight"])


def _latent(x, W, p, z, lens, pos):
    H, d, r = z["heads"], z["nope"], z["rank"]
    q = _lin(x, W[p + "q_proj.weight"]).view(-1, H, d + z["rope"])
    kv = _lin(x, W[p + "kv_a_proj_with_mqa"])
    c = _rms(kv[:, :r], W[p + "kv_a_layernorm"])
    qr = _rope(q[..., d:], pos, z["theta"])
    kr = _rope(kv[:, None, r:], pos, z["theta"])
    wk, wv = W[p + "w_kc"].to(F64), W[p + "w_vc"].to(F64)
    k = (c @ wk.reshape(H * d, r).T).view(-1, H, d)
    v = (c @ wv.transpose(0, 1).reshape(r, H * d)).view(-1, H, d)
    k = torch.cat([k, kr.expand(-1, H, -1)], -1)
    q = torch.cat([q[..., :d], qr], -1)
    o = torch.cat([_attend(a, b, e, (d + z["rope"]) ** -0.5)
                   for a, b, e in zip(q.split(lens), k.split(lens),
                                      v.split(lens))])
    return _lin(o.reshape(len(x), -1), W[p + "o_proj.weight"])


def _as_quantized(w, group=128):
    """w as 4-bit codes of its groups say it (asymmetric, in f32)."""
    v = w.float().reshape(w.shape[0], -1, group)
    hi, lo = v.amax(-1), v.amin(-1)
    scale = (hi - lo).clamp(min=1e-8) / 15.0
    zero = (-lo / scale).round().clamp(0, 15)
    q = (v / scale[..., None] + zero[..., None]).round().clamp(0, 15)
    q, scale = q.to(F64), scale.to(F64)
    return ((q - zero.to(F64)[..., None]) * scale[..., None]).reshape(w.shape)


@torch.no_grad()
def exact(case, seed):
    z = _sizes(case)
    W = dict(_weights(case, seed))
    if case["weights"] == "w4a16":
        for name in W:
            if name.startswith("layers.") and name.endswith("proj.weight"):
                W[name] = _as_quantized(W[name])
    known = _tokens(case, seed, z["vocab"])
    lens = [len(t) for t in known]
    ids = torch.tensor(sum(known, []), device=DEV)
    pos = torch.cat([torch.arange(n, device=DEV) for n in lens])
    x = W["embed_tokens.weight"][ids].to(F64)
    m = case["model"]
    if m == "gurapel":
        x = x + W["pos_embed"][pos].to(F64)
    for i in range(z["layers"]):
        p = "layers.%d." % i
        if m == "gurapel":
            if i % 3 == 0:
                y = _delta(x, W, p + "mixer.", z, lens)
            else:
                y = 0.5 * (_rms(_windowed(x, W, p + "attn.", z, lens),
                                W[p + "attn_out_norm"])
                           + _rms(_recurrent(x, W, p + "rglru.", z, lens),
                                  W[p + "rglru_out_norm"]))
            x = x + _rms(y, W[p + "norm1"])
            y = _top_softmax(x, W, p + "mlp.", z["top"])
            x = x + _rms(y, W[p + "norm2"])
            continue
        y = _rms(x, W[p + "input_layernorm"])
        x = x + (_latent(y, W, p + "self_attn.", z, lens, pos)
                 if m == "mla-moe" else
                 _rotary(y, W, p + "self_attn.", z, lens, pos,
                         case["kv"] == "fp8"))
        y = _rms(x, W[p + "post_attention_layernorm"])
        q = p + "mlp."
        if q + "gate" not in W:
            x = x + _swiglu(y, W[q + "gate_up_proj.weight"],
                            W[q + "down_proj.weight"])
        elif m == "mla-moe":
            x = x + _corrected(y, W, q, z)
        else:
            x = x + _top_softmax(y, W, q, z["top"])
    last = torch.tensor(lens, device=DEV).cumsum(0) - 1
    x = _rms(x[last], W["norm"])
    logits = _lin(x, W["lm_head" if m == "gurapel" else "lm_head.weight"])
    if case["phase"] == "decode":
        return logits
    # one block of rows per step that completes a prompt
    left, out, row = list(lens), [], 0
    for step in _steps(case, known):
        n = 0
        for i, k in step:
            left[i] -= k
            n += left[i] == 0
        if n:
            out.append(logits[row:row + n])
            row += n
    return out
