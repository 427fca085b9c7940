"""The serving steps whose speed is followed from one change to the next.

A case is ONE step of the engine's model runner on a batch that the engine's
own scheduler assembled: a prompt step (ModelRunner.forward_logits), a chunk
behind a cached history (the same call), or a decode step (the captured graph
and the greedy sampler, ModelRunner.execute_async). The models are stacks of
the framework's own presets and bench configurations cut to four layers, with
random weights of the sizes named there, and with the full vocabulary head:

* "llama": llama-3-8b, the flagship of bench.py;
* "moe":   qwen3-30b-a3b, 128 experts, 8 a token;
* "hybrid": the medium Livasun stack of the layer bench — windowed attention
  without rotation, a mamba2 mixer and a lightning mixer on an fp32 stream.

Weights, cached keys and values, recurrent states and tokens come from the
seed. Scores have a spread of about two, routers decide clearly and an expert
adds a fraction of the stream, as trained ones do; with the flat scores of plain
random weights a rounding error sends a row to another expert of the same
weight, and a step then differs from `exact` by 2 to 7 % however it is computed
(router gains of 1, 2, 3, 4: 2.6, 1.9, 1.4, 1.1 % at 64 rows).

`exact` computes a step in float64 with plain torch from the same numbers.
"""
from __future__ import annotations

import math
import zlib

import torch

from gpustack_amd.bench.layer_bench import SIZES, livasun_spec
from gpustack_amd.engine import EngineConfig
from gpustack_amd.engine.model_runner import ModelRunner
from gpustack_amd.engine.scheduler import Scheduler
from gpustack_amd.engine.sequence import SamplingParams, Sequence, SeqStatus

LAYERS = 4
PRESET = {"llama": "llama-3-8b", "moe": "qwen3-30b-a3b"}


# --- the cases -------------------------------------------------------------

def _case(model, kind, seqs, lo, hi, hist=0, kv="bf16", w4=False):
    """`lo`..`hi`: rows per sequence of a prompt step, or the tokens already
    cached per sequence of a decode step; `hist`: cached tokens in front of
    every sequence's rows of a chunk."""
    return {"model": model, "kind": kind, "seqs": seqs, "lo": lo, "hi": hi,
            "hist": hist, "kv": kv, "w4": w4}


def listed():
    rows = [
        # one user chatting: the smallest step, bound by the weight stream
        # and the number of launches
        ("decode-1", _case("llama", "decode", 1, 1000, 1000)),
        # bench.py's steady state: 512 requests of 256 + 128 tokens
        ("decode-512", _case("llama", "decode", 512, 256, 383)),
        # long conversations on the fp8 cache (--kv-dtype fp8)
        ("decode-48-long-fp8", _case("llama", "decode", 48, 3500, 7900,
                                     kv="fp8")),
        # a short question arriving alone: time to first token
        ("prompt-77", _case("llama", "prompt", 1, 77, 77)),
        # bench.py's admission wave: 32 prompts of 256
        ("prompt-32x256", _case("llama", "prompt", 32, 256, 256)),
        # one long document, as much as a step's token budget takes
        ("prompt-7999", _case("llama", "prompt", 1, 7999, 7999)),
        # chunked prefill, or a prompt behind a cached prefix
        ("chunk-2039", _case("llama", "chunk", 1, 2039, 2039, hist=6001)),
        # packed int4 weights (--quantize w4), a handful of users
        ("decode-16-w4", _case("llama", "decode", 16, 300, 1200, w4=True)),
        # mixture of experts, both directions
        ("moe-decode-64", _case("moe", "decode", 64, 200, 2000)),
        ("moe-prompt-9", _case("moe", "prompt", 9, 203, 701)),
        # recurrent and windowed layers, both directions
        ("hybrid-prompt-6", _case("hybrid", "prompt", 6, 301, 1900)),
        ("hybrid-decode-64", _case("hybrid", "decode", 64, 200, 3000)),
    ]
    return [{"name": n, **c} for n, c in rows]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    form = rng.choice(["decode", "decode", "decode-fp8", "decode-w4",
                       "prompt", "prompt", "chunk", "moe-decode",
                       "moe-prompt", "hybrid-prompt", "hybrid-decode"])
    if form == "decode":
        n = _log(rng, 1, 512)
        lo = _log(rng, 20, 2000)
        return _case("llama", "decode", n, lo, min(7900, int(lo * rng.uniform(1, 3))))
    if form == "decode-fp8":
        n = _log(rng, 1, 64)
        lo = _log(rng, 200, 5000)
        return _case("llama", "decode", n, lo, min(7900, int(lo * rng.uniform(1, 2))),
                     kv="fp8")
    if form == "decode-w4":
        n = _log(rng, 1, 64)
        lo = _log(rng, 50, 1500)
        return _case("llama", "decode", n, lo, int(lo * rng.uniform(1, 2)),
                     w4=True)
    if form == "chunk":
        return _case("llama", "chunk", 1, *(2 * [_log(rng, 33, 2039)]),
                     hist=_log(rng, 64, 6001))
    model, _, kind = form.rpartition("-")
    model = model or "llama"
    if kind == "decode":
        n = _log(rng, 1, 64)
        lo = _log(rng, 100, 2000)
        return _case(model, kind, n, lo, int(lo * rng.uniform(1, 1.5)))
    # prompts share a budget of rows
    total = _log(rng, 33, 7999 if model == "llama" else 4000)
    n = min(_log(rng, 1, 32), max(1, total // 33))
    mid = total // n
    lo = max(1, int(mid * rng.uniform(0.5, 1)))
    return _case(model, kind, n, lo, max(lo, 2 * mid - lo))


def _lens(case):
    """The sequences' sizes, spread over lo..hi in no particular order."""
    lo, hi = case["lo"], case["hi"]
    return [lo + int((hi - lo) * ((i * 0.6180339887 + 0.5) % 1.0))
            for i in range(case["seqs"])]


def _rows(case):
    """(cached tokens, rows of the step) of every sequence."""
    if case["kind"] == "decode":
        return [(n, 1) for n in _lens(case)]
    return [(case["hist"], n) for n in _lens(case)]


# --- numbers from the seed -------------------------------------------------

def _normal(seed, key, shape, std=1.0, base=0.0):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + zlib.crc32(key.encode())) % (1 << 62))
    t = torch.randn(*shape, generator=g, dtype=torch.float32, device="cuda")
    return t.mul_(std).add_(base)


def _tokens(seed, n, vocab):
    g = torch.Generator()
    g.manual_seed(int(seed) + 77)
    return torch.randint(2, vocab, (n,), generator=g)


def _spec(case):
    if case["model"] == "hybrid":
        return livasun_spec(dict(SIZES["medium"], layers=LAYERS))
    spec = EngineConfig(model=PRESET[case["model"]], device="cpu").spec
    spec.num_layers = LAYERS
    return spec


def _weight(seed, name, shape, dtype, case):
    """One weight, by name: projections keep the size of what they read,
    norms are near 1, queries and routers a little larger."""
    leaf = name.rsplit(".", 1)[-1]
    std, base = 0.05, 0.0
    if leaf == "embed":
        std = 1.0
    elif leaf == "conv_w":
        std = 0.5
    elif leaf == "v_lam":
        base = 0.3
    elif leaf == "dt_bias":
        std, base = 0.5, -1.0
    elif leaf == "a_log":
        std = 0.5
    elif leaf in ("conv_b",):
        std = 0.3
    elif len(shape) > 1:
        std = shape[-1] ** -0.5
        if leaf == "router_w":
            std *= 4.0
        elif leaf == "down_w" and case["model"] == "moe":
            std *= 0.5
    elif not leaf.endswith("_b"):
        base = 2.0 if leaf in ("q_norm", "q_head_norm") else 1.0
    t = _normal(seed, name, shape, std, base)
    if leaf == "qkv_w" and case["model"] == "llama":
        t[:32 * 128] *= 2.0
    return t.to(dtype)


def _cached(seed, what, layer, n, heads, width, kv):
    t = _normal(seed, "%s%d" % (what, layer), (n, heads, width))
    return t.to(torch.float8_e4m3fn if kv == "fp8" else torch.bfloat16)


# --- the step ---------------------------------------------------------------

def prepare(case, seed):
    """A runner with its weights, the pools with what the sequences have
    cached, and the scheduled batch."""
    rows = _rows(case)
    need = sum((h + n + 16) // 16 + 1 for h, n in rows) + 8
    longest = max(h + n for h, n in rows)
    cfg = EngineConfig(
        model=PRESET.get(case["model"], "layer-bench"), device="cuda:0",
        max_num_seqs=len(rows), max_model_len=longest + 16,
        kv_cache_blocks=need, kv_cache_dtype=case["kv"], seed=int(seed) % 1000,
        admission_min_seqs=1)
    cfg.spec = _spec(case)
    runner = ModelRunner(cfg)
    for name, p in runner.model.named_parameters():
        p.data.copy_(_weight(seed, name, tuple(p.shape), p.dtype, case))
    if case["w4"]:
        from gpustack_amd.models.weights import convert_to_w4_runtime

        convert_to_w4_runtime(runner.model, cfg)
    kv = runner.init_kv_cache()
    sch = Scheduler(cfg, kv)
    toks = _tokens(seed, sum(h + n for h, n in rows), cfg.spec.vocab_size).tolist()
    seqs, at, slots = [], 0, []
    for i, (h, n) in enumerate(rows):
        s = Sequence("r%d" % i, toks[at:at + h + n],
                     SamplingParams(max_tokens=1 << 20, ignore_eos=True))
        at += h + n
        seqs.append(s)
        if h:
            s.block_table = kv.allocator.allocate(kv.blocks_needed(h))
            s.num_cached_tokens = h
            if kv.state_allocator is not None:
                s.state_slot = kv.state_allocator.allocate()
            slots.append(torch.as_tensor(kv.slots_for(s.block_table, 0, h)))
    if slots:
        _fill(case, seed, cfg.spec, kv, torch.cat(slots).cuda(), seqs)
    if case["kind"] == "decode":
        for s in seqs:
            s.status = SeqStatus.RUNNING
        sch.running.extend(seqs)
        batch = sch.schedule()
    elif case["kind"] == "chunk":
        batch = sch.schedule_forced([(s, n, [n - 1]) for s, (_, n) in
                                     zip(seqs, rows)])
    else:
        for s in seqs:
            sch.add(s)
        batch = sch.schedule()
    assert len(batch.seqs) == len(rows), "the whole batch in one step"
    assert [s.request_id for s in batch.seqs] == [s.request_id for s in seqs]
    return {"case": case, "runner": runner, "batch": batch}


def _fill(case, seed, spec, kv, slots, seqs):
    blk, off = slots // 16, slots % 16
    for i in range(LAYERS):
        if case["model"] != "hybrid":
            for what, pool in (("k", kv.k_caches[i]), ("v", kv.v_caches[i])):
                t = _cached(seed, what, i, slots.numel(), spec.num_kv_heads,
                            spec.head_dim, case["kv"])
                if case["kv"] == "fp8":
                    pool, t = pool.view(torch.uint8), t.view(torch.uint8)
                pool[blk, :, off] = t
            continue
        ls = spec.layers[i]
        if ls.mixer_type == "paged_attention":
            m = ls.mixer
            kv.k_caches[i][blk, :, off] = _cached(
                seed, "k", i, slots.numel(), m.kv_heads, m.qk_dim, "bf16")
            kv.v_caches[i][blk, :, :, off] = _cached(
                seed, "v", i, slots.numel(), m.kv_heads, m.v_dim, "bf16")
        else:
            at = torch.tensor([s.state_slot for s in seqs], device="cuda")
            state, conv = kv.ssm_states[i], kv.conv_states[i]
            state[at] = _normal(seed, "s%d" % i,
                                (len(seqs), *state.shape[1:]))
            if conv is not None:
                conv[at] = _normal(seed, "c%d" % i, (
                    len(seqs), *conv.shape[1:])).to(conv.dtype)


def run(state):
    """One step: its logits, and the pools that it wrote to."""
    runner, batch = state["runner"], state["batch"]
    if state["case"]["kind"] != "decode":
        logits = runner.forward_logits(batch)
    else:
        runner.execute_async(batch, reuse_tokens=False)
        gr = runner.graph_runner
        n = len(batch.seqs)
        logits = gr.outs[next(b for b in gr.buckets if b >= n)][:n]
    kv = runner.kv
    pools = [t for t in (*kv.k_caches, *kv.v_caches, *kv.ssm_states,
                         *kv.conv_states) if t is not None and t.numel()]
    return {"logits": logits, "pools": pools}


# --- what a step cannot do without ------------------------------------------

def work(case):
    spec, rows = _spec(case), _rows(case)
    T, n = sum(r for _, r in rows), len(rows)
    h, V = spec.hidden_size, spec.vocab_size
    byts = 2.0 * V * h + 2.0 * n * V + 2.0 * T * h
    flops = 2.0 * n * V * h

    def linear(rows_, out, inp, copies=1.0):
        nonlocal byts, flops
        byts += copies * out * inp * (0.5 if case["w4"] else 2.0)
        flops += 2.0 * rows_ * out * inp

    def attention(hq, hkv, d, window=0):
        nonlocal byts, flops
        b = 1 if case["kv"] == "fp8" else 2
        for hist, r in rows:
            seen = sum(min(hist + t + 1, window or hist + t + 1)
                       for t in range(r))
            keys = min(hist + r, (window + r) if window else hist + r)
            byts += 2.0 * b * hkv * d * (keys + r)
            flops += 4.0 * hq * d * seen

    for i in range(LAYERS):
        if case["model"] != "hybrid":
            hq, hkv, d = spec.num_heads, spec.num_kv_heads, spec.head_dim
            linear(T, (hq + 2 * hkv) * d, h)
            linear(T, h, hq * d)
            attention(hq, hkv, d)
            if spec.num_experts:
                E, k, f = (spec.num_experts, spec.num_experts_per_tok,
                           spec.moe_intermediate_size)
                hit = E * (1.0 - (1.0 - k / E) ** T)
                linear(T, E, h)
                linear(T * k, 3 * f, h, hit)
            else:
                linear(T, 3 * spec.intermediate_size, h)
            continue
        ls = spec.layers[i]
        m = ls.mixer
        if ls.mixer_type == "paged_attention":
            linear(T, (m.heads + 2 * m.kv_heads) * m.qk_dim, h)
            linear(T, h, m.heads * m.v_dim)
            attention(m.heads, m.kv_heads, m.qk_dim, m.window)
        else:
            inner = m.heads * m.vdim
            wide = (2 * inner + 2 * m.groups * m.state + m.heads
                    if m.kind == "mamba2" else 4 * inner)
            linear(T, wide, h)
            linear(T, h, inner)
            moved = sum(2 if hist else 1 for hist, _ in rows)
            byts += 4.0 * moved * inner * m.state
            flops += 5.0 * T * inner * m.state
        linear(T, 3 * ls.mlp.ff, h)
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    """bf16 operands through four layers: the steps are 0.7 to 1.0 % (llama),
    about 1 % (experts) and 0.3 % (hybrid, on an fp32 stream) away from
    `exact`."""
    return {"rel": 0.012 if case["model"] == "hybrid" else 0.03, "max": 0.5}


# --- the same step in float64 -------------------------------------------------

def exact(case, seed):
    spec = _spec(case)
    rows = _rows(case)
    toks = _tokens(seed, sum(h + n for h, n in rows), spec.vocab_size)
    now, at = [], 0
    for h, n in rows:
        now.append(toks[at + h:at + h + n])
        at += h + n
    ids = torch.cat(now).cuda()
    last, r0 = [], 0
    for _, n in rows:
        last.append(r0 + n - 1)
        r0 += n
    last = torch.tensor(last, device="cuda")
    x = (_exact_hybrid if case["model"] == "hybrid" else _exact_llama)(
        case, seed, spec, rows, ids, last)
    head = _w64(case, seed, "lm_head", (spec.vocab_size, spec.hidden_size))
    # the pools hold the same keys and values in pages of the engine's own
    return {"logits": x @ head.T, "pools": None}


def _w64(case, seed, name, shape, dtype=torch.bfloat16):
    w = _weight(seed, name, shape, dtype, case)
    leaf = name.rsplit(".", 1)[-1]
    if case["w4"] and leaf in ("qkv_w", "o_w", "gate_up_w", "down_w",
                               "lm_head"):
        # groups of 128 along the row, 4 bits, scale and offset in bf16
        g = w.float().view(shape[0], -1, 128)
        scale = ((g.amax(-1) - g.amin(-1)) / 15).clamp_min(1e-8)
        zero = (-g.amin(-1) / scale).round().clamp(0, 15)
        q = (g / scale.unsqueeze(-1) + zero.unsqueeze(-1)).round().clamp(0, 15)
        return (q.double() * scale.bfloat16().double().unsqueeze(-1)
                - (zero * scale).bfloat16().double().unsqueeze(-1)).view(shape)
    return w.double()


def _rms(x, w, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w


def _attend(q, k, v, hist, window=0, slopes=None):
    """q [n, H, D] behind hist keys, k / v [hist + n, G, D]."""
    n, H, D = q.shape
    L, G, _ = k.shape
    out = torch.empty(n, H, v.shape[2], dtype=torch.float64, device=q.device)
    pos = torch.arange(hist, hist + n, device=q.device)[:, None]
    key = torch.arange(L, device=q.device)[None, :]
    hide = key > pos
    if window:
        hide = hide | (pos - key >= window)
    step = max(1, min(H // G, int(2e8 // max(1, n * L))))
    for h0 in range(0, H, step):
        h1 = min(h0 + step, H)
        kk = k[:, [h * G // H for h in range(h0, h1)]].transpose(0, 1)
        vv = v[:, [h * G // H for h in range(h0, h1)]].transpose(0, 1)
        s = torch.bmm(q[:, h0:h1].transpose(0, 1),
                      kk.transpose(1, 2).contiguous()) * D ** -0.5
        if slopes is not None:
            s = s - slopes[h0:h1, None, None] * (pos - key)
        s = s.masked_fill_(hide, float("-inf")).softmax(-1)
        out[:, h0:h1] = torch.bmm(s, vv.contiguous()).transpose(0, 1)
    return out


def _history(case, seed, i, rows, heads, width):
    total = sum(h for h, _ in rows)
    if not total:
        return None, None
    return tuple(_cached(seed, w, i, total, heads, width, case["kv"])
                 .to(torch.float32).double() for w in ("k", "v"))


def _over_sequences(q, k, v, kc, vc, rows, **kw):
    out, r, c = [], 0, 0
    for h, n in rows:
        kk, vv = k[r:r + n], v[r:r + n]
        if h:
            kk = torch.cat([kc[c:c + h], kk])
            vv = torch.cat([vc[c:c + h], vv])
        out.append(_attend(q[r:r + n], kk, vv, h, **kw))
        r, c = r + n, c + h
    return torch.cat(out)


def _exact_llama(case, seed, spec, rows, ids, last):
    hq, hkv, d = spec.num_heads, spec.num_kv_heads, spec.head_dim
    H, eps = spec.hidden_size, spec.rms_norm_eps
    W = lambda name, *shape: _w64(case, seed, name, shape)
    pos = torch.cat([torch.arange(h, h + n) for h, n in rows]).cuda().double()
    inv = spec.rope_theta ** (-torch.arange(0, d, 2, device="cuda").double() / d)
    ang = pos[:, None] * inv
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rot(t):
        a, b = t[..., :d // 2], t[..., d // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    x = W("embed", spec.vocab_size, H)[ids]
    for i in range(LAYERS):
        p = "layers.%d." % i
        y = _rms(x, W(p + "input_norm", H), eps)
        qkv = (y @ W(p + "attn.qkv_w", (hq + 2 * hkv) * d, H).T).view(-1, hq + 2 * hkv, d)
        q, k, v = qkv[:, :hq], qkv[:, hq:hq + hkv], qkv[:, hq + hkv:]
        if spec.qk_norm:
            q = _rms(q, W(p + "attn.q_norm", d), eps)
            k = _rms(k, W(p + "attn.k_norm", d), eps)
        o = _over_sequences(rot(q), rot(k), v,
                            *_history(case, seed, i, rows, hkv, d), rows)
        x = x + o.reshape(-1, hq * d) @ W(p + "attn.o_w", H, hq * d).T
        y = _rms(x, W(p + "post_attn_norm", H), eps)
        if not spec.num_experts:
            f = spec.intermediate_size
            if i + 1 == LAYERS:
                x, y = x[last], y[last]
            gu = y @ W(p + "mlp.gate_up_w", 2 * f, H).T
            x = x + (torch.nn.functional.silu(gu[:, :f]) * gu[:, f:]) \
                @ W(p + "mlp.down_w", H, f).T
            continue
        E, f = spec.num_experts, spec.moe_intermediate_size
        top, ex = torch.topk(y @ W(p + "mlp.router_w", E, H).T,
                             spec.num_experts_per_tok, -1)
        top = top.softmax(-1)
        up = _weight(seed, p + "mlp.gate_up_w", (E, 2 * f, H), torch.bfloat16, case)
        down = _weight(seed, p + "mlp.down_w", (E, H, f), torch.bfloat16, case)
        out = torch.zeros_like(x)
        for e in range(E):
            t, j = (ex == e).nonzero(as_tuple=True)
            gu = y[t] @ up[e].double().T
            out.index_add_(0, t, ((torch.nn.functional.silu(gu[:, :f]) * gu[:, f:])
                                  @ down[e].double().T) * top[t, j, None])
        x = x + out
    if spec.num_experts:
        x = x[last]
    return _rms(x, W("final_norm", H), eps)


def _exact_hybrid(case, seed, spec, rows, ids, last):
    H, eps = spec.hidden_size, spec.rms_norm_eps
    f32 = torch.float32
    W = lambda name, *shape: _w64(case, seed, name, shape)
    F = lambda name, *shape: _w64(case, seed, name, shape, f32)
    silu, sig = torch.nn.functional.silu, torch.sigmoid
    starts, r = [], 0
    for _, n in rows:
        starts.append(r)
        r += n
    S, N = len(rows), max(n for _, n in rows)
    # [sequence, step] -> row, a spare row behind the last sequence's steps
    grid = torch.full((S, N), r)
    for i, (_, n) in enumerate(rows):
        grid[i, :n] = torch.arange(starts[i], starts[i] + n)
    grid = grid.cuda()
    pos = torch.cat([torch.arange(h, h + n) for h, n in rows]).cuda().double()

    def norm(x, name):
        d = x - x.mean(-1, keepdim=True)
        bias = name[:-2] + "_b" if name.endswith("_w") else name + "_b"
        return d * torch.rsqrt((d * d).mean(-1, keepdim=True) + eps) \
            * F(name, H) + F(bias, H)

    def scan(q, k, v, a, state):
        """S <- a S + k v^T; y = S^T q over every sequence's rows; q, k
        [rows, heads, state], v [rows, heads, vdim], a [rows, heads]."""
        pad = lambda t: torch.cat([t, torch.zeros_like(t[:1])])[grid]
        q, k, v, a = pad(q), pad(k), pad(v), pad(a)
        y = torch.empty(S, N, *v.shape[2:], dtype=torch.float64, device="cuda")
        for t in range(N):
            state = a[:, t, :, None, None] * state \
                + k[:, t, :, :, None] * v[:, t, :, None, :]
            y[:, t] = (state * q[:, t, :, :, None]).sum(2)
        out = torch.empty(r + 1, *v.shape[2:], dtype=torch.float64, device="cuda")
        out[grid.reshape(-1)] = y.reshape(S * N, *v.shape[2:])
        return out[:r]

    x = W("embed", spec.vocab_size, H)[ids] * (spec.embed_scale or 1.0)
    v_first = None
    cached = bool(rows[0][0])
    for i in range(LAYERS):
        ls, p = spec.layers[i], "layers.%d." % i
        m = ls.mixer
        y = norm(x, p + "norm1_w")
        if ls.mixer_type == "paged_attention":
            d, hq, hkv = m.qk_dim, m.heads, m.kv_heads
            qkv = (y @ W(p + "mixer.qkv_w", (hq + 2 * hkv) * d, H).T).view(-1, hq + 2 * hkv, d)
            q, k, v = qkv[:, :hq], qkv[:, hq:hq + hkv], qkv[:, hq + hkv:]
            q = _rms(q, F(p + "mixer.q_head_norm", d), eps)
            k = _rms(k, F(p + "mixer.k_head_norm", d), eps)
            coef, every = m.q_temp
            q = q * (1.0 + coef * torch.log(torch.floor((pos + 1) / every) + 1))[:, None, None]
            if v_first is None:
                v_first = v
            else:
                lam = F(p + "mixer.v_lam", 1)
                v = (1 - lam) * v + lam * v_first
            slopes = 2.0 ** (-8.0 * (torch.arange(hq, device="cuda").double() + 1) / hq)
            o = _over_sequences(q, k, v,
                                *_history(case, seed, i, rows, hkv, d), rows,
                                window=m.window, slopes=slopes)
            a = o.reshape(-1, hq * d) @ W(p + "mixer.o_w", H, hq * d).T
        else:
            nh, ns, vd = m.heads, m.state, m.vdim
            inner = nh * vd
            state = (_normal(seed, "s%d" % i, (S, nh, ns, vd)).double()
                     if cached else torch.zeros(S, nh, ns, vd, dtype=torch.float64, device="cuda"))
            if m.kind == "mamba2":
                gn = m.groups * ns
                C = inner + 2 * gn
                u = y @ W(p + "mixer.in_w", 2 * inner + 2 * gn + nh, H).T
                z, xbc, dt = u[:, :inner], u[:, inner:inner + C], u[:, inner + C:]
                old = (_normal(seed, "c%d" % i, (S, m.conv - 1, C)).to(torch.bfloat16).double()
                       if cached else torch.zeros(S, m.conv - 1, C, dtype=torch.float64, device="cuda"))
                cw, cb = F(p + "mixer.conv_w", C, m.conv), F(p + "mixer.conv_b", C)
                parts = []
                for s, (_, n) in enumerate(rows):
                    full = torch.cat([old[s], xbc[starts[s]:starts[s] + n]])
                    parts.append(cb + sum(full[j:j + n] * cw[:, j] for j in range(m.conv)))
                xbc = silu(torch.cat(parts))
                rep = nh // m.groups
                v = xbc[:, :inner].view(-1, nh, vd)
                k = xbc[:, inner:inner + gn].view(-1, m.groups, ns).repeat_interleave(rep, 1)
                q = xbc[:, inner + gn:].view(-1, m.groups, ns).repeat_interleave(rep, 1)
                dt = torch.nn.functional.softplus(dt + F(p + "mixer.dt_bias", nh))
                o = scan(q, k * dt[:, :, None], v,
                         torch.exp(-torch.exp(F(p + "mixer.a_log", nh)) * dt), state)
                o = (o + F(p + "mixer.skip", nh)[:, None] * v).reshape(-1, inner) * silu(z)
                o = _rms(o.view(-1, m.norm_groups, inner // m.norm_groups), 1.0, eps)
                o = o.reshape(-1, inner) * F(p + "mixer.norm", inner)
            else:
                u = y @ W(p + "mixer.qkvg_w", 2 * nh * ns + 2 * inner, H).T
                q, k, v = (silu(u[:, j * nh * ns:(j + 1) * nh * ns]).view(-1, nh, ns)
                           for j in range(3))
                a = torch.tensor(m.decay, dtype=torch.float64).to(f32).cuda().double()
                o = scan(q, k, v, a.expand(r, nh), state).reshape(-1, inner)
                o = _rms(o, F(p + "mixer.norm", inner), eps) * sig(u[:, 2 * nh * ns + inner:])
            a = o @ W(p + "mixer.o_w", H, inner).T
        x = x + a
        y = norm(x, p + "norm2_w")
        f = ls.mlp.ff
        gu = y @ W(p + "mlp.up_w", 2 * f, H).T
        x = x + (silu(gu[:, :f]) * gu[:, f:]) @ W(p + "mlp.down_w", H, f).T
    return norm(x[last], "final_norm")
