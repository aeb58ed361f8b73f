"""Performance cases of the candidate-group attention framework.

A case is one piece of the work a completion service does with this package,
through its public entry points and at the shapes of the package's own model
configurations (aios_amd.config.MODELS):

  decode         the attention of one decode step in every layer (q/k norm +
                 RoPE, KV append, shared-prefix decode), replayed from a
                 captured graph as the engine replays its steps
  prefill        the attention of a prefill or of a keystroke's extension of a
                 cached prefix; up to 64 new tokens from a captured graph (the
                 engine's rule), more of them eagerly
  layers         the projections of a decode step's layers with their norms
                 and activation, from a captured graph
  head           final norm and LM head of a decode step, from a captured graph
  pick           one sampled token per candidate from its logits, from a
                 captured graph
  mixer          the Block-AttnRes depth mixers of one forward, from a
                 captured graph (chunks of one length)
  model_decode   a whole decode step's forward, from a captured graph
  model_prefill  a whole prefill forward, eager (longer than the engine graphs)

``listed`` names the cases, ``draw`` gives more over the same ranges.
"""
from __future__ import annotations

import math
from dataclasses import replace

import torch
import torch.nn.functional as F

from aios_amd.attention import Mi355xAttentionBackend
from aios_amd.config import MODELS
from aios_amd.core import Batch, Context, Req, SamplingParams, reset_global_ctx, set_global_ctx
from aios_amd.kvcache import MHAKVCache
from aios_amd.layers import HipOps
from aios_amd.minimind_ime import DepthBank
from aios_amd.qwen3 import Qwen3ForCausalLM, init_weights
from aios_amd.sample import sample_step

DEV = "cuda"
GRAPHED_PREFILL = 64  # new tokens up to which a prefill is graph-replayed


# -- the cases ---------------------------------------------------------------

def listed():
    return [
        # The smallest attention step: 8 candidates on a short typed prefix
        # (the single-layer op test's shape, in all 14 layers of that model).
        {"name": "decode-short", "kind": "decode", "model": "minimind-0.1b", "layers": 14,
         "rows": 8, "prefix": 24, "suffix": 16},
        # Candidates over a long document: the long-context benchmark step.
        {"name": "decode-long", "kind": "decode", "model": "qwen3-4b", "layers": 36, "rows": 24,
         "prefix": 4096, "suffix": 64},
        # The longest contexts a service keeps, with many candidates.
        {"name": "decode-longest", "kind": "decode", "model": "qwen3-0.6b", "layers": 28,
         "rows": 48, "prefix": 16000, "suffix": 100},
        # A keystroke adds a few tokens to a long cached document.
        {"name": "extend-long", "kind": "prefill", "model": "qwen3-4b", "layers": 8, "new": 6,
         "cached": 4093},
        # A long document read for the first time: the prefill benchmark.
        {"name": "prefill-long", "kind": "prefill", "model": "qwen3-4b", "layers": 1,
         "new": 4096, "cached": 0},
        # The projections of a small model's decode step.
        {"name": "layers-small", "kind": "layers", "model": "minimind-0.1b", "layers": 14,
         "rows": 8},
        # The same for the largest model with the long-context group size.
        {"name": "layers-large", "kind": "layers", "model": "qwen3-4b", "layers": 4, "rows": 24},
        # The LM head of that step.
        {"name": "head-large", "kind": "head", "model": "qwen3-4b", "rows": 24},
        # Sampling with the service's default temperature, top-k and top-p.
        {"name": "pick-default", "kind": "pick", "vocab": 151936, "rows": 24,
         "temperature": 0.35, "top_k": 50, "top_p": 0.9},
        # Depth mixers of a prompt chunk in the 0.214B trunk (65 mixers).
        {"name": "mixer-chunk", "kind": "mixer", "hidden": 768, "blocks": 8, "per_block": 4,
         "tokens": 512},
        # One whole decode step of the deployed model.
        {"name": "model-decode", "kind": "model_decode", "model": "minimind-ime-0.1b",
         "layers": 14, "rows": 8, "prefix": 130, "suffix": 16},
        # One whole prefill of a pasted document.
        {"name": "model-prefill", "kind": "model_prefill", "model": "qwen3-0.6b", "layers": 28,
         "new": 2048},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "layers",
                       "layers", "head", "pick", "mixer", "model_decode", "model_prefill"])
    shapes = ["minimind-0.1b", "minimind-ime-0.1b", "qwen3-0.6b", "qwen3-4b"]
    model = rng.choice(shapes)
    cfg = MODELS[model]
    if kind == "decode":
        prefix = _log(rng, 16, 16384)
        kv = prefix * cfg.num_kv_heads * cfg.head_dim * 4
        return {"kind": kind, "model": model, "rows": _log(rng, 1, 64), "prefix": prefix,
                "suffix": rng.randint(0, 128),
                "layers": max(2, min(cfg.num_layers, (1 << 30) // kv))}
    if kind == "prefill":
        new = _log(rng, 1, 4096)
        cached = 0 if rng.random() < 0.3 else _log(rng, 8, 12000)
        return {"kind": kind, "model": model, "new": new, "cached": cached,
                "layers": rng.randint(4, 12) if new <= GRAPHED_PREFILL else 1}
    if kind == "layers":
        return {"kind": kind, "model": model, "rows": _log(rng, 1, 64), "layers": rng.randint(2, 6)}
    if kind == "head":
        return {"kind": kind, "model": model, "rows": _log(rng, 1, 64)}
    if kind == "pick":
        t, k, p = rng.choice([(0.35, 50, 0.9), (0.75, 96, 0.95), (0.95, 160, 0.95), (0.0, -1, 1.0)])
        return {"kind": kind, "vocab": rng.choice([6400, 16384, 151936]), "rows": _log(rng, 1, 64),
                "temperature": t, "top_k": k, "top_p": p}
    if kind == "mixer":
        return {"kind": kind, "hidden": 768, "blocks": 8, "per_block": rng.randint(1, 4),
                "tokens": _log(rng, 1, 2048)}
    if kind == "model_decode":
        return {"kind": kind, "model": model, "layers": rng.randint(2, 8), "rows": _log(rng, 1, 32),
                "prefix": _log(rng, 16, 4096), "suffix": rng.randint(0, 32)}
    return {"kind": kind, "model": model, "layers": rng.randint(2, 8),
            "new": rng.randint(GRAPHED_PREFILL + 1, 2048)}


# -- inputs ------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, shape, std=1.0, mean=0.0):
    x = torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)
    return (x * std + mean).to(torch.bfloat16)


def _config(case):
    cfg = MODELS[case["model"]]
    if cfg.residual_type != "standard":
        cfg = replace(cfg, residual_type="standard", attnres_num_blocks=0)
    return cfg.with_layers(case["layers"]) if "layers" in case else cfg


def _suffixes(case, seed):
    """Tokens each candidate has behind the prefix before this step, ragged."""
    g = torch.Generator().manual_seed(seed + 7)
    return torch.randint(0, case["suffix"] + 1, (case["rows"],), generator=g).tolist()


class _Pool:
    """A filled KV pool and page table: the prefix on scattered pages, each
    row's suffix on others, and the step's new tokens on the last ones, in a
    row, as the page allocator hands them out."""

    def __init__(self, cfg, cached, suffixes, new, seed):
        g = _gen(seed)
        old = cached + sum(suffixes)
        self.pages = old + new
        self.first_new = old
        self.kv = MHAKVCache(cfg.num_kv_heads, cfg.num_layers, cfg.head_dim, self.pages, 1,
                             torch.bfloat16, DEV)
        for i in range(cfg.num_layers):
            shape = self.kv.k_cache(i).shape
            self.kv.k_cache(i).copy_(_normal(g, shape))
            self.kv.v_cache(i).copy_(_normal(g, shape, 0.5))
        perm = torch.randperm(old, generator=torch.Generator().manual_seed(seed + 1))
        self.prefix = perm[:cached]
        self.suffix = torch.split(perm[cached:], suffixes) if suffixes else ()
        self.out_loc = torch.arange(old, old + new, dtype=torch.int32, device=DEV)

    def table(self, rows):
        width = max(len(r) for r in rows)
        t = torch.zeros((len(rows), width), dtype=torch.int32)
        for i, r in enumerate(rows):
            t[i, : len(r)] = r.to(torch.int32)
        return t.to(DEV)

    def written(self):
        """The pool rows the step writes, all layers: views of K and of V."""
        n, out = self.kv.num_layers, []
        for cache in (self.kv.k_cache, self.kv.v_cache):
            first = cache(0)
            layer = first.numel()
            out.append(first.as_strided((n, self.pages - self.first_new) + first.shape[1:],
                                        (layer,) + first.stride(),
                                        first.storage_offset()
                                        + self.first_new * first.stride(0)))
        return out


def _decode_pool(case, cfg, seed):
    suffixes = _suffixes(case, seed)
    pool = _Pool(cfg, case["prefix"], suffixes, case["rows"], seed)
    rows = [torch.cat([pool.prefix, s, torch.tensor([pool.first_new + i])])
            for i, s in enumerate(pool.suffix)]
    return pool, rows


def _prefill_pool(case, cfg, seed):
    cached = case.get("cached", 0)
    pool = _Pool(cfg, cached, [], case["new"], seed)
    return pool, [torch.cat([pool.prefix, torch.arange(cached, cached + case["new"])])]


def _attention_inputs(case, cfg, seed):
    tokens = case["rows"] if case["kind"] == "decode" else case["new"]
    g = _gen(seed + 2)
    width = (cfg.num_qo_heads + 2 * cfg.num_kv_heads) * cfg.head_dim
    qkv = _normal(g, (cfg.num_layers, tokens, width))
    norms = [{"q_norm": _normal(g, (cfg.head_dim,), 0.1, 1.0),
              "k_norm": _normal(g, (cfg.head_dim,), 0.1, 1.0)} for _ in range(cfg.num_layers)]
    return qkv, norms


def _layer_inputs(case, cfg, seed):
    g = _gen(seed)
    w = init_weights(replace(cfg, vocab_size=16), seed + 1, DEV)["layers"]
    for lw in w:
        for n in ("input_norm", "post_norm"):
            lw[n] = _normal(g, (cfg.hidden_size,), 0.1, 1.0)
    shape = (case["rows"], cfg.hidden_size)
    return w, _normal(g, shape, 0.5), _normal(g, shape)


def _head_inputs(case, cfg, seed):
    g = _gen(seed)
    shape = (case["rows"], cfg.hidden_size)
    return (_normal(g, (cfg.vocab_size, cfg.hidden_size), 0.02), _normal(g, shape, 0.5),
            _normal(g, shape), _normal(g, (cfg.hidden_size,), 0.1, 1.0))


def _pick_inputs(case, seed):
    """Logits with a broad bulk and a few likely continuations a row."""
    g = _gen(seed)
    rows, vocab = case["rows"], case["vocab"]
    x = torch.randn((rows, vocab), generator=g, device=DEV) * 2.0
    top = torch.randint(0, vocab, (rows, 64), generator=g, device=DEV)
    x.scatter_add_(1, top, 4.0 + 8.0 * torch.rand((rows, 64), generator=g, device=DEV))
    u = torch.rand((rows, 4), generator=g, device=DEV)
    blocked = torch.tensor([2, 3], dtype=torch.int32, device=DEV)
    return x.to(torch.bfloat16), u, blocked


def _mixer_inputs(case, seed):
    g = _gen(seed)
    n, d, layers = case["tokens"], case["hidden"], case["blocks"] * case["per_block"]
    first = _normal(g, (n, d))
    deltas = [_normal(g, (n, d), 0.3) for _ in range(2 * layers)]
    wq = [torch.randn(d, generator=g, device=DEV) * 0.02 for _ in range(2 * layers + 1)]
    return first, deltas, wq


def _model_inputs(case, cfg, seed):
    w = init_weights(cfg, seed + 1, DEV)
    # embeddings of the size of what the layers add, as in a trained model
    w["embed"] = w["embed"] * 25
    n = case["rows"] if case["kind"] == "model_decode" else case["new"]
    ids = torch.randint(0, cfg.vocab_size, (n,), generator=_gen(seed + 3), device=DEV)
    return w, ids


# -- what a program keeps ------------------------------------------------------

def _capture(call):
    """The call's HIP graph and its outputs, warmed once as the engine does."""
    cur = torch.cuda.current_stream()
    stream = torch.cuda.Stream()
    stream.wait_stream(cur)
    with torch.cuda.stream(stream), torch.inference_mode():
        call()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream), torch.inference_mode():
        out = call()
    cur.wait_stream(stream)
    return graph, out


def _context(pool, table, backend):
    reset_global_ctx()
    ctx = Context(page_size=1)
    ctx.kv_cache = pool.kv
    ctx.attn_backend = backend
    ctx.page_table = table
    set_global_ctx(ctx)
    return ctx


def _attention_state(case, cfg, seed, weights=None, ids=None):
    """Model, batch and metadata of a decode step or a prefill."""
    decode = case["kind"] in ("decode", "model_decode")
    pool, rows = (_decode_pool if decode else _prefill_pool)(case, cfg, seed)
    table = pool.table(rows)
    backend = Mi355xAttentionBackend(cfg)
    longest = max(len(r) for r in rows)
    model = Qwen3ForCausalLM(cfg, weights, DEV, attn_backend=backend, max_positions=longest)
    ctx = _context(pool, table, backend)
    new = 1 if decode else case["new"]
    reqs = [Req(input_ids=torch.empty(len(r), dtype=torch.long), cached_len=len(r) - new,
                output_len=1, uid=i, table_idx=i, sampling_params=SamplingParams(max_tokens=1))
            for i, r in enumerate(rows)]
    batch = Batch(reqs=reqs, phase="decode" if decode else "prefill")
    batch.out_loc = pool.out_loc
    if ids is not None:
        batch.input_ids = ids
    if decode:
        batch.positions = torch.tensor([len(r) - 1 for r in rows], dtype=torch.int32, device=DEV)
        batch.shared_prefix_len = case["prefix"]
        batch.fused_append = True
    else:
        batch.positions = torch.arange(longest - new, longest, dtype=torch.int32, device=DEV)
    if not decode and new <= GRAPHED_PREFILL:
        # as the engine plans its graphed prefills: for the length rounded up to 64
        cap = -(-longest // 64) * 64
        wide = F.pad(table, (0, cap - longest))
        md = backend.prepare_static_prefill(new, cap, wide)
        md.refresh(torch.full((1,), longest, dtype=torch.int32, device=DEV))
        batch.attn_metadata = md
    else:
        backend.prepare_metadata(batch)
    return {"model": model, "batch": batch, "pool": pool, "ctx": ctx}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        cfg = _config(case)
        qkv, norms = _attention_inputs(case, cfg, seed)
        s = _attention_state(case, cfg, seed, {"layers": norms})

        def attention():
            return [s["model"].attention_core(i, qkv[i], s["batch"].positions, s["pool"].kv,
                                              s["batch"]) for i in range(cfg.num_layers)]

        s["call"] = lambda: attention() + s["pool"].written()
        graphed = kind == "decode" or case["new"] <= GRAPHED_PREFILL
    elif kind == "layers":
        cfg = _config(case)
        weights, h0, r0 = _layer_inputs(case, cfg, seed)
        ops, eps, q = HipOps(), cfg.rms_norm_eps, cfg.num_qo_heads * cfg.head_dim

        def layers():
            h, res, out = h0, r0, []
            for lw in weights:
                qkv, res = ops.add_rmsnorm_linear(h, res, lw["input_norm"], eps, lw["qkv"])
                x = ops.linear(qkv[:, :q], lw["o"])  # (the q part stands for the attention)
                act, res = ops.add_rmsnorm_linear(x, res, lw["post_norm"], eps, lw["gate_up"],
                                                  silu=True)
                h = ops.linear(act, lw["down"])
                out += [qkv, h, res]
            return out

        s, graphed = {"call": layers}, True
    elif kind == "head":
        cfg = _config(case)
        w, h, res, norm = _head_inputs(case, cfg, seed)
        ops = HipOps()
        s = {"call": lambda: ops.add_rmsnorm_linear(h, res, norm, cfg.rms_norm_eps, w)}
        graphed = True
    elif kind == "pick":
        logits, u, blocked = _pick_inputs(case, seed)
        params = SamplingParams(temperature=case["temperature"], top_k=case["top_k"],
                                top_p=case["top_p"])
        step = torch.ones(1, dtype=torch.int64, device=DEV)
        s = {"call": lambda: sample_step(logits, params, u, step, blocked, 2)}
        graphed = True
    elif kind == "mixer":
        first, deltas, wq = _mixer_inputs(case, seed)
        bank = torch.empty((case["blocks"] + 1,) + first.shape, dtype=first.dtype, device=DEV)
        bank[0] = first
        part = torch.empty_like(first)
        ops = HipOps()

        def mixers():
            depth, out = DepthBank(bank, part, ops, 1e-5), []
            for i, delta in enumerate(deltas):
                out.append(depth.mix(wq[i]))
                depth.add(delta, closes_block=(i + 1) % (2 * case["per_block"]) == 0)
            out.append(depth.mix(wq[-1]))
            return out[-60:] + [bank]  # (the first mixes are copies or two-source sums)

        s, graphed = {"call": mixers}, True
    else:
        cfg = _config(case)
        weights, ids = _model_inputs(case, cfg, seed)
        s = _attention_state(case, cfg, seed, weights, ids)

        def forward():
            reset_global_ctx()
            set_global_ctx(s["ctx"])
            with s["ctx"].forward_batch(s["batch"]):
                logits = s["model"].forward()
            return [logits] + s["pool"].written()

        s["call"] = forward
        graphed = kind == "model_decode"
    if graphed:
        s["graph"], s["out"] = _capture(s["call"])
    return s


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    with torch.inference_mode():
        return state["call"]()


# -- what a pass cannot do without ---------------------------------------------

def _attention_work(cfg, new, cached_rows, shared):
    """One layer: ``cached_rows`` = KV positions each request has behind the
    shared ones, ``new`` = tokens each adds."""
    hq, hkv, d = cfg.num_qo_heads, cfg.num_kv_heads, cfg.head_dim
    tokens = new * len(cached_rows)
    old = shared + sum(cached_rows)
    io = tokens * (hq + 2 * hkv) * d * 2 + tokens * hq * d * 2 + tokens * 2 * hkv * d * 2
    pairs = sum(new * (shared + c) + new * (new + 1) // 2 for c in cached_rows)
    return old * 2 * hkv * d * 2 + io + 4 * (old + tokens), 4 * hq * d * pairs


def _layer_params(cfg):
    q, kv = cfg.num_qo_heads * cfg.head_dim, cfg.num_kv_heads * cfg.head_dim
    return cfg.hidden_size * (2 * q + 2 * kv + 3 * cfg.intermediate_size)


def work(case):
    kind = case["kind"]
    if kind == "pick":
        n = case["rows"] * case["vocab"]
        return {"bytes": 2 * n + case["rows"] * 16, "flops": 2 * n}
    if kind == "mixer":
        # every mix reads the sources there are and its delta, and writes the
        # partial and the mix
        n, mixes, sources = case["tokens"] * case["hidden"], 2 * case["blocks"] * case["per_block"], 0
        for i in range(mixes + 1):
            sources += 1 + (i - 1) // (2 * case["per_block"]) + (2 if i else 0) if i else 1
        return {"bytes": 2 * n * (sources + 2 * mixes + 1), "flops": 6 * n * sources}
    cfg = _config(case)
    h, vocab = cfg.hidden_size, cfg.vocab_size
    if kind == "head":
        rows = case["rows"]
        return {"bytes": 2 * (vocab * h + rows * (3 * h + vocab)), "flops": 2 * rows * vocab * h}
    if kind == "layers":
        rows = case["rows"]
        params = _layer_params(cfg) * cfg.num_layers
        return {"bytes": 2 * params + 8 * rows * h * cfg.num_layers, "flops": 2 * rows * params}
    if kind in ("decode", "model_decode"):
        mid = [case["suffix"] // 2] * case["rows"]
        b, f = _attention_work(cfg, 1, mid, case["prefix"])
        tokens, out = case["rows"], case["rows"]
    else:
        b, f = _attention_work(cfg, case["new"], [case.get("cached", 0)], 0)
        tokens, out = case["new"], 1
    b, f = b * cfg.num_layers, f * cfg.num_layers
    if kind.startswith("model"):
        params = _layer_params(cfg) * cfg.num_layers
        b += 2 * (params + vocab * h + out * vocab)
        f += 2 * (tokens * params + out * vocab * h)
    return {"bytes": b, "flops": f}


def tolerance(case):
    kind = case["kind"]
    if kind == "pick":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.0}
    # bf16 results of fp32 sums (half a unit is 2e-3 of a value), about four
    # times what sums in another order and other split lengths show: attention
    # 0.004, one projection or mixer 0.002 to 0.004, a chain of layers 0.01
    # (there a changed rounding goes through every later projection).
    if kind in ("layers", "model_decode", "model_prefill"):
        return {"rel": 0.03, "max": 0.2}
    return {"rel": 0.015, "max": 0.1}


# -- the same in 64 bits ---------------------------------------------------------

def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, pos, base):
    """x [T, H, D] at positions pos [T]."""
    d = x.shape[-1]
    inv = base ** (-torch.arange(0, d, 2, dtype=torch.float64, device=x.device) / d)
    a = (pos.double()[:, None] * inv).repeat(1, 2)[:, None, :]
    turned = torch.cat([-x[..., d // 2:], x[..., : d // 2]], -1)
    return x * a.cos() + turned * a.sin()


def _exact_decode(q, k, v, kc, vc, prefix, suffixes):
    """One layer's decode: q [N, Hq, D], new k, v [N, Hkv, D], caches
    [pages, Hkv, D] in bf16, prefix and suffixes lists of page ids."""
    n, hq, d = q.shape
    hkv = k.shape[1]
    out = torch.empty((n, hq, d), dtype=torch.float64, device=q.device)
    widest = max((len(s) for s in suffixes), default=0)
    ids = torch.zeros((n, widest), dtype=torch.long)
    live = torch.zeros((n, widest), dtype=torch.bool)
    for i, s in enumerate(suffixes):
        ids[i, : len(s)] = s
        live[i, : len(s)] = True
    ids, live, prefix = ids.to(q.device), live.to(q.device), prefix.to(q.device)
    for h in range(hkv):
        g = hq // hkv
        qh = q[:, h * g:(h + 1) * g] * d ** -0.5
        kp, vp = kc[prefix, h].double(), vc[prefix, h].double()
        ks, vs = kc[ids, h].double(), vc[ids, h].double()
        s1 = (qh.reshape(-1, d) @ kp.t()).view(n, g, -1)
        s2 = torch.matmul(qh, ks.transpose(1, 2)).masked_fill(~live[:, None, :], -math.inf)
        s3 = (qh * k[:, h, None]).sum(-1, keepdim=True)
        p = torch.cat([s1, s2, s3], -1).softmax(-1)
        m = len(prefix)
        o = (p[..., :m].reshape(n * g, m) @ vp).view(n, g, d)
        o = o + torch.matmul(p[..., m:m + widest], vs) + p[..., -1:] * v[:, h, None]
        out[:, h * g:(h + 1) * g] = o
    return out


def _exact_prefill(q, k, v, kc, vc, prefix):
    """One layer's causal prefill of T tokens behind the cached ones."""
    t, hq, d = q.shape
    hkv = k.shape[1]
    prefix = prefix.to(q.device)
    c, g = len(prefix), hq // hkv
    late = torch.ones((t, c + t), dtype=torch.bool, device=q.device).triu(c + 1)
    out = torch.empty((t, hq, d), dtype=torch.float64, device=q.device)
    for h in range(hkv):
        kh = torch.cat([kc[prefix, h].double(), k[:, h]])
        vh = torch.cat([vc[prefix, h].double(), v[:, h]])
        for j in range(h * g, (h + 1) * g):
            s = (q[:, j] * d ** -0.5) @ kh.t()
            out[:, j] = s.masked_fill_(late, -math.inf).softmax(-1) @ vh
    return out


def _exact_attention(cfg, i, qkv, pos, q_norm, k_norm, pool, decode):
    """(attention output [T, Hq * D], new K, new V) of layer i from its
    projections qkv [T, (Hq + 2 Hkv) * D] in 64 bits."""
    hq, hkv, d = cfg.num_qo_heads, cfg.num_kv_heads, cfg.head_dim
    t = qkv.shape[0]
    q, k, v = qkv.split([hq * d, hkv * d, hkv * d], -1)
    q = _rope(_rms(q.view(t, hq, d), q_norm, cfg.rms_norm_eps), pos, cfg.rope_theta)
    k = _rope(_rms(k.view(t, hkv, d), k_norm, cfg.rms_norm_eps), pos, cfg.rope_theta)
    v = v.view(t, hkv, d)
    kc = pool.kv.k_cache(i).view(-1, hkv, d)
    vc = pool.kv.v_cache(i).view(-1, hkv, d)
    o = (_exact_decode(q, k, v, kc, vc, pool.prefix, pool.suffix) if decode
         else _exact_prefill(q, k, v, kc, vc, pool.prefix))
    return o.reshape(t, -1), k, v


def _exact_sample(case, seed):
    logits, u, blocked = _pick_inputs(case, seed)
    x = logits.double()
    raw = x.log_softmax(-1)
    y = x.clone()
    y[:, blocked.long()] = -math.inf
    if case["temperature"] <= 0.0:
        tok = y.argmax(-1)  # (ties: checked against the first below)
        tok = (y == y.gather(1, tok[:, None])).double().argmax(-1)
    else:
        # descending, lower id first among equals
        val, order = (y / case["temperature"]).sort(dim=-1, descending=True, stable=True)
        val, order = val[:, : case["top_k"]], order[:, : case["top_k"]]
        p = val.softmax(-1)
        before = p.cumsum(-1) - p
        cut = before > case["top_p"]
        cut[:, 0] = False
        p = p.masked_fill(cut, 0.0)
        p = p / p.sum(-1, keepdim=True)
        at = (p.cumsum(-1) < u[:, 1:2].double()).sum(-1).clamp(max=case["top_k"] - 1)
        tok = order.gather(1, at[:, None])[:, 0]
    return tok, raw.gather(1, tok[:, None])[:, 0]


def _exact_mixers(case, seed):
    first, deltas, wq = _mixer_inputs(case, seed)
    bank, partial, out = [first.double()], None, []

    def mix(w):
        x = torch.stack(bank + ([partial] if partial is not None else []))
        score = (x * w.double()).sum(-1) * torch.rsqrt((x * x).mean(-1) + 1e-5)
        return (score.softmax(0)[..., None] * x).sum(0)

    for i, delta in enumerate(deltas):
        out.append(mix(wq[i]))
        partial = delta.double() if partial is None else partial + delta.double()
        if (i + 1) % (2 * case["per_block"]) == 0:
            bank.append(partial)
            partial = None
    out.append(mix(wq[-1]))
    return out[-60:] + [torch.stack(bank)]


@torch.inference_mode()
def exact(case, seed):
    kind = case["kind"]
    if kind == "pick":
        return _exact_sample(case, seed)
    if kind == "mixer":
        return _exact_mixers(case, seed)
    cfg = _config(case)
    eps = cfg.rms_norm_eps
    if kind == "head":
        w, h, res, norm = _head_inputs(case, cfg, seed)
        r = h.double() + res.double()
        x = _rms(r, norm, eps)
        return torch.cat([x @ c.double().t() for c in w.split(16384)], -1), r
    if kind == "layers":
        weights, h, res = _layer_inputs(case, cfg, seed)
        h, res, out, q = h.double(), res.double(), [], cfg.num_qo_heads * cfg.head_dim
        for lw in weights:
            res = res + h
            qkv = _rms(res, lw["input_norm"], eps) @ lw["qkv"].double().t()
            h = qkv[:, :q] @ lw["o"].double().t()
            attn = res + h
            gate, up = (_rms(attn, lw["post_norm"], eps)
                        @ lw["gate_up"].double().t()).chunk(2, -1)
            res = attn
            h = (F.silu(gate) * up) @ lw["down"].double().t()
            out += [qkv, h, res]
        return out
    decode = kind in ("decode", "model_decode")
    pool, rows = (_decode_pool if decode else _prefill_pool)(case, cfg, seed)
    new = 1 if decode else case["new"]
    pos = (torch.tensor([len(r) - 1 for r in rows], device=DEV) if decode
           else torch.arange(len(rows[0]) - new, len(rows[0]), device=DEV))
    ks, vs = [], []
    if kind in ("decode", "prefill"):
        qkv, norms = _attention_inputs(case, cfg, seed)
        out = []
        for i, n in enumerate(norms):
            o, k, v = _exact_attention(cfg, i, qkv[i].double(), pos, n["q_norm"], n["k_norm"], pool,
                                       decode)
            out.append(o)
            ks.append(k)
            vs.append(v)
        out = [o.view(-1, cfg.num_qo_heads * cfg.head_dim) for o in out]
        return out + [torch.stack(ks)[:, :, None], torch.stack(vs)[:, :, None]]
    w, ids = _model_inputs(case, cfg, seed)
    res = w["embed"][ids].double()
    for i, lw in enumerate(w["layers"]):
        qkv = _rms(res, lw["input_norm"], eps) @ lw["qkv"].double().t()
        o, k, v = _exact_attention(cfg, i, qkv, pos, lw["q_norm"], lw["k_norm"], pool, decode)
        ks.append(k)
        vs.append(v)
        res = res + o @ lw["o"].double().t()
        gate, up = (_rms(res, lw["post_norm"], eps) @ lw["gate_up"].double().t()).chunk(2, -1)
        res = res + (F.silu(gate) * up) @ lw["down"].double().t()
    x = _rms(res if decode else res[-1:], w["final_norm"], eps)
    logits = torch.cat([x @ c.double().t() for c in w["embed"].split(16384)], -1)
    return [logits, torch.stack(ks)[:, :, None], torch.stack(vs)[:, :, None]]
