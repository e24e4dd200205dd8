"""Performance cases: the work a user of this library has it do, through its public entry points.

Every case is one Llama-3.1-8B call of the serving path in bf16 (the library's storage type), at
the model's own shapes:

  decode_step    ie_decode_step: one token of one sequence through the whole model (chat decoding)
  decode_layer   ie_decoder_layer_decode: one decoder layer of it, long contexts included
  batched_layer  ie_decoder_layer_batched: one layer of a batched step, sequences of mixed lengths
  batched_paged  ie_decode_step_batched_paged: a whole batched step over long paged contexts
  prefill_layer  ie_decoder_layer_prefill: one layer of a prompt, from a short question to a document
  chunk_attn     ie_attn_prefill_core_paged: a prompt chunk's attention over the pages before it
  head           ie_final_norm_lm_head: final norm and vocabulary product of one row or a batch
  sample         ie_sample_top_p: temperature / nucleus sampling of one row or a batch

listed() fixes twelve of them; draw() gives others of the same ranges.
"""
import ctypes as C
import functools
import random

import torch

from infengine_amd import ModelWeightsStruct, check, lib
from infengine_amd.engine import Context, device_view, kv_cache_size, ptr, workspace_size

H, F, V, LAYERS = 4096, 14336, 128256, 32
QH, KVH, D = 32, 8, 128
MAX_CTX, MAX_LONG, PAGE = 8192, 131072, 64
LAYER = 5  # the layer that single-layer cases run
LAYER_PARAMS = 2 * H * H + 2 * 1024 * H + 3 * F * H
STD = 0.02          # weights, as the library's random init
OUT_STD = STD / 8   # whole models: O and down projections scaled by 1 / sqrt(2 layers), as trained
                    # models start, so that the residual stream is more than the last layers
KV_STD = 1.28       # keys and values of such a model: sqrt(4096) * 0.02


# ------------------------------------------------------------------------------- cases
def listed():
    return [
        # one token of a chat, 600 tokens in: the latency a single user sees
        {"name": "decode_step_600", "kind": "decode_step", "ctx": 600},
        # one layer late in a long conversation, near the end of the cache
        {"name": "decode_layer_7000", "kind": "decode_layer", "ctx": 7000},
        # a full batch of chats of mixed lengths, one layer of a step
        {"name": "batched_layer_16x1800", "kind": "batched_layer", "batch": 16, "ctx": 1800},
        # six long documents being answered at once, over the page pool
        {"name": "batched_paged_6x20000", "kind": "batched_paged", "batch": 6, "ctx": 20000},
        # a one-sentence question
        {"name": "prefill_layer_48", "kind": "prefill_layer", "rows": 48},
        # a paragraph, an odd number of tokens
        {"name": "prefill_layer_291", "kind": "prefill_layer", "rows": 291},
        # a page of text
        {"name": "prefill_layer_777", "kind": "prefill_layer", "rows": 777},
        # the benchmark's long prompt
        {"name": "prefill_layer_2048", "kind": "prefill_layer", "rows": 2048},
        # a document that nearly fills the reference-layout cache
        {"name": "prefill_layer_6000", "kind": "prefill_layer", "rows": 6000},
        # the next turn of a long conversation: a short chunk over 30000 cached positions
        {"name": "chunk_attn_200_at_30000", "kind": "chunk_attn", "rows": 200, "start": 30000},
        # the head of a half-full batch
        {"name": "head_8", "kind": "head", "rows": 8},
        # sampling for a full batch
        {"name": "sample_16", "kind": "sample", "rows": 16, "temperature": 0.7, "top_p": 0.9},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["decode_step", "decode_layer", "batched_layer", "batched_paged",
                       "prefill_layer", "prefill_layer", "prefill_layer", "chunk_attn",
                       "chunk_attn", "head", "sample"])
    if kind in ("decode_step", "decode_layer"):
        return {"kind": kind, "ctx": _log(rng, 2, MAX_CTX - 1)}
    if kind == "batched_layer":
        return {"kind": kind, "batch": rng.randint(2, 16), "ctx": _log(rng, 64, 8000)}
    if kind == "batched_paged":
        return {"kind": kind, "batch": rng.randint(2, 6), "ctx": _log(rng, 1000, 20000)}
    if kind == "prefill_layer":
        return {"kind": kind, "rows": _log(rng, 17, 6000)}
    if kind == "chunk_attn":
        return {"kind": kind, "rows": _log(rng, 16, 1024), "start": _log(rng, 1000, 60000)}
    if kind == "head":
        return {"kind": kind, "rows": rng.randint(1, 16)}
    return {"kind": "sample", "rows": rng.randint(1, 16),
            "temperature": round(rng.uniform(0.4, 1.2), 2), "top_p": round(rng.uniform(0.5, 0.98), 2)}


def _lens(case):
    """The batch's context lengths: between an eighth of the longest and the longest, which is
    ctx."""
    r = random.Random(case["batch"] * 1000003 + case["ctx"])
    lens = [r.randint(max(1, case["ctx"] // 8), case["ctx"]) for _ in range(case["batch"])]
    lens[r.randrange(case["batch"])] = case["ctx"]
    return lens


def work(case):
    k = case["kind"]
    if k == "decode_step":
        params, c = LAYERS * LAYER_PARAMS + V * H, case["ctx"]
        return {"bytes": 2 * params + LAYERS * 4096 * c + 4 * V,
                "flops": 2 * params + LAYERS * 4 * QH * D * c}
    if k == "decode_layer":
        c = case["ctx"]
        return {"bytes": 2 * LAYER_PARAMS + 4096 * c, "flops": 2 * LAYER_PARAMS + 4 * QH * D * c}
    if k == "batched_layer":
        n = sum(_lens(case))
        return {"bytes": 2 * LAYER_PARAMS + 4096 * n,
                "flops": 2 * case["batch"] * LAYER_PARAMS + 4 * QH * D * n}
    if k == "batched_paged":
        params, n = LAYERS * LAYER_PARAMS + V * H, sum(_lens(case))
        return {"bytes": 2 * params + LAYERS * 4096 * n + 4 * V * case["batch"],
                "flops": 2 * case["batch"] * params + LAYERS * 4 * QH * D * n}
    if k == "prefill_layer":
        s = case["rows"]
        return {"bytes": 2 * LAYER_PARAMS + 4 * s * H + 4096 * s,
                "flops": 2 * s * LAYER_PARAMS + 4 * QH * D * s * (s + 1) // 2}
    if k == "chunk_attn":
        s, p = case["rows"], case["start"]
        return {"bytes": 4 * s * H + 4096 * (p + s),
                "flops": 4 * QH * D * (s * p + s * (s + 1) // 2)}
    if k == "head":
        r = case["rows"]
        return {"bytes": 2 * V * H + r * (2 * H + 4 * V), "flops": 2 * r * V * H}
    # the logits are read once; a few operations each
    return {"bytes": case["rows"] * V * 4, "flops": case["rows"] * V * 10}


def tolerance(case):
    k = case["kind"]
    if k == "sample":
        return "exact"              # token ids
    if k in ("decode_step", "batched_paged"):
        # 32 layers of bf16 residuals: the batched step's kernels against the single step's on
        # the same token differ by 2.2e-2 (largest 0.1)
        return {"rel": 3e-2, "max": 0.4}
    if k in ("chunk_attn", "head"):
        return {"rel": 9e-3}        # 2.2e-3 from 64 bits (bf16 probabilities, bf16 norm output)
    return {"rel": 1.3e-2}          # one layer: 3.3e-3 between two K splits of its products


# ------------------------------------------------------------------------------- inputs
@functools.cache
def _stream():
    return torch.cuda.Stream(0)


def _context():
    """A context per state (it keeps the captured graphs of the state's buffers), all on one
    stream, which is torch's current stream too."""
    return Context(0, stream=_stream())


@functools.cache
def _rope():
    cos, sin = C.c_void_p(), C.c_void_p()
    check(lib.ie_init_rope_buffer(C.byref(cos), C.byref(sin)))
    return tuple(device_view(p.value, (MAX_LONG, D // 2), torch.float32) for p in (cos, sin))


class _Gen:
    """Seeded normal tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def bf16(self, *shape, mean=0.0, std=1.0):
        return torch.empty(*shape, dtype=torch.bfloat16, device="cuda").normal_(
            mean, std, generator=self.g)

    def ids(self, n):
        return torch.randint(0, V, (n,), dtype=torch.int32, device="cuda", generator=self.g)


LAYER_SHAPES = {"input_layernorm": (H,), "post_attention_layernorm": (H,), "w_q": (H, H),
                "w_k": (KVH * D, H), "w_v": (KVH * D, H), "w_o": (H, H), "w_gate": (F, H),
                "w_up": (F, H), "w_down": (H, F)}


def _layer_weights(g, out_std=STD):
    return {n: g.bf16(*s, mean=1.0, std=0.02) if len(s) == 1
            else g.bf16(*s, std=out_std if n in ("w_o", "w_down") else STD)
            for n, s in LAYER_SHAPES.items()}


def _model(g, whole):
    """(the weights' tensors, the library's struct over them).  A single-layer case points all
    32 layers at one layer's tensors; the head and the embedding are not read there."""
    w = {"final_norm": g.bf16(H, mean=1.0, std=0.02)}
    if whole:
        w["emb_lookup"], w["lm_head"] = g.bf16(V, H, std=1.0), g.bf16(V, H, std=STD)
        w["layers"] = [_layer_weights(g, OUT_STD) for _ in range(LAYERS)]
    else:
        w["emb_lookup"] = w["lm_head"] = g.bf16(1, H, std=STD)
        w["layers"] = [_layer_weights(g)] * LAYERS
    s = ModelWeightsStruct()
    for n in ("emb_lookup", "lm_head", "final_norm"):
        setattr(s, n, w[n].data_ptr())
    for l, t in enumerate(w["layers"]):
        for n, v in t.items():
            part = s.layers[l]
            if n in ("w_q", "w_k", "w_v", "w_o"):
                part = part.transformer
            elif n in ("w_gate", "w_up", "w_down"):
                part = part.ffn_block
            setattr(part, n, v.data_ptr())
    cos, sin = _rope()
    s.rope.cos, s.rope.sin, s.rope_rows = cos.data_ptr(), sin.data_ptr(), MAX_LONG
    return w, s


def _pages(g, lens, layers):
    """A shuffled page pool for sequences of these lengths, [pages][32][2][8][64][128], the given
    layers filled, and the block tables [batch][stride]."""
    need = [-(-n // PAGE) for n in lens]
    pool = torch.empty(sum(need), LAYERS, 2, KVH, PAGE, D, dtype=torch.bfloat16, device="cuda")
    for l in layers:
        pool[:, l] = g.bf16(sum(need), 2, KVH, PAGE, D, std=KV_STD)
    order = torch.randperm(sum(need), device="cuda", generator=g.g).to(torch.int32)
    table = torch.zeros(len(lens), max(need), dtype=torch.int32, device="cuda")
    at = 0
    for b, n in enumerate(need):
        table[b, :n] = order[at:at + n]
        at += n
    return pool, table


def prepare(case, seed):
    k, ctx = case["kind"], _context()
    g = _Gen(seed)
    s = {"kind": k, "ctx": ctx, "case": case}
    bf = functools.partial(torch.empty, dtype=torch.bfloat16, device="cuda")
    if k == "decode_step":
        n = case["ctx"]
        s["w"], s["W"] = _model(g, True)
        s["tokens"] = torch.zeros(MAX_CTX, dtype=torch.int32, device="cuda")
        s["tokens"][:n] = g.ids(n)
        s["kv"] = bf(LAYERS, 2, KVH, MAX_CTX, D)
        for l in range(LAYERS):
            s["kv"][l, :, :, :n - 1] = g.bf16(2, KVH, n - 1, D, std=KV_STD)
        s["data"], s["aux"], s["attn"] = bf(1, H), bf(1, H), bf(1, H)
        s["logits"] = torch.empty(V, dtype=torch.float32, device="cuda")
        s["token"] = torch.empty(1, dtype=torch.int32, device="cuda")
        s["ws"] = torch.empty(workspace_size(n), dtype=torch.uint8, device="cuda")
        s["new_kv"] = s["kv"][:, :, :, n - 1]
    elif k == "decode_layer":
        n = case["ctx"]
        s["w"], s["W"] = _model(g, False)
        s["kv"] = bf(LAYERS, 2, KVH, MAX_CTX, D)
        s["kv"][LAYER, :, :, :n - 1] = g.bf16(2, KVH, n - 1, D, std=KV_STD)
        s["x"], s["attn"] = g.bf16(1, H), bf(1, H)
        s["ws"] = torch.empty(workspace_size(n), dtype=torch.uint8, device="cuda")
        s["new_kv"] = s["kv"][LAYER, :, :, n - 1]
    elif k == "batched_layer":
        lens, b = _lens(case), case["batch"]
        s["w"], s["W"] = _model(g, False)
        s["kv"] = torch.empty(b, kv_cache_size() // 2, dtype=torch.bfloat16, device="cuda")
        planes = s["kv"].view(b, LAYERS, 2, KVH, MAX_CTX, D)[:, LAYER]
        for i, n in enumerate(lens):
            planes[i, :, :, :n - 1] = g.bf16(2, KVH, n - 1, D, std=KV_STD)
        s["planes"] = planes
        s["x"], s["attn"] = g.bf16(b, H), bf(b, H)
        s["lens"] = (C.c_int * b)(*lens)
        s["ws"] = torch.empty(lib.ie_batch_workspace_size(b), dtype=torch.uint8, device="cuda")
    elif k == "batched_paged":
        lens, b = _lens(case), case["batch"]
        s["w"], s["W"] = _model(g, True)
        s["pool"], s["table"] = _pages(g, lens, range(LAYERS))
        s["tokens"] = g.ids(b * case["ctx"]).view(b, case["ctx"])
        s["data"], s["attn"] = bf(b, H), bf(b, H)
        s["logits"] = torch.empty(b, V, dtype=torch.float32, device="cuda")
        s["token"] = torch.empty(b, dtype=torch.int32, device="cuda")
        s["out"], s["lens"] = (C.c_int * b)(), (C.c_int * b)(*lens)
        s["ws"] = torch.empty(lib.ie_batch_workspace_size(b), dtype=torch.uint8, device="cuda")
    elif k == "prefill_layer":
        n = case["rows"]
        s["w"], s["W"] = _model(g, False)
        s["kv"] = bf(LAYERS, 2, KVH, MAX_CTX, D)
        s["x"], s["aux"], s["attn"] = g.bf16(n, H), bf(n, H), bf(n, H)
        s["ws"] = torch.empty(workspace_size(n), dtype=torch.uint8, device="cuda")
        s["new_kv"] = s["kv"][LAYER, :, :, :n]
    elif k == "chunk_attn":
        n = case["start"] + case["rows"]
        s["pool"], s["table"] = _pages(g, [n], [LAYER])
        s["q"], s["out"] = g.bf16(case["rows"], QH, D, std=KV_STD), bf(case["rows"], H)
    elif k == "head":
        s["x"], s["norm"] = g.bf16(case["rows"], H), g.bf16(H, mean=1.0, std=0.02)
        s["lm_head"] = g.bf16(V, H, std=STD)
        s["logits"] = torch.empty(case["rows"], V, dtype=torch.float32, device="cuda")
    else:
        r = case["rows"]
        s["logits"] = torch.empty(r, V, device="cuda").normal_(0.0, 2.0, generator=g.g)
        s["seed"] = seed
        s["token"] = torch.empty(r, dtype=torch.int32, device="cuda")
        s["ws"] = torch.empty(lib.ie_top_p_workspace_size(r, V), dtype=torch.uint8, device="cuda")
    return s


# ------------------------------------------------------------------------------- one pass
def run(s):
    k, c, h = s["kind"], s["case"], s["ctx"].handle
    if k == "decode_step":
        check(lib.ie_decode_step(h, C.byref(s["W"]), c["ctx"], ptr(s["tokens"]), ptr(s["data"]),
                                 ptr(s["aux"]), ptr(s["attn"]), ptr(s["logits"]), ptr(s["token"]),
                                 ptr(s["ws"]), ptr(s["kv"])))
        return {"logits": s["logits"], "new_kv": s["new_kv"]}
    if k == "decode_layer":
        check(lib.ie_decoder_layer_decode(h, C.byref(s["W"]), LAYER, c["ctx"], ptr(s["x"]),
                                          ptr(s["attn"]), ptr(s["ws"]), ptr(s["kv"])))
        return {"x": s["x"], "new_kv": s["new_kv"]}
    if k == "batched_layer":
        check(lib.ie_decoder_layer_batched(h, C.byref(s["W"]), LAYER, c["batch"], s["lens"],
                                           ptr(s["x"]), ptr(s["attn"]), ptr(s["ws"]),
                                           ptr(s["kv"])))
        return {"x": s["x"], "new_kv": [s["planes"][i, :, :, n - 1] for i, n in enumerate(s["lens"])]}
    if k == "batched_paged":
        check(lib.ie_decode_step_batched_paged(
            h, C.byref(s["W"]), c["batch"], s["lens"], ptr(s["tokens"]), c["ctx"], ptr(s["data"]),
            ptr(s["attn"]), ptr(s["logits"]), ptr(s["token"]), s["out"], ptr(s["ws"]),
            ptr(s["pool"]), s["pool"].shape[0], ptr(s["table"]), s["table"].shape[1]))
        return {"logits": s["logits"]}
    if k == "prefill_layer":
        check(lib.ie_decoder_layer_prefill(h, C.byref(s["W"]), LAYER, c["rows"], ptr(s["x"]),
                                           ptr(s["aux"]), ptr(s["attn"]), ptr(s["ws"]),
                                           ptr(s["kv"])))
        return {"x": s["x"], "new_kv": s["new_kv"]}
    if k == "chunk_attn":
        check(lib.ie_attn_prefill_core_paged(h, c["rows"], c["start"], ptr(s["q"]),
                                             ptr(s["pool"]), s["pool"].shape[0], ptr(s["table"]),
                                             LAYER, ptr(s["out"])))
        return s["out"]
    if k == "head":
        check(lib.ie_final_norm_lm_head(h, c["rows"], ptr(s["x"]), ptr(s["norm"]),
                                        ptr(s["lm_head"]), ptr(s["logits"])))
        return s["logits"]
    check(lib.ie_sample_top_p(h, c["rows"], V, ptr(s["logits"]), c["temperature"], c["top_p"],
                              s["seed"], 1, ptr(s["token"]), ptr(s["ws"])))
    return s["token"]


# ------------------------------------------------------------------------------- 64 bits
def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * w.double()


def _mul64(x, w):
    """x . w^T in float64, the weight converted in slices."""
    return torch.cat([x @ p.double().t() for p in w.split(16384)], dim=-1)


def _rot64(x, pos):
    """RoPE of x [n][heads][128] at the positions, from the library's fp32 tables."""
    cos, sin = (t[pos].double()[:, None] for t in _rope())
    a, b = x[..., :64], x[..., 64:]
    return torch.cat([a * cos - b * sin, a * sin + b * cos], dim=-1)


def _attend64(q, k, v, first):
    """q [n][32][128] at positions first.., k and v [8][first + n][128] -> [n][4096]."""
    n, m = q.shape[0], k.shape[1]
    out = torch.empty(n, QH, D, dtype=torch.float64, device=q.device)
    for g in range(KVH):
        kt, vg = k[g].double().t().contiguous(), v[g].double()
        for h in range(4 * g, 4 * g + 4):
            for r in range(0, n, 1024):
                s = (q[r:r + 1024, h] @ kt) * D ** -0.5
                rows = torch.arange(first + r, first + r + s.shape[0], device=q.device)
                s.masked_fill_(torch.arange(m, device=q.device)[None] > rows[:, None], float("-inf"))
                out[r:r + 1024, h] = torch.softmax(s, dim=-1) @ vg
    return out.reshape(n, H)


def _qkv64(x, w, pos):
    a = _norm64(x, w["input_layernorm"])
    n = x.shape[0]
    q = _rot64(_mul64(a, w["w_q"]).view(n, QH, D), pos)
    k = _rot64(_mul64(a, w["w_k"]).view(n, KVH, D), pos)
    return q, k, _mul64(a, w["w_v"]).view(n, KVH, D)


def _rest64(x, att, w):
    x = x + _mul64(att, w["w_o"])
    b = _norm64(x, w["post_attention_layernorm"])
    return x + _mul64(torch.nn.functional.silu(_mul64(b, w["w_gate"])) * _mul64(b, w["w_up"]),
                      w["w_down"])


def _token64(x, w, lens, past):
    """One layer for the new token of each sequence: x [b][4096], past(i) the K and V rows
    [2][8][lens[i]-1][128] of sequence i.  Returns the rows and the new K/V [b][2][8][128]."""
    pos = torch.tensor([n - 1 for n in lens], device=x.device)
    q, k, v = _qkv64(x, w, pos)
    att, new = [], torch.stack([k, v], dim=1)
    for i, n in enumerate(lens):
        kv = torch.cat([past(i).double(), new[i][:, :, None]], dim=2)
        att.append(_attend64(q[i:i + 1], kv[0], kv[1], n - 1))
    return _rest64(x, torch.cat(att), w), new


def _rows64(pool, table, layer, n):
    """The K and V rows [2][8][n][128] of a sequence's pages."""
    p = pool[table[:-(-n // PAGE)].long(), layer]
    return p.permute(1, 2, 0, 3, 4).reshape(2, KVH, -1, D)[:, :, :n]


def exact(case, seed):
    s = prepare(case, seed)
    k = s["kind"]
    if k == "decode_step":
        n, w = case["ctx"], s["w"]
        x, new = w["emb_lookup"][s["tokens"][n - 1:n].long()].double(), []
        for l in range(LAYERS):
            x, kv = _token64(x, w["layers"][l], [n], lambda i: s["kv"][l, :, :, :n - 1])
            new.append(kv[0])
        return {"logits": _mul64(_norm64(x, w["final_norm"]), w["lm_head"])[0],
                "new_kv": torch.stack(new)}
    if k == "decode_layer":
        n = case["ctx"]
        x, kv = _token64(s["x"].double(), s["w"]["layers"][LAYER], [n],
                         lambda i: s["kv"][LAYER, :, :, :n - 1])
        return {"x": x, "new_kv": kv[0]}
    if k == "batched_layer":
        lens = _lens(case)
        x, kv = _token64(s["x"].double(), s["w"]["layers"][LAYER], lens,
                         lambda i: s["planes"][i, :, :, :lens[i] - 1])
        return {"x": x, "new_kv": list(kv)}
    if k == "batched_paged":
        lens, w = _lens(case), s["w"]
        ids = torch.stack([s["tokens"][i, n - 1] for i, n in enumerate(lens)])
        x = w["emb_lookup"][ids.long()].double()
        for l in range(LAYERS):
            x, _ = _token64(x, w["layers"][l], lens,
                            lambda i: _rows64(s["pool"], s["table"][i], l, lens[i] - 1))
        return {"logits": _mul64(_norm64(x, w["final_norm"]), w["lm_head"])}
    if k == "prefill_layer":
        w, x = s["w"]["layers"][LAYER], s["x"].double()
        q, kk, v = _qkv64(x, w, torch.arange(case["rows"], device="cuda"))
        new = torch.stack([kk, v]).transpose(1, 2).contiguous()
        return {"x": _rest64(x, _attend64(q, new[0], new[1], 0), w), "new_kv": new}
    if k == "chunk_attn":
        kv = _rows64(s["pool"], s["table"][0], LAYER, case["start"] + case["rows"])
        return _attend64(s["q"].double(), kv[0], kv[1], case["start"])
    if k == "head":
        return _mul64(_norm64(s["x"].double(), s["norm"]), s["lm_head"])
    return None  # token ids have no nearby values
