"""Performance cases of the Qwen3-4B decode path on one MI355X.

Each case is one unit of work that a decode or serving program hands to this
package: an MLP, an attention half of a decoder layer, the attention launch
alone, the vocabulary head, the row kernels of a prefill layer, or a whole
greedy decode step.  ``prepare`` builds what such a program holds between
calls (weights, caches, workspaces and, where the program captures its step
once, the captured HIP graph), ``run`` does one pass, ``exact`` restates the
pass in float64 torch.

Shapes are those of the model this package serves (``Qwen3Config``); rows,
batch, context length and tree size vary over what a server sees: one
sequence up to the 128 rows of a batch-16 x 8-node speculative verify.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from starter_amd import decode as D
from starter_amd import kernels as K

BF16 = torch.bfloat16
F64 = torch.float64
CFG = D.Qwen3Config()
H, I, V = CFG.hidden, CFG.intermediate, CFG.vocab
HQ, HKV, HD = CFG.heads, CFG.kv_heads, CFG.head_dim
QKV = (HQ + 2 * HKV) * HD
EPS = CFG.eps
DEV = "cuda:0"


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # The MLP of a decoder layer (residual add + norm + gate/up + SwiGLU,
        # then down), replayed from a graph: one sequence, the batch-16 decode
        # step, five sequences of an 8-node draft tree, and the batch-16 x
        # 8-node verify pass.
        {"name": "mlp_m1", "kind": "mlp", "M": 1},
        {"name": "mlp_m16", "kind": "mlp", "M": 16},
        {"name": "mlp_m40", "kind": "mlp", "M": 40},
        {"name": "mlp_m128", "kind": "mlp", "M": 128},
        # The attention half of a decoder layer (norm + qkv, rotary step +
        # cache write + attention, o_proj), replayed from a graph: a single
        # chat sequence some 2000 tokens in, and the verify pass of a batch.
        {"name": "attn_half_b1", "kind": "attn_half", "B": 1, "R": 1, "ctx": 2000, "cap": 4096},
        {"name": "attn_half_verify_b16x8", "kind": "attn_half", "B": 16, "R": 8, "ctx": 1151, "cap": 1408},
        # The attention launch alone: a batch whose sequences have come to
        # different lengths, and two long documents.
        {"name": "attention_b16_mixed", "kind": "attention", "B": 16, "R": 1, "ctx": 1400, "cap": 1408},
        {"name": "attention_b2_long", "kind": "attention", "B": 2, "R": 1, "ctx": 32000, "cap": 32768},
        # One projection called without a graph, as while a program is being
        # brought up: the launch path counts as much as the kernel.
        {"name": "o_proj_m4_eager", "kind": "o_proj", "M": 4},
        # Logits of every verify row and their eight best tokens (the drafts
        # of the next round).
        {"name": "head_topk_m128", "kind": "head_topk", "M": 128, "k": 8},
        # What this package runs in a prefill layer beside the library's large
        # products: two residual adds + norms, the rotary step with its cache
        # write, and SwiGLU, over 16 prompts of 1024 tokens.
        {"name": "prefill_rows_16x1024", "kind": "prefill_rows", "B": 16, "T": 1024},
        # A whole greedy step of 16 sequences (four layers and the full
        # vocabulary), replayed from the plan's graph.
        {"name": "decode_b16", "kind": "decode", "B": 16, "T": 1024, "layers": 4},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["mlp", "mlp", "attn_half", "attn_half", "attention", "attention", "o_proj", "head_topk",
                       "head_argmax", "prefill_rows", "decode"])
    if kind == "mlp" or kind == "head_argmax":
        return {"kind": kind, "M": _log_int(rng, 1, 128)}
    if kind == "o_proj":
        return {"kind": kind, "M": _log_int(rng, 1, 128)}
    if kind == "head_topk":
        return {"kind": kind, "M": _log_int(rng, 1, 128), "k": rng.choice([4, 8, 16])}
    if kind == "prefill_rows":
        B = _log_int(rng, 1, 16)
        return {"kind": kind, "B": B, "T": _log_int(rng, 17, 16384 // B)}
    if kind == "decode":
        return {"kind": kind, "B": _log_int(rng, 1, 16), "T": _log_int(rng, 64, 1200), "layers": rng.randint(2, 4)}
    R = rng.choice([1, 1, 2, 3, 4, 5, 7, 8])
    B = _log_int(rng, 1, min(64, 128 // R))
    ctx = _log_int(rng, 64, min(32000, 65536 // B))
    return {"kind": kind, "B": B, "R": R, "ctx": ctx, "cap": (ctx + R + rng.randint(64, 2048) + 63) // 64 * 64}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

class _Source:
    """Tensors of one seed, drawn on the GPU in a fixed order."""

    def __init__(self, seed: int):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed))

    def normal(self, *shape, std: float = 1.0) -> torch.Tensor:
        return torch.empty(shape, dtype=BF16, device=DEV).normal_(0.0, std, generator=self.g)

    def weight(self, *shape) -> torch.Tensor:
        return self.normal(*shape, std=0.02)

    def gain(self, n: int) -> torch.Tensor:
        return (1.0 + 0.1 * torch.randn(n, generator=self.g, device=DEV)).to(BF16)

    def ints(self, lo: int, hi: int, n: int, dtype=torch.int32) -> torch.Tensor:
        return torch.randint(lo, hi, (n,), generator=self.g, device=DEV).to(dtype)


def _tree(R: int) -> tuple[list[int], list[int]]:
    """Parents and depths of an R-node draft tree (two children per node)."""
    parents = [-1] + [(t - 1) // 2 for t in range(1, R)]
    depth = [0] * R
    for t in range(1, R):
        depth[t] = depth[parents[t]] + 1
    return parents, depth


def _positions(src: _Source, case: dict) -> torch.Tensor:
    """Sequences of a batch stand between half the context and all of it."""
    B, ctx = case["B"], case["ctx"]
    return src.ints(ctx // 2, ctx + 1, B) if B > 1 else torch.full((1,), ctx, dtype=torch.int32, device=DEV)


def _attention_inputs(src: _Source, case: dict) -> dict:
    B, R, cap = case["B"], case["R"], case["cap"]
    cos, sin = D.rope_tables(CFG, cap, DEV)
    s = {"q_norm": src.gain(HD), "k_norm": src.gain(HD), "cos": cos, "sin": sin, "pos": _positions(src, case),
         "k_cache": src.normal(B, HKV, cap, HD), "v_cache": src.normal(B, HKV, cap, HD), "tree": None, "depth": None}
    if R > 1:
        parents, depth = _tree(R)
        s["tree"] = torch.tensor(K.ancestor_masks(parents), dtype=torch.int64, device=DEV)
        s["depth"] = torch.tensor(depth, dtype=torch.int32, device=DEV)
    return s


def _inputs(case: dict, seed: int) -> dict:
    """The tensors of a case, the same for ``prepare`` and ``exact``."""
    src = _Source(seed)
    kind = case["kind"]
    if kind == "mlp":
        M = case["M"]
        return {"x": src.normal(M, H), "y": src.normal(M, H), "norm": src.gain(H), "wgu": src.weight(2 * I, H),
                "wd": src.weight(H, I)}
    if kind == "o_proj":
        return {"a": src.normal(case["M"], HQ * HD), "wo": src.weight(H, HQ * HD)}
    if kind in ("head_topk", "head_argmax"):
        M = case["M"]
        return {"x": src.normal(M, H), "y": src.normal(M, H), "norm": src.gain(H), "lm_head": src.weight(V, H)}
    if kind == "attention":
        s = _attention_inputs(src, case)
        s["qkv"] = src.normal(case["B"] * case["R"], QKV)
        return s
    if kind == "attn_half":
        s = _attention_inputs(src, case)
        M = case["B"] * case["R"]
        s.update(x=src.normal(M, H), y=src.normal(M, H), norm=src.gain(H), wqkv=src.weight(QKV, H),
                 wo=src.weight(H, HQ * HD))
        return s
    if kind == "prefill_rows":
        B, T = case["B"], case["T"]
        cap = (T + 64 + 63) // 64 * 64
        cos, sin = D.rope_tables(CFG, cap, DEV)
        N = B * T
        return {"x": src.normal(N, H), "o": src.normal(N, H), "norm1": src.gain(H), "gu": src.normal(N, 2 * I),
                "d": src.normal(N, H), "norm2": src.gain(H), "qkv": src.normal(N, QKV), "q_norm": src.gain(HD),
                "k_norm": src.gain(HD), "cos": cos, "sin": sin, "cap": cap}
    raise ValueError(kind)


def _captured(call) -> dict:
    """The program's step captured once: its replay, its outputs, and the step
    itself, whose plans own the workspaces that the replay uses."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    return {"call": call, "graph": graph, "out": out}


def _decode_plan(case: dict, seed: int):
    cfg = D.Qwen3Config(layers=case["layers"])
    model = D.SyntheticModel(cfg, device=DEV, seed=int(seed), norm_noise=0.1)
    plan = D.DecodePlan(model, case["B"], case["T"], 128)
    src = _Source(seed + 1)
    plan.k_cache.normal_(0.0, 1.0, generator=src.g)
    plan.v_cache.normal_(0.0, 1.0, generator=src.g)
    tok = src.ints(0, V, case["B"], torch.int64)
    pos = torch.full((case["B"],), case["T"] + 64, dtype=torch.int32, device=DEV)   # halfway through the answer
    return plan, tok, pos


def prepare(case: dict, seed: int):
    kind = case["kind"]
    if kind == "decode":
        plan, tok, pos = _decode_plan(case, seed)
        plan.tok.copy_(tok)
        plan.pos.copy_(pos)
        plan.capture()
        return {"kind": kind, "plan": plan, "tok": tok, "pos": pos}

    s = _inputs(case, seed)
    s["kind"] = kind
    if kind == "mlp":
        gu = K.pick_normed("gateup", s["x"], s["y"], s["norm"], s["wgu"], EPS)
        down = K.pick_matmul(torch.empty((case["M"], I), dtype=BF16, device=DEV), s["wd"])
        xout = torch.empty_like(s["x"])

        def call():
            act = gu(s["x"], s["y"], s["norm"], xout, s["wgu"])
            return {"xout": xout, "act": act, "y": down(act, s["wd"])}

        s.update(_captured(call))
    elif kind == "o_proj":
        s["mm"] = K.pick_matmul(s["a"], s["wo"])
    elif kind == "head_topk":
        mm = K.pick_normed("matmul", s["x"], s["y"], s["norm"], s["lm_head"], EPS)
        xout = torch.empty_like(s["x"])

        def call():
            logits = mm(s["x"], s["y"], s["norm"], xout, s["lm_head"])
            vals, idxs = K.fast_topk(logits, case["k"])
            return {"xout": xout, "logits": logits, "vals": vals, "idxs": idxs}

        s.update(_captured(call))
    elif kind == "head_argmax":
        mm = K.pick_lm_argmax(s["x"], s["lm_head"], EPS)
        xout = torch.empty_like(s["x"])

        def call():
            ids, maxv = mm(s["x"], s["y"], s["norm"], xout, s["lm_head"])
            return {"xout": xout, "ids": ids, "maxv": maxv}

        s.update(_captured(call))
    elif kind in ("attention", "attn_half"):
        B, R, cap = case["B"], case["R"], case["cap"]
        attn = K.pick_attention(B, HQ, HKV, HD, cap, case["ctx"], DEV, R=R, tree=R > 1, maxlen=cap)
        attn_out = torch.empty((B, R, HQ, HD), dtype=BF16, device=DEV)

        def attend(qkv):
            attn.rope_attend(qkv, s["q_norm"], s["k_norm"], s["cos"], s["sin"], s["pos"], s["k_cache"], s["v_cache"],
                             attn_out, EPS, tree=s["tree"], depth=s["depth"])

        if kind == "attention":
            def call():
                attend(s["qkv"])
                return {"out": attn_out, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
        else:
            mm_qkv = K.pick_normed("matmul", s["x"], s["y"], s["norm"], s["wqkv"], EPS)
            mm_o = K.pick_matmul(attn_out.view(B * R, HQ * HD), s["wo"])
            xout = torch.empty_like(s["x"])

            def call():
                attend(mm_qkv(s["x"], s["y"], s["norm"], xout, s["wqkv"]))
                o = mm_o(attn_out.view(B * R, HQ * HD), s["wo"])
                return {"xout": xout, "out": attn_out, "o": o, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}

        s.update(_captured(call))
    elif kind == "prefill_rows":
        B, T, cap = case["B"], case["T"], s["cap"]
        s["pos"] = torch.zeros((B,), dtype=torch.int32, device=DEV)
        s["q"] = torch.empty((B, HQ, T, HD), dtype=BF16, device=DEV)
        s["k_cache"] = torch.zeros((B, HKV, cap, HD), dtype=BF16, device=DEV)
        s["v_cache"] = torch.zeros((B, HKV, cap, HD), dtype=BF16, device=DEV)
        s["x1"], s["x2"] = torch.empty_like(s["x"]), torch.empty_like(s["x"])
        s["T"] = T
    return s


def run(s):
    kind = s["kind"]
    if kind == "decode":
        # every pass is the same step: the token and position it starts from
        plan = s["plan"]
        plan.tok.copy_(s["tok"])
        plan.pos.copy_(s["pos"])
        plan.g_decode.replay()
        # Not the tokens: with random weights the two best logits of a row are
        # often closer than a change of rounding in the layers moves them.
        return {"x": plan.xa, "max_logit": plan.maxv_out, "k_cache": plan.k_cache, "v_cache": plan.v_cache}
    if kind == "o_proj":
        return s["mm"](s["a"], s["wo"])
    if kind == "prefill_rows":
        K.qk_norm_rope_cache(s["qkv"], s["q_norm"], s["k_norm"], s["cos"], s["sin"], s["pos"], s["q"], s["k_cache"],
                             s["v_cache"], s["T"], EPS)
        h1 = K.add_rms_norm(s["x"], s["o"], s["norm1"], EPS, xout=s["x1"])
        act = K.swiglu(s["gu"])
        h2 = K.add_rms_norm(s["x1"], s["d"], s["norm2"], EPS, xout=s["x2"])
        return {"q": s["q"], "k_cache": s["k_cache"], "v_cache": s["v_cache"], "x1": s["x1"], "h1": h1, "act": act,
                "x2": s["x2"], "h2": h2}
    s["graph"].replay()
    return s["out"]


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how far apart two right answers may be
# ---------------------------------------------------------------------------

def _keys(case: dict) -> float:
    """Keys one pass reads, over the batch (the mean of the drawn lengths)."""
    B, R, ctx = case["B"], case["R"], case["ctx"]
    return B * (R + (0.75 * ctx if B > 1 else ctx))


def _attention_work(case: dict) -> tuple[float, float]:
    B, R = case["B"], case["R"]
    keys = _keys(case)
    nbytes = keys * HKV * HD * 4 + B * R * (QKV + HQ * HD) * 2
    return nbytes, 4.0 * keys * R * HQ * HD


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "mlp":
        M = case["M"]
        return {"bytes": 2.0 * (3 * I * H + M * (4 * H + 2 * I) + H), "flops": 6.0 * M * I * H}
    if kind == "o_proj":
        M = case["M"]
        return {"bytes": 2.0 * (H * HQ * HD + M * (H + HQ * HD)), "flops": 2.0 * M * H * HQ * HD}
    if kind == "head_topk":
        M = case["M"]
        return {"bytes": 2.0 * (V * H + M * (3 * H + 2 * V)) + 8.0 * M * case["k"], "flops": 2.0 * M * V * H}
    if kind == "head_argmax":
        M = case["M"]
        return {"bytes": 2.0 * (V * H + 3 * M * H) + 12.0 * M, "flops": 2.0 * M * V * H}
    if kind == "attention":
        nbytes, flops = _attention_work(case)
        return {"bytes": nbytes, "flops": flops}
    if kind == "attn_half":
        M = case["B"] * case["R"]
        nbytes, flops = _attention_work(case)
        return {"bytes": nbytes + 2.0 * (QKV * H + H * HQ * HD + M * (4 * H + QKV + HQ * HD)),
                "flops": flops + 2.0 * M * (QKV * H + H * HQ * HD)}
    if kind == "prefill_rows":
        N = case["B"] * case["T"]
        return {"bytes": 2.0 * N * (2 * QKV + 8 * H + 3 * I), "flops": N * (10.0 * QKV + 20.0 * H + 8.0 * I)}
    B, L = case["B"], case["layers"]
    layer = QKV * H + H * HQ * HD + 3 * I * H
    keys = B * (case["T"] + 65.0)
    return {"bytes": 2.0 * (L * layer + V * H) + L * keys * HKV * HD * 4,
            "flops": 2.0 * B * (L * layer + V * H) + L * 4.0 * keys * HQ * HD}


def tolerance(case: dict):
    # Outputs are bf16 after several bf16 roundings inside each block; the
    # float64 restatement (which rounds nowhere) is 0.2-0.4% away for a block
    # and about 1% after the layers of a whole step.
    if case["kind"] == "decode":
        return {"rel": 0.03, "max": 0.5}
    if case["kind"] in ("head_topk", "head_argmax"):
        return {"rel": 0.01, "max": 0.2, "differ": 0.01}
    return {"rel": 0.01, "max": 0.2}


# ---------------------------------------------------------------------------
# The same passes in float64
# ---------------------------------------------------------------------------

def _mm(a: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """a @ w.T in float64, the weight rows converted a block at a time."""
    return torch.cat([a @ w[n:n + 16384].to(F64).t() for n in range(0, w.shape[0], 16384)], 1)


def _norm(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.to(F64)


def _rotate(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    half = x.shape[-1] // 2
    return x * cos + torch.cat((-x[..., half:], x[..., :half]), -1) * sin


def _attend(qkv, s, k_cache, v_cache, B: int, R: int):
    """Rotary step, cache write (into the given float64 caches) and attention."""
    rows = qkv.view(B, R, HQ + 2 * HKV, HD)
    depth = s["depth"].long() if s["depth"] is not None else torch.arange(R, device=DEV)
    masks = s["tree"].tolist() if s["tree"] is not None else [(1 << (t + 1)) - 1 for t in range(R)]
    out = torch.empty((B, R, HQ, HD), dtype=F64, device=DEV)
    for b in range(B):
        p = int(s["pos"][b])
        cos, sin = (s[n][p + depth].to(F64)[:, None] for n in ("cos", "sin"))
        q = _rotate(_norm(rows[b, :, :HQ], s["q_norm"]), cos, sin)
        k = _rotate(_norm(rows[b, :, HQ:HQ + HKV], s["k_norm"]), cos, sin)
        k_cache[b, :, p:p + R] = k.transpose(0, 1)
        v_cache[b, :, p:p + R] = rows[b, :, HQ + HKV:].transpose(0, 1)
        seen = torch.ones((R, p + R), dtype=torch.bool, device=DEV)
        for t in range(R):
            seen[t, p:] = torch.tensor([bool((masks[t] >> j) & 1) for j in range(R)], device=DEV)
        kk, vv = k_cache[b, :, :p + R], v_cache[b, :, :p + R]
        qg = q.transpose(0, 1).reshape(HKV, HQ // HKV * R, HD)                 # head-major, then row
        score = (qg @ kk.transpose(1, 2).contiguous()) / math.sqrt(HD)
        score = score.view(HKV, HQ // HKV, R, p + R).masked_fill(~seen, -math.inf)
        o = score.softmax(-1).view(HKV, HQ // HKV * R, p + R) @ vv
        out[b] = o.view(HQ, R, HD).transpose(0, 1)
    return out


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "decode":
        plan, tok, pos = _decode_plan(case, seed)
        m, B = plan.model, case["B"]
        k_cache, v_cache = plan.k_cache.to(F64), plan.v_cache.to(F64)
        x = m.embed[tok].to(F64)
        for i, layer in enumerate(m.layers):
            s = {"q_norm": layer.q_norm, "k_norm": layer.k_norm, "cos": plan.cos, "sin": plan.sin, "pos": pos,
                 "tree": None, "depth": None}
            o = _attend(_mm(_norm(x, layer.in_norm), layer.wqkv), s, k_cache[i], v_cache[i], B, 1)
            x = x + _mm(o.view(B, HQ * HD), layer.wo)
            gu = _mm(_norm(x, layer.post_norm), layer.wgu)
            x = x + _mm(F.silu(gu[:, :I]) * gu[:, I:], layer.wd)
        logits = _mm(_norm(x, m.final_norm), m.lm_head)
        return {"x": x, "max_logit": logits.max(-1).values, "k_cache": k_cache, "v_cache": v_cache}
    s = _inputs(case, seed)
    if kind == "o_proj":
        return _mm(s["a"].to(F64), s["wo"])
    if kind == "prefill_rows":
        B, T = case["B"], case["T"]
        rows = s["qkv"].view(B, T, HQ + 2 * HKV, HD)
        cos, sin = s["cos"][:T].to(F64)[:, None], s["sin"][:T].to(F64)[:, None]
        k_cache = torch.zeros((B, HKV, s["cap"], HD), dtype=F64, device=DEV)
        v_cache = torch.zeros_like(k_cache)
        q = torch.empty((B, HQ, T, HD), dtype=F64, device=DEV)
        for b in range(B):
            r = rows[b].to(F64)
            q[b] = _rotate(_norm(r[:, :HQ], s["q_norm"]), cos, sin).transpose(0, 1)
            k_cache[b, :, :T] = _rotate(_norm(r[:, HQ:HQ + HKV], s["k_norm"]), cos, sin).transpose(0, 1)
            v_cache[b, :, :T] = r[:, HQ + HKV:].transpose(0, 1)
        x1 = s["x"].to(F64) + s["o"].to(F64)
        gu = s["gu"]
        act = F.silu(gu[:, :I].to(F64)) * gu[:, I:].to(F64)
        x2 = x1 + s["d"].to(F64)
        return {"q": q, "k_cache": k_cache, "v_cache": v_cache, "x1": x1, "h1": _norm(x1, s["norm1"]), "act": act,
                "x2": x2, "h2": _norm(x2, s["norm2"])}
    if kind == "attention":
        k_cache, v_cache = s["k_cache"].to(F64), s["v_cache"].to(F64)
        out = _attend(s["qkv"].to(F64), s, k_cache, v_cache, case["B"], case["R"])
        return {"out": out, "k_cache": k_cache, "v_cache": v_cache}
    xout = s["x"].to(F64) + s["y"].to(F64)
    h = _norm(xout, s["norm"])
    if kind == "mlp":
        gu = _mm(h, s["wgu"])
        act = F.silu(gu[:, :I]) * gu[:, I:]
        return {"xout": xout, "act": act, "y": _mm(act, s["wd"])}
    if kind == "attn_half":
        B, R = case["B"], case["R"]
        k_cache, v_cache = s["k_cache"].to(F64), s["v_cache"].to(F64)
        out = _attend(_mm(h, s["wqkv"]), s, k_cache, v_cache, B, R)
        return {"xout": xout, "out": out, "o": _mm(out.view(B * R, HQ * HD), s["wo"]), "k_cache": k_cache,
                "v_cache": v_cache}
    logits = _mm(h, s["lm_head"])
    if kind == "head_argmax":
        return {"xout": xout, "ids": None, "maxv": logits.max(-1).values}
    # the values of ranks past the first follow the kernel's documented
    # approximation (one candidate per lane), so they have no exact value here
    return {"xout": xout, "logits": logits, "vals": None, "idxs": None}
