"""The work this backend is measured on: the layers and steps of the decoder
and the vision encoder, each through the public ops of the package, at the
sizes the model's configuration, the tests and bench.py use.

`listed()` gives the cases, `draw(rng)` more of the same ranges. `prepare`
makes what a program holds before the call (inputs, weights, workspaces, a
captured decode step), `run` is one pass, `exact` the same outputs in 64-bit
torch with the roundings to bf16 that the ops document.
"""

import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """The package (its directory is not an identifier) as module uocr_rocm."""
    if "uocr_rocm" not in sys.modules:
        path = os.path.join(ROOT, "grpc-unlimited-ocr_amd", "__init__.py")
        spec = importlib.util.spec_from_file_location("uocr_rocm", path)
        mod = importlib.util.module_from_spec(spec)
        sys.modules["uocr_rocm"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["uocr_rocm"]


# The decoder's dimensions: hidden, heads x head dim, the dense layer's FFN,
# routed experts and their FFN, the shared experts' FFN, the vocabulary, the
# block router's key width; SAM's and CLIP's widths.
HIDDEN, HEADS, HD, DENSE_FFN = 1280, 10, 128, 6848
EXPERTS, TOP_K, EXPERT_FFN, SHARED_FFN = 64, 6, 896, 1792
VOCAB, ROUTER_D, BLOCK, LOCAL, TOP_M, TOP_BLOCKS = 129280, 128, 32, 4, 16, 12
N_TOK, PAGE_MOD = 63, 2  # rope: 63 token pairs and one page pair
SAM_W, SAM_HEADS, SAM_MLP, SAM_WINDOW = 768, 12, 3072, 14
CLIP_W, CLIP_HEADS, CLIP_MLP = 1024, 16, 4096
EPS = 1e-6


def listed():
    return [
        # Batch-1 decode's small ops called one by one: the embedding row with
        # the residual add and RMSNorm, then RoPE on q and k. The smallest call.
        {"name": "decode_chain", "kind": "chain_step", "hidden": 2048, "q_heads": 16, "k_heads": 4, "dtype": "bf16"},
        # One token through a mixture-of-experts layer (11 of the model's 12)
        # of the block-routed decode step, replayed as a captured graph as a
        # program decodes, over a full fp32 cache of 8192 positions.
        {"name": "decode_moe", "kind": "decode", "moe": True, "cap": 8192, "pos": 8191, "cache": "f32"},
        # One token through the dense layer attending to every position of a
        # bf16 cache, then the final norm and LM head: the step's two ends.
        {"name": "decode_dense_head", "kind": "decode", "moe": False, "cap": 4096, "pos": 2777, "cache": "bf16"},
        # The fused prefill ops of a layer over a long prompt (the benchmark's
        # headline chain): add + RMSNorm, SwiGLU, RoPE.
        {"name": "prefill_chain", "kind": "chain", "rows": 8192, "hidden": 2048, "ffn": 1408, "q_heads": 16,
         "k_heads": 4, "dtype": "bf16"},
        # The dense layer's MLP over a 4096-token prompt: gate and up stacked.
        {"name": "prefill_mlp", "kind": "mlp", "rows": 4096, "ffn": DENSE_FFN},
        # The routed experts of one layer over a prompt, expert by expert.
        {"name": "prefill_experts", "kind": "experts", "rows": 4096, "experts": EXPERTS},
        # What a layer's routing computes over a prompt: the router's norms,
        # rope, block summaries, scores and key mask, the gate's logits and
        # top experts.
        {"name": "prefill_routing", "kind": "routing", "rows": 4096, "first": 0},
        # The prompt's attention under the routed key mask, into bf16 for the
        # output projection.
        {"name": "prefill_attention", "kind": "attention", "rows": 4096, "first": 0, "heads": HEADS, "hd": HD,
         "mask": "routed", "out": "bf16", "workspace": True},
        # Attention of a head dim without a one-pass kernel: scores product,
        # scale + mask + softmax, values product, over a second prompt's rows.
        {"name": "attention_products", "kind": "products", "rows": 1003, "first": 517, "heads": 10, "hd": 96},
        # One CLIP layer over a 1024-pixel view's 257 tokens.
        {"name": "clip_layer", "kind": "clip", "grid": 16},
        # One SAM block with global attention over a 1024-pixel view's 64 x 64
        # grid, and one with 14 x 14 windows (8 of the encoder's 12).
        {"name": "sam_global", "kind": "sam", "grid": 64, "windowed": False},
        {"name": "sam_windows", "kind": "sam", "grid": 64, "windowed": True},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["chain_step", "decode", "decode", "chain", "mlp", "experts", "routing", "attention",
                       "attention", "products", "clip", "sam", "sam"])
    if kind == "chain_step":
        return {"kind": kind, "hidden": 8 * _log(rng, 64, 512), "q_heads": rng.randint(1, 32),
                "k_heads": rng.randint(1, 8), "dtype": rng.choice(["bf16", "f32"])}
    if kind == "decode":
        cap = BLOCK * _log(rng, 8, 512)
        return {"kind": kind, "moe": rng.random() < 0.6, "cap": cap, "pos": rng.randint(1, cap - 1),
                "cache": rng.choice(["f32", "bf16"])}
    if kind == "chain":
        return {"kind": kind, "rows": _log(rng, 16, 8192), "hidden": rng.choice([1280, 2048]),
                "ffn": rng.choice([896, 1408, 1792]), "q_heads": rng.choice([10, 16]),
                "k_heads": rng.choice([4, 10]), "dtype": rng.choice(["bf16", "f32"])}
    if kind == "mlp":
        return {"kind": kind, "rows": _log(rng, 16, 4096), "ffn": rng.choice([SHARED_FFN, DENSE_FFN])}
    if kind == "experts":
        return {"kind": kind, "rows": _log(rng, 32, 4096), "experts": rng.choice([16, 32, 64])}
    if kind == "routing":
        rows = _log(rng, 16, 4096)
        return {"kind": kind, "rows": rows, "first": rng.choice([0, rng.randint(1, 1024)])}
    if kind == "attention":
        rows = _log(rng, 16, 4096)
        mask = rng.choice(["routed", "causal", "none"])
        return {"kind": kind, "rows": rows, "first": 0 if mask == "none" else rng.choice([0, rng.randint(1, 1024)]),
                "heads": rng.choice([10, 12, 16]), "hd": rng.choice([64, 128]), "mask": mask,
                "out": rng.choice(["bf16", "f32"]), "workspace": mask != "none" and rng.random() < 0.75}
    if kind == "products":
        return {"kind": kind, "rows": _log(rng, 16, 1536), "first": rng.choice([0, rng.randint(1, 512)]),
                "heads": rng.randint(2, 16), "hd": 4 * rng.randint(4, 40)}
    if kind == "clip":
        return {"kind": kind, "grid": rng.randint(3, 24)}
    return {"kind": "sam", "grid": 4 * rng.randint(2, 16), "windowed": rng.random() < 0.6}


# ---- inputs ------------------------------------------------------------------


def _tables():
    """PageRope's frequency tables, float32 of 64-bit powers."""
    i = np.arange(N_TOK, dtype=np.float64)
    return torch.from_numpy((1.0 / 1e4 ** (i / N_TOK)).astype(np.float32)).cuda(), torch.ones(1, device="cuda")


def _rope_inv(n):
    return torch.from_numpy((1.0 / 1e4 ** (np.arange(n, dtype=np.float64) / n)).astype(np.float32)).cuda()


class _Source:
    """Inputs on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))

    def f32(self, *shape, scale=1.0):
        return torch.randn(*shape, device="cuda", generator=self.g) * scale

    def bf16(self, *shape, scale=1.0):
        out = torch.empty(*shape, device="cuda", dtype=torch.bfloat16)
        flat = out.view(-1)
        for at in range(0, flat.numel(), 1 << 26):  # no full-size fp32 copy of the large tables
            part = flat[at:at + (1 << 26)]
            part.copy_(torch.randn(part.numel(), device="cuda", generator=self.g) * scale)
        return out

    def norm(self, n):
        return 1 + 0.02 * self.f32(n)

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, device="cuda", generator=self.g)


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def _dtype(name):
    return torch.bfloat16 if name == "bf16" else torch.float32


def _inputs(case, seed):
    """The inputs and weights of a case, before any workspace or output."""
    s, kind = _Source(seed), case["kind"]
    t = {}
    if kind == "chain_step":
        n, dt = case["hidden"], _dtype(case["dtype"])
        vocab = 128000
        t["table"] = s.bf16(vocab, n)
        t["delta"], t["w"] = s.f32(n).to(dt), s.norm(n)
        t["q"], t["k"] = s.f32(case["q_heads"] * HD).to(dt), s.f32(case["k_heads"] * HD).to(dt)
        t["inv"] = _rope_inv(HD // 2)
        token, pos = int(s.ints(0, vocab, 1)), int(s.ints(0, 32768, 1))
        t["step"] = torch.tensor([token, pos, pos, 0, -1], device="cuda")
    elif kind == "decode":
        cap, pos, width, moe = case["cap"], case["pos"], HEADS * HD, case["moe"]
        dt = _dtype(case["cache"])
        t["x"], t["delta"] = s.f32(HIDDEN), s.f32(HIDDEN)
        t["in"], t["post"] = s.norm(HIDDEN), s.norm(HIDDEN)
        t["proj"] = s.bf16(3 * width + (2 * ROUTER_D if moe else 0), HIDDEN, scale=0.03)
        t["o"] = s.bf16(HIDDEN, width, scale=0.03)
        t["kc"], t["vc"] = s.f32(cap, width).to(dt), s.f32(cap, width).to(dt)
        f = SHARED_FFN if moe else DENSE_FFN
        t["gate"], t["up"] = s.bf16(f, HIDDEN, scale=0.03), s.bf16(f, HIDDEN, scale=0.03)
        t["down"] = s.bf16(HIDDEN, f, scale=0.03)
        t["inv_tok"], t["inv_page"] = _tables()
        # positions past a prompt of pages: the prompt is the first half of
        # the cache, eight blocks a page, the query confined to one page of it
        page = int(s.ints(0, 4, 1))
        t["step"] = torch.tensor([0, pos, max(0, pos - cap // 4), 17, page], device="cuda")
        if moe:
            t["rqn"], t["rkn"], t["cls"] = s.f32(ROUTER_D, scale=0.1), s.f32(ROUTER_D, scale=0.1), s.f32(ROUTER_D)
            t["rkeys"], t["summ"] = s.f32(cap, ROUTER_D), s.f32(cap // BLOCK, ROUTER_D)
            t["pages"] = torch.arange(max(1, cap // BLOCK // 2), device="cuda") // 8
            t["router"] = s.f32(EXPERTS, HIDDEN, scale=0.05)
            t["gs"] = s.bf16(EXPERTS * EXPERT_FFN, HIDDEN, scale=0.03)
            t["us"] = s.bf16(EXPERTS * EXPERT_FFN, HIDDEN, scale=0.03)
            t["ds"] = s.bf16(EXPERTS, HIDDEN, EXPERT_FFN, scale=0.03)
        else:
            t["lm"], t["final"] = s.bf16(VOCAB, HIDDEN, scale=0.03), s.norm(HIDDEN)
    elif kind == "chain":
        rows, n, f, dt = case["rows"], case["hidden"], case["ffn"], _dtype(case["dtype"])
        t["x"], t["delta"], t["w"] = s.f32(rows, n).to(dt), s.f32(rows, n).to(dt), s.norm(n)
        t["gu"] = s.f32(rows, 2 * f).to(dt)
        t["q"], t["k"] = s.f32(rows, case["q_heads"] * HD).to(dt), s.f32(rows, case["k_heads"] * HD).to(dt)
        t["pos"], t["inv"] = torch.arange(rows, device="cuda") + int(s.ints(0, 4096, 1)), _rope_inv(HD // 2)
    elif kind == "mlp":
        t["h"] = s.f32(case["rows"], HIDDEN)
        t["gate_up"] = s.bf16(2 * case["ffn"], HIDDEN, scale=0.03)
        t["down"] = s.bf16(HIDDEN, case["ffn"], scale=0.03)
    elif kind == "experts":
        rows, e = case["rows"], case["experts"]
        t["h"] = s.f32(rows, HIDDEN)
        t["gate"] = s.bf16(e * EXPERT_FFN, HIDDEN, scale=0.03)
        t["up"] = s.bf16(e * EXPERT_FFN, HIDDEN, scale=0.03)
        t["down"] = s.bf16(e, HIDDEN, EXPERT_FFN, scale=0.03)
        # each row's experts and weights: a softmax over logits with a spread
        # between the experts, as a gate's loads differ
        score = torch.softmax(s.f32(rows, e) + 0.3 * s.f32(1, e), -1)
        weight, ids = torch.topk(score, TOP_K, -1)
        for j in range(e):
            row, slot = torch.nonzero(ids == j, as_tuple=True)
            t["row%d" % j], t["weight%d" % j] = row.contiguous(), weight[row, slot].contiguous()
    elif kind == "routing":
        rows, first = case["rows"], case["first"]
        keys = first + rows
        nblk = -(-keys // BLOCK)
        t["rq"], t["rk"] = s.f32(rows, ROUTER_D), s.f32(rows, ROUTER_D)
        t["rkeys"] = s.f32(keys, ROUTER_D)
        t["rqn"], t["rkn"], t["cls"] = s.f32(ROUTER_D, scale=0.1), s.f32(ROUTER_D, scale=0.1), s.f32(ROUTER_D)
        t["inv_tok"], t["inv_page"] = _tables()
        t["tok"] = torch.arange(first, keys, device="cuda")
        t["page"] = t["tok"] // 257
        # the scores the mask is made from are given, so that the mask's
        # choices do not hang on the last bit of the scores product
        t["z_given"] = s.f32(rows, nblk)
        t["blocks"] = torch.arange(nblk, device="cuda") // 8
        t["query_page"] = torch.where(s.ints(0, 4, rows) == 0, t["tok"] // 256 // 2, -1)
        t["h"], t["gate"] = s.f32(rows, HIDDEN), s.f32(EXPERTS, HIDDEN, scale=0.05)
    elif kind == "attention":
        rows, first, heads, hd = case["rows"], case["first"], case["heads"], case["hd"]
        keys = first + rows
        t["q"], t["k"], t["v"] = (s.f32(n, heads * hd) for n in (rows, keys, keys))
        t["mask"] = None if case["mask"] == "none" else _mask(s, case["mask"], rows, first)
    elif kind == "products":
        rows, keys, width = case["rows"], case["rows"] + case["first"], case["heads"] * case["hd"]
        t["q"], t["k"], t["v"] = (s.f32(n, width) for n in (rows, keys, keys))
        t["mask"] = _mask(s, "causal", rows, case["first"])
    elif kind in ("clip", "sam"):
        c, mlp = (CLIP_W, CLIP_MLP) if kind == "clip" else (SAM_W, SAM_MLP)
        n = case["grid"] ** 2 + (1 if kind == "clip" else 0)
        t["x"] = s.f32(n, c)
        for name in ("ln1", "ln2"):
            t[name + "_w"], t[name + "_b"] = s.norm(c), 0.02 * s.f32(c)
        for name, (o, k) in {"qkv": (3 * c, c), "proj": (c, c), "fc1": (mlp, c), "fc2": (c, mlp)}.items():
            t[name], t[name + "_b"] = s.bf16(o, k, scale=1 / math.sqrt(k)), 0.02 * s.f32(o)
        if kind == "sam":
            side = SAM_WINDOW if case["windowed"] else case["grid"]
            hd = SAM_W // SAM_HEADS
            t["rh"], t["rw"] = s.f32(side, side, hd, scale=0.1), s.f32(side, side, hd, scale=0.1)
            if case["windowed"]:
                t["slots"] = _window_rows(case["grid"])
    else:
        raise ValueError("unknown kind %r" % kind)
    return t


def _mask(s, kind, rows, first):
    """A prompt's key mask [rows, keys]: causal, or routed (the local window of
    4 blocks and 12 earlier blocks a row with a bias each, rows near each
    other choosing much the same blocks)."""
    keys = first + rows
    pos = torch.arange(first, keys, device="cuda")[:, None]
    key = torch.arange(keys, device="cuda")[None, :]
    ninf = float("-inf")
    if kind == "causal":
        return torch.where(key <= pos, 0.0, ninf).float().contiguous()
    nblk = -(-keys // BLOCK)
    groups = torch.arange(rows, device="cuda") // 32
    z = s.f32(int(groups[-1]) + 1, nblk)[groups] + 0.3 * s.f32(rows, nblk)
    blk = torch.arange(nblk, device="cuda")[None, :]
    z = torch.where(blk <= pos // BLOCK - LOCAL, z, ninf)
    top = torch.topk(z, min(TOP_BLOCKS, nblk), -1)
    bias = torch.full((rows, nblk), ninf, device="cuda")
    bias.scatter_(1, top.indices, torch.where(torch.isfinite(top.values), top.values - 1.5, ninf))
    mask = bias.repeat_interleave(BLOCK, 1)[:, :keys]
    mask = torch.where(key > pos - LOCAL * BLOCK, 0.0, mask)
    return torch.where(key <= pos, mask, ninf).float().contiguous()


def _window_rows(g):
    """The grid row of every window slot (window-major), g * g for padding."""
    per = -(-g // SAM_WINDOW)
    y = torch.arange(per * SAM_WINDOW, device="cuda")
    at = torch.where((y[:, None] < g) & (y[None, :] < g), y[:, None] * g + y[None, :], g * g)
    at = at.view(per, SAM_WINDOW, per, SAM_WINDOW).permute(0, 2, 1, 3)
    return at.reshape(-1).contiguous()


# ---- one pass ----------------------------------------------------------------


def prepare(case, seed):
    be = _package()
    t = _inputs(case, seed)
    kind = case["kind"]
    st = {"case": dict(case), "be": be, "t": t}
    if kind == "chain_step":
        st["x"], st["h"] = _empty(case["hidden"], dtype=_dtype(case["dtype"])), _empty(case["hidden"], dtype=_dtype(case["dtype"]))
    elif kind == "decode":
        _prepare_decode(st)
    elif kind == "chain":
        dt = _dtype(case["dtype"])
        st["h"] = _empty(case["rows"], case["hidden"], dtype=dt)
        st["act"] = _empty(case["rows"], case["ffn"], dtype=dt)
    elif kind == "mlp":
        rows, f = case["rows"], case["ffn"]
        st["hb"], st["gu"], st["act"] = _empty(rows, HIDDEN, dtype=torch.bfloat16), _empty(rows, 2 * f), _empty(rows, f)
        st["ab"], st["y"] = _empty(rows, f, dtype=torch.bfloat16), _empty(rows, HIDDEN)
    elif kind == "experts":
        most = max(t["row%d" % e].numel() for e in range(case["experts"]))
        st["in"], st["g"], st["u"], st["res"] = (_empty(most * n) for n in (HIDDEN, EXPERT_FFN, EXPERT_FFN, HIDDEN))
        st["inb"], st["gb"] = (_empty(most * n, dtype=torch.bfloat16) for n in (HIDDEN, EXPERT_FFN))
        st["out"] = _empty(case["rows"], HIDDEN)
        st["rows_of"] = [t["row%d" % e].numel() for e in range(case["experts"])]
    elif kind == "routing":
        rows, keys = case["rows"], case["rows"] + case["first"]
        nblk = -(-keys // BLOCK)
        st["summ"], st["z"], st["mask"] = _empty(nblk, ROUTER_D), _empty(rows, nblk), _empty(rows, keys)
        st["logits"] = _empty(rows, EXPERTS)
        st["ids"], st["wts"] = _empty(rows, TOP_K, dtype=torch.int64), _empty(rows, TOP_K)
        st["params"] = be.RouteParams()
    elif kind == "attention":
        rows, keys, heads, hd = case["rows"], case["rows"] + case["first"], case["heads"], case["hd"]
        st["out"] = _empty(rows, heads * hd, dtype=_dtype(case["out"]))
        st["ws"] = _empty(be.attention_workspace_floats(heads, rows, keys, hd)) if case["workspace"] else None
    elif kind == "products":
        rows, keys, heads = case["rows"], case["rows"] + case["first"], case["heads"]
        st["scores"], st["out"] = _empty(heads, rows, keys), _empty(rows, heads * case["hd"])
    else:
        _prepare_vision(st)
    return st


def run(state):
    return _RUN[state["case"]["kind"]](state, state["be"], state["t"], state["case"])


def _run_chain_step(st, be, t, case):
    be.embed_add_rms_norm_step(t["table"], t["step"], t["w"], st["x"], st["h"], t["delta"], EPS)
    be.rope_qk_step(t["q"], case["q_heads"], t["k"], case["k_heads"], HD, t["step"], t["inv"], None, 0)
    return {"x": st["x"], "h": st["h"], "q": t["q"], "k": t["k"]}


def _prepare_decode(st):
    """The layer's buffers and its captured step."""
    be, t, case = st["be"], st["t"], st["case"]
    width, moe = HEADS * HD, case["moe"]
    f = SHARED_FFN if moe else DENSE_FFN
    st.update(x1=_empty(HIDDEN), x2=_empty(HIDDEN), proj=_empty(t["proj"].shape[0]), o=_empty(HIDDEN), act=_empty(f),
              delta=_empty(HIDDEN))
    q, k, v = (st["proj"][i * width:(i + 1) * width] for i in range(3))
    scale = 1.0 / math.sqrt(HD)
    if moe:
        params = be.RouteParams(BLOCK, LOCAL, TOP_M, TOP_BLOCKS)
        max_live = (TOP_BLOCKS + LOCAL) * BLOCK
        rq, rk = st["proj"][3 * width:3 * width + ROUTER_D], st["proj"][3 * width + ROUTER_D:]
        st.update(segs=_empty(be.KEY_SEGMENT_WORDS, dtype=torch.int32), h=_empty(HIDDEN), logits=_empty(EXPERTS),
                  ids=_empty(TOP_K, dtype=torch.int64), wts=_empty(TOP_K),
                  scratch=_empty(be.attend_segments_scratch_floats(HEADS, HD, max_live)),
                  escratch=_empty(be.expert_scratch_floats(TOP_K, EXPERT_FFN)))
    else:
        st.update(attn=_empty(width), logits=_empty(VOCAB),
                  scratch=_empty(be.attend_scratch_floats(HEADS, HD, case["cap"])))

    def step():
        be.add_rms_norm_gemv_bf16(t["x"], t["proj"], st["proj"], delta=t["delta"], x_out=st["x1"], w_norm=t["in"],
                                  eps=EPS)
        if moe:
            be.route_decode_step(rq, rk, t["rqn"], t["rkn"], EPS, t["inv_tok"], t["inv_page"], PAGE_MOD, t["cls"],
                                 t["rkeys"], t["summ"], t["pages"], t["pages"], t["step"], params, None,
                                 segments=st["segs"])
            be.attend_rope_kv_step_segments(q, k, v, t["kc"], t["vc"], HEADS, HD, st["segs"], max_live, scale,
                                            t["step"], t["inv_tok"], t["inv_page"], PAGE_MOD, st["scratch"], None)
            be.attend_merge_gemv_bf16(st["scratch"], HEADS, HD, max_live, t["o"], st["o"])
            be.add_rms_norm_swiglu_router_gemv_bf16(st["x1"], t["gate"], t["up"], st["act"], t["router"], st["logits"],
                                                    delta=st["o"], x_out=st["x2"], w_norm=t["post"], eps=EPS,
                                                    h_out=st["h"])
            be.moe_ffn_one(st["h"], t["gs"], t["us"], t["ds"], st["logits"], st["ids"], st["wts"], st["act"],
                           t["down"], st["escratch"], st["delta"])
        else:
            be.attend_rope_kv_step(q, k, v, t["kc"], t["vc"], HEADS, HD, None, scale, t["step"], t["inv_tok"],
                                   t["inv_page"], PAGE_MOD, st["scratch"], st["attn"])
            be.gemv_bf16(st["attn"], t["o"], st["o"])
            be.add_rms_norm_swiglu_gemv_bf16(st["x1"], t["gate"], t["up"], st["act"], delta=st["o"], x_out=st["x2"],
                                             w_norm=t["post"], eps=EPS)
            be.gemv_bf16(st["act"], t["down"], st["delta"])
            be.add_rms_norm_gemv_bf16(st["x2"], t["lm"], st["logits"], delta=st["delta"], w_norm=t["final"], eps=EPS)

    torch.cuda.synchronize()
    st["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(st["graph"]):
        step()


def _run_decode(st, be, t, case):
    st["graph"].replay()
    out = {"x": st["x2"], "delta": st["delta"], "logits": st["logits"], "k": t["kc"], "v": t["vc"]}
    if case["moe"]:
        out.update(router_keys=t["rkeys"], ids=st["ids"], weights=st["wts"])
    return out


def _run_chain(st, be, t, case):
    be.add_rms_norm(t["x"], t["delta"], t["w"], st["h"], EPS)
    be.swiglu(t["gu"], st["act"])
    be.rope_qk(t["q"], case["q_heads"], t["k"], case["k_heads"], HD, t["pos"], None, t["inv"], None, 0)
    return {"x": t["x"], "h": st["h"], "act": st["act"], "q": t["q"], "k": t["k"]}


def _run_mlp(st, be, t, case):
    be.round_bf16(t["h"], st["hb"])
    be.linear(st["hb"], t["gate_up"], st["gu"])
    be.swiglu(st["gu"], st["act"])
    be.round_bf16(st["act"], st["ab"])
    be.linear(st["ab"], t["down"], st["y"])
    return {"y": st["y"]}


def _run_experts(st, be, t, case):
    st["out"].zero_()
    for e, n in enumerate(st["rows_of"]):
        if n == 0:
            continue
        w = slice(e * EXPERT_FFN, (e + 1) * EXPERT_FFN)
        row = t["row%d" % e]
        x, g, u, res = (st[k][:n * c].view(n, c) for k, c in
                        (("in", HIDDEN), ("g", EXPERT_FFN), ("u", EXPERT_FFN), ("res", HIDDEN)))
        xb, gb = (st[k][:n * c].view(n, c) for k, c in (("inb", HIDDEN), ("gb", EXPERT_FFN)))
        be.gather_rows(t["h"], row, x)
        be.round_bf16(x, xb)
        be.linear(xb, t["gate"][w], g)
        be.linear(xb, t["up"][w], u)
        be.silu_mul(g, u)
        be.round_bf16(g, gb)
        be.linear(gb, t["down"][e], res)
        be.scatter_add_rows(st["out"], row, t["weight%d" % e], res)
    return {"out": st["out"]}


def _run_routing(st, be, t, case):
    rows, first = case["rows"], case["first"]
    keys = first + rows
    nblk = -(-keys // BLOCK)
    for x, w in ((t["rq"], t["rqn"]), (t["rk"], t["rkn"])):
        be.router_norm(x, w, EPS)
        be.rope(x, 1, ROUTER_D, t["tok"], t["page"], t["inv_tok"], t["inv_page"], PAGE_MOD)
    be.block_summaries(t["rkeys"], t["cls"], BLOCK, st["summ"])
    be.gemm_nt(rows, nblk, ROUTER_D, 1.0 / math.sqrt(ROUTER_D), t["rq"], ROUTER_D, 0, st["summ"], ROUTER_D, 0, st["z"],
               nblk, 0)
    be.route_blocks(t["z_given"], first, keys, t["blocks"], t["blocks"], t["query_page"], -1, st["params"], st["mask"])
    be.gemm_nt(rows, EXPERTS, HIDDEN, 1.0, t["h"], HIDDEN, 0, t["gate"], HIDDEN, 0, st["logits"], EXPERTS, 0)
    be.expert_topk(st["logits"], TOP_K, st["ids"], st["wts"])
    return {"rq": t["rq"], "rk": t["rk"], "summaries": st["summ"], "z": st["z"], "mask": st["mask"],
            "logits": st["logits"], "ids": st["ids"], "weights": st["wts"]}


def _run_attention(st, be, t, case):
    rows, keys, heads, hd = case["rows"], case["rows"] + case["first"], case["heads"], case["hd"]
    at = (0, heads * hd, hd)  # each head's columns in place
    be.attention(t["q"], t["k"], t["v"], st["out"], heads, rows, keys, hd, 1.0 / math.sqrt(hd), t["mask"],
                 strides={"q": at, "k": at, "v": at, "out": at}, workspace=st["ws"])
    return {"out": st["out"]}


def _run_products(st, be, t, case):
    rows, keys, heads, hd = case["rows"], case["rows"] + case["first"], case["heads"], case["hd"]
    w = heads * hd
    be.gemm_nt(rows, keys, hd, 1.0, t["q"], w, hd, t["k"], w, hd, st["scores"], keys, rows * keys, heads)
    be.scale_mask_softmax_rows(st["scores"], 1.0 / math.sqrt(hd), t["mask"], heads, rows, keys)
    be.gemm_nn(rows, hd, keys, st["scores"], keys, rows * keys, t["v"], w, hd, st["out"], w, hd, heads)
    return {"scores": st["scores"], "out": st["out"]}


def _prepare_vision(st):
    be, t, case = st["be"], st["t"], st["case"]
    n, c = t["x"].shape
    mlp = t["fc1"].shape[0]
    rows = t["slots"].numel() if "slots" in t else n
    if "slots" in t:
        st["normed"] = torch.zeros(n + 1, c, dtype=torch.bfloat16, device="cuda")  # the last row: windows' padding
        st["in"] = _empty(rows, c, dtype=torch.bfloat16)
    else:
        st["in"] = _empty(n, c, dtype=torch.bfloat16)
    st["h"] = _empty(n, c, dtype=torch.bfloat16)
    st["qkv"], st["merged"] = _empty(rows, 3 * c), _empty(rows, c, dtype=torch.bfloat16)
    st["wide"], st["act"] = _empty(n, mlp), _empty(n, mlp, dtype=torch.bfloat16)
    shapes = [(rows, c, 3 * c), (n, c, c), (n, c, mlp), (n, mlp, c)]
    st["ws"] = _empty(max([1] + [be.linear_workspace_floats(*s) for s in shapes]))
    if case["kind"] == "sam":
        side = t["rh"].shape[0]
        slices = SAM_HEADS * (rows // (side * side))
        st["dots"] = _empty(max(1, be.attention_rel_pos_workspace_floats(slices, side, side)))


def _run_vision(st, be, t, case):
    x, ws = t["x"], st["ws"]
    n, c = x.shape
    if case["kind"] == "sam" and case["windowed"]:
        be.layer_norm_to_bf16(x, t["ln1_w"], t["ln1_b"], st["normed"][:n], EPS)
        be.gather_rows(st["normed"].view(torch.float32), t["slots"], st["in"].view(torch.float32))
    else:
        be.layer_norm_to_bf16(x, t["ln1_w"], t["ln1_b"], st["in"], EPS)
    be.linear_ws(st["in"], t["qkv"], st["qkv"], ws, t["qkv_b"])
    if case["kind"] == "clip":
        hd = c // CLIP_HEADS
        q, k, v = st["qkv"], st["qkv"].view(-1)[c:], st["qkv"].view(-1)[2 * c:]
        at = (0, 3 * c, hd)
        be.attention(q, k, v, st["merged"], CLIP_HEADS, n, n, hd, 1.0 / math.sqrt(hd),
                     strides={"q": at, "k": at, "v": at, "out": (0, c, hd)})
    else:
        hd, side = c // SAM_HEADS, t["rh"].shape[0]
        be.attention_rel_pos_windows(st["qkv"], st["merged"], SAM_HEADS, st["qkv"].shape[0] // (side * side), side,
                                     side, hd, 1.0 / math.sqrt(hd), t["rh"], t["rw"], st["dots"])
    if "slots" in t:
        be.linear_add_rows(st["merged"], t["proj"], x, t["slots"], t["proj_b"])
    else:
        be.linear_add(st["merged"], t["proj"], x, ws, t["proj_b"])
    quick = case["kind"] == "clip"
    be.layer_norm_to_bf16(x, t["ln2_w"], t["ln2_b"], st["h"], EPS)
    if n >= 128:
        be.linear_ws(st["h"], t["fc1"], st["wide"], ws, t["fc1_b"])
        be.act_to_bf16(st["wide"], st["act"], quick)
    else:
        be.linear_act(st["h"], t["fc1"], st["act"], t["fc1_b"], quick)
    be.linear_add(st["act"], t["fc2"], x, ws, t["fc2_b"])
    return {"x": x, "qkv": st["qkv"], "attention": st["merged"]}


_RUN = {"chain_step": _run_chain_step, "decode": _run_decode, "chain": _run_chain, "mlp": _run_mlp,
        "experts": _run_experts, "routing": _run_routing, "attention": _run_attention, "products": _run_products,
        "clip": _run_vision, "sam": _run_vision}


# ---- what a pass cannot do without ----------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "chain_step":
        e, n = 2 if case["dtype"] == "bf16" else 4, case["hidden"]
        return {"bytes": 2 * n + 4 * n + 3 * e * n + 2 * e * HD * (case["q_heads"] + case["k_heads"]), "flops": 6 * n}
    if kind == "decode":
        e, w = 2 if case["cache"] == "bf16" else 4, HEADS * HD
        moe = case["moe"]
        live = min(case["pos"] + 1, (TOP_BLOCKS + LOCAL) * BLOCK) if moe else case["pos"] + 1
        weights = HIDDEN * (3 * w + w)
        if moe:
            weights += HIDDEN * (2 * ROUTER_D + 3 * SHARED_FFN + 3 * TOP_K * EXPERT_FFN)
        else:
            weights += HIDDEN * (3 * DENSE_FFN + VOCAB)
        other = 4 * EXPERTS * HIDDEN + 4 * ROUTER_D * (case["pos"] // BLOCK + BLOCK) if moe else 4 * VOCAB
        return {"bytes": 2 * weights + 2 * e * live * w + other, "flops": 2 * weights + 4 * live * w}
    if kind == "chain":
        e, rows = 2 if case["dtype"] == "bf16" else 4, case["rows"]
        per = 4 * case["hidden"] + 3 * case["ffn"] + 2 * HD * (case["q_heads"] + case["k_heads"])
        return {"bytes": rows * (e * per + 8), "flops": 5 * rows * per}
    if kind == "mlp":
        rows, f = case["rows"], case["ffn"]
        return {"bytes": 8 * rows * HIDDEN + 6 * f * HIDDEN, "flops": 6 * rows * f * HIDDEN}
    if kind == "experts":
        rows, e = case["rows"], case["experts"]
        return {"bytes": 8 * rows * HIDDEN + 6 * e * EXPERT_FFN * HIDDEN + 12 * rows * TOP_K,
                "flops": 6 * rows * TOP_K * EXPERT_FFN * HIDDEN}
    if kind == "routing":
        rows, keys = case["rows"], case["rows"] + case["first"]
        nblk = -(-keys // BLOCK)
        return {"bytes": 4 * (4 * rows * ROUTER_D + keys * ROUTER_D + 2 * rows * nblk + rows * keys
                              + rows * (HIDDEN + EXPERTS + 3 * TOP_K)),
                "flops": 2 * rows * (nblk * ROUTER_D + EXPERTS * HIDDEN) + 4 * keys * ROUTER_D}
    if kind in ("attention", "products"):
        rows, first, heads, hd = case["rows"], case["first"], case["heads"], case["hd"]
        keys = rows + first
        mask = case.get("mask", "causal")
        if mask == "none":
            live = rows * keys
        else:
            live = rows * first + rows * (rows + 1) // 2
            if mask == "routed":
                live = sum(min(p + 1, (TOP_BLOCKS + LOCAL) * BLOCK) for p in range(first, keys))
        e = 2 if case.get("out") == "bf16" else 4
        nbytes = heads * hd * (4 * rows + 8 * keys + e * rows) + (0 if mask == "none" else 4 * rows * keys)
        if kind == "products":
            nbytes += 4 * heads * rows * keys
        return {"bytes": nbytes, "flops": 4 * heads * hd * live}
    c, mlp, heads = (CLIP_W, CLIP_MLP, CLIP_HEADS) if kind == "clip" else (SAM_W, SAM_MLP, SAM_HEADS)
    n = case["grid"] ** 2 + (1 if kind == "clip" else 0)
    keys = SAM_WINDOW ** 2 if case.get("windowed") else n
    return {"bytes": 8 * n * c + 12 * n * c + 2 * n * c + 2 * c * (4 * c + 2 * mlp),
            "flops": 2 * n * c * (4 * c + 2 * mlp) + 4 * n * keys * c}


# Stated from what `exact` showed (about four times the error of the ops
# against 64 bits): one bf16 rounding is about 1.7e-3 in the 2-norm, fp32
# sums stay near 1e-6.
_TOLERANCE = {"chain_step": {"bf16": {"rel": 7e-3, "max": 4e-2}, "f32": {"rel": 4e-6, "max": 1e-4}},
              "chain": {"bf16": {"rel": 7e-3, "max": 4e-2}, "f32": {"rel": 4e-6, "max": 1e-4}}}


def tolerance(case):
    kind = case["kind"]
    if kind in _TOLERANCE:
        return _TOLERANCE[kind][case["dtype"]]
    if kind == "routing":  # ids: two experts whose scores meet in the last bits
        return {"rel": 8e-6, "max": 1e-4, "differ": 1e-3}
    if kind == "products" or (kind == "attention" and case["out"] == "f32"):
        return {"rel": 8e-6, "max": 1e-4}
    if kind == "attention":
        return {"rel": 7e-3, "max": 4e-2}
    # layers of several products: an fp32 sum's last bit moves a bf16 rounding
    # of the next product's input (4e-5 against 64 bits over a whole MLP); the
    # vision layers return the attention in bf16 beside their rows
    if kind in ("clip", "sam"):
        return {"rel": 7e-3, "max": 5e-2}
    if kind == "decode":  # one moved rounding of the attention row reaches every later product: 1.6e-3
        return {"rel": 6e-3, "max": 5e-2, "differ": 0.0}
    return {"rel": 2e-4, "max": 2e-2}


# ---- the same outputs in 64 bits ----------------------------------------------------


def _r(x):
    """The nearest bf16 values, in 64 bits."""
    return x.float().to(torch.bfloat16).double()


def _mm(x, w):
    """bf16(x) . w^T in 64 bits."""
    return _r(x) @ w.double().T


def _rms(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def _layer_norm(x, w, b):
    d = x - x.mean(-1, keepdim=True)
    return d * torch.rsqrt(d.pow(2).mean(-1, keepdim=True) + EPS) * w.double() + b.double()


def _router_norm(x, w):
    n = (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS)).clamp(-1e4, 1e4)
    return (n * (1 + w.double())).clamp(-1e4, 1e4)


def _angles(tok, inv_tok, page=None, inv_page=None, page_mod=0):
    """Rotation angles [rows, pairs]: fp32 products, then 64 bits."""
    a = (tok.float()[:, None] * inv_tok).double()
    if inv_page is None:
        return a
    return torch.cat([a, ((page % page_mod).float()[:, None] * inv_page).double()], -1)


def _rotate(x, heads, ang):
    v = x.double().view(ang.shape[0], heads, 2, -1)
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    return torch.stack([v[:, :, 0] * c - v[:, :, 1] * s, v[:, :, 1] * c + v[:, :, 0] * s], 2).reshape(x.shape)


def _silu(x):
    return x * torch.sigmoid(x)


def _gelu(x, quick=False):
    return x * torch.sigmoid(1.702 * x) if quick else 0.5 * x * (1 + torch.erf(x / math.sqrt(2.0)))


def _attend(q, k, v, scale, bias=None):
    """softmax(scale q k^T + bias) v for one head, rows in parts."""
    out = torch.empty(q.shape[0], v.shape[1], dtype=torch.float64, device="cuda")
    for at in range(0, q.shape[0], 1024):
        s = scale * (q[at:at + 1024] @ k.T)
        if bias is not None:
            s += bias[at:at + 1024]
        out[at:at + 1024] = torch.softmax(s, -1).nan_to_num(0.0) @ v
    return out


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    return {"chain_step": _exact_chain_step, "decode": _exact_decode, "chain": _exact_chain, "mlp": _exact_mlp,
            "experts": _exact_experts, "routing": _exact_routing, "attention": _exact_attention,
            "products": _exact_products, "clip": _exact_vision, "sam": _exact_vision}[kind](case, t)


def _exact_chain_step(case, t):
    step = t["step"]
    x = t["table"][step[0]].double() + t["delta"].double()
    x32 = x.float().to(t["delta"].dtype).double()  # the stored x is rounded; h is formed from the sum
    ang = _angles(step[2:3], t["inv"])
    return {"x": x32, "h": _rms(x, t["w"]), "q": _rotate(t["q"][None], case["q_heads"], ang)[0],
            "k": _rotate(t["k"][None], case["k_heads"], ang)[0]}


def _exact_chain(case, t):
    x = t["x"].double() + t["delta"].double()
    f = case["ffn"]
    gu = t["gu"].double()
    ang = _angles(t["pos"], t["inv"])
    return {"x": x, "h": _rms(x, t["w"]), "act": _silu(gu[:, :f]) * gu[:, f:],
            "q": _rotate(t["q"], case["q_heads"], ang), "k": _rotate(t["k"], case["k_heads"], ang)}


def _exact_mlp(case, t):
    f = case["ffn"]
    gu = _mm(t["h"], t["gate_up"])
    return {"y": _mm(_silu(gu[:, :f]) * gu[:, f:], t["down"])}


def _exact_experts(case, t):
    out = torch.zeros(case["rows"], HIDDEN, dtype=torch.float64, device="cuda")
    for e in range(case["experts"]):
        row, w = t["row%d" % e], slice(e * EXPERT_FFN, (e + 1) * EXPERT_FFN)
        if row.numel():
            x = t["h"][row]
            y = _mm(_silu(_mm(x, t["gate"][w])) * _mm(x, t["up"][w]), t["down"][e])
            out[row] += t["weight%d" % e].double()[:, None] * y
    return {"out": out}


def _summaries(keys, cls):
    """Per block of 32 keys the softmax(k . cls / sqrt d)-weighted mean."""
    n, d = keys.shape
    nblk = -(-n // BLOCK)
    a = ((keys @ cls.double()) / math.sqrt(d)).clamp(-1e4, 1e4)
    pad = nblk * BLOCK - n
    a = torch.cat([a, a.new_full((pad,), float("-inf"))]).view(nblk, BLOCK)
    p = torch.softmax(a, -1)
    return torch.einsum("bt,btd->bd", p, torch.cat([keys, keys.new_zeros(pad, d)]).view(nblk, BLOCK, d))


def _select(z, remote, allowed):
    """The blocks a row reads and their biases, rows of scores z [rows, nblk]
    in 64 bits: the top 16 candidates through 1.5-entmax, the first 12 kept
    with log-probability biases about their mean; -inf elsewhere."""
    rows, nblk = z.shape
    cand = remote & allowed
    cand = torch.where(cand.any(-1, keepdim=True), cand, remote)
    x = torch.where(cand, z * math.sqrt(128.0), -1e4)
    m = max(1, min(TOP_M, nblk))
    k = max(1, min(TOP_BLOCKS, m))
    top, at = torch.sort(x, dim=-1, descending=True, stable=True)
    top, at = top[:, :m], at[:, :m]
    v = (top - top[:, :1]) / 2
    rho = torch.arange(1, m + 1, device="cuda", dtype=torch.float64)
    mean, sq = v.cumsum(-1) / rho, (v * v).cumsum(-1) / rho
    tau = mean - torch.sqrt(((1 - rho * (sq - mean * mean)) / rho).clamp_min(0))
    support = (tau <= v).sum(-1, keepdim=True).clamp_min(1)
    p = (v - tau.gather(1, support - 1)).clamp_min(0) ** 2
    at, p = at[:, :k], p[:, :k]
    valid = cand.gather(1, at)
    logp = torch.log(p.clamp_min(np.float64(np.float32(1e-4))))
    mu = (logp * valid).sum(-1, keepdim=True) / valid.sum(-1, keepdim=True).clamp_min(1)
    bias = torch.full((rows, nblk), float("-inf"), dtype=torch.float64, device="cuda")
    bias.scatter_(1, at, torch.where(valid, logp - mu, float("-inf")))
    return bias


def _key_mask(bias, pos, keys):
    key = torch.arange(keys, device="cuda")[None, :]
    mask = bias.repeat_interleave(BLOCK, 1)[:, :keys]
    mask = torch.where(key > pos - LOCAL * BLOCK, 0.0, mask)
    return torch.where(key <= pos, mask, float("-inf"))


def _exact_routing(case, t):
    rows, first = case["rows"], case["first"]
    keys = first + rows
    ang = _angles(t["tok"], t["inv_tok"], t["page"], t["inv_page"], PAGE_MOD)
    rq = _rotate(_router_norm(t["rq"].double(), t["rqn"]), 1, ang)
    rk = _rotate(_router_norm(t["rk"].double(), t["rkn"]), 1, ang)
    summ = _summaries(t["rkeys"].double(), t["cls"])
    pos = torch.arange(first, keys, device="cuda")[:, None]
    blk = torch.arange(-(-keys // BLOCK), device="cuda")[None, :]
    page = t["query_page"][:, None]
    known = t["blocks"][None, :]
    allowed = (page < 0) | (known == page)
    bias = _select(t["z_given"].double(), blk <= pos // BLOCK - LOCAL, allowed)
    logits = t["h"].double() @ t["gate"].double().T
    w, ids = torch.topk(torch.softmax(logits, -1), TOP_K, -1)
    return {"rq": rq, "rk": rk, "summaries": summ, "z": rq @ summ.T / math.sqrt(ROUTER_D),
            "mask": _key_mask(bias, pos, keys), "logits": logits, "ids": ids, "weights": w}


def _exact_attention(case, t):
    heads, hd = case["heads"], case["hd"]
    bias = None if t["mask"] is None else t["mask"].double()
    at = [slice(h * hd, (h + 1) * hd) for h in range(heads)]
    return {"out": torch.cat([_attend(t["q"][:, c].double(), t["k"][:, c].double(), t["v"][:, c].double(),
                                      1.0 / math.sqrt(hd), bias) for c in at], 1)}


def _exact_products(case, t):
    heads, hd = case["heads"], case["hd"]
    at = [slice(h * hd, (h + 1) * hd) for h in range(heads)]
    p = torch.stack([torch.softmax(t["q"][:, c].double() @ t["k"][:, c].double().T / math.sqrt(hd)
                                   + t["mask"].double(), -1) for c in at])
    return {"scores": p, "out": torch.cat([p[h] @ t["v"][:, c].double() for h, c in enumerate(at)], 1)}


def _exact_vision(case, t):
    clip = case["kind"] == "clip"
    x = t["x"].double()
    n, c = x.shape
    heads = CLIP_HEADS if clip else SAM_HEADS
    hd = c // heads
    normed = _layer_norm(x, t["ln1_w"], t["ln1_b"])
    if "slots" in t:
        normed = torch.cat([normed, normed.new_zeros(1, c)])[t["slots"]]
    qkv = _mm(normed, t["qkv"]) + t["qkv_b"].double()
    side = None if clip else t["rh"].shape[0]
    per = n if clip else side * side
    merged = torch.empty(qkv.shape[0], c, dtype=torch.float64, device="cuda")
    for at in range(0, qkv.shape[0], per):
        for h in range(heads):
            q, k, v = (qkv[at:at + per, i * c + h * hd:i * c + (h + 1) * hd] for i in range(3))
            bias = None
            if not clip:
                g = q.view(side, side, hd)
                bh = torch.matmul(g, t["rh"].double().transpose(1, 2).contiguous())  # [y, x, ky]
                bw = torch.matmul(g.transpose(0, 1).contiguous(), t["rw"].double().transpose(1, 2).contiguous())
                bias = (bh[:, :, :, None] + bw.transpose(0, 1)[:, :, None, :]).reshape(per, per)
            merged[at:at + per, h * hd:(h + 1) * hd] = _attend(q, k, v, 1.0 / math.sqrt(hd), bias)
    y = _mm(merged, t["proj"]) + t["proj_b"].double()
    if "slots" in t:
        kept = t["slots"] < n
        x = x.index_add(0, t["slots"][kept], y[kept])
    else:
        x = x + y
    act = _gelu(_mm(_layer_norm(x, t["ln2_w"], t["ln2_b"]), t["fc1"]) + t["fc1_b"].double(), clip)
    return {"x": x + _mm(act, t["fc2"]) + t["fc2_b"].double(), "qkv": qkv, "attention": merged}


def _exact_decode(case, t):
    pos, moe, w = case["pos"], case["moe"], HEADS * HD
    x1 = t["x"].double() + t["delta"].double()
    proj = _mm(_rms(x1, t["in"])[None], t["proj"])[0]
    step = t["step"]
    ang = _angles(step[2:3], t["inv_tok"], step[3:4], t["inv_page"], PAGE_MOD)
    q, k = (_rotate(proj[None, i * w:(i + 1) * w], HEADS, ang)[0] for i in range(2))
    kc, vc = t["kc"].double(), t["vc"].double()
    kc[pos], vc[pos] = (_r(k), _r(proj[2 * w:3 * w])) if case["cache"] == "bf16" else (k, proj[2 * w:3 * w])
    bias, extra = None, {}
    if moe:
        rq = _rotate(_router_norm(proj[None, 3 * w:3 * w + ROUTER_D], t["rqn"]), 1, ang)
        rkeys = t["rkeys"].double()
        rkeys[pos] = _rotate(_router_norm(proj[None, 3 * w + ROUTER_D:], t["rkn"]), 1, ang)[0]
        nblk = pos // BLOCK + 1
        summ = t["summ"].double()[:nblk]
        summ[nblk - 1] = _summaries(rkeys[(nblk - 1) * BLOCK:pos + 1], t["cls"])[0]
        z = (rq @ summ.T / math.sqrt(ROUTER_D)).clamp(-1e4, 1e4)
        blk = torch.arange(nblk, device="cuda")[None, :]
        known = torch.full((1, nblk), -1, device="cuda")
        m = min(nblk, t["pages"].numel())
        known[0, :m] = t["pages"][:m]
        bias = _key_mask(_select(z, blk <= pos // BLOCK - LOCAL, known == step[4]), pos, pos + 1)
        extra["router_keys"] = rkeys
    attn = torch.cat([_attend(q[None, h * HD:(h + 1) * HD], kc[:pos + 1, h * HD:(h + 1) * HD],
                              vc[:pos + 1, h * HD:(h + 1) * HD], 1.0 / math.sqrt(HD), bias)[0] for h in range(HEADS)])
    x2 = x1 + _mm(attn[None], t["o"])[0]
    h = _rms(x2, t["post"])
    act = _silu(_mm(h[None], t["gate"])[0]) * _mm(h[None], t["up"])[0]
    delta = _mm(act[None], t["down"])[0]
    if moe:
        logits = t["router"].double() @ h
        weights, ids = torch.topk(torch.softmax(logits, -1), TOP_K)
        for p, e in zip(weights.tolist(), ids.tolist()):
            at = slice(e * EXPERT_FFN, (e + 1) * EXPERT_FFN)
            a = _silu(_mm(h[None], t["gs"][at])) * _mm(h[None], t["us"][at])
            delta = delta + p * _mm(a, t["ds"][e])[0]
        extra.update(ids=ids, weights=weights)
    else:
        logits = _mm(_rms(x2 + delta, t["final"])[None], t["lm"])[0]
    return {"x": x2, "delta": delta, "logits": logits, "k": kc, "v": vc, **extra}
