"""Timed cases of the framework: draft tree build, one decoder layer of the
tree-verify step (full attention and GatedDeltaNet), the prompt prefill and its
blocks, and a whole verify forward, each through public entry points.

Model geometries are the package's own configurations (QWEN3_4B, QWEN35_4B,
QWEN35_9B) cut to the layers a case runs; vocabularies of layer cases are cut
to 4096, since they are about the layers. Weights are seeded: linear weights
N(0, 0.02) in bf16, or the same quantised to 4-bit groups of 64.

`exact` is plain torch in float64. The KV cache is a bf16 format, so attention
reads keys and values rounded to bf16 there as well.
"""
import math
import random
import sys
from dataclasses import replace
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parent.parent / "dtree-mlx_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import ctypes as C  # noqa: E402

from dtree_hip import QWEN35_4B, QWEN35_9B, QWEN3_4B  # noqa: E402
from dtree_hip import Qwen35TargetAdapter, Qwen35TreeModel, Qwen3TargetAdapter, Qwen3TreeModel  # noqa: E402
from dtree_hip import Qwen35Weights, Qwen3Weights  # noqa: E402
from dtree_hip import _native as N  # noqa: E402
from dtree_hip.weights import (W_TILED, W_TILED_F16, GdnLayerWeights, LayerWeights, Q4Linear,  # noqa: E402
                               interleave_gate_up, q4_to_tiled, tile_weight_f16)

MODELS = {"qwen3-4b": QWEN3_4B, "qwen35-4b": QWEN35_4B, "qwen35-9b": QWEN35_9B}
LAYER_VOCAB = 4096
F64 = torch.float64


# ---- the cases -------------------------------------------------------------------
def listed():
    return [
        # The smallest call: the draft tree of one decode step (15 draft rows,
        # 24 draft nodes) from the drafter's logits.
        dict(name="tree_build_d15_b24", kind="tree", depth=15, vocab=151936, budget=24),
        # One decoder layer of the tree-verify step, the decode loop's work:
        # a 25-node tree over a 1024-key prefix in bf16, the same model with
        # q4 weights over a shorter prefix, and the hybrid models' gated
        # attention and GatedDeltaNet layers (25 nodes in bf16; 65 nodes in q4,
        # the attention over a long prefix).
        dict(name="verify_attn_4b_bf16_25n", kind="layer", model="qwen3-4b", mixer="attn", quant="bf16", nodes=25,
             past=1024),
        dict(name="verify_attn_4b_q4_25n", kind="layer", model="qwen3-4b", mixer="attn", quant="q4", nodes=25,
             past=509),
        dict(name="verify_gated_9b_q4_65n_p8192", kind="layer", model="qwen35-9b", mixer="attn", quant="q4", nodes=65,
             past=8192),
        dict(name="verify_gdn_4b_bf16_25n", kind="layer", model="qwen35-4b", mixer="gdn", quant="bf16", nodes=25,
             past=2048),
        dict(name="verify_gdn_9b_q4_65n", kind="layer", model="qwen35-9b", mixer="gdn", quant="q4", nodes=65,
             past=8192),
        # The compute-bound blocks of a prompt's prefill: the MLP of a
        # 1024-token segment in bf16, of a short ragged prompt in q4, and a
        # GatedDeltaNet layer's core over a 1024-token segment.
        dict(name="prefill_mlp_4b_bf16_1024", kind="mlp", model="qwen3-4b", quant="bf16", tokens=1024),
        dict(name="prefill_mlp_9b_q4_300", kind="mlp", model="qwen35-9b", quant="q4", tokens=300),
        dict(name="prefill_gdn_chain_1024", kind="chain", model="qwen35-4b", tokens=1024),
        # A prompt through the adapter: one full-attention layer over a ragged
        # 1000-token prompt, and one period of the q4 hybrid (three
        # GatedDeltaNet layers, one gated attention layer) over 4096 tokens.
        dict(name="prefill_4b_bf16_1000", kind="prompt", model="qwen3-4b", quant="bf16", layers=1, tokens=1000,
             past=0),
        dict(name="prefill_hybrid_9b_q4_4096", kind="prompt", model="qwen35-9b", quant="q4", layers=4, tokens=4096,
             past=0),
        # The whole model once: a verify forward of 36 layers and the logits of
        # every tree node (the sampling path of a decode step).
        dict(name="verify_forward_4b_bf16_25n", kind="step", model="qwen3-4b", quant="bf16", layers=36, nodes=25,
             past=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["tree", "layer", "layer", "layer", "mlp", "mlp", "chain", "prompt", "prompt", "step"])
    quant = rng.choice(["bf16", "q4"])
    if kind == "tree":
        return dict(kind=kind, depth=rng.randint(1, 15), vocab=4 * _log(rng, 1000, 37984),
                    budget=rng.choice([8, 16, 24, 31, 48, 64, 100, 127]))
    if kind == "layer":
        model = rng.choice(list(MODELS))
        mixer = "attn" if model == "qwen3-4b" else rng.choice(["attn", "gdn"])
        return dict(kind=kind, model=model, mixer=mixer, quant=quant,
                    nodes=rng.choice([1, rng.randint(2, 32), rng.randint(17, 32), rng.randint(33, 96)]),
                    past=_log(rng, 1, 8192) - 1)
    if kind == "mlp":
        return dict(kind=kind, model=rng.choice(list(MODELS)), quant=quant, tokens=_log(rng, 100, 4096))
    if kind == "chain":
        return dict(kind=kind, model="qwen35-4b", tokens=_log(rng, 1, 4096))
    if kind == "prompt":
        model = rng.choice(list(MODELS))
        full = model == "qwen3-4b"
        return dict(kind=kind, model=model, quant=quant, layers=1 if full else 4, tokens=_log(rng, 128, 3000),
                    past=rng.choice([0, 0, _log(rng, 1, 4096)]) if full else 0)
    return dict(kind="step", model="qwen3-4b", quant=quant, layers=rng.choice([4, 8]), nodes=rng.randint(1, 32),
                past=_log(rng, 1, 4096) - 1)


# ---- seeded inputs (shared by prepare and exact) -----------------------------------
def _gen(seed, *salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + sum((i + 1) * 7919 * s for i, s in enumerate(salt))) % (1 << 62))
    return g


def _normal(g, *shape, std=1.0):
    return torch.empty(*shape, device="cuda").normal_(0.0, std, generator=g)


def _lin_bf16(g, n, k):
    """bf16 [n, k] ~ N(0, 0.02), magnitudes under 2^-17 flushed (exact in fp16)."""
    t = _normal(g, n, k, std=0.02).to(torch.bfloat16)
    return torch.where(t.abs() < 2.0 ** -17, torch.zeros_like(t), t)


def _lin_q4(g, n, k):
    """N(0, 0.02) quantised to 4-bit affine groups of 64: (q, scales, biases)."""
    w = _normal(g, n, k // 64, 64, std=0.02)
    lo, hi = w.amin(-1), w.amax(-1)
    s = ((hi - lo) / 15.0).to(torch.bfloat16)
    b = lo.to(torch.bfloat16)
    q = ((w - b.float().unsqueeze(-1)) / s.float().unsqueeze(-1)).round_().clamp_(0, 15).to(torch.uint8)
    return q.reshape(n, k), s, b


class _Mat:
    """A seeded linear weight: a bf16 matrix or q4 group-64 parts."""

    def __init__(self, g, n, k, quant, zero_rows=0):
        self.quant = quant
        self.parts = _lin_q4(g, n, k) if quant == "q4" else (_lin_bf16(g, n, k),)
        if zero_rows:
            self.parts = tuple(torch.cat([t, t.new_zeros(zero_rows, *t.shape[1:])]) for t in self.parts)

    def exact(self):
        if self.quant != "q4":
            return self.parts[0].to(F64)
        q, s, b = self.parts
        n, k = q.shape
        return (q.to(F64).reshape(n, k // 64, 64) * s.to(F64).unsqueeze(-1) + b.to(F64).unsqueeze(-1)).reshape(n, k)

    def packed(self, up=None):
        """The device layout (with `up`: gate / up rows interleaved)."""
        if self.quant != "q4":
            return tile_weight_f16(self.parts[0] if up is None else interleave_gate_up(self.parts[0], up.parts[0]))

        def words(q):
            v = q.to(torch.int32).reshape(q.shape[0], -1, 8)
            out = v[..., 0].clone()
            for i in range(1, 8):
                out |= v[..., i] << (4 * i)
            return out

        q, s, b = words(self.parts[0]), self.parts[1], self.parts[2]
        if up is not None:
            q = interleave_gate_up(q, words(up.parts[0]))
            s, b = interleave_gate_up(s, up.parts[1]), interleave_gate_up(b, up.parts[2])
        return Q4Linear(*q4_to_tiled(q, s, b))


def _norm_w(g, n):
    return (1.0 + _normal(g, n, std=0.1)).to(torch.bfloat16)


def _layer_mats(cfg, mixer, quant, seed, li):
    """Seeded weights of layer li by name."""
    g = _gen(seed, 11, li)
    H, F = cfg.hidden_size, cfg.intermediate_size
    m = dict(input_norm=_norm_w(g, H), post_norm=_norm_w(g, H))
    if mixer == "gdn":
        Hv = cfg.linear_num_value_heads
        rows = cfg.conv_dim + cfg.value_dim + 2 * Hv
        m["w_in"] = _Mat(g, rows, H, quant, zero_rows=cfg.in_proj_dim - rows)
        m["conv_w"] = (torch.rand(cfg.linear_conv_kernel_dim, cfg.conv_dim, device="cuda", generator=g) - 0.5).to(
            torch.bfloat16).float()
        m["A_log"] = torch.log(1.0 + 15.0 * torch.rand(Hv, device="cuda", generator=g))
        # decays of trained models sit near 1: dt = softplus(a + dt_bias) ~ 0.001 .. 0.1
        m["dt_bias"] = torch.log(torch.expm1(torch.exp(
            math.log(1e-3) + math.log(100.0) * torch.rand(Hv, device="cuda", generator=g))))
        m["gnorm"] = _norm_w(g, cfg.linear_value_head_dim)
        m["w_out"] = _Mat(g, H, cfg.value_dim, quant)
    else:
        qkv = cfg.qkv_dim if cfg.model_type == "qwen3" else cfg.attn_qkv_dim
        m["wqkv"] = _Mat(g, qkv, H, quant)
        m["q_norm"], m["k_norm"] = _norm_w(g, cfg.head_dim), _norm_w(g, cfg.head_dim)
        m["wo"] = _Mat(g, H, cfg.q_dim, quant)
    m["gate"], m["up"], m["down"] = _Mat(g, F, H, quant), _Mat(g, F, H, quant), _Mat(g, H, F, quant)
    return m


def _globals(cfg, quant, seed):
    g = _gen(seed, 5)
    return _Mat(g, cfg.vocab_size, cfg.hidden_size, quant), _norm_w(g, cfg.hidden_size)


def _is_gdn(cfg, li):
    return cfg.model_type != "qwen3" and cfg.is_linear(li)


def _config(case):
    cfg = MODELS[case["model"]]
    kw = dict(vocab_size=LAYER_VOCAB if case["kind"] != "step" else cfg.vocab_size,
              num_hidden_layers=case.get("layers", 1))
    if case["kind"] == "layer" and cfg.model_type != "qwen3":
        kw["full_attention_interval"] = 1 if case["mixer"] == "attn" else 4
    return replace(cfg, **kw)


def _model(case, seed, max_past, max_nodes=32):
    cfg, quant = _config(case), case["quant"]
    emb, fnorm = _globals(cfg, quant, seed)
    layers = []
    for li in range(cfg.num_hidden_layers):
        gdn = _is_gdn(cfg, li)
        m = _layer_mats(cfg, "gdn" if gdn else "attn", quant, seed, li)
        rest = dict(input_norm=m["input_norm"], post_norm=m["post_norm"], wgu=m["gate"].packed(m["up"]),
                    wd=m["down"].packed())
        if gdn:
            layers.append(GdnLayerWeights(w_in=m["w_in"].packed(), conv_w=m["conv_w"], A_log=m["A_log"],
                                          dt_bias=m["dt_bias"], gnorm=m["gnorm"], w_out=m["w_out"].packed(), **rest))
        else:
            layers.append(LayerWeights(wqkv=m["wqkv"].packed(), q_norm=m["q_norm"], k_norm=m["k_norm"],
                                       wo=m["wo"].packed(), **rest))
    q3 = cfg.model_type == "qwen3"
    w = (Qwen3Weights if q3 else Qwen35Weights)(cfg=cfg, embed=emb.packed(), final_norm=fnorm, layers=layers,
                                                layout=W_TILED if quant == "q4" else W_TILED_F16, quant=quant)
    return (Qwen3TreeModel if q3 else Qwen35TreeModel)(cfg, w, max_past=max_past, max_nodes=max_nodes)


def _prefix(cfg, seed, li, past):
    """Cached keys (unit RMS, as k_norm leaves them) and values of a prefix."""
    g = _gen(seed, 23, li)
    shape = (past, cfg.num_key_value_heads, cfg.head_dim)
    return _normal(g, *shape).to(torch.bfloat16), _normal(g, *shape).to(torch.bfloat16)


def _gdn_state(cfg, seed, li):
    """A committed conv window and recurrent state."""
    g = _gen(seed, 31, li)
    return (_normal(g, cfg.linear_conv_kernel_dim - 1, cfg.conv_dim),
            _normal(g, cfg.linear_num_value_heads, cfg.linear_value_head_dim, cfg.linear_key_head_dim, std=0.1))


def _draft(case, seed, vocab):
    """A draft tree (tokens, depths, parents): best nodes first, up to 8 deep."""
    r = random.Random(seed * 7 + 3)
    n = case["nodes"]
    parents, depths = [-1], [0]
    for i in range(1, n):
        p = max(r.randrange(i), r.randrange(i)) if r.random() < 0.7 else r.randrange(i)
        while depths[p] >= 15:
            p = parents[p]
        parents.append(p)
        depths.append(depths[p] + 1)
    tokens = [r.randrange(vocab) for _ in range(n)]
    path = [n - 1]
    while parents[path[-1]] >= 0:
        path.append(parents[path[-1]])
    return tokens, depths, parents, path[::-1]


def _prompt(case, seed, vocab):
    r = random.Random(seed * 13 + 5)
    return [r.randrange(vocab) for _ in range(case["tokens"])]


def _write_prefix(cfg, kv, seed, past):
    if past:
        for ai, li in enumerate([i for i in range(cfg.num_hidden_layers) if not _is_gdn(cfg, i)]):
            kv.write_logical(ai, *_prefix(cfg, seed, li, past))


def _st():
    return torch.cuda.current_stream().cuda_stream


class _Graph:
    """A captured launch sequence (dtree_graph_*), as a serving loop keeps it."""

    def __init__(self, launch):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        N.call("dtree_graph_begin", side.cuda_stream)
        try:
            launch(side.cuda_stream)
        finally:
            ex = C.c_void_p()
            N.call("dtree_graph_end", side.cuda_stream, C.byref(ex))
        self.ex = ex
        torch.cuda.current_stream().wait_stream(side)

    def __del__(self):
        torch.cuda.synchronize()
        N.lib().dtree_graph_destroy(self.ex)


# ---- prepare / run -------------------------------------------------------------------
def prepare(case, seed):
    return {"tree": _prep_tree, "layer": _prep_layer, "mlp": _prep_mlp, "chain": _prep_chain, "prompt": _prep_prompt,
            "step": _prep_step}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _tree_logits(case, seed):
    """Draft logits: flat noise plus a few confident tokens per row."""
    g = _gen(seed, 41)
    D, V = case["depth"], case["vocab"]
    x = _normal(g, D, V) - torch.log(-torch.log(torch.rand(D, V, device="cuda", generator=g).clamp_(1e-7, 1 - 1e-7)))
    top = torch.rand(D, V, device="cuda", generator=g).topk(4, dim=1).indices
    return x.scatter_add_(1, top, 10.0 + 8.0 * torch.rand(D, 4, device="cuda", generator=g))


def _prep_tree(case, seed):
    D, V, B = case["depth"], case["vocab"], case["budget"]
    k = min(B, V)
    lib = N.lib()
    need = lib.dtree_tree_build_workspace_bytes(D, V, k)
    dev = dict(device="cuda")
    return dict(run=_run_tree, D=D, V=V, k=k, B=B, logits=_tree_logits(case, seed),
                ws=torch.zeros(need, dtype=torch.uint8, **dev),
                desc=torch.zeros(C.sizeof(N.StepDesc), dtype=torch.uint8, **dev),
                out=torch.zeros(1 + 3 * N.MAX_NODES, dtype=torch.int32, **dev),
                ids=torch.zeros(D, k, dtype=torch.int32, **dev), lp=torch.zeros(D, k, **dev))


def _run_tree(s):
    N.call("dtree_tree_build", s["logits"].data_ptr(), s["V"], s["D"], s["V"], s["k"], s["B"], 1, 1024,
           s["ws"].data_ptr(), s["ws"].numel(), s["desc"].data_ptr(), s["out"].data_ptr(), s["ids"].data_ptr(),
           s["lp"].data_ptr(), _st())
    return [s["out"], s["ids"], s["lp"]]


def _prep_layer(case, seed):
    n, P = case["nodes"], case["past"]
    model = _model(case, seed, max_past=max(P, 1), max_nodes=n)
    cfg, eng = model.args, model.engine
    cache = eng.new_cache()
    kv = cache if cfg.model_type == "qwen3" else cache.kv
    _write_prefix(cfg, kv, seed, P)
    gdn = _is_gdn(cfg, 0)
    if gdn:
        w, s = _gdn_state(cfg, seed, 0)
        cache.windows[0].copy_(w)
        cache.states[0].copy_(s)
    tokens, depths, parents, path = _draft(case, seed, cfg.vocab_size)
    cache.offset = P
    eng.set_step(tokens, [P + d for d in depths], parents, P, accepted=path)

    def launch(st):
        eng.launch_forward(cache, st, norm_hidden=True)
        if gdn:
            eng.launch_compact(cache, st, select_hidden=False)

    outs = [eng.x, eng.norm_hidden]
    outs += [cache.windows_next, cache.states_next] if gdn else [kv.k_pages, kv.v_pages]
    torch.cuda.synchronize()
    return dict(run=_run_graph, graph=_Graph(launch), outs=outs, keep=(model, cache))


def _run_graph(s):
    N.check(N.lib().dtree_graph_launch(s["graph"].ex, _st()), "graph launch")
    return s["outs"]


def _mlp_args(cfg, quant, x, w, epi, rows, **kw):
    n, k = w.shape
    a = N.GemmArgs()
    lay = N.W_TILED if quant == "q4" else N.W_TILED_F16
    a.x = x.data_ptr(); a.x_layout = lay; a.ldx = k; a.rows_padded = rows
    if quant == "q4":
        a.w = w.words.data_ptr(); a.w_scales = w.sb.data_ptr(); a.w_layout = N.W_Q4G64
    else:
        a.w = w.data_ptr(); a.w_layout = lay
    a.n = n; a.k = k; a.epilogue = epi; a.norm_dim = cfg.hidden_size; a.eps = cfg.rms_norm_eps
    a.out_layout = lay
    for name, v in kw.items():
        setattr(a, name, v.data_ptr() if isinstance(v, torch.Tensor) else v)
    return a


def _prep_mlp(case, seed):
    """Token rows, then the post-attention RMSNorm and MLP of a layer."""
    cfg, quant = _config(case), case["quant"]
    H, F = cfg.hidden_size, cfg.intermediate_size
    emb, fnorm = _globals(cfg, quant, seed)
    m = _layer_mats(cfg, "attn", quant, seed, 0)
    n = case["tokens"]
    rows = 128 * ((n + 127) // 128)
    q4 = quant == "q4"
    s = dict(run=_run_mlp, n=n, rows=rows, H=H, vocab=cfg.vocab_size, q4=q4, emb=emb.packed(), norm=m["post_norm"],
             wgu=m["gate"].packed(m["up"]), wd=m["down"].packed(), fnorm=fnorm,
             tokens=torch.tensor(_prompt(case, seed, cfg.vocab_size), dtype=torch.int32, device="cuda"))
    dt = torch.bfloat16 if q4 else torch.float16
    z = lambda *sh, dtype=torch.float32: torch.zeros(*sh, dtype=dtype, device="cuda")  # noqa: E731
    s["x"], s["xg"], s["ss"] = z(rows, H), z(rows, H, dtype=dt), z(rows // 32, H // 32, 32)
    s["act"], s["hidden"] = z(rows, F, dtype=dt), z(rows, H, dtype=torch.bfloat16)
    s["gu"] = _mlp_args(cfg, quant, s["xg"], s["wgu"], N.EPI_SWIGLU, rows, ss_in=s["ss"], ss_tiles=H // 32,
                        out_bf16=s["act"], ld_out_bf16=F)
    s["down"] = _mlp_args(cfg, quant, s["act"], s["wd"], N.EPI_RESIDUAL, rows, out_f32=s["x"], ld_out_f32=H,
                          out_bf16=s["xg"], ld_out_bf16=H, next_norm=fnorm, ss_out=s["ss"], hidden_out=s["hidden"],
                          ld_hidden=H)
    return s


def _run_mlp(s):
    lib, st = N.lib(), _st()
    q4, e = s["q4"], s["emb"]
    N.check(lib.dtree_embed_tokens(
        s["tokens"].data_ptr(), s["n"], e.words.data_ptr() if q4 else e.data_ptr(),
        N.W_Q4G64 if q4 else N.W_TILED_F16, e.sb.data_ptr() if q4 else None, s["vocab"], s["H"], s["norm"].data_ptr(),
        s["rows"], s["x"].data_ptr(), s["xg"].data_ptr(), None, N.W_TILED if q4 else N.W_TILED_F16,
        s["ss"].data_ptr(), st), "embed tokens")
    N.check(lib.dtree_gemm_long(C.byref(s["gu"]), st), "gate/up")
    N.check(lib.dtree_gemm_long(C.byref(s["down"]), st), "down")
    return [s["x"], s["xg"], s["ss"], s["hidden"]]


def _chain_inputs(case, seed):
    """A projection [T, qkv | z | b | a] as in_proj gives it, and layer weights."""
    cfg = replace(MODELS[case["model"]], num_hidden_layers=1)
    T = case["tokens"]
    g = _gen(seed, 53)
    proj = _normal(g, T, cfg.in_proj_dim)
    m = _layer_mats(replace(cfg, hidden_size=64, intermediate_size=64), "gdn", "bf16", seed, 0)
    return cfg, proj, m, _gdn_state(cfg, seed, 0)


def _prep_chain(case, seed):
    cfg, proj, m, (win, st) = _chain_inputs(case, seed)
    T = case["tokens"]
    rows = 128 * ((T + 127) // 128)
    Hv = cfg.linear_num_value_heads
    z = lambda *sh, dtype=torch.float32: torch.zeros(*sh, dtype=dtype, device="cuda")  # noqa: E731
    s = dict(run=_run_chain, T=T, m=m, proj=z(rows, cfg.in_proj_dim), q=z(rows, cfg.key_dim), k=z(rows, cfg.key_dim),
             v=z(rows, cfg.value_dim), g=z(rows, Hv), beta=z(rows, Hv), y=z(rows, cfg.value_dim),
             out=z(rows, cfg.value_dim, dtype=torch.float16), window=win.clone(), state=st.clone(), win0=win, st0=st)
    s["proj"][:T] = proj
    a = N.GdnArgs()
    a.rows_padded = rows
    a.num_k_heads, a.num_v_heads = cfg.linear_num_key_heads, Hv
    a.head_k_dim, a.head_v_dim = cfg.linear_key_head_dim, cfg.linear_value_head_dim
    a.conv_keep = cfg.linear_conv_kernel_dim - 1
    a.ld_proj = cfg.in_proj_dim
    for name in ("proj", "window", "state", "q", "k", "v", "g", "beta", "y", "out"):
        setattr(a, name, s[name].data_ptr())
    a.conv_w, a.A_log, a.dt_bias = (m[t].data_ptr() for t in ("conv_w", "A_log", "dt_bias"))
    a.norm_w, a.eps = m["gnorm"].data_ptr(), cfg.rms_norm_eps
    a.out_layout, a.ld_out = N.W_TILED_F16, cfg.value_dim
    s["args"] = a
    return s


def _run_chain(s):
    s["window"].copy_(s["win0"])  # a prompt that continues a kept prefix
    s["state"].copy_(s["st0"])
    N.check(N.lib().dtree_gdn_layer_chain(C.byref(s["args"]), s["T"], _st()), "gdn chain")
    return [s["out"], s["window"], s["state"]]


def _prep_prompt(case, seed):
    P, T = case["past"], case["tokens"]
    model = _model(case, seed, max_past=P + T)
    cfg = model.args
    q3 = cfg.model_type == "qwen3"
    adapter = Qwen3TargetAdapter() if q3 else Qwen35TargetAdapter()
    cache = adapter.make_cache(model)
    kv = cache if q3 else cache.kv
    _write_prefix(cfg, kv, seed, P)
    return dict(run=_run_prompt, model=model, adapter=adapter, cache=cache, kv=kv, P=P, q3=q3,
                prompt=_prompt(case, seed, cfg.vocab_size), ids=[cfg.num_hidden_layers - 1])


def _run_prompt(s):
    cache = s["cache"]
    cache.reset(s["P"])
    logits, hidden = s["adapter"].forward_with_hidden_states(s["model"], s["prompt"], cache, s["ids"])
    outs = [logits, hidden, s["kv"].k_pages, s["kv"].v_pages]
    return outs if s["q3"] else outs + [cache.windows, cache.states]


def _prep_step(case, seed):
    n, P = case["nodes"], case["past"]
    model = _model(case, seed, max_past=max(P, 1))
    cfg = model.args
    adapter = Qwen3TargetAdapter()
    cache = adapter.make_cache(model)
    _write_prefix(cfg, cache, seed, P)
    cache.offset = P
    tokens, depths, parents, _ = _draft(case, seed, cfg.vocab_size)
    mask = np.ones((n, P + n), dtype=bool)
    mask[:, P:] = _visible(parents)
    return dict(run=_run_step, model=model, adapter=adapter, cache=cache, tokens=tokens, parents=parents, mask=mask,
                pos=[P + d for d in depths], n=n, ids=[cfg.num_hidden_layers // 2, cfg.num_hidden_layers - 1])


def _run_step(s):
    ad, model, cache = s["adapter"], s["model"], s["cache"]
    norm, hidden = ad.forward_tree_with_hidden_states(model, s["tokens"], cache, s["ids"], s["parents"], s["pos"],
                                                      s["mask"])
    logits = ad.lm_head_logits(model, norm)
    ad.rewind_kv_caches(cache, s["n"])  # nothing accepted: the tree's rows are dropped
    return [logits, norm, hidden]


# ---- work ----------------------------------------------------------------------------
def _mat_bytes(n, k, quant):
    return n * k * 9 // 16 if quant == "q4" else 2 * n * k


def _layer_linears(cfg, gdn):
    H, F = cfg.hidden_size, cfg.intermediate_size
    if gdn:
        mix = [(cfg.in_proj_dim, H), (H, cfg.value_dim)]
    else:
        mix = [(cfg.qkv_dim if cfg.model_type == "qwen3" else cfg.attn_qkv_dim, H), (H, cfg.q_dim)]
    return mix + [(2 * F, H), (H, F)]


def _mixer_work(cfg, gdn, rows, past, causal):
    if gdn:
        Hv, Dk, Dv = cfg.linear_num_value_heads, cfg.linear_key_head_dim, cfg.linear_value_head_dim
        return 8 * Hv * Dk * Dv, 6 * rows * Hv * Dk * Dv
    D, Hq, Hkv = cfg.head_dim, cfg.num_attention_heads, cfg.num_key_value_heads
    keys = past + (rows + 1) / 2 if causal else past + rows
    return 4 * (past + rows) * Hkv * D, int(4 * rows * keys * Hq * D)


def work(case):
    kind = case["kind"]
    if kind == "tree":
        D, V = case["depth"], case["vocab"]
        return dict(bytes=4 * D * V, flops=3 * D * V)
    cfg = _config(case) if kind != "chain" else MODELS[case["model"]]
    H = cfg.hidden_size
    if kind == "mlp":
        n, F = case["tokens"], cfg.intermediate_size
        return dict(bytes=_mat_bytes(3 * F, H, case["quant"]) + n * H * 2 + n * H * 8, flops=6 * n * H * F)
    if kind == "chain":
        T = case["tokens"]
        b, f = _mixer_work(cfg, True, T, 0, True)
        return dict(bytes=b + 4 * T * cfg.in_proj_dim + 2 * T * cfg.value_dim, flops=f)
    rows, past = (case["tokens"], case["past"]) if kind == "prompt" else (case["nodes"], case["past"])
    byts, flops = 2 * rows * H, 0
    for li in range(cfg.num_hidden_layers):
        gdn = _is_gdn(cfg, li)
        for n, k in _layer_linears(cfg, gdn):
            byts += _mat_bytes(n, k, case["quant"])
            flops += 2 * rows * n * k
        b, f = _mixer_work(cfg, gdn, rows, past, kind == "prompt")
        byts, flops = byts + b, flops + f
    if kind == "step":
        byts += _mat_bytes(cfg.vocab_size, H, case["quant"]) + 4 * rows * cfg.vocab_size
        flops += 2 * rows * cfg.vocab_size * H
    return dict(bytes=byts, flops=flops)


def tolerance(case):
    """About four times the distance from `exact` measured per kind: fp16
    activations and bf16 outputs for bf16 models, bf16 activations for q4."""
    kind, q4 = case["kind"], case.get("quant") == "q4"
    if kind == "tree":  # log-probs: fp32 sums; tokens and tree exact
        return {"rel": 1e-6}
    if kind == "chain":  # fp32 recurrence, fp16 output
        return {"rel": 8e-4}
    if kind == "step":
        return {"rel": 5e-2 if q4 else 1.4e-2}
    if kind == "prompt" and q4:
        return {"rel": 5e-2 if case["layers"] > 1 else 2.5e-2}
    return {"rel": 2e-2 if q4 else 8e-3}


# ---- exact (float64, plain torch) --------------------------------------------------------
def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * (1.0 if w is None else w.to(F64))


def _rope(x, pos, dims, base):
    half = dims // 2
    inv = base ** (-torch.arange(half, dtype=F64, device="cuda") * 2.0 / dims)
    ang = pos.to(F64)[:, None] * inv
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = x[..., :half], x[..., half:dims]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., dims:]], -1)


def _visible(parents):
    vis = np.zeros((len(parents), len(parents)), dtype=bool)
    for i, p in enumerate(parents):
        if p >= 0:
            vis[i] = vis[p]
        vis[i, i] = True
    return vis


def _mlp(m, x, eps):
    h = _rms(x, m["post_norm"], eps)
    gate = h @ m["gate"].exact().T
    return x + (gate * torch.sigmoid(gate) * (h @ m["up"].exact().T)) @ m["down"].exact().T


def _attn(cfg, m, x, pos, prefix, vis):
    """-> (x + attention, k rows, v rows); vis: [n, n] visibility among the rows."""
    n, D, Hq, Hkv = x.shape[0], cfg.head_dim, cfg.num_attention_heads, cfg.num_key_value_heads
    q3 = cfg.model_type == "qwen3"
    y = _rms(x, m["input_norm"], cfg.rms_norm_eps) @ m["wqkv"].exact().T
    nq = cfg.q_dim if q3 else 2 * cfg.q_dim
    q, k, v = y[:, :nq].reshape(n, Hq, -1), y[:, nq:nq + Hkv * D].reshape(n, Hkv, D), y[:, nq + Hkv * D:]
    v = v.reshape(n, Hkv, D)
    gate = None if q3 else q[..., D:]
    dims = D if q3 else cfg.rope_dims
    q = _rope(_rms(q[..., :D], m["q_norm"], cfg.rms_norm_eps), pos, dims, cfg.rope_theta)
    k = _rope(_rms(k, m["k_norm"], cfg.rms_norm_eps), pos, dims, cfg.rope_theta)
    P = 0 if prefix is None else prefix[0].shape[0]
    K, V = k.to(torch.bfloat16).to(F64), v.to(torch.bfloat16).to(F64)
    if P:
        K, V = torch.cat([prefix[0].to(F64), K]), torch.cat([prefix[1].to(F64), V])
    out = torch.empty(n, Hq, D, dtype=F64, device="cuda")
    for r0 in range(0, n, 1024):
        r1 = min(n, r0 + 1024)
        for h in range(Hq):
            s = q[r0:r1, h] @ K[:, h // (Hq // Hkv)].T * D ** -0.5
            s[:, P:].masked_fill_(~vis[r0:r1], -math.inf)
            out[r0:r1, h] = torch.softmax(s, -1) @ V[:, h // (Hq // Hkv)]
    if gate is not None:
        out = out * torch.sigmoid(gate)
    return x + out.reshape(n, -1) @ m["wo"].exact().T, k, v


def _gdn_core(cfg, m, proj, window, state, parents):
    """conv, gates, recurrence and gated norm over nodes in topological order;
    -> (gated output [n, value_dim], per-node windows, state after each node)."""
    n, Hk, Hv = proj.shape[0], cfg.linear_num_key_heads, cfg.linear_num_value_heads
    Dk, Dv, Cd, kd = cfg.linear_key_head_dim, cfg.linear_value_head_dim, cfg.conv_dim, cfg.key_dim
    x, z = proj[:, :Cd], proj[:, Cd:Cd + cfg.value_dim].reshape(n, Hv, Dv)
    b, a = proj[:, Cd + cfg.value_dim:][:, :Hv], proj[:, Cd + cfg.value_dim + Hv:][:, :Hv]
    keep = window.shape[0]
    rows = torch.cat([window.to(F64), x])
    idx = np.zeros((n, keep + 1), dtype=np.int64)  # conv rows of node t, oldest first
    for t, p in enumerate(parents):
        prev = np.arange(keep) if p < 0 else idx[p, 1:]
        idx[t] = np.append(prev, keep + t)
    idx = torch.from_numpy(idx).cuda()
    conv = sum(rows[idx[:, j]] * m["conv_w"][j].to(F64) for j in range(keep + 1))
    conv = conv * torch.sigmoid(conv)
    grp = Hv // Hk
    q = (_rms(conv[:, :kd].reshape(n, Hk, Dk), None, 1e-6) / Dk).repeat_interleave(grp, 1)
    k = (_rms(conv[:, kd:2 * kd].reshape(n, Hk, Dk), None, 1e-6) * Dk ** -0.5).repeat_interleave(grp, 1)
    v = conv[:, 2 * kd:].reshape(n, Hv, Dv)
    g = torch.exp(-torch.exp(m["A_log"].to(F64)) * torch.nn.functional.softplus(a + m["dt_bias"].to(F64)))
    beta = torch.sigmoid(b)
    chain = all(p == i - 1 for i, p in enumerate(parents))
    y = torch.empty(n, Hv, Dv, dtype=F64, device="cuda")
    S0, states = state.to(F64), {}
    for t, p in enumerate(parents):
        S = (S0 if p < 0 else states[p]) * g[t][:, None, None]
        d = (v[t] - (S @ k[t].unsqueeze(-1)).squeeze(-1)) * beta[t][:, None]
        S = S + d.unsqueeze(-1) * k[t].unsqueeze(1)
        y[t] = (S @ q[t].unsqueeze(-1)).squeeze(-1)
        if chain:
            states.pop(p, None)
        states[t] = S
    o = _rms(y, m["gnorm"], cfg.rms_norm_eps) * (z * torch.sigmoid(z))
    return o.reshape(n, -1), lambda t: rows[idx[t, 1:]], states


def _gdn(cfg, m, x, window, state, parents):
    proj = _rms(x, m["input_norm"], cfg.rms_norm_eps) @ m["w_in"].exact().T
    o, win, states = _gdn_core(cfg, m, proj, window, state, parents)
    return x + o @ m["w_out"].exact().T, win, states


def _tiled(t):
    """[n, k] in the 32 x 64 tile order of the GEMM operands."""
    n, k = t.shape
    return t.reshape(n // 32, 32, k // 64, 2, 4, 8).permute(0, 2, 4, 3, 1, 5).reshape(n, k)


def _pages(rows, n_pages, which):
    """[T, heads, D] -> [n_pages, heads, 64 * D] in the cache's fragment order."""
    T, Hkv, D = rows.shape
    slot, d = torch.arange(64, device="cuda").view(64, 1), torch.arange(D, device="cuda").view(1, D)
    if which == "k":
        r = slot & 31
        r = (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1)
        off = ((((slot >> 5) * (D >> 4) + (d >> 4)) * 64 + ((d >> 3) & 1) * 32 + r) << 3) + (d & 7)
    else:
        off = ((((slot >> 4) * (D >> 5) + (d >> 5)) * 64 + ((slot >> 3) & 1) * 32 + (d & 31)) << 3) + (slot & 7)
    full = torch.zeros(n_pages * 64, Hkv, D, dtype=F64, device="cuda")
    full[:T] = rows
    src = full.reshape(n_pages, 64, Hkv, D).permute(0, 2, 1, 3).reshape(n_pages, Hkv, 64 * D)
    out = torch.empty_like(src)
    out[:, :, off.reshape(-1)] = src
    return out


def _pad(t, rows):
    return torch.cat([t, t.new_zeros(rows - t.shape[0], *t.shape[1:])])


def exact(case, seed):
    kind = case["kind"]
    if kind == "tree":
        lp = torch.log_softmax(_tree_logits(case, seed).to(F64), -1)
        return [None, None, lp.topk(min(case["budget"], case["vocab"]), dim=-1).values]
    if kind == "chain":
        cfg, proj, m, (win, st) = _chain_inputs(case, seed)
        T = case["tokens"]
        o, window, states = _gdn_core(cfg, m, proj.to(F64), win, st, list(range(-1, T - 1)))
        return [_tiled(_pad(o, 128 * ((T + 127) // 128))), window(T - 1), states[T - 1]]
    cfg, quant = _config(case), case["quant"]
    emb, fnorm = _globals(cfg, quant, seed)
    E = emb.exact()
    eps = cfg.rms_norm_eps
    if kind == "mlp":
        rows = 128 * ((case["tokens"] + 127) // 128)
        x = E[torch.tensor(_prompt(case, seed, cfg.vocab_size), device="cuda")]
        x = _pad(_mlp(_layer_mats(cfg, "attn", quant, seed, 0), x, eps), rows)
        ss = x.square().reshape(rows // 32, 32, -1, 32).sum(-1).transpose(1, 2)
        return [x, _tiled(x * fnorm.to(F64)), ss, x]
    prompt = kind == "prompt"
    P = case["past"]
    if prompt:
        tokens = _prompt(case, seed, cfg.vocab_size)
        n, parents = len(tokens), list(range(-1, len(tokens) - 1))
        pos = torch.arange(P, P + n, device="cuda")
        vis = torch.ones(n, n, dtype=torch.bool, device="cuda").tril_()
    else:
        tokens, depths, parents, path = _draft(case, seed, cfg.vocab_size)
        n = len(tokens)
        pos = torch.tensor([P + d for d in depths], device="cuda")
        vis = torch.from_numpy(_visible(parents)).cuda()
    x = E[torch.tensor(tokens, device="cuda")]
    n_pages = (max(P, 1) + n + 63) // 64 if kind == "layer" else (P + n + 32 + 63) // 64
    keys, vals, wins, sts, hid = [], [], [], [], {}
    for li in range(cfg.num_hidden_layers):
        gdn = _is_gdn(cfg, li)
        m = _layer_mats(cfg, "gdn" if gdn else "attn", quant, seed, li)
        if gdn:
            win, st = _gdn_state(cfg, seed, li)
            if prompt:  # a new prompt starts from an empty state
                win, st = torch.zeros_like(win), torch.zeros_like(st)
            x, window, states = _gdn(cfg, m, x, win, st, parents)
            last = n - 1 if prompt else path[-1]
            wins.append(window(last))
            sts.append(states[last])
        else:
            pre = _prefix(cfg, seed, li, P) if P else None
            x, k, v = _attn(cfg, m, x, pos, pre, vis)
            if kind != "step":
                keys.append(_pages(k if pre is None else torch.cat([pre[0].to(F64), k]), n_pages, "k"))
                vals.append(_pages(v if pre is None else torch.cat([pre[1].to(F64), v]), n_pages, "v"))
        x = _mlp(m, x, eps)
        hid[li] = x
    norm = _rms(x, fnorm, eps)
    if kind == "layer":
        rows = 32 * ((n + 31) // 32)
        tail = [torch.stack(wins), torch.stack(sts)] if wins else [torch.stack(keys), torch.stack(vals)]
        return [_pad(x, rows), _pad(norm, rows)] + tail
    if prompt:
        outs = [(norm[-1:] @ E.T)[None], x[None], torch.stack(keys), torch.stack(vals)]
        return outs + ([torch.stack(wins), torch.stack(sts)] if wins else [])
    nl = cfg.num_hidden_layers
    return [(norm @ E.T)[None], norm[None], torch.cat([hid[nl // 2], hid[nl - 1]], -1)[None]]
