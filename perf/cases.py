"""The work that is timed: single layers, operators and whole decoder calls of the
Qwen3.6-35B-A3B shape (and the small shape that the tests use), through the package's
public entry points.

Kinds of case:

* ``qmv``    one quantised operator (``NpuIQ4MatVec`` / ``NpuQuantMatVec``) on one or a
             few vectors: an expert matrix driven from a caller's own loop;
* ``linear`` one dense bf16 projection (``NpuLinear``) on a prompt or a step's vector;
* ``chain``  consecutive MoE blocks with RMSNorm and residual (``GpuMoeChain``): a decode
             step of 1 to 8 sequences;
* ``moe``    one MoE block (``GpuMoeBlock``) over a prompt's tokens: IQ4_XS / IQ3_XXS
             experts, or the K-quant experts of the model's outlier layers;
* ``attn``   the gated attention layer (``attn_forward``): a decode step on a filled
             cache, or a prompt (from position 0 or on a cached prefix);
* ``ssm``    the Gated DeltaNet layer (``ssm_forward``): a prompt or a step;
* ``model``  the whole ``forward``: three DeltaNet layers and one attention layer (the
             model's pattern), each with its MoE block, output norm and lm_head.

Where a call updates its state in place, ``run`` starts from the same saved state every
time, as a program does that answers several continuations of one prefix: it sets the KV
cache's length back, and hands over a copy of the DeltaNet states.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from npu_amd import qwen_core as QN
from npu_amd.gguf_types import GGMLQuantizationType as QT
from npu_amd.linear import NpuLinear
from npu_amd.moe import GpuMoeBlock, GpuMoeChain
from npu_amd.quant_mv import NpuQuantMatVec
from npu_amd.quant_mv_iq4 import NpuIQ4MatVec

DEV = "cuda"
EPS = 1e-6

# The model's dimensions, and the small ones of the tests.
SHAPES = {
    "model": dict(D=2048, n_head=16, n_head_kv=2, head_dim=256, rope_dim=64, theta=1e7, d_inner=4096, d_state=128,
                  n_k_heads=16, n_v_heads=32, E=256, k=8, FF=512, vocab=248_320),
    "small": dict(D=512, n_head=4, n_head_kv=2, head_dim=128, rope_dim=32, theta=1e6, d_inner=256, d_state=64,
                  n_k_heads=2, n_v_heads=4, E=16, k=4, FF=256, vocab=1000),
}
MAX_POS = 4096                # Model.load's default
PATTERN = [False, False, False, True]       # is_attention of the four layers of a "model" case

# (weights, bytes) of a block, byte offsets of its fp16 scales, and a typical size of the
# scale (weights of a trained layer are a few hundredths)
FORMATS = {
    "iq4_xs": (int(QT.IQ4_XS), 256, 136, (0,), 2e-5),
    "iq3_xxs": (int(QT.IQ3_XXS), 256, 98, (0,), 1.5e-4),
    "q8_0": (int(QT.Q8_0), 32, 34, (0,), 4e-4),
    "q4_k": (int(QT.Q4_K), 256, 144, (0, 2), 1e-4),
    "q5_k": (int(QT.Q5_K), 256, 176, (0, 2), 5e-5),
    "q6_k": (int(QT.Q6_K), 256, 210, (208,), 2e-5),
}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one expert's gate matrix times one vector: the smallest call, all latency
        dict(name="iq4_vector", kind="qmv", fmt="iq4_xs", M=512, K=2048, T=1),
        # an attention layer's input projection over a prompt
        dict(name="linear_prompt", kind="linear", M=9216, K=2048, T=300),
        # MoE blocks of a decode step: one sequence, and a full batch of eight
        dict(name="chain_one", kind="chain", shape="model", layers=4, T=1, gate="iq4_xs", down="iq3_xxs"),
        dict(name="chain_eight", kind="chain", shape="model", layers=4, T=8, gate="iq4_xs", down="iq3_xxs"),
        # one MoE block over an ordinary prompt, over the longest that the default cache
        # takes, and an outlier layer (K-quant experts) over a short one
        dict(name="moe_512", kind="moe", shape="model", T=512, gate="iq4_xs", down="iq3_xxs", shared="iq"),
        dict(name="moe_4096", kind="moe", shape="model", T=4096, gate="iq4_xs", down="iq3_xxs", shared="iq"),
        dict(name="moe_outlier_150", kind="moe", shape="model", T=150, gate="q5_k", down="q6_k", shared="q6_k"),
        # attention: a step late in a conversation, and a follow-up turn of 1021 tokens
        dict(name="attn_step", kind="attn", shape="model", T=1, start=3001),
        dict(name="attn_prompt", kind="attn", shape="model", T=1021, start=300),
        # Gated DeltaNet over a first prompt
        dict(name="ssm_prompt", kind="ssm", shape="model", T=1000, saved=False),
        # whole calls: a decode step after 700 tokens, and a short prompt
        dict(name="model_step", kind="model", shape="model", T=1, start=700),
        dict(name="model_prompt", kind="model", shape="model", T=57, start=0),
    ]


def _log(rng, lo, hi):
    """A whole number of lo .. hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["qmv", "linear", "chain", "moe", "moe", "outlier", "attn_step", "attn", "ssm", "model"])
    shape = "small" if rng.random() < 0.15 else "model"
    if kind == "qmv":
        return dict(kind="qmv", fmt=rng.choice(["iq4_xs", "iq3_xxs"]), M=_log(rng, 256, 4096),
                    K=256 * _log(rng, 1, 16), T=1 if rng.random() < 0.5 else _log(rng, 2, 64))
    if kind == "linear":
        M, K = rng.choice([(8192, 2048), (4096, 2048), (2048, 4096), (9216, 2048),
                           (_log(rng, 500, 9000), 32 * _log(rng, 16, 128))])
        return dict(kind="linear", M=M, K=K, T=1 if rng.random() < 0.25 else _log(rng, 2, 600))
    gate, down = rng.choice([("iq4_xs", "iq3_xxs")] * 3 + [("iq3_xxs", "iq4_xs"), ("iq4_xs", "iq4_xs"),
                                                           ("iq3_xxs", "iq3_xxs")])
    if kind == "chain":
        return dict(kind="chain", shape="model", layers=rng.choice([2, 3, 5, 6]), T=rng.randint(1, 8), gate=gate, down=down)
    if kind == "moe":
        return dict(kind="moe", shape=shape, T=_log(rng, 9, 4000), gate=gate, down=down,
                    shared=rng.choice(["iq", "iq", "q6_k"]))
    if kind == "outlier":
        return dict(kind="moe", shape=shape, T=_log(rng, 9, 500), gate=rng.choice(["q5_k", "q6_k", "q8_0", "q4_k"]),
                    down=rng.choice(["q5_k", "q6_k"]), shared="q6_k")
    if kind == "attn_step":
        return dict(kind="attn", shape=shape, T=1, start=_log(rng, 1, 4000))
    if kind == "attn":
        T = _log(rng, 2, 900)
        return dict(kind="attn", shape=shape, T=T, start=rng.choice([0, 0, _log(rng, 1, 1500)]))
    if kind == "ssm":
        return dict(kind="ssm", shape=shape, T=1 if rng.random() < 0.25 else _log(rng, 2, 950),
                    saved=rng.random() < 0.5)
    T = 1 if rng.random() < 0.5 else _log(rng, 2, 200)
    return dict(kind="model", shape="small" if rng.random() < 0.3 else "model", T=T,
                start=_log(rng, 10, 2000) if T == 1 else 0)


# ------------------------------------------------------------------ inputs
def _gen(seed, part):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1009 + part)
    return g


def _randn(g, *shape, scale=1.0):
    return torch.randn(*shape, device=DEV, generator=g) * scale


def _bf(t):
    return t.to(torch.bfloat16).float()


def _blocks(g, fmt, *shape_k):
    """Raw bytes [..., M, row bytes] of an [..., M, K] matrix: uniform quants and scales,
    fp16 block scales |N(0, 1)| times the format's typical one (every block's at least a
    tenth of it, as trained blocks are never empty)."""
    _, bw, bb, at, d = FORMATS[fmt]
    *lead, K = shape_k
    n = math.prod(lead) * (K // bw)
    raw = torch.randint(0, 256, (n, bb), dtype=torch.uint8, device=DEV, generator=g)
    for o in at:
        s = ((torch.randn(n, device=DEV, generator=g).abs() + 0.1) * d).to(torch.float16)
        raw[:, o:o + 2] = s.view(torch.uint8).reshape(n, 2)
    return raw.reshape(*lead, (K // bw) * bb)


def _moe_inputs(c, seed, part=0, layer=0):
    s, g = SHAPES[c["shape"]], _gen(seed, 100 + layer)
    D, FF, E = s["D"], s["FF"], s["E"]
    sh = c.get("shared", "iq")
    gate_sh, down_sh = (c["gate"], c["down"]) if sh == "iq" else (sh, sh)
    w = dict(gate=_blocks(g, c["gate"], E, FF, D), up=_blocks(g, c["gate"], E, FF, D),
             down=_blocks(g, c["down"], E, D, FF), gate_sh=_blocks(g, gate_sh, FF, D), up_sh=_blocks(g, gate_sh, FF, D),
             down_sh=_blocks(g, down_sh, D, FF))
    # the file's router and shared gate are F32; a trained router is sure of its first picks
    # (logits of a few units) and uses the experts unevenly (here through a bias)
    w["router"] = _randn(g, E, D, scale=0.06)
    w["sh_gate_inp"] = _randn(g, D, scale=0.02)
    w["router_bias"] = _randn(g, E, scale=0.5)
    w["norm_w"] = 1 + _randn(g, D, scale=0.1)
    return w, gate_sh, down_sh


def _moe_block(c, w, gate_sh, down_sh):
    s = SHAPES[c["shape"]]
    return GpuMoeBlock(q_gate=FORMATS[c["gate"]][0], q_down=FORMATS[c["down"]][0], q_gate_sh=FORMATS[gate_sh][0],
                       q_down_sh=FORMATS[down_sh][0], D=s["D"], FF=s["FF"], E=s["E"], k=s["k"], norm_eps=EPS,
                       device=DEV, **w)


def _cfg(shape):
    s = SHAPES[shape]
    return QN.Config(d_model=s["D"], n_layer=len(PATTERN), n_head=s["n_head"], n_head_kv=s["n_head_kv"],
                     head_dim=s["head_dim"], rms_eps=EPS, rope_theta=s["theta"], rope_dim=s["rope_dim"],
                     n_expert=s["E"], n_expert_used=s["k"], d_expert_ff=s["FF"], vocab_size=s["vocab"],
                     ssm_d_conv=4, ssm_d_inner=s["d_inner"], ssm_d_state=s["d_state"], ssm_n_k_heads=s["n_k_heads"],
                     ssm_n_v_heads=s["n_v_heads"], is_attention=list(PATTERN))


def _attn_weights(shape, seed, layer=0):
    s, g = SHAPES[shape], _gen(seed, 200 + layer)
    D, Hq, Hkv, Dh = s["D"], s["n_head"], s["n_head_kv"], s["head_dim"]
    return dict(attn_norm=1 + _randn(g, D, scale=0.1), post_norm=1 + _randn(g, D, scale=0.1),
                wq=_bf(_randn(g, 2 * Hq * Dh, D, scale=0.02)), wk=_bf(_randn(g, Hkv * Dh, D, scale=0.02)),
                wv=_bf(_randn(g, Hkv * Dh, D, scale=0.02)), wo=_bf(_randn(g, D, Hq * Dh, scale=0.02)),
                q_norm=1 + _randn(g, Dh, scale=0.1), k_norm=1 + _randn(g, Dh, scale=0.1))


def _ssm_weights(shape, seed, layer=0):
    s, g = SHAPES[shape], _gen(seed, 300 + layer)
    D, Hv, Sk = s["D"], s["n_v_heads"], s["d_state"]
    C = 2 * s["n_k_heads"] * Sk + Hv * Sk
    return dict(attn_norm=1 + _randn(g, D, scale=0.1), post_norm=1 + _randn(g, D, scale=0.1),
                w_in=_bf(_randn(g, C, D, scale=0.02)), w_gate=_bf(_randn(g, Hv * Sk, D, scale=0.02)),
                conv1d=_randn(g, C, 4, scale=0.5), a=-2 * torch.rand(Hv, device=DEV, generator=g),
                alpha=_randn(g, Hv, D, scale=0.05), beta=_randn(g, Hv, D, scale=0.05), dt_bias=_randn(g, Hv, scale=0.5),
                ssm_norm=1 + _randn(g, Sk, scale=0.1), w_out=_bf(_randn(g, D, Hv * Sk, scale=0.02)))


def _prefix(shape, seed, start, layer=0):
    """k and v rows of ``start`` cached positions."""
    s, g = SHAPES[shape], _gen(seed, 400 + layer)
    return (_randn(g, start, s["n_head_kv"], s["head_dim"]),
            _randn(g, start, s["n_head_kv"], s["head_dim"], scale=0.5))


def _ssm_state(shape, seed, layer=0):
    s, g = SHAPES[shape], _gen(seed, 500 + layer)
    Sk, C = s["d_state"], 2 * s["n_k_heads"] * s["d_state"] + s["n_v_heads"] * s["d_state"]
    return _randn(g, 1, C, 3, scale=0.5), _randn(g, 1, s["n_v_heads"], Sk, Sk, scale=0.05)


def _cache(cfg, prefix):
    c = QN.KVCache(cfg, MAX_POS)
    n = prefix[0].shape[0]
    c.k[:n], c.v[:n] = prefix
    c.length = n
    return c


def _inputs_x(c, seed):
    D = c["K"] if "K" in c else SHAPES[c["shape"]]["D"]
    return _randn(_gen(seed, 1), c["T"], D)


def _tokens(c, seed):
    return torch.randint(0, SHAPES[c["shape"]]["vocab"], (c["T"],), device=DEV, generator=_gen(seed, 2))


def _model_weights(shape, seed):
    s, g = SHAPES[shape], _gen(seed, 600)
    return dict(embd=_randn(g, s["vocab"], s["D"]), onorm=1 + _randn(g, s["D"], scale=0.1),
                head=_randn(g, s["vocab"], s["D"], scale=0.02).to(torch.bfloat16))


def _model_case(c, layer):
    """The MoE block of a model case's layer: the file's usual formats."""
    return dict(shape=c["shape"], gate="iq4_xs", down="iq3_xxs", shared="q6_k")


# ------------------------------------------------------------------ prepare / run
def prepare(case, seed):
    c, kind = case, case["kind"]
    st = dict(case=c)
    if kind == "qmv":
        cls = NpuIQ4MatVec if c["fmt"] == "iq4_xs" else NpuQuantMatVec
        st["op"] = cls(_blocks(_gen(seed, 0), c["fmt"], c["M"], c["K"]).cpu().numpy().reshape(-1), c["M"], c["K"])
        st["x"] = _inputs_x(c, seed)[0] if c["T"] == 1 else _inputs_x(c, seed)
        st["op"](st["x"])                                  # the first call uploads the weight
    elif kind == "linear":
        st["op"] = NpuLinear(_bf(_randn(_gen(seed, 0), c["M"], c["K"], scale=0.02)))
        st["x"] = _inputs_x(c, seed)
        st["op"](st["x"])
    elif kind == "chain":
        st["op"] = GpuMoeChain([_moe_block(c, *_moe_inputs(c, seed, layer=i)) for i in range(c["layers"])])
        st["x"] = _inputs_x(c, seed)
    elif kind == "moe":
        st["op"] = _moe_block(c, *_moe_inputs(c, seed))
        st["x"] = _inputs_x(c, seed)
    elif kind in ("attn", "ssm"):
        cfg = st["cfg"] = _cfg(c["shape"])
        st["x"] = _inputs_x(c, seed).unsqueeze(0)
        if kind == "attn":
            st["layer"] = QN.AttnLayer(i=0, **_attn_weights(c["shape"], seed))
            st["layer"].gpu = QN.GpuAttn(st["layer"], cfg)
            st["rope"] = QN.build_partial_rope_cache(cfg.rope_dim, MAX_POS, cfg.rope_theta, device=DEV)
            st["cache"] = _cache(cfg, _prefix(c["shape"], seed, c["start"]))
        else:
            st["layer"] = QN.SSMLayer(i=0, **_ssm_weights(c["shape"], seed))
            st["layer"].gpu = QN.GpuSsm(st["layer"], cfg)
            st["saved"] = _ssm_state(c["shape"], seed) if c["saved"] else None
    else:
        cfg, w = _cfg(c["shape"]), _model_weights(c["shape"], seed)
        cos, sin = QN.build_partial_rope_cache(cfg.rope_dim, MAX_POS, cfg.rope_theta, device=DEV)
        layers, kv, ssm = [], [], []
        for i, is_attn in enumerate(PATTERN):
            mc = _model_case(c, i)
            mw, gs, ds = _moe_inputs(mc, seed, layer=i)
            mw.pop("norm_w")                               # the decoder hands over the layer's post_norm
            blk = _moe_block(mc, mw, gs, ds)
            if is_attn:
                core = QN.AttnLayer(i=i, **_attn_weights(c["shape"], seed, i))
                core.gpu = QN.GpuAttn(core, cfg)
                core.wq = core.wk = core.wv = core.wo = None     # the device copy is what runs
                kv.append(_cache(cfg, _prefix(c["shape"], seed, c["start"], i)))
                ssm.append(None)
            else:
                core = QN.SSMLayer(i=i, **_ssm_weights(c["shape"], seed, i))
                core.gpu = QN.GpuSsm(core, cfg)
                core.w_in = core.w_gate = core.w_out = None
                kv.append(None)
                ssm.append(_ssm_state(c["shape"], seed, i) if c["start"] else None)
            layers.append((core, blk))
        st["model"] = QN.Model(cfg=cfg, token_embd=w["embd"], output_norm=w["onorm"], lm_head=w["head"], layers=layers,
                               rope_cos=cos, rope_sin=sin)
        st["kv"], st["saved"] = kv, ssm
        # a decode loop hands over the sampled token as it lies on the GPU, a prompt comes
        # as a tokenizer's list
        st["tokens"] = _tokens(c, seed) if c["T"] == 1 else _tokens(c, seed).tolist()
        # stages the head and the tables, and fills the blocks' workspaces
        _run_model(st)
    return st


def _clone(state):
    return None if state is None else tuple(t.clone() for t in state)


def _run_model(st):
    c = st["case"]
    for cache in st["kv"]:
        if cache is not None:
            cache.length = c["start"]
    logits, kv, ssm = QN.forward(st["model"], st["tokens"], start_pos=c["start"], kv_caches=st["kv"],
                                 ssm_states=[_clone(s) for s in st["saved"]])
    new = slice(c["start"], c["start"] + c["T"])
    return dict(logits=logits, k=kv[-1].k[new], v=kv[-1].v[new], ssm=[list(s) for s in ssm if s is not None])


def run(state):
    c, kind = state["case"], state["case"]["kind"]
    if kind in ("qmv", "linear"):
        return state["op"](state["x"])
    if kind == "chain":
        return state["op"](state["x"], residual=True)
    if kind == "moe":
        return state["op"](state["x"])
    if kind == "attn":
        cache = state["cache"]
        cache.length = c["start"]
        y, cache = QN.attn_forward(state["x"], state["layer"], state["cfg"], *state["rope"], cache, c["start"])
        new = slice(c["start"], c["start"] + c["T"])
        return dict(y=y, k=cache.k[new], v=cache.v[new])
    if kind == "ssm":
        y, (conv, S) = QN.ssm_forward(state["x"], state["layer"], state["cfg"], _clone(state["saved"]))
        return dict(y=y, conv=conv, S=S)
    return _run_model(state)


# ------------------------------------------------------------------ work
def _wbytes(fmt, n):
    _, bw, bb, _, _ = FORMATS[fmt]
    return n // bw * bb


def _moe_work(c, T):
    s = SHAPES[c["shape"]]
    D, FF, E, k = s["D"], s["FF"], s["E"], s["k"]
    used = E * (1 - (1 - k / E) ** T)                       # distinct experts of T tokens, about
    sh = c.get("shared", "iq")
    gs, ds = (c["gate"], c["down"]) if sh == "iq" else (sh, sh)
    w = used * (2 * _wbytes(c["gate"], FF * D) + _wbytes(c["down"], FF * D)) + 2 * _wbytes(gs, FF * D) \
        + _wbytes(ds, FF * D) + 4 * (E + 1) * D
    return w + 8 * T * D, 2 * T * D * (3 * FF * (k + 1) + E + 1)


def _attn_work(c, T, start):
    s = SHAPES[c["shape"]]
    D, Hq, Hkv, Dh = s["D"], s["n_head"], s["n_head_kv"], s["head_dim"]
    w = ((2 * Hq + 2 * Hkv) * Dh + Hq * Dh) * D
    pairs = T * start + T * (T + 1) // 2
    return 2 * w + 8 * T * D + 8 * Hkv * Dh * (start + 2 * T), 2 * T * w + 4 * Hq * Dh * pairs


def _ssm_work(c, T):
    s = SHAPES[c["shape"]]
    D, Sk, Hv = s["D"], s["d_state"], s["n_v_heads"]
    C = 2 * s["n_k_heads"] * Sk + Hv * Sk
    w = (C + 2 * Hv * Sk) * D
    return 2 * w + 8 * Hv * D + 8 * T * D + 8 * Hv * Sk * Sk + 24 * C, \
        2 * T * w + 4 * T * Hv * D + T * (8 * C + 7 * Hv * Sk * Sk)


def work(case):
    c, kind, T = case, case["kind"], case["T"]
    if kind == "qmv":
        return dict(bytes=_wbytes(c["fmt"], c["M"] * c["K"]) + 4 * T * (c["M"] + c["K"]), flops=2 * T * c["M"] * c["K"])
    if kind == "linear":
        return dict(bytes=2 * c["M"] * c["K"] + 4 * T * (c["M"] + c["K"]), flops=2 * T * c["M"] * c["K"])
    if kind == "chain":
        b, f = _moe_work(c, T)
        return dict(bytes=c["layers"] * b, flops=c["layers"] * f)
    if kind == "moe":
        b, f = _moe_work(c, T)
    elif kind == "attn":
        b, f = _attn_work(c, T, c["start"])
    elif kind == "ssm":
        b, f = _ssm_work(c, T)
    else:
        s = SHAPES[c["shape"]]
        parts = [_attn_work(c, T, c["start"]) if a else _ssm_work(c, T) for a in PATTERN]
        parts += [_moe_work(_model_case(c, i), T) for i in range(len(PATTERN))]
        b = sum(p[0] for p in parts) + 2 * s["vocab"] * s["D"] + 4 * T * s["vocab"]
        f = sum(p[1] for p in parts) + 2 * T * s["vocab"] * s["D"]
    return dict(bytes=b, flops=f)


# ------------------------------------------------------------------ tolerance
def tolerance(case):
    """About four times the error against 64 bits that the kinds show. Sums in 32 bits: 1e-7
    to 7e-7 (the chains and the whole step most). MoE blocks over more than 8 tokens whose
    experts are in the IQ formats multiply 16-bit activations: 1.7e-3. A decoder call that
    holds such blocks: 2e-3, and 8e-3 on 57 tokens where one token's eighth expert is so near
    to its ninth that the rounding decides between them."""
    if case["T"] > 8 and case["kind"] == "model":
        return {"rel": 2.5e-2}
    if case["T"] > 8 and case["kind"] == "moe" and case["gate"].startswith("iq"):
        return {"rel": 7e-3}
    return {"rel": 3e-6}


# ------------------------------------------------------------------ in 64 bits
# The IQ3_XXS grid: four values a point, each an octal digit into _GRID_LEVELS.
_GRID_LEVELS = (4, 12, 20, 28, 36, 44, 52, 62)
_GRID = (
    "000020004000110031007100020022001300240037005700101030100110211012105210031023101410451007100020"
    "202040201120022022201320332073201520752057201030703001302130523007303140734044407540374057401050"
    "705023502550536046600170417061703470167010013001010121011201320103012301430174010501001120111111"
    "021122111021302101212121122103212721003120310231133164316631104150410541025142516451175150612271"
    "047100022002110231020202220262021302240210123012501201122112121203123612761207120022202211227122"
    "022222227322042255221032013241320732473253423542305272521452475210723072617254721003010321031203"
    "320305035603270300132013021313134413641310233023012352232523272311333333034374432743005360532253"
    "555341636363366333730673400471045304730435047504471402247324042406246624703454344044154446445254"
    "345407545074017421740374210514050705001560156215551541252325272520353535014532457245274520551355"
    "056542752475420644066406460612161616712646260336633644465056255633663076127630075007700701072307"
    "2507621704172127542725270037513733370637124714470057205742570367"
)
_KVALUES = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _half(raw, o):
    return raw[:, o:o + 2].contiguous().view(torch.float16).double()


def _dequant(fmt, raw, K):
    """Raw rows [M, row bytes] -> float64 [M, K], from the formats' definitions."""
    _, bw, bb, _, _ = FORMATS[fmt]
    M = raw.shape[0]
    b = raw.reshape(-1, bb)
    n = b.shape[0]
    u = b.long()
    ar = lambda m: torch.arange(m, device=raw.device)      # noqa: E731
    if fmt == "q8_0":
        w = _half(b, 0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif fmt == "iq4_xs":
        high = u[:, 2] | u[:, 3] << 8
        ls = (u[:, 4:8].repeat_interleave(2, 1) >> (4 * (ar(8) % 2)) & 15) | ((high[:, None] >> 2 * ar(8) & 3) << 4)
        q = u[:, 8:].reshape(n, 8, 16)
        kv = torch.tensor(_KVALUES, device=raw.device, dtype=torch.float64)
        w = (_half(b, 0) * (ls - 32)).unsqueeze(2) * kv[torch.cat([q & 15, q >> 4], 2)]
    elif fmt == "iq3_xxs":
        lv = torch.tensor(_GRID_LEVELS, device=raw.device, dtype=torch.float64)
        grid = lv[torch.tensor([int(d) for d in _GRID], device=raw.device)].reshape(256, 4)
        g = grid[u[:, 2:66]].reshape(n, 8, 4, 8)
        aux = (u[:, 66:].reshape(n, 8, 4) << 8 * ar(4)).sum(2)
        s7 = aux.unsqueeze(2) >> 7 * ar(4) & 127
        bits = s7.unsqueeze(3) >> ar(8) & 1                # the eighth sign is the parity of the other seven
        bits[..., 7] = bits[..., :7].sum(3) & 1
        scale = _half(b, 0) * (0.5 + (aux >> 28).double()) * 0.5
        w = scale[:, :, None, None] * g * (1 - 2 * bits)
    elif fmt == "q6_k":
        ql, qh = u[:, :128].reshape(n, 2, 2, 32), u[:, 128:192].reshape(n, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)
        q = (low | ((qh >> (2 * ar(4))[:, None] & 3) << 4)) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        w = (_half(b, 208) * sc).repeat_interleave(16, 1) * q.reshape(n, 256)
    else:                                                  # q4_k, q5_k
        s = u[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6) << 4], 1)
        mn = torch.cat([s[:, 4:8] & 63, s[:, 8:] >> 4 | (s[:, 4:8] >> 6) << 4], 1)
        qs = u[:, -128:].reshape(n, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
        if fmt == "q5_k":
            q = q | (u[:, 16:48].unsqueeze(1) >> ar(8)[:, None] & 1) << 4
        w = (_half(b, 0) * sc).unsqueeze(2) * q - (_half(b, 2) * mn).unsqueeze(2)
    return w.reshape(M, K)


def _rms(x, w):
    return x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt() * w


def _moe64(x, c, w, gate_sh, down_sh, norm_w):
    s = SHAPES[c["shape"]]
    D, FF = s["D"], s["FF"]
    xn = _rms(x, norm_w.double())

    def ffn(t, gate, up, down, fg, fd):
        h = F.silu(t @ _dequant(fg, gate, D).T) * (t @ _dequant(fg, up, D).T)
        return h @ _dequant(fd, down, FF).T

    p = torch.softmax(xn @ w["router"].double().T + w["router_bias"].double(), -1)
    top, ids = p.topk(s["k"], -1)
    top = top / top.sum(-1, keepdim=True)
    y = torch.zeros_like(x)
    for e in ids.unique().tolist():
        t, j = (ids == e).nonzero(as_tuple=True)
        y[t] += top[t, j, None] * ffn(xn[t], w["gate"][e], w["up"][e], w["down"][e], c["gate"], c["down"])
    share = torch.sigmoid(xn @ w["sh_gate_inp"].double()).unsqueeze(1)
    return y + share * ffn(xn, w["gate_sh"], w["up_sh"], w["down_sh"], gate_sh, down_sh)


def _attn64(x, shape, W, prefix, start):
    s = SHAPES[shape]
    Hq, Hkv, Dh, rd = s["n_head"], s["n_head_kv"], s["head_dim"], s["rope_dim"]
    T = x.shape[0]
    W = {n: t.double() for n, t in W.items()}
    h = _rms(x, W["attn_norm"])
    q, gate = (h @ W["wq"].T).reshape(T, Hq, 2, Dh).unbind(2)
    k, v = (h @ W["wk"].T).reshape(T, Hkv, Dh), (h @ W["wv"].T).reshape(T, Hkv, Dh)
    q, k = _rms(q, W["q_norm"]), _rms(k, W["k_norm"])
    # the angles as the callers hand them over: a table in 32 bits
    cos, sin = (t[start:start + T, None].double() for t in
                QN.build_partial_rope_cache(rd, MAX_POS, s["theta"], device=DEV))

    def rope(t):
        a, b, rest = t[..., :rd // 2], t[..., rd // 2:rd], t[..., rd:]
        return torch.cat([t[..., :rd] * cos + torch.cat([-b, a], -1) * sin, rest], -1)

    q, k = rope(q), rope(k)
    ka, va = torch.cat([prefix[0].double(), k]), torch.cat([prefix[1].double(), v])
    out = torch.empty_like(q)
    mask = torch.arange(start + T, device=DEV)[None] > start + torch.arange(T, device=DEV)[:, None]
    for i in range(Hq):
        j = i * Hkv // Hq
        p = torch.softmax((q[:, i] @ ka[:, j].T / Dh ** 0.5).masked_fill(mask, -math.inf), -1)
        out[:, i] = p @ va[:, j]
    return (out * torch.sigmoid(gate)).reshape(T, Hq * Dh) @ W["wo"].T, k, v


def _ssm64(x, shape, W, state):
    s = SHAPES[shape]
    Hk, Hv, Sk, T = s["n_k_heads"], s["n_v_heads"], s["d_state"], x.shape[0]
    Ck = Hk * Sk
    W = {n: t.double() for n, t in W.items()}
    h = _rms(x, W["attn_norm"])
    mixed, z = (h @ W["w_in"].T).T, h @ W["w_gate"].T
    g = F.softplus(h @ W["alpha"].T + W["dt_bias"]) * W["a"]
    beta = torch.sigmoid(h @ W["beta"].T)
    conv0, S = (t[0].double() for t in state) if state is not None else (
        mixed.new_zeros(mixed.shape[0], 3), mixed.new_zeros(Hv, Sk, Sk))
    seen = torch.cat([conv0, mixed], 1)
    conv = F.silu(sum(W["conv1d"][:, j, None] * seen[:, j:j + T] for j in range(4))).T
    unit = lambda t: t / t.square().sum(-1, keepdim=True).clamp_min(EPS).sqrt()     # noqa: E731
    q = unit(conv[:, :Ck].reshape(T, Hk, Sk)).repeat(1, Hv // Hk, 1) / Sk ** 0.5
    k = unit(conv[:, Ck:2 * Ck].reshape(T, Hk, Sk)).repeat(1, Hv // Hk, 1)
    v = conv[:, 2 * Ck:].reshape(T, Hv, Sk)
    o = torch.empty_like(v)
    for t in range(T):
        S = S * torch.exp(g[t])[:, None, None]
        d = (v[t] - (S * k[t][:, :, None]).sum(1)) * beta[t][:, None]
        S = S + k[t][:, :, None] * d[:, None]
        o[t] = (S * q[t][:, :, None]).sum(1)
    o = _rms(o, W["ssm_norm"]).reshape(T, Hv * Sk) * F.silu(z)
    return o @ W["w_out"].T, seen[:, -3:].unsqueeze(0), S.unsqueeze(0)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "qmv":
        x = _inputs_x(c, seed).double()
        y = x @ _dequant(c["fmt"], _blocks(_gen(seed, 0), c["fmt"], c["M"], c["K"]), c["K"]).T
        return y[0] if c["T"] == 1 else y
    if kind == "linear":
        return _inputs_x(c, seed).double() @ _bf(_randn(_gen(seed, 0), c["M"], c["K"], scale=0.02)).double().T
    if kind in ("chain", "moe"):
        x = _inputs_x(c, seed).double()
        for i in range(c.get("layers", 1)):
            w, gs, ds = _moe_inputs(c, seed, layer=i)
            y = _moe64(x, c, w, gs, ds, w["norm_w"])
            x = x + y
        return x if kind == "chain" else y
    if kind == "attn":
        y, k, v = _attn64(_inputs_x(c, seed).double(), c["shape"], _attn_weights(c["shape"], seed),
                          _prefix(c["shape"], seed, c["start"]), c["start"])
        return dict(y=y.unsqueeze(0), k=k, v=v)
    if kind == "ssm":
        y, conv, S = _ssm64(_inputs_x(c, seed).double(), c["shape"], _ssm_weights(c["shape"], seed),
                            _ssm_state(c["shape"], seed) if c["saved"] else None)
        return dict(y=y.unsqueeze(0), conv=conv, S=S)
    w = _model_weights(c["shape"], seed)
    x = w["embd"][_tokens(c, seed)].double()
    states = []
    for i, is_attn in enumerate(PATTERN):
        mc = _model_case(c, i)
        if is_attn:
            W = _attn_weights(c["shape"], seed, i)
            y, k, v = _attn64(x, c["shape"], W, _prefix(c["shape"], seed, c["start"], i), c["start"])
        else:
            W = _ssm_weights(c["shape"], seed, i)
            y, conv, S = _ssm64(x, c["shape"], W, _ssm_state(c["shape"], seed, i) if c["start"] else None)
            states.append([conv, S])
        mw, gs, ds = _moe_inputs(mc, seed, layer=i)
        x = x + y
        x = x + _moe64(x, mc, mw, gs, ds, W["post_norm"])
    return dict(logits=_rms(x, w["onorm"].double()) @ w["head"].double().T, k=k, v=v, ssm=states)
