"""The many-token kernels against plain 64-bit references at the edges of their tiles: the
dense bf16 GEMM, the prompts of the core layers, and the grouped MoE kernels over I8 rows."""
import numpy as np
import pytest
import torch

from npu_amd import ops
from npu_amd.gguf_types import GGMLQuantizationType as QT

pytestmark = pytest.mark.gpu


# (M, K, T): 128 x 64 tiles with an odd M (scalar stores) and a last half step, in few steps
# and in 17 (both LDS buffers in turn); K split in two with a K of one step, and with an odd
# count of steps and a short second part; K split in four with a last part that is short, and
# parts that hold no step at all, one token past a tile; the few-token kernel's last sizes and
# the first ones that the tiles take: over 16 tokens, over 32, and for a short K
@pytest.mark.parametrize("M,K,T", [(4099, 96, 700), (4096, 32, 300), (2050, 1056, 260), (3072, 160, 65),
                                   (3072, 2048, 17), (3072, 2048, 16), (4099, 1056, 700), (2050, 1056, 520),
                                   (3072, 160, 129), (5872, 2048, 32), (5888, 2048, 17), (3184, 1024, 64),
                                   (3200, 1024, 64), (5184, 544, 64), (5200, 544, 64)])
def test_gemm_bf16_tiles(gpu, M, K, T):
    g = torch.Generator().manual_seed(M + K + T)
    w = (torch.randn(M, K, generator=g) * 0.05).to(torch.bfloat16)
    x = torch.randn(T, K, generator=g) * torch.exp(torch.randn(T, 1, generator=g))
    print(f"gemm case M={M} K={K} T={T}", flush=True)
    y = ops.matvec(QT.BF16, w.to(gpu), M, K, x.to(gpu)).cpu().double()
    ref = x.double() @ w.double().T
    # every product is exact; a value is a chain of at most 24 + K / 64 additions of 32-product
    # sums, each rounding at most 2^-24 of the sum of magnitudes (twice that for the inner sums)
    bound = (2 * 24 + K / 64 + 4) * 2.0 ** -24 * (x.abs().double() @ w.abs().double().T)
    assert bool(((y - ref).abs() <= bound).all())
    assert float((y - ref).norm() / ref.norm()) <= 1e-6


# the three tile shapes, and the few-token kernel as the core layers' prompts run it
@pytest.mark.parametrize("M,T", [(9216, 300), (9216, 120), (9216, 57), (1024, 12)])
def test_bf16_products_unbiased(gpu, M, T):
    """The mean error of a prompt's v rows against 64 bits, in units of their size: an attention
    over them averages out everything else.  Rounding errors of either sign leave 1.2e-7 over
    the root of their number (at most 1e-9 here); sums that all round down leave 2e-8 to 3e-8."""
    from npu_amd import qwen_core as QN
    print(f"gemm bias case M={M} T={T}", flush=True)
    D, Hkv, Dh = 2048, 1, 256
    cfg = QN.Config(d_model=D, n_head=(M - 2 * Hkv * Dh) // (2 * Dh), n_head_kv=Hkv, head_dim=Dh, rope_dim=0)
    g = torch.Generator().manual_seed(M + T)
    bf = lambda *s: (torch.randn(*s, generator=g) * 0.02).to(torch.bfloat16).float()
    Hq = cfg.n_head
    ones = torch.ones(Dh)
    layer = QN.AttnLayer(i=0, attn_norm=torch.ones(D), post_norm=torch.ones(D), wq=bf(2 * Hq * Dh, D), wk=bf(Hkv * Dh, D),
                         wv=bf(Hkv * Dh, D), wo=bf(D, Hq * Dh), q_norm=ones, k_norm=ones)
    err, n, size = 0.0, 0, 0.0
    for _ in range(max(1, 400 // T)):
        x = torch.randn(1, T, D, generator=g)
        _, c = QN.attn_forward(x.to(gpu), layer, cfg, torch.zeros(T, 0), torch.zeros(T, 0), None, 0)
        xd = x[0].double()
        ref = (xd * (xd.square().mean(1, keepdim=True) + cfg.rms_eps).rsqrt()) @ layer.wv.double().T
        e = c.v[:T, 0].cpu().double() - ref
        err, n, size = err + float(e.sum()), n + e.numel(), size + float(ref.square().sum())
    assert abs(err / n) / (size / n) ** 0.5 <= 3e-9, err / n / (size / n) ** 0.5


# ---- prompts through the core layers (gm_attn_prefill / gm_ssm_prefill)
def _cfgs(**kw):
    from npu_amd import qwen_core as QN
    from oracle import qwen_core as QC
    kw = dict(dict(d_model=512, n_head=4, n_head_kv=2, head_dim=128, rope_dim=32, rope_theta=1e6,
                   ssm_d_inner=256, ssm_d_state=64, ssm_n_k_heads=2, ssm_n_v_heads=4), **kw)
    return QC.CoreCfg(**kw), QN.Config(**kw)


def _rel(a, b):
    return float((a.double().cpu() - b.double()).abs().max() / b.double().abs().max())


def _attn(ocfg, seed):
    g = torch.Generator().manual_seed(seed)
    D, Hq, Hkv, Dh = ocfg.d_model, ocfg.n_head, ocfg.n_head_kv, ocfg.head_dim
    bf = lambda *s: (torch.randn(*s, generator=g) * 0.03).to(torch.bfloat16).float()
    nw = lambda n: 1 + 0.1 * torch.randn(n, generator=g)
    return dict(attn_norm=nw(D), post_norm=nw(D), wq=bf(2 * Hq * Dh, D), wk=bf(Hkv * Dh, D), wv=bf(Hkv * Dh, D),
                wo=bf(D, Hq * Dh), q_norm=2 * nw(Dh), k_norm=2 * nw(Dh))


# one query block with its keys in 5 parts, blocks that end inside a position's heads (G = 3),
# every head_dim, a rotation over the whole head, one token past a block and past the part of
# 1024, no rotation
@pytest.mark.parametrize("kw,parts", [
    (dict(), (2, 700, 2, 17)),
    (dict(n_head=6, n_head_kv=2, head_dim=64, rope_dim=64), (5, 43, 1, 22)),
    (dict(n_head=16, n_head_kv=2, head_dim=256, rope_dim=96), (9, 8, 130)),
    (dict(n_head=2, n_head_kv=2, head_dim=512, rope_dim=0), (3, 65)),
    (dict(n_head=4, n_head_kv=1, head_dim=64, rope_dim=16), (1025, 2)),
])
def test_attention_prompts(gpu, kw, parts):
    """A sequence fed in parts of several tokens, each on the cache of the parts before, against
    the oracle fed the same way: fp32 sums in another order, bar 1e-4 as for single steps."""
    from npu_amd import qwen_core as QN
    from oracle import qwen_core as QC
    print(f"attention prompt case {kw} {parts}", flush=True)
    ocfg, ncfg = _cfgs(**kw)
    W = _attn(ocfg, 31)
    OL, NL = QC.AttnW(**W), QN.AttnLayer(i=0, **W)
    cos, sin = QC.build_partial_rope_cache(ocfg.rope_dim, sum(parts) + 3, ocfg.rope_theta)
    x = torch.randn(1, sum(parts), ocfg.d_model, generator=torch.Generator().manual_seed(32))
    oc = nc = None
    pos = 0
    for i, n in enumerate(parts):
        xp = x[:, pos:pos + n]
        yo, oc = QC.attn_forward(xp, OL, ocfg, cos, sin, oc, pos)
        yn, nc = QN.attn_forward(xp.to(gpu), NL, ncfg, cos, sin, nc, pos, residual=i == 1)
        pos += n
        assert nc.length == pos
        assert _rel(yn - xp.to(gpu) if i == 1 else yn, yo) <= 1e-4, f"part {i}"
    rep = ocfg.n_head // ocfg.n_head_kv
    assert _rel(nc.k[:pos], oc[0][0, :, ::rep]) <= 1e-5 and _rel(nc.v[:pos], oc[1][0, :, ::rep]) <= 1e-5
    assert not nc.k[pos:].any()                            # nothing past the filled positions


# eight, three and one row a position, on a cache whose keys are cut into parts and without one
@pytest.mark.parametrize("kw,prefix", [(dict(n_head=8, n_head_kv=1, head_dim=256), 300),
                                       (dict(n_head=6, n_head_kv=2, head_dim=64), 0),
                                       (dict(n_head=2, n_head_kv=2, head_dim=128), 400)])
def test_attention_prompt_non_finite_token(gpu, kw, prefix):
    """A token with a NaN or infinity reaches itself and the tokens after it, as one token at a
    time: the finite outputs are the same ones, with the same values to fp32 sums (2-norm)."""
    from npu_amd import qwen_core as QN
    print(f"attention non-finite case {kw} {prefix}", flush=True)
    ocfg, ncfg = _cfgs(**kw)
    NL = QN.AttnLayer(i=0, **_attn(ocfg, 33))
    T = 61
    cos, sin = QN.build_partial_rope_cache(ocfg.rope_dim, prefix + T, ocfg.rope_theta)
    g = torch.Generator().manual_seed(34)
    x = torch.randn(1, T, ocfg.d_model, generator=g)
    x[0, 21, 5], x[0, 45, 7] = float("nan"), float("inf")
    x = x.to(gpu)
    caches = [QN.KVCache(ncfg, prefix + T) for _ in range(2)]
    k, v = (torch.randn(prefix, ocfg.n_head_kv, ocfg.head_dim, generator=g).to(gpu) for _ in range(2))
    for c in caches:
        c.k[:prefix], c.v[:prefix], c.length = k, v, prefix
    y, _ = QN.attn_forward(x, NL, ncfg, cos, sin, caches[0], prefix)
    steps = [QN.attn_forward(x[:, t:t + 1], NL, ncfg, cos, sin, caches[1], prefix + t)[0] for t in range(T)]
    ref = torch.cat(steps, 1)
    assert torch.equal(y.isfinite(), ref.isfinite())
    assert bool(y[0, :21].isfinite().all()) and not y[0, 21:].isfinite().any()
    # each within 5e-7 of 64 bits
    assert float((y[0, :21] - ref[0, :21]).double().norm() / ref[0, :21].double().norm()) <= 1e-6


# 128 and 256 dims a head, on a cache whose keys are cut into parts
@pytest.mark.parametrize("kw", [dict(), dict(d_model=1024, n_head=8, n_head_kv=1, head_dim=256)])
def test_attention_prompt_no_less_exact_than_steps(gpu, kw):
    """A prompt's outputs, k and v against 64 bits, beside the error of the same tokens one at a
    time: sums of some 60,000 rounding errors of either sign and more, whose norms chance moves
    by less than a hundredth; the bar leaves two."""
    from npu_amd import qwen_core as QN
    print(f"attention precision case {kw}", flush=True)
    ocfg, ncfg = _cfgs(**kw)
    W = _attn(ocfg, 61)
    W["q_norm"], W["k_norm"] = W["q_norm"] / 2, W["k_norm"] / 2        # scores of about one
    T, prefix = 120, 500
    Hq, Hkv, Dh, rd = ocfg.n_head, ocfg.n_head_kv, ocfg.head_dim, ocfg.rope_dim
    cos, sin = QN.build_partial_rope_cache(rd, prefix + T, ocfg.rope_theta)
    g = torch.Generator().manual_seed(62)
    x = torch.randn(1, T, ocfg.d_model, generator=g)
    k0, v0 = torch.randn(prefix, Hkv, Dh, generator=g), 0.5 * torch.randn(prefix, Hkv, Dh, generator=g)
    # in 64 bits
    w64 = {n: t.double() for n, t in W.items()}
    rms = lambda t, w: t * (t.square().mean(-1, keepdim=True) + ocfg.rms_eps).rsqrt() * w
    h = rms(x[0].double(), w64["attn_norm"])
    q, gate = (h @ w64["wq"].T).reshape(T, Hq, 2, Dh).unbind(2)
    k, v = (h @ w64["wk"].T).reshape(T, Hkv, Dh), (h @ w64["wv"].T).reshape(T, Hkv, Dh)
    c, s = (t[prefix:, None].double() for t in (cos, sin))
    rope = lambda t: torch.cat([t[..., :rd] * c + torch.cat([-t[..., rd // 2:rd], t[..., :rd // 2]], -1) * s, t[..., rd:]], -1)
    q, k = rope(rms(q, w64["q_norm"])), rope(rms(k, w64["k_norm"]))
    ka, va = (torch.cat([p.double(), t]).repeat_interleave(Hq // Hkv, 1) for p, t in ((k0, k), (v0, v)))
    mask = torch.arange(prefix + T)[None] > prefix + torch.arange(T)[:, None]
    sc = torch.stack([q[:, i] @ ka[:, i].T for i in range(Hq)]) / Dh ** 0.5
    pr = torch.softmax(sc.masked_fill(mask, float("-inf")), -1)
    o = torch.stack([pr[i] @ va[:, i] for i in range(Hq)], 1) * torch.sigmoid(gate)
    ref = (o.reshape(T, -1) @ w64["wo"].T, k, v)
    layer = QN.AttnLayer(i=0, **W)

    def run(parts):
        cache = QN.KVCache(ncfg, prefix + T)
        cache.k[:prefix], cache.v[:prefix], cache.length = k0.to(gpu), v0.to(gpu), prefix
        ys = [QN.attn_forward(xp.to(gpu), layer, ncfg, cos, sin, cache, cache.length)[0] for xp in x.split(parts, 1)]
        return torch.cat(ys, 1)[0], cache.k[prefix:], cache.v[prefix:]
    err = lambda a, b: float((a.double().cpu() - b).norm() / b.norm())
    for n, a, b, r in zip("ykv", run(T), run(1), ref):
        print(f"{n} {err(a, r):.3e} against {err(b, r):.3e}", flush=True)
        assert err(a, r) <= 1.02 * err(b, r), n


# d_state 64 / 128 / 256, prompts around the 16 staged tokens (8 at 256) and past the part of
# 1024, conv kernels of 1, 2 and 8 taps, and a prompt shorter than the conv state
@pytest.mark.parametrize("kw,parts", [
    (dict(), (2, 16, 1, 33)),
    (dict(ssm_d_inner=512, ssm_d_state=128, ssm_d_conv=8), (3, 2, 31)),
    (dict(ssm_d_inner=1024, ssm_d_state=256, ssm_d_conv=2, ssm_n_k_heads=1), (9, 8)),
    (dict(ssm_d_conv=1, ssm_n_k_heads=4), (5, 18)),
    (dict(ssm_d_inner=128, ssm_n_k_heads=1, ssm_n_v_heads=2), (1026, 3)),
])
def test_ssm_prompts(gpu, kw, parts):
    from npu_amd import qwen_core as QN
    from oracle import qwen_core as QC
    print(f"ssm prompt case {kw} {parts}", flush=True)
    ocfg, ncfg = _cfgs(**kw)
    g = torch.Generator().manual_seed(41)
    D, Hv, Hk, S = ocfg.d_model, ocfg.ssm_n_v_heads, ocfg.ssm_n_k_heads, ocfg.ssm_d_state
    C = 2 * Hk * S + Hv * S
    bf = lambda *s: (torch.randn(*s, generator=g) * 0.03).to(torch.bfloat16).float()
    r = lambda *s, sc=1.0: torch.randn(*s, generator=g) * sc
    W = dict(attn_norm=1 + r(D, sc=0.1), post_norm=1 + r(D, sc=0.1), w_in=bf(C, D), w_gate=bf(Hv * S, D),
             conv1d=r(C, ocfg.ssm_d_conv, sc=0.5), a=-torch.rand(Hv, generator=g), alpha=r(Hv, D, sc=0.05),
             beta=r(Hv, D, sc=0.05), dt_bias=r(Hv, sc=0.5), ssm_norm=1 + r(S, sc=0.1), w_out=bf(D, Hv * S))
    OL, NL = QC.SSMW(**W), QN.SSMLayer(i=0, **W)
    x = torch.randn(1, sum(parts), D, generator=torch.Generator().manual_seed(42))
    ck = ocfg.ssm_d_conv
    os_ = (torch.zeros(1, C, ck - 1), torch.zeros(1, Hv, S, S))
    ns = None
    pos = 0
    for i, n in enumerate(parts):
        xp = x[:, pos:pos + n]
        # the oracle's new conv state is cin[..., -(ck - 1):], which for one tap is everything
        yo, os_ = QC.ssm_forward(xp, OL, ocfg, os_)
        os_ = (os_[0][..., :ck - 1] if ck == 1 else os_[0], os_[1])
        yn, ns = QN.ssm_forward(xp.to(gpu), NL, ncfg, ns, residual=i == 1)
        pos += n
        assert _rel(yn - xp.to(gpu) if i == 1 else yn, yo) <= 1e-4, f"part {i}"
        assert _rel(ns[1], os_[1]) <= 1e-4, f"part {i}: recurrent state"
        if ck > 1:
            assert _rel(ns[0], os_[0]) <= 1e-5, f"part {i}: conv state"


def test_ssm_prompt_no_less_exact_than_steps(gpu):
    """A prompt's outputs and new state against 64 bits, beside the error of the same tokens one
    at a time.  Both are sums of some 1e6 rounding errors of either sign, whose norms over as
    many values differ by less than a hundredth by chance; the bar leaves five."""
    from npu_amd import qwen_core as QN
    from oracle import qwen_core as QC
    kw = dict(d_model=2048, ssm_d_inner=1024, ssm_d_state=128, ssm_n_k_heads=4, ssm_n_v_heads=8)
    print("ssm precision case", flush=True)
    ocfg, ncfg = _cfgs(**kw)
    g = torch.Generator().manual_seed(51)
    D, Hv, Hk, S = 2048, 8, 4, 128
    C = 2 * Hk * S + Hv * S
    r = lambda *s, sc=1.0: torch.randn(*s, generator=g) * sc
    bf = lambda *s: r(*s, sc=0.02).to(torch.bfloat16).float()
    W = dict(attn_norm=1 + r(D, sc=0.1), post_norm=1 + r(D, sc=0.1), w_in=bf(C, D), w_gate=bf(Hv * S, D),
             conv1d=r(C, 4, sc=0.5), a=-torch.rand(Hv, generator=g), alpha=r(Hv, D, sc=0.05), beta=r(Hv, D, sc=0.05),
             dt_bias=r(Hv, sc=0.5), ssm_norm=1 + r(S, sc=0.1), w_out=bf(D, Hv * S))
    T = 500
    x = r(1, T, D)
    ref, (_, Sr) = QC.ssm_forward(x.double(), QC.SSMW(**{n: t.double() for n, t in W.items()}), ocfg,
                                  (torch.zeros(1, C, 3).double(), torch.zeros(1, Hv, S, S).double()))
    layer = QN.SSMLayer(i=0, **W)
    y, st = QN.ssm_forward(x.to(gpu), layer, ncfg, None)
    steps, ss = [], None
    for t in range(T):
        yt, ss = QN.ssm_forward(x[:, t:t + 1].to(gpu), layer, ncfg, ss)
        steps.append(yt)
    err = lambda a, b: float((a.double().cpu() - b).norm() / b.norm())
    y1, s1 = torch.cat(steps, 1), ss[1]
    print(f"y {err(y, ref):.3e} against {err(y1, ref):.3e}, state {err(st[1], Sr):.3e} against {err(s1, Sr):.3e}", flush=True)
    assert err(y, ref) <= 1.05 * err(y1, ref)
    assert err(st[1], Sr) <= 1.05 * err(s1, Sr)


# the widths from which two tokens are two steps, and those below where they are a prompt; past
# 3500 cached positions an attention layer of any width
@pytest.mark.parametrize("D,prefix,steps", [(1024, 3, True), (992, 3, False), (512, 3500, True), (512, 3499, False)])
def test_two_tokens(gpu, D, prefix, steps, monkeypatch):
    """Two tokens go the faster way: the bits of two single calls, or one prompt call."""
    from npu_amd import qwen_core as QN
    print(f"two tokens case {D} {prefix}", flush=True)
    ocfg, ncfg = _cfgs(d_model=D)
    g = torch.Generator().manual_seed(81)
    r = lambda *s, sc=1.0: torch.randn(*s, generator=g) * sc
    bf = lambda *s: r(*s, sc=0.03).to(torch.bfloat16).float()
    A = QN.AttnLayer(i=0, **_attn(ocfg, 82))
    S = QN.SSMLayer(i=0, attn_norm=1 + r(D, sc=0.1), post_norm=1 + r(D, sc=0.1), w_in=bf(512, D), w_gate=bf(256, D),
                    conv1d=r(512, 4, sc=0.5), a=-torch.rand(4, generator=g), alpha=r(4, D, sc=0.05),
                    beta=r(4, D, sc=0.05), dt_bias=r(4, sc=0.5), ssm_norm=1 + r(64, sc=0.1), w_out=bf(D, 256))
    cos, sin = QN.build_partial_rope_cache(ocfg.rope_dim, prefix + 2, ocfg.rope_theta)
    x = r(1, 2, D).to(gpu)
    k, v = r(prefix, 2, 128).to(gpu), r(prefix, 2, 128).to(gpu)
    prompts = []
    for cls in (QN.GpuAttn, QN.GpuSsm):
        monkeypatch.setattr(cls, "prompt", lambda self, *a, _f=cls.prompt, _c=cls: (prompts.append(_c), _f(self, *a))[1])

    def attn(parts):
        c = QN.KVCache(ncfg, prefix + 2)
        c.k[:prefix], c.v[:prefix], c.length = k, v, prefix
        y = torch.cat([QN.attn_forward(xp, A, ncfg, cos, sin, c, c.length)[0] for xp in x.split(parts, 1)], 1)
        assert c.length == prefix + 2
        return y, c.k, c.v

    def ssm(parts):
        st, ys = None, []
        for xp in x.split(parts, 1):
            y, st = QN.ssm_forward(xp, S, ncfg, st)
            ys.append(y)
        return torch.cat(ys, 1), *st

    for fn, cls, one in ((attn, QN.GpuAttn, steps), (ssm, QN.GpuSsm, D >= 1024)):
        two, single = fn(2), fn(1)
        assert (cls not in prompts) == one
        for a, b in zip(two, single):
            assert torch.equal(a, b) if one else float((a - b).norm() / b.norm()) <= 1e-6


# wide enough for the 128 x 64 tiles in the input projections (of two matrices in the DeltaNet
# layer) and for the same with K split in two in the output projection with its residual
@pytest.mark.parametrize("kind", ["attn", "ssm"])
def test_wide_core_prompts(gpu, kind):
    """Against the same tokens one at a time: each within 4e-7 of 64 bits (2-norm)."""
    from npu_amd import qwen_core as QN
    print(f"wide prompt case {kind}", flush=True)
    ocfg, ncfg = _cfgs(d_model=2048, n_head=16, n_head_kv=2, head_dim=256, rope_dim=64, ssm_d_inner=4096,
                       ssm_d_state=128, ssm_n_k_heads=16, ssm_n_v_heads=32)
    T, g = 520, torch.Generator().manual_seed(71)
    r = lambda *s, sc=1.0: torch.randn(*s, generator=g) * sc
    bf = lambda *s: r(*s, sc=0.02).to(torch.bfloat16).float()
    x = r(1, T, 2048).to(gpu)
    if kind == "attn":
        layer = QN.AttnLayer(i=0, **_attn(ocfg, 72))
        cos, sin = QN.build_partial_rope_cache(64, T, ocfg.rope_theta)
        call = lambda xp, st: QN.attn_forward(xp, layer, ncfg, cos, sin, st, st.length if st else 0, residual=True)
    else:
        layer = QN.SSMLayer(i=0, attn_norm=1 + r(2048, sc=0.1), post_norm=1 + r(2048, sc=0.1), w_in=bf(8192, 2048),
                            w_gate=bf(4096, 2048), conv1d=r(8192, 4, sc=0.5), a=-torch.rand(32, generator=g),
                            alpha=r(32, 2048, sc=0.05), beta=r(32, 2048, sc=0.05), dt_bias=r(32, sc=0.5),
                            ssm_norm=1 + r(128, sc=0.1), w_out=bf(2048, 4096))
        call = lambda xp, st: QN.ssm_forward(xp, layer, ncfg, st, residual=True)
    y, st = call(x, None)
    ys, ss = [], None
    for t in range(T):
        yt, ss = call(x[:, t:t + 1], ss)
        ys.append(yt)
    state = lambda s: (s.k[:T], s.v[:T]) if kind == "attn" else s
    for a, b in zip((y - x, *state(st)), (torch.cat(ys, 1) - x, *state(ss))):
        assert float((a - b).double().norm() / b.double().norm()) <= 1e-6


# ---- MoE blocks with I8 routed experts over more than 8 tokens (prefill_i8.hip)
def _i8_block(gpu, D, FF, E, k, q_gate, q_down, shared, seed):
    from npu_amd import synth
    from npu_amd.moe import GpuMoeBlock
    h = synth.host_moe_layer(seed, D=D, FF=FF, E=E, k=k, q_gate=q_gate, q_down=q_down, shared=shared, norm=True)
    return GpuMoeBlock.from_host(h, device=gpu)


# the first T past the decode kernels (mostly one token an expert), experts with two whole
# segments and one token, or about two segments (few experts), one row tile, odd counts of 128-wide steps, no shared expert
@pytest.mark.parametrize("D,FF,E,k,T,q_gate,q_down,shared", [
    (512, 256, 64, 8, 9, QT.Q6_K, QT.Q5_K, True),
    (256, 256, 2, 2, 33, QT.Q8_0, QT.Q6_K, True),
    (256, 512, 4, 1, 128, QT.Q5_K, QT.Q4_K, False),
    (768, 256, 16, 4, 130, QT.Q4_K, QT.Q8_0, True),
    (2048, 512, 256, 8, 41, QT.Q6_K, QT.Q6_K, True),
])
def test_moe_i8_prompts(gpu, D, FF, E, k, T, q_gate, q_down, shared):
    """Against the same tokens through the decode kernels, eight at a time.  Both keep the
    weights exact and the activations to 2^-23 with fp32 sums (each within 1e-6 of 64 bits),
    so their difference is held to 3e-6 of the outputs; ids and weights come from the same
    logits to fp32 rounding."""
    print(f"i8 prompt case D={D} FF={FF} E={E} k={k} T={T} {q_gate} {q_down} {shared}", flush=True)
    blk = _i8_block(gpu, D, FF, E, k, q_gate, q_down, shared, 300 + T)
    g = torch.Generator().manual_seed(T)
    x = (torch.randn(T, D, generator=g) * torch.exp(torch.randn(T, 1, generator=g))).to(gpu)
    y = blk(x, residual=True)
    ids = blk.stages(T)["topk_ids"].clone()
    parts, pids = [], []
    for t in range(0, T, 8):
        parts.append(blk(x[t:t + 8], residual=True))
        pids.append(blk.stages(len(x[t:t + 8]))["topk_ids"].clone())
    assert torch.equal(ids, torch.cat(pids))
    ref = torch.cat(parts).double()
    err = (y.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= 3e-6, float(err.max())
    assert torch.equal(y, blk(x, residual=True))           # fixed order: the same bits again


@pytest.mark.parametrize("side", ["x", "h"])
def test_moe_i8_prompt_quiet_sub_blocks(gpu, side):
    """Activations beside an outlier of their row that meets zero weights only, so that all of
    the outputs comes from the quiet ones: as exact as through the decode kernels (each
    sub-block of 32 to 2^-23 of its own largest), bar as above."""
    from npu_amd import synth
    from npu_amd.moe import GpuMoeBlock
    D, FF, E, k, T = 512, 256, 4, 2, 40
    print(f"i8 quiet case {side}", flush=True)
    h = synth.host_moe_layer(370, D=D, FF=FF, E=E, k=k, q_gate=QT.Q8_0, q_down=QT.Q8_0)
    half = lambda v: np.frombuffer(np.float16(v).tobytes(), np.uint8)
    blocks = lambda w: w.reshape(*w.shape[:-1], -1, 34)    # 34 bytes per 32 weights, the scale first
    x = torch.randn(T, D, generator=torch.Generator().manual_seed(371))
    if side == "x":
        x[:, 3] = 2.0 ** 24
        for w in (h.gate, h.up, h.gate_sh, h.up_sh):
            blocks(w)[..., 0, :2] = 0
        h.router[:, 3] = 0
        h.sh_gate_inp[3] = 0
    else:                                                  # hidden value 5 at about 2^20 times the others and more
        for w in (h.gate, h.up, h.gate_sh, h.up_sh):
            blocks(w)[..., 5, :, :2] = half(2000.0)
        for w in (h.down, h.down_sh):
            blocks(w)[..., 0, :2] = 0
    blk = GpuMoeBlock.from_host(h, device=gpu)
    x = x.to(gpu)
    y = blk(x).double()
    ref = torch.cat([blk(x[t:t + 8]) for t in range(0, T, 8)]).double()
    err = (y - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= 3e-6, float(err.max())


@pytest.mark.parametrize("q_gate,q_down", [(QT.Q8_0, QT.Q5_K), (QT.Q6_K, QT.Q6_K), (QT.Q4_K, QT.Q5_K)])
def test_moe_i8_prompt_no_less_exact_than_steps(gpu, q_gate, q_down):
    """Against 64 bits, beside the error of the decode kernels on the same tokens (both are some
    80,000 sums of rounding errors of either sign: norms that chance alone moves by less than a
    hundredth; the bar leaves five)."""
    from npu_amd import synth
    from npu_amd.moe import GpuMoeBlock
    from oracle import moe as OM
    T = 40
    print(f"i8 precision case {q_gate} {q_down}", flush=True)
    h = synth.host_moe_layer(380, D=2048, FF=512, E=8, k=8, q_gate=q_gate, q_down=q_down)
    blk = GpuMoeBlock.from_host(h, device=gpu)
    x = torch.randn(T, 2048, generator=torch.Generator().manual_seed(381))
    ref = OM.moe_forward_dense64(x, OM.OracleLayer(h))
    err = lambda y: float((y.cpu().double() - ref).norm() / ref.norm())
    y, steps = blk(x.to(gpu)), torch.cat([blk(x[t:t + 8].to(gpu)) for t in range(0, T, 8)])
    print(f"{err(y):.3e} against {err(steps):.3e}", flush=True)
    assert err(y) <= 1.05 * err(steps)


@pytest.mark.parametrize("D,f32", [(2048, True), (2048, False), (4096, True)])
def test_moe_i8_prompt_logits_no_less_exact_than_steps(gpu, D, f32):
    """The router's logits against 64 bits, beside the decode kernels' on the same tokens: norms
    over 6,400 rounding errors, which chance moves by about a hundredth; the bar leaves five."""
    from npu_amd import synth
    from npu_amd.moe import GpuMoeBlock
    from oracle import moe as OM
    T, E = 100, 64
    print(f"i8 logits case D={D} {f32}", flush=True)
    h = synth.host_moe_layer(390, D=D, FF=256, E=E, k=4, q_gate=QT.Q8_0, q_down=QT.Q8_0, shared=False, router_f32=f32)
    blk = GpuMoeBlock.from_host(h, device=gpu)
    x = torch.randn(T, D, generator=torch.Generator().manual_seed(391))
    ref = OM.router_logits64(x, OM.OracleLayer(h))

    def logits(xp):
        blk(xp.to(gpu))
        return blk.stages(len(xp))["ffn_moe_logits"].double().cpu()
    err = lambda a: float((a - ref).norm() / ref.norm())
    one, steps = err(logits(x)), err(torch.cat([logits(xp) for xp in x.split(4)]))
    print(f"{one:.3e} against {steps:.3e}", flush=True)
    assert one <= 1.05 * steps


def test_moe_i8_prompt_in_a_small_workspace(gpu):
    """A workspace too small for the planes of the I8 GEMMs still runs the tokens (as decode
    chunks): the static scratch of gm_moe_forward_noalloc, at a T that fits an IQ layer."""
    import ctypes
    from npu_amd import _lib as L, synth
    from npu_amd.moe import GpuMoeBlock
    blk = _i8_block(gpu, 2048, 512, 16, 8, QT.Q6_K, QT.Q6_K, True, 350)
    iq = GpuMoeBlock.from_host(synth.host_moe_layer(351, D=2048, FF=512, E=16, k=8, norm=True), device=gpu)
    limit = 16 << 20
    T = max(t for t in range(9, 400) if ops.moe_workspace_bytes(iq.struct, t) <= limit)
    assert ops.moe_workspace_bytes(blk.struct, T) > limit
    x = torch.randn(T, 2048, generator=torch.Generator().manual_seed(1)).to(gpu)
    y = torch.empty_like(x)
    L.check(L.lib().gm_moe_forward_noalloc(ctypes.byref(blk.struct), L.ptr(x), L.ptr(y), T, 0, L.stream_ptr()), "noalloc")
    ref = blk(x).double()
    assert float((y.double() - ref).norm() / ref.norm()) <= 3e-6


# ---- MoE blocks with IQ routed experts (prefill.hip)
# segments of 64 tokens (many pairs per expert and enough of them to fill the chip) in every
# format pair, with one row group per block (D = 256) and ragged last segments; the SwiGLU width
# of three superblocks, in segments of 32
@pytest.mark.parametrize("D,FF,E,k,T,q_gate,q_down", [
    (512, 512, 16, 4, 1040, QT.IQ4_XS, QT.IQ3_XXS),
    (256, 256, 8, 4, 2053, QT.IQ3_XXS, QT.IQ4_XS),
    (1024, 512, 12, 8, 515, QT.IQ3_XXS, QT.IQ3_XXS),
    (256, 512, 16, 8, 601, QT.IQ4_XS, QT.IQ4_XS),
    (512, 768, 8, 2, 77, QT.IQ4_XS, QT.IQ3_XXS),
    (256, 768, 8, 2, 40, QT.IQ3_XXS, QT.IQ4_XS),
])
def test_moe_iq_prompt_segments(gpu, D, FF, E, k, T, q_gate, q_down):
    """Against the oracle, to the prefill tests' tolerance (f16 and bf16 operands: 2^-9 of a
    product each, max-norm over a row of sums)."""
    from npu_amd import synth
    from test_gpu_prefill import _check
    h = synth.host_moe_layer(400 + T, D=D, FF=FF, E=E, k=k, q_gate=q_gate, q_down=q_down, bias=True)
    _check(gpu, h, T, seed=T)
