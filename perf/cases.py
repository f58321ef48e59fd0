"""The workloads this framework is timed on, from single layers to whole models, through the entry
points a program calls: pulsatrix_amd.models (CausalLM, Block, NextTokenLogits) and the kernel
library's C ABI through pulsatrix_amd.native.

listed() names the cases, draw() gives more of the same ranges, prepare() makes what a program holds
before the call (weights loaded, inputs in HBM, outputs allocated), run() is one call of the path,
work() its unavoidable bytes and operations, exact() the same results from float64 torch, and
tolerance() how far another fp32 implementation may be from the present one.
"""
import ctypes
import math

import numpy as np
import torch

from pulsatrix_amd import models
from pulsatrix_amd import native as N

# ---- the models ---------------------------------------------------------------------------------
# The repository's own shapes: the SmolLM2-135M one of the headline benchmark, Llama-3.2-1B's widths
# and Gemma-3-270m's. `layers` and `vocab` of a case replace the defaults.
SHAPES = {
    "smol": dict(vocab_size=49152, hidden_size=576, num_layers=30, num_heads=9, num_kv_heads=3, head_dim=64,
                 intermediate_size=1536, rms_norm_eps=1e-5, rope_theta=100000.0),
    "llama1b": dict(vocab_size=128256, hidden_size=2048, num_layers=16, num_heads=32, num_kv_heads=8, head_dim=64,
                    intermediate_size=8192, rms_norm_eps=1e-5, rope_theta=500000.0),
    "gemma270m": dict(vocab_size=262144, hidden_size=640, num_layers=18, num_heads=4, num_kv_heads=1, head_dim=256,
                      intermediate_size=2048, rms_norm_eps=1e-6, rope_theta=1e6, hidden_act=1, qk_norm=1, post_norms=1,
                      norm_weight_offset=1.0, embed_scale=float(np.float32(np.sqrt(640.0))),
                      query_pre_attn_scalar=256.0, rope_local_base=10000.0, sliding_window=512),
}
LXT_EPS = 1e-9
RULES = {  # LRPRuleConfig settings: AttnLRP as LXT runs it, the default epsilon rule, Zennit's Gamma
    "lxt": dict(rule=N.EPSILON, epsilon=LXT_EPS, bias_in_denominator=True),
    "eps": dict(rule=N.EPSILON, epsilon=1e-6),
    "gamma": dict(rule=N.GAMMA, epsilon=1e-6, gamma=0.25),
}
HEADS = {"smol": (9, 3, 64), "llama1b": (32, 8, 64), "wide": (8, 2, 128), "narrow": (4, 2, 40)}


def listed():
    return [
        # The headline: one 512-token sequence explained by a program that captured the step once.
        dict(name="explain_512_graph", kind="explain", shape="smol", layers=30, batch=1, seq=512, rule="lxt", graph=True),
        # A short prompt explained eagerly, its length new to the program: bound by launches.
        dict(name="explain_24", kind="explain", shape="smol", layers=30, batch=1, seq=24, rule="lxt", graph=False),
        # A long document through a shallower model (attention dominates).
        dict(name="explain_3072", kind="explain", shape="smol", layers=6, batch=1, seq=3072, rule="lxt", graph=False),
        # Two ragged sentences under Zennit's Gamma rule on every Linear and the head.
        dict(name="explain_gamma_2x203", kind="explain", shape="smol", layers=6, batch=2, seq=203, rule="gamma",
             graph=False),
        # A batch of long sequences at the 1B widths: the large GEMMs and wide attention grids.
        dict(name="explain_1b_8x1024", kind="explain", shape="llama1b", layers=2, vocab=49152, batch=8, seq=1024,
             rule="lxt", graph=False),
        # One TransformerBlock called on host arrays, forward and relevance (the module API).
        dict(name="block_128", kind="block", shape="smol", batch=1, seq=128),
        # Batched greedy decoding over KV caches.
        dict(name="generate_4x32", kind="generate", shape="gemma270m", layers=18, batch=4, prompt=64, new=32),
        # Every generated token explained over its prefix.
        dict(name="explain_generated_2x24", kind="explain_generated", shape="gemma270m", layers=18, batch=2, prompt=48,
             new=24, rule="lxt"),
        # A chat turn through the next-token function: a prompt, then one token a call, logits to the host.
        dict(name="next_token_200", kind="next_token", shape="smol", layers=30, prompt=200, steps=16),
        # One Linear of no round size: forward with bias, its epsilon relevance and its weight gradient.
        dict(name="linear_1000x577x1531", kind="linear", rows=1000, inputs=577, outputs=1531, bias=True),
        # One attention layer, forward and AttnLRP, three ragged sequences.
        dict(name="attention_3x777", kind="attention", heads="llama1b", batch=3, seq=777),
        # The row and element kernels a training step runs around its GEMMs, forward and backward.
        dict(name="rows_4096x2048", kind="rows", rows=4096, cols=2048),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["explain", "explain", "explain", "linear", "linear", "attention", "attention", "block",
                       "next_token", "generate", "explain_generated", "rows"])
    if kind == "explain":
        shape = rng.choice(["smol", "smol", "llama1b", "gemma270m"])
        layers = {"smol": rng.randint(2, 12), "llama1b": rng.randint(1, 2), "gemma270m": rng.choice([3, 6])}[shape]
        seq = _log(rng, 2, 700 if shape == "gemma270m" else 2400)
        batch = rng.randint(1, max(1, min(4, 4096 // seq)))
        rule = rng.choice(["lxt", "lxt", "eps", "gamma"]) if shape == "smol" and batch * seq <= 1024 else "lxt"
        c = dict(kind=kind, shape=shape, layers=layers, batch=batch, seq=seq, rule=rule, graph=rng.random() < 0.5)
        return dict(c, vocab=49152) if shape != "smol" else c
    if kind == "linear":
        while True:
            m, i, o = _log(rng, 1, 8192), _log(rng, 16, 8192), _log(rng, 16, 8192)
            if m * i * o <= 1 << 36:
                return dict(kind=kind, rows=m, inputs=i, outputs=o, bias=rng.random() < 0.5)
    if kind == "attention":
        while True:
            heads, b, s = rng.choice(sorted(HEADS)), rng.randint(1, 8), _log(rng, 1, 2048)
            if b * s * s * HEADS[heads][0] <= 8 * 1024 * 1024 * 32:
                return dict(kind=kind, heads=heads, batch=b, seq=s)
    if kind == "block":
        return dict(kind=kind, shape="smol", batch=rng.randint(1, 3), seq=_log(rng, 1, 512))
    if kind == "next_token":
        return dict(kind=kind, shape="smol", layers=rng.choice([10, 30]), prompt=_log(rng, 9, 700), steps=rng.randint(1, 24))
    if kind == "generate":
        return dict(kind=kind, shape="gemma270m", layers=rng.choice([6, 18]), batch=rng.randint(1, 8),
                    prompt=_log(rng, 2, 128), new=rng.randint(2, 32))
    if kind == "explain_generated":
        return dict(kind=kind, shape="gemma270m", layers=rng.choice([3, 6]), batch=rng.randint(1, 3),
                    prompt=_log(rng, 4, 64), new=rng.randint(2, 24), rule="lxt")
    while True:
        m, c = _log(rng, 1, 16384), _log(rng, 8, 8192)
        if m * c <= 1 << 24:
            return dict(kind="rows", rows=m, cols=c)


def _fields(case):
    f = dict(SHAPES[case["shape"]])
    f["num_layers"] = case.get("layers", 1)
    if "vocab" in case:
        f["vocab_size"] = case["vocab"]
    if f.get("sliding_window"):  # every sixth layer attends fully, the others slide
        f["sliding_layers"] = sum(1 << i for i in range(f["num_layers"]) if i % 6 != 5)
    return f


def _layout(f, block=False):
    """(name, shape) of every parameter in the flat blob's order."""
    d, H, K, D, F = (f[k] for k in ("hidden_size", "num_heads", "num_kv_heads", "head_dim", "intermediate_size"))
    layer = [("norm1", (d,)), ("q", (d, H * D)), ("k", (d, K * D)), ("v", (d, K * D)), ("o", (H * D, d))]
    if f.get("qk_norm"):
        layer += [("q_norm", (D,)), ("k_norm", (D,))]
    layer += [("norm2", (d,)), ("gate", (d, F)), ("up", (d, F)), ("down", (F, d))]
    if f.get("post_norms"):
        layer += [("post_attn", (d,)), ("post_mlp", (d,))]
    if block:
        return layer
    every = [("embed", (f["vocab_size"], d))]
    for i in range(f["num_layers"]):
        every += [("%d.%s" % (i, n), s) for n, s in layer]
    return every + [("norm", (d,))]


def _weights(f, seed, block=False):
    """The parameter blob (fp32, on the GPU) and its named views: N(0, 0.02), norm scales around 1."""
    lay = _layout(f, block)
    g = torch.Generator(device="cuda").manual_seed(seed)
    blob = torch.empty(sum(math.prod(s) for _, s in lay), device="cuda")
    blob.normal_(0.0, 0.02, generator=g)
    named, at = {}, 0
    for name, s in lay:
        v = blob[at:at + math.prod(s)].view(s)
        if len(s) == 1:
            v.mul_(5.0).add_(1.0 - f.get("norm_weight_offset", 0.0))
        named[name] = v
        at += math.prod(s)
    return blob, named


def _ids(case, seed, rows, cols):
    v = _fields(case)["vocab_size"]
    g = torch.Generator(device="cuda").manual_seed(seed + 77)
    return torch.randint(0, v, (rows, cols), device="cuda", generator=g)


class _DeviceArray:
    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f4", data=(ptr, False), version=2, strides=None)


def _view(ptr, shape):
    return torch.as_tensor(_DeviceArray(int(ptr), shape), device="cuda")


def _randn(g, *shape, scale=1.0):
    return torch.randn(*shape, device="cuda", generator=g) * scale


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


# ---- whole models -----------------------------------------------------------------------------------
def _lm(case, seed):
    f = _fields(case)
    blob, _ = _weights(f, seed)
    return models.CausalLM(N.model_config(**f), blob.cpu().numpy()), f


def _prepare_explain(case, seed):
    lm, f = _lm(case, seed)
    n, l = case["batch"], case["seq"]
    s = dict(lm=lm, n=n, l=l, f=f, rule=N.lrp_rule(**RULES[case["rule"]]), ids=_ids(case, seed, n, l).float(),
             tok=torch.zeros(n, l, device="cuda"), targets=torch.zeros(n, dtype=torch.int64, device="cuda"))
    s["run"] = _run_explain
    if case["graph"]:
        torch.cuda.synchronize()
        lm.capture_explain_rule(s["ids"].data_ptr(), n, l, s["rule"], s["tok"].data_ptr(), s["targets"].data_ptr())
        s["run"] = _run_replay
    return s


def _explain_outputs(s):
    lm, f = s["lm"], s["f"]
    emb = N.host().pxa_lm_last_embedding_relevance(lm.h)
    return dict(tokens=s["tok"], targets=s["targets"],
                logits=_view(lm.last_logits_ptr(), (s["n"], s["l"], f["vocab_size"])),
                embedding=_view(emb, (s["n"], s["l"], f["hidden_size"])))


def _run_explain(s):
    s["lm"].explain_device_rule(s["ids"].data_ptr(), s["n"], s["l"], s["rule"], s["tok"].data_ptr(),
                                s["targets"].data_ptr())
    return _explain_outputs(s)


def _run_replay(s):
    s["lm"].replay()
    return _explain_outputs(s)


def _prepare_generate(case, seed):
    lm, f = _lm(case, seed)
    n, p, new = case["batch"], case["prompt"], case["new"]
    ids = torch.zeros(n, p + new, device="cuda")
    ids[:, :p] = _ids(case, seed, n, p)
    return dict(run=_run_generate, lm=lm, n=n, p=p, new=new, ids=ids, picked=torch.zeros(n, p + new, device="cuda"))


def _run_generate(s):
    s["lm"].generate_device(s["ids"].data_ptr(), s["n"], s["p"], s["new"], s["p"] + s["new"], s["picked"].data_ptr())
    return dict(ids=s["ids"], logits=s["picked"])


def _prepare_explain_generated(case, seed):
    lm, f = _lm(case, seed)
    n, p, new = case["batch"], case["prompt"], case["new"]
    return dict(run=_run_explain_generated, lm=lm, n=n, p=p, new=new, ids=_ids(case, seed, n, p + new).float(),
                rule=N.lrp_rule(**RULES[case["rule"]]), rel=torch.zeros(new, n, p + new - 1, device="cuda"))


def _run_explain_generated(s):
    s["lm"].explain_generated_device(s["ids"].data_ptr(), s["n"], s["p"], s["new"], s["p"] + s["new"], s["rule"],
                                     s["rel"].data_ptr())
    return dict(tokens=s["rel"])


def _prepare_next_token(case, seed):
    lm, f = _lm(case, seed)
    total = case["prompt"] + case["steps"]
    return dict(run=_run_next_token, f=lm.next_token_logits(total), prompt=case["prompt"], steps=case["steps"],
                tokens=_ids(case, seed, 1, total)[0].cpu().numpy())


def _run_next_token(s):
    return [s["f"](s["tokens"][:s["prompt"] + i]) for i in range(s["steps"] + 1)]


def _prepare_block(case, seed):
    f = _fields(case)
    f["rope_theta"] = 10000.0
    blob, _ = _weights(f, seed, block=True)
    g = torch.Generator(device="cuda").manual_seed(seed + 5)
    x = _randn(g, case["batch"], case["seq"], f["hidden_size"])
    return dict(run=_run_block, block=models.Block(N.model_config(**dict(f, num_layers=1, vocab_size=0)), blob.cpu().numpy()),
                x=x.cpu().numpy())


def _run_block(s):
    y = s["block"].forward(s["x"])
    r = np.zeros_like(y)
    r[..., 0] = y[..., 0]  # the relevance of the output's first channel
    return dict(y=y, relevance=s["block"].relevance(r, 1e-6, False))


# ---- single layers --------------------------------------------------------------------------------
def _desc(m, n, k, a, lda, b, ldb, c, **more):
    d = N.GemmDesc()
    d.m, d.n, d.k, d.batch, d.inner, d.kgroups = m, n, k, 1, 1, 1
    d.a, d.b, d.c = N.operand(a.data_ptr(), lda), N.operand(b.data_ptr(), ldb), N.operand(c.data_ptr(), n)
    for key, v in more.items():
        setattr(d, key, v)
    return d


def _linear_inputs(case, seed):
    m, i, o = case["rows"], case["inputs"], case["outputs"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    x, w = _randn(g, m, i), _randn(g, i, o, scale=i ** -0.5)
    b = _randn(g, o, scale=0.1) if case["bias"] else None
    z = (x.double() @ w.double()).float()  # the forward's cached pre-bias output
    grad = _randn(g, m, o)                 # the gradient arriving at the output
    r = (z if b is None else z + b) * grad  # and the relevance: output times gradient
    return x, w, b, z, grad, r


def _prepare_linear(case, seed):
    m, i, o = case["rows"], case["inputs"], case["outputs"]
    x, w, b, z, grad, r = _linear_inputs(case, seed)
    y_z, y, r_in, dw = (torch.empty(*s, device="cuda") for s in ((m, o), (m, o), (m, i), (i, o)))
    # y = x W (+ b); r_in = x * ((r / stab(z (+ b))) W^T), LXT's epsilon rule; dW = x^T grad
    ops = [_desc(m, o, i, x, i, w, o, y_z, epilogue=N.EPI_STORE_BIAS if case["bias"] else N.EPI_STORE),
           _desc(m, i, o, r, o, w, o, r_in, trans_b=1, prologue=N.PRO_DIV_STAB, epilogue=N.EPI_MUL_X, eps=LXT_EPS,
                 z=N.operand(z.data_ptr(), o), x=N.operand(x.data_ptr(), i)),
           _desc(i, o, m, x, i, grad, o, dw, trans_a=1)]
    if b is not None:
        ops[0].c2, ops[0].e_bias = N.operand(y.data_ptr(), o), N.operand(b.data_ptr(), 0)
        ops[1].z_bias = N.operand(b.data_ptr(), 0)
    ws = torch.empty(max([N.gemm_workspace(d) // 4 for d in ops] + [4]), device="cuda")
    for d in ops:
        d.workspace, d.workspace_bytes = ws.data_ptr(), ws.numel() * 4
    out = dict(z=y_z, relevance=r_in, weight_gradient=dw)
    if b is not None:
        out["y"] = y
    return dict(run=_run_linear, ops=ops, out=out, keep=(x, w, b, z, grad, r, ws))


def _run_linear(s):
    stream = torch.cuda.current_stream().cuda_stream
    for d in s["ops"]:
        N.gemm(d, stream)
    return s["out"]


def _rope_tables(l, D, theta):
    inv = 1.0 / theta ** (torch.arange(0, D, 2, device="cuda", dtype=torch.float64) / D)
    a = torch.arange(l, device="cuda", dtype=torch.float64)[:, None] * inv
    return a.cos().float(), a.sin().float()


def _rotate(x, cos, sin):
    """Rotate-half RoPE of x (..., l, D) at positions 0 .. l - 1; sin negated turns it back."""
    h = x.shape[-1] // 2
    a, b = x[..., :h], x[..., h:]
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)


def _attention_inputs(case, seed):
    H, K, D = HEADS[case["heads"]]
    n, l = case["batch"], case["seq"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    z = _randn(g, n, l, H + 2 * K, D, scale=1.5)  # the packed q | k | v projections
    cos, sin = _rope_tables(l, D, 500000.0)
    rot = _rotate(z[:, :, :H + K].transpose(1, 2), cos, sin).transpose(1, 2).contiguous()
    spv = _randn(g, n, l, H, D)  # r_ctx / (2 ctx), what the output projection's relevance hands down
    return z, rot, spv, cos, sin


def _prepare_attention(case, seed):
    H, K, D = HEADS[case["heads"]]
    n, l = case["batch"], case["seq"]
    z, rot, spv, cos, sin = _attention_inputs(case, seed)
    e = lambda *s: torch.empty(*s, device="cuda")  # noqa: E731
    stats, ctx, row_sum, g = e(n, H, l, 2), e(n, l, H, D), e(n, H, l), e(n, l, H + 2 * K, D)
    key_rel, value_rel, p, sc = e(n, l, K, D), e(n, l, K, D), e(n, H, l, l), e(n, H, l, l)
    qd, kd, w3, rw = H * D, K * D, (H + 2 * K) * D, (H + K) * D
    zp, rp, gp = z.data_ptr(), rot.data_ptr(), g.data_ptr()
    common = dict(n=n, l=l, heads=H, kv_heads=K, head_dim=D, eps=LXT_EPS, causal=1, rope=1, rope_half=1,
                  cos_t=cos.data_ptr(), sin_t=sin.data_ptr(), ld_g=w3, spv=spv.data_ptr(), ld_spv=qd, q=rp, ld_q=rw,
                  k=rp + 4 * qd, ld_k=rw, v=zp + 4 * rw, ld_v=w3, s=sc.data_ptr(), ld_z=w3)
    rq = N.AttnRelDesc(scale=D ** -0.5, q_pre=zp, ld_q_pre=w3, z=zp, g=gp, ctx=ctx.data_ptr(), ld_ctx=qd,
                       stats=stats.data_ptr(), row_sum=row_sum.data_ptr(), p_out=p.data_ptr(), **common)
    rk = N.AttnRelKvDesc(p=p.data_ptr(), k_pre=zp + 4 * qd, ld_k_pre=w3, z_k=zp + 4 * qd, z_v=zp + 4 * rw,
                         key_rel=key_rel.data_ptr(), value_rel=value_rel.data_ptr(), ld_rel=kd, g_k=gp + 4 * qd,
                         g_v=gp + 4 * rw, **common)
    fwd = (rp, rw, rp + 4 * qd, rw, zp + 4 * rw, w3, None, None, stats.data_ptr(), ctx.data_ptr(), qd, n, l, H, K, D,
           D ** -0.5, 1)
    out = dict(context=ctx, stats=stats, row_sums=row_sum, shares=g, key=key_rel, value=value_rel)
    return dict(run=_run_attention, fwd=fwd, rq=rq, rk=rk, out=out, keep=(z, rot, spv, cos, sin, p, sc))


def _run_attention(s):
    lib, stream = N.pxk(), torch.cuda.current_stream().cuda_stream
    N.call("pxk_attention_forward_stats", *s["fwd"], stream)
    N.check(lib.pxk_attention_relevance_q(ctypes.byref(s["rq"]), stream))
    N.check(lib.pxk_attention_relevance_kv(ctypes.byref(s["rk"]), stream))
    return s["out"]


def _rows_inputs(case, seed):
    m, c = case["rows"], case["cols"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    return _randn(g, m, c), 1.0 + _randn(g, c, scale=0.1), _randn(g, m, c), _randn(g, m, c, scale=2.0)


def _prepare_rows(case, seed):
    m, c = case["rows"], case["cols"]
    x, gamma, grad, scores = _rows_inputs(case, seed)
    e = lambda *s: torch.empty(*s, device="cuda")  # noqa: E731
    out = dict(norm=e(m, c), rms=e(m), act=e(m, c), act_grad=e(m, c), x_grad=e(m, c), gamma_grad=e(c), softmax=e(m, c),
               score_grad=e(m, c), logsumexp=e(m))
    terms, silu = e(m, c), ctypes.c_int(4)
    calls = [("pxk_rms_norm_forward", x, gamma, out["norm"], out["rms"], m, c, 1e-5),
             ("pxk_elementwise", silu, out["norm"], out["act"], m * c),
             ("pxk_elementwise_backward", silu, out["norm"], grad, out["act_grad"], m * c),
             ("pxk_rms_norm_backward", out["act_grad"], gamma, x, out["rms"], out["x_grad"], terms, m, c),
             ("pxk_column_sums", terms, out["gamma_grad"], m, c, 0.0),
             ("pxk_softmax_rows", scores, out["softmax"], m, c),
             ("pxk_softmax_rows_backward", out["softmax"], grad, out["score_grad"], m, c),
             ("pxk_logsumexp_rows", scores, out["logsumexp"], m, c)]
    return dict(run=_run_rows, calls=[(getattr(N.pxk(), name), [_c(v) for v in args]) for name, *args in calls], out=out,
                keep=(x, gamma, grad, scores, terms))


def _c(v):
    """An argument as the C ABI takes it (the training ops are not in native's table of signatures)."""
    if isinstance(v, torch.Tensor):
        return ctypes.c_void_p(v.data_ptr())
    return ctypes.c_float(v) if isinstance(v, float) else ctypes.c_int64(v) if isinstance(v, int) else v


def _run_rows(s):
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for fn, args in s["calls"]:
        N.check(fn(*args, stream))
    return s["out"]


_PREPARE = dict(explain=_prepare_explain, generate=_prepare_generate, explain_generated=_prepare_explain_generated,
                next_token=_prepare_next_token, block=_prepare_block, linear=_prepare_linear,
                attention=_prepare_attention, rows=_prepare_rows)


# ---- unavoidable work -------------------------------------------------------------------------------
def _layer_params(f):
    d, H, K, D, F = (f[k] for k in ("hidden_size", "num_heads", "num_kv_heads", "head_dim", "intermediate_size"))
    return d * (H + 2 * K) * D + H * D * d + 3 * d * F


def _visible(l):
    return l * (l + 1) / 2


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, i, o = case["rows"], case["inputs"], case["outputs"]
        return dict(bytes=4.0 * (2 * m * i + 2 * i * o + (4 + case["bias"]) * m * o), flops=6.0 * m * i * o)
    if kind == "attention":
        H, K, D = HEADS[case["heads"]]
        n, l = case["batch"], case["seq"]
        rows = 4.0 * n * l * D
        return dict(bytes=rows * ((H + 2 * K) + (H + K) + H + H + (H + 2 * K) + 2 * K), flops=14.0 * n * H * _visible(l) * D)
    if kind == "rows":
        return dict(bytes=4.0 * 8 * case["rows"] * case["cols"], flops=40.0 * case["rows"] * case["cols"])
    f = _fields(case)
    d, V, H, D, layers, per = f["hidden_size"], f["vocab_size"], f["num_heads"], f["head_dim"], f["num_layers"], _layer_params(f)
    weights = 4.0 * (layers * per + V * d)
    # forward products per row, and per row and visible key
    if kind == "block":
        m, vis = case["batch"] * case["seq"], case["batch"] * _visible(case["seq"])
        return dict(bytes=4.0 * (per + 4 * m * d), flops=4.0 * m * per + 14.0 * vis * H * D)
    if kind == "explain":
        n, l = case["batch"], case["seq"]
        m, vis = n * l, n * _visible(l)
        back = 4 if case["rule"] == "gamma" else 1  # Gamma: two denominators and two backward products each way
        flops = 2.0 * m * layers * per * (1 + back) + 14.0 * vis * layers * H * D + 2.0 * m * d * V
        return dict(bytes=weights + 4.0 * m * (V + d + 1), flops=flops)
    if kind == "generate":
        n, p, new = case["batch"], case["prompt"], case["new"]
        rows = n * (p + new - 1)
        return dict(bytes=weights * new + 4.0 * n * new, flops=2.0 * rows * layers * per + 2.0 * n * new * d * V)
    if kind == "next_token":
        p, t = case["prompt"], case["steps"]
        return dict(bytes=weights * (t + 1) + 4.0 * V * (t + 1), flops=2.0 * (p + t) * layers * per + 2.0 * (t + 1) * d * V)
    n, p, new = case["batch"], case["prompt"], case["new"]
    rows = sum(n * (p + t) for t in range(new))
    return dict(bytes=weights + 4.0 * new * n * (p + new - 1),
                flops=2.0 * layers * per * (rows + n * (p + new - 1)) + 4.0 * new * n * d * V)


# About four times what the present code is off float64 (measured: logits, single layers and row kernels
# 1e-7 .. 4e-6, the relevance of whole models 8e-6 through 30 layers, 1.2e-4 through the Gemma blocks,
# whose QK-Norm and sandwich norms leave more near-zero denominators).
def tolerance(case):
    if case["kind"] in ("explain", "explain_generated"):
        return {"rel": 1e-3, "max": 0.05, "differ": 0.005} if case["shape"] == "gemma270m" else {"rel": 1e-4, "max": 0.02, "differ": 0.005}
    return {"rel": 1e-5, "differ": 0.005} if case["kind"] == "generate" else {"rel": 1e-5}


# ---- the same in float64 ------------------------------------------------------------------------------
def _stab(z, eps):
    return z + eps * torch.where(z >= 0, 1.0, -1.0).to(z.dtype)


def _rms(x, gamma, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * gamma


def _linear_rule(x, w, z, r, rule):
    """Relevance through z = x w (no bias) under the epsilon or the Gamma rule."""
    eps = rule["epsilon"]
    if rule["rule"] == N.EPSILON:
        return x * ((r / _stab(z, eps)) @ w.T)
    g, xp, xn = rule["gamma"], x.clamp(min=0), x.clamp(max=0)
    wa, wb = w + g * w.clamp(min=0), w + g * w.clamp(max=0)
    gp = torch.where(z > 0, r / _stab(xp @ wa + xn @ wb, eps), 0.0)
    gn = torch.where(z < 0, r / _stab(xp @ wb + xn @ wa, eps), 0.0)
    return xp * (gp @ wa.T + gn @ wb.T) + xn * (gp @ wb.T + gn @ wa.T)


def _split(a, b, r, eps):
    s = _stab(a + b, eps)
    return a / s * r, b / s * r


class _Layer:
    """One transformer block in float64, its forward cached for the relevance."""

    def __init__(self, f, w, slides=False):
        self.f, self.off = f, f.get("norm_weight_offset", 0.0)
        self.w = {k: v.double() + (self.off if v.dim() == 1 else 0.0) for k, v in w.items()}
        self.window = f.get("sliding_window", 0) if slides else 0
        self.theta = f["rope_local_base"] if slides and f.get("rope_local_base") else f["rope_theta"]

    def heads(self, t, h):
        n, l = t.shape[:2]
        return t.view(n, l, h, self.f["head_dim"]).transpose(1, 2)

    def forward(self, x):
        f, w, eps = self.f, self.w, self.f["rms_norm_eps"]
        H, K, D = f["num_heads"], f["num_kv_heads"], f["head_dim"]
        n, l, _ = x.shape
        self.x, self.x1 = x, _rms(x, w["norm1"], eps)
        self.zq, self.zk, self.zv = self.x1 @ w["q"], self.x1 @ w["k"], self.x1 @ w["v"]
        self.pq, self.pk, v = self.heads(self.zq, H), self.heads(self.zk, K), self.heads(self.zv, K)
        if f.get("qk_norm"):
            self.pq, self.pk = _rms(self.pq, w["q_norm"], eps), _rms(self.pk, w["k_norm"], eps)
        self.cos, self.sin = (t.double() for t in _rope_tables(l, D, self.theta))
        self.q, self.k = _rotate(self.pq, self.cos, self.sin), _rotate(self.pk, self.cos, self.sin)
        self.kk, self.vv = self.k.repeat_interleave(H // K, 1), v.repeat_interleave(H // K, 1)
        self.scale = (f.get("query_pre_attn_scalar") or D) ** -0.5
        i = torch.arange(l, device=x.device)
        self.seen = i[None, :] <= i[:, None]
        if self.window:
            self.seen = self.seen & (i[None, :] > i[:, None] - self.window)
        self.raw = self.q @ self.kk.transpose(-1, -2)
        self.p = (self.raw * self.scale).masked_fill(~self.seen, -math.inf).softmax(-1)
        self.ctx = self.p @ self.vv
        self.merged = self.ctx.transpose(1, 2).reshape(n, l, H * D)
        self.zo = self.merged @ w["o"]
        self.attn = _rms(self.zo, w["post_attn"], eps) if f.get("post_norms") else self.zo
        self.y1 = x + self.attn
        self.x2 = _rms(self.y1, w["norm2"], eps)
        self.zg, self.zu = self.x2 @ w["gate"], self.x2 @ w["up"]
        act = torch.nn.functional
        self.gate = act.gelu(self.zg, approximate="tanh") if f.get("hidden_act") else act.silu(self.zg)
        self.hid = self.gate * self.zu
        self.zd = self.hid @ w["down"]
        self.ffn = _rms(self.zd, w["post_mlp"], eps) if f.get("post_norms") else self.zd
        return self.y1 + self.ffn

    def relevance(self, r, rule):
        f, w, eps = self.f, self.w, rule["epsilon"]
        H, K, D = f["num_heads"], f["num_kv_heads"], f["head_dim"]
        n, l, _ = r.shape
        r_y1, r_ffn = _split(self.y1, self.ffn, r, eps)
        r_hid = _linear_rule(self.hid, w["down"], self.zd, r_ffn, rule)
        half = self.hid / (2 * self.hid + eps * torch.where(self.hid >= 0, 1.0, -1.0)) * r_hid
        r_y1 = r_y1 + _linear_rule(self.x2, w["gate"], self.zg, half, rule) + _linear_rule(self.x2, w["up"], self.zu, half, rule)
        r_x, r_attn = _split(self.x, self.attn, r_y1, eps)
        r_ctx = self.heads(_linear_rule(self.merged, w["o"], self.zo, r_attn, rule), H)
        spv = r_ctx / (2 * self.ctx + eps * torch.where(self.ctx >= 0, 1.0, -1.0))
        rq, rk, rv = self.core(spv, eps)[:3]
        flat = lambda t: t.transpose(1, 2).reshape(n, l, -1)  # noqa: E731
        return (r_x + _linear_rule(self.x1, w["q"], self.zq, flat(rq), rule)
                + _linear_rule(self.x1, w["k"], self.zk, flat(rk), rule)
                + _linear_rule(self.x1, w["v"], self.zv, flat(rv), rule))

    def core(self, spv, eps):
        """The attention core's AttnLRP: relevance of q, k (before RoPE) and v, and the row sums."""
        n, H, l, D = self.q.shape
        K = self.k.shape[1]
        r_p = self.p * (spv @ self.vv.transpose(-1, -2))
        rows = r_p.sum(-1, keepdim=True)
        r_s = self.scale * self.raw * (r_p - self.p * rows)
        del r_p
        s = (r_s / (2 * self.raw + eps * torch.where(self.raw >= 0, 1.0, -1.0))).masked_fill(~self.seen, 0.0)
        del r_s
        group = lambda t: t.view(n, K, H // K, l, D).sum(2)  # noqa: E731
        r_q = self.q * (s @ self.kk)
        r_k = group(self.kk * (s.transpose(-1, -2) @ self.q))
        r_v = group(self.vv * (self.p.transpose(-1, -2) @ spv))
        back = lambda x, y, r: x * _rotate(r / _stab(y, eps), self.cos, -self.sin)  # noqa: E731
        return back(self.pq, self.q, r_q), back(self.pk, self.k, r_k), r_v, rows[..., 0]


class _Model:
    def __init__(self, case, seed):
        self.f = f = _fields(case)
        _, w = _weights(f, seed)
        self.embed = w["embed"].double()
        slide = f.get("sliding_layers", 0)
        self.layers = [_Layer(f, {k.split(".")[1]: v for k, v in w.items() if k.startswith("%d." % i)}, slide >> i & 1)
                       for i in range(f["num_layers"])]
        self.norm = w["norm"].double() + f.get("norm_weight_offset", 0.0)

    def hidden(self, ids):
        x = self.embed[ids] * (self.f.get("embed_scale") or 1.0)
        for layer in self.layers:
            x = layer.forward(x)
        self.h = _rms(x, self.norm, self.f["rms_norm_eps"])
        return self.h

    def relevance(self, targets, rule):
        """The relevance of each sequence's last row's logit `targets`, at the embeddings."""
        h = self.h[:, -1]
        z = h @ self.embed.T
        r = torch.zeros_like(z).scatter_(1, targets[:, None], z.gather(1, targets[:, None]))
        top = torch.zeros_like(self.h)
        top[:, -1] = _linear_rule(h, self.embed.T, z, r, rule)
        for layer in reversed(self.layers):
            top = layer.relevance(top, rule)
        return top


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def _exact_explain(case, seed):
    m, ids = _Model(case, seed), _ids(case, seed, case["batch"], case["seq"])
    logits = m.hidden(ids) @ m.embed.T
    targets = logits[:, -1].argmax(-1)
    r = m.relevance(targets, RULES[case["rule"]])
    return dict(tokens=r.sum(-1), targets=targets, logits=logits, embedding=r)


def _exact_generate(case, seed):
    m, n, p, new = _Model(case, seed), case["batch"], case["prompt"], case["new"]
    ids = _ids(case, seed, n, p)
    picked = torch.zeros(n, p + new, device="cuda", dtype=torch.float64)
    for t in range(new):
        top = (m.hidden(ids)[:, -1] @ m.embed.T).max(-1)
        picked[:, p + t] = top.values
        ids = torch.cat([ids, top.indices[:, None]], 1)
    return dict(ids=ids.double(), logits=picked)


def _exact_explain_generated(case, seed):
    m, n, p, new = _Model(case, seed), case["batch"], case["prompt"], case["new"]
    ids = _ids(case, seed, n, p + new)
    out = torch.zeros(new, n, p + new - 1, device="cuda", dtype=torch.float64)
    for t in range(new):
        m.hidden(ids[:, :p + t])
        out[t, :, :p + t] = m.relevance(ids[:, p + t], RULES[case["rule"]]).sum(-1)
    return dict(tokens=out)


def _exact_next_token(case, seed):
    m, p, t = _Model(case, seed), case["prompt"], case["steps"]
    logits = m.hidden(_ids(case, seed, 1, p + t))[0, p - 1:] @ m.embed.T
    return [row for row in logits]


def _exact_block(case, seed):
    f = dict(_fields(case), rope_theta=10000.0)
    layer = _Layer(f, _weights(f, seed, block=True)[1])
    g = torch.Generator(device="cuda").manual_seed(seed + 5)
    y = layer.forward(_randn(g, case["batch"], case["seq"], f["hidden_size"]).double())
    r = torch.zeros_like(y)
    r[..., 0] = y[..., 0]
    return dict(y=y, relevance=layer.relevance(r, dict(rule=N.EPSILON, epsilon=1e-6)))


def _exact_linear(case, seed):
    x, w, b, z, grad, r = (None if t is None else t.double() for t in _linear_inputs(case, seed))
    y = x @ w
    zb = z if b is None else z + b
    out = dict(z=y, relevance=x * ((r / _stab(zb, LXT_EPS)) @ w.T), weight_gradient=x.T @ grad)
    return out if b is None else dict(out, y=y + b)


def _exact_attention(case, seed):
    H, K, D = HEADS[case["heads"]]
    z, rot, spv, cos, sin = (t.double() for t in _attention_inputs(case, seed))
    n, l = z.shape[:2]
    a = _Layer(dict(num_heads=H, num_kv_heads=K, head_dim=D, rope_theta=1.0), {})
    heads = lambda t: t.transpose(1, 2)  # noqa: E731
    a.pq, a.pk, v = heads(z[:, :, :H]), heads(z[:, :, H:H + K]), heads(z[:, :, H + K:])
    a.q, a.k, a.cos, a.sin = heads(rot[:, :, :H]), heads(rot[:, :, H:]), cos, sin
    a.kk, a.vv, a.scale = a.k.repeat_interleave(H // K, 1), v.repeat_interleave(H // K, 1), D ** -0.5
    i = torch.arange(l, device=z.device)
    a.seen = i[None, :] <= i[:, None]
    a.raw = a.q @ a.kk.transpose(-1, -2)
    x = (a.raw * a.scale).masked_fill(~a.seen, -math.inf)
    a.p = x.softmax(-1)
    top = x.max(-1).values
    stats = torch.stack([top, 1.0 / (x - top[..., None]).exp().sum(-1)], -1)
    ctx = a.p @ a.vv
    rq, rk, rv, rows = a.core(heads(spv), LXT_EPS)
    shares = torch.cat([heads(t) for t in (rq, rk, rv)], 2) / _stab(z, LXT_EPS)
    return dict(context=heads(ctx), stats=stats, row_sums=rows, shares=shares, key=heads(rk), value=heads(rv))


def _exact_rows(case, seed):
    x, gamma, grad, scores = (t.double() for t in _rows_inputs(case, seed))
    rms = (x.square().mean(-1) + 1e-5).sqrt()
    norm = x / rms[:, None] * gamma
    sig = norm.sigmoid()
    back = grad * sig * (1 + norm * (1 - sig))
    terms = back * x / rms[:, None]
    gx = back * gamma
    x_grad = (gx - x * (gx * x).mean(-1, keepdim=True) / rms[:, None].square()) / rms[:, None]
    p = scores.softmax(-1)
    return dict(norm=norm, rms=rms, act=norm * sig, act_grad=back, x_grad=x_grad, gamma_grad=terms.sum(0), softmax=p,
                score_grad=p * (grad - (p * grad).sum(-1, keepdim=True)), logsumexp=scores.logsumexp(-1))


_EXACT = dict(explain=_exact_explain, generate=_exact_generate, explain_generated=_exact_explain_generated,
              next_token=_exact_next_token, block=_exact_block, linear=_exact_linear, attention=_exact_attention,
              rows=_exact_rows)
