"""The workloads the framework's speed is measured on.

Each listed case is one thing a user of the library has it do, through its
public entry points (include/intllm_hip.h by way of the ctypes bindings in
int-llm_amd/intllm, and the C host's model calls): GEMVs, the decode MLP,
decode attention, the token-batched GEMM, prefill attention, and whole
generate / decode / prefill calls.  Sizes are those of the repository's own
configurations (the tiny Llama and the TinyLlama shape) and generic ones.
Every result is an integer and must be the same word for word.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "int-llm_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import intllm  # noqa: E402

ONE = 1 << 48
DEV = "cuda:0"
MAX_SEQ = 4096      # cache rows of the attention and long-context cases
EMBED_ROWS = 64     # rows of the embedding table in the decode MLP cases

# dim, n_heads, n_kv_heads, head_dim, n_layers, ffn, vocab
TINY = dict(dim=256, nh=8, nkv=2, hd=32, layers=2, ffn=688, vocab=512)
TINYLLAMA = dict(dim=2048, nh=32, nkv=4, hd=64, layers=22, ffn=5632, vocab=32000)


def listed():
    return [
        # a whole greedy generate on the tiny model: prompt and 24 tokens, the
        # smallest call a program makes; launches and host calls are all of it
        dict(name="generate_tiny", kind="generate", **TINY, T=16, n=24),
        # one projection of odd sizes, as a model with unusual dims has them
        dict(name="gemv_ragged", kind="gemv", M=1031, K=2047),
        # the MLP of one decoded token: embedding row, gate|up with SwiGLU,
        # down with the residual, int64 weights
        dict(name="decode_mlp", kind="mlp", dim=2048, ffn=5632, bf16=False),
        # the same with bfloat16-resident weights
        dict(name="decode_mlp_bf16", kind="mlp", dim=2048, ffn=5632, bf16=True),
        # one decoded token's attention, chat-sized context
        dict(name="attn_decode_short", kind="attn", nh=32, nkv=4, hd=64, pos=120),
        # and over a long cache
        dict(name="attn_decode_long", kind="attn", nh=32, nkv=4, hd=64, pos=2060),
        # the q|k|v projection of a short prompt, weights as they are
        dict(name="gemm_128", kind="gemm", T=128, N=2560, K=2048, prepared=False),
        # gate|up of a long prompt, weight planes prepared once
        dict(name="gemm_2048", kind="gemm", T=2048, N=11264, K=2048, prepared=True),
        # a later chunk of a long prompt attending to itself and what came before
        dict(name="attn_prefill_chunk", kind="pfattn", nh=32, nkv=4, hd=64, T=512, p0=512),
        # the headline: 32 greedy tokens of the TinyLlama shape from position 40
        dict(name="decode_tinyllama", kind="decode", **TINYLLAMA, T=40, n=32, bf16=False,
             sampled=False),
        # long-context sampled decoding with bfloat16-resident weights
        dict(name="decode_long_sampled", kind="decode", **TINYLLAMA, T=2060, n=16, bf16=True,
             sampled=True),
        # the prompt of a long document, the last row's logits
        dict(name="prefill_tinyllama", kind="prefill", **TINYLLAMA, T=1500),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["generate", "gemv", "mlp", "attn", "attn", "gemm", "gemm", "pfattn",
                       "decode", "prefill"])
    if kind == "gemv":
        K = _logint(rng, 64, 8192)
        return dict(kind=kind, M=_logint(rng, 64, min(32000, (1 << 26) // K)), K=K)
    if kind == "mlp":
        bf16 = rng.random() < 0.5
        step = 512 if bf16 else rng.choice([2, 16, 64])
        dim = max(step, _logint(rng, 256, 4096) // step * step)
        return dict(kind=kind, dim=dim, ffn=max(step, _logint(rng, 256, 8192) // step * step),
                    bf16=bf16)
    if kind in ("attn", "pfattn"):
        hd = rng.choice([32, 64, 64, 128])
        nkv = rng.choice([1, 2, 4, 8])
        nh = nkv * rng.choice([1, 2, 4, 7, 8])
        if kind == "attn":
            return dict(kind=kind, nh=nh, nkv=nkv, hd=hd, pos=_logint(rng, 8, MAX_SEQ) - 1)
        T = _logint(rng, 16, 1024)
        return dict(kind=kind, nh=min(nh, 32) // nkv * nkv, nkv=nkv, hd=hd, T=T,
                    p0=rng.choice([0, rng.randrange(0, 1024)]))
    if kind == "gemm":
        return dict(kind=kind, T=_logint(rng, 2, 2048), N=_logint(rng, 128, 11264),
                    K=_logint(rng, 128, 5632), prepared=rng.random() < 0.5)
    # whole models between the tiny and the TinyLlama shape, few layers
    hd = rng.choice([32, 64, 128])
    nkv = rng.choice([2, 4])
    nh = nkv * rng.choice([2, 4])
    bf16 = kind == "decode" and rng.random() < 0.4
    if bf16:
        nh = max(nh, 512 // hd) // nkv * nkv
        nh = nh if nh * hd % 512 == 0 else 8 * nkv
    m = dict(dim=nh * hd, nh=nh, nkv=nkv, hd=hd, layers=rng.randrange(1, 5),
             ffn=_logint(rng, 1, 11) * 512 if bf16 else _logint(rng, 300, 5632),
             vocab=_logint(rng, 500, 32000))
    if kind == "generate":
        return dict(kind=kind, **m, T=_logint(rng, 2, 300), n=rng.randrange(4, 25))
    if kind == "prefill":
        return dict(kind=kind, **m, T=_logint(rng, 3, 2000))
    return dict(kind=kind, **m, T=_logint(rng, 8, 3000), n=rng.randrange(4, 33), bf16=bf16,
                sampled=rng.random() < 0.4)


# ---- inputs ------------------------------------------------------------------

_contexts = {}


def _context(hd=0):
    """A program's one context; its RoPE tables serve one head size, so the
    attention cases keep one context per head size."""
    if hd not in _contexts:
        _contexts[hd] = intllm.Context(0)
        if hd:
            _contexts[hd].rope_init(hd, MAX_SEQ, 10000)
    return _contexts[hd]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & ((1 << 62) - 1))


def _weights(g, n, sigma=0.02, mean=0.0):
    """bfloat16 values as Q16.48 words: what bfloat16_to_q1648 makes of a
    checkpoint's N(0, 0.02) weights (toward zero where bits fall below 2^-48)."""
    w = (torch.randn(n, generator=g, device=DEV) * sigma + mean).to(torch.bfloat16)
    return (w.double() * float(ONE)).to(torch.int64)


def _acts(g, n, sigma=1.0):
    """Activations: every fraction bit in use."""
    return (torch.randn(n, generator=g, device=DEV, dtype=torch.float64) * (sigma * ONE)).to(
        torch.int64)


def _empty(*shape):
    return torch.zeros(shape, dtype=torch.int64, device=DEV)


class _Model:
    """A HostModel with random weights, uploaded through a pinned buffer."""

    def __init__(self, case, seed, max_seq):
        self.ctx = _context()
        dim, kvd, ffn = case["dim"], case["nkv"] * case["hd"], case["ffn"]
        self.cfg = intllm.Config(dim, case["nh"], case["nkv"], case["hd"], case["layers"], ffn,
                                 case["vocab"], max_seq, 10000)
        self.m = intllm.HostModel(self.ctx, self.cfg)
        g = _gen(seed)
        big = max(case["vocab"] * dim, dim * dim, ffn * dim)
        host = torch.empty(big, dtype=torch.int64, pin_memory=True)

        def up(name, n, **kw):
            host[:n].copy_(_weights(g, n, **kw))
            self.m.upload(name, host[:n].numpy())

        up("model.embed_tokens.weight", case["vocab"] * dim)
        up("model.norm.weight", dim, sigma=0.1, mean=1.0)
        up("lm_head.weight", case["vocab"] * dim)
        for i in range(case["layers"]):
            p = "model.layers.%d." % i
            up(p + "input_layernorm.weight", dim, sigma=0.1, mean=1.0)
            up(p + "post_attention_layernorm.weight", dim, sigma=0.1, mean=1.0)
            for t, n in (("self_attn.q_proj", dim * dim), ("self_attn.k_proj", kvd * dim),
                         ("self_attn.v_proj", kvd * dim), ("self_attn.o_proj", dim * dim),
                         ("mlp.gate_proj", ffn * dim), ("mlp.up_proj", ffn * dim),
                         ("mlp.down_proj", dim * ffn)):
                up(p + t + ".weight", n)
        rng = np.random.RandomState(seed & 0x7FFFFFFF)
        self.tokens = [int(t) for t in rng.randint(3, case["vocab"], case["T"])]
        self.seed = int(seed)

    def __del__(self):
        m = self.__dict__.get("m")
        if m is not None:
            m.free()


def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    s = dict(case=case)
    if kind == "gemv":
        s.update(ctx=_context(), W=_weights(g, case["M"] * case["K"]), x=_acts(g, case["K"]),
                 y=_empty(case["M"]))
    elif kind == "mlp":
        dim, ffn, ctx = case["dim"], case["ffn"], _context()
        s.update(ctx=ctx, table=_weights(g, EMBED_ROWS * dim),
                 token=int(seed) % EMBED_ROWS, norm=_weights(g, dim, sigma=0.1, mean=1.0),
                 Wgu=_weights(g, 2 * ffn * dim), Wd=_weights(g, dim * ffn),
                 hidden=_empty(dim), h=_empty(ffn), stats=_empty(intllm.stats_words(dim)),
                 stats2=_empty(intllm.stats_words(dim)))
        if case["bf16"]:
            torch.cuda.synchronize()
            for name in ("Wgu", "Wd"):
                b = torch.empty(s[name].numel(), dtype=torch.int16, device=DEV)
                if not ctx.bf16_pack(b.data_ptr(), s[name].data_ptr(), b.numel()):
                    raise RuntimeError("weights are not bfloat16 values")
                s[name] = b
    elif kind == "attn":
        nh, nkv, hd = case["nh"], case["nkv"], case["hd"]
        s.update(ctx=_context(hd), q=_acts(g, nh * hd), k=_acts(g, nkv * hd),
                 v=_acts(g, nkv * hd), kc=_acts(g, MAX_SEQ * nkv * hd),
                 vc=_acts(g, MAX_SEQ * nkv * hd), out=_empty(nh, hd))
    elif kind == "pfattn":
        nh, nkv, hd = case["nh"], case["nkv"], case["hd"]
        s.update(ctx=_context(hd), qkv=_acts(g, case["T"] * (nh + 2 * nkv) * hd),
                 kc=_acts(g, MAX_SEQ * nkv * hd), vc=_acts(g, MAX_SEQ * nkv * hd),
                 out=_empty(case["T"], nh, hd))
    elif kind == "gemm":
        T, N, K, ctx = case["T"], case["N"], case["K"], _context()
        s.update(ctx=ctx, W=_weights(g, N * K), X=_acts(g, T * K), Y=_empty(T, N))
        if case["prepared"]:
            s["Wp"] = torch.empty(ctx.gemm_planes_bytes(N, K), dtype=torch.uint8, device=DEV)
            torch.cuda.synchronize()
            ctx.gemm_prepare(s["Wp"].data_ptr(), s["W"].data_ptr(), N, K)
    else:
        max_seq = 2048 if case["T"] + case.get("n", 0) <= 2048 else MAX_SEQ
        model = s["model"] = _Model(case, seed, max_seq)
        if kind == "decode":
            # the cache a program has before it decodes: its prompt's
            model.m.prefill(model.tokens, 0, case["vocab"], logits=False, choose=False)
            if case["bf16"]:
                model.m.set_bf16(True)
    return s


# ---- one pass ----------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "gemv":
        s["ctx"].gemv(s["y"].data_ptr(), s["W"].data_ptr(), s["x"].data_ptr(), case["M"],
                      case["K"])
        return s["y"]
    if kind == "mlp":
        ctx, dim, ffn = s["ctx"], case["dim"], case["ffn"]
        p = {k: v.data_ptr() for k, v in s.items() if isinstance(v, torch.Tensor)}
        ctx.embed_stats(p["hidden"], p["table"], s["token"], dim, p["stats"])
        up, down = ((ctx.norm_gemv_swiglu_stats_bf16, ctx.gemv_residual_stats_bf16)
                    if case["bf16"] else (ctx.norm_gemv_swiglu_stats, ctx.gemv_residual_stats))
        up(p["h"], p["Wgu"], p["hidden"], p["norm"], p["stats"], ffn, dim)
        down(p["hidden"], p["Wd"], p["h"], dim, ffn, p["stats2"])
        return [s["hidden"], s["h"], s["stats2"]]
    if kind == "attn":
        s["ctx"].attn_decode_rope(s["out"].data_ptr(), s["q"].data_ptr(), s["kc"].data_ptr(),
                                  s["vc"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), 0,
                                  case["pos"], case["nh"], case["nkv"], case["hd"], MAX_SEQ)
        return [s["out"], s["kc"], s["vc"]]
    if kind == "pfattn":
        s["ctx"].attn_prefill(s["out"].data_ptr(), s["qkv"].data_ptr(), s["kc"].data_ptr(),
                              s["vc"].data_ptr(), 0, case["p0"], case["T"], case["nh"],
                              case["nkv"], case["hd"], MAX_SEQ)
        return s["out"]
    if kind == "gemm":
        args = (s["X"].data_ptr(), case["T"], case["N"], case["K"])
        if case["prepared"]:
            s["ctx"].gemm_prepared(s["Y"].data_ptr(), s["W"].data_ptr(), s["Wp"].data_ptr(), *args)
        else:
            s["ctx"].gemm(s["Y"].data_ptr(), s["W"].data_ptr(), *args)
        return s["Y"]
    model = s["model"]
    m = model.m
    if kind == "generate":
        toks, _, _ = m.generate(model.tokens, case["n"], hashes=False)
        return {"tokens": np.array(toks, dtype=np.int64), "logits": m.read_logits()}
    if kind == "prefill":
        m.prefill(model.tokens, 0, case["vocab"], logits=False, choose=False)
        return m.read_logits()
    m.set_sampling(ONE * 8 // 10 if case["sampled"] else 0, 40, ONE * 9 // 10, model.seed)
    _, toks, _ = m.decode_graph(model.tokens[-1], case["T"], case["n"])
    return {"tokens": np.array(toks, dtype=np.int64), "logits": m.read_logits()}


# ---- what a pass cannot do without -------------------------------------------

def _model_work(case, rows, kv_rows, heads, wbytes):
    """rows: tokens that go through the layers, in one pass over the weights;
    kv_rows: sum over those tokens of the cache rows each attends to."""
    dim, kvd, ffn = case["dim"], case["nkv"] * case["hd"], case["ffn"]
    per_layer = (dim + 2 * kvd) * dim + dim * dim + 3 * ffn * dim
    lm = case["vocab"] * dim
    macs = case["layers"] * (rows * per_layer + 2 * kv_rows * dim) + heads * lm
    nbytes = wbytes * (case["layers"] * per_layer + lm) + 8 * heads * case["vocab"]
    return macs, nbytes


def work(case):
    """flops: two for each Q16.48 multiply-add (a 64 x 64 -> 128-bit product
    and its exact sum), however the kernels make it."""
    kind = case["kind"]
    if kind == "gemv":
        M, K = case["M"], case["K"]
        return {"bytes": 8 * (M * K + K + M), "flops": 2 * M * K}
    if kind == "mlp":
        dim, ffn = case["dim"], case["ffn"]
        return {"bytes": (2 if case["bf16"] else 8) * 3 * dim * ffn + 8 * (3 * dim + ffn),
                "flops": 6 * dim * ffn}
    if kind in ("attn", "pfattn"):
        nh, nkv, hd = case["nh"], case["nkv"], case["hd"]
        if kind == "attn":
            S = case["pos"] + 1
            return {"bytes": 16 * S * nkv * hd + 16 * (nh + nkv) * hd, "flops": 4 * S * nh * hd}
        T, p0 = case["T"], case["p0"]
        pairs = T * p0 + T * (T + 1) // 2
        return {"bytes": 16 * (p0 + T) * nkv * hd + 16 * T * nh * hd, "flops": 4 * pairs * nh * hd}
    if kind == "gemm":
        T, N, K = case["T"], case["N"], case["K"]
        return {"bytes": 8 * (T * K + N * K + T * N), "flops": 2 * T * N * K}
    T, n, kvd = case["T"], case.get("n", 0), case["nkv"] * case["hd"]
    wbytes = 2 if case.get("bf16") else 8
    macs = nbytes = 0
    if kind in ("generate", "prefill"):     # the prompt: one pass over the weights
        macs, nbytes = _model_work(case, T, T * (T + 1) // 2, 1, wbytes)
        nbytes += 16 * case["layers"] * T * kvd
    steps = n - 1 if kind == "generate" else n
    for i in range(steps):                  # each decoded token: all weights and its cache rows
        a, b = _model_work(case, 1, T + i + 1, 1, wbytes)
        macs += a
        nbytes += b + 16 * case["layers"] * (T + i + 1) * kvd
    return {"bytes": nbytes, "flops": 2 * macs}


def tolerance(case):
    """Fixed-point integers: any correct implementation gives the same words."""
    return "exact"


# ---- the products in 64 bits -------------------------------------------------

def _limbs(v):
    """An int64 tensor as four 16-bit limbs in float64, the top one signed."""
    return [((v >> (16 * i)) & 0xFFFF).double() for i in range(3)] + [(v >> 48).double()]


def _exact_product(X, W):
    """(sum_k X[t][k] W[n][k]) >> 48 mod 2^64: limb products in float64 (every
    sum below 2^53, so exact), carried up in int64."""
    xs, ws = _limbs(X), [w.t().contiguous() for w in _limbs(W)]
    out, acc = torch.zeros(X.shape[0], W.shape[0], dtype=torch.int64, device=DEV), 0
    for d in range(7):
        q = sum(torch.mm(xs[a], ws[d - a]).to(torch.int64)
                for a in range(4) if 0 <= d - a <= 3)
        acc = q + acc
        if d >= 3:
            out += (acc & 0xFFFF) << (16 * (d - 3))
        acc = acc >> 16
    return out


def exact(case, seed):
    """The plain products; the other kinds go through fixed-point exponentials
    and divisions whose truncations plain 64-bit arithmetic does not have."""
    if case["kind"] not in ("gemv", "gemm"):
        return None
    g = _gen(seed)
    if case["kind"] == "gemv":
        M, K = case["M"], case["K"]
        W, x = _weights(g, M * K), _acts(g, K)
        return _exact_product(x.view(1, K), W.view(M, K)).view(M)
    T, N, K = case["T"], case["N"], case["K"]
    W, X = _weights(g, N * K), _acts(g, T * K)
    return _exact_product(X.view(T, K), W.view(N, K))
