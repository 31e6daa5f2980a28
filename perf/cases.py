"""The attention work that programs built on this framework do, as measured cases.

A case is a dict of plain values.  ``listed()`` names the fixed ones,
``draw(rng)`` makes one more of the same ranges; ``prepare`` builds what a
program holds before the call, ``run`` is one pass through the public entry
points (``triton_attn_func`` or an attention layer), ``exact`` the same pass in
plain 64-bit torch, ``work`` the bytes and operations the pass cannot do
without, and ``tolerance`` the error another correct implementation may show.
"""
import math

import torch

from trinix_amd import FastGroupedQueryAttention, triton_attn_func

DEV = "cuda"
DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}

# Largest relative error (2-norm) of any output against 64 bits that one pass
# showed over these ranges, times about four: attention 8.1e-7 (fp32), 6.4e-4
# (fp16) and 5.0e-3 (bf16), the gradients of q and k; the layer 1.1e-3 (fp16)
# and 9.6e-3 (bf16), the projections' gradients.
_TOL_ATTN = {"fp32": 3.3e-6, "fp16": 2.6e-3, "bf16": 2e-2}
_TOL_LAYER = {"bf16": 3e-2, "fp16": 4.5e-3}


def _attn(name, B, Sq, Sk, H, Hkv, D, dtype, causal=True, window=0, rope=0.0, alibi=False, mask=False, dropout=0.0,
          grad=False):
    """One ``triton_attn_func`` call, with its backward when ``grad``."""
    c = dict(kind="attn", B=B, Sq=Sq, Sk=Sk, H=H, Hkv=Hkv, D=D, dtype=dtype, causal=causal, window=window, rope=rope,
             alibi=alibi, mask=mask, dropout=dropout, grad=grad)
    return dict(name=name, **c) if name else c


def _layer(name, B, S, H, Hkv, D, dtype, norm, rope, grad):
    """One ``FastGroupedQueryAttention`` call with qk-norm and RoPE, with its backward when ``grad``."""
    c = dict(kind="layer", B=B, Sq=S, Sk=S, H=H, Hkv=Hkv, D=D, E=H * D, dtype=dtype, norm=norm, rope=rope, grad=grad,
             causal=True, window=0)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one sequence being generated: a token against a short cache, where launches and latency count
        _attn("decode_b1_s2048", 1, 1, 2048, 32, 8, 128, "bf16", causal=False),
        # a serving batch's decode step against long caches (8B-parameter GQA shape)
        _attn("decode_b16_s8192", 16, 1, 8192, 32, 8, 128, "bf16", causal=False),
        # GPT-2-small evaluation
        _attn("gpt2_forward", 4, 1024, 1024, 12, 12, 64, "bf16"),
        # GPT-2-small training, with the attention dropout it is trained with
        _attn("gpt2_train_dropout", 4, 1024, 1024, 12, 12, 64, "bf16", dropout=0.1, grad=True),
        # prompt of a Llama-3-8B-shaped model, RoPE fused
        _attn("llama_prefill_s8192", 1, 8192, 8192, 32, 8, 128, "bf16", rope=500000.0),
        # the same model's attention in training
        _attn("llama_train_s8192", 1, 8192, 8192, 32, 8, 128, "bf16", rope=500000.0, grad=True),
        # long prompts through sliding-window attention (Mistral shape)
        _attn("window_prefill_s16384", 2, 16384, 16384, 32, 8, 128, "bf16", window=4096, rope=10000.0),
        # ALiBi with an additive block mask, fp16 (packed or sparse batches)
        _attn("alibi_mask_fp16", 8, 2048, 2048, 16, 16, 64, "fp16", causal=False, alibi=True, mask=True),
        # training in torch's default dtype, as a first run of any model has it
        _attn("fp32_train_s1024", 4, 1024, 1024, 12, 12, 64, "fp32", grad=True),
        # training of a model with wide heads (head_dim 256, grouped queries)
        _attn("head256_train_s2048", 2, 2048, 2048, 8, 4, 256, "bf16", grad=True),
        # cross attention in training: unequal odd lengths, a head_dim that is no power of two
        _attn("cross_train_d80", 3, 777, 1111, 10, 10, 80, "fp16", causal=False, grad=True),
        # a whole attention layer in training: projections, RoPE, qk-norm, grouped queries
        _layer("gqa_layer_train_s2048", 2, 2048, 16, 4, 128, "bf16", "rmsnorm", 500000.0, True),
    ]


def draw(rng):
    def size(lo, hi):  # spread over the logarithm; odd sizes as likely as even ones
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    half = rng.choice(["bf16", "bf16", "fp16"])
    pick = rng.randrange(11)
    if pick == 0:  # decode, one to sixteen sequences
        H, Hkv = rng.choice([(32, 8), (16, 16), (16, 4), (16, 1)])
        return _attn(None, size(1, 16), rng.choice([1, 1, 1, 4]), size(300, 8192), H, Hkv, rng.choice([64, 128]), half,
                     causal=False)
    if pick == 1:  # evaluation of a small model
        return _attn(None, *_square(size(1, 4), size(128, 1024)), *_mha(rng.choice([8, 12])), 64, half)
    if pick == 2:  # its training, with dropout
        return _attn(None, *_square(size(1, 4), size(128, 1024)), *_mha(rng.choice([8, 12])), 64, half,
                     dropout=rng.choice([0.1, 0.2]), grad=True)
    if pick == 3:  # prompts of a model with grouped queries
        H, Hkv = rng.choice([(32, 8), (16, 4), (16, 16)])
        return _attn(None, *_square(1, size(700, 8192)), H, Hkv, 128, half, rope=500000.0)
    if pick == 4:  # its training
        H, Hkv = rng.choice([(32, 8), (16, 4), (16, 16)])
        return _attn(None, *_square(1, size(700, 8192)), H, Hkv, 128, half, rope=500000.0, grad=True)
    if pick == 5:  # sliding windows
        return _attn(None, *_square(rng.choice([1, 2]), size(2048, 16384)), 32, 8, 128, half, window=size(500, 4096),
                     rope=10000.0)
    if pick == 6:  # ALiBi and a mask, grouped down to a single KV head
        return _attn(None, *_square(size(1, 8), size(200, 2048)), 16, rng.choice([16, 1]), 64, half, causal=False,
                     alibi=True, mask=True)
    if pick == 7:  # fp32, forward or training
        D = rng.choice([64, 64, 128])
        return _attn(None, *_square(size(1, 4), size(100, 1024 if D == 64 else 700)), *_mha(rng.choice([4, 8, 12])), D,
                     "fp32", causal=rng.random() < 0.7, grad=rng.random() < 0.7)
    if pick == 8:  # wide heads, forward or training
        H, Hkv = rng.choice([(8, 4), (8, 8), (8, 1)])
        return _attn(None, *_square(size(1, 2), size(200, 2048)), H, Hkv, 256, half, grad=rng.random() < 0.7)
    if pick == 9:  # cross attention, ragged lengths and head_dims
        return _attn(None, size(1, 4), size(60, 1200), size(60, 1500), *_mha(rng.choice([8, 10])),
                     rng.choice([40, 72, 80, 96, 112]), half, causal=False, grad=rng.random() < 0.7)
    # layers, forward or training; layernorm forward only: its bias on k shifts a row's scores alike, so that its
    # gradient is zero and what is computed for it is rounding alone
    H, Hkv = rng.choice([(16, 4), (8, 8), (8, 2)])
    grad = rng.random() < 0.6
    return _layer(None, size(1, 2), size(200, 2048), H, Hkv, 128, half,
                  "rmsnorm" if grad else rng.choice(["rmsnorm", "layernorm"]), 500000.0, grad)


def _square(B, S):
    return B, S, S


def _mha(H):
    return H, H


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _rope_tables(S, D, base, dtype):
    inv = 1.0 / base ** (torch.arange(0, D, 2, device=DEV).float() / D)
    f = torch.outer(torch.arange(S, device=DEV).float(), inv)
    e = torch.cat((f, f), dim=-1)
    return e.cos().to(dtype), e.sin().to(dtype)


def _alibi_slopes(H):
    n = 2 ** math.floor(math.log2(H))
    s = [2.0 ** (-8.0 * (i + 1) / n) for i in range(n)] + [2.0 ** (-4.0 * (2 * i + 1) / n) for i in range(H - n)]
    return torch.tensor(s, dtype=torch.float32, device=DEV)


def _block_mask(Sq, Sk, g):
    """0, and -inf on about a tenth of the 64 x 64 blocks; key block 0 stays open."""
    grid = torch.rand((-(-Sq // 64), -(-Sk // 64)), generator=g, device=DEV) < 0.1
    grid[:, 0] = False
    full = grid.repeat_interleave(64, 0).repeat_interleave(64, 1)[:Sq, :Sk]
    return torch.zeros((Sq, Sk), device=DEV).masked_fill_(full, float("-inf"))


def prepare(case, seed):
    c, dt = case, DTYPES[case["dtype"]]
    g = torch.Generator(device=DEV).manual_seed(seed)

    def randn(*shape):
        return torch.randn(shape, generator=g, device=DEV).to(dt)

    if c["kind"] == "layer":
        before = torch.get_default_dtype()
        torch.set_default_dtype(dt)  # 16-bit parameters; the RoPE frequencies stay fp32
        try:
            with torch.device(DEV):
                layer = FastGroupedQueryAttention(c["E"], c["H"], c["Hkv"], bias=False, causal=True, head_dim=c["D"],
                                                  position_method="rope", rope_base=c["rope"], max_seq_len=c["Sq"],
                                                  qk_norm=True, qk_norm_type=c["norm"])
        finally:
            torch.set_default_dtype(before)
        with torch.no_grad():
            for name, p in layer.named_parameters():
                if p.dim() == 2:
                    p.normal_(0.0, c["E"] ** -0.5, generator=g)
                elif name.endswith("weight"):
                    p.normal_(1.0, 0.1, generator=g)
                else:
                    p.normal_(0.0, 0.1, generator=g)
        layer.train(c["grad"])
        x = randn(c["B"], c["Sq"], c["E"]).requires_grad_(c["grad"])
        return dict(case=c, layer=layer, x=x, dout=randn(c["B"], c["Sq"], c["E"]) if c["grad"] else None)
    q = randn(c["B"], c["Sq"], c["H"], c["D"]).requires_grad_(c["grad"])
    k = randn(c["B"], c["Sk"], c["Hkv"], c["D"]).requires_grad_(c["grad"])
    v = randn(c["B"], c["Sk"], c["Hkv"], c["D"]).requires_grad_(c["grad"])
    kw = dict(causal=c["causal"])
    if c["window"]:
        kw["window_size"] = (c["window"], 0)
    if c["rope"]:
        kw["rotary_cos"], kw["rotary_sin"] = _rope_tables(max(c["Sq"], c["Sk"]), c["D"], c["rope"], dt)
    if c["alibi"]:
        kw["alibi_slopes"] = _alibi_slopes(c["H"])
    if c["mask"]:
        kw["attn_mask"] = _block_mask(c["Sq"], c["Sk"], g)
    if c["dropout"]:
        kw["dropout_p"] = c["dropout"]
    return dict(case=c, q=q, k=k, v=v, kw=kw, seed=seed, dout=randn(*q.shape) if c["grad"] else None)


def run(state):
    c = state["case"]
    if c["kind"] == "layer":
        layer, x = state["layer"], state["x"]
        if not c["grad"]:
            with torch.no_grad():
                return layer(x)[0]
        out = layer(x)[0]
        return [out, *torch.autograd.grad(out, [x, *layer.parameters()], state["dout"])]
    q, k, v = state["q"], state["k"], state["v"]
    if c["dropout"]:
        torch.default_generator.manual_seed(state["seed"])  # a step that can be repeated, as a resumed run needs it
    out = triton_attn_func(q, k, v, **state["kw"])
    if not c["grad"]:
        return out
    return [out, *torch.autograd.grad(out, [q, k, v], state["dout"])]


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how exact it is
# ---------------------------------------------------------------------------
def _pairs(c):
    """Allowed (query, key) pairs of one head."""
    Sq, Sk = c["Sq"], c["Sk"]
    if not c["causal"]:
        n = Sq * Sk
    else:
        w = c["window"] or Sq
        m = min(Sq, w + 1)  # rows that see every key up to their own
        n = m * (m + 1) // 2 + (Sq - m) * (w + 1)
    return n * 0.9 if c.get("mask") else n


def work(case):
    c = case
    esz = 4 if c["dtype"] == "fp32" else 2
    qn, kn = c["B"] * c["Sq"] * c["H"] * c["D"], c["B"] * c["Sk"] * c["Hkv"] * c["D"]
    flops = 4.0 * c["D"] * c["B"] * c["H"] * _pairs(c)
    flops *= 3.5 if c["grad"] else 1.0
    if c["kind"] == "layer":
        wn = c["E"] * c["D"] * (2 * c["H"] + 2 * c["Hkv"])
        xn = c["B"] * c["Sq"] * c["E"]
        flops += 2.0 * c["B"] * c["Sq"] * wn * (3 if c["grad"] else 1)
        return {"bytes": float(esz * ((2 * wn + 4 * xn) if c["grad"] else (wn + 2 * xn))), "flops": flops}
    n = 2 * qn + 2 * kn
    if c["grad"]:
        n += 2 * qn + 2 * kn  # dout read; dq, dk and dv written
    return {"bytes": float(esz * n + (4 * c["Sq"] * c["Sk"] if c["mask"] else 0)), "flops": flops}


def tolerance(case):
    if case["kind"] == "layer":
        return {"rel": _TOL_LAYER[case["dtype"]]}
    return {"rel": _TOL_ATTN[case["dtype"]]}


def _rotate64(x, cos, sin):
    """RoPE of (B, S, H, D) in 64 bits."""
    c, s = (t.double()[: x.shape[1], None, :] for t in (cos, sin))
    x1, x2 = x.chunk(2, dim=-1)
    return x * c + torch.cat((-x2, x1), dim=-1) * s


def _attend64(q, k, v, causal, window, slopes, mask):
    """Attention of (B, S, H, D) in 64 bits, head by head and in bands of rows, with gradients where asked for."""
    B, Sq, H, D = q.shape
    Sk, G = k.shape[1], H // k.shape[2]
    rows = max(64, min(Sq, (1 << 26) // Sk))
    out = []
    for b in range(B):
        heads = []
        for h in range(H):
            bands = []
            for i0 in range(0, Sq, rows):
                i1 = min(Sq, i0 + rows)
                j0 = max(0, i0 - window) if window else 0
                j1 = min(Sk, i1) if causal else Sk
                d = torch.arange(j0, j1, device=DEV)[None, :] - torch.arange(i0, i1, device=DEV)[:, None]
                z = q[b, i0:i1, h] @ k[b, j0:j1, h // G].t().contiguous() * D ** -0.5
                if slopes is not None:
                    z = z - slopes[h].double() * d.abs()
                if mask is not None:
                    z = z + mask[i0:i1, j0:j1].double()
                if causal:
                    z = z.masked_fill(d > 0, float("-inf"))
                if window:
                    z = z.masked_fill(d < -window, float("-inf"))
                bands.append(torch.softmax(z, dim=-1) @ v[b, j0:j1, h // G])
            heads.append(torch.cat(bands))
        out.append(torch.stack(heads, dim=1))
    return torch.stack(out)


def exact(case, seed):
    c = case
    if c.get("dropout"):
        return None  # which weights are dropped is the library's own choice
    s = prepare(case, seed)
    if c["kind"] == "layer":
        layer, eps = s["layer"], s["layer"].q_norm.eps
        P = {n: p.detach().double().requires_grad_(c["grad"]) for n, p in layer.named_parameters()}
        x = s["x"].detach().double().requires_grad_(c["grad"])
        cos, sin = _rope_tables(c["Sq"], c["D"], c["rope"], DTYPES[c["dtype"]])

        def proj(t, name):
            return torch.nn.functional.linear(t, P[name + ".weight"])

        def norm(t, name):
            if c["norm"] == "layernorm":
                return torch.nn.functional.layer_norm(t, (c["D"],), P[name + ".weight"], P[name + ".bias"], eps)
            return t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + eps) * P[name + ".weight"]

        def split(t, heads):
            return t.view(c["B"], c["Sq"], heads, c["D"])

        q = norm(_rotate64(split(proj(x, "q_proj"), c["H"]), cos, sin), "q_norm")
        k = norm(_rotate64(split(proj(x, "k_proj"), c["Hkv"]), cos, sin), "k_norm")
        a = _attend64(q, k, split(proj(x, "v_proj"), c["Hkv"]), True, 0, None, None)
        out = proj(a.reshape(c["B"], c["Sq"], -1), "o_proj")
        if not c["grad"]:
            return out
        return [out.detach(), *torch.autograd.grad(out, [x, *P.values()], s["dout"].double())]
    q, k, v = (s[n].detach().double() for n in ("q", "k", "v"))
    kw = s["kw"]
    args = (c["causal"], c["window"], kw.get("alibi_slopes"), kw.get("attn_mask"))

    def attend(q, k, v):
        if c["rope"]:
            q, k = (_rotate64(t, kw["rotary_cos"], kw["rotary_sin"]) for t in (q, k))
        return q, k, v

    if not c["grad"]:
        return _attend64(*attend(q, k, v), *args)
    # one KV head at a time: the graph of one group's rows is all that is held
    G = c["H"] // c["Hkv"]
    out, grads = torch.empty_like(q), [torch.empty_like(t) for t in (q, k, v)]
    for b in range(c["B"]):
        for j in range(c["Hkv"]):
            at = (slice(b, b + 1), slice(None))
            own = [t[at + (w,)].clone().requires_grad_() for t, w in ((q, slice(j * G, j * G + G)),
                                                                      (k, slice(j, j + 1)), (v, slice(j, j + 1)))]
            sub = (c["causal"], c["window"], args[2][j * G:j * G + G] if args[2] is not None else None, args[3])
            o = _attend64(*attend(*own), *sub)
            got = torch.autograd.grad(o, own, s["dout"][at + (slice(j * G, j * G + G),)].double())
            out[at + (slice(j * G, j * G + G),)] = o.detach()
            for t, gr, w in zip(grads, got, (slice(j * G, j * G + G), slice(j, j + 1), slice(j, j + 1))):
                t[at + (w,)] = gr
    return [out, *grads]
