"""GPU tests of the kernels whose P and dZ enter their products with more bits
than a 16-bit operand has: the fp32 forward and backward (24 bits), and the
16-bit backward at head_dim 256 (two 16-bit terms: 16 bits in bf16, about 21 in
fp16) (``csrc/attn_fwd_f32.hip``, ``csrc/attn_bwd_generic.h``), at the edges of
their 32-row tiles and 64/128-row blocks, with one and with two wavefronts per
32 keys or rows.

Bars against float64 autograd of the oracle.  Elementwise the repository's
(twice the eager error of the dtype plus 2e-3, or for fp32 1e-5, of the
scale).  In the 2-norm, 16-bit: the inputs' products are exact and P and dZ
carry 16 or more bits, so what is left is the rounding of each gradient and of
the saved output (through delta), uniform within u of an element: u / sqrt(3)
of the norm each, 0.82 u together; the bar is u (P and dZ rounded to 16 bits
show 1.2 u)."""
import pytest
import torch

from oracle import attention_oracle as orc
from trinix_amd import triton_attn_func

pytestmark = pytest.mark.gpu
DEV = "cuda"
UNIT = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}

SHAPES = [(31, 33), (64, 65), (97, 200), (129, 127), (1, 300), (260, 5)]
KINDS = [(torch.float32, 64), (torch.float32, 128), (torch.float32, 256), (torch.bfloat16, 256), (torch.float16, 256)]


def _data(B, Sq, Sk, H, Hkv, D, dtype, seed, do_scale=1.0):
    g = torch.Generator().manual_seed(seed)
    ts = [torch.randn(s, generator=g).to(dtype) for s in ((B, Sq, H, D), (B, Sk, Hkv, D), (B, Sk, Hkv, D))]
    return ts, (torch.randn(B, Sq, H, D, generator=g) * do_scale).to(dtype)


def _grads(fn, ts, do, **kw):
    leaves = [t.detach().clone(memory_format=torch.preserve_format).requires_grad_(True) for t in ts]
    out = fn(*leaves, **kw)
    return [out.detach(), *torch.autograd.grad(out, leaves, do)]


def _compare(hip, ts, do, dtype, **kw):
    truth = _grads(orc.functional_attention, [t.double() for t in ts], do.double(), **kw)
    eager = _grads(orc.functional_attention, ts, do, **kw)
    for name, h, e, t in zip(("out", "dq", "dk", "dv"), hip, eager, truth):
        h, e = h.cpu().double(), e.double()
        scale, err_h, err_e = t.abs().max().item(), (h - t).abs().max().item(), (e - t).abs().max().item()
        assert err_h <= 2 * err_e + (1e-5 if dtype == torch.float32 else 2e-3) * scale, (name, err_h, err_e, scale)
        if dtype in UNIT and name != "out":
            assert (h - t).norm() <= UNIT[dtype] * t.norm(), (name, (h - t).norm() / t.norm())


@pytest.mark.parametrize("ks", ["1", "2"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("dtype,D", KINDS, ids=lambda v: str(v))
def test_tile_edges(monkeypatch, dtype, D, shape, ks):
    Sq, Sk = shape
    print(f"generic tile edges {dtype} {D} {shape} ks {ks}", flush=True)
    monkeypatch.setenv("TRINIX_BWD_GENERIC", f"{ks},{ks}")
    monkeypatch.setenv("TRINIX_F32_KS", ks)
    for n, kw in enumerate((dict(), dict(causal=True), dict(window_size=(40, 17), alibi_slopes=orc.alibi_slopes(2)))):
        if kw.get("window_size") and Sk < Sq:
            continue  # rows past Sk + 40 would see no key
        if kw.get("causal") and Sq == 1:
            continue  # a single key: dq and dk are exactly zero, what is computed is rounding alone
        ts, do = _data(2, Sq, Sk, 2, 1, D, dtype, 31 * Sq + Sk + n)
        gkw = {k: v.to(DEV) if torch.is_tensor(v) else v for k, v in kw.items()}
        _compare(_grads(triton_attn_func, [t.to(DEV) for t in ts], do.to(DEV), **gkw), ts, do, dtype, **kw)


@pytest.mark.parametrize("D", [64, 128, 256])
def test_fp32_rows_without_16_byte_alignment(D):
    """fp32 operands sliced out of wider rows (4-byte aligned) are read in
    place, element by element: bitwise the contiguous operands' results."""
    B, S, H = 1, 75, 2
    ts, do = _data(B, S, S, H, H, D, torch.float32, D)
    wide = [torch.zeros(B, S, H, D + 3, device=DEV) for _ in ts]
    views = []
    for w, t in zip(wide, ts):
        w[..., 1:D + 1] = t.to(DEV)
        views.append(w[..., 1:D + 1])
    want = _grads(triton_attn_func, [t.to(DEV) for t in ts], do.to(DEV), causal=True)
    leaves = [v.requires_grad_(True) for v in views]
    out = triton_attn_func(*leaves, causal=True)
    got = [out.detach(), *torch.autograd.grad(out, leaves, do.to(DEV))]
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("exponent", [-12, -6, 8])
def test_fp16_head_dim_256_gradient_range(exponent):
    """fp16 dZ is held at a power of two of its own, so gradients keep their
    relative accuracy for output gradients far from 1 (here rows that differ
    by 2^8 among themselves, the large ones last: the factor is lowered on the
    way).  Gradients stay in fp16's normal range at these scales, except the
    smallest one's, whose quantum of 2^-24 is allowed for."""
    B, S, H, D = 1, 160, 2, 256
    ts, do = _data(B, S, S, H, H, D, torch.float16, 9)
    rows = torch.where(torch.arange(S) < S // 2, 2.0 ** -8, 1.0)[None, :, None, None]
    do = (do.float() * rows * 2.0 ** exponent).half()
    hip = _grads(triton_attn_func, [t.to(DEV) for t in ts], do.to(DEV), causal=True)
    truth = _grads(orc.functional_attention, [t.double() for t in ts], do.double(), causal=True)
    for name, h, t in list(zip(("out", "dq", "dk", "dv"), hip, truth))[1:]:
        err = (h.cpu().double() - t).norm()
        assert err <= UNIT[torch.float16] * t.norm() + 2.0 ** -24 * t.numel() ** 0.5, (name, (err / t.norm()).item())
