"""The forward's key split on 32-key tiles (head_dim 128 and 256): pairs of
wavefronts take alternate tiles of a 32-row group and merge through LDS."""
import math

import pytest
import torch

from oracle import attention_oracle as orc
from trinix_amd.kernels import TritonAttentionKernel
from trinix_amd.kernels.attention_kernel import attention
from trinix_amd.kernels.qk_norm_kernel import qk_rmsnorm

pytestmark = pytest.mark.gpu

DEV = "cuda"
CFG = {128: "4,2,32,2", 256: "4,1,32,2"}

CASES = [
    # (B, Sq, Sk, H, Hkv, causal, window, alibi): one key (an empty odd half), 32 | 33 | 65 keys, partial row groups,
    # rows without keys on one side, Sq != Sk both ways
    (1, 1, 1, 2, 1, True, None, False),
    (1, 33, 32, 2, 2, False, None, False),
    (2, 64, 33, 2, 1, False, None, True),
    (1, 65, 65, 4, 2, True, None, False),
    (1, 200, 130, 2, 2, True, None, True),
    (2, 97, 300, 4, 1, False, (70, 20), False),
    (1, 300, 300, 2, 2, True, (40, 0), False),
]


def _rand(shape, dtype, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(DEV, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [128, 256])
@pytest.mark.parametrize("case", CASES, ids=[str(c) for c in CASES])
def test_split_matches_the_closed_form(case, D, dtype, monkeypatch):
    """The kernel rounds P to 16 bits and sums the rounded P (relative error u
    of every p: u sum p|v| in O, u in the row sum, so u in lse), then rounds
    the output (u again); fp32 sums, exp2 and the score's rounding get a tenth
    of that."""
    B, Sq, Sk, H, Hkv, causal, window, alibi = case
    q, k, v = _rand((B, Sq, H, D), dtype, 1), _rand((B, Sk, Hkv, D), dtype, 2), _rand((B, Sk, Hkv, D), dtype, 3)
    slopes = orc.alibi_slopes(H).to(DEV, torch.float32) if alibi else None
    monkeypatch.setenv("TRINIX_ATTN_CFG", CFG[D])
    monkeypatch.setattr("trinix_amd.kernels.attention_kernel.SPLITKV_ENABLED", False)
    out, lse = TritonAttentionKernel.apply(q, k, v, causal=causal, window_size=window, alibi_slopes=slopes,
                                           return_lse=True)
    q, k, v, out, lse = (t.cpu().double() for t in (q, k, v, out, lse))
    k, v = (t.repeat_interleave(H // Hkv, 2) for t in (k, v))
    s = torch.einsum("bihd,bjhd->bhij", q, k) / math.sqrt(D)
    i, j = torch.arange(Sq)[:, None], torch.arange(Sk)[None]
    if alibi:
        s = s - slopes.cpu().double()[None, :, None, None] * (i - j).abs()
    ok = torch.ones(Sq, Sk, dtype=torch.bool)
    if causal:
        ok &= j <= i
    if window is not None:
        ok &= (j >= i - window[0]) & (j <= i + window[1])
    s = s.masked_fill(~ok, -math.inf)
    live = ok.any(1)
    p = s.softmax(-1)
    ref = torch.einsum("bhij,bjhd->bihd", p, v)
    mass = torch.einsum("bhij,bjhd->bihd", p, v.abs())
    u = torch.finfo(dtype).eps / 2  # 8 and 11 significant bits
    assert torch.isnan(out[:, ~live]).all()
    assert ((out - ref)[:, live].abs() <= 1.1 * u * (mass + 2 * ref.abs())[:, live] + 1e-7).all()
    assert ((lse - s.logsumexp(-1))[..., live].abs() <= 1.1 * u).all()


@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (256, torch.float16)])
def test_split_with_the_fused_q_norm(D, dtype, monkeypatch):
    """The norm in the prologue, and the normalised q it leaves for the
    backward: bit for bit the two-kernel path on the same tiles."""
    monkeypatch.setenv("TRINIX_ATTN_CFG", CFG[D])
    B, S, H, HKV, eps = 2, 170, 4, 2, 1e-5
    q0, k0, v0 = _rand((B, S, H, D), dtype, 4) * 2, _rand((B, S, HKV, D), dtype, 5), _rand((B, S, HKV, D), dtype, 6)
    w0, do = _rand((D,), dtype, 7) * 0.2 + 1, _rand((B, S, H, D), dtype, 8)
    res = []
    for fused in (True, False):
        q, k, v, w = (t.clone().requires_grad_(True) for t in (q0, k0, v0, w0))
        if fused:
            out = attention(q, k, v, causal=True, q_norm_weight=w, q_norm_eps=eps)
        else:
            out = attention(qk_rmsnorm(q, w, eps), k, v, causal=True)
        out.backward(do)
        res.append([out.detach()] + [t.grad for t in (q, k, v, w)])
    for name, a, b in zip(("out", "dq", "dk", "dv", "dweight"), *res):
        assert torch.equal(a, b), name
