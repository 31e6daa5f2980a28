"""GPU tests of head dims between the kernels': q, k and v zero-padded by one
``trinix_pad_heads`` launch, the other tensors at their own width
(``trinix_attn_fwd_narrow`` / ``trinix_attn_bwd_narrow``) where the head_dim is a
multiple of 8 of at most 128, sliced from padded ones elsewhere.  Gradients
within the repository's bar: twice the eager error against float64 plus 2e-3
of the scale."""
import pytest
import torch

from oracle import attention_oracle as orc
from trinix_amd import triton_attn_func

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _tensors(B, Sq, Sk, H, Hkv, D, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(s, generator=g).to(dtype)
            for s in ((B, Sq, H, D), (B, Sk, Hkv, D), (B, Sk, Hkv, D), (B, Sq, H, D))]


def _run(fn, ts, do, **kw):
    out = fn(*ts, **kw)
    return [out.detach(), *torch.autograd.grad(out, ts, do)]


def _check(got, ts, dtype, **kw):
    def ref(dt):
        leaves = [t.to(dt).requires_grad_(True) for t in ts[:3]]
        return _run(orc.functional_attention, leaves, ts[3].to(dt), **kw)

    for name, h, e, t in zip(("out", "dq", "dk", "dv"), got, ref(dtype), ref(torch.float64)):
        h, e, t = h.cpu().double(), e.double(), t.double()
        scale = t.abs().max().item()
        err_h, err_e = (h - t).abs().max().item(), (e - t).abs().max().item()
        assert h.shape == t.shape and err_h <= 2 * err_e + 2e-3 * scale, (name, err_h, err_e, scale)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [8, 36, 40, 63, 72, 80, 96, 100, 112, 120, 160])
def test_padded_head_dims(D, dtype):
    for n, kw in enumerate((dict(), dict(causal=True), dict(alibi_slopes=orc.alibi_slopes(4), window_size=(50, 30)))):
        ts = _tensors(2, 70, 70 + 35 * (n == 0), 4, 2, D, dtype, D + n)
        print(f"padded heads D {D} {dtype} {n}", flush=True)
        gkw = {k: v.to(DEV) if torch.is_tensor(v) else v for k, v in kw.items()}

        def step():
            return _run(triton_attn_func, [t.to(DEV).requires_grad_(True) for t in ts[:3]], ts[3].to(DEV), **gkw)

        first, again = step(), step()  # the second from the layout's launch templates
        for a, b in zip(first, again):
            assert torch.equal(a, b)
        _check(first, ts, dtype, **kw)
        with torch.no_grad():
            gpu = [t.to(DEV) for t in ts[:3]]
            for _ in range(2):
                assert torch.equal(triton_attn_func(*gpu, **gkw), first[0])


@pytest.mark.parametrize("D", [72, 80, 100])
def test_padded_heads_from_other_layouts(D):
    """Transposed (B, H, S, D) operands, slices of one projection with odd
    starts, and a gradient that is not contiguous: the contiguous results."""
    B, S, H, dtype = 2, 60, 3, torch.bfloat16
    ts = [t.to(DEV) for t in _tensors(B, S, S, H, H, D, dtype, 5)]
    want = _run(triton_attn_func, [t.clone().requires_grad_(True) for t in ts[:3]], ts[3], causal=True)
    trans = [t.transpose(1, 2).contiguous().transpose(1, 2).requires_grad_(True) for t in ts[:3]]
    do = ts[3].transpose(1, 2).contiguous().transpose(1, 2)
    packed = torch.zeros(B, S, H, 3 * D + 5, dtype=dtype, device=DEV)
    for n in range(3):
        packed[..., 1 + n * D:1 + (n + 1) * D] = ts[n]
    slices = [packed[..., 1 + n * D:1 + (n + 1) * D].requires_grad_(True) for n in range(3)]
    for got in (_run(triton_attn_func, trans, do, causal=True), _run(triton_attn_func, slices, do, causal=True)):
        for a, b in zip(got, want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("keep_map", ["0", "1"])
def test_padded_heads_with_dropout_and_mask(monkeypatch, keep_map):
    """Dropout and a mask run the same narrow path: bitwise the result of the
    operands padded by hand (the zero columns change no sum)."""
    B, S, H, D, dtype = 2, 90, 2, 80, torch.float16
    monkeypatch.setenv("TRINIX_DROPOUT_KEEP_MAP", keep_map)
    ts = [t.to(DEV) for t in _tensors(B, S, S, H, H, D, dtype, 6)]
    m = torch.where(torch.rand(S, S, generator=torch.Generator().manual_seed(1)) < 0.2, float("-inf"), 0.0)
    m[:, 0] = 0
    kw = dict(attn_mask=m.to(DEV), dropout_p=0.25, softmax_scale=D ** -0.5)
    torch.manual_seed(3)
    got = _run(triton_attn_func, [t.clone().requires_grad_(True) for t in ts[:3]], ts[3], **kw)
    pad = [torch.nn.functional.pad(t, (0, 128 - D)) for t in ts]
    torch.manual_seed(3)
    want = _run(triton_attn_func, [t.requires_grad_(True) for t in pad[:3]], pad[3], **kw)
    for a, b in zip(got, want):
        assert torch.equal(a, b[..., :D])


@pytest.mark.parametrize("D", [80, 100])
def test_padded_heads_output_written_before_the_backward(D):
    """The backward reads its own copy of the output: scaling the returned one
    in place scales the gradients alone (by a power of two, bitwise)."""
    ts = [t.to(DEV) for t in _tensors(2, 70, 90, 3, 3, D, torch.float16, 8)]
    leaves = [t.requires_grad_(True) for t in ts[:3]]
    for _ in range(2):  # the second from the layout's launch templates
        want = torch.autograd.grad(triton_attn_func(*leaves), leaves, ts[3])
        got = torch.autograd.grad(triton_attn_func(*leaves).mul_(0.5), leaves, ts[3] * 2)
        for a, b in zip(got, want):
            assert torch.equal(a, b)


def test_empty_operands_take_the_general_path():
    """No head_dim columns: an empty output (and empty gradients) where the
    caller gives the scale; no rows or keys: the forward's own error."""
    q, k = torch.empty(2, 5, 3, 0, dtype=torch.bfloat16, device=DEV), torch.empty(2, 7, 3, 0, dtype=torch.bfloat16, device=DEV)
    for _ in range(2):
        assert triton_attn_func(q, k, k, softmax_scale=1.0).shape == (2, 5, 3, 0)
        leaves = [t.clone().requires_grad_(True) for t in (q, k, k)]
        out = triton_attn_func(*leaves, softmax_scale=1.0)
        grads = torch.autograd.grad(out, leaves, torch.empty_like(out))
        assert [g.shape for g in grads] == [q.shape, k.shape, k.shape]
    for Sq, Sk in ((0, 7), (5, 0)):
        for D in (72, 100):
            q, k = (torch.empty(2, n, 3, D, dtype=torch.bfloat16, device=DEV) for n in (Sq, Sk))
            with pytest.raises(ValueError, match="trinix_attn_fwd.*: invalid or inconsistent sizes"):
                triton_attn_func(q, k, k)
