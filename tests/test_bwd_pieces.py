"""dK/dV in pieces (``trinix_attn_bwd_ws``): a key block's items cut into runs
that leave fp32 partial sums for a reduction (``csrc/attn_bwd16.h``,
``plan_bwd_pieces`` in ``csrc/host_plan.cpp``)."""
import ctypes

import pytest
import torch

import trinix_amd.kernels.attention_kernel as ak
from oracle import attention_oracle as orc
from trinix_amd import _native as nat
from trinix_amd import triton_attn_func

DEV = "cuda"


def _args(B, S, Hq, Hkv, D, causal=True, dtype=nat.TRINIX_BF16):
    a = nat.AttnBwdArgs()
    for f in ("q", "k", "v", "out", "dout", "lse", "delta", "dq", "dk", "dv"):
        setattr(a, f, 4096)
    for f, h in (("q", Hq), ("k", Hkv), ("v", Hkv), ("out", Hq), ("dout", Hq), ("dq", Hq), ("dk", Hkv), ("dv", Hkv)):
        setattr(a, f + "_stride", nat.int64x4((S * h * D, h * D, D, 1)))
    a.batch, a.seqlen_q, a.seqlen_k, a.nheads_q, a.nheads_kv, a.head_dim = B, S, S, Hq, Hkv, D
    a.dtype, a.softmax_scale, a.causal = dtype, D ** -0.5, int(causal)
    return a


def _workspace(a):
    n = ctypes.c_int64(-1)
    rc = nat.load_library().trinix_attn_bwd_workspace(ctypes.byref(a), ctypes.byref(n))
    return rc, n.value


@pytest.fixture
def built():
    if not nat.LIB_PATH.exists():
        pytest.skip("the HIP library is not built")


def test_workspace_plan(built, monkeypatch):
    monkeypatch.delenv("TRINIX_BWD_PIECES", raising=False)
    # few KV heads: pieces; 128 keys x D x (dk, dv) fp32 each, one to two per CU
    rc, n = _workspace(_args(2, 2048, 16, 4, 128))
    piece = 2 * 128 * 128 * 4
    assert rc == 0 and n % (8 * piece) == 0 and 128 * piece < n <= 512 * piece
    # a grid that fills the chip, a single item per block, fp32 and head_dim 256: whole blocks
    for a in (_args(1, 8192, 32, 8, 128), _args(1, 64, 4, 4, 128), _args(2, 2048, 16, 4, 128, dtype=nat.TRINIX_F32),
              _args(2, 2048, 16, 4, 256)):
        assert _workspace(a) == (0, 0)
    # more key blocks than a wavefront counts
    assert _workspace(_args(1, 64 * 128 + 1, 4, 1, 128)) == (0, 0)
    assert _workspace(_args(1, 0, 4, 1, 128))[0] == nat.TRINIX_ERR_BAD_SHAPE
    lib = nat.load_library()
    assert lib.trinix_attn_bwd_workspace(ctypes.byref(_args(1, 64, 4, 4, 128)), None) == nat.TRINIX_ERR_NULL_POINTER


def test_workspace_is_checked_before_any_launch(built, monkeypatch):
    monkeypatch.delenv("TRINIX_BWD_PIECES", raising=False)
    lib, a = nat.load_library(), _args(2, 2048, 16, 4, 128)
    need = _workspace(a)[1]
    for ws, n in ((None, need), (4096, need - 1), (4100, need)):
        assert lib.trinix_attn_bwd_ws(ctypes.byref(a), ws, n, None) == nat.TRINIX_ERR_BAD_ARGUMENT


SHAPES = [
    # (B, Sq, Sk, Hq, Hkv, D, kwargs): one and several groups per XCD, key blocks of one item and none, partial tiles
    (1, 300, 300, 4, 1, 128, dict(causal=True)),
    (8, 130, 200, 2, 1, 64, dict()),
    (2, 257, 129, 6, 2, 128, dict(window_size=(60, 10))),
    (1, 100, 500, 2, 2, 64, dict(causal=True)),
    (2, 200, 200, 4, 2, 128, dict(causal=True, dropout_p=0.2)),
]


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 2, 5])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", range(len(SHAPES)))
def test_pieces_match_whole_blocks(monkeypatch, case, dtype, T):
    """Pieces sum the same products in another order, in fp32 (1e-5 of the
    scale), so two results round to the same or to neighbouring 16-bit values:
    one ulp, at most 2u of the element, apart; bitwise the same every run."""
    B, Sq, Sk, Hq, Hkv, D, kw = SHAPES[case]
    print(f"pieces {SHAPES[case]} {dtype} T {T}", flush=True)
    g = torch.Generator().manual_seed(case)
    ts = [torch.randn(s, generator=g).to(dtype).to(DEV)
          for s in ((B, Sq, Hq, D), (B, Sk, Hkv, D), (B, Sk, Hkv, D), (B, Sq, Hq, D))]

    def grads(pieces):
        monkeypatch.setenv("TRINIX_BWD_PIECES", str(pieces))
        monkeypatch.setattr(ak, "_TRAIN_LAUNCHES", {})
        torch.manual_seed(77)
        leaves = [t.clone().requires_grad_(True) for t in ts[:3]]
        return torch.autograd.grad(triton_attn_func(*leaves, **kw), leaves, ts[3])

    whole, first, second = grads(0), grads(T), grads(T)
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for name, w, a, b in zip(("dq", "dk", "dv"), whole, first, second):
        assert torch.equal(a, b), name
        d, scale = (a.double() - w.double()).abs(), w.double().abs().max()
        assert (d <= 2 * u * w.double().abs() + 1e-5 * scale).all(), (name, d.max().item(), scale.item())



FEATURES = [
    # (B, Sq, Sk, Hq, Hkv, D, kwargs): the mask and ALiBi variants of the kernel, and head_dims between the kernels'
    # (narrow rows, the partial sums behind a padded dout)
    (2, 150, 260, 4, 2, 64, dict(attn_mask=True)),
    (1, 260, 260, 4, 1, 128, dict(attn_mask=True, alibi_slopes=True)),
    (2, 130, 200, 4, 2, 64, dict(alibi_slopes=True, causal=True)),
    (1, 140, 270, 4, 2, 128, dict(attn_mask=True, dropout_p=0.25)),
    (1, 140, 140, 2, 1, 64, dict(attn_mask=True, alibi_slopes=True, dropout_p=0.25, causal=True)),
    (2, 150, 260, 4, 2, 40, dict(causal=True)),
    (1, 260, 150, 4, 1, 80, dict()),
    (2, 150, 260, 4, 2, 72, dict(attn_mask=True, alibi_slopes=True)),
    (1, 140, 270, 4, 2, 112, dict(dropout_p=0.25, causal=True)),
    (1, 140, 270, 4, 2, 56, dict(attn_mask=True, dropout_p=0.25)),
]


@pytest.mark.gpu
@pytest.mark.parametrize("T", [0, 1, 3])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", range(len(FEATURES)))
def test_features_in_pieces(monkeypatch, case, dtype, T):
    """Whole blocks (T = 0) and pieces against float64 autograd: twice the eager
    error plus 2e-3 of the scale, the bar of the other gradient tests; with
    dropout, pieces against whole blocks of the same seed alone (bound as in
    test_pieces_match_whole_blocks)."""
    B, Sq, Sk, Hq, Hkv, D, kw = FEATURES[case]
    print(f"pieces {FEATURES[case]} {dtype} T {T}", flush=True)
    g = torch.Generator().manual_seed(100 + case)
    ts = [torch.randn(s, generator=g).to(dtype)
          for s in ((B, Sq, Hq, D), (B, Sk, Hkv, D), (B, Sk, Hkv, D), (B, Sq, Hq, D))]
    kw = dict(kw)
    if "attn_mask" in kw:  # a block mask: some 64-key blocks are skipped, key block 0 stays open
        m = torch.zeros(Sq, Sk)
        m[: Sq // 2, 64:128] = float("-inf")
        m[Sq // 2:, 192:] = -1.5
        kw["attn_mask"] = m
    if "alibi_slopes" in kw:
        kw["alibi_slopes"] = orc.alibi_slopes(Hq)
    gpu = {k: v.to(DEV) if torch.is_tensor(v) else v for k, v in kw.items()}

    def grads(pieces):
        monkeypatch.setenv("TRINIX_BWD_PIECES", str(pieces))
        monkeypatch.setattr(ak, "_TRAIN_LAUNCHES", {})
        torch.manual_seed(77)
        leaves = [t.to(DEV).requires_grad_(True) for t in ts[:3]]
        return [t.cpu().double() for t in torch.autograd.grad(triton_attn_func(*leaves, **gpu), leaves, ts[3].to(DEV))]

    got = grads(T)
    if "dropout_p" in kw:
        u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
        for name, w, a in zip(("dq", "dk", "dv"), grads(0), got):
            d, scale = (a - w).abs(), w.abs().max()
            assert (d <= 2 * u * w.abs() + 1e-5 * scale).all(), (name, d.max().item(), scale.item())
        return

    def ref(dt):
        leaves = [t.to(dt).requires_grad_(True) for t in ts[:3]]
        return [t.double() for t in torch.autograd.grad(orc.functional_attention(*leaves, **kw), leaves, ts[3].to(dt))]

    for name, h, e, t in zip(("dq", "dk", "dv"), got, ref(dtype), ref(torch.float64)):
        scale = t.abs().max().item()
        err_h, err_e = (h - t).abs().max().item(), (e - t).abs().max().item()
        assert err_h <= 2 * err_e + 2e-3 * scale, (name, err_h, err_e, scale)


@pytest.mark.gpu
def test_changed_switch_between_calls_of_one_layout(monkeypatch):
    """The backward's template keeps the workspace size of the plan it was
    built with; a call whose plan has come to need more plans anew."""
    B, S, Hq, Hkv, D = 1, 300, 4, 1, 128
    g = torch.Generator().manual_seed(5)
    ts = [torch.randn(s, generator=g).to(torch.bfloat16).to(DEV)
          for s in ((B, S, Hq, D), (B, S, Hkv, D), (B, S, Hkv, D), (B, S, Hq, D))]
    monkeypatch.setattr(ak, "_TRAIN_LAUNCHES", {})
    launch, sizes = ak._launch_bwd, []

    def record(a, ws, *rest):
        sizes.append(ws)
        return launch(a, ws, *rest)

    monkeypatch.setattr(ak, "_launch_bwd", record)

    def grads(pieces):
        monkeypatch.setenv("TRINIX_BWD_PIECES", pieces)
        leaves = [t.clone().requires_grad_(True) for t in ts[:3]]
        return torch.autograd.grad(triton_attn_func(*leaves, causal=True), leaves, ts[3])

    first = {}
    for pieces in ("5", "5", "1", "0", "5", "1"):  # the template is built by the first call
        got = grads(pieces)
        want = first.setdefault(pieces, got)
        assert all(torch.equal(a, b) for a, b in zip(got, want)), pieces
    few, many = (n * 2 * 128 * D * 4 for n in (4 + 3 + 1, 20 + 12 + 4))  # 4 heads x 5, 3 and 1 query tiles
    assert sizes == [few, few, few, many, few, few, few, many]
    monkeypatch.setattr(ak, "_TRAIN_LAUNCHES", {})
    assert all(torch.equal(a, b) for a, b in zip(grads("0"), first["0"]))
