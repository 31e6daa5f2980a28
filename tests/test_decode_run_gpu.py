"""The chunks a decode launch runs (``decode_run_plan``): one to four
workgroups per CU inside the planned workspace, with and without
non-temporal K/V loads."""
import pytest
import torch

from oracle import attention_oracle as orc
from test_attn_gpu import assert_parity_or_more_accurate, oracle_on, rand
from trinix_amd import triton_attn_func

pytestmark = pytest.mark.gpu

CASES = [
    # (B, Sq, Sk, Hq, Hkv, D, kwargs)
    (32, 1, 513, 8, 8, 128, dict()),                      # 256 items: unsplit, streamed
    (24, 1, 300, 8, 8, 128, dict()),                      # 192: unsplit, CUs idle
    (20, 1, 700, 16, 8, 128, dict(window_size=(0, 600))),  # 160 items, 3 chunks, a window's span
    (48, 1, 400, 8, 8, 128, dict()),                      # 384 items, short rows: unsplit, through the caches
    (48, 1, 1200, 8, 8, 128, dict()),                     # 384 items, 2 chunks each, streamed in three rounds
    (2, 3, 5000, 8, 1, 128, dict()),                      # 2 items, 24 rows: two row groups per KV head
    (64, 1, 257, 4, 4, 64, dict()),                       # head_dim 64, one workgroup per CU
    (12, 1, 1000, 16, 16, 64, dict()),                    # head_dim 64, the planned count
    (16, 1, 1001, 32, 8, 128, dict(mask=True)),           # 128 items, 2 chunks, a ragged last step, mask + ALiBi
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=[str(c) for c in CASES])
def test_run_chunks_match_the_oracle_and_the_planned_chunks(case, dtype, monkeypatch):
    """Against the oracle, and the planned chunks (P and the partial sums are
    fp32 in both: one rounding of the output apart, and 1e-5 of sum p|v| for
    sums in another order)."""
    B, Sq, Sk, H, Hkv, D, kw = case
    q, k, v = rand((B, Sq, H, D), dtype, 11), rand((B, Sk, Hkv, D), dtype, 12), rand((B, Sk, Hkv, D), dtype, 13)
    kw = dict(kw)
    if kw.pop("mask", False):
        m = torch.randn((Sq, Sk), generator=torch.Generator().manual_seed(14))
        m[:, 5:90] = float("-inf")
        kw.update(attn_mask=m.to(q.device), alibi_slopes=orc.alibi_slopes(H).to(q.device))
    out, lse = triton_attn_func(q, k, v, return_lse=True, **kw)
    monkeypatch.setenv("TRINIX_SPLITKV_CFG", "1024,128")
    planned, plse = triton_attn_func(q, k, v, return_lse=True, **kw)
    monkeypatch.delenv("TRINIX_SPLITKV_CFG")
    eps = torch.finfo(dtype).eps
    assert ((out.float() - planned.float()).abs() <= eps * planned.float().abs() + 1e-5 * v.float().abs().max()).all()
    assert ((lse - plse).abs() <= 1e-5 * (1 + plse.abs())).all()
    ckw = {a: (b.cpu() if torch.is_tensor(b) else b) for a, b in kw.items()}
    ref = oracle_on(q, k, v, **ckw)
    assert_parity_or_more_accurate(out, ref, orc.closed_form(q.cpu(), k.cpu(), v.cpu(), **ckw), dtype, str(case))
