"""The fp32 forward's row sums (``csrc/attn_fwd_f32.hip``): summed per 32-key
tile, then over the tiles, so that a long row's denominator (and the lse the
backward exponentiates) carries the rounding of its tiles, not of its keys."""
import math

import pytest
import torch

from trinix_amd.kernels.attention_kernel import TritonAttentionKernel


@pytest.mark.gpu
@pytest.mark.parametrize("D,ks", [(64, 1), (64, 2), (128, 1), (128, 2), (256, 1)])
def test_row_sum_error_grows_with_tiles(monkeypatch, D, ks):
    """One key at score 0 and n - 1 at -delta: the weights are 1 and one value
    p < 1, whose sum a running fp32 total rounds the same way at every step
    (2.4e-4 for this delta, by emulation).  Bound, with u = 2^-24: 16 terms of a
    lane's tile, one add per tile, one for the two lanes and, with two
    wavefronts, a merge: (16 + tiles + 3) u; p itself 4u; the lse's own
    rounding 2u |lse|."""
    n, delta = 32768, 0.7488721804511279
    print(f"row sum D={D} ks={ks}", flush=True)
    monkeypatch.setenv("TRINIX_F32_KS", str(ks))
    q = torch.zeros(1, 32, 1, D)
    q[..., 0] = 1.0
    k = torch.zeros(1, n, 1, D)
    k[:, 1:, :, 0] = -delta
    v = torch.randn(1, n, 1, D, generator=torch.Generator().manual_seed(0))
    _, lse = TritonAttentionKernel.apply(q.cuda(), k.cuda(), v.cuda(), scale=1.0, return_lse=True)
    want = math.log1p((n - 1) * math.exp(k[0, 1, 0, 0].double().item()))
    u = 2.0 ** -24
    bound = (16 + n // 32 + 3 + 4) * u + 2 * u * abs(want)
    err = (lse.double().cpu() - want).abs().max().item()
    assert err <= bound, (err, bound)
