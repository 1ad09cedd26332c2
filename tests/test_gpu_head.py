"""mtl_lm_head (the lm_head of at most 16 rows) against the float64 product and
the library's, at the ends of its ranges and where a tile is partial."""
import math

import pytest
import torch
import torch.nn.functional as F

from mamba_lite import ops

pytestmark = pytest.mark.gpu


# M, N, K: the fewest and most rows, N below one tile, of one partial tile, not a multiple of the tile, more tiles than
# workgroups; K at both ends and in between (an odd number of blocks)
@pytest.mark.parametrize("dtype,ks", [(torch.float32, (1024, 1152, 2048)), (torch.bfloat16, (2048, 2304, 4096))])
@pytest.mark.parametrize("M,N", [(1, 4), (16, 20), (7, 1000), (3, 50280), (16, 33000)])
def test_matches_float64(M, N, dtype, ks):
    for K in ks:
        g = torch.Generator(device="cuda").manual_seed(N + K)
        x = torch.randn(M, K, device="cuda", generator=g).to(dtype)
        w = (torch.randn(N, K, device="cuda", generator=g) * 0.02).to(dtype)
        ref = x.double() @ w.double().t()
        e = float((ops.lm_head(x, w).double() - ref).norm() / ref.norm())
        # fp32: a random walk of K rounded adds, 2^-24 sqrt(K); bf16: the output's rounding, 8 significand bits, at most 2^-8 (half of 2^-7)
        assert e < (2.0 ** -24 * math.sqrt(K) if dtype == torch.float32 else 2.0 ** -8), (K, e)


def test_where_it_is_taken():
    x, w = torch.randn(5, 2048, device="cuda"), torch.randn(32768, 2048, device="cuda")
    assert ops.lm_head_ok(x, w) and not ops.lm_head_ok(x, w[:20000]) and not ops.lm_head_ok(x, w.bfloat16())
    assert not ops.lm_head_ok(torch.randn(17, 2048, device="cuda"), w)
    assert not ops.lm_head_ok(x[:, :768].contiguous(), w[:, :768].contiguous())
    wp = torch.nn.Parameter(w)
    assert not ops.lm_head_ok(x, wp)          # gradients are being recorded
    with torch.no_grad():
        assert ops.lm_head_ok(x, wp)
        a, b = ops.lm_head(x, wp), F.linear(x, wp)
    assert float((a - b).norm() / b.norm()) < 2e-6
