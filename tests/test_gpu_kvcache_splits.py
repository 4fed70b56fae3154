"""GPU: KV-cache attention at both sides of the lines where a call gives up splitting the keys
(decode: caches of 384 and 1088 rows, 128 (row, head) pairs; several new rows: the tiles against the
partials) or change a decode workgroup's size (64 cache rows, 256 pairs), with empty, ragged and full caches, against the oracle.

Tolerance per element: half a bf16 ulp of the reference (2^-8 |ref|, the output's own rounding)
plus 2^-14 max|V| for fp32 sums in another order."""
import pytest
import torch

from oracle.kvcache_oracle import kvcache_attention
from prefixlm import flash_attn_with_kvcache

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("B,S,H,Smax", [
    (1, 1, 1, 1), (2, 1, 3, 64), (2, 1, 3, 65), (3, 1, 3, 127), (3, 1, 3, 129), (2, 1, 3, 384), (2, 1, 3, 385),
    (8, 1, 16, 384), (129, 1, 1, 384), (256, 1, 1, 300), (257, 1, 1, 300), (16, 1, 16, 1023),
    (9, 1, 16, 1087), (9, 1, 16, 1088), (18, 1, 20, 1090),
    (1, 5, 8, 128), (1, 5, 8, 256), (1, 5, 8, 257), (1, 64, 8, 128), (1, 64, 8, 129), (4, 64, 16, 512),
    (4, 64, 16, 513), (4, 100, 16, 256), (4, 100, 16, 480), (16, 33, 16, 200), (16, 20, 8, 500)])
def test_matches_oracle(B, S, H, Smax):
    g = torch.Generator().manual_seed(B + S + Smax)
    q, k, v, kc, vc = (torch.randn(B, n, H, 128, generator=g).to(torch.bfloat16) for n in (S, S, S, Smax, Smax))
    lens = torch.linspace(0, Smax - S, B).to(torch.int32)
    ref, kr, vr = kvcache_attention(q, kc, vc, k, v, lens, True)
    d = [t.to(DEV) for t in (q, k, v, kc, vc)]
    out = flash_attn_with_kvcache(d[0], d[3], d[4], k=d[1], v=d[2], cache_seqlens=lens.to(DEV), causal=True)
    assert torch.equal(d[3].cpu(), kr) and torch.equal(d[4].cpu(), vr)
    err = (out.float().cpu() - ref).abs()
    tol = ref.abs() * 2.0 ** -8 + vc.float().abs().max().item() * 2.0 ** -14
    assert (err <= tol).all(), f"worst {(err - tol).max().item():.3e} over, max_abs {err.max().item():.3e}"
