"""GPU: prompts into an empty cache (forward and append in one launch) at the edges of the
128-row tiles, with head counts that do not divide over the XCDs, strided and larger caches.

Tolerance per element: half a bf16 ulp of the reference (2^-8 |ref|) for the output, and
2^-9 max|V| for P rounded to bf16 (a relative 2^-9 of every probability; they sum to 1)."""
import pytest
import torch

from oracle.kvcache_oracle import kvcache_attention
from prefixlm import flash_attn_with_kvcache

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,S,H,Smax", [(1, 1, 1, 1), (3, 1, 2, 8), (2, 127, 10, 200), (3, 128, 3, 128), (2, 129, 12, 300),
                                        (1, 515, 20, 515)])
def test_prefill_edges(B, S, H, Smax, causal):
    g = torch.Generator().manual_seed(S)
    mk = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)  # noqa: E731
    q, k, v = mk(B, S, H, 128), mk(B, S, H, 128), mk(B, S, H, 128)
    kc, vc = mk(B, H, Smax, 128).transpose(1, 2), mk(B, Smax, H, 128)   # k_cache laid out heads first
    ref, kr, vr = kvcache_attention(q, kc, vc, k, v, 0, causal)
    kd, vd = kc.transpose(1, 2).to(DEV).transpose(1, 2), vc.to(DEV)
    out = flash_attn_with_kvcache(q.to(DEV), kd, vd, k=k.to(DEV), v=v.to(DEV), cache_seqlens=0, causal=causal)
    assert torch.equal(kd.cpu(), kr) and torch.equal(vd.cpu(), vr)
    err = (out.float().cpu() - ref).abs()
    assert (err <= ref.abs() * 2.0 ** -8 + v.abs().max().item() * 2.0 ** -9).all(), f"max_abs {err.max().item():.3e}"


@pytest.mark.parametrize("causal", [False, True])
def test_prefill_of_more_tiles_than_the_chip_holds(causal):
    """17 sequences x 3 tiles x 20 heads: one sequence after another without a causal mask."""
    B, S, H = 17, 300, 20
    g = torch.Generator().manual_seed(S)
    q, k, v, kc, vc = (torch.randn(B, S, H, 128, generator=g).to(torch.bfloat16) for _ in range(5))
    ref, kr, vr = kvcache_attention(q, kc, vc, k, v, 0, causal)
    kd, vd = kc.to(DEV), vc.to(DEV)
    out = flash_attn_with_kvcache(q.to(DEV), kd, vd, k=k.to(DEV), v=v.to(DEV), cache_seqlens=0, causal=causal)
    assert torch.equal(kd.cpu(), kr) and torch.equal(vd.cpu(), vr)
    err = (out.float().cpu() - ref).abs()
    assert (err <= ref.abs() * 2.0 ** -8 + v.abs().max().item() * 2.0 ** -9).all(), f"max_abs {err.max().item():.3e}"
