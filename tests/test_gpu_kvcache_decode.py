"""GPU: one new row per sequence at the edges of the decode kernel's key steps (64) and
splits: lengths from an empty to a full cache, one split written directly, up to 64 splits
merged, and a cache row shared by the batch (where the append keeps a launch of its own).

Tolerance per element: half a bf16 ulp of the reference (2^-8 |ref|) plus 2^-14 max|V| for
fp32 sums in another order."""
import pytest
import torch

from oracle.kvcache_oracle import kvcache_attention
from prefixlm import flash_attn_with_kvcache

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _run(B, H, Smax, lens, shared=False):
    g = torch.Generator().manual_seed(B * 1000 + Smax)
    mk = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)  # noqa: E731
    q, k, v = mk(B, 1, H, 128), mk(B, 1, H, 128), mk(B, 1, H, 128)
    kc, vc = mk(1 if shared else B, Smax, H, 128), mk(1 if shared else B, Smax, H, 128)
    kd, vd = kc.to(DEV), vc.to(DEV)
    if shared:
        k, v = (x[:1].expand(B, -1, -1, -1) for x in (k, v))
        kc, vc, kd, vd = (x.expand(B, -1, -1, -1) for x in (kc, vc, kd, vd))
    lens = torch.tensor(lens, dtype=torch.int32)
    ref, kr, vr = kvcache_attention(q, kc, vc, k, v, lens)
    out = flash_attn_with_kvcache(q.to(DEV), kd, vd, k=k.to(DEV), v=v.to(DEV), cache_seqlens=lens.to(DEV))
    assert torch.equal(kd.cpu(), kr) and torch.equal(vd.cpu(), vr)
    err = (out.float().cpu() - ref).abs()
    tol = ref.abs() * 2.0 ** -8 + v.abs().max().item() * 2.0 ** -14
    assert (err <= tol).all(), f"max_abs {err.max().item():.3e}"


# 11 splits of one step; 64 splits of 128 keys, the last 24 without keys; one split of a short cache in
# a batch that fills the chip
@pytest.mark.parametrize("B,H,Smax", [(9, 5, 700), (1, 2, 5000), (130, 2, 129)])
def test_decode_lengths(B, H, Smax):
    edges = [0, 1, 63, 64, 65, 127, 128, Smax // 2, Smax - 1, Smax]
    _run(B, H, Smax, [min(edges[i % len(edges)] if B > 1 else Smax - 1, Smax) for i in range(B)])


def test_decode_shared_cache_row():
    _run(3, 4, 300, [200, 200, 200], shared=True)


@pytest.mark.parametrize("value", [float("-inf"), -3.3e38])
@pytest.mark.parametrize("where", ["new", "cached", "all"])
@pytest.mark.parametrize("B,H,Smax", [(10, 4, 700), (130, 2, 129), (2, 2, 300)])
def test_decode_keys_of_score_minus_infinity(B, H, Smax, where, value):
    """Keys whose score is -inf weigh nothing: the new one, every cached one of the first two key
    steps, or all of a row's, which alone makes its output NaN. A row without keys is 0."""
    print(f"[case] decode -inf B={B} Smax={Smax} {where} {value}", flush=True)
    g = torch.Generator().manual_seed(B + Smax)
    mk = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)  # noqa: E731
    q, k, v, kc, vc = mk(B, 1, H, 128), mk(B, 1, H, 128), mk(B, 1, H, 128), mk(B, Smax, H, 128), mk(B, Smax, H, 128)
    q[..., 7] = 16.0                              # 16 * -3.3e38 is past the range of fp32, scaled or not
    if where != "cached":
        k[..., 7] = value
    if where != "new":
        kc[:, :128 if where == "cached" else Smax, :, 7] = value
    edges = [1, 16, 17, 63, 64, 65, 128, Smax // 2, Smax - 2, 0]
    lens = torch.tensor([min(edges[(i + (where == "cached")) % 10], Smax - 1) for i in range(B)], dtype=torch.int32)
    ref, _, _ = kvcache_attention(q, kc, vc, k, v, lens)
    assert torch.isnan(ref).any() == (where == "all" or (where == "new" and 0 in lens.tolist()))
    d = [t.to(DEV) for t in (q, k, v, kc, vc)]
    out = flash_attn_with_kvcache(d[0], d[3], d[4], k=d[1], v=d[2], cache_seqlens=lens.to(DEV)).float().cpu()
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    err, tol = (out - ref).abs(), ref.abs() * 2.0 ** -8 + 5.0 * 2.0 ** -14
    assert (torch.isnan(ref) | (err <= tol)).all()
    none = flash_attn_with_kvcache(d[0], d[3], d[4], cache_seqlens=torch.zeros_like(lens).to(DEV))
    assert (none == 0).all()
