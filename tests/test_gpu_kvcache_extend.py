"""GPU: several new rows per sequence onto filled caches (the extend kernel) against the
oracle, at the edges of its query blocks (32, 64, 128 rows), key tiles (32, 64, 128 keys)
and key splits, with rows that fall past the cache, cached-only calls, strided and shared
caches, and non-finite values.

Tolerance per element: half a bf16 ulp of the reference (2^-8 |ref|, the output's own
rounding) plus 2^-14 max|V|: P enters P V with its fp32 bits, and fp32 sums of up to 1500 terms in
another order stay below 2^-15."""
import pytest
import torch

from oracle.kvcache_oracle import kvcache_attention
from prefixlm import flash_attn_with_kvcache

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _inputs(B, S, H, Smax, seed):
    g = torch.Generator().manual_seed(seed)
    mk = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)  # noqa: E731
    return mk(B, S, H, 128), mk(B, S, H, 128), mk(B, S, H, 128), mk(B, Smax, H, 128), mk(B, Smax, H, 128)


def _check(got, ref, v_max):
    got = got.float().cpu()
    err, tol = (got - ref).abs(), ref.abs() * 2.0 ** -8 + v_max * 2.0 ** -14
    assert (err <= tol).all(), f"worst {(err - tol).max().item():.3e} over, max_abs {err.max().item():.3e}"


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("S", [2, 31, 32, 33, 64, 65, 127, 128, 130])
def test_extend_matches_oracle(S, causal):
    B, H, Smax = 4, 3, 700
    q, k, v, kc, vc = _inputs(B, S, H, Smax, S)
    lens = torch.tensor([0, 127, 500, Smax - S], dtype=torch.int32)
    ref, kr, vr = kvcache_attention(q, kc, vc, k, v, lens, causal)
    d = [t.to(DEV) for t in (q, k, v, kc, vc)]
    out = flash_attn_with_kvcache(d[0], d[3], d[4], k=d[1], v=d[2], cache_seqlens=lens.to(DEV), causal=causal)
    assert torch.equal(d[3].cpu(), kr) and torch.equal(d[4].cpu(), vr)
    _check(out, ref, v.abs().max().item())


@pytest.mark.parametrize("B,S,H,Smax", [(2, 40, 16, 1500), (70, 70, 16, 70), (9, 300, 16, 320)])
def test_extend_splits(B, S, H, Smax):
    """Many splits of few units, and more units than the grid wants (one split, written directly)."""
    q, k, v, kc, vc = _inputs(B, S, H, Smax, B)
    lens = torch.arange(B, dtype=torch.int32) * 7 % (Smax - S + 1)
    ref, kr, vr = kvcache_attention(q, kc, vc, k, v, lens, True)
    d = [t.to(DEV) for t in (q, k, v, kc, vc)]
    out = flash_attn_with_kvcache(d[0], d[3], d[4], k=d[1], v=d[2], cache_seqlens=lens.to(DEV), causal=True)
    assert torch.equal(d[3].cpu(), kr) and torch.equal(d[4].cpu(), vr)
    _check(out, ref, v.abs().max().item())


@pytest.mark.parametrize("new", [True, False])
def test_extend_past_the_cache_and_cached_only(new):
    """Rows past Smax are dropped; without new rows the queries see the cached ones."""
    B, S, H, Smax = 3, 20, 2, 200
    q, k, v, kc, vc = _inputs(B, S, H, Smax, 3)
    lens = torch.tensor([190, 60, 200], dtype=torch.int32)
    ref, kr, vr = kvcache_attention(q, kc, vc, k if new else None, v if new else None, lens, False)
    d = [t.to(DEV) for t in (q, k, v, kc, vc)]
    out = flash_attn_with_kvcache(d[0], d[3], d[4], k=d[1] if new else None, v=d[2] if new else None,
                                  cache_seqlens=lens.to(DEV))
    assert torch.equal(d[3].cpu(), kr) and torch.equal(d[4].cpu(), vr)
    _check(out, ref, 5.0)


@pytest.mark.parametrize("layout", ["heads_first", "shared_batch", "negative_scale"])
def test_extend_strides(layout):
    """Caches laid out [B, H, Smax, D]; one cache row shared by the whole batch (appended
    before it is read, so every sequence must see the same rows); a negative softmax scale."""
    B, S, H, Smax = 2, 33, 3, 300
    q, k, v, kc, vc = _inputs(B, S, H, Smax, 11)
    lens = torch.tensor([100, 230], dtype=torch.int32)
    scale = -0.05 if layout == "negative_scale" else None
    if layout == "shared_batch":
        k, v, lens = k[:1].expand(B, -1, -1, -1), v[:1].expand(B, -1, -1, -1), torch.tensor([100, 100], dtype=torch.int32)
        kc, vc = kc[:1].expand(B, -1, -1, -1), vc[:1].expand(B, -1, -1, -1)
        kd, vd = (x[:1].to(DEV).expand(B, -1, -1, -1) for x in (kc, vc))
    elif layout == "heads_first":
        kd, vd = (x.to(DEV).transpose(1, 2).contiguous().transpose(1, 2) for x in (kc, vc))
    else:
        kd, vd = kc.to(DEV), vc.to(DEV)
    ref, kr, vr = kvcache_attention(q, kc, vc, k, v, lens, True, scale)
    out = flash_attn_with_kvcache(q.to(DEV), kd, vd, k=k.to(DEV), v=v.to(DEV), cache_seqlens=lens.to(DEV), causal=True,
                                  softmax_scale=scale)
    assert torch.equal(kd.cpu(), kr) and torch.equal(vd.cpu(), vr)
    _check(out, ref, v.abs().max().item())


@pytest.mark.parametrize("S", [6, 50, 100])
def test_extend_non_finite_values(S):
    """A value row that is infinite reaches the queries that see it, as +-inf and not as NaN,
    and no other query."""
    B, H, Smax = 2, 2, 400
    q, k, v, kc, vc = _inputs(B, S, H, Smax, 21)
    lens = torch.tensor([150, 301], dtype=torch.int32)
    bad = S - 3                                    # the new row only the last three queries see
    v[:, bad] = float("inf")
    v[:, bad, :, 5] = float("-inf")
    ref, _, _ = kvcache_attention(q, kc, vc, k, v.nan_to_num(posinf=0.0, neginf=0.0), lens, True)
    d = [t.to(DEV) for t in (q, k, v, kc, vc)]
    out = flash_attn_with_kvcache(d[0], d[3], d[4], k=d[1], v=d[2], cache_seqlens=lens.to(DEV), causal=True).float().cpu()
    _check(out[:, :bad], ref[:, :bad], 5.0)
    want = torch.full_like(out[:, bad:], float("inf"))
    want[..., 5] = float("-inf")
    assert torch.equal(out[:, bad:], want)


@pytest.mark.parametrize("value_inf", [False, True])
@pytest.mark.parametrize("where", ["first", "all"])
@pytest.mark.parametrize("B,S,Smax", [(2, 6, 400), (2, 50, 400), (2, 100, 400), (70, 6, 60)])
def test_extend_keys_of_score_minus_infinity(B, S, Smax, where, value_inf):
    """Cached keys whose score is -inf weigh nothing, with and without a value row that is infinite
    (seen by the last three queries only); a query whose keys are all such is NaN."""
    print(f"[case] extend -inf B={B} S={S} {where} {value_inf}", flush=True)
    H = 2
    q, k, v, kc, vc = _inputs(B, S, H, Smax, 23)
    lens = torch.full((B,), min(150, Smax - S), dtype=torch.int32)
    lens[1] = Smax - S
    q[..., 3] = 2.0
    kc[:, :40, :, 3] = float("-inf")
    if where == "all":
        kc[1, ..., 3] = k[1, :S // 2, :, 3] = float("-inf")
    last = S - 3
    if value_inf:
        v[:, last] = float("inf")
    ref, _, _ = kvcache_attention(q, kc, vc, k, v.nan_to_num(posinf=0.0), lens, True)
    d = [t.to(DEV) for t in (q, k, v, kc, vc)]
    out = flash_attn_with_kvcache(d[0], d[3], d[4], k=d[1], v=d[2], cache_seqlens=lens.to(DEV), causal=True).float().cpu()
    rows = slice(0, last) if value_inf else slice(0, S)
    got, ref = out[:, rows], ref[:, rows]
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.isnan(ref).any() == (where == "all")
    _check(got.nan_to_num(), ref.nan_to_num(), 5.0)
    if value_inf:
        assert (out[:, last:] == float("inf")).all()


@pytest.mark.parametrize("S", [2, 40, 100])
@pytest.mark.parametrize("Smax,at", [(128, (0, 1, 2)), (1000, (700, 5, 6)), (1000, (0, 5, 800))])
def test_extend_keeps_the_bits_of_the_probabilities(S, Smax, at):
    """Three keys count: one of weight 1 and value 0, and two of nearly the same weight, 0.4 to 0.9,
    with values +1 and -1, whose difference of about 1e-4 is the output.

    Bound: half a bf16 ulp of the result plus 2^-21, four times what fp32 weights leave (an exponent
    below 2 in magnitude, rounded twice, and exp2 to 1 ulp, each weight less than 0.4 of the sum:
    2 * 0.4 * 2^-22.5). Weights of 16 bits are off by up to 2^-18 each."""
    B, H = 2, 5
    q, k, v, kc, vc = (torch.zeros(B, n, H, 128, dtype=torch.bfloat16) for n in (S, S, S, Smax, Smax))
    g = torch.Generator().manual_seed(S + Smax)
    q[..., 0] = (0.08 + 0.6 * torch.rand(B, S, H, generator=g)).to(torch.bfloat16)
    kc[..., 0], k[..., 0] = -3e4, -3e4
    for j, a, x in zip(at, (16.0, 1.0, 1.0078125), (0.0, 1.0, -1.0)):
        kc[:, j, :, 0], vc[:, j] = a, x
    lens = torch.full((B,), Smax - S, dtype=torch.int32)
    d = [t.to(DEV) for t in (q, k, v, kc, vc)]
    out = flash_attn_with_kvcache(d[0], d[3], d[4], k=d[1], v=d[2], cache_seqlens=lens.to(DEV), causal=True).double().cpu()
    w = torch.softmax(q[..., :1].double() * torch.tensor([16.0, 1.0, 1.0078125], dtype=torch.float64) / 128 ** 0.5, -1)
    ref = (w[..., 1] - w[..., 2]).unsqueeze(-1)
    worst = ((out - ref).abs() - ref.abs() * 2.0 ** -8).max().item()
    assert worst <= 2.0 ** -21, f"{worst:.3e}"


@pytest.mark.parametrize("scale", [None, -0.05])
@pytest.mark.parametrize("S", [1, 2, 40, 100])
def test_extend_scores_past_the_range_before_the_scale(S, scale):
    """Keys of about the type's lowest value: q k is -6e38, infinite in fp32, and -5e37 with the
    softmax scale. Every key of the first sequence scores the same, so its output is the mean of
    the values that a query sees; the second sequence sees one other key, which takes it all."""
    B, H, Smax = 2, 3, 300
    q, k, v, kc, vc = _inputs(B, S, H, Smax, 31)
    q.zero_(), k.zero_(), kc.zero_()
    q[..., 0] = 2.0 if scale is None else -2.0
    kc[..., 0] = k[..., 0] = -3e38
    kc[1, 7, :, 0] = 0.0
    lens = torch.tensor([130, 200], dtype=torch.int32)
    d = [t.to(DEV) for t in (q, k, v, kc, vc)]
    out = flash_attn_with_kvcache(d[0], d[3], d[4], k=d[1], v=d[2], cache_seqlens=lens.to(DEV), causal=True,
                                  softmax_scale=scale).float().cpu()
    rows = torch.cat((vc[0, :130], v[0])).double()
    mean = torch.stack([rows[:130 + i + 1].mean(0) for i in range(S)])
    _check(out[0], mean.float(), 5.0)
    assert torch.equal(out[1], vc[1, 7].float().expand(S, H, 128))
