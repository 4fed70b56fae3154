"""GPU: the forward of small grids, which deals an item's key tiles to two groups of waves,
around where it begins (segments of 256 rows, at most one workgroup per CU) and where its
groups are uneven: odd tile counts, rows that see keys of one group only, empty prefixes, both
head dims, both masks; O, the LSE and the gradients against the oracle.

Tolerance: half a bf16 ulp of the output (2^-8 |ref|) plus 2^-9 max|V| for P in bf16;
for the gradients the bar of the parity tests (2e-2), LSE 1e-3."""
import pytest
import torch

from oracle.prefixlm_oracle import attention_bwd, attention_fwd, segments_from_meta
from prefixlm import op
from prefixlm.synth import make_batch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("is_causal", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("prefix,causal,H", [([0], [255], 2), ([0], [256], 2), ([257], [0], 3), ([31, 0], [290, 33], 2),
                                             ([500, 1], [13, 0], 4), ([0, 64], [1, 700], 1),
                                             ([0], [1024], 32), ([0], [1152], 32)])
def test_small_grids(prefix, causal, H, D, is_causal):
    T = sum(prefix) + sum(causal) + 5
    b = make_batch(prefix, causal, T, H, D, seed=T + D, device=DEV)
    segs = segments_from_meta(b.prefix.tolist() + [0], b.causal.tolist() + [0], b.seq_tensors["cu_seqlens"], len(prefix))
    out, lse, lo, qa = op.varlen_fwd(b.q, b.k, b.v, is_causal, *b.seq_info.values(), D ** -0.5)
    ref, ref_lse = attention_fwd(b.q.float(), b.k.float(), b.v.float(), segs, is_causal)
    n = T - 5
    err = (out.float() - ref).abs()
    assert (err <= ref.abs() * 2.0 ** -8 + b.v.float().abs().max() * 2.0 ** -9).all(), f"max_abs {err.max().item():.3e}"
    assert (lse[:, :n] - ref_lse[:, :n]).abs().max().item() <= 1e-3
    assert (out[n:] == 0).all() and torch.isneginf(lse[:, n:]).all()
    got = op.varlen_bwd(b.q, b.k, b.v, is_causal, b.dout, out, lse, lo, qa, *b.seq_info.values(), D ** -0.5)
    want = attention_bwd(b.q.float(), b.k.float(), b.v.float(), b.dout.float(), segs, is_causal)
    for x, y in zip(got, want):
        assert (x.float() - y).abs().max().item() <= 2e-2
