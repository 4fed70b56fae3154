"""GPU: the forward that finds its work items from the metadata, around where it begins and
ends (64 segments, 320 workgroups on 256 CUs, 768 with segments of at most 1024 rows), with
empty segments and padding rows: bitwise the outputs of the same call over a host-built list,
since an item's result depends on neither its place in the grid nor the others; and the error
word that an inconsistent segment leaves."""
import pytest
import torch

from prefixlm import build_plan, op
from prefixlm.synth import make_batch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")

SHAPES = {
    "one_row": ([1], [0], 3),
    "empty_segments": ([0, 0, 130, 0], [0, 200, 0, 0], 8),
    "63_segments": ([i % 5 for i in range(63)], [1 + i % 40 for i in range(63)], 2),
    "64_segments": ([i % 7 for i in range(64)], [i % 60 for i in range(64)], 2),
    "65_segments": ([i % 7 for i in range(65)], [1 + i % 60 for i in range(65)], 2),
    "many_segments_end_of_tiles": ([128, 0, 127, 1, 256], [0, 128, 1, 128, 1], 9),
    # (rows / 128 + segments) x heads workgroups: 320 and 336 with a segment above 1024 rows
    "at_320": ([1000, 100], [1200, 4], 16),
    "above_320": ([1000, 100], [1200, 132], 16),
    # 768 and 784 with none
    "at_768": ([512] * 5, [500] * 5, 16),
    "above_768": ([512] * 5, [512] * 4 + [436], 17),
}


@pytest.mark.parametrize("is_causal", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_same_as_over_a_list(shape, D, is_causal):
    prefix, causal, H = SHAPES[shape]
    b = make_batch(prefix, causal, sum(prefix) + sum(causal) + 3, H, D, seed=D + H, device=DEV)
    plan = torch.from_numpy(build_plan(b.seq_tensors, b.seq_scalars, is_causal)).to(DEV)
    got = op.varlen_fwd(b.q, b.k, b.v, is_causal, *b.seq_info.values(), D ** -0.5)
    want = op.varlen_fwd(b.q, b.k, b.v, is_causal, *b.seq_info.values(), D ** -0.5, plan)
    for name, x, y in zip(("out", "lse", "out_lo"), got, want):
        assert torch.equal(x, y), name
    # the max |Q| slots belong to workgroups; the backward only uses each head's largest
    args = (b.dout, *got[:3])
    for x, y in zip(op.varlen_bwd(b.q, b.k, b.v, is_causal, *args, got[3], *b.seq_info.values(), D ** -0.5),
                    op.varlen_bwd(b.q, b.k, b.v, is_causal, *args, want[3], *b.seq_info.values(), D ** -0.5)):
        assert torch.equal(x, y)


@pytest.mark.parametrize("field,index,value", [("cu_seqlens", 0, 1), ("prefix_lens", 1, -1), ("causal_lens", 2, 500)])
def test_error_word(field, index, value, monkeypatch):
    monkeypatch.setattr(op, "_CHECK_METADATA", True)
    b = make_batch([10, 20, 30], [40, 50, 60], 220, 2, 128, seed=1, device=DEV)
    op.varlen_fwd(b.q, b.k, b.v, False, *b.seq_info.values(), 128 ** -0.5)
    b.seq_info[field][index] = value
    with pytest.raises(RuntimeError):
        op.varlen_fwd(b.q, b.k, b.v, False, *b.seq_info.values(), 128 ** -0.5)
