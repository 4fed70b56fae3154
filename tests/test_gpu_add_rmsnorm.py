"""The residual add fused with the norm after it: bitwise the separate operations, over row
lengths around the kernel's chunk counts, strided, repeated and overlapping rows, and inside
the stack, where a hook on a block takes the separate operations."""
import pytest
import torch

from prefixlm import fused_attention_layer, rms_norm
from prefixlm import op as op_module
from prefixlm.hrm_stack import FusedLayer, HRMStack, HRMStackConfig, packed_position_ids
from prefixlm.norm_mlp import add_rms_norm, add_rms_scales, rms_norm_fwd, rms_norm_swiglu, rms_scaled_swiglu
from prefixlm.synth import metadata_tensors

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS = 1e-6


def _rand(*shape, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return torch.randn(shape, generator=g).to(torch.bfloat16).to(DEV)


def _same(got, want):
    assert got.shape == want.shape and got.dtype == want.dtype and got.is_contiguous()
    torch.testing.assert_close(got, want, rtol=0, atol=0, equal_nan=True)


@pytest.fixture(params=["native", "ops"])
def path(request, monkeypatch):
    if request.param == "ops":
        import prefixlm.norm_mlp as m
        monkeypatch.setattr(m, "_native_calls", lambda: None)
    else:
        assert op_module._native_calls() is not None
    return request.param


@pytest.mark.parametrize("rows,cols", [(1, 8), (3, 504), (5, 512), (7, 520), (9, 1024), (4, 1032), (130, 2048),
                                       (2, 2056), (3, 4096), (3, 4104), (2, 8192)])
def test_add_rms_norm(path, rows, cols):
    print(f"[case] add_rms_norm {path} rows={rows} cols={cols}", flush=True)
    wide = _rand(rows, cols + 8)
    one = _rand(cols, seed=1)
    over = _rand(rows * 8 + cols, seed=2).as_strided((rows, cols), (8, 1))
    odd = _rand(rows, cols + 3, seed=3)[:, 1:cols + 1]
    pairs = [(_rand(rows, cols), wide[:, 8:]), (one.expand(rows, cols), wide[:, :cols]),
             (wide[:, 8:], one.expand(rows, cols)), (over, odd), (odd, over)]
    for x, r in pairs:
        s, y = add_rms_norm(x, r, EPS)
        want, rstd = rms_norm_fwd(x + r, EPS)
        _same(s, x + r)
        _same(y, want)
        s, got = add_rms_scales(x, r, EPS)
        _same(s, x + r)
        _same(got, rstd)


def test_values_at_the_ends(path):
    x, r = _rand(6, 64), _rand(6, 64, seed=1)
    x[0, 3], x[1, 0], r[1, 0], x[2, 5] = float("inf"), float("inf"), -float("inf"), float("nan")
    x[3], r[3] = 3.3e38, 3.3e38
    x[4], r[4] = 0, 0
    s, y = add_rms_norm(x, r, EPS)
    _same(s, x + r)
    _same(y, rms_norm(x + r, EPS))
    empty = _rand(0, 64)
    s, y = add_rms_norm(empty, empty, EPS)
    assert s.shape == y.shape == (0, 64)


@pytest.mark.parametrize("rows", [1, 100, 129, 300])
def test_scaled_projection(path, rows):
    x, r, w = _rand(rows, 256), _rand(rows, 256, seed=1), _rand(512, 256, seed=2)
    s, rstd = add_rms_scales(x, r, EPS)
    _same(rms_scaled_swiglu(s, w, rstd, EPS), rms_norm_swiglu(x + r, w, EPS))


@pytest.mark.parametrize("rows", [1, 64, 100, 128, 129])
def test_scaled_projection_takes_the_given_scales(path, rows):
    """Scales that are not those of x are applied as given and not written, for few rows as for
    many. Bound per element as in the projection tests: one bf16 rounding plus fp32 accumulation."""
    x, w = _rand(rows, 256), _rand(512, 256, seed=2)
    _, rstd = add_rms_scales(x, torch.zeros_like(x), EPS)
    before = rstd.clone()
    for factor in (0.125, -2.0):
        got = rms_scaled_swiglu(x, w, factor * rstd, EPS)
        y = (x.double() * rstd.double().unsqueeze(1) * factor) @ w.double().t()
        gate, up = y.chunk(2, -1)
        want = gate * torch.sigmoid(gate) * up
        size = x.double().abs() * rstd.double().unsqueeze(1).abs() * abs(factor) @ w.double().abs().t()
        sg, su = size.chunk(2, -1)
        s = torch.sigmoid(gate)
        bound = 1.02 * 2.0 ** -8 * want.abs() + 2.0 ** -18 * ((s * (1 + gate * (1 - s)) * up).abs() * sg
                                                             + (gate * s).abs() * su) + 1e-12
        assert ((got.double() - want).abs() <= bound).all()
    assert torch.equal(rstd, before)


@pytest.mark.parametrize("fused_gemm", [False, True])
def test_stack(fused_gemm):
    cfg = HRMStackConfig(hidden_size=256, num_heads=2, layers_per_module=2, H_cycles=1, L_cycles=2, max_seq_len=256,
                         fused_elementwise=True, fused_gemm=fused_gemm)
    net = HRMStack(cfg).init_weights(3).to(torch.bfloat16).to(DEV)
    prefix, causal, T = [20, 0, 64], [30, 50, 36], 208
    info = {}
    for part in metadata_tensors(prefix, causal, T, DEV):
        info.update(part)
    pos = packed_position_ids(prefix, causal, T, DEV)
    x = _rand(T, 256)
    attn = FusedLayer(fused_attention_layer)
    with torch.no_grad():
        fused = net(x, pos, attn, info)
        seen = []
        for m in (net.H, net.L):
            m.layers[0].register_forward_hook(lambda mod, args, out: seen.append(out.shape))
        separate = net(x, pos, attn, info)
    assert len(seen) == 3
    _same(fused, separate)
