"""GPU: the native host path of the public calls against the Python path they replace:
bitwise the same results and gradients, the same refusals, and the calls it hands back
(operands that need a copy, recorded and batched backwards, dispatch and function modes,
saved-tensor hooks that give back other tensors)."""
import pytest
import torch

from prefixlm import (_native, flash_attn_varlen_prefixlm, flash_attn_with_kvcache, fused_attention_layer, plan_inputs,
                      rms_norm, swiglu)
from prefixlm.hrm_stack import rotary_cos_sin
from prefixlm.norm_mlp import add_rms_scales, rms_norm_linear, rms_norm_swiglu, rms_scaled_swiglu
from prefixlm.synth import make_batch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.fixture(params=["native", "python"])
def path(request, monkeypatch):
    assert _native.calls() is not None, "the native host path is not built"
    if request.param == "python":
        monkeypatch.setattr(_native, "_module", None)
    return request.param


def _rand(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16).to(DEV)


def _both(fn, monkeypatch):
    """fn's results on the native and on the Python path."""
    assert _native.calls() is not None
    a = fn()
    with monkeypatch.context() as m:
        m.setattr(_native, "_module", None)
        b = fn()
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and torch.equal(x, y)


@pytest.mark.parametrize("plan", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("ints", [False, True])
def test_varlen_bitwise(plan, D, ints, monkeypatch):
    b = make_batch([10, 130, 0], [40, 7, 90], 300, 4, D, seed=5, device=DEV)
    info = dict(b.seq_info)
    if plan:
        info.update(plan_inputs(b.seq_tensors, b.seq_scalars, DEV))
    if ints:
        info = {k: int(x) if isinstance(x, torch.Tensor) and x.dim() == 0 else x for k, x in info.items()}

    def run():
        q, k = (t.clone().requires_grad_() for t in (b.q, b.k))
        v = torch.stack((b.v, b.v), 1)[:, 1].requires_grad_()        # a strided view
        out = flash_attn_varlen_prefixlm(q, k, v, False, **info)
        g = torch.autograd.grad(out, (q, k, v), b.dout, retain_graph=True)
        g2 = torch.autograd.grad(out.float().sum(), (q, k, v))       # an expanded gradient
        with torch.no_grad():
            o = flash_attn_varlen_prefixlm(q, k, v, True, **info)
        return out, *g, *g2, o
    _both(run, monkeypatch)


def test_layer_norm_activation_projection_bitwise(monkeypatch):
    T, H = 260, 2
    b = make_batch([60, 20], [100, 70], T, H, 128, seed=6, device=DEV, with_dout=False)
    cos, sin = rotary_cos_sin(torch.arange(T, device=DEV), 128, 10000.0, 1024)
    gq, dy = _rand(T, 4 * H, 128, seed=1), _rand(T, H, 128, seed=2)
    x, gu, w = _rand(7, 9, 256, seed=3), _rand(40, 512, seed=4), _rand(512, 256, seed=5)

    def run():
        g = gq.clone().requires_grad_()
        y = fused_attention_layer(g, cos, sin, False, **b.seq_info)
        xx, uu = x.clone().requires_grad_(), gu.clone().requires_grad_()
        n, a = rms_norm(xx, 1e-6), swiglu(uu)
        grads = torch.autograd.grad((y, n, a), (g, xx, uu), (dy, x, a.detach()))
        with torch.no_grad():
            return (y, n, a, *grads, rms_norm(x[:, ::2], 1e-5), swiglu(gu), rms_norm_linear(x, torch.nn.Parameter(w), 1e-6),
                    rms_norm_swiglu(x.view(63, 256)[:, :256], w, 1e-6))
    _both(run, monkeypatch)


@pytest.mark.parametrize("S", [1, 5])
def test_kvcache_bitwise_and_in_place(S, monkeypatch):
    B, H, Smax = 2, 3, 150
    q, k, v = (_rand(B, S, H, 128, seed=i) for i in range(3))
    caches = _rand(2, B, Smax, H, 128, seed=9)
    lens = torch.tensor([20, 140], dtype=torch.int32, device=DEV)

    def run():
        kc, vc = caches[0].clone(), caches[1].clone()
        before = kc._version, vc._version
        o = flash_attn_with_kvcache(q, kc, vc, k=k, v=v, cache_seqlens=lens, causal=True)
        assert (kc._version, vc._version) == tuple(n + 1 for n in before)
        o2 = flash_attn_with_kvcache(q, kc, vc, cache_seqlens=30)
        return o, kc, vc, o2
    _both(run, monkeypatch)


def test_refusals(path):
    b = make_batch([10], [40], 64, 2, 128, seed=5, device=DEV)
    with pytest.raises(TypeError):
        flash_attn_varlen_prefixlm(b.q.float(), b.k, b.v, False, **b.seq_info)
    with pytest.raises(ValueError):
        flash_attn_varlen_prefixlm(b.q, b.k[:32], b.v, False, **b.seq_info)
    with pytest.raises(AssertionError):
        flash_attn_varlen_prefixlm(b.q, b.k, b.v, False, **{**b.seq_info, "numseqs": torch.tensor(1, device=DEV)})
    with pytest.raises(RuntimeError, match="total_seqlen"):
        flash_attn_varlen_prefixlm(b.q, b.k, b.v, False, **{**b.seq_info, "total_seqlen": torch.tensor(65)})
    with pytest.raises(RuntimeError, match="multiple"):
        rms_norm(_rand(4, 12), 1e-6)
    with pytest.raises(ValueError):
        swiglu(_rand(4, 24))
    q = b.q.clone().requires_grad_()
    out = flash_attn_varlen_prefixlm(q, b.k, b.v, False, **b.seq_info)
    with torch.no_grad():
        q.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()


def test_recorded_backward_is_the_custom_op(path):
    """create_graph: the gradient carries a graph whose own backward is refused."""
    b = make_batch([10], [40], 64, 2, 128, seed=5, device=DEV)
    q = b.q.clone().requires_grad_()
    out = flash_attn_varlen_prefixlm(q, b.k, b.v, False, **b.seq_info)
    (g,) = torch.autograd.grad(out, q, b.dout.clone().requires_grad_(), create_graph=True)
    assert g.requires_grad
    with pytest.raises(RuntimeError):
        g.float().sum().backward()


def test_hooks_checkpoint_and_other_streams(path):
    b = make_batch([10, 30], [40, 20], 128, 2, 128, seed=5, device=DEV)
    q = b.q.clone().requires_grad_()
    f = lambda q: flash_attn_varlen_prefixlm(q, b.k, b.v, False, **b.seq_info)  # noqa: E731
    want, = torch.autograd.grad(f(q), q, b.dout)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t.clone(), lambda t: t):
        out = f(q)
    assert torch.equal(torch.autograd.grad(out, q, b.dout)[0], want) and len(packed) >= 7
    out = torch.utils.checkpoint.checkpoint(f, q, use_reentrant=False)
    assert torch.equal(torch.autograd.grad(out, q, b.dout)[0], want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        out = f(q)
        got, = torch.autograd.grad(out, q, b.dout)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    with torch.inference_mode():
        assert torch.equal(f(q.detach()), out.detach())


def _wide(t):
    """t's values in rows of twice the length."""
    return torch.cat((t, t), -1)[..., :t.shape[-1]]


def _shifted(t):
    """t's values one element off its alignment."""
    return torch.cat((t.flatten()[:1], t.flatten()))[1:].view(t.shape)


# which saved tensor (by dtype and number of dimensions, the n-th such), what a hook gives back for
# it, and what the backward then does: the same gradients, or this error
HOOKS = {
    "q_fp32": ("varlen", (torch.bfloat16, 3, 0), lambda t: t.float(), TypeError),
    "k_cpu": ("varlen", (torch.bfloat16, 3, 1), lambda t: t.cpu(), ValueError),
    "v_off_alignment": ("varlen", (torch.bfloat16, 3, 2), _shifted, RuntimeError),
    "out_wide": ("varlen", (torch.bfloat16, 3, 3), _wide, None),
    "lse_transposed": ("varlen", (torch.float32, 2, 0), lambda t: t.t().contiguous().t(), None),
    "lse_double": ("varlen", (torch.float32, 2, 0), lambda t: t.double(), ValueError),
    "residual_strided": ("varlen", (torch.int8, 3, 0), lambda t: torch.stack((t, t), -1)[..., 0], None),
    "residual_short": ("varlen", (torch.int8, 3, 0), lambda t: t[:-1], ValueError),
    "q_amax_short": ("varlen", (torch.float32, 1, 0), lambda t: t[:-1], ValueError),
    "q_amax_strided": ("varlen", (torch.float32, 1, 0), lambda t: torch.stack((t, t), -1)[:, 0], None),
    "lens_long": ("varlen", (torch.int32, 1, 0), lambda t: t.long(), None),
    "plan_off_alignment": ("varlen", (torch.int32, 1, 3), _shifted, None),
    "scalar_gpu": ("varlen", (torch.int64, 0, 0), lambda t: t.to(DEV), AssertionError),
    "gqkv_wide": ("layer", (torch.bfloat16, 3, 0), _wide, None),
    "gqkv_fp32": ("layer", (torch.bfloat16, 3, 0), lambda t: t.float(), ValueError),
    "cos_wide": ("layer", (torch.float32, 2, 1), lambda t: torch.cat((t, t), -1)[:, :128].contiguous(), None),
    "sin_short": ("layer", (torch.float32, 2, 2), lambda t: t[:-1], ValueError),
    "rstd_strided": ("rms_norm", (torch.float32, 1, 0), lambda t: torch.stack((t, t), -1)[:, 0], None),
    "rstd_short": ("rms_norm", (torch.float32, 1, 0), lambda t: t[:-1], ValueError),
    "gu_fp32": ("swiglu", (torch.bfloat16, 2, 0), lambda t: t.float(), ValueError),
}


@pytest.mark.parametrize("name", HOOKS)
def test_hooks_that_give_back_other_tensors(name, path):
    """A saved-tensors hook may change what the backward gets: the operands are checked again, and
    copied or refused as the custom ops do."""
    print(f"[case] hook {name} {path}", flush=True)
    call, which, change, error = HOOKS[name]
    T, H = 300, 2
    b = make_batch([60, 20], [100, 70], T, H, 128, seed=6, device=DEV)
    info = {**b.seq_info, **plan_inputs(b.seq_tensors, b.seq_scalars, DEV)}
    cos, sin = rotary_cos_sin(torch.arange(T, device=DEV), 128, 10000.0, 1024)
    x, f, dy = {
        "varlen": (b.q, lambda q: flash_attn_varlen_prefixlm(q, b.k, b.v, False, **info), b.dout),
        "layer": (_rand(T, 4 * H, 128, seed=1), lambda g: fused_attention_layer(g, cos, sin, False, **info), b.dout),
        "rms_norm": (_rand(40, 256, seed=1), lambda x: rms_norm(x, 1e-6), _rand(40, 256, seed=2)),
        "swiglu": (_rand(40, 512, seed=1), swiglu, _rand(40, 256, seed=2)),
    }[call]
    x = x.clone().requires_grad_()
    want, = torch.autograd.grad(f(x), x, dy)
    seen, given = {}, []

    def pack(t):
        key = (t.dtype, t.dim())
        n = seen.get(key, 0)
        seen[key] = n + 1
        return t, (*key, n) == which

    def unpack(p):
        given.append(p[1])
        return change(p[0].detach()) if p[1] else p[0]

    with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
        y = f(x)
    if error is None:
        assert torch.equal(torch.autograd.grad(y, x, dy)[0], want)
    else:
        with pytest.raises(error):
            torch.autograd.grad(y, x, dy)
    assert given.count(True) == 1


def test_the_profiler_sees_the_calls(path):
    """torch.profiler shows each call and each backward under its operator's name, once, with shapes."""
    b = make_batch([10, 30], [40, 20], 128, 2, 128, seed=5, device=DEV)
    cos, sin = rotary_cos_sin(torch.arange(128, device=DEV), 128, 10000.0, 1024)
    q, g = b.q.clone().requires_grad_(), _rand(128, 8, 128).requires_grad_()
    x, gu, w = _rand(40, 256).requires_grad_(), _rand(40, 512, seed=1).requires_grad_(), _rand(512, 256, seed=2)
    kq, cache = _rand(1, 1, 2, 128), _rand(2, 1, 64, 2, 128)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], record_shapes=True) as prof:
        torch.autograd.grad(flash_attn_varlen_prefixlm(q, b.k, b.v, False, **b.seq_info), q, b.dout)
        torch.autograd.grad(fused_attention_layer(g, cos, sin, False, **b.seq_info), g, b.dout)
        torch.autograd.grad(rms_norm(x, 1e-6), x, _rand(40, 256, seed=3))
        torch.autograd.grad(swiglu(gu), gu, _rand(40, 256, seed=3))
        with torch.no_grad():
            rms_norm_linear(x, w, 1e-6)
            s, rstd = add_rms_scales(x, x, 1e-6)
            rms_scaled_swiglu(s, w, rstd, 1e-6)
            flash_attn_with_kvcache(kq, cache[0], cache[1], k=kq, v=kq, cache_seqlens=0)
    seen = {e.key: e for e in prof.key_averages(group_by_input_shape=True) if e.key.startswith("prefixlm::")}
    assert {k: e.count for k, e in seen.items()} == {f"prefixlm::{n}": 1 for n in (
        "varlen_fwd", "varlen_bwd", "attn_layer_fwd", "attn_layer_bwd", "rms_norm_fwd", "rms_norm_bwd", "swiglu_fwd",
        "swiglu_bwd", "proj_gemm", "add_rmsnorm", "proj_gemm_scaled", "kvcache_attn")}
    assert seen["prefixlm::varlen_fwd"].input_shapes[0] == [128, 2, 128]


def _call(name, plan):
    """(leaf input, call, output gradient) of one differentiable call."""
    T, H = 300, 2
    b = make_batch([60, 20], [100, 70], T, H, 128, seed=6, device=DEV)
    info = {**b.seq_info, **(plan_inputs(b.seq_tensors, b.seq_scalars, DEV) if plan else {})}
    cos, sin = rotary_cos_sin(torch.arange(T, device=DEV), 128, 10000.0, 1024)
    x, f, dy = {
        "varlen": (b.q, lambda q: flash_attn_varlen_prefixlm(q, b.k, b.v, False, **info), b.dout),
        "layer": (_rand(T, 4 * H, 128, seed=1), lambda g: fused_attention_layer(g, cos, sin, False, **info), b.dout),
        "rms_norm": (_rand(40, 256, seed=1), lambda x: rms_norm(x, 1e-6), _rand(40, 256, seed=2)),
        "swiglu": (_rand(40, 512, seed=1), swiglu, _rand(40, 256, seed=2)),
    }[name]
    return x.clone().requires_grad_(), f, dy


CALLS = [("varlen", False), ("varlen", True), ("layer", False), ("layer", True), ("rms_norm", False), ("swiglu", False)]


@pytest.mark.parametrize("name,plan", CALLS)
def test_recorded_backwards_give_the_same_gradient(name, plan):
    """create_graph takes the custom op, whose arguments the native node lines up by hand."""
    assert _native.calls() is not None
    x, f, dy = _call(name, plan)
    want, = torch.autograd.grad(f(x), x, dy)
    got, = torch.autograd.grad(f(x), x, dy.clone().requires_grad_(), create_graph=True)
    assert got.requires_grad and torch.equal(got.detach(), want)


@pytest.mark.parametrize("name,plan", CALLS)
def test_modes_see_the_operators(name, plan):
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    assert _native.calls() is not None
    seen = []

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    x, f, dy = _call(name, plan)
    y = f(x)
    want, = torch.autograd.grad(y, x, dy)
    for mode in (Dispatch, Function):
        with mode():
            z = f(x)
            got, = torch.autograd.grad(z, x, dy)
        assert torch.equal(z, y) and torch.equal(got, want)
    assert sum(op.startswith("prefixlm.") for op in seen) == 2


@pytest.mark.parametrize("name,plan", CALLS)
def test_batched_gradients_as_on_the_python_path(name, plan, monkeypatch):
    def run():
        x, f, dy = _call(name, plan)
        try:
            return torch.autograd.grad(f(x), x, torch.stack((dy, 2 * dy)), is_grads_batched=True)[0]
        except Exception as e:
            return type(e)
    assert _native.calls() is not None
    a = run()
    with monkeypatch.context() as m:
        m.setattr(_native, "_module", None)
        b = run()
    assert torch.equal(a, b) if isinstance(a, torch.Tensor) and isinstance(b, torch.Tensor) else a is b
