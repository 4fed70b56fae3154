"""GPU: the projection GEMM where its tiling can go wrong: few rows, 128- and 256-row
tiles, one K stage, an odd number of stages, one W tile, tile counts below and off the
multiples of 8 and of the CUs, strided rows of x, against float64.

Bound per element as in the other projection tests: one bf16 rounding of the result plus
fp32 accumulation over the summed terms (1.02 * 2^-8 |ref| + 2^-18 size)."""
import pytest
import torch

from prefixlm.norm_mlp import proj_gemm

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
EPS = 1e-6


@pytest.mark.parametrize("swiglu", [True, False])
@pytest.mark.parametrize("M,K,N", [(1, 64, 256), (31, 192, 512), (33, 2048, 512), (64, 1280, 256), (65, 320, 768),
                                   (128, 1024, 512), (129, 64, 256), (257, 192, 512), (700, 128, 2304),
                                   (2300, 320, 2816), (5000, 64, 4096)])
def test_proj_gemm_tiles(M, K, N, swiglu):
    g = torch.Generator().manual_seed(M + K + N)
    x = torch.randn(M, K + 8, generator=g).to(torch.bfloat16).to(DEV)[:, :K]
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(DEV)
    for norm in (True, False):
        y = proj_gemm(x, w, swiglu, norm, EPS).double()
        xd, wd = x.double(), w.double()
        r = torch.rsqrt(xd.square().mean(-1, keepdim=True) + EPS) if norm else torch.ones(M, 1, device=DEV).double()
        ref, size = (xd * r) @ wd.t(), r * (xd.abs() @ wd.abs().t())
        if swiglu:
            gate, up = ref.chunk(2, -1)
            sg, su = size.chunk(2, -1)
            s = torch.sigmoid(gate)
            size = (s * (1 + gate * (1 - s)) * up).abs() * sg + (gate * s).abs() * su
            ref = gate * s * up
        bound = 1.02 * 2.0 ** -8 * ref.abs() + 2.0 ** -18 * size + 1e-12
        worst = ((y - ref).abs() / bound).max().item()
        assert worst <= 1.0, (norm, worst)


@pytest.mark.parametrize("M,K,N", [(3778, 2048, 11264), (1537, 128, 8192), (1150, 2048, 16384)])
def test_repeats_over_several_tiles_per_workgroup(M, K, N):
    """A workgroup's stages of successive tiles share two buffers: every pass gives the same bits."""
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(DEV)
    first = proj_gemm(x, w, True, True, EPS)
    assert all(torch.equal(proj_gemm(x, w, True, True, EPS), first) for _ in range(40))
