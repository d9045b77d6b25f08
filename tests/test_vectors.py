"""Weights with one diagonal factor and nothing else: update and application in one launch each (csrc/elem.hip,
vec_update_kernel and vec_apply_kernel) up to 16384 elements, a launch per stage above."""
import ctypes

import pytest
import torch

from psgd_pro_amd import _lib as L
from tests.test_gpu_parity import assert_fp32, run_pair

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("sizes", [(2, 63), (1023, 1024, 1025), (1, 1531, 16384), (16385,)])
@pytest.mark.parametrize("gdt", [torch.float32, torch.bfloat16])
def test_vectors_with_a_diagonal_factor(sizes, gdt):
    """Against the float64 oracle at the fp32 bar, sizes around the workgroup's 1024 threads and the one-launch limit, as
    columns and as rows; equal sizes share a launch."""
    shapes = [s for n in sizes for s in ((n,), (n, 1), (1, n))]
    worst, base = run_pair(shapes, steps=3, skew=1.0, gdt=gdt, grad_eps=float(torch.finfo(gdt).eps))
    assert_fp32(worst, base)


@pytest.mark.parametrize("n", [5, 1500, 16384, 16390])
@pytest.mark.parametrize("over", ["G", "P"])
def test_preconditioned_gradient_in_place(n, over):
    """psgdk_kron2d_apply with pre_out and clipped_out over the fp32 gradient, or pre_out over P: pre = G P once, the
    weight's step from it. Five element-wise roundings of 2^-24, and of the RMS a sum of n squares in fp32: 1e-6."""
    g = torch.Generator().manual_seed(n)
    G, P, W = torch.randn(n, generator=g), torch.rand(n, generator=g) + 0.5, torch.zeros(n)
    dG, dP, dW = G.to(DEV), P.to(DEV), W.to(DEV)
    k = L.Kron2d()
    k.nb, k.prec, k.m, k.n, k.g_dtype, k.p_dtype = 1, L.PREC_F32, 1, n, L.F32, L.F32
    k.kind[0], k.kind[1] = L.FACTOR_NONE, L.FACTOR_DIAG
    k.G[0] = dG.data_ptr()
    k.P[1][0] = k.Q[1][0] = k.L[1][0] = dP.data_ptr()
    pre = dG if over == "G" else dP
    o = L.ApplyOpts(1e-3, 0.5, 1.0, 0)
    L.call_ws(L.lib().psgdk_kron2d_apply, k, o, L.ptrs([dW]), L.ptrs([pre]), L.ptrs([dG]) if over == "G" else None,
              ws=L.Workspace(), device=dG.device, stream=L.stream_of(dG))
    x = G.double() * P.double()
    rms = x.square().mean().sqrt()
    step = (x * (0.5 / rms) if rms > 0.5 else x).clamp(-1.0, 1.0)
    torch.testing.assert_close(dW.cpu().double(), -1e-3 * step, rtol=1e-6, atol=1e-10)
    torch.testing.assert_close(pre.cpu().double(), step if over == "G" else x, rtol=1e-6, atol=1e-10)
