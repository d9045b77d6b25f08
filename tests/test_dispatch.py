"""Which kernel the size rules give a product (psgdk_profile_start / _stop), on both sides of each line, and its result."""
import pytest
import torch

from psgd_pro_amd import _lib as L
from psgd_pro_amd import ops as K

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _launches(f):
    L.profile_start()
    out = f()
    return out, [r.kernel_id for r in L.profile_stop()]


@pytest.mark.parametrize("n,k,small", [(1920, 1032, True), (2048, 1024, True), (2048, 1032, False), (2432, 1024, True),
                                       (2560, 1024, False)])
def test_bf16_syrk(n, k, small):
    """The small-problem kernel below 128 128-tiles, up to k 1024 below 192 (2432: 190, 2560: 210). Its sums are the other
    kernels', in k order: fp32 sums of exact products, k 2^-24 of |X||X|^T at most."""
    X = torch.randn(n, k, generator=torch.Generator().manual_seed(n)).to(DEV).bfloat16()
    C, ids = _launches(lambda: K.syrk(X, False, L.OUT_MIRROR, True))
    assert [i // 1000 for i in ids] == [7 if small else 5]
    x = X.double()
    assert ((C - x @ x.T).abs() <= k * 2.0 ** -24 * (x.abs() @ x.abs().T)).all()


@pytest.mark.parametrize("m,n,k,wide", [(2048, 2048, 96, False), (2048, 2049, 96, True), (2944, 1500, 64, True)])
def test_fp32_product(m, n, k, wide):
    """128 x 256 tiles from 129 of them on (2048 x 2048: 128; 2048 x 2049: 144; 2944 x 1500: 138), else 64 x 64. k 2^-24 of
    |A||B| bounds both."""
    g = torch.Generator().manual_seed(m + n)
    A, B = torch.randn(m, k, generator=g).to(DEV), torch.randn(k, n, generator=g).to(DEV)
    C, ids = _launches(lambda: K.gemm(A, B, False, False, False))
    assert ids == [6000 + (0 if wide else 10)]
    a, b = A.double(), B.double()
    assert ((C - a @ b).abs() <= k * 2.0 ** -24 * (a.abs() @ b.abs())).all()
