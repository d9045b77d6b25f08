"""Norm bounds whose V A products run on 16-column workgroups (csrc/nlb.hip, vmm_strip_kernel): matrices read from their
upper triangle, and launches of few fully stored ones, at the edges of the kernel's column blocks and k chunks."""
import pytest
import torch

from oracle.psgd_oracle import norm_lower_bound
from psgd_pro_amd import _lib as L

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _bound(fn, mats, Vs, sign, *extra):
    n, outs = mats[0].shape[0], [torch.empty((), device=DEV) for _ in mats]
    L.call_ws(fn, n, sign, len(mats), L.ptrs(mats), mats[0].stride(0), *extra, L.ptrs(Vs), L.ptrs(outs),
              ws=L.Workspace(), device=mats[0].device, stream=L.stream_of(mats[0]))
    return [float(o) for o in outs]


# k chunks hold 512 fp32 or 1024 bf16; n 4 and 8 are less than one column block, 509 has no 16-byte rows (the split-K
# route), 516 and 1032 end a chunk after 4 and 8, 1040 is a whole number of blocks
@pytest.mark.parametrize("n", [4, 8, 16, 509, 512, 516, 1032, 1040])
@pytest.mark.parametrize("sign", [1, -1])
def test_bound_by_column_strips(n, sign):
    """Against float64: fp32 sums of n products and five roundings per pass leave far less than 1e-5 of the norms here
    (sqrt(n) 2^-24 is 2e-6); bf16 storage rounds each of the iteration's vectors by up to 2^-8 (rel 2e-2)."""
    g = torch.Generator().manual_seed(n)
    mats, Vs = [], []
    for b in range(2):
        X = torch.randn(n, n + 8, generator=g)
        S = X @ X.T if sign > 0 else X[:, :n] - X[:, :n].T
        mats.append(S / n)
        Vs.append(torch.randn(32, n, generator=g))
    lib, dv = L.lib(), [v.to(DEV) for v in Vs]
    ref = [float(norm_lower_bound(M.double(), V.double(), skew=sign < 0)) for M, V in zip(mats, Vs)]
    wide = []  # a row stride over n, and NaN wherever only the other triangle's reader may look
    for M in mats:
        W = torch.full((n, n + 4), float("nan"), device=DEV)
        W[:, :n] = torch.where(torch.ones(n, n).triu().bool(), M, torch.tensor(float("nan"))).to(DEV)
        wide.append(W)
    tri = _bound(lib.psgdk_norm_lower_bound, wide, dv, sign)
    full = _bound(lib.psgdk_norm_lower_bound_full, [M.to(DEV) for M in mats], dv, sign, 0)
    b16 = [M.to(DEV).bfloat16() for M in mats]
    low = _bound(lib.psgdk_norm_lower_bound_full, b16, dv, sign, 1)
    for r, t, f, q in zip(ref, tri, full, low):
        assert t == pytest.approx(r, rel=1e-5) and f == pytest.approx(r, rel=1e-5)
        assert q == pytest.approx(r, rel=2e-2)
