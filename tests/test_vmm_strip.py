"""Norm bounds of one launch (csrc/nlb.hip, nlb_small_kernel) and those whose V A products run on 16-column workgroups
(vmm_strip_kernel): matrices read from their upper triangle, launches of few fully stored ones and rows at odd addresses,
at the edges of the kernels' sides, column blocks and k chunks; and row norms and products of groups of triangles."""
import pytest
import torch

from oracle.psgd_oracle import norm_lower_bound
from psgd_pro_amd import _lib as L
from tests.metrics import rel_err_norm

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _bound(fn, mats, Vs, sign, *extra):
    n, outs = mats[0].shape[0], [torch.empty((), device=DEV) for _ in mats]
    L.call_ws(fn, n, sign, len(mats), L.ptrs(mats), mats[0].stride(0), *extra, L.ptrs(Vs), L.ptrs(outs),
              ws=L.Workspace(), device=mats[0].device, stream=L.stream_of(mats[0]))
    return [float(o) for o in outs]


# One launch: up to 128 (fp32), 256 (bf16, and fp32 rows that are not 16-byte aligned). Strips: k chunks hold 512 fp32 or
# 1024 bf16; 257, 509 and 1030 end in a partial piece, 516 and 1032 end a chunk after 4 and 8.
@pytest.mark.parametrize("n", [1, 3, 16, 127, 128, 129, 132, 254, 256, 257, 264, 509, 512, 516, 1030, 1032, 1040])
@pytest.mark.parametrize("sign", [1, -1])
def test_bounds_at_the_edges(n, sign):
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
    nan, wide, up = float("nan"), [], []  # a row stride over n; NaN wherever the bound must not look
    for M in mats:
        wide.append(torch.full((n, n + 4), nan, device=DEV))
        wide[-1][:, :n] = M.to(DEV)
        up.append(torch.where(torch.ones(n, n + 4, device=DEV).triu().bool(), wide[-1], nan))
    tri = _bound(lib.psgdk_norm_lower_bound, up, dv, sign)
    full = _bound(lib.psgdk_norm_lower_bound_full, wide, dv, sign, 0)
    b16 = [M.to(DEV).bfloat16() for M in mats]
    low = _bound(lib.psgdk_norm_lower_bound_full, b16, dv, sign, 1)
    for r, t, f, q in zip(ref, tri, full, low):
        assert t == pytest.approx(r, rel=1e-5) and f == pytest.approx(r, rel=1e-5)
        assert q == pytest.approx(r, rel=2e-2)


@pytest.mark.parametrize("nb", [3, 16])
@pytest.mark.parametrize("n", [130, 129])
def test_row_norms_of_several_matrices(nb, n):
    """psgdk_tri_rownorm2 on a group: every matrix's squared row norms and largest element are its own (scales a factor of
    two apart), and every output is written. rn2: n squares summed in fp32, 1e-6 as for one matrix."""
    g = torch.Generator().manual_seed(n + nb)
    X = [torch.randn(n, n, generator=g) * 2.0 ** b for b in range(nb)]
    mats = [(x + x.T) for x in X]
    up = [torch.where(torch.ones(n, n).triu().bool(), m, torch.tensor(float("nan"))).to(DEV) for m in mats]
    rn2 = [torch.full((n,), float("nan"), device=DEV) for _ in mats]
    amax = [torch.full((), float("nan"), device=DEV) for _ in mats]
    L.call_ws(L.lib().psgdk_tri_rownorm2, n, 1, nb, L.ptrs(up), n, L.ptrs(rn2), L.ptrs(amax), ws=L.Workspace(),
              device=up[0].device, stream=L.stream_of(up[0]))
    for m, r, a in zip(mats, rn2, amax):
        assert float(a) == float(m.abs().max())
        assert rel_err_norm(r, m.double().square().sum(1)) < 1e-6


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("n", [7, 130, 513, 1028])
@pytest.mark.parametrize("sign", [1, -1])
def test_products_of_triangles(n, sign, in_place):
    """psgdk_tri_vmm on a group of three, into outputs of its own or over V: V A_sym, NaN below the triangles. Sums of n
    products in fp32 stay below 1e-6 normwise, as for one matrix."""
    g = torch.Generator().manual_seed(n)
    S = [torch.randn(n, n, generator=g) for _ in range(3)]
    S = [s + s.T if sign > 0 else s - s.T for s in S]
    V = [torch.randn(32, n, generator=g) for _ in S]
    up = [torch.where(torch.ones(n, n).triu().bool(), s, torch.tensor(float("nan"))).to(DEV) for s in S]
    dv = [v.to(DEV) for v in V]
    W = dv if in_place else [torch.empty_like(v) for v in dv]
    L.call_ws(L.lib().psgdk_tri_vmm, n, sign, 3, L.ptrs(dv), L.ptrs(up), n, L.ptrs(W), ws=L.Workspace(),
              device=up[0].device, stream=L.stream_of(up[0]))
    for w, v, s in zip(W, V, S):
        assert rel_err_norm(w, v.double() @ s.double()) < 1e-6


@pytest.mark.parametrize("lda", [2 ** 20 - 4, 2 ** 20])
def test_triangles_past_two_gib(lda):
    """Rows so far apart that the matrix spans 2.3 GiB: up to 2^20 the 16-column kernel, whose offsets are relative to a
    chunk's first row, from there on split products of the converting engine. Errors as in the tests above."""
    n = 600
    g = torch.Generator().manual_seed(n)
    X = torch.randn(n, n + 8, generator=g)
    S, V = X @ X.T / n, torch.randn(32, n, generator=g)
    wide = torch.full((n, lda), float("nan"), device=DEV)
    wide[:, :n] = torch.where(torch.ones(n, n).triu().bool(), S, torch.tensor(float("nan"))).to(DEV)
    dv, W = V.to(DEV), torch.empty(32, n, device=DEV)
    r = float(norm_lower_bound(S.double(), V.double(), skew=False))
    assert _bound(L.lib().psgdk_norm_lower_bound, [wide], [dv], 1) == [pytest.approx(r, rel=1e-5)]
    L.call_ws(L.lib().psgdk_tri_vmm, n, 1, 1, L.ptrs([dv]), L.ptrs([wide]), lda, L.ptrs([W]), ws=L.Workspace(),
              device=wide.device, stream=L.stream_of(wide))
    assert rel_err_norm(W, V.double() @ S.double()) < 1e-6


def test_products_of_triangles_sum_in_short_chains():
    """P = 0.5 I + A A^T / 2 at n 4096: V P within 2e-7 of float64 normwise. Every rounding after the diagonal's term is of
    its size, uniform in 2^-24 of it or less: the split products' few come to 9e-8 (measured), fp32 MFMA chains of 32 k to
    1.5e-7, one over 512 k to 4.2e-7."""
    n = 4096
    g = torch.Generator().manual_seed(1)
    a = torch.randn(n, n, generator=g).to(DEV) / n ** 0.5
    P = 0.5 * (a @ a.T)
    P.diagonal().add_(0.5)
    P = 0.5 * (P + P.T)
    V = torch.randn(32, n, generator=g).to(DEV)
    W = torch.empty_like(V)
    L.call_ws(L.lib().psgdk_tri_vmm, n, 1, 1, L.ptrs([V]), L.ptrs([P]), n, L.ptrs([W]), ws=L.Workspace(), device=P.device,
              stream=L.stream_of(P))
    assert rel_err_norm(W, V.double() @ P.double()) < 2e-7
