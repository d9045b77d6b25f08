"""The converting MFMA engine (csrc/gemm_cv.hip): every tile configuration at the edges of its tiles, in both precisions
and every layout it reads, against float64."""
import ctypes

import pytest
import torch

from psgd_pro_amd import _lib as L
from psgd_pro_amd import ops as K
from tests.metrics import rel_err_norm
from tests.test_gpu_parity import assert_fp32, run_pair

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(params=[-1, 0, 1, 2, 3])
def engine(request):
    """The engine alone (option 10 = 0: no small-problem kernels), in one tile configuration (option 13)."""
    hip = L.lib()
    L.check(hip.psgdk_set_option(13, request.param))
    L.check(hip.psgdk_set_option(10, 0))
    yield hip
    L.check(hip.psgdk_set_option(13, -1))
    L.check(hip.psgdk_set_option(10, 128))


def _rnd(rows, cols, seed):
    # a view one column into a wider matrix: rows that no 16-byte access is aligned to
    x = torch.randn(rows, cols + 3, generator=torch.Generator().manual_seed(seed))
    return x.to(DEV)[:, 1:1 + cols]


def _check(C, A, B, bf16, what):
    """|C - A B| <= c |A| |B| elementwise. fp32: the split drops under 2^-23 of each product, and a product takes part in
    at most 6 roundings per 16 k of its 128-k block (a truncation counting two) and one per block, each 2^-24 of sums
    that |A| |B| bounds. bf16: two operand
    roundings of 2^-8 besides. (The last term: results below the smallest normal.) And fp32 normwise 1e-6, five times the
    measured 2e-7: without a third plane, or without m m', random operands are 2e-6 to 6e-6 off."""
    A, B = A.double().cpu(), B.double().cpu()
    u = 2.0 ** -24
    c = u * (2 + 2 * 6 * 8 + A.shape[1] / 64 + 4) + (2.0 ** -7 + 2.0 ** -16 if bf16 else 0.0)
    bad = (C.double().cpu() - A @ B).abs() > c * (A.abs() @ B.abs()) + 2.0 ** -126
    assert not bad.any(), (what, int(bad.sum()))
    if not bf16 and (A @ B).norm() > 2.0 ** -100:
        assert rel_err_norm(C, A @ B) < 1e-6, (what, rel_err_norm(C, A @ B))


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (31, 63, 33), (64, 64, 64), (65, 129, 127), (129, 257, 130),
                                   (200, 500, 321)])
@pytest.mark.parametrize("bf16", [False, True])
def test_converting_engine(engine, m, n, k, bf16):
    for ta in (False, True):
        for tb in (False, True):
            A, B = _rnd(*((k, m) if ta else (m, k)), seed=m + k), _rnd(*((n, k) if tb else (k, n)), seed=n + k)
            for dt in (torch.float32, torch.bfloat16):
                a, b = A.to(dt), B.to(dt)
                C = K.gemm(a, b, ta, tb, bf16)
                _check(C, a.T if ta else a, b.T if tb else b, bf16, (ta, tb, dt))
    A, S = _rnd(m, k, 1), _rnd(m, m, 2)
    _check(K.symm(S, A, 1, bf16), torch.triu(S) + torch.triu(S, 1).T, A, bf16, "symm")
    _check(K.symm_right(A.T, S, -1, bf16), A.T, torch.triu(S, 1) - torch.triu(S, 1).T, bf16, "symm_right")
    _check(K.trmm(S, A, bf16), torch.triu(S), A, bf16, "trmm")
    for trans in (False, True):
        x = A.T if trans else A
        full = K.syrk(A, trans, L.OUT_MIRROR, bf16)
        assert torch.equal(full, full.T)
        _check(full, x, x.T, bf16, "syrk")
        i, j = torch.triu_indices(len(x), len(x))
        assert torch.equal(K.syrk(A, trans, L.OUT_PACKED, bf16), full[i, j])
        assert torch.equal(torch.triu(K.syrk(A, trans, L.OUT_UPPER, bf16)), torch.triu(full))
    if bf16:
        return
    # rows holding an infinity, a NaN, a value over the bfloat16 range or under its normals: as on fp32 MFMAs
    A, B = _rnd(m, k, 3).clone(), _rnd(k, n, 4)
    for i, v in enumerate((float("inf"), float("nan"), 3.4e38, 1e-41)):
        A[i * 9 % m, i % k] = v
    C = K.gemm(A, B, False, False, False)
    L.check(engine.psgdk_set_option(8, 0))
    R = K.gemm(A, B, False, False, False)
    L.check(engine.psgdk_set_option(8, 1))
    fin = torch.isfinite(R)
    assert torch.equal(fin, torch.isfinite(C)) and torch.equal(torch.isnan(R), torch.isnan(C))
    assert torch.equal(R[torch.isinf(R)], C[torch.isinf(R)])
    ok = fin.all(1)
    _check(C[ok], A[ok], B, False, "finite rows")


@pytest.mark.parametrize("m,n,k", [(2, 2, 2), (31, 63, 33), (65, 129, 127), (129, 257, 130), (200, 500, 321)])
def test_operands_stored_in_bf16(engine, m, n, k):
    """Products of the bf16 precision with one or both operands in bf16, at rows of even stride (read four elements at a
    time, whatever the rows' length) and of odd stride."""
    for dA, dB in ((torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16)):
        for pad in (3, 4):
            def put(x, dt):
                y = torch.full((x.shape[0], x.shape[1] // 2 * 2 + pad), float("nan"), dtype=dt, device=DEV)
                y[:, 2:2 + x.shape[1]] = x
                return y[:, 2:2 + x.shape[1]]
            for ta in (False, True):
                for tb in (False, True):
                    a = put(_rnd(*((k, m) if ta else (m, k)), seed=m), dA)
                    b = put(_rnd(*((n, k) if tb else (k, n)), seed=n), dB)
                    _check(K.gemm(a, b, ta, tb, True), a.T if ta else a, b.T if tb else b, True, (ta, tb, dA, dB, pad))


@pytest.mark.parametrize("k", [512, 1280, 1288, 3072])
@pytest.mark.parametrize("sign", [False, True])
def test_split_products_are_no_further_off_than_fp32_mfmas(engine, k, sign):
    """Against float64, the fp32 products by splits are as close as fp32 MFMA chains of 128 k (option 8 = 0, 64 x 64
    tiles) for operands of random and of one sign: there the sum of the blocks bounds both, which the splits must not cut
    shorter for long k. One percent for the two samples of the same rounding."""
    g = torch.Generator().manual_seed(k)
    A, B = torch.randn(256, k, generator=g), torch.randn(k, 512, generator=g)
    if sign:
        A, B = A.abs(), B.abs()
    a, b, R = A.to(DEV), B.to(DEV), A.double() @ B.double()
    C = K.gemm(a, b, False, False, False)
    cfg = ctypes.c_int(0)
    L.check(engine.psgdk_get_option(13, ctypes.byref(cfg)))
    L.check(engine.psgdk_set_option(13, 1))
    L.check(engine.psgdk_set_option(8, 0))
    ref = rel_err_norm(K.gemm(a, b, False, False, False), R)
    L.check(engine.psgdk_set_option(8, 1))
    L.check(engine.psgdk_set_option(13, cfg.value))
    assert rel_err_norm(C, R) < 1.01 * ref, (rel_err_norm(C, R), ref)


def test_operands_far_from_one(engine):
    """fp32 products keep fp32's accuracy over its range: operands down to its subnormals (whole matrices, and single rows
    and columns of ordinary ones), sums beyond what the scaled split can hold, and operands beyond it."""
    m, n, k = 70, 130, 96
    A, B = _rnd(m, k, 5), _rnd(k, n, 6)
    for ea, eb in ((-100, 90), (-113, 100), (-121, 100), (-126, 110), (-136, 100), (100, -113), (90, -136), (60, 50),
                   (120, -30), (-126, 120)):
        a, b = torch.ldexp(A, torch.tensor(ea, device=DEV)), torch.ldexp(B, torch.tensor(eb, device=DEV))
        _check(K.gemm(a, b, False, False, False), a, b, False, (ea, eb))
        _check(K.symm_right(a.T, torch.ldexp(_rnd(m, m, 7), torch.tensor(eb, device=DEV)), -1, False), a.T,
               (lambda u: u - u.T)(torch.ldexp(torch.triu(_rnd(m, m, 7), 1), torch.tensor(eb, device=DEV))), False, "symm")
    rows = torch.tensor([-120 if i % 5 == 3 else -136 if i % 5 == 1 else 0 for i in range(m)], device=DEV)
    cols = torch.tensor([-119 if j % 7 == 2 else 0 for j in range(n)], device=DEV)
    a, b = torch.ldexp(A, rows[:, None]), torch.ldexp(B, cols[None])
    C = K.gemm(a, torch.ldexp(b, torch.tensor(40, device=DEV)), False, False, False)
    _check(C, a, torch.ldexp(b, torch.tensor(40, device=DEV)), False, "rows")


@pytest.mark.parametrize("cfg", [-1, 1, 3])
def test_gram_diagonal_keeps_its_small_squares(cfg):
    """X^T X for X near the identity: the small squares beside a diagonal entry's large one are not lost to its
    alignment, which would lower every entry by their sum."""
    n = 192
    X = (torch.eye(n) + 2.0 ** -13 * torch.randn(n, n, generator=torch.Generator().manual_seed(5))).to(DEV)
    L.check(L.lib().psgdk_set_option(13, cfg))
    try:
        C = K.syrk(X, True, L.OUT_MIRROR, False)
    finally:
        L.check(L.lib().psgdk_set_option(13, -1))
    d = C.diagonal().double() - X.double().square().sum(0)
    # one rounding of at most 2^-24 per entry and either sign (1 <= C_ii < 2), so a mean of n of them within 4 standard
    # deviations 2^-24 / sqrt(3 n); the seven squares lost would make it -7 * 2^-26
    assert d.mean().abs().item() < 4 * 2.0 ** -24 / (3 * n) ** 0.5, d.mean()


@pytest.mark.parametrize("m,n", [(1032, 1032), (24, 390), (129, 257)])
def test_application_in_every_configuration(engine, m, n):
    """P1 G P2, its sum of squares and the clipped update of two fp32 weights, from a workspace of exactly the queried size
    between guard bytes that stay as they are. Two products of up to 1032 terms, 2e-7 each, and six element-wise roundings
    of 2^-24: 1e-6 normwise leaves a factor of two."""
    g = torch.Generator().manual_seed(m + n)
    P = [[(lambda x: x @ x.T)(torch.randn(d, d, generator=g) / d ** 0.5 + torch.eye(d)) for d in (m, n)] for _ in range(2)]
    G = [torch.randn(m, n, generator=g) for _ in range(2)]
    W = [torch.randn(m, n, generator=g) for _ in range(2)]
    k = L.Kron2d()
    k.nb, k.prec, k.m, k.n, k.g_dtype, k.p_dtype = 2, L.PREC_F32, m, n, L.F32, L.F32
    k.kind[0] = k.kind[1] = L.FACTOR_DENSE
    dP, dG, dW = [[p.to(DEV) for p in ps] for ps in P], [x.to(DEV) for x in G], [x.to(DEV) for x in W]
    for b in range(2):
        k.G[b] = dG[b].data_ptr()
        for f in range(2):
            k.P[f][b] = k.Q[f][b] = k.L[f][b] = dP[b][f].data_ptr()
    pre = [torch.full((m, n), float("nan"), device=DEV) for _ in range(2)]
    o = L.ApplyOpts(1e-3, 0.5, 1.0, 0)
    args = (k, o, L.ptrs(dW), L.ptrs(pre), None)
    sz, st = ctypes.c_size_t(0), L.stream_of(dG[0])
    L.check(engine.psgdk_kron2d_apply(*args, None, ctypes.byref(sz), st))
    ws = torch.full((sz.value + 8192,), 0xA5, dtype=torch.uint8, device=DEV)
    L.check(engine.psgdk_kron2d_apply(*args, ctypes.c_void_p(ws.data_ptr() + 4096), ctypes.byref(sz), st))
    assert (ws[:4096] == 0xA5).all() and (ws[4096 + sz.value:] == 0xA5).all()
    for b in range(2):
        x = P[b][0].double() @ G[b].double() @ P[b][1].double()
        assert rel_err_norm(pre[b], x) < 1e-6
        rms = x.square().mean().sqrt()
        step = (x * (0.5 / rms) if rms > 0.5 else x).clamp(-1.0, 1.0)
        assert rel_err_norm(W[b].double() - dW[b].double().cpu(), 1e-3 * step) < 1e-4  # W - step rounds at 2^-24 of W


@pytest.mark.parametrize("cfg", [-1, 1, 3])
@pytest.mark.parametrize("n", [192, 1601, 3072])
@pytest.mark.parametrize("trans,dt", [(False, torch.float32), (True, torch.float32), (False, torch.bfloat16)])
def test_gram_diagonal_is_unbiased(n, trans, dt, cfg):
    """X X^T and X^T X for X near the identity, at sizes that take the 128 x 256 tiles otherwise: no entry of the diagonal
    loses the seven squares beside its large one. Without their own MFMA the mean is -2e-7 here; the roundings of n entries
    of either sign leave less than 2^-24 / 8."""
    X = (torch.eye(n) + 2.0 ** -10 * torch.randn(n, n, generator=torch.Generator().manual_seed(5))).to(DEV).to(dt)
    L.check(L.lib().psgdk_set_option(13, cfg))
    L.check(L.lib().psgdk_set_option(10, 0))
    try:
        C = K.syrk(X, trans, L.OUT_MIRROR, False)
    finally:
        L.check(L.lib().psgdk_set_option(13, -1))
        L.check(L.lib().psgdk_set_option(10, 128))
    x = X.double()
    d = C.diagonal().double() - x.square().sum(0 if trans else 1)
    assert d.mean().abs().item() < 2.0 ** -27, d.mean()


@pytest.mark.parametrize("r2", [False, True])
def test_steps_at_the_edges_of_tiles(engine, r2):
    """Whole fp32 steps against the float64 oracle at the fp32 bar, in every tile configuration: the epilogues of the factor
    update, of both Procrustes steps (their traces, their reads of Q and R Q, the triangular grid) and of the application,
    at sides one past a tile, inside one, and past two tile rows of 128."""
    worst, base = run_pair([(129, 257), (390, 64)], steps=2, skew=float("inf"), r2=r2,
                           grad_eps=float(torch.finfo(torch.float32).eps))
    assert_fp32(worst, base)


def _epilogue_results(hip, d, value):
    """The outputs of the factor update, both Procrustes steps and the application with `value` in single places."""
    g = torch.Generator().manual_seed(d)
    ws, st = L.Workspace(), L.stream_of(torch.empty(1, device=DEV))
    dev = torch.device(DEV)
    Q = torch.eye(d) + 0.05 * torch.randn(d, d, generator=g)
    X = torch.randn(d, d, generator=g) / d ** 0.5
    T = X @ X.T
    T[d // 3, d // 2] = T[d // 2, d // 3] = value
    V = torch.randn(32, d, generator=g).to(DEV)
    out = []
    q, t, Lv = Q.to(DEV), T.to(DEV), torch.full((1,), 1.0, device=DEV)
    qo = torch.empty_like(q)
    L.call_ws(hip.psgdk_factor_update, 0, d, 1, L.ptrs([t]), 0, L.ptrs([q]), L.ptrs([qo]), L.ptrs([Lv]), L.ptrs([V]), 0.1,
              0.9, 3.0, ws=ws, device=dev, stream=st)
    out += [qo, Lv]
    Q[d // 4, d // 5] = value
    q = Q.to(DEV)
    for fn in (hip.psgdk_procrustes, hip.psgdk_procrustes_r2):
        out.append(torch.empty_like(q))
        L.call_ws(fn, 0, d, 1, L.ptrs([q]), L.ptrs([out[-1]]), L.ptrs([V]), ws=ws, device=dev, stream=st)
    G = torch.randn(d, d, generator=g)
    G[1, 2] = value
    G, P = G.to(DEV), (T.clamp(max=1.0) + torch.eye(d)).to(DEV)
    W, pre = torch.zeros(d, d, device=DEV), torch.empty(d, d, device=DEV)
    k = L.Kron2d()
    k.nb, k.prec, k.m, k.n, k.g_dtype, k.p_dtype = 1, L.PREC_F32, d, d, L.F32, L.F32
    k.kind[0] = k.kind[1] = L.FACTOR_DENSE
    k.G[0] = G.data_ptr()
    for f in range(2):
        k.P[f][0] = k.Q[f][0] = k.L[f][0] = P.data_ptr()
    L.call_ws(hip.psgdk_kron2d_apply, k, L.ApplyOpts(1e-3, 0.5, 1.0, 0), L.ptrs([W]), L.ptrs([pre]), None, ws=ws,
              device=dev, stream=st)
    return [o.cpu() for o in out + [pre, W]]


@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.4e38, 2.0 ** 113, 2.0 ** 60])
@pytest.mark.parametrize("d", [130, 300])
def test_epilogues_of_sums_that_are_not_finite(engine, d, value):
    """Values that the split cannot hold, in front of every epilogue: infinities and NaNs fall where fp32 MFMAs (option 8 = 0)
    put them, and what is finite agrees row by row to 1e-5 of the row's largest value (both are fp32 sums, 3e-7, of
    products that reach the outputs through up to three more)."""
    got = _epilogue_results(engine, d, value)
    L.check(engine.psgdk_set_option(8, 0))
    ref = _epilogue_results(engine, d, value)
    L.check(engine.psgdk_set_option(8, 1))
    for i, (x, y) in enumerate(zip(got, ref)):
        assert torch.equal(torch.isnan(x), torch.isnan(y)) and torch.equal(torch.isinf(x), torch.isinf(y)), i
        fin = torch.isfinite(y)
        assert torch.equal(x[~fin & ~torch.isnan(y)], y[~fin & ~torch.isnan(y)]), i
        x, y = (torch.where(fin, v, 0.0).double().reshape(-1, v.shape[-1]) for v in (x, y))
        assert ((x - y).abs() <= 1e-5 * y.abs().amax(1, keepdim=True)).all(), i


@pytest.mark.parametrize("n,k", [(130, 70), (129, 129), (200, 333), (64, 1)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_gram_products_beside_their_own_k(engine, n, k, dt):
    """X X^T and X^T X from rows amid NaN, with fewer, as many and more k than rows: the rows' own k end inside a diagonal
    tile, and what lies beyond must not reach it."""
    for trans in (False, True):
        r, c = (k, n) if trans else (n, k)
        wide = torch.full((r + 2, c + 5), float("nan"), device=DEV, dtype=dt)
        X = wide[1:1 + r, 3:3 + c]
        X.copy_(torch.randn(r, c, generator=torch.Generator().manual_seed(n + k)))
        x = X.T if trans else X
        _check(K.syrk(X, trans, L.OUT_MIRROR, False), x, x.T, False, (n, k, trans, dt))
