"""The INT8 / INT4 GEMV band's matrix-core form against float64 products:
ragged rows, columns and K, each plan, K in parts, both activation types."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
# fp32 throughout: input limbs 2^-23, sums of a few 2^-24 each
TOL = 2e-7


def _case(int4, m, n, k, seed, f16=False):
    import torch
    g = torch.Generator().manual_seed(seed)
    lo, hi = (-8, 8) if int4 else (-128, 128)
    q = torch.randint(lo, hi, (n, k), generator=g, dtype=torch.int8)
    sc = 0.001 + torch.rand(n * k // 32, generator=g)
    a = torch.randn(m, k, generator=g) * torch.exp(2 * torch.randn(m, 1, generator=g))
    if f16:
        a = a.half()
    hs = 0.5 + torch.rand((n + 6) // 7, generator=g)
    q, sc, a, hs = (t.cuda() for t in (q, sc, a, hs))
    w = q.double().reshape(n, k // 32, 32) * sc.double().reshape(n, k // 32, 1)
    ref = a.double() @ w.reshape(n, k).t()
    if int4:
        ref = ref * hs.double()[torch.arange(n, device="cuda") // 7]
        u = (q & 15).view(torch.uint8)
        q = u[:, 0::2] | (u[:, 1::2] << 4)
    return a, q.contiguous(), sc, hs, ref


def _run(int4, a, q, sc, hs, m, n, k, c=None, force=False):
    import gq
    if int4:
        return gq.launch_int4_wt(a, q, sc, hs, m, n, k, head_dim=7, force_gemv=force, c=c)
    return gq.launch_int8_wt(a, q, sc, m, n, k, c=c)


def _rel(c, ref):
    return float((c.double() - ref).norm() / ref.norm())


# Shapes of every launch of the matrix-core form (row tiles of 16 x parts of K a
# workgroup; activation rows): ragged last tiles, K that ends inside a window
SHAPES = [
    (2, 14337, 2080),   # (two rows: the VALU kernels)
    (8, 14337, 2080), (8, 16500, 544),  # 4 x 2, 8 rows: a short K; more workgroups than CUs
    (8, 8300, 6272),    # 4 x 4, 8 rows, the last workgroup of three tiles
    (8, 20001, 256),    # 4 x 1, one window
    (8, 7001, 800), (8, 7001, 736),     # 2 x 4; 2 x 1: fewer windows than K parts
    (8, 4100, 4096), (8, 6001, 1056),   # 1 x 8, 1 x 4
    (3, 3001, 14304),   # 8 rows, K in parts over workgroups
    (12, 16500, 544), (9, 14337, 2080), (16, 14337, 352),  # 16 rows, four row tiles: 4 x 2, 4 x 4, 4 x 1
    (16, 7001, 1056), (16, 7001, 800), (16, 7001, 384),    # two row tiles: 2 x 8, 2 x 4, 2 x 1
    (9, 4100, 1248), (16, 3000, 4128), (16, 6001, 800), (32, 6001, 352),  # one row tile: 1 x 8 twice, 1 x 4, 1 x 1
    (16, 3000, 14304),  # 16 rows, K in parts over workgroups
    (17, 16500, 544), (31, 14336, 96), (32, 6500, 992),    # 32 rows: 4 x 2, 4 x 1, 4 x 4
    (17, 4097, 4096), (32, 1500, 8224),  # 32 rows, K in parts over workgroups
    (32, 1024, 2048),   # ... not in two
]


@pytest.mark.parametrize("int4", [True, False])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_rows_match_float64(dev, int4, m, n, k):
    a, q, sc, hs, ref = _case(int4, m, n, k, m + k)
    assert _rel(_run(int4, a, q, sc, hs, m, n, k), ref) <= TOL


@pytest.mark.parametrize("m,n,k", SHAPES[1::2])
def test_rows_of_fp16_activations(dev, m, n, k):
    a, q, sc, hs, ref = _case(True, m, n, k, m + k, f16=True)
    assert _rel(_run(True, a, q, sc, hs, m, n, k), ref) <= TOL


def test_fp16_activations_and_force_gemv(dev):
    m, n, k = 70, 4100, 1056
    a, q, sc, hs, ref = _case(True, m, n, k, 5, f16=True)
    assert _rel(_run(True, a, q, sc, hs, m, n, k, force=True), ref) <= TOL


@pytest.mark.parametrize("int4", [True, False])
def test_wide_range_and_nonfinite_rows(dev, int4):
    """Rows near fp32's ends stay exact to TOL; Inf and NaN stay in their row."""
    import torch
    m, n, k = 8, 4112, 4096
    a, q, sc, hs, _ = _case(int4, m, n, k, 9)
    a[0] *= 1e30
    a[1] *= 1e-36
    a[2, 300:] = 0.0
    a[3, 77] = float("inf")
    a[4, 4000] = float("nan")
    a[5] = 0.0
    w = (q if not int4 else torch.stack([q & 15, q >> 4], 2).reshape(n, k).to(torch.int16).add_(8).bitwise_and_(15).sub_(8))
    w = (w.double().reshape(n, k // 32, 32) * sc.double().reshape(n, k // 32, 1)).reshape(n, k)
    ref = a.double() @ w.t()
    if int4:
        ref = ref * hs.double()[torch.arange(n, device="cuda") // 7]
    c = _run(int4, a, q, sc, hs, m, n, k)
    for row in (0, 2, 6, 7):
        assert _rel(c[row], ref[row]) <= TOL, row
    assert _rel(c[1].double() * 2.0**60, ref[1] * 2.0**60) <= TOL
    assert bool((c[5] == 0).all())
    assert bool((torch.isnan(c[3]) == torch.isnan(ref[3])).all()) and bool((torch.isinf(c[3]) == torch.isinf(ref[3])).all())
    assert bool((c[3][torch.isinf(c[3])] == ref[3][torch.isinf(c[3])].float()).all())
    assert bool(torch.isnan(c[4]).all())


@pytest.mark.parametrize("int4,f16", [(True, False), (False, False), (True, True)])
@pytest.mark.parametrize("m,n,k", [(8, 4112, 4096), (13, 4112, 4128), (32, 2000, 8224), (8, 13000, 1056)])
def test_outlier_under_a_zero_code(dev, int4, f16, m, n, k):
    """One entry of each row far above the others, in a column whose codes are 0:
    the others count in full.  (fp16 activations: the others mostly subnormal.)"""
    import torch
    a, q, sc, hs, _ = _case(int4, m, n, k, m + n, f16=f16)
    w = torch.stack([q & 15, q >> 4], 2).reshape(n, k).to(torch.int16).add_(8).bitwise_and_(15).sub_(8) if int4 else q.clone()
    col = torch.arange(m, device="cuda") * 37 % k
    a = torch.randn(m, k, generator=torch.Generator().manual_seed(n)).cuda()
    if f16:
        a = (a * 2.0**-16).half()   # mostly subnormal
        big = torch.full((m,), 60000.0, device="cuda")
    else:
        big = 10.0 ** (4 + torch.arange(m, device="cuda") % 9).float()
    a[torch.arange(m, device="cuda"), col] = big.to(a.dtype)
    w[:, col] = 0
    if int4:
        u = (w & 15).to(torch.uint8)
        q = (u[:, 0::2] | (u[:, 1::2] << 4)).contiguous()
    else:
        q = w.contiguous()
    wd = (w.double().reshape(n, k // 32, 32) * sc.double().reshape(n, k // 32, 1)).reshape(n, k)
    ref = a.double() @ wd.t()
    if int4:
        ref = ref * hs.double()[torch.arange(n, device="cuda") // 7]
    c = _run(int4, a, q, sc, hs, m, n, k)
    err = (c.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= TOL, err


@pytest.mark.parametrize("int4", [True, False])
@pytest.mark.parametrize("m,n,k", [(8, 4112, 4096), (16, 4112, 4096), (32, 4112, 4096)])
def test_tiny_windows(dev, int4, m, n, k):
    """Windows of a row down to fp32's smallest normal values beside windows of
    zeros and of each other's sizes: every row's sum as its largest window's."""
    import torch
    a, q, sc, hs, _ = _case(int4, m, n, k, 31)
    w = torch.stack([q & 15, q >> 4], 2).reshape(n, k).to(torch.int16).add_(8).bitwise_and_(15).sub_(8) if int4 else q
    a = torch.randn(m, k, generator=torch.Generator().manual_seed(n)).cuda()
    for row in range(m):
        a[row] *= 2.0 ** -(8 * row % 124)
        a[row, 256 * (row % 8):256 * (row % 8) + 256] *= 2.0**-40
        a[row, 3000:3000 + 20 * row] = 0.0
    a[a.abs() < 2.0**-126] = 0.0
    wd = (w.double().reshape(n, k // 32, 32) * sc.double().reshape(n, k // 32, 1)).reshape(n, k)
    ref = a.double() @ wd.t()
    if int4:
        ref = ref * hs.double()[torch.arange(n, device="cuda") // 7]
    c = _run(int4, a, q, sc, hs, m, n, k).double()
    up = 2.0**60
    err = ((c - ref) * up).norm(dim=1) / (ref * up).norm(dim=1)
    assert float(err.max()) <= TOL, err


def test_captured_without_scratch(dev):
    import torch
    m, n, k = 16, 2000, 14336
    a, q, sc, hs, ref = _case(True, m, n, k, 11)
    c = _run(True, a, q, sc, hs, m, n, k)
    cg = torch.empty_like(c)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        _run(True, a, q, sc, hs, m, n, k, c=cg)
    for _ in range(3):
        cg.zero_()
        g.replay()
        _run(True, a, q, sc, hs, m, n, k, c=c)
        torch.cuda.synchronize()
        assert _rel(cg, ref) <= TOL and _rel(c, ref) <= TOL
    assert np.isfinite(cg.cpu().numpy()).all()


@pytest.mark.parametrize("int4", [True, False])
@pytest.mark.parametrize("n,k", [(33, 32), (130, 1024), (100, 1056), (257, 544), (16, 2080)])
def test_mfma_route_conversion(dev, int4, n, k):
    """M > 32: rows converted to the tiled layout at the edges of a workgroup's
    512 bytes of a row and of its 16 rows.  A and w s rounded to fp16 once each:
    about 3.5e-4 (of the scale to fp16 as well)."""
    a, q, sc, hs, ref = _case(int4, 40, n, k, n + k)
    assert _rel(_run(int4, a, q, sc, hs, 40, n, k), ref) <= 1e-3
