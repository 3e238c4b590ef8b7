"""Tiled-GEMM routes of Q6_K and fp16 weights (and int8 x int8) against float64 products of the
dequantized weights (the oracle's), at the edges of each tile shape."""
import threading

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
# A and W rounded once to fp16 each: relative error <= 2^-11 per factor, about
# 3.5e-4 over a row in the 2-norm; 1e-3 bounds it
TOL = 1e-3


def _ref(fmt, w, a, n, k):
    import torch
    wd = torch.from_numpy(O.dequant(fmt, w).reshape(n, k)).cuda().double()
    return a.double().cuda() @ wd.t()


def _rel(c, ref):
    return float((c.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("fmt", [O.Q6_K, O.Q6_K_GGML])
@pytest.mark.parametrize("m,n,k", [
    (4865, 5300, 256),   # 256 x 256 tiles, one row and 180 columns over
    (700, 8300, 512),    # 128 x 256
    (641, 4200, 1024),   # 128 x 128 in two K groups
    (300, 4100, 256),    # 64 x 128 in four K groups, one step each
])
def test_q6k_tiled_gemm(dev, fmt, m, n, k):
    import gq
    import torch
    w = O.gen_weights(fmt, n, k, seed=m)
    packed = torch.from_numpy(gq.repack_host(fmt, w, n, k)).to(dev)
    a = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).to(dev)
    ref = _ref(fmt, w, a, n, k)
    c = gq.gemm(fmt, packed, a, n, k)
    assert _rel(c, ref) <= TOL
    cb = gq.gemm(fmt, packed, a, n, k, out_dtype=torch.bfloat16)
    assert torch.equal(cb, c.bfloat16())


@pytest.mark.parametrize("m,n,k", [
    (130, 1400, 3072), (130, 1400, 256),    # one round of 16-row blocks; one chunk
    (41, 8200, 2048), (64, 8200, 4096),     # two rounds, full chunks
    (300, 832, 1024), (300, 1024, 3072),    # single row tiles; chunks three quarters full
    (1000, 300, 4096), (40, 20000, 256),    # more than 12 row blocks; up to 40 rows
])
def test_q6k_gemm_skinny_or_tiled(dev, m, n, k):
    """Both sides of the limits between the skinny and the tiled kernel."""
    import gq
    import torch
    w = O.gen_weights(O.Q6_K, n, k, seed=n)
    packed = torch.from_numpy(gq.repack_host(O.Q6_K, w, n, k)).to(dev)
    a = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).to(dev)
    assert _rel(gq.gemm(O.Q6_K, packed, a, n, k), _ref(O.Q6_K, w, a, n, k)) <= TOL


@pytest.mark.parametrize("m,n,k", [
    (49, 33, 4352), (33, 8192, 4352), (130, 8200, 4608), (300, 100, 14336),
    (48, 33, 4352), (23, 1000, 14336), (24, 1000, 14336), (17, 4200, 14336),  # about the GEMV passes' limits
])
def test_q6k_matmul_long_k(dev, m, n, k):
    """K > 4096: the tiled kernel on scratch memory, the 16-row GEMVs under
    capture; the same within the bound, replayed with eager calls between."""
    import gq
    import torch
    w = O.gen_weights(O.Q6_K, n, k, seed=k)
    packed = torch.from_numpy(gq.repack_host(O.Q6_K, w, n, k)).to(dev)
    a = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).to(dev)
    ref = _ref(O.Q6_K, w, a, n, k)
    c = torch.empty(m, n, device=dev)
    gq.matmul(O.Q6_K, packed, a, n, k, c=c)
    assert _rel(c, ref) <= TOL
    g = torch.cuda.CUDAGraph()
    cg = torch.empty(m, n, device=dev)
    with torch.cuda.graph(g):
        gq.matmul(O.Q6_K, packed, a, n, k, c=cg)
    for _ in range(3):
        cg.zero_()
        g.replay()
        gq.matmul(O.Q6_K, packed, a, n, k, c=c)
        torch.cuda.synchronize()
        assert _rel(cg, ref) <= TOL and _rel(c, ref) <= TOL


def test_scratch_routes_on_streams(dev):
    """Calls of four threads on streams of their own: each has its own scratch."""
    import gq
    import torch
    m, n, k = 100, 500, 5120
    w = O.gen_weights(O.Q6_K, n, k, seed=1)
    packed = torch.from_numpy(gq.repack_host(O.Q6_K, w, n, k)).to(dev)
    a = [torch.randn(m, k, generator=torch.Generator().manual_seed(i)).to(dev) for i in range(4)]
    want = [gq.matmul(O.Q6_K, packed, x, n, k) for x in a]
    got = [torch.zeros(m, n, device=dev) for _ in a]
    torch.cuda.synchronize()

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(10):
                gq.matmul(O.Q6_K, packed, a[i], n, k, c=got[i])
        s.synchronize()

    th = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert all(np.array_equal(x.cpu().numpy(), y.cpu().numpy()) for x, y in zip(got, want))


@pytest.mark.parametrize("m,n,k", [(100, 500, 5120), (64, 1000, 14336)])  # (the second splits K: two blocks a call)
def test_scratch_routes_of_many_threads(dev, m, n, k):
    """Twelve threads on streams of their own: more than blocks are kept.  Each call
    runs the kernels it runs alone, bit for bit."""
    import gq
    import torch
    w = O.gen_weights(O.Q6_K, n, k, seed=1)
    packed = torch.from_numpy(gq.repack_host(O.Q6_K, w, n, k)).to(dev)
    a = [torch.randn(m, k, generator=torch.Generator().manual_seed(i)).to(dev) for i in range(12)]
    want = [gq.matmul(O.Q6_K, packed, x, n, k) for x in a]
    got = [[torch.zeros(m, n, device=dev) for _ in range(20)] for _ in a]
    torch.cuda.synchronize()
    go = threading.Barrier(len(a))

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            go.wait()
            for c in got[i]:
                gq.matmul(O.Q6_K, packed, a[i], n, k, c=c)
        s.synchronize()

    th = [threading.Thread(target=work, args=(i,)) for i in range(len(a))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    bad = sum(not torch.equal(c, y) for x, y in zip(got, want) for c in x)
    assert bad == 0, bad


def test_scratch_of_many_streams_and_sizes(dev):
    """One thread, ten streams with work pending on each, sizes that grow and
    shrink: blocks are replaced and handed on in every state."""
    import gq
    import torch
    k = 4096
    w = torch.randn(700, k, generator=torch.Generator().manual_seed(2)).half().to(dev)
    a = torch.randn(900, k, generator=torch.Generator().manual_seed(3)).to(dev)
    sizes = [(17, 700), (900, 100), (64, 300), (300, 700), (40, 64), (600, 512)]
    want = {(m, n): gq.gemm_f16w(w[:n], a[:m], n, k) for m, n in sizes}
    big = torch.randn(2048, 2048, device=dev)
    streams = [torch.cuda.Stream() for _ in range(10)]
    torch.cuda.synchronize()
    got = []
    for turn in range(12):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                if turn % 3 == 0:
                    big @ big
                m, n = sizes[(turn * 7 + i) % len(sizes)]
                c = torch.zeros(m, n, device=dev)
                got.append(((m, n), gq.gemm_f16w(w[:n], a[:m], n, k, c=c)))
    torch.cuda.synchronize()
    assert all(torch.equal(c, want[mn]) for mn, c in got)


@pytest.mark.parametrize("m,n,k", [
    (4865, 5300, 96),     # 256 x 256 tiles; K past the last whole 64-k step
    (700, 8300, 160),     # 128 x 256
    (641, 4200, 1056),    # 128 x 128 in two K groups
    (300, 4100, 32),      # 64 x 128 in four K groups, K within one step
    (17, 33, 4128),       # K in parts, 64-row tiles, an odd count of outputs
    (131, 300, 14304),    # K in parts of unequal length, 128-row tiles
    (17, 100, 64), (40, 64, 512), (49, 64, 512),  # about the batch GEMVs' limits
    (32, 64, 512), (33, 64, 512), (17, 2560, 2048), (17, 2561, 2048),
])
def test_f16w_tiled(dev, m, n, k):
    """Columns past K hold Inf in the next row's weights: they must not count."""
    import gq
    import torch
    g = torch.Generator().manual_seed(m + k)
    w = torch.randn(n + 1, k, generator=g).half()
    w[n] = float("inf")  # (the row after the matrix)
    w = w.to(dev)
    a = torch.randn(m, k, generator=g).to(dev)
    a[m // 2] *= 1e6     # a row beyond fp16's range
    c = torch.full((m + 1, n), 7.0, device=dev)
    gq.gemm_f16w(w[:n], a, n, k, c=c[:m])
    ref = a.double() @ w[:n].double().t()
    err = (c[:m].double() - ref).norm(dim=1) / ref.norm(dim=1)
    # one row of n outputs: a little over the bound of a long row
    assert float(err.max()) <= 2 * TOL and _rel(c[:m], ref) <= TOL
    assert bool((c[m] == 7.0).all())


# Rows of every tile shape and conversion kernel of the two routes that scale
# windows of 256 k by themselves: (fp16 weights?, m, n, k)
WINDOW_SHAPES = [
    (True, 300, 4100, 512), (True, 641, 4200, 1024), (True, 700, 8300, 512), (True, 4865, 5300, 512),  # tiles
    (True, 50, 130, 4064), (True, 100, 300, 4096),      # K parts, 64 and 128 rows
    (True, 64, 300, 16384), (True, 1030, 600, 5120), (True, 50, 100, 33024),  # conversions
    (False, 49, 33, 4352), (False, 300, 4100, 4352), (False, 641, 4200, 4352), (False, 700, 8300, 4352),
    (False, 4865, 5300, 4352), (False, 64, 1000, 14336),  # (the last: K parts)
]


def _window_weights(f16, n, k, live):
    """Weights that are zero outside of row n's window live[n] (None: none zero):
    as the call takes them, and in float64."""
    import gq
    import torch
    if f16:
        w = torch.randn(n, k, generator=torch.Generator().manual_seed(n)).cuda().half()
        if live is not None:
            w *= live.cuda()[:, None] == torch.arange(k, device="cuda")[None] // 256
        return w, w.double()
    b = O.gen_weights(O.Q6_K, n, k, seed=n).reshape(n, k // 256, 210)
    if live is not None:
        dead = live.numpy()[:, None] != np.arange(k // 256)[None]
        b[dead, :128] = 0      # code 32 in all places: weight 0
        b[dead, 128:192] = 0xAA
    b = b.reshape(-1)
    return (torch.from_numpy(gq.repack_host(O.Q6_K, b, n, k)).cuda(),
            torch.from_numpy(O.dequant(O.Q6_K, b).reshape(n, k)).cuda().double())


def _window_run(f16, w, a, n, k):
    import gq
    return gq.gemm_f16w(w, a, n, k) if f16 else gq.matmul(O.Q6_K, w, a, n, k)


@pytest.mark.parametrize("f16,m,n,k", WINDOW_SHAPES)
def test_small_windows_beside_large_ones(dev, f16, m, n, k):
    """Windows of a row up to 2^80 apart, each output from one of them alone: all
    keep their bits.  A is rounded once to fp16, 2^-11 of each product (Q6_K: its
    scales and weights once each too), and an entry 2^-29 or less of the row's, where
    its window is not scaled up, to 2^-19 of the window's largest."""
    import torch
    g = torch.Generator().manual_seed(m)
    nw = -(-k // 256)
    w, wd = _window_weights(f16, n, k, torch.arange(n) % nw)
    a = torch.randn(m, k, generator=g).cuda()
    down = torch.randint(0, 81, (m, nw), generator=g).cuda()
    down[torch.arange(m) % 3 == 1] //= 8   # up to 10: not scaled
    down[torch.arange(m) % 3 == 2] //= 3   # around the limit of 20
    a *= torch.exp2(-down.double()).float().repeat_interleave(256, 1)[:, :k]
    a[3 % m] = 0.0
    ref = a.double() @ wd.t()
    top = torch.nn.functional.pad(a.double().abs(), (0, 256 * nw - k)).reshape(m, nw, 256).amax(2)
    tol = (2.0**-10 if f16 else 2.0**-9) * (a.double().abs() @ wd.abs().t())
    tol += 2.0**-18 * top[:, torch.arange(n, device="cuda") % nw] * wd.abs().sum(1)
    c = _window_run(f16, w, a, n, k)
    bad = (c.double() - ref).abs() > tol
    assert not bool(bad.any()), (int(bad.sum()), bad.nonzero()[:4])
    # rows without such windows: the bits they have in a call of their own kind
    if m > 64:
        b = torch.randn(m, k, generator=g).cuda()
        x = b.clone()
        x[5] = a[0]
        y, z = _window_run(f16, w, b, n, k), _window_run(f16, w, x, n, k)
        y[5] = z[5]
        assert torch.equal(y, z)


@pytest.mark.parametrize("f16,m,n,k", WINDOW_SHAPES[3:10])
def test_large_values_beside_an_inf(dev, f16, m, n, k):
    """Finite values past fp16's range in a row with an Inf stay finite: the outputs
    are Infs by the sign of the Inf's weight, not the NaN of two Infs."""
    import torch
    g = torch.Generator().manual_seed(m)
    w, wd = _window_weights(f16, n, k, None)
    a = torch.randn(m, k, generator=g).cuda()
    rows = torch.arange(0, m, 7, device="cuda")
    a[rows] *= 1e9
    col = (rows * 131) % k
    a[rows, col] = float("inf")
    c = _window_run(f16, w, a, n, k)
    at = wd[:, col].t()
    want = torch.sign(at) * float("inf")  # (0: NaN)
    assert torch.equal(torch.nan_to_num(c[rows].double(), nan=0.0, posinf=1.0, neginf=-1.0),
                       torch.nan_to_num(want, nan=0.0, posinf=1.0, neginf=-1.0))
    rest = torch.ones(m, dtype=torch.bool, device="cuda")
    rest[rows] = False
    assert _rel(c[rest], a[rest].double() @ wd.t()) <= TOL


@pytest.mark.parametrize("f16,k,fit", [(True, 16384, 3840), (False, 16128, 4096)])
@pytest.mark.parametrize("extra", [1, 70])
def test_second_block_of_rows(dev, f16, k, fit, extra):
    """More rows than one scratch block converts at a time: the last block, of a few
    rows, takes another tile (and could split K).  Every row against float64."""
    import torch
    m, n = fit + extra, 70
    w, wd = _window_weights(f16, n, k, None)
    a = torch.randn(m, k, generator=torch.Generator(device="cuda").manual_seed(extra), device="cuda")
    c = _window_run(f16, w, a, n, k)
    worst = 0.0
    for r in range(0, m, 512):
        ref = a[r:r + 512].double() @ wd.t()
        worst = max(worst, float(((c[r:r + 512].double() - ref).norm(dim=1) / ref.norm(dim=1)).max()))
    # one row of 70 outputs: a little over the bound of a long row
    assert worst <= 2 * TOL, worst


@pytest.mark.parametrize("m,n,k", [(49, 1, 32), (64, 3, 64), (50, 7, 32), (70, 1, 288), (300, 2, 96)])
def test_f16w_fewer_weights_than_a_padded_row(dev, m, n, k):
    """Steps past K start beyond the matrix's end: they read zeros, not the Inf
    that follows it.  A rounded once to fp16: 2^-11 of each product, 2^-10 bounds
    it with the fp32 sums."""
    import gq
    import torch
    g = torch.Generator().manual_seed(m + k)
    w = torch.randn(n * k + 4096, generator=g).half()
    w[n * k:] = float("inf")
    w = w.to(dev)
    wm = w[:n * k].view(n, k)
    a = torch.randn(m, k, generator=g).to(dev)
    c = gq.gemm_f16w(wm, a, n, k).double()
    ref = a.double() @ wm.double().t()
    assert bool(((c - ref).abs() <= 2.0**-10 * (a.double().abs() @ wm.double().abs().t())).all())


@pytest.mark.parametrize("m,n,k", [(300, 4100, 352), (700, 8300, 352), (641, 4200, 352), (4865, 5300, 352)])
def test_f16w_infinite_weight(dev, m, n, k):
    """One infinite weight of a step whose buffer a step past K takes next: its
    output is +-Inf, and NaN only if the buffer still held it against zeros."""
    import gq
    import torch
    g = torch.Generator().manual_seed(n)
    w = torch.randn(n, k, generator=g).half()
    w[::2, 200] = float("inf")
    w[1::2, 330] = float("inf")
    w = w.to(dev)
    a = torch.randn(m, k, generator=g).abs().add_(0.1).to(dev)
    c = torch.empty(m, n, device=dev)
    gq.gemm_f16w(w, a, n, k, c=c)
    assert bool((c == float("inf")).all())


@pytest.mark.parametrize("m,n,k", [(1, 16, 32), (130, 140, 96), (129, 257, 4128), (260, 100, 1056)])
@pytest.mark.parametrize("inf", [False, True])
def test_q8_i8_scales(dev, m, n, k, inf):
    """Exact integer sums under fp32 scales; with infinite weight scales the
    tile takes the form that keeps them infinite (NaN where the sum is 0)."""
    import gq
    import torch
    w = O.gen_weights(O.Q8_0, n, k, seed=k).reshape(-1, 34)
    if inf:
        w[(n - 1) * (k // 32), 0:2] = (0x00, 0x7C)  # +Inf, the last row's first block
        w[0, 0:2] = (0x00, 0xFC)                    # -Inf, row 0
        w[0, 2:] = 0
    qa, da = gq.quantize_act_q8(torch.randn(m, k, generator=torch.Generator().manual_seed(k)).to(dev))
    packed = torch.from_numpy(gq.repack_host(O.Q8_0, w.ravel(), n, k)).to(dev)
    c = gq.gemm_q8_i8(packed, qa, da, n).double().cpu().numpy()
    q = w[:, 2:].view(np.int8).astype(np.float64).reshape(n, k // 32, 32)
    d = w[:, :2].copy().view(np.float16).astype(np.float64).reshape(n, k // 32)
    p = np.einsum("mbe,nbe->mnb", qa.cpu().numpy().astype(np.float64).reshape(m, k // 32, 32), q)
    with np.errstate(invalid="ignore"):
        ref = (p * d[None] * da.cpu().numpy().astype(np.float64)[:, None]).sum(2)
    assert np.array_equal(np.isnan(c), np.isnan(ref)) and np.array_equal(np.isinf(c), np.isinf(ref))
    assert np.array_equal(c[np.isinf(c)], ref[np.isinf(ref)])
    ok = np.isfinite(ref)
    # two roundings per block and one per sum, K / 32 blocks: under 2e-6
    assert np.linalg.norm(c[ok] - ref[ok]) <= 2e-6 * np.linalg.norm(ref[ok])


@pytest.mark.parametrize("fmt", [O.Q4_0, O.Q8_0, O.Q4_K, O.Q6_K])
@pytest.mark.parametrize("m,n,k,adt,odt", [
    (33, 130, 8448, "float32", "float32"),
    (64, 4096, 14336, "bfloat16", "bfloat16"),
    (301, 333, 9216, "float32", "float32"),      # an odd count of outputs, parts of unequal length
    (129, 1000, 16384, "float16", "float32"),
])
def test_gemm_k_parts(dev, fmt, m, n, k, adt, odt):
    """K over workgroups: gq_gemm with a workspace, gq_gemm_static's own memory
    (the same sums), and the unsplit form under capture."""
    import ctypes

    import gq
    import torch
    adt, odt = getattr(torch, adt), getattr(torch, odt)
    w = O.gen_weights(fmt, n, k, seed=m)
    packed = torch.from_numpy(gq.repack_host(fmt, w, n, k)).to(dev)
    a = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).to(adt).to(dev)
    ref = _ref(fmt, w, a, n, k)
    tol = TOL if odt == torch.float32 else 4e-3  # (one rounding to bf16: 2^-9)
    if fmt == O.Q6_K:
        c = gq.matmul(fmt, packed, a.float(), n, k)
        assert _rel(c, ref) <= TOL
        return
    c = gq.gemm(fmt, packed, a, n, k, out_dtype=odt, workspace=gq.Workspace(dev))
    assert _rel(c, ref) <= tol
    cs = torch.empty_like(c)
    dt = {torch.bfloat16: gq.DT_BF16, torch.float16: gq.DT_F16, torch.float32: gq.DT_F32}
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    st = gq.load().gq_gemm_static(fmt, p(packed), p(a), dt[adt], p(cs), dt[odt], m, n, k,
                                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == 0 and torch.equal(c, cs)
    ws, cg = gq.Workspace(dev, gq.gemm_workspace_bytes(fmt, m, k)), torch.empty_like(c)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        gq.gemm(fmt, packed, a, n, k, out_dtype=odt, c=cg, workspace=ws)
    for _ in range(3):
        cg.zero_()
        g.replay()
        gq.gemm(fmt, packed, a, n, k, out_dtype=odt, c=c, workspace=ws)
        torch.cuda.synchronize()
        assert _rel(cg, ref) <= tol and _rel(c, ref) <= tol


@pytest.mark.parametrize("fmt", [O.Q4_0, O.Q8_0, O.Q4_K, O.Q6_K])
@pytest.mark.parametrize("b,n,k", [(9, 1025, 8448), (16, 6500, 8192), (13, 2000, 14336)])
def test_gemv_k_parts(dev, fmt, b, n, k):
    """Batch 9..16 with K over workgroups, and the unsplit kernel under capture."""
    import gq
    import torch
    w = O.gen_weights(fmt, n, k, seed=b)
    packed = torch.from_numpy(gq.repack_host(fmt, w, n, k)).to(dev)
    x = torch.randn(b, k, generator=torch.Generator().manual_seed(b)).to(dev)
    x[b - 1] *= 1e6
    ref = _ref(fmt, w, x, n, k)
    y, yg = gq.gemv(fmt, packed, x, n, k), torch.empty(b, n, device=dev)
    rel = lambda t: float(((t.double() - ref).norm(dim=1) / ref.norm(dim=1)).max())  # noqa: E731
    assert rel(y) <= TOL
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        gq.gemv(fmt, packed, x, n, k, y=yg)
    for _ in range(3):
        yg.zero_()
        g.replay()
        gq.gemv(fmt, packed, x, n, k, y=y)
        torch.cuda.synchronize()
        assert rel(yg) <= TOL and rel(y) <= TOL
