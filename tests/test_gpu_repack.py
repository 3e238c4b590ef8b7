"""Device repack at the edges of a workgroup's span of K and of its row tile,
from data at any byte address: the host repack, bit for bit."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
FMTS = [O.Q4_0, O.Q8_0, O.Q4_K, O.Q4_K_GGML, O.Q6_K, O.Q6_K_GGML]


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("n,spans", [(16, 1), (17, 2), (33, 1.5), (15, 0.25), (1, 2.25), (160, 3)])
def test_repack_spans(dev, fmt, n, spans):
    import gq
    import torch
    k = int(1024 * spans) if fmt not in (O.Q8_0,) else int(512 * spans)
    for k in (k, k + 32) if fmt in (O.Q4_0, O.Q8_0) else (k,):
        w = O.gen_weights(fmt, n, k, seed=n + k)
        host = gq.repack_host(fmt, w, n, k)
        for shift in (0, 1, 2, 6):
            src = torch.zeros(w.size + shift, dtype=torch.uint8, device=dev)
            src[shift:] = torch.from_numpy(w).to(dev)
            got = gq.repack(fmt, src[shift:], n, k).cpu().numpy()
            assert np.array_equal(got, host), (k, shift)


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("n", [1, 16, 35])
def test_repack_short_and_partial_rows(dev, fmt, n):
    """Rows of one or two chunks, and last spans of every length in blocks."""
    import gq
    import torch
    step = 32 if fmt in (O.Q4_0, O.Q8_0) else 256
    for k in range(step, 36 * step if step == 32 else 9 * step, step):
        w = O.gen_weights(fmt, n, k, seed=n + k)
        host = gq.repack_host(fmt, w, n, k)
        shift = (k // step) % 3
        # bytes after the rows that must not be taken in
        src = torch.full((w.size + shift + 64,), 0xA5, dtype=torch.uint8, device=dev)
        src[shift:shift + w.size] = torch.from_numpy(w).to(dev)
        got = gq.repack(fmt, src[shift:shift + w.size], n, k).cpu().numpy()
        assert np.array_equal(got, host), (k, shift)
