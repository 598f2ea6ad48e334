"""The lane-group reductions of the row operators (groups of 8, 16, 32 and 64 lanes): every lane's value has to reach every
lane. Each row carries one outlier, its column walking through all of the row's 16-byte chunks, so a lost or doubled lane
moves the row's maximum, sum, mean or variance far beyond rounding."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import to_dev, to_np
from oracle import refs
from softhier_mlir_amd import data, shops

pytestmark = pytest.mark.gpu
A = shops.addr


@pytest.mark.parametrize("cols", [8, 64, 104, 128, 256, 264, 512, 1000, 1001, 1024, 2048, 4096, 5000])
@pytest.mark.parametrize("rows", [67, 2049])
def test_every_lane_counts(lib, gpu, rows, cols):
    import torch
    if rows * cols > 2049 * 2048:
        rows = 515
    chunks = (cols + 7) // 8
    x = data.normal((rows, cols), 21)
    r = np.arange(rows)
    x[r, np.minimum(8 * (r % chunks) + r % 8, cols - 1)] = 12.0
    g, b = data.normal((1, cols), 22, 1.0, 0.1), data.normal((1, cols), 23)
    X, G, B, Y = to_dev(x), to_dev(g), to_dev(b), torch.zeros(rows, cols, dtype=torch.float16, device="cuda")
    ops = [(lambda: lib.sh_softmax_rows(A(Y), A(X), rows, cols, cols, 0.5, shops.SH_ALL), refs.softmax(x, 0.5)),
           (lambda: lib.sh_softmax_rows(A(Y), A(X), rows, cols, cols, -0.5, shops.SH_ALL), refs.softmax(x, -0.5)),
           (lambda: lib.sh_layernorm(A(Y), A(X), A(G), A(B), rows, cols, cols, 1e-6, shops.SH_ALL), refs.layernorm(x, g, b, 1e-6))]
    if cols % 4 == 0 and cols <= 4096:
        ops.append((lambda: lib.sh_rmsnorm(A(Y), A(X), A(G), rows, cols, cols, 1e-6, shops.SH_ALL), refs.rmsnorm(x, g, 1e-6)))
    for fn, want in ops:
        fn()
        assert shops.last_error()[0] == 0, shops.last_error()
        bad, err, _ = refs.close(to_np(Y), want)
        assert bad == 0, err
