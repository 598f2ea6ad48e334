"""Row operators on dense tensors of odd widths and on odd bases (the any-alignment kernels) against the oracle: widths around
the 8-half chunk, totals that end inside a chunk, a bias chunk that spans two rows, outputs aliasing their input, and nothing
written outside the tensor. Exact operators (add, add_bias: one rounding; transpose) are compared bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import to_np
from oracle import refs
from softhier_mlir_amd import data, shops

pytestmark = pytest.mark.gpu
A = shops.addr
ALL = shops.SH_ALL


def _buf(x, off):
    """x's halves `off` halves into a padded buffer of sevens."""
    import torch
    t = torch.full((x.size + 16,), 7.0, dtype=torch.float16, device="cuda")
    t[off:off + x.size] = torch.from_numpy(x.reshape(-1)).cuda()
    return t


def _out(t, n, off, shape):
    v = to_np(t)
    assert (v[:off] == 7.0).all() and (v[off + n:] == 7.0).all(), "wrote outside"
    return v[off:off + n].reshape(shape)


@pytest.mark.parametrize("rows,cols", [(1, 8), (3, 9), (7, 12), (5, 15), (33, 100), (129, 131), (64, 513), (10, 1001), (3, 4099)])
@pytest.mark.parametrize("off", [0, 1, 5])
def test_dense_odd_widths(lib, gpu, rows, cols, off):
    x, y = data.normal((rows, cols), 5), data.normal((rows, cols), 6)
    g, b = data.normal((1, cols), 7, 1.0, 0.1), data.normal((1, cols), 8)
    n, r16 = rows * cols, refs.r16
    G, B = _buf(g, off), _buf(b, off)

    def run(fn, *srcs):
        """fn(y, srcs...) out of place and in place; both views of the result."""
        got = []
        for inplace in (False, True):
            S = [_buf(s, off) for s in srcs]
            Y = S[0] if inplace else _buf(np.zeros_like(x), off)
            fn(A(Y, off), *[A(s, off) for s in S])
            assert shops.last_error()[0] == 0, shops.last_error()
            got.append(_out(Y, n, off, (rows, cols)))
        assert np.array_equal(got[0].view(np.uint16), got[1].view(np.uint16))
        return got[0]

    z = run(lambda o, a, c: lib.sh_add(o, a, c, rows, cols, cols, ALL), x, y)
    assert np.array_equal(z.astype(np.float32), r16(refs.add(x, y)))
    z = run(lambda o, a: lib.sh_add_bias(o, a, A(B, off), rows, cols, cols, ALL), x)
    assert np.array_equal(z.astype(np.float32), r16(refs.add_bias(x, b)))
    z = run(lambda o, a: lib.sh_scale(o, a, rows, cols, cols, 0.25, ALL), x)
    assert np.array_equal(z.astype(np.float32), r16(refs.scale(x, 0.25)))
    for fn, want in ((lambda o, a: lib.sh_gelu(o, a, rows, cols, cols, ALL), refs.gelu(x)),
                     (lambda o, a: lib.sh_layernorm(o, a, A(G, off), A(B, off), rows, cols, cols, 1e-6, ALL), refs.layernorm(x, g, b, 1e-6)),
                     (lambda o, a: lib.sh_softmax_rows(o, a, rows, cols, cols, 0.5, ALL), refs.softmax(x, 0.5))):
        bad, err, _ = refs.close(run(fn, x), want)
        assert bad == 0, err
    if cols % 4 == 0:
        assert refs.close(run(lambda o, a, c: lib.sh_silu_mul(o, a, c, rows, cols, cols, ALL), x, y), refs.silu_mul(x, y))[0] == 0
        assert refs.close(run(lambda o, a: lib.sh_rmsnorm(o, a, A(G, off), rows, cols, cols, 1e-6, ALL), x), refs.rmsnorm(x, g, 1e-6))[0] == 0
    X, T = _buf(x, off), _buf(np.zeros_like(x), off)
    lib.sh_transpose(A(T, off), A(X, off), rows, cols, cols, rows, ALL)
    assert np.array_equal(_out(T, n, off, (cols, rows)).view(np.uint16), x.T.view(np.uint16))
