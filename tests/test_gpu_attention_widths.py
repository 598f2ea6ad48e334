"""Head widths and key-block splits of the attention kernels against the oracle: the one-pass kernel at every width it has a
build for, on sequences that end inside, at and past a key block (64) and a query block (128) and at few workgroups, and the
key-splitting kernel of token-masked heads at the edges of its 32-query items and of its wavefronts' key blocks."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import _KEEP, to_dev, to_np
from oracle import refs
from softhier_mlir_amd import data, shops

pytestmark = pytest.mark.gpu
A = shops.addr


@pytest.mark.parametrize("dh", [32, 64, 72, 80, 96, 128])
@pytest.mark.parametrize("S", [1, 63, 65, 129, 200, 580])
def test_one_pass_widths(lib, gpu, S, dh):
    """Packed q | k | v rows of two sequences; values in the last columns of V and K rows reach only their own head (a width
    that is no multiple of 32 reads past a row inside the kernel): a NaN planted in the next head's V must not leak."""
    import torch
    B, H = 2, 3
    D = H * dh
    q, k, v = (data.normal((B * S, D), 70 + i) for i in range(3))
    v[:, dh:2 * dh] = np.nan                                  # head 1's values: heads 0 and 2 must stay finite
    X = to_dev(np.concatenate([q, k, v], 1))
    O = torch.full((B * S, D + 8), 7.0, dtype=torch.float16, device="cuda")
    rc = lib.sh_attention_batched(A(X), A(X, D), A(X, 2 * D), A(O), B, S, D, H, 3 * D, 3 * D, 3 * D, D + 8,
                                  S * 3 * D, S * 3 * D, S * 3 * D, S * (D + 8), dh ** -0.5, 0)
    assert rc == 0, shops.last_error()
    o = to_np(O)
    assert (o[:, D:] == 7.0).all()
    for h in (0, 2):
        c = slice(h * dh, (h + 1) * dh)
        want = refs.attention_batched(q[:, c], k[:, c], v[:, c], B, 1, dh ** -0.5)
        bad, err, _ = refs.close(o[:, c], want)
        assert bad == 0, (h, err)
    assert np.isnan(o[:, dh:2 * dh]).all()


@pytest.mark.parametrize("S,H", [(132, 3), (192, 4), (196, 12), (257, 2), (512, 2), (1000, 4)])
@pytest.mark.parametrize("scale", [0.125, -0.3, 2.0])
def test_few_workgroups_unmasked(lib, gpu, S, H, scale):
    D = 64 * H
    q, k, v = (data.normal((S, D), 80 + i) for i in range(3))
    import torch
    O = torch.zeros((S, D), dtype=torch.float16, device="cuda")
    rc = lib.sh_attention_batched(A(to_dev(q)), A(to_dev(k)), A(to_dev(v)), A(O), 1, S, D, H, D, D, D, D, 0, 0, 0, 0, scale, 0)
    assert rc == 0, shops.last_error()
    # against float64 (the oracle rounds its scores to fp16, which a scale of 2 makes visible): the numerators' fp16 rounding
    # moves the weighted mean of V by at most 2^-11 max|v| in the sum and as much in its normalisation, the output's own
    # rounding adds 2^-11 max|v|, and the fp32 exponents (|c s| < 256, 2^-24 relative) less than 2^-15: below 2^-9 max|v|
    o, x64 = to_np(O).astype(np.float64), [t.astype(np.float64) for t in (q, k, v)]
    for h in range(H):
        c = slice(64 * h, 64 * (h + 1))
        t = scale * (x64[0][:, c] @ x64[1][:, c].T)
        p = np.exp(t - t.max(1, keepdims=True))
        want = (p / p.sum(1, keepdims=True)) @ x64[2][:, c]
        assert np.abs(o[:, c] - want).max() <= 2.0 ** -9 * np.abs(x64[2][:, c]).max(), h


@pytest.mark.parametrize("dh", [32, 64, 72, 80, 96, 128])
@pytest.mark.parametrize("S", [4, 36, 64, 68, 200])
def test_split_keys_masked(lib, gpu, S, dh):
    """Causal tokens, a token array one element into its buffer, padding queries (uniform) and a first block whose keys no
    query of a later class order may see."""
    import torch
    H, Hkv = 4, 2
    D, DKV = H * dh, Hkv * dh
    q, k, v = data.normal((S, D), 91), data.normal((S, DKV), 92), data.normal((S, DKV), 93)
    Q, K, V = to_dev(q), to_dev(k), to_dev(v)
    down = np.arange(S, dtype=np.uint32)[::-1].copy()         # query i sees keys j >= i
    mix = np.array([(j % 3) if j % 11 else refs.LLM_PAD for j in range(S)], np.uint32)
    for tok in (refs.llm_tokens(S, "causal"), down, mix):
        T = torch.from_numpy(np.concatenate([[0], tok]).astype(np.uint16).view(np.int16)).cuda()
        _KEEP.append(T)
        O = torch.zeros((S, D), dtype=torch.float16, device="cuda")
        assert lib.sh_attention_gqa(A(Q), A(K), A(V), A(O), S, D, H, Hkv, D, DKV, DKV, D, 0.125, A(T, 1), shops.SH_ALL) == 0, shops.last_error()
        bad, err, _ = refs.close(to_np(O), refs.attention_gqa(q, k, v, H, Hkv, tok))
        assert bad == 0, err


@pytest.mark.parametrize("dh", [32, 72, 80, 96])
@pytest.mark.parametrize("S,scale", [(1, 0.125), (63, -0.3), (64, 2.0), (129, 0.125), (300, 0.0), (580, 0.125)])
def test_one_pass_widths_store_the_general_kernel_bits(lib, gpu, S, scale, dh):
    """The same heads one element into their buffers run on the register-staged kernel of any alignment: the same running
    maximum, numerators and sums in the same order, so the same bits, infinite scores included."""
    import torch
    B, H = 2, 3
    D = H * dh
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(B * S, 3 * D, generator=g, device="cuda").half()
    x[:, :D] *= 4                                             # scores over a few tens: the maximum moves in later blocks
    x[S // 2, D:D + 2] = float("inf")                         # one key of head 0, sequence 0: scores +-inf and NaN
    outs = []
    for off in (0, 1):
        xb = torch.zeros(B * S * 3 * D + 8, device="cuda", dtype=torch.float16)
        xb[off:off + x.numel()] = x.reshape(-1)
        ob = torch.zeros(B * S * D + 8, device="cuda", dtype=torch.float16)
        rc = lib.sh_attention_batched(A(xb, off), A(xb, off + D), A(xb, off + 2 * D), A(ob, off), B, S, D, H, 3 * D, 3 * D, 3 * D, D,
                                      S * 3 * D, S * 3 * D, S * 3 * D, S * D, scale, 0)
        assert rc == 0, shops.last_error()
        outs.append(ob[off:off + B * S * D].clone())
    nan = [torch.isnan(o) for o in outs]
    assert torch.equal(*nan)
    assert torch.equal(outs[0].view(torch.int16)[~nan[0]], outs[1].view(torch.int16)[~nan[0]])


@pytest.mark.parametrize("dh", [32, 64, 72, 80, 96, 128])
def test_low_tail(lib, gpu, dh):
    """One key a few units above a long tail that is far below 0, the reference of an unmoved exponent: the tail's numerators
    keep the weight that their row sum counts. Against float64 in units of max|v|: numerators and output rounded to fp16 once
    each (2^-11 + 2^-11), and the tail's S numerators, fp16 subnormals, by at most 2^-25 of the largest each. (64 and 128 wide heads start
    from m = 0 while the first maximum is within 8 of it, their numerators up to 2^8 smaller: S 2^-17, and their row sums are those
    of the rounded numerators.)"""
    import torch
    S = 2048
    q = np.zeros((S, dh), np.float16); k = np.zeros((S, dh), np.float16)
    q[:, 0] = 1.0
    top, low = (-7.9, -25.5) if dh not in (64, 128) else (-7.9, -20.0)
    k[:, 0] = low
    k[7, 0] = top
    v = np.abs(data.normal((S, dh), 95)).astype(np.float16) + np.float16(1)
    v[7] = 0
    scale = float(np.log(2.0))                                # scores in log2 units
    O = torch.zeros((S, dh), dtype=torch.float16, device="cuda")
    rc = lib.sh_attention_batched(A(to_dev(q)), A(to_dev(k)), A(to_dev(v)), A(O), 1, S, dh, 1, dh, dh, dh, dh, 0, 0, 0, 0, scale, 0)
    assert rc == 0, shops.last_error()
    t = k[:, 0].astype(np.float64)
    p = 2.0 ** (t - t.max())
    want = (p / p.sum()) @ v.astype(np.float64)
    sub = S * (2.0 ** -17 if dh in (64, 128) else 2.0 ** -25)
    assert np.abs(to_np(O).astype(np.float64) - want).max() <= (2 * 2.0 ** -11 + sub) * v.max(), dh


@pytest.mark.parametrize("dh", [32, 72, 80, 96])
def test_masked_tail_keeps_fp32_weights(lib, gpu, dh):
    """Masked heads of these widths weigh keys in fp32: a tail 25.5 (log2) below its maximum, which one fp16 numerator cannot
    hold, carries the whole output here (the largest key's values are 0). Against float64: the output's rounding 2^-11, fp32 exponents (25.5
    in log2, 2^-24 relative) 2^-19, S sums 2^-24 each and numerators 2^-22, together below 2^-10."""
    import torch
    S = 256
    q = np.zeros((S, dh), np.float16); k = np.zeros((S, dh), np.float16)
    q[:, 0] = 1.0
    k[:, 0] = -25.5
    k[7, 0] = 0.0
    v = np.full((S, dh), 60000.0, np.float16) - np.abs(data.normal((S, dh), 96)).astype(np.float16) * np.float16(4096)
    v[7] = 0
    T = torch.zeros(S, dtype=torch.int16, device="cuda")      # one class: every key allowed
    O = torch.zeros((S, dh), dtype=torch.float16, device="cuda")
    rc = lib.sh_attention_gqa(A(to_dev(q)), A(to_dev(k)), A(to_dev(v)), A(O), S, dh, 1, 1, dh, dh, dh, dh, float(np.log(2.0)), A(T), shops.SH_ALL)
    assert rc == 0, shops.last_error()
    p = 2.0 ** k[:, 0].astype(np.float64)
    want = (p / p.sum()) @ v.astype(np.float64)
    assert np.abs(to_np(O).astype(np.float64) / want - 1).max() <= 2.0 ** -10


@pytest.mark.parametrize("dh", [32, 64, 72, 80, 96, 128, 88])
@pytest.mark.parametrize("S", [12, 132])
def test_masked_infinite_scores(lib, gpu, S, dh):
    """Keys that score -inf take no weight; a query whose allowed keys all do averages V uniformly over the S keys, as a
    padding query does. (88 wide heads: the per-query kernel.) Means of values in (0, 4) rounded to fp16 weights and once more."""
    import torch
    q, k = np.abs(data.normal((S, dh), 97)) + 1, data.normal((S, dh), 98)
    v = np.minimum(np.abs(data.normal((S, dh), 99)), 4).astype(np.float16)
    k[:5, 0] = -np.inf                                        # causal: queries 0 .. 4 see no other key
    T = torch.arange(S, dtype=torch.int32, device="cuda").to(torch.int16)
    O = torch.zeros((S, dh), dtype=torch.float16, device="cuda")
    rc = lib.sh_attention_gqa(A(to_dev(q)), A(to_dev(k)), A(to_dev(v)), A(O), S, dh, 1, 1, dh, dh, dh, dh, 0.125, A(T), shops.SH_ALL)
    assert rc == 0, shops.last_error()
    q, k, v = (t.astype(np.float16).astype(np.float64) for t in (q, k, v))
    want = np.empty((S, dh))
    for i in range(S):
        s = 0.125 * (k[5:i + 1] @ q[i])
        p = np.exp(s - s.max()) if i >= 5 else np.ones(S)
        want[i] = (p / p.sum()) @ (v[5:i + 1] if i >= 5 else v)
    assert np.abs(to_np(O).astype(np.float64) - want).max() <= 2 * 2.0 ** -11 * 4 + 2.0 ** -11 * 4
