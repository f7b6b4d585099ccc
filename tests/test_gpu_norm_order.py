"""RMSNorm's double sum of squares runs in one order wherever a call promises another's words.

The float mean moves with the order of the sum only where the sum falls within
its own rounding error of a midpoint between two floats.  The rows here are
steered there: two elements are set so that the exact mean square is a midpoint
to within half an ulp of the double sum, and the weights so that either
neighbour of the mean is seen in the result (for Q8_0, whose block scales are
rounded to fp16, each block's largest product is put at an fp16 midpoint).
"""
import math

import numpy as np
import pytest
import torch

import edgexpu_amd as E
from edgexpu_amd import synth

pytestmark = pytest.mark.gpu
EPS = np.float32(1e-5)
F = np.float32


def bits(t):
    return t.cpu().numpy().view(np.uint32)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def scale_of(mean):
    return F(1.0) / np.sqrt(F(mean + EPS))


def steered_row(rng, n):
    """(row, the scales of the two floats its mean square lies between), n a power of two."""
    while True:
        x = rng.normal(0, 1, n).astype(F)
        x[:2] = 0.0
        rest = math.fsum(float(v) * float(v) for v in x)
        lo = F((rest + 1.0) / n)
        hi = np.nextafter(lo, F(np.inf))
        r = (float(lo) + float(hi)) / 2 * n - rest  # exact: n is a power of two
        z1 = F(math.sqrt(r))
        while float(z1) ** 2 > r:
            z1 = np.nextafter(z1, F(0))
        x[0], x[1] = z1, F(math.sqrt(r - float(z1) ** 2))
        scales = scale_of(lo), scale_of(hi)
        if scales[0] != scales[1]:
            at = rng.permutation(n)
            return x[at], scales


def telling_weights(rng, x, scales):
    """RMSNorm weights that give each 32-element block another fp16 scale for either row scale."""
    w = rng.uniform(0.9, 1.1, x.size).astype(F)
    for b in range(0, x.size, 32):
        i = b + int(np.argmax(np.abs(x[b:b + 32])))
        v = [F(abs(x[i])) * s for s in scales]
        d = np.float16(1.3 * float(v[0]) / 127)  # w[i] of about 1.3: the block's largest product
        mid = (float(d) + float(np.nextafter(d, np.float16(np.inf)))) / 2
        g = F(mid * 127 / float(v[0]))
        for _ in range(40):
            g = np.nextafter(g, F(0))
        for _ in range(80):
            a, c = (np.float16(F(u * g) / F(127.0)) for u in v)
            if a != c:
                break
            g = np.nextafter(g, F(np.inf))
        w[i] = g
    return w


@pytest.mark.parametrize("n_in", [512, 1024, 2048])
def test_short_q80_rows_equal_the_fused_gemv(hipdev, n_in):
    """One token of few Q8_0 rows (csrc/gemv_q80_row.hip) and of many (the fused
    GEMV): the rows both hold get the same words."""
    rng = np.random.default_rng(n_in)
    big = 9000
    w = dev(synth.np_weights(8, big, n_in, rng))
    for k in range(40):
        x, scales = steered_row(rng, n_in)
        nw, xd = dev(telling_weights(rng, x, scales)), dev(x[None, :])
        few, = E.layer_linear([w[:16]], 8, xd, [16], n_in, norm_weight=nw)
        many, = E.layer_linear([w], 8, xd, [big], n_in, norm_weight=nw)
        assert np.array_equal(bits(few), bits(many[:, :16])), k


@pytest.mark.parametrize("qt", [12, 14, 8])
@pytest.mark.parametrize("n_in", [512, 2048, 8192])
def test_few_token_layer_calls_equal_rmsnorm_and_product(hipdev, qt, n_in):
    """RMSNorm in the few-token pack (csrc/gemm_small.hip) and as a call of its own."""
    rng = np.random.default_rng(qt + n_in)
    m, n_out = 6, 48
    w = dev(synth.np_weights(qt, n_out, n_in, rng))
    for k in range(20):
        rows = [steered_row(rng, n_in) for _ in range(m)]
        x = dev(np.stack([r[0] for r in rows]))
        nw = dev(telling_weights(rng, *rows[0]) if qt == 8 else rng.uniform(0.9, 1.1, n_in).astype(F))
        layer, = E.layer_linear([w], qt, x, [n_out], n_in, norm_weight=nw, eps=float(EPS))
        steps = E.linear_quant_batch(w, qt, E.rmsnorm(x, nw, float(EPS)), n_out, n_in)
        assert np.array_equal(bits(layer), bits(steps)), k
