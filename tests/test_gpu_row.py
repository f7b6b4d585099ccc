"""One token of short Q8_0 rows (csrc/gemv_q80_row.hip) equals the fused GEMV word for word.

Up to 8192 rows of at most 2048 elements take the short launch, more rows the
fused kernel: the first rows of a 9000-row matrix computed alone must be the
words the whole matrix gives, at one to 64 blocks a row (16, 32 and 64 lanes a
row, full and not) and row counts around a wave's and a workgroup's, and within
1e-5 of the conditioning scale of the oracle; so must the RMSNorm, SiLU-mul,
residual and gate / up forms.
"""
import numpy as np
import pytest
import torch

import edgexpu_amd as E
import npref
from edgexpu_amd import synth

pytestmark = pytest.mark.gpu
BIG = 9000


def bits(t):
    return t.cpu().numpy().view(np.uint32)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


@pytest.mark.parametrize("n_in", [32, 512, 544, 1024, 1056, 2048])
def test_row_equals_fused(hipdev, ora, n_in):
    rng = np.random.default_rng(n_in)
    w = synth.np_weights(8, BIG, n_in, rng)
    w2 = synth.np_weights(8, BIG, n_in, rng)
    x = synth.np_activations(1, n_in, rng)
    b = rng.normal(0, 0.3, BIG).astype(np.float32)
    r = rng.normal(0, 2, (1, BIG)).astype(np.float32)
    y = dev(rng.normal(0, 1, (1, n_in)).astype(np.float32))
    nw = dev(rng.normal(1, 0.2, n_in).astype(np.float32))
    wd, w2d, xd, bd, rd = dev(w), dev(w2), dev(x), dev(b), dev(r)

    def forms(n):
        ws, bs, rs = wd[:n], bd[:n], rd[:, :n].contiguous()
        return [E.linear_quant_batch(ws, 8, xd, n, n_in, bias=bs),
                E.layer_linear([ws], 8, xd, [n], n_in, norm_weight=nw)[0],
                E.layer_linear([ws], 8, xd, [n], n_in, x2=y, residuals=[rs])[0],
                E.layer_linear([ws], 8, xd, [n], n_in, biases=[bs], residuals=[rs])[0],
                E.gate_up_silu(ws, w2d[:n], 8, xd, n, n_in, norm_weight=nw, b_up=bs),
                E.gate_up_silu(ws, w2d[:n], 8, xd, n, n_in)]

    full = forms(BIG)
    for n in (1, 3, 4, 5, 16, 33):
        for k, (a, c) in enumerate(zip(forms(n), full)):
            assert np.array_equal(bits(a), bits(c[:, :n])), (n, k)
    group = E.linear_quant_group([wd[:5], w2d[:1], wd[5:22]], 8, xd, [5, 1, 17], n_in)
    plain = E.linear_quant_batch(wd, 8, xd, BIG, n_in)
    assert np.array_equal(bits(group[0]), bits(plain[:, :5])) and np.array_equal(bits(group[2]), bits(plain[:, 5:22]))
    xq = ora.quantize_q8_0(x[0])
    want = ora.linear_quant_batch(x, w[:33], 8, b[:33], 1, 33, n_in)
    S = np.array([npref.q8_dot_f64(8, v, xq)[1] for v in w[:33]]) + np.abs(b[:33])
    assert np.all(np.abs(forms(33)[0].cpu().numpy() - want) <= 1e-5 * S)
