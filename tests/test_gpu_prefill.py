"""The prefill GEMMs (csrc/gemm.hip, gemm_kq.hip, gemm_g32.hip) where Q4_K, Q6_K and Q8_0 calls reach them.

Fewer rows or tokens take the few-token GEMM, so every case here first asserts
that the dispatch rule leaves it to the prefill GEMM of its format: ragged rows
and tokens, one super-block, rows that end inside a record, the K split and none,
two chains per super-block, quantized input, exact integers.  Outputs are checked
at a sample of rows (the first and last tiles' among them) and every token
against the float64 restatement, and at a few tokens against the oracle.
"""
import ctypes as C

import numpy as np
import pytest
import torch

import edgexpu_amd as E
import npref
from edgexpu_amd import synth
from test_gpu_parity import _q4k_headers, _q80_rows, _q8k_rows, assert_tol, bits, dev, special_blocks

pytestmark = pytest.mark.gpu

SHAPES = {
    12: [(14336, 1030, 897), (4096, 4099, 577), (2560, 50001, 33), (1024, 2000, 1700), (256, 16385, 500)],
    14: [(2560, 2570, 513), (9728, 1100, 577), (256, 8321, 700), (1024, 3001, 640), (14336, 150, 4300)],
    8: [(576, 1537, 2300), (96, 16385, 1100), (4096, 4097, 300), (14336, 770, 800), (160, 9999, 1200)],
}


def assert_prefill(qt, n_out, n_in, m):
    f = E.hip().lib._Z15gemm_small_takeiiii
    f.restype = C.c_bool
    f.argtypes = [C.c_int] * 4
    assert not f(qt, n_out, n_in, m), "the few-token GEMM takes this shape"


def sample_rows(n_out, rng):
    if n_out <= 300:
        return np.arange(n_out)
    ends = np.r_[0:40, n_out - 40:n_out]
    return np.unique(np.r_[ends, rng.choice(n_out, 220, replace=False)])


def f64(qt, w, xq):
    return (npref.g32_q80_gemm_f64 if qt == 8 else npref.kq_q8k_gemm_f64)(qt, w, xq)


def f64_gemm(qt, w, xq):
    return npref.q4k_q8k_gemm_f64(w, xq) if qt == 12 else f64(qt, w, xq)


@pytest.mark.parametrize("qt,n_in,n_out,m", [(qt, *s) for qt, v in SHAPES.items() for s in v])
def test_prefill_shapes(hipdev, ora, qt, n_in, n_out, m):
    """f32 and quantized input give the same bits, twice in a row (the K split's
    arrival counters are back at zero), within the bound of both references."""
    assert_prefill(qt, n_out, n_in, m)
    rng = np.random.default_rng(qt + n_in + n_out + m)
    w = synth.np_weights(qt, n_out, n_in, rng)
    x = synth.np_activations(m, n_in, rng)
    bias = rng.normal(0, 0.5, n_out).astype(np.float32)
    wd, xd, bd = dev(w), dev(x), dev(bias)
    got = E.linear_quant_batch(wd, qt, xd, n_out, n_in, bias=bd)
    again = E.linear_quant_batch(wd, qt, xd, n_out, n_in, bias=bd)
    xq = _q80_rows(ora, x) if qt == 8 else _q8k_rows(ora, x)
    blocks = E.gemv_q8(wd, qt, dev(xq), m, n_out, n_in, bias=bd)
    assert torch.equal(got.view(torch.int32), again.view(torch.int32))
    assert torch.equal(got.view(torch.int32), blocks.view(torch.int32))
    rows = sample_rows(n_out, rng)
    got = got.cpu().numpy()[:, rows]
    exact, S = f64_gemm(qt, w[rows], xq)
    S = S + np.abs(bias[rows])[None, :]
    assert_tol(got, (exact + bias[rows][None, :].astype(np.float64)).astype(np.float32), S, "vs float64")
    tok = np.r_[0, m - 1, rng.choice(m, 2, replace=False)]
    want = ora.linear_quant_batch(x[tok], w[rows], qt, bias[rows], tok.size, rows.size, n_in)
    assert_tol(got[tok], want, S[tok], "vs oracle")


@pytest.mark.parametrize("n_in,n_out,m", [(2048, 4224, 900), (14336, 256, 3500)])
def test_prefill_q4k_integers_exact(hipdev, n_in, n_out, m):
    """Unit scales and activations that are their own Q8_K codes: every fp32
    step is exact, so the output is the integer closed form, with the K range
    unsplit (136 tiles) and split in four (28 tiles)."""
    assert_prefill(12, n_out, n_in, m)
    rng = np.random.default_rng(5150 + n_out)
    w = _q4k_headers(synth.np_weights(12, n_out, n_in, rng), 1.0, 1.0)
    x = rng.integers(-127, 128, (m, n_in)).astype(np.float32)
    x.reshape(m, -1, 256)[:, :, 0] = -127.0
    got = E.linear_quant_batch(dev(w), 12, dev(x), n_out, n_in).cpu().numpy()
    rows = sample_rows(n_out, rng)
    xq = np.stack([npref.quantize_q8_k(x[t]) for t in range(m)])
    want, _ = npref.q4k_q8k_gemm_f64(w[rows], xq)
    assert np.abs(want).max() < 2**24
    assert np.array_equal(got[:, rows].astype(np.float64), want)


@pytest.mark.parametrize("qt,n_in,n_out,m", [(14, 512, 3001, 1000), (8, 640, 4001, 800)])
def test_prefill_integers_exact(hipdev, qt, n_in, n_out, m):
    """The same for Q6_K (largest and smallest scales included) and Q8_0 (code -128 in every block)."""
    assert_prefill(qt, n_out, n_in, m)
    rng = np.random.default_rng(4500 + qt)
    w = synth.np_weights(qt, n_out, n_in, rng)
    one = np.array([1.0], np.float16).view(np.uint8)
    x = rng.integers(-127, 128, (m, n_in)).astype(np.float32)
    if qt == 14:
        wb = w.reshape(n_out, -1, 210)
        wb[:, :, 208:210] = one
        sc = wb[:, :, 192:208].view(np.int8)
        sc[:, :, 0], sc[:, :, 1] = -128, 127
        x.reshape(m, -1, 256)[:, :, 0] = -127.0
        xq = np.stack([npref.quantize_q8_k(v) for v in x])
    else:
        wb = w.reshape(n_out, -1, 34)
        wb[:, :, 0:2] = one
        wb[:, :, 2] = 0x80
        x.reshape(m, -1, 32)[:, :, 5] = 127.0
        xq = np.stack([npref.quantize_q8_0(v) for v in x])
    got = E.linear_quant_batch(dev(w), qt, dev(x), n_out, n_in).cpu().numpy()
    rows = sample_rows(n_out, rng)
    want, _ = f64(qt, w[rows], xq)
    assert np.abs(want).max() < 2**24
    assert np.array_equal(got[:, rows].astype(np.float64), want)


def test_prefill_two_chains(hipdev, ora):
    """Tokens whose Q8_K codes are all +-127 (sum |q8| = 32512 per super-block,
    beyond the 17753 one exact chain allows) run every super-block as two
    chains; rows with every scale and min 63 and every code 15 push sumi to
    30.7 M.  Ordinary tokens beside them in the same and in other blocks."""
    n_in, n_out, m = 2048, 6000, 500
    assert_prefill(12, n_out, n_in, m)
    rng = np.random.default_rng(6161)
    w = synth.np_weights(12, n_out, n_in, rng)
    for o in (0, 1, 150, n_out - 1):
        w[o].reshape(-1, 144)[:, 4:144] = 0xFF
    x = synth.np_activations(m, n_in, rng)
    x[:150] = np.where(rng.random((150, n_in)) < 0.5, -1.0, 1.0).astype(np.float32)
    x[:150] *= rng.uniform(0.5, 2.0, (150, 1)).astype(np.float32)
    got = E.linear_quant_batch(dev(w), 12, dev(x), n_out, n_in).cpu().numpy()
    rows = np.unique(np.r_[0, 1, 150, sample_rows(n_out, rng)])
    exact, S = npref.q4k_q8k_gemm_f64(w[rows], _q8k_rows(ora, x))
    assert_tol(got[:, rows], exact.astype(np.float32), S, "two chains vs float64")
    want = ora.linear_quant_batch(x[:4], w[rows], 12, None, 4, rows.size, n_in)
    assert_tol(got[:4][:, rows], want, S[:4], "two chains vs oracle")


@pytest.mark.parametrize("qt,n_out", [(12, 2100), (14, 1100)])
def test_prefill_special_blocks(hipdev, ora, qt, n_out):
    """The prefill pack's Q8_K quantization of blocks a quantizer can go wrong
    on (zeros, ties of opposite sign, NaN, subnormals, .5 ties), bit for bit the
    GEMM over the oracle's Q8_K bytes."""
    n_in, m = 1024, 1637
    assert_prefill(qt, n_out, n_in, m)
    rng = np.random.default_rng(4242 + qt)
    x = special_blocks(m, n_in, rng)
    w = synth.np_weights(qt, n_out, n_in, rng)
    bias = rng.normal(0, 0.5, n_out).astype(np.float32)
    wd, bd = dev(w), dev(bias)
    got = E.linear_quant_batch(wd, qt, dev(x), n_out, n_in, bias=bd).cpu().numpy()
    want = E.gemv_q8(wd, qt, dev(_q8k_rows(ora, x)), m, n_out, n_in, bias=bd).cpu().numpy()
    assert np.array_equal(bits(got), bits(want))
    tok = [t for t in range(12) if np.isfinite(x[t]).all()]
    rows = sample_rows(n_out, rng)
    ref = ora.linear_quant_batch(x[tok], w[rows], qt, bias[rows], len(tok), rows.size, n_in)
    _, S = f64_gemm(qt, w[rows], _q8k_rows(ora, x[tok]))
    assert_tol(got[tok][:, rows], ref, S + np.abs(bias[rows])[None, :], "special blocks vs oracle")
