"""Products of a few tokens, and of more against few rows (csrc/gemm_small.hip), against the oracle.

Q4_K, Q6_K and Q8_0 rows on the integer matrix cores, 16 rows by up to 64
tokens per workgroup with K split over its waves: every output within 1e-5 of
its conditioning scale (the block integers are exact; what differs from the
oracle is the order of the f32 sum over blocks), at the edges of the token
tiles (16), the row tiles (16, 32), the K units (one super-block, one 32-element
block, counts that do not divide the waves) and the wave counts (1 to 16).
"""
import ctypes as C

import numpy as np
import pytest
import torch

import edgexpu_amd as E
import npref
from edgexpu_amd import synth

pytestmark = pytest.mark.gpu
TOL = 1e-5


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def quantize(ora, qt, x):
    return np.stack([(ora.quantize_q8_0 if qt == 8 else ora.quantize_q8_k)(r) for r in x])


def scales(qt, w, xq):
    """S[t][i] of the integer dot (float64)."""
    return np.stack([[npref.q8_dot_f64(qt, r, q)[1] for r in w] for q in xq])


@pytest.mark.parametrize("qt,n_in", [(12, 256), (12, 2560), (12, 4352), (14, 256), (14, 2816), (14, 9728), (8, 32),
                                     (8, 576), (8, 2080)])
@pytest.mark.parametrize("m", [5, 16, 17, 33, 64, 70, 100, 131])
def test_small_vs_oracle(hipdev, ora, qt, n_in, m):
    """A group of ragged row counts (one below a tile, one past it, one row),
    with and without bias; equal to the call of each matrix alone and to the
    call over quantized blocks bit for bit.  70 and 100 tokens are five and
    seven token tiles in two blocks, whose last one reads past the pack's."""
    n_outs = (15, 33, 1)
    rng = np.random.default_rng(100 * qt + n_in + m)
    ws = [synth.np_weights(qt, n, n_in, rng) for n in n_outs]
    x = synth.np_activations(m, n_in, rng)
    biases = [rng.normal(0, 0.3, n).astype(np.float32) if z != 1 else None for z, n in enumerate(n_outs)]
    wd, xd = [dev(w) for w in ws], dev(x)
    bd = [None if b is None else dev(b) for b in biases]
    outs = E.linear_quant_group(wd, qt, xd, list(n_outs), n_in, biases=bd)
    xq = quantize(ora, qt, x)
    for z, n in enumerate(n_outs):
        got = outs[z].cpu().numpy()
        want = ora.linear_quant_batch(x, ws[z], qt, biases[z], m, n, n_in)
        S = scales(qt, ws[z], xq) + (0 if biases[z] is None else np.abs(biases[z])[None, :])
        assert np.all(np.abs(got - want) <= TOL * S), f"matrix {z}"
        one = E.linear_quant_batch(wd[z], qt, xd, n, n_in, bias=bd[z]).cpu().numpy()
        assert np.array_equal(bits(got), bits(one)), f"matrix {z} alone"
        blk = E.gemv_q8(wd[z], qt, dev(xq), m, n, n_in, bias=bd[z]).cpu().numpy()
        assert np.array_equal(bits(got), bits(blk)), f"matrix {z} from blocks"


@pytest.mark.parametrize("qt,n_in", [(12, 256), (14, 512), (8, 96)])
@pytest.mark.parametrize("m", [12, 16, 17, 70, 100])
def test_small_many_rows(hipdev, qt, n_in, m):
    """From 8192 rows a wave may take two row tiles: the same words as the rows
    computed in parts below that, the last tiles ragged."""
    n_out = 8203
    rng = np.random.default_rng(qt + m)
    w = dev(synth.np_weights(qt, n_out, n_in, rng))
    x = dev(synth.np_activations(m, n_in, rng))
    got = E.linear_quant_batch(w, qt, x, n_out, n_in).cpu().numpy()
    for r0, r1 in ((0, 3000), (3000, 8170), (8170, n_out)):
        part = E.linear_quant_batch(w[r0:r1].contiguous(), qt, x, r1 - r0, n_in).cpu().numpy()
        assert np.array_equal(bits(got[:, r0:r1]), bits(part)), r0


@pytest.mark.parametrize("qt,n_in,n_out", [(12, 4096, 8200), (14, 2560, 300), (8, 576, 100)])
@pytest.mark.parametrize("m", [7, 40])
def test_small_layer_calls_equal_the_steps(hipdev, qt, n_in, n_out, m):
    """RMSNorm and SiLU-mul in the pack, the residual in the store (also over
    itself) and the gate / up pair: equal to the separate device calls bit for
    bit.  An output that overlaps another matrix's residual takes the steps,
    where every product is complete before a residual is read."""
    rng = np.random.default_rng(qt + n_in + m)
    w, w2 = (dev(synth.np_weights(qt, n_out, n_in, rng)) for _ in range(2))
    x, y = (dev(rng.normal(0, 1, (m, n_in)).astype(np.float32)) for _ in range(2))
    nw = dev(rng.normal(1, 0.2, n_in).astype(np.float32))
    b, b2 = (dev(rng.normal(0, 0.5, n_out).astype(np.float32)) for _ in range(2))
    res = dev(rng.normal(0, 4, (m, n_out)).astype(np.float32))

    def eq(a, c):
        assert np.array_equal(bits(a.cpu().numpy()), bits(c.cpu().numpy()))

    lin = lambda a, ww, bb: E.linear_quant_batch(ww, qt, a, n_out, n_in, bias=bb)  # noqa: E731
    norm = E.rmsnorm(x, nw, 1e-5)
    r = res.clone()
    E.layer_linear([w], qt, x, (n_out,), n_in, norm_weight=nw, biases=[b], residuals=[r], outs=[r])
    eq(r, E.add(res, lin(norm, w, b)))
    got, = E.layer_linear([w], qt, x, (n_out,), n_in, x2=y, residuals=[res])
    eq(got, E.add(res, lin(E.silu_mul(x, y), w, None)))
    act = E.gate_up_silu(w, w2, qt, x, n_out, n_in, norm_weight=nw, b_gate=b, b_up=b2)
    eq(act, E.silu_mul(lin(norm, w, b), lin(norm, w2, b2)))
    # out 0 is matrix 1's residual
    o0, o1 = res.clone(), torch.empty_like(res)
    E.layer_linear([w, w2], qt, x, (n_out, n_out), n_in, residuals=[res, o0], outs=[o0, o1])
    eq(o0, E.add(res, lin(x, w, None)))
    eq(o1, E.add(o0, lin(x, w2, None)))


def takes_small(qt, n_out, n_in, m):
    """The dispatch rule itself (gemm_small_take in csrc/gemm_small.hip)."""
    f = E.hip().lib._Z15gemm_small_takeiiii
    f.restype = C.c_bool
    f.argtypes = [C.c_int] * 4
    return f(qt, n_out, n_in, m)


@pytest.mark.parametrize("qt,n_in,n_outs,m", [(12, 2560, (9728, 1024, 9728), 300), (14, 2560, (9728, 300), 200),
                                              (8, 2048, (20000, 40), 200)])
def test_group_equals_each_matrix_across_the_line(hipdev, qt, n_in, n_outs, m):
    """Past 64 tokens a group may hold matrices on either side of the line to
    the prefill GEMM: each gives the words of its own call, plain, as a layer
    call and as a gate / up pair."""
    taken = [takes_small(qt, n, n_in, m) for n in n_outs]
    assert True in taken and False in taken
    rng = np.random.default_rng(qt + m)
    wd = [dev(synth.np_weights(qt, n, n_in, rng)) for n in n_outs]
    bd = [dev(rng.normal(0, 0.3, n).astype(np.float32)) for n in n_outs]
    rd = [dev(rng.normal(0, 3, (m, n)).astype(np.float32)) for n in n_outs]
    x = dev(synth.np_activations(m, n_in, rng))
    nw = dev(rng.normal(1, 0.2, n_in).astype(np.float32))

    def eq(a, b, what):
        assert np.array_equal(bits(a.cpu().numpy()), bits(b.cpu().numpy())), what

    group = E.linear_quant_group(wd, qt, x, list(n_outs), n_in, biases=bd)
    layer = E.layer_linear(wd, qt, x, list(n_outs), n_in, norm_weight=nw, biases=bd, residuals=rd)
    for z, n in enumerate(n_outs):
        eq(group[z], E.linear_quant_batch(wd[z], qt, x, n, n_in, bias=bd[z]), ("group", z))
        eq(layer[z], E.layer_linear([wd[z]], qt, x, [n], n_in, norm_weight=nw, biases=[bd[z]],
                                    residuals=[rd[z]])[0], ("layer", z))
    n = n_outs[0]
    up = wd[0].flip(0).contiguous()
    gu = E.linear_quant_group([wd[0], up], qt, x, [n, n], n_in)
    for z, w in enumerate((wd[0], up)):
        eq(gu[z], E.linear_quant_batch(w, qt, x, n, n_in), ("pair", z))
    eq(E.gate_up_silu(wd[0], up, qt, x, n, n_in), E.silu_mul(gu[0], gu[1]), "gate_up_silu")


@pytest.mark.parametrize("m", [8, 40])
def test_group_with_a_matrix_at_another_address(hipdev, m):
    """Q4_K blocks off a 16-byte address keep to the GEMV; the other matrices
    of their group give the words of their own calls."""
    n_out, n_in = 100, 2560
    rng = np.random.default_rng(m)
    w = [synth.np_weights(12, n_out, n_in, rng) for _ in range(2)]
    x = dev(synth.np_activations(m, n_in, rng))
    off = torch.empty(w[1].size + 16, dtype=torch.uint8, device="cuda:0")
    off[4:4 + w[1].size] = dev(w[1].reshape(-1))
    wd = [dev(w[0]), off[4:4 + w[1].size]]
    group = E.linear_quant_group(wd, 12, x, [n_out, n_out], n_in)
    for z in range(2):
        one = E.linear_quant_batch(wd[z], 12, x, n_out, n_in)
        assert np.array_equal(bits(group[z].cpu().numpy()), bits(one.cpu().numpy())), z


@pytest.mark.parametrize("qt,n_in", [(12, 2560), (14, 2560), (8, 576)])
def test_small_special_activations(hipdev, ora, qt, n_in):
    """Tokens holding zeros, infinities and NaN: finite tokens beside them are
    untouched, and each output is finite exactly where the one-token call's is."""
    m, n_out = 9, 40
    rng = np.random.default_rng(qt)
    w = synth.np_weights(qt, n_out, n_in, rng)
    x = synth.np_activations(m, n_in, rng)
    x[1] = 0.0
    x[3, 5] = np.inf
    x[4, 300] = np.nan
    x[6, :40] = 1e-40
    got = E.linear_quant_batch(dev(w), qt, dev(x), n_out, n_in).cpu().numpy()
    for t in range(m):
        one = E.linear_quant_batch(dev(w), qt, dev(x[t:t + 1]), n_out, n_in).cpu().numpy()[0]
        assert np.array_equal(np.isfinite(got[t]), np.isfinite(one)), t
    fin = np.isfinite(x).all(axis=1)
    want = ora.linear_quant_batch(x[fin], w, qt, None, int(fin.sum()), n_out, n_in)
    assert np.all(np.abs(got[fin] - want) <= TOL * scales(qt, w, quantize(ora, qt, x[fin])))
