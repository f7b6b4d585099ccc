"""The few-token GEMM's workspace (csrc/shim.hip) under captured graphs.

A captured call holds the workspace's address.  Later calls with larger packs,
of more tokens or of longer rows, must leave that memory allocated and to
itself: every replay equals the eager result bit for bit, with the larger calls
and fresh tensors that would land in freed memory between the replays.
"""
import numpy as np
import pytest
import torch

import edgexpu_amd as E
from edgexpu_amd import synth

pytestmark = pytest.mark.gpu


def bits(t):
    return t.cpu().numpy().view(np.uint32)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


@pytest.fixture
def fresh(hipdev):
    """The library with no workspace yet (earlier tests may have grown it)."""
    torch.cuda.synchronize()
    hipdev.shutdown()
    hipdev.check(hipdev.init(0), "init")
    return hipdev


# larger packs than 4 MiB: more tokens, and the longest rows 15 tokens can have below that
LARGER = [(1024, 4096), (1500, 4096), (15, 65536)]


@pytest.mark.parametrize("m", [8, 40])
def test_captured_call_survives_larger_calls(fresh, m):
    rng = np.random.default_rng(m)
    n_outs, n_in = (48, 16, 16), 4096
    ws = [dev(synth.np_weights(12, n, n_in, rng)) for n in n_outs]
    x = dev(synth.np_activations(m, n_in, rng))
    want = [o.clone() for o in E.linear_quant_group(ws, 12, x, list(n_outs), n_in)]
    outs = [torch.empty_like(o) for o in want]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        E.linear_quant_group(ws, 12, x, list(n_outs), n_in, outs=outs)
    for big_m, big_k in LARGER:
        wb = dev(synth.np_weights(12, 16, big_k, rng))
        xb = dev(synth.np_activations(big_m, big_k, rng))
        first = E.linear_quant_batch(wb, 12, xb, 16, big_k)
        junk = [torch.full((1 << 20,), float("nan"), device="cuda:0") for _ in range(8)]
        for rep in range(3):
            for o in outs:
                o.fill_(float("nan"))
            graph.replay()
            again = E.linear_quant_batch(wb, 12, xb, 16, big_k)
            torch.cuda.synchronize()
            for z, (o, r) in enumerate(zip(outs, want)):
                assert np.array_equal(bits(o), bits(r)), (big_m, big_k, rep, z)
            assert np.array_equal(bits(again), bits(first)), (big_m, big_k, rep)
        assert all(bool(torch.isnan(j).all()) for j in junk), "a replay wrote into another tensor"


@pytest.mark.parametrize("qt", [8, 12, 14])
def test_decode_and_prefill_on_two_streams(fresh, qt):
    """A few-token call of a decode step beside one of a prefill, each on its
    own stream: the two packs are in different buffers, so every result is
    that of the call alone."""
    rng = np.random.default_rng(qt)
    n_out, n_in = 48, 4096
    w = dev(synth.np_weights(qt, n_out, n_in, rng))
    xs = [dev(synth.np_activations(m, n_in, rng)) for m in (8, 15, 700)]
    want = [E.linear_quant_batch(w, qt, x, n_out, n_in).clone() for x in xs]
    torch.cuda.synchronize()
    decode, prefill = torch.cuda.Stream(), torch.cuda.Stream()
    got = [[torch.empty_like(o) for _ in range(40)] for o in want]
    for i in range(40):
        with torch.cuda.stream(prefill):
            E.linear_quant_batch(w, qt, xs[2], n_out, n_in, out=got[2][i])
        with torch.cuda.stream(decode):
            for z in (0, 1):
                E.linear_quant_batch(w, qt, xs[z], n_out, n_in, out=got[z][i])
    torch.cuda.synchronize()
    for z, o in enumerate(want):
        for i in range(40):
            assert np.array_equal(bits(got[z][i]), bits(o)), (z, i)


@pytest.mark.parametrize("m", [8, 40])
def test_capture_before_any_few_token_call(fresh, m):
    """Captured with the other paths' workspaces in place but no earlier call
    of a few tokens: the capture succeeds, and every replay is the eager result."""
    rng = np.random.default_rng(m)
    n_out, n_in = 48, 4096
    w = dev(synth.np_weights(12, n_out, n_in, rng))
    x = dev(synth.np_activations(m, n_in, rng))
    E.logits(w, 12, x[:1].contiguous(), n_out, n_in)
    out = torch.empty((m, n_out), device="cuda:0")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):  # global capture mode
        E.linear_quant_batch(w, 12, x, n_out, n_in, out=out)
    want = E.linear_quant_batch(w, 12, x, n_out, n_in)
    for rep in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(bits(out), bits(want)), rep
