"""The line between the few-token GEMM and the prefill GEMMs (gemm_small_take in csrc/gemm_small.hip)."""
import ctypes as C

import pytest

import edgexpu_amd as E

# type, rows, K, tokens, measured us of the few-token and of the prefill GEMM
MEASURED = [
    (12, 4096, 4096, 512, 47.0, 51.1), (12, 4096, 4096, 768, 66.1, 62.1), (12, 9728, 2560, 192, 41.7, 44.5),
    (12, 9728, 2560, 256, 51.1, 46.3), (12, 65536, 2560, 32, 46.1, 51.3), (12, 65536, 2560, 48, 73.0, 54.8),
    (12, 12000, 1024, 256, 34.9, 38.1), (12, 12000, 1024, 320, 42.9, 33.0), (12, 28672, 4096, 64, 51.4, 57.3),
    (12, 32000, 4096, 64, 53.3, 61.0), (12, 14336, 4096, 192, 69.0, 58.7), (12, 4096, 14336, 192, 68.7, 83.2),
    (14, 9728, 2560, 64, 30.5, 40.0), (14, 9728, 2560, 128, 48.2, 45.2), (14, 9728, 2560, 192, 72.3, 53.7),
    (14, 2560, 9728, 192, 49.1, 58.3), (14, 2560, 9728, 256, 67.3, 62.2), (14, 1024, 4096, 512, 29.7, 38.8),
    (14, 28672, 4096, 64, 83.7, 120.4), (8, 2560, 2560, 512, 47.9, 42.7), (8, 4096, 4096, 192, 42.0, 48.6),
    (8, 49152, 576, 128, 65.7, 57.3), (8, 1536, 576, 768, 19.1, 25.2), (8, 14336, 4096, 128, 86.2, 89.7),
]


def take(*a):
    f = E.hip().lib._Z15gemm_small_takeiiii
    f.restype = C.c_bool
    f.argtypes = [C.c_int] * 4
    return f(*a)


@pytest.mark.parametrize("qt,n_out,n_in,m,few,prefill", MEASURED)
def test_line_takes_the_faster(qt, n_out, n_in, m, few, prefill):
    """At the shapes measured nearest the line, the kernel it gives is within 10 % of the faster one."""
    assert (few if take(qt, n_out, n_in, m) else prefill) <= 1.1 * min(few, prefill)


def test_line_bounds():
    for qt in (12, 14, 8):
        assert not take(qt, 4096, 4096, 4) and take(qt, 4096, 4096, 5) and take(qt, 128256, 4096, 32)
        assert not take(qt, 1, 256, 64 * 4096 + 1)
    assert not any(take(qt, 64, 256, 64) for qt in (0, 1, 2, 6, 13))
