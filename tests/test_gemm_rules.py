"""The rule that sends a model's projection to the few-row GEMM or to the library, and hk_linear to its few-row
or its 256 x 256 tiles: products measured on both sides, of which the rule has to take the faster one. Runs the cost
function of the built library on the CPU."""
import ctypes as C

import pytest

from huncho_amd import abi

STORE, RESIDUAL, SWIGLU = 0, 1, 2


class GemmArgs(C.Structure):
    _fields_ = [("x", C.c_void_p), ("w", C.c_void_p), ("c", C.c_void_p), ("y", C.c_void_p), ("ldx", C.c_long),
                ("ldw", C.c_long), ("ldc", C.c_long), ("ldy", C.c_long), ("M", C.c_int), ("N", C.c_int), ("K", C.c_int),
                ("w2", C.c_void_p), ("y2", C.c_void_p), ("ldy2", C.c_long), ("N2", C.c_int)]


def few_us(epi, m, n, k):
    f = abi.lib().hk_gemm_few_rows_cost
    f.restype, f.argtypes = C.c_float, [C.c_int, C.POINTER(GemmArgs)]
    return 2.2 + k / 1024 * f(epi, C.byref(GemmArgs(M=m, N=n, K=k)))


def library_us(m, n, k):
    return 5 + 2.2 * k / 1024 + 1.8e-9 * m * n * k


def native_us(m, n, k):
    return 30 * k / 1024 * -(-(n // 256 * -(-m // 256)) // 256)


# rows, columns, K: measured us on the few-row kernel's best tile, and on the other
@pytest.mark.parametrize("epi,m,n,k,few,library", [
    (STORE, 1024, 8192, 1024, 30.4, 21.7), (RESIDUAL, 2048, 1024, 3584, 27.9, 25.4), (RESIDUAL, 4096, 1024, 3584, 46.1, 36.6),
    (RESIDUAL, 4096, 1024, 2048, 26.4, 22.3), (RESIDUAL, 2704, 768, 1152, 14.6, 12.7), (RESIDUAL, 4096, 768, 1152, 16.7, 14.8),
    (RESIDUAL, 4096, 768, 768, 13.4, 11.9),
    (STORE, 169, 8192, 1024, 9.3, 12.7), (RESIDUAL, 169, 1024, 3584, 10.8, 11.2), (RESIDUAL, 512, 1024, 3584, 13.2, 17.4),
    (STORE, 300, 8192, 1024, 12.3, 14.1), (RESIDUAL, 1700, 768, 1152, 9.6, 10.6), (STORE, 16384, 32, 1024, 5.4, 10.1)])
def test_projections(epi, m, n, k, few, library):
    assert (few_us(epi, m, n, k) <= 0.93 * library_us(m, n, k)) == (few < library)


def test_the_pinned_choices_are_reached():
    """The shapes of the full scoring batch keep the library's solution that was chosen for them by timing."""
    for epi, n, k in ((STORE, 8192, 1024), (STORE, 32, 1024), (RESIDUAL, 1024, 2048), (RESIDUAL, 1024, 3584)):
        assert few_us(epi, 32768, n, k) > 0.93 * library_us(32768, n, k)


@pytest.mark.parametrize("epi,m,n,k,few,native", [
    (RESIDUAL, 8192, 1024, 3584, 88, 109), (SWIGLU, 2704, 7168, 1024, 66.0, 61.1), (SWIGLU, 4096, 7168, 1024, 97.7, 72.3),
    (RESIDUAL, 4096, 1024, 3584, 46.1, 98.8), (SWIGLU, 1024, 7168, 1024, 28.2, 35.3), (RESIDUAL, 6000, 1024, 3584, 67.8, 99.4)])
def test_linear(epi, m, n, k, few, native):
    assert (few_us(epi, m, n, k) - 2.2 < native_us(m, n, k)) == (few < native)
