"""The planner of the run-time-length transforms, for all lengths (no GPU): factorisation, the
registers and LDS that a launch shape has to hold, the divisions by multiplication, and that the GPU
tests run every launch shape."""

import ctypes

from mr_recon_amd._lib import check, lib
from test_gpu_any_fft_shapes import LENGTHS

LDS = 160 * 1024


def _shape(L):
    s = (ctypes.c_int * 16)()
    check(lib().mra_fft_any_shape(L, s))
    return s[0], s[1], s[2], s[3], s[4], list(s[6:6 + s[5]])


def _largest_prime(n):
    p = 1
    for f in range(2, n + 1):
        while n % f == 0:
            n, p = n // f, f
    return p


def test_lengths_outside_are_refused():
    s = (ctypes.c_int * 16)()
    assert all(lib().mra_fft_any_shape(L, s) != 0 for L in (-1, 0, 1, 641, 1 << 20))


def test_plans():
    for L in range(2, 641):
        M, threads, nt, kind, lds, radices = _shape(L)
        n = 1
        for r in radices:
            # butterflies a thread keeps through a pass: 1 from radix 9, 2 from 5, else 4
            held = 1 if r >= 9 else 2 if r >= 5 else 4
            assert M % r == 0 and held * threads >= M // r * nt
            inv = 2 ** 32 // n + 1
            assert n == 1 or all((j * inv) >> 32 == j // n for j in range(M // r))
            n *= r
        assert n == M
        largest = _largest_prime(L)
        assert kind == (1 if largest > 19 else 2 if largest > 16 else 0)
        assert M == L if kind != 1 else M >= 2 * L - 1 and max(radices) <= 16
        assert threads % nt == 0 and threads <= 1024 and nt in (8, 16)
        assert lds >= 8 * (M * (nt + 1) + M) and lds + 1024 <= LDS  # static arrays: under 1 KB
        inv = 2 ** 32 // L + 1
        assert all((e * inv) >> 32 == e // L for e in range(nt * L))


def test_gpu_tests_reach_every_launch_shape():
    key = lambda L: _shape(L)[1:4]
    assert {key(L) for L in LENGTHS} == {key(L) for L in range(2, 641)}
