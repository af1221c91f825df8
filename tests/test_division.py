"""The kernels' 64-bit division (``csrc/gd_divide.h``), compiled for the host, against integer division: the same steps with a reciprocal that is off
by as much as the hardware's may be (CPU only)."""

from __future__ import annotations

import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "env-gradoom-turbo-torch_amd", "csrc")

DRIVER = r"""
#include "gd_divide.h"
#include <cstdint>

static std::uint64_t state;
static std::uint64_t next() { state ^= state << 13; state ^= state >> 7; state ^= state << 17; return state; }
static std::uint64_t of_bits(int bits) { return bits == 0 ? 0 : (next() >> (64 - bits)) | (1ULL << (bits - 1)); }

static long long expected(long long a, long long b) { return b == 0 ? 0 : (b == -1 ? (long long)(0 - (std::uint64_t)a) : a / b); }

// How many of the quotients are wrong where the reciprocal is off by up to `off` of its value (either way, by `off` itself half of the time).
extern "C" long long wrong_quotients(std::uint64_t seed, long long pairs, int most_bits, double off) {
    state = seed;
    long long wrong = 0;
    auto check = [&](std::uint64_t ua, std::uint64_t ub) {
        const std::uint64_t coin = next();
        const double part = (coin & 1) ? 1.0 : (double)(next() >> 11) * 0x1p-53, error = (coin & 2) ? off * part : -off * part;
        auto reciprocal = [error](double d) { const double r = 1.0 / d; return r + r * error; };
        const long long a = (long long)((coin & 4) ? 0 - ua : ua), b = (long long)((coin & 8) ? 0 - ub : ub);
        wrong += truncated_quotient(a, b, reciprocal) != expected(a, b);
    };
    for (long long k = 0; k < pairs; ++k) {
        const std::uint64_t b = of_bits(1 + (int)(next() % (unsigned)most_bits));
        check(of_bits((int)(next() % (unsigned)(most_bits + 1))), b);
        // about a multiple of the divisor, the largest quotients among them
        const std::uint64_t top = ((1ULL << most_bits) - 1) / b, many = (next() & 1) ? top - next() % (top < 4 ? top + 1 : 4) : next() % (top + 1), near = many * b;
        check(near, b);
        check(near + 1, b);
        check(near ? near - 1 : 0, b);
    }
    // about the magnitude from which on the other way is taken, the largest ones, and nothing
    const std::uint64_t ends[] = {0, 1, 2, 3, 5, (1ULL << 26) - 1, 1ULL << 26, (1ULL << 51) - 1, 1ULL << 51, (1ULL << 52) - 3, (1ULL << 52) - 1, 1ULL << 52, (1ULL << 52) + 1,
                                  (1ULL << 62) + 1, (1ULL << 63) - 1, 1ULL << 63};
    for (std::uint64_t a : ends) for (std::uint64_t b : ends) for (int k = 0; k < 16; ++k) check(a, b);
    return wrong;
}
"""


@pytest.fixture(scope="module")
def wrong_quotients(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("division") / "libdivision.so")
    command = ["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fno-fast-math", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-D__device__=", "-D__forceinline__=inline",
               "-I", CSRC, "-x", "c++", "-o", path, "-"]
    subprocess.run(command, input=DRIVER, text=True, check=True)
    function = C.CDLL(path).wrong_quotients
    function.restype = C.c_longlong
    function.argtypes = [C.c_uint64, C.c_longlong, C.c_int, C.c_double]
    return function


# The instruction is off by 2^-24.3 of the value at most over 2.1e9 divisors; the steps are good for 2^-22 by their argument.
@pytest.mark.parametrize("off", [0.0, 2.0**-53, 2.0**-30, 2.0**-24, 2.0**-22])
def test_quotients_are_those_of_integer_division(wrong_quotients, off):
    assert wrong_quotients(12345, 400_000, 52, off) == 0        # float64 arithmetic
    assert wrong_quotients(54321, 20_000, 63, off) == 0         # both ways


def test_a_reciprocal_of_a_few_bits_is_found_out(wrong_quotients):
    assert wrong_quotients(12345, 20_000, 52, 2.0**-6) > 0
