"""Lengths the chirp-z row transforms take (any_dft_length of
axs_anydft.hpp, host code of the library; no GPU)."""
import ctypes

import pytest

from pyaxisymflow_amd import _lib


def length(n, primes=13):
    f = ctypes.CDLL(_lib.LIB_PATH)["_ZN3axs14any_dft_lengthEiPbi"]
    blue = ctypes.c_bool()
    return f(n, ctypes.byref(blue), primes), blue.value


# the shortest length keeps a lone radix 2 where the next one without it has
# as many stages (or puts a thirteenth wave where twelve were)
@pytest.mark.parametrize("n,l", [(253, 512), (317, 640), (373, 750), (487, 1000), (571, 1152),
                                 (613, 1250), (757, 1536), (3301, 6750)])
def test_shortest_length_where_the_longer_one_is_slower(n, l):
    assert length(n) == (l, True)


# fewer stages; smaller butterflies per thread or more rows in flight
@pytest.mark.parametrize("n,l", [(513, 1125), (677, 1500), (941, 2000), (2049, 4500), (1019, 2160),
                                 (1579, 3375), (1867, 3840), (1949, 4096), (2437, 5120)])
def test_longer_length_where_it_is_faster(n, l):
    assert length(n) == (l, True)


def test_direct_lengths_and_batches():
    assert length(770) == (770, False) and length(770, 5) == (1600, True)
    assert length(2048) == (2048, False) and length(4095) == (4095, False)
    assert length(613, 5) == (1250, True) and length(1025, 5) == (2160, True)
    assert length(4097)[0] > 8192  # refused
