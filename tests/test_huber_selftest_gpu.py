"""The TV layer's Huber terms from one transcendental instruction: the bits of the IEEE root and divisions for every square of a
norm from 2^-96 to 2^80, and for 0."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def test_huber_terms_match_ieee_on_the_gpu():
    from customnetworklayers_amd._lib import last_error, lib

    out = (ctypes.c_ulonglong * 4)()
    rc = lib.inpaint_selftest_huber(out)
    assert rc == 0, last_error()
    print("mismatches: forward factor %d, adjoint %d; %d reciprocals off, wrong quotients by them %d" % tuple(out), flush=True)
    assert out[0] == out[1] == out[3] == 0
    assert 0 < out[2] <= 4096  # all of them were listed, and their quotients checked
