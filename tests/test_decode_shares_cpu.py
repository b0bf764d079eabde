"""Which decode steps of 1 to 4 sequences multiply with the output projection inside the attention (vy_dec_shares_pay of
vyomai_amd/csrc/vy_runtime.hip): those that it makes faster."""
import ctypes as C

import pytest


def pays(B, h, hk, S):
    from vyomai_amd import _lib
    rule = _lib.load()._Z17vy_dec_shares_payiiil
    rule.argtypes, rule.restype = [C.c_int, C.c_int, C.c_int, C.c_int64], C.c_bool
    return rule(B, h, hk, 2 * B * hk * S * 64 * 2)


@pytest.mark.parametrize("h,hk,B,short,long", [
    # heads, key heads, sequences; behind 60 and behind 600 tokens
    (12, 12, 1, True, True), (12, 4, 1, True, True), (16, 16, 1, False, False), (16, 8, 1, False, True), (16, 2, 1, False, False),
    (8, 8, 4, True, True), (12, 12, 2, True, True), (12, 12, 3, False, False), (12, 12, 4, False, False), (12, 6, 4, True, True),
    (16, 16, 2, False, False), (16, 8, 2, False, False), (16, 4, 4, False, False), (16, 2, 3, False, False),
    (12, 4, 2, False, True), (12, 4, 4, False, True), (12, 3, 2, False, False), (12, 3, 3, False, True), (8, 2, 4, False, True),
    (12, 2, 2, True, True), (12, 2, 4, False, True), (12, 1, 3, False, False), (8, 1, 4, True, True)])
def test_rule(h, hk, B, short, long):
    assert (pays(B, h, hk, 60), pays(B, h, hk, 600)) == (short, long)
