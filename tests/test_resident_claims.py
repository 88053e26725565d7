"""Claims from a job-table entry of the resident program while its job is
replaced: in every order of the accesses (specs/claim_word.h, on the host) each
item of the new job is granted once, with that job's fields. The order of
accesses that reads the limit after the add, planted in the oracle, is found."""

import ctypes

import oracle_lib as O


def orders(planted):
    f = O.lib().oracle_claim_orders
    f.restype, f.argtypes = ctypes.c_uint64, [ctypes.c_int, ctypes.POINTER(ctypes.c_uint64)]
    wrong = ctypes.c_uint64()
    return f(planted, ctypes.byref(wrong)), wrong.value


def test_no_order_grants_an_item_twice():
    n, wrong = orders(0)
    assert n > 100 and wrong == 0


def test_a_limit_read_after_the_add_is_found():
    n, wrong = orders(1)
    assert 0 < wrong < n
