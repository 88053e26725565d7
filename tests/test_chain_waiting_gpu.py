"""Lane chaining and promises that wait: a group whose lanes hold promises that
requeue themselves until another one has run still makes that one. Numbers
around those at which lanes go on without looking for work (60), up to the 63
that leave a link of the stash open."""

import ctypes

import pytest

import harmonize_amd as hz

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("waiting", [0, 1, 59, 60, 61, 63])
@pytest.mark.parametrize("cycles", [1 << 16, 500])
def test_waiting_lanes_let_work_be_made(waiting, mixed, cycles):
    passed = ctypes.c_uint32()
    hz.check(hz.lib().hz_wait_selftest(waiting, mixed, cycles, 4, ctypes.byref(passed)), "hz_wait_selftest")
    assert passed.value == waiting
