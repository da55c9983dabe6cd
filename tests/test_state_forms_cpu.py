"""The forms a state, an address and a stream can be passed in, and host jumps by bytes of the step."""
import ctypes
from types import SimpleNamespace

import numpy as np
import pytest

import mrg8_amd

P = 2**31 - 1
WORDS = [5, 0, P, 1, 2, P - 1, 7, 2**30]


@pytest.mark.parametrize("form", [list, tuple, lambda w: np.array(w, np.uint32), lambda w: np.array(w, np.int64),
                                  lambda w: np.array([w, w], np.uint32).T[:, 0], lambda w: [np.uint32(x) for x in w],
                                  lambda w: [float(x) for x in w]])
def test_state_forms_agree(form, oracle_mod):
    assert mrg8_amd.advance_state(form(WORDS), 12345).tolist() == oracle_mod.jump(np.array(WORDS, np.uint32), 12345).tolist()


@pytest.mark.parametrize("bad", [[1] * 7, (1,) * 9, [-1] + [1] * 7, [2**32] + [1] * 7, np.ones((8, 1), np.uint32)])
def test_bad_states_are_refused(bad):
    with pytest.raises(ValueError):
        mrg8_amd.advance_state(bad, 1)


@pytest.mark.parametrize("step", [0, 1, 7, 8, 255, 256, 257, 0xff00ff, 1 << 32, (1 << 56) + 1, 2**64 - 1])
@pytest.mark.parametrize("state", [WORDS, [0] * 8, [P] * 8, [0, 0, 0, 0, 0, 0, 0, 9], [0, 3, 0, 0, 0, 0, 0, 0]])
def test_host_jump_bytes(step, state, oracle_mod):
    assert mrg8_amd.advance_state(state, step).tolist() == oracle_mod.jump(np.array(state, np.uint32), step).tolist()


@pytest.mark.parametrize("address", [0, 4096, np.int64(1 << 40), np.uint64(2**64 - 4096)])
def test_addresses_and_streams_of_any_integer_type(address):
    want = ctypes.c_void_p(int(address)).value
    for p in (SimpleNamespace(data_ptr=lambda: address), SimpleNamespace(ptr=address), address):
        assert ctypes.c_void_p(mrg8_amd._ptr(p)).value == want
    for s in (SimpleNamespace(cuda_stream=address), SimpleNamespace(handle=int(address)), address):
        got = mrg8_amd._stream(s)
        assert (got if isinstance(got, ctypes.c_void_p) else ctypes.c_void_p(got)).value == want
    assert mrg8_amd._stream(None) is None


@pytest.mark.parametrize("bad", [None, "0", SimpleNamespace(data_ptr=lambda: None), SimpleNamespace(cuda_stream=None)])
def test_what_is_no_address_is_refused(bad):
    with pytest.raises((TypeError, ValueError)):
        ctypes.c_void_p(mrg8_amd._ptr(bad)).value + 0
