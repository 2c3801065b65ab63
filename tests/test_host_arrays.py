"""Pointer arrays and records of the host entries: a stack gives the addresses that its
images give one by one, and what was refused stays refused."""
import ctypes

import numpy as np
import pytest

from isac_amd import binding


@pytest.mark.parametrize("shape", [(1, 4, 4), (5, 3, 3), (7, 16)])
def test_stack_addresses(shape):
    x = np.zeros(shape, np.float32)
    a, b = binding.get_c_ptr_array(x), binding.get_c_ptr_array([x[i] for i in range(shape[0])])
    assert type(a) is type(b)
    for p, q in zip(a, b):
        assert ctypes.addressof(p.contents) == ctypes.addressof(q.contents)


@pytest.mark.parametrize("bad", [np.zeros((3, 4, 4)), np.zeros((3, 4, 8), np.float32)[:, :, ::2]])
def test_stack_refusals(bad):
    with pytest.raises(AssertionError):
        binding.get_c_ptr_array(bad)


def test_params_round_trip():
    prm = (binding.AlignParam * 3)()
    ptr = ctypes.cast(prm, ctypes.POINTER(binding.AlignParam))
    acc = np.array([[0.1, -2.5], [1e-9, 3.0], [7.0, 0.3]])
    binding._set_shifts(ptr, acc)
    prm[1].mirror, prm[2].angle, prm[0].ref_id = True, 12.5, 4
    got = binding.params_to_numpy(ptr, 3)
    np.testing.assert_array_equal(got["shift_x"], acc[:, 0].astype(np.float32))
    np.testing.assert_array_equal(got["shift_y"], acc[:, 1].astype(np.float32))
    assert got["mirror"].tolist() == [0, 1, 0] and got["mirror"].dtype == np.int32
    assert got["angle"].tolist() == [0.0, 0.0, 12.5] and got["ref_id"].tolist() == [4, 0, 0]
