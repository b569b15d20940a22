"""Which test sets an evaluation refuses (the check itself, on the CPU)."""
import warnings

import numpy as np
import pytest
import torch

GOOD = [[0, 0, 9], [9, 2, 0], [4, 1, 4]]


@pytest.mark.parametrize("dtype", [np.int64, np.int32, np.uint8, np.uint64, np.float64])
def test_ids_inside_the_tables_become_int64(dtype):
    from dicee_amd.evaluator import check_triple_ids
    for t in (np.array(GOOD, dtype=dtype), np.array(GOOD, dtype=dtype, order="F"), np.zeros((0, 3), dtype=dtype)):
        ids = check_triple_ids(t, 10, 3)
        assert ids.dtype == np.int64 and ids.flags.c_contiguous
        np.testing.assert_array_equal(ids, t.astype(np.int64))


@pytest.mark.parametrize("bad", [(0, 10), (0, -1), (1, 3), (1, -1), (2, 10), (2, -2**63), (0, 2**62)])
def test_ids_outside_their_table_are_refused(bad):
    from dicee_amd.evaluator import check_triple_ids
    t = np.array(GOOD, dtype=np.int64)
    t[1, bad[0]] = bad[1]
    with pytest.raises(IndexError):
        check_triple_ids(t, 10, 3)
    with pytest.raises(IndexError):
        check_triple_ids(np.array([[-0.5, 0, 1]]), 10, 3)
    with pytest.raises(IndexError):
        check_triple_ids(np.array([[0, 0, 2**70]], dtype=object), 10, 3)
    with pytest.raises(IndexError):
        check_triple_ids(np.array([[0, 0, -2**70]], dtype=object), 10, 3)


def test_a_read_only_test_set_goes_to_torch_without_a_warning(tmp_path):
    """A memory-mapped file, or an array whose owner locked it: torch.from_numpy warns of memory it may not write."""
    from dicee_amd.evaluator import check_triple_ids
    np.save(tmp_path / "t.npy", np.array(GOOD, dtype=np.int64))
    locked = np.array(GOOD, dtype=np.int64)
    locked.flags.writeable = False
    for t in (np.asarray(np.load(tmp_path / "t.npy", mmap_mode="r")), locked):
        with warnings.catch_warnings():
            warnings.simplefilter("error")
            got = torch.from_numpy(check_triple_ids(t, 10, 3))
        np.testing.assert_array_equal(got.numpy(), GOOD)
