"""The Python binding's conversions, without a device: token ids of any sequence convert as int() and a
C int take them, and collect()'s result is a plain dict to every reader whether or not the K/V array
was asked for."""

import copy
import pickle

import numpy as np
import pytest

from tiles_amd import runtime as R


@pytest.mark.parametrize("ids", [[1, 2, 3], (4, 5), [], [1.7, 2], [2**40 + 5, -1], np.array([3, 4]), range(4),
                                 [np.int64(7), True], ["9"]])
def test_token_ids_convert_one_by_one_or_together(ids):
    assert list(R._token_array(ids)) == list((R.token_id * len(ids))(*[int(t) for t in ids]))


def test_unrequested_cache_reads_as_zeros():
    make = lambda: R._Diagnostics(np.ones(2), 4, None, np.zeros(3))  # noqa: E731
    zeros = np.zeros(4, dtype=np.float32)
    readers = (lambda d: d["kv"], lambda d: d.get("kv"), lambda d: dict(d)["kv"], lambda d: {**d}["kv"], lambda d: d.pop("kv"),
               lambda d: list(d.values())[1], lambda d: dict(d.items())["kv"], lambda d: d.copy()["kv"],
               lambda d: copy.deepcopy(d)["kv"], lambda d: pickle.loads(pickle.dumps(d))["kv"], lambda d: (d | {})["kv"])
    for read in readers:
        got = read(make())
        assert got.dtype == np.float32 and np.array_equal(got, zeros)
    d = make()
    assert set(d) == {"logits", "kv", "block_outputs"} and len(d) == 3 and "kv" in d
    d["kv"][1] = 5.0  # an array of its own
    assert d["kv"][1] == 5.0 and make()["kv"][1] == 0.0
