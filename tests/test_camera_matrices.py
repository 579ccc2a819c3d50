"""The renderer's camera matrices as rows of 16 floats: the forms it takes, and
those it refuses."""
import numpy as np
import pytest

from ngt.renderer import _mat_list


@pytest.mark.parametrize("mats", [
    [np.eye(4), np.arange(16.0).reshape(4, 4)], [np.eye(4, dtype=np.float32)], np.arange(32.0).reshape(2, 4, 4),
    [np.eye(4), np.arange(16.0)], (list(range(16)),)])
def test_rows(mats):
    rows = _mat_list(mats)
    assert rows.dtype == np.float32 and rows.shape == (len(mats), 16)
    for r, m in zip(rows, mats):
        assert np.array_equal(r, np.asarray(m, dtype=np.float32).reshape(16))


@pytest.mark.parametrize("mats", [[], np.eye(4), [np.ones((2, 4)), np.ones((2, 4))]])
def test_refused(mats):
    with pytest.raises(ValueError):
        _mat_list(mats)
