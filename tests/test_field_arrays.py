"""The arrays a download fills: independent of each other in memory."""
import numpy as np
import pytest

from hydropad_amd.hydro import FIELDS, field_arrays


@pytest.mark.parametrize("shape", [(9, 9, 9), (38, 38, 38), (70, 41, 99)])
def test_each_field_owns_its_memory(shape):
    """Keeping one field of a download keeps that field alone."""
    out = field_arrays(shape)
    assert tuple(out) == FIELDS
    for k, a in out.items():
        assert a.shape == shape and a.dtype == np.float64 and a.flags.f_contiguous and a.flags.writeable
        assert a.flags.owndata and a.base is None, k
        a[...] = 1.0 + FIELDS.index(k)
    for k, a in out.items():
        assert np.all(a == 1.0 + FIELDS.index(k))
