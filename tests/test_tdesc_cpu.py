"""A tensor descriptor holds what its fields would be assigned one by one, for
integer and integer-like entries and for lists of unlike lengths."""
import numpy as np
import pytest

from tenet_hip import _lib as L
from tenet_hip.device import tdesc


@pytest.mark.parametrize("shape,labels,strides", [
    ((), (), None), ((3,), (1,), None), ((np.int64(3), 4.0), (1, 2), None), ((3, 4), (5, 6), (4, 1)),
    (tuple(range(1, 9)), range(8), None), ((2, 3, 4), (1, 2), None), (np.array([2, 3]), (1, 2), None)])
def test_fields(shape, labels, strides):
    st, acc = [], 1
    for s in shape:
        st.append(acc)
        acc *= int(s)
    d, z = L.TDesc(), tdesc(shape, labels, strides)
    d.rank = len(shape)
    for i, (e, s, lab) in enumerate(zip(shape, strides or st, labels)):
        d.extent[i], d.stride[i], d.label[i] = int(e), int(s), int(lab)
    assert bytes(d) == bytes(z)


def test_rank_limit():
    with pytest.raises(ValueError, match="rank above 8"):
        tdesc(range(9), range(9))


def test_zero_dimensional_floats_and_generators():
    """What int() takes is taken: 0-d float arrays (which have an __index__ that
    refuses), and label and stride sequences that can be read only once."""
    want = tdesc((2, 3), (5, 6), (1, 2))
    assert bytes(tdesc((np.array(2.0), np.array(3.0)), (5, 6), (1, 2))) == bytes(want)
    assert bytes(tdesc((2.0, 3), (x for x in (5, 6)), (x for x in (1, 2)))) == bytes(want)
    with pytest.raises(TypeError):
        tdesc((2, None), (5, 6), (1, 2))
