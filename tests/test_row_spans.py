"""Stages of several tokens reach their input rows by 32-bit offsets: rows further apart than that are refused, on host-only graphs."""
import pytest

from mirage import _capi
from test_unread_program import _attach, _linear, _pk, B


@pytest.mark.parametrize("stride,fits", [(2 ** 28, True), (2 ** 32 // (2 * (B - 1)) + 1, False), (2 ** 31 - 8, False)])
def test_rows_far_apart(stride, fits):
    pk = _pk()
    x, (y, _) = pk.new_tensor((B, 64), strides=(stride, 1), name="x"), _attach(pk, "y", B, 64)
    _linear(pk, x, 64, y)
    if fits:
        assert len(pk.describe_program().splitlines()) == 1
    else:
        with pytest.raises(_capi.MkError, match="4 GiB"):
            pk.describe_program()
