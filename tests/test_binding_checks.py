"""Sizes that the Python binding checks before a call whose C entry trusts them."""
import numpy as np
import pytest

from pyiid_amd import _lib


class Stub:
    """In the library's place: notes the call, fails nothing."""

    def __init__(self):
        self.rows = []

    def pyiid_grad_pdf(self, handle, grad, rows, out, flags):
        self.rows.append(rows)
        return 0

    def pyiid_set_transform(self, *args):
        return 0

    def pyiid_destroy(self, handle):
        return 0


@pytest.fixture
def context():
    c = _lib.Context.__new__(_lib.Context)
    c.lib, c.handle = Stub(), None
    c.set_transform(0.01, 0.1, 0.01 * np.arange(40), 0.0, 30)
    return c


@pytest.mark.parametrize("shape,n_r,out", [
    ((12, 30), 40, None),            # rows of a flat array: 360 of them were taken
    ((30,), 40, None), ((2, 2, 3, 30), 40, None),
    ((4, 3, 29), 40, None), ((4, 3, 31), 40, None),
    ((4, 3, 30), 39, None), ((4, 3, 30), 41, None),
    ((4, 3, 30), 40, (4, 3, 39)), ((4, 3, 30), 40, (3, 3, 40)), ((4, 3, 30), 40, (13, 40))])
def test_grad_pdf_refuses_sizes_that_do_not_fit(context, shape, n_r, out):
    with pytest.raises(ValueError):
        context.grad_pdf(np.zeros(shape, np.float32), n_r,
                         out=None if out is None else np.zeros(out))
    assert context.lib.rows == []


def test_grad_pdf_passes_sizes_that_fit(context):
    assert context.grad_pdf(np.zeros((4, 3, 30), np.float32), 40).shape == (4, 3, 40)
    assert context.grad_pdf(np.zeros((7, 1, 30)), 40, out=np.zeros((7, 40))).shape == (7, 40)
    assert context.grad_pdf(np.zeros((0, 3, 30)), 40).shape == (0, 3, 40)
    assert context.lib.rows == [12, 7, 0]
