"""Configuration.copy_to_host with a stand-in for the native context: rows that
the library can fill are filled in place, read-only ones (a colarray around a
memory map opened for reading) are an error and stay as they are, rows of
another type are converted."""
import numpy as np
import pytest

import gamdpy_amd as gp


class Context:
    """Hands out ones, through the rows' memory as the library does."""

    def __init__(self, N):
        self.N = N
        self.in_place = False

    def download(self, vectors=None):
        N = self.N
        self.in_place = vectors is not None
        rows = vectors if vectors is not None else [np.empty((N, 3), np.float32) for _ in range(3)]
        for a in rows:
            b = np.frombuffer((gp._native.ctypes.c_char * a.nbytes).from_address(a.ctypes.data), a.dtype)
            b[:] = 1.0
        return (*rows, np.ones((N, 4), np.float32), np.ones(N, np.int32), np.ones((N, 3), np.int32))

    def current_box(self):
        return None


def _conf(array):
    conf = gp.Configuration(D=3, N=array.shape[1])
    conf.vectors = gp.configuration.colarray(conf.vector_columns, array.shape[1:], array=array)
    conf.attach(Context(conf.N))
    return conf


@pytest.mark.parametrize("dtype,in_place", [(np.float32, True), (np.float64, False)])
def test_rows_are_filled(dtype, in_place):
    conf = _conf(np.zeros((3, 5, 3), dtype))
    conf.copy_to_host()
    assert conf._ctx.in_place == in_place
    assert np.all(conf.vectors.array == 1.0) and conf.vectors.array.dtype == dtype and np.all(conf.ptype == 1)


def test_read_only_rows_are_an_error():
    array = np.zeros((3, 5, 3), np.float32)
    array.flags.writeable = False
    conf = _conf(array)
    with pytest.raises(ValueError, match="read-only"):
        conf.copy_to_host()
    assert not np.any(array) and not np.any(conf.ptype)
