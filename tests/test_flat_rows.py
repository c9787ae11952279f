"""Neighbour rows of the pair interface as one flat array with row addresses: every
kind of row that a conversion one by one takes, and its refusals."""
import ctypes as C

import numpy as np
import pytest

from ann_amd.gpu import _flat_rows

ROWS = [[3, 1, 2], [], [7], [0, 5, 2 ** 31 - 1, -1]]


def _read(num, ptrs):
    return [list((C.c_int * n).from_address(int(p))) if n else [] for n, p in zip(num, ptrs)]


@pytest.mark.parametrize("kind", [
    lambda: [np.array(r, np.int32) for r in ROWS], lambda: [np.array(r, np.int64) for r in ROWS],
    lambda: [np.array(r, np.float64) for r in ROWS], lambda: ROWS, lambda: tuple(map(tuple, ROWS)),
    lambda: iter(ROWS), lambda: (np.array(r, np.int32) for r in ROWS),
    lambda: [np.repeat(np.array(r, np.int32), 2)[::2] for r in ROWS],
    lambda: [np.array(r, np.int32).reshape(-1, 1) for r in ROWS],
    lambda: [np.array(ROWS[0], np.int32).reshape(-1, 1)] + [np.array(r, np.int32) for r in ROWS[1:]],
    lambda: [ROWS[0], np.array([], np.int64), 7, np.array(ROWS[3])]])
def test_rows(kind):
    num, flat, ptrs = _flat_rows(kind(), 4)
    assert flat.dtype == np.int32 and ptrs.dtype == np.uintp and _read(num, ptrs) == ROWS


def test_matrix_and_empty():
    matrix = np.arange(12).reshape(4, 3)
    num, flat, ptrs = _flat_rows(matrix, 4)
    assert len(flat) == 12 and _read(num, ptrs) == matrix.tolist()
    num, flat, ptrs = _flat_rows([[], []], 2)
    assert list(num) == [0, 0] and len(flat) == 0 and len(ptrs) == 2
    assert len(_flat_rows([], 0)[0]) == 0


def test_refused():
    for big in (2 ** 31, -2 ** 31 - 1, 2 ** 40):
        with pytest.raises(OverflowError):
            _flat_rows([[1, big], [0]], 2)
    with pytest.raises(ValueError):
        _flat_rows([[1], [0]], 3)
    with pytest.raises(ValueError):
        _flat_rows([[1], [0]], 1)
    with pytest.raises(ValueError):
        _flat_rows([["x"], [0]], 2)
