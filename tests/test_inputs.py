"""Arrays that a caller may hand over (on the CPU): any order and sign of strides,
read-only, either byte order, lists; the values arrive as contiguous float64 rows."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from jaccpot_amd.solver import FastMultipoleMethod

N = 7


def _as_inputs(x, m):
    fmm = object.__new__(FastMultipoleMethod)  # without a GPU: only the device is read
    fmm.device = torch.device("cpu")
    return fmm._as_inputs(x, m)


def _readonly(a):
    a = a.copy()
    a.flags.writeable = False
    return a


FORMS = {
    "rows": lambda a: a.copy(),
    "columns first": np.asfortranarray,
    "reversed": lambda a: a[::-1].copy()[::-1],
    "reversed columns": lambda a: a[..., ::-1].copy()[..., ::-1],
    "every second": lambda a: np.repeat(a, 2, axis=0)[::2],
    "read-only": _readonly,
    "big endian": lambda a: a.astype(a.dtype.newbyteorder(">")),
}


@pytest.mark.filterwarnings("error")
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("dtype", (np.float32, np.float64, np.float16))
def test_numpy_inputs(form, dtype):
    rng = np.random.default_rng(3)
    x, m = rng.normal(size=(N, 3)).astype(dtype), rng.uniform(size=N).astype(dtype)
    xd, md, kind, in_dtype, in_dev = _as_inputs(FORMS[form](x), FORMS[form](m))
    assert kind == "numpy" and in_dev is None and in_dtype == FORMS[form](x).dtype
    for got, want in ((xd, x), (md, m)):
        assert got.dtype == torch.float64 and got.is_contiguous()
        assert np.array_equal(got.numpy(), want.astype(np.float64))


def test_lists_and_shapes():
    xd, md, *_ = _as_inputs([[0, 1, 2], [3, 4, 5]], [1, 2])
    assert xd.tolist() == [[0, 1, 2], [3, 4, 5]] and md.tolist() == [1, 2]
    for x, m in ((np.zeros((3, 2)), np.zeros(3)), (np.zeros((3, 3)), np.zeros(4)), (np.zeros((0, 3)), np.zeros(0))):
        with pytest.raises(ValueError):
            _as_inputs(x, m)
