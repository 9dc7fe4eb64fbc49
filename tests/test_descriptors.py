"""Tensor descriptors and the row-alignment test against their plain forms (CPU)."""
import pytest
import torch

from saga_amd import _lib, ops

VIEWS = {
    "scalar": lambda: torch.zeros(()),
    "vector": lambda: torch.zeros(7, dtype=torch.int32),
    "empty": lambda: torch.zeros(0, 3),
    "rows": lambda: torch.zeros(3, 40, dtype=torch.bool)[:, 8:],
    "packed8": lambda: torch.zeros(2, 3, 512, dtype=torch.bfloat16),
    "heads": lambda: torch.zeros(2, 3, 4, 64, dtype=torch.bfloat16).transpose(1, 2),
    "expanded": lambda: torch.zeros(1, 3, 4, 64, dtype=torch.float16).expand(5, 3, 4, 64),
    "unaligned": lambda: torch.zeros(2, 3, 4, 72, dtype=torch.bfloat16)[..., 1:65],
    "odd_rows": lambda: torch.zeros(2, 3, 4, 65, dtype=torch.bfloat16)[..., :64],
    "odd_single": lambda: torch.zeros(4 * 64 + 3).as_strided((1, 1, 4, 64), (259, 3, 64, 1)),
    "strided": lambda: torch.zeros(2, 3, 4, 128, dtype=torch.bfloat16)[..., ::2],
}


@pytest.mark.parametrize("name", VIEWS)
def test_descriptor(name):
    t = VIEWS[name]()
    d = _lib.descriptor(t)
    n = max(t.dim(), 1)
    assert (d.data or 0) == t.data_ptr() and d.dtype == _lib.dtype_code(t.dtype) and d.ndim == n
    assert list(d.shape) == (list(t.shape) or [1]) + [0] * (4 - n)
    assert list(d.stride) == (list(t.stride()) or [1]) + [0] * (4 - n)


def test_descriptor_refuses():
    with pytest.raises(ValueError):
        _lib.descriptor(torch.zeros(1, 1, 1, 1, 1))
    with pytest.raises(TypeError):
        _lib.descriptor(torch.zeros(2, dtype=torch.float64))


@pytest.mark.parametrize("name", VIEWS)
def test_vec_ready(name):
    t = VIEWS[name]()
    if t.dim() == 0:
        return
    es = t.element_size()
    ok = t.stride(-1) == 1 and t.data_ptr() % 16 == 0 and all(
        (s * es) % 16 == 0 for s, n in zip(t.stride()[:-1], t.shape[:-1]) if n > 1)
    got = ops._vec_ready(t)
    assert (got is t) == (ok or t.is_contiguous())
