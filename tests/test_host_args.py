"""The host helpers that pass a tensor through where it already has the wanted form: the same memory
and values as the conversion they skip, over the forms a caller may hand in."""
import sys
import pathlib

import pytest
import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent.parent / "qwen-mla-vllm_amd"))
from qmla import _lib  # noqa: E402


@pytest.mark.parametrize("make", [lambda: torch.tensor(0.37), lambda: torch.tensor([0.37, 9.0]),
                                  lambda: torch.tensor([[9.0, 0.37], [1.0, 2.0]])[:, 1], lambda: torch.tensor(0.37).expand(3),
                                  lambda: torch.tensor(0.375, dtype=torch.float64), lambda: torch.tensor([0.375]).half()])
def test_scale_first_element(make):
    t = make()
    s = _lib.as_scale(t, t.device)
    want = t.reshape(-1)[:1].to(torch.float32)
    assert s.dtype == torch.float32 and s.flatten()[0] == want[0]
    assert (s.data_ptr() == t.data_ptr()) == (t.dtype == torch.float32)


@pytest.mark.parametrize("shape", [(5, 8), (5, 2, 4), (5,), (1, 8), (5, 1, 8)])
def test_rows_flattened(shape):
    t = torch.arange(40)[:torch.Size(shape).numel()].reshape(shape)
    got, want = _lib.rows2d(t), t.reshape(t.shape[0], -1)
    assert got.shape == want.shape and got.stride() == want.stride() and got.data_ptr() == t.data_ptr()
    assert torch.equal(got, want)
    wide = torch.zeros(4, 16)[:, :8]          # a row stride of its own is kept
    assert _lib.rows2d(wide).stride() == (16, 1)


def test_no_rows_stay_refused():
    with pytest.raises(RuntimeError):
        _lib.rows2d(torch.zeros(0, 8))
