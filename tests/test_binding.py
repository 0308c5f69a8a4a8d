"""Arguments the compiled binding (csrc/binding.cpp) does not take: it answers with a negative status, they reach the
checks of ops.py and end as Python exceptions, never as a C++ exception that leaves a C function."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from vectorsparse_amd import _lib, ops

ENTRIES = {"wmmaSpmm": "wmma_spmm", "cudaSpmm": "cuda_spmm", "wmmaSddmm": "wmma_sddmm", "cudaSddmm": "cuda_sddmm",
           "sddmm_batched": "wmma_sddmm_batched", "sparse_softmax": "sparse_softmax", "spmm_batched": "wmma_spmm_batched"}


def _operands(device):
    make = lambda shape, dtype: torch.empty(shape, dtype=dtype, device=device)
    indices = [make(4, torch.int32), make(5, torch.int32), make(16, torch.int32)]
    return indices, make((16, 4), torch.float16), make((8, 8), torch.float16), make((16, 8), torch.float16)


def _calls(device):
    idx, values, rhs, out = _operands(device)
    q = torch.empty((2, 16, 8), dtype=torch.float16, device=device)
    scores = torch.empty((2, 16, 4), dtype=torch.float16, device=device)
    return {
        "wmmaSpmm": lambda: ops.spmm.wmmaSpmm(4, 4, 8, 8, *idx, values, rhs, out),
        "cudaSpmm": lambda: ops.spmm.cudaSpmm(4, 4, 8, 8, *idx, values, rhs, out),
        "wmmaSddmm": lambda: ops.sddmm.wmmaSddmm(4, 8, 8, 16, *idx, out, rhs, values, 4),
        "cudaSddmm": lambda: ops.sddmm.cudaSddmm(4, 8, 8, 16, *idx, out, rhs, values, 4),
        "sddmm_batched": lambda: ops.sddmm_batched(4, 8, 16, 16, *idx, q, q, scores, 4),
        "sparse_softmax": lambda: ops.sparse_softmax(4, 4, idx[0], idx[1], scores),
        "spmm_batched": lambda: ops.spmm_batched(4, 4, 8, 16, *idx, scores, q, q),
    }


class _Recorder:
    """The compiled binding, with every answer noted."""

    def __init__(self):
        _lib.lib()
        from vectorsparse_amd import _binding
        self.binding, self.answers = _binding, []

    def __getattr__(self, name):
        def call(*args):
            self.answers.append((name, getattr(self.binding, name)(*args)))
            return self.answers[-1][1]
        return call


@pytest.fixture
def recorder(monkeypatch):
    r = _Recorder()
    monkeypatch.setattr(ops, "_native", r)
    return r


@pytest.mark.parametrize("name", sorted(ENTRIES))
def test_tensors_without_storage_raise(name, recorder):
    with FakeTensorMode():
        call = _calls("cuda")[name]
        with pytest.raises((RuntimeError, ValueError)):
            call()
    assert recorder.answers == [(ENTRIES[name], -1)]


@pytest.mark.parametrize("name", sorted(ENTRIES))
def test_host_tensors_raise(name, recorder):
    with pytest.raises(ValueError, match="device memory"):
        _calls("cpu")[name]()
    assert recorder.answers == [(ENTRIES[name], -1)]


def test_wrong_argument_counts_and_types_are_unusual_not_fatal():
    binding = _Recorder().binding
    for name in dir(binding):
        if not name.startswith("_"):
            assert getattr(binding, name)() == -1
            assert getattr(binding, name)(*range(17)) == -1
            assert getattr(binding, name)(*([None] * 12)) == -1
            assert getattr(binding, name)(1 << 80, "x", 2.5) == -1
