"""Arguments the compiled binding (csrc/binding.cpp) does not take: they reach the checks of ops.py and end as Python
exceptions, never as a C++ exception that leaves a C function."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from vectorsparse_amd import ops


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


@pytest.mark.parametrize("name", sorted(_calls("cpu")))
def test_tensors_without_storage_raise(name):
    with FakeTensorMode():
        call = _calls("cuda")[name]
        with pytest.raises(Exception):
            call()


@pytest.mark.parametrize("name", ["wmmaSpmm", "cudaSpmm", "wmmaSddmm", "cudaSddmm"])
def test_host_tensors_raise(name):
    with pytest.raises(Exception):
        _calls("cpu")[name]()
