"""Which calls of a convolution block take the package's kernel and which go on to the library; without a GPU, the kernel
stands in as the library's convolution in a recorder."""
import pytest
import torch
import torch.nn.functional as F

from spgt_amd._lib import SpgtError
from spgt_amd.extension.bind import datamove


@pytest.fixture
def kernel_calls(monkeypatch):
    """The calls that would have reached the kernel."""
    calls = []

    def stand_in(X, weight, bias, activation, count, turned):
        calls.append((X, weight, bias, turned))
        return F.conv_transpose2d(X, weight, None, padding=1) if turned else F.conv2d(X, weight, bias, padding=1)

    monkeypatch.setattr(datamove, "_conv3x3", stand_in)
    return calls


@pytest.mark.parametrize("fn", [datamove.conv3x3, datamove.conv3x3_train])
def test_wrappers_refuse_operands_off_the_gpu(kernel_calls, fn):
    with pytest.raises(SpgtError):
        fn(torch.zeros(1, 4, 5, 6), torch.zeros(8, 4, 3, 3), torch.zeros(7))
    assert not kernel_calls
