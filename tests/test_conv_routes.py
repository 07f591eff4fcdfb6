"""Which calls of a convolution block take the package's kernel and which go on to the library; without a GPU, the kernel
stands in as the library's convolution in a recorder."""
import pytest
import torch
import torch.nn.functional as F

from spgt_amd._lib import SpgtError
from spgt_amd.extension.bind import datamove
from spgt_amd.network.layer import ConvResBlock2D


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


@pytest.fixture
def block(monkeypatch, kernel_calls):
    """A block whose operands the kernel would serve, wherever they live."""
    monkeypatch.setattr(ConvResBlock2D, "_own_kernel", lambda self, X: True)
    monkeypatch.setattr(datamove, "_check_conv3x3", lambda *operands: None)
    torch.manual_seed(1)
    return ConvResBlock2D(3, 5, 3, 1, 0.0, "silu")


def test_plain_call_takes_the_kernel(block, kernel_calls):
    block(torch.randn(1, 3, 6, 7))
    assert len(kernel_calls) == 1


@pytest.mark.parametrize("hook", ["forward", "forward_pre", "full_backward", "full_backward_pre", "global_forward",
                                  "global_forward_pre", "global_full_backward", "global_full_backward_pre"])
def test_hooked_convolutions_are_called(block, kernel_calls, hook):
    """Every kind of hook on the convolution, or on all modules, sees it."""
    seen = []

    def note(*args):
        if args[0] is block.conv_layer:
            seen.append(args)

    if hook.startswith("global_"):
        handle = getattr(torch.nn.modules.module, f"register_module_{hook[7:]}_hook")(note)
    else:
        handle = getattr(block.conv_layer, f"register_{hook}_hook")(note)
    try:
        block(torch.randn(1, 3, 6, 7, requires_grad=True)).sum().backward()
    finally:
        handle.remove()
    assert seen and not kernel_calls


def test_replaced_forwards_are_called(block, kernel_calls):
    forward = block.conv_layer.forward
    block.conv_layer.forward = lambda X: 2 * forward(X)
    x = torch.randn(1, 3, 6, 7)
    assert torch.equal(block(x), F.silu(2 * forward(x))) and not kernel_calls
