"""Which calls of a convolution block take the package's kernel and which go on to the library; without a GPU, the kernel
stands in as the library's convolution in a recorder."""
import pytest
import torch
import torch.nn.functional as F

from spgt_amd import _lib
from spgt_amd._lib import SpgtError
from spgt_amd.extension.bind import datamove
from spgt_amd.network.layer import ConvResBlock2D
from spgt_amd.network.model import UpScaler2D


@pytest.fixture
def kernel_calls(monkeypatch):
    """The calls that would have reached the kernel."""
    calls = []

    def stand_in(X, weight, bias, activation, count, turned):
        assert X.data_ptr() and weight.data_ptr()
        calls.append((X, weight, bias, turned))
        X, weight = X.detach(), weight.detach()
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
    monkeypatch.setattr(ConvResBlock2D, "_own_kernel", lambda self, X, with_gradient=False: True)
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


@pytest.fixture
def leaves_and_output(block):
    x = torch.randn(2, 3, 6, 7, requires_grad=True)
    leaves = [x, block.conv_layer.weight, block.conv_layer.bias]
    return leaves, datamove.conv3x3_train(*leaves), F.conv2d(*leaves, padding=1)


def test_batched_gradients_go_to_the_library(kernel_calls, leaves_and_output):
    leaves, y, want = leaves_and_output
    dy = torch.randn(4, *y.shape)
    del kernel_calls[:]
    got = torch.autograd.grad(y, leaves, dy, is_grads_batched=True, retain_graph=True)
    for a, b in zip(got, torch.autograd.grad(want, leaves, dy, is_grads_batched=True, retain_graph=True)):
        assert torch.equal(a, b)
    got = torch.func.vmap(lambda g: torch.autograd.grad(y, leaves[0], g, retain_graph=True)[0])(dy)
    assert torch.equal(got, torch.func.vmap(lambda g: torch.autograd.grad(want, leaves[0], g, retain_graph=True)[0])(dy))
    assert not kernel_calls


def test_forward_mode_derivatives_of_a_gradient_go_to_the_library(kernel_calls, leaves_and_output):
    import torch.autograd.forward_ad as forward_ad
    leaves, y, want = leaves_and_output
    dy, tangent = torch.randn_like(y), torch.randn_like(y)
    del kernel_calls[:]
    with forward_ad.dual_level():
        dual = forward_ad.make_dual(dy, tangent)
        got, ref = (forward_ad.unpack_dual(torch.autograd.grad(t, leaves[0], dual)[0]).tangent for t in (y, want))
    assert got is not None and torch.equal(got, ref) and not kernel_calls


def test_modes_see_the_gradient(kernel_calls, leaves_and_output):
    from torch.utils.flop_counter import FlopCounterMode
    leaves, y, want = leaves_and_output
    del kernel_calls[:]
    counts = []
    for t in (y, want):
        with FlopCounterMode(display=False) as counter:
            torch.autograd.grad(t, leaves, torch.ones_like(t), retain_graph=True)
        counts.append(counter.get_total_flops())
    assert not kernel_calls and counts[0] == counts[1] > 0


def test_plain_gradients_take_the_kernel(kernel_calls, leaves_and_output):
    leaves, y, want = leaves_and_output
    dy = torch.randn_like(y)
    del kernel_calls[:]
    got = torch.autograd.grad(y, leaves, dy)
    for a, b in zip(got, torch.autograd.grad(want, leaves, dy)):
        assert (a - b).abs().max() <= 1e-5 * b.abs().max()
    assert len(kernel_calls) == 1 and kernel_calls[0][3]


def test_watched_operators_are_not_replaced():
    """Compilers, tracers, modes and tensor classes see the library's convolution; a default device changes nothing."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.overrides import TorchFunctionMode
    from torch.utils.flop_counter import FlopCounterMode
    x = torch.randn(2, 3)
    assert datamove.run_eagerly(x, torch.nn.Parameter(x))
    with torch.device("cpu"):
        assert datamove.run_eagerly(x)
    with FlopCounterMode(display=False):
        assert not datamove.run_eagerly(x)
    with TorchFunctionMode():
        assert not datamove.run_eagerly(x)
    fake = FakeTensorMode()
    assert not datamove.run_eagerly(fake.from_tensor(x))
    assert not datamove.run_eagerly(x.as_subclass(type("Other", (torch.Tensor,), {})))
    seen = []
    torch.jit.trace(lambda t: (seen.append(datamove.run_eagerly(t)), t + 1)[1], x, check_trace=False)
    torch.fx.experimental.proxy_tensor.make_fx(lambda t: (seen.append(datamove.run_eagerly(t)), t + 1)[1])(x)
    assert seen and not any(seen)


def test_function_modes_are_seen_in_a_fresh_process():
    """... whatever parts of torch have been imported by then."""
    import subprocess
    import sys
    from conftest import ROOT
    code = ("import torch\nfrom torch.overrides import BaseTorchFunctionMode\nfrom spgt_amd.extension.bind import datamove\n"
            "with BaseTorchFunctionMode():\n    assert not datamove.run_eagerly(torch.zeros(1))")
    done = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True)
    assert done.returncode == 0, done.stderr


def test_block_compiles_into_one_graph():
    block = ConvResBlock2D(3, 5, 3, 1, 0.0, "silu")
    x = torch.randn(1, 3, 6, 7)
    torch._dynamo.reset()
    assert torch.equal(torch.compile(block, backend="eager", fullgraph=True)(x), block(x))


def test_sizes_that_the_library_is_quicker_at():
    """(batch, in, out channels, rows): the down-scaler's convolutions and the ends of the ranges that were measured
    (256 compute units, also without a GPU)."""
    pays = _lib.load().spgt_conv3x3_pays
    inference = {(1, 128, 42, 30): 1, (1, 42, 44, 30): 1, (4, 128, 42, 122): 1, (4, 42, 44, 363): 1, (16, 16, 16, 64): 1,
                 (4, 256, 256, 64): 1, (4, 512, 512, 64): 1, (16, 128, 512, 8): 0, (1, 256, 64, 30): 0, (1, 512, 512, 8): 0,
                 (4, 512, 64, 64): 0, (1, 1024, 512, 64): 0, (1, 5000, 8, 8): 0}
    training = {(4, 42, 42, 122): 0, (4, 42, 44, 363): 1, (4, 128, 42, 89): 0, (4, 128, 42, 122): 1, (16, 64, 64, 64): 1,
                (4, 64, 64, 122): 0, (4, 64, 1, 256): 1, (4, 16, 16, 256): 0, (1, 512, 512, 64): 0}
    for sizes, with_gradient in ((inference, 0), (training, 1)):
        for (n, cin, cout, r), want in sizes.items():
            assert pays(n, cin, cout, r, r + 1, with_gradient) == want, (n, cin, cout, r)


def test_weight_gradients_that_the_library_is_quicker_at():
    """(batch, in, out channels, height, width): either side of the lines that were measured, and sizes that no kernel takes."""
    pays = _lib.load().spgt_conv3x3_weight_grad_pays
    wanted = {(64, 256, 256, 8, 9): 0, (97, 256, 256, 16, 16): 0, (14, 256, 256, 200, 9): 0, (106, 192, 384, 2, 128): 0,
              (23, 256, 256, 33, 33): 1, (49, 256, 256, 4, 128): 1, (59, 256, 256, 20, 21): 1, (4, 512, 512, 122, 123): 1,
              (1366, 128, 128, 8, 9): 0, (848, 96, 96, 16, 16): 1, (5462, 64, 64, 8, 9): 0, (2731, 64, 64, 12, 12): 1,
              (19661, 64, 64, 4, 5): 0, (8239, 42, 42, 4, 5): 0, (3363, 42, 42, 7, 7): 1, (32769, 16, 16, 8, 9): 1,
              (4, 42, 42, 363, 364): 1, (4, 128, 42, 90, 91): 1, (1, 1, 1, 1, 1): 0, (0, 64, 64, 64, 64): 0,
              (1, 5000, 64, 64, 64): 0}
    for sizes, want in wanted.items():
        assert pays(*sizes) == want, sizes


@pytest.mark.parametrize("cin,cout,trained,inferred", [(128, 128, (71, 72), (82, 83)), (256, 512, (71, 72), (82, 83)),
                                                       (128, 64, (78, 79), (82, 83)), (256, 32, (78, 79), (90, 91)),
                                                       (64, 128, (90, 91), (90, 91)), (64, 512, (90, 91), (90, 91))])
def test_up_scaler_reorders_where_it_is_quicker(cin, cout, trained, inferred):
    """From 64 x 64 pixels: the last size that takes the convolution and the first that mixes the channels before."""
    scaler = UpScaler2D([[128] * 2, [90] * 2, [64] * 2, [90] * 2, [128] * 2], cin, cout, 0.0, "silu")
    x = torch.empty(1, 64, 64, cin)
    for training, sizes in ((True, trained), (False, inferred)):
        assert [scaler._resamples_enough(x, (r, r), training) for r in sizes] == [False, True]
