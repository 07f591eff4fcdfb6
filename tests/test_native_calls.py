"""The native calls (csrc/native_calls.cpp): they serve the plain case with the Python operators' results and leave every
other to those operators."""
import os
import shutil
import subprocess
import sys
import threading

import pytest
import torch

from spgt_amd import _lib
from spgt_amd.extension.bind import datamove as dm
from spgt_amd.extension.bind import galerkin_attention as ga
from spgt_amd.extension.bind import linear as ln


def test_serves_nothing_but_the_bound_library_and_gpu_tensors():
    lib = _lib.load()
    x, w = torch.zeros(3, 128), torch.zeros(128, 128)
    for first in (None, lib, object()):
        assert _lib.fast.linear(first, x, w, None, None, 0, False, 1) is None
    assert _lib.fast.linear(lib, x, w) is None and _lib.fast.weight_grad(lib, 1, "x", None) is None
    assert _lib.fast.encoder_layer(lib, x, None, [], 1e-6, 0) is None
    with pytest.raises(_lib.SpgtError):
        ln.fused_linear(x, w)


@pytest.mark.parametrize("content", [None, b"not a shared object"])
def test_missing_or_unusable_build_is_named(monkeypatch, tmp_path, content):
    path = tmp_path / "_native_calls.so"
    if content is not None:
        path.write_bytes(content)
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "NATIVE_PATH", str(path))
    with pytest.raises(_lib.SpgtError, match="_native_calls.*python -m spgt_amd.build"):
        _lib.load()


@pytest.mark.parametrize("stale", [None, b"not a shared object"])
def test_built_and_loaded_in_one_process(tmp_path, stale):
    """A checkout without libraries, or with a native module that cannot be loaded, imports the package, builds and loads
    what it has built.  (The compilers' part is played by a copy of this tree's libraries.)"""
    root, built = os.path.dirname(_lib.PKG_DIR), [_lib.LIB_PATH, _lib.NATIVE_PATH]
    shutil.copytree(_lib.PKG_DIR, tmp_path / "spgt_amd", ignore=shutil.ignore_patterns("*.so", "build", "__pycache__"))
    shutil.copy(os.path.join(root, "__graft_entry__.py"), tmp_path)
    if stale is not None:
        (tmp_path / "spgt_amd" / "_native_calls.so").write_bytes(stale)
    code = f"""
import os, shutil
import __graft_entry__
import spgt_amd.build as recipe
from spgt_amd import _lib
assert os.path.samefile(_lib.PKG_DIR, {str(tmp_path / "spgt_amd")!r})
def copied(**_):
    for path in {built!r}:
        target = os.path.join(_lib.PKG_DIR, os.path.basename(path))
        shutil.copy(path, target + ".tmp")
        os.replace(target + ".tmp", target)
    return _lib.LIB_PATH
recipe.build = copied
__graft_entry__.build()
assert _lib.fast.__file__ == _lib.NATIVE_PATH and _lib.fast.linear(None) is None
"""
    done = subprocess.run([sys.executable, "-c", code], cwd=tmp_path, capture_output=True, text=True)
    assert done.returncode == 0, done.stderr


def _calls(gpu):
    """By name: a call of an operator (some with more than one native call in them) and the native functions that serve it."""
    g = torch.Generator().manual_seed(1)
    r = lambda *s: torch.randn(*s, generator=g).to(gpu)
    x, w, b = r(2, 300, 128), r(128, 384) / 11, r(384)
    q, k, v, pos = r(2, 300, 128), r(2, 300, 128), r(2, 300, 128), r(2, 300, 2)
    norm = [r(4, 32) for _ in range(4)]
    heads = [r(2, 4, 34, 300) for _ in range(3)]
    out, ktv = ga.gexts.galerkin_attention_fused_forward(q, k, v, pos, *norm, 1e-6, 4, 2, return_ktv=True)
    tail = (r(2, 300, 136), x, r(136, 128) / 11, r(128), r(128, 256) / 11, r(256), r(256, 128) / 16, r(128), "silu")
    y, u, w5 = r(2, 24, 60, 32), r(2, 24, 60, 32), [r(12, 12, 32, 32, 2) for _ in range(2)]
    gh = torch.complex(r(24, 60), r(24, 60))
    table, field, lin = r(60, 24), r(2, 60, 60, 32), r(32, 32)
    operand = dm.inverse_table_operand(table)
    gf = ga.gexts
    layer_x, layer_pos = r(1, 6400, 128), r(1, 6400, 2)
    layer = {dp: [r(*(shape or (128, 4 * (32 + dp)))) / 11 for _, shape in ln.ENCODER_LAYER_SHAPES] for dp in (0, 2)}
    residual, square, wide = r(2, 300, 384), w[:, :128].contiguous(), w[:, :256].contiguous()
    hidden, planes = torch.relu(r(2, 300, 256)), torch.stack([q, k, v])
    image, taps, image_bias = r(2, 8, 9, 11), r(12, 8, 3, 3), r(12)
    to_136, pre = r(128, 136) / 11, x.view(600, 128)
    calls = {
        "linear": (lambda: ln.fused_linear(x, w, b, "relu", residual, planes=1), ["linear"]),
        "linear_after": (lambda: ln.fused_linear(x, w, b, "silu", residual, True), ["linear"]),
        "planes": (lambda: ln.fused_linear(x, w, None, "none", planes=3), ["linear"]),
        "input_grad": (lambda: ln.linear_input_grad(x, to_136), ["input_grad"]),
        "masked": (lambda: ln.linear_input_grad(x, wide, relu_output=hidden), ["input_grad"]),
        "added": (lambda: ln.linear_input_grad(x, wide, add=hidden), ["input_grad"]),
        "projection_input_grad": (lambda: ln.projection_input_grad(x, square), ["projection_input_grad"]),
        "packed": (lambda: ln.packed_input_grad(planes.view(3, 600, 128), [w[:, i:i + 128].contiguous() for i in (0, 128, 256)],
                                                pre), ["packed_input_grad"]),
        "weight_grad": (lambda: ln.linear_weight_grad(x, q) + ln.linear_weight_grad(x, q, out_major=True), ["weight_grad"] * 2),
        "weight_grad_batched": (lambda: ln.linear_weight_grad_batched(x, planes), ["weight_grad_batched"]),
        "attention": (lambda: gf.galerkin_attention_fused_forward(q, k, v, pos, *norm, 1e-6, 4, 2, return_ktv=True) +
                      gf.galerkin_attention_fused_backward(out, q, k, v, pos, *norm, 1e-6, ktv, 4, 2),
                      ["attention_forward", "attention_backward"]),
        "attention_forward": (lambda: gf.galerkin_attention_fused_forward(q, k, v, None, *norm, 1e-6, 4, 0, return_ktv=True),
                              ["attention_forward"]),
        "encoder_tail": (lambda: ln.fused_encoder_tail(*tail), ["encoder_tail"]),
        "modes_middle": (lambda: dm._spectral_modes_middle(y, gh, gh.t().contiguous(), *w5), ["modes_middle"]),
        "dft_forward": (lambda: dm.truncated_dft_rows_forward(field, table, planar=True), ["dft_rows_planar"]),
        "dft_inverse": (lambda: dm.truncated_dft_rows_inverse(y, table, planar=True), ["dft_rows_planar"]),
        "inverse_linear": (lambda: dm.spectral_inverse_linear(u, operand, field, lin, b[:32], "silu"), ["inverse_linear"]),
        "inverse_linear_plain": (lambda: dm.spectral_inverse_linear(u, operand, field, lin, None, None), ["inverse_linear"]),
        "conv3x3": (lambda: dm.conv3x3(image, taps, image_bias, "silu", 2), ["conv3x3"]),
        "projection": (lambda: gf.multihead_projection_with_position_rrc_forward(x, square, b[:128], pos, 300, 128, 4, 32, 2, 2),
                       ["projection"]),
        "projection_layernorm": (lambda: gf.multihead_projection_layernorm_with_position_rrc_forward(
            x, square, b[:128], norm[0], norm[1], 1e-5, pos, 300, 128, 4, 32, 2, 2), ["projection"]),
        "cccr": (lambda: (gf.multihead_galerkin_attention_cccr_forward(*heads, 2, 4, 34, 300),) +
                 gf.multihead_galerkin_attention_cccr_backward(heads[0].transpose(2, 3).contiguous(), *heads, 2, 4, 34, 300),
                 ["cccr_forward", "cccr_backward"]),
        "heads_to_tokens": (lambda: ga._heads_feature_to_token_major(heads[0], 2, 4, 2, 32, 300), ["heads_to_tokens"]),
        "layernorm": (lambda: ga._layernorm_heads_backward(pre, q, norm[0], 1e-6, 4, 32), ["layernorm_heads_backward"]),
    }
    for dp in (0, 2):
        position = layer_pos if dp else None

        def encoder_layer(position=position, parameters=layer[dp]):
            got = ln.fused_encoder_layer_if_plain(layer_x, position, parameters, 1e-5, "relu")
            return ln.fused_encoder_layer(layer_x, position, parameters, 1e-5, "relu") if got is None else got

        calls[f"encoder_layer_{dp}"] = encoder_layer, ["encoder_layer"]
    return calls


class _Recorder:
    """The native calls, noting which were made and whether they served."""

    def __init__(self, native):
        self.native, self.served, self.refused = native, [], []

    def __getattr__(self, name):
        def call(*args):
            got = getattr(self.native, name)(*args)
            (self.refused if got is None else self.served).append(name)
            return got

        return call


def _flat(t):
    return [t] if isinstance(t, torch.Tensor) else list(t)


@pytest.mark.gpu
def test_same_results_as_the_python_operators(gpu, monkeypatch):
    """Bit for bit, shapes, strides and all; every native function is among the calls and serves its own."""
    _lib.load()
    native, served = {}, set()
    calls = _calls(gpu)
    for name, (call, functions) in calls.items():
        recorder = _Recorder(_lib.fast)
        with monkeypatch.context() as patch:
            patch.setattr(_lib, "fast", recorder)
            native[name] = _flat(call())
        assert recorder.served == functions and not recorder.refused, name
        served.update(functions)
    assert served == {n for n in dir(_lib.fast) if not n.startswith("_")} - {"bind"}
    monkeypatch.setattr(_lib, "fast", _lib._NotBuilt())
    for name, (call, _) in calls.items():
        for a, b in zip(native[name], _flat(call()), strict=True):
            assert a.shape == b.shape and a.is_contiguous() == b.is_contiguous() and torch.equal(a, b), name
            assert not a.requires_grad


@pytest.mark.gpu
def test_on_other_streams_and_threads(gpu):
    """Every native call runs on the stream that is current in its thread: behind a fill of its input on that stream, and from
    four threads with streams of their own at once."""
    _lib.load()
    calls = _calls(gpu)
    want = {name: [t.clone() for t in _flat(call())] for name, (call, _) in calls.items()}
    x, w = torch.zeros(4096, 128, device=gpu), torch.randn(128, 128, device=gpu)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        busy = torch.randn(4096, 4096, device=gpu)
        for _ in range(8):
            busy = busy @ busy / 64
        x.fill_(1.0)  # late on this stream
        got = ln.fused_linear(x, w)
    side.synchronize()
    assert torch.equal(got, ln.fused_linear(torch.ones_like(x), w))
    failed = []

    def work():
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(3):
                    for name, (call, _) in calls.items():
                        got = [t.clone() for t in _flat(call())]
                        torch.cuda.current_stream().synchronize()
                        failed.extend(name for a, b in zip(got, want[name], strict=True) if not torch.equal(a, b))
        except BaseException as e:  # shown by the assertion below
            failed.append(e)

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed


@pytest.mark.gpu
def test_leaves_the_rest_to_the_python_operators(gpu):
    lib, fast = _lib.load(), _lib.fast
    x, w = torch.randn(40, 128, device=gpu), torch.randn(128, 128, device=gpu)
    plain = lambda a, b, *more: fast.linear(lib, a, b, *(more or (None, None, 0, False, 1)))
    assert plain(x, w) is not None and plain(torch.nn.Parameter(x), torch.nn.Parameter(w)) is not None

    class Marked(torch.Tensor):
        pass

    refused = [(x.as_subclass(Marked), w), (x.double(), w), (x[:, ::2], w), (x.t(), w), (x, w[:, :31]), (x[:0], w), (x.cpu(), w),
               (torch.empty(40 * 128 + 1, device=gpu)[1:].view(40, 128), w), (x._neg_view(), w)]
    assert all(plain(a, b) is None for a, b in refused)
    assert plain(x, w, torch.zeros(127, device=gpu), None, 0, False, 1) is None  # bias of another size
    assert plain(x, w, None, x[:39], 0, False, 1) is None and plain(x, w, None, None, 7, False, 1) is None
    with torch.utils._python_dispatch._disable_current_modes(), torch.overrides.BaseTorchFunctionMode():
        assert plain(x, w) is None
    assert torch.equal(torch.func.vmap(lambda t: t * 1)(x), x)

    def inside(t):
        assert plain(t, w) is None
        return t

    torch.func.vmap(inside)(x.view(2, 20, 128))
    lib2 = _lib.open_library(_lib.LIB_PATH)
    assert fast.linear(lib2, x, w, None, None, 0, False, 1) is None


@pytest.mark.gpu
def test_missing_layernorm_parameters_are_refused(gpu):
    """... by the operator with LayerNorm, also where the native call without it would serve the rest."""
    _lib.load()
    x, w = torch.randn(2, 300, 128, device=gpu), torch.randn(128, 128, device=gpu)
    b, pos = torch.randn(128, device=gpu), torch.randn(2, 300, 2, device=gpu)
    project = ga.gexts.multihead_projection_layernorm_with_position_rrc_forward
    norm = torch.randn(4, 32, device=gpu)
    for weight, bias in ((None, None), (norm, None), (None, norm)):
        with pytest.raises((TypeError, AttributeError)):
            project(x, w, b, weight, bias, 1e-5, pos, 300, 128, 4, 32, 2, 2)


@pytest.mark.gpu
def test_residuals_of_another_row_length_are_refused(gpu):
    """... where they have two dimensions; any other shape is taken as rows of the result."""
    _lib.load()
    x, w = torch.randn(2, 300, 128, device=gpu), torch.randn(128, 128, device=gpu)
    for shape in ((1200, 64), (300, 256)):
        with pytest.raises(ValueError):
            ln.fused_linear(x, w, residual=torch.randn(shape, device=gpu))
    rows = torch.randn(600, 128, device=gpu)
    want = ln.fused_linear(x, w, residual=rows.view(2, 300, 128))
    for residual in (rows, rows.view(-1), rows.view(4, 150, 128), rows.view(2, 150, 256)):
        assert torch.equal(ln.fused_linear(x, w, residual=residual), want)
