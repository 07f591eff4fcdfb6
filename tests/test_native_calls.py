"""The native calls (csrc/native_calls.cpp): they serve the plain case with the Python operators' results and leave every
other to those operators."""
import os
import shutil
import subprocess
import sys

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
    g = torch.Generator().manual_seed(1)
    r = lambda *s: torch.randn(*s, generator=g).to(gpu)
    x, w, b = r(2, 300, 128), r(128, 384) / 11, r(384)
    q, k, v, pos = r(2, 300, 128), r(2, 300, 128), r(2, 300, 128), r(2, 300, 2)
    norm = [r(4, 32) for _ in range(4)]
    heads = [r(2, 4, 34, 300) for _ in range(3)]
    out, ktv = ga.gexts.galerkin_attention_fused_forward(q, k, v, pos, *norm, 1e-6, 4, 2, return_ktv=True)
    tail = (r(2, 300, 136), x, r(136, 128) / 11, r(128), r(128, 256) / 11, r(256), r(256, 128) / 16, r(128), "silu")
    y, w5 = r(2, 24, 60, 32), [r(12, 12, 32, 32, 2) for _ in range(2)]
    gh = torch.complex(r(24, 60), r(24, 60))
    gf = ga.gexts
    return {
        "linear": lambda: ln.fused_linear(x, w, b, "relu", r(2, 300, 384) * 0 + 1, planes=1),
        "planes": lambda: ln.fused_linear(x, w, None, "none", planes=3),
        "input_grad": lambda: ln.linear_input_grad(x, r(128, 136) * 0 + 0.1),
        "masked": lambda: ln.linear_input_grad(x, w[:, :256].contiguous(), relu_output=torch.relu(ln.fused_linear(x, w[:, :256].contiguous()))),
        "packed": lambda: ln.packed_input_grad(torch.stack([q, k, v]).view(3, 600, 128), [w[:, i:i + 128].contiguous() for i in (0, 128, 256)], x.view(600, 128)),
        "weight_grad": lambda: ln.linear_weight_grad(x, q) + ln.linear_weight_grad(x, q, out_major=True),
        "weight_grad_batched": lambda: ln.linear_weight_grad_batched(x, torch.stack([q, k, v])),
        "attention": lambda: (out, ktv) + gf.galerkin_attention_fused_backward(r(2, 300, 136) * 0 + out, q, k, v, pos, *norm, 1e-6, ktv, 4, 2),
        "attention_forward": lambda: gf.galerkin_attention_fused_forward(q, k, v, None, *norm, 1e-6, 4, 0, return_ktv=True),
        "encoder_tail": lambda: ln.fused_encoder_tail(*tail),
        "modes_middle": lambda: dm._spectral_modes_middle(y, gh, gh.t().contiguous(), *w5),
        "conv3x3": lambda: dm.conv3x3(r(2, 8, 9, 11) * 0 + 1, r(12, 8, 3, 3) * 0 + 0.5, r(12) * 0, "silu", 2),
        "projection": lambda: gf.multihead_projection_layernorm_with_position_rrc_forward(x, w[:, :128].contiguous(), b[:128], norm[0], norm[1], 1e-5, pos, 300, 128, 4, 32, 2, 2),
        "cccr": lambda: (gf.multihead_galerkin_attention_cccr_forward(*heads, 2, 4, 34, 300),) + gf.multihead_galerkin_attention_cccr_backward(heads[0].transpose(2, 3).contiguous(), *heads, 2, 4, 34, 300),
        "layernorm": lambda: ga._layernorm_heads_backward(x.view(600, 128), q, norm[0], 1e-6, 4, 32),
    }


@pytest.mark.gpu
def test_same_results_as_the_python_operators(gpu, monkeypatch):
    """Bit for bit, shapes, strides and all."""
    flat = lambda t: [t] if isinstance(t, torch.Tensor) else list(t)
    native = {name: flat(call()) for name, call in _calls(gpu).items()}
    monkeypatch.setattr(_lib, "fast", _lib._NotBuilt())
    for name, call in _calls(gpu).items():
        for a, b in zip(native[name], flat(call()), strict=True):
            assert a.shape == b.shape and a.is_contiguous() == b.is_contiguous() and torch.equal(a, b), name
            assert not a.requires_grad


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
