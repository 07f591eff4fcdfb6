"""What the spectral layer's training route promises beside its kernels' numbers, on the CPU: the kernels' parts are played
by torch products that record nothing, as the kernels do."""
import pytest
import torch

from spgt_amd.network import truncated_dft as td


def _rows_forward(x, table, planar=True):
    return torch.einsum("nhwc,wk->nkhc", x.detach(), table).contiguous()


def _rows_inverse(u, table, planar=True):
    return torch.einsum("nkhc,wk->nhwc", u.detach(), table).contiguous()


def _modes_middle(y, gh, ghi, w1, w2):
    w = torch.view_as_complex(torch.cat([w1, w2]).detach())
    z = torch.einsum("kh,nwhc->nkwc", gh, torch.complex(y[:, 0::2], y[:, 1::2]).detach())
    u = torch.einsum("hk,nkwo->nwho", ghi, torch.einsum("nkwc,kwco->nkwo", z, w))
    return torch.stack([u.real, u.imag], dim=2).flatten(1, 2).contiguous()


def _inverse_linear(u, table, x, weight_kn, bias, activation):
    return x.detach() @ weight_kn.detach() + bias.detach() + _rows_inverse(u, table)


def _weight_adjoint(w1, w2, width):
    w = torch.view_as_complex(torch.stack([w1, w2]).detach()).conj().transpose(3, 4)  # [2, m, m, cout, cin]
    return torch.stack([torch.view_as_real(part.contiguous()) for part in w.resolve_conj().split(width, dim=4)])


def _input_grad_into(dx, c0, u, table, grad, weight):
    width = u.shape[3]
    dx[..., c0:c0 + width] = grad.detach() @ weight[:, c0:c0 + width] + _rows_inverse(u, table)


def _weight_grad(y, gh, du, gh_adjoint):
    z = torch.einsum("kh,nwhc->nkwc", gh, torch.complex(y[:, 0::2], y[:, 1::2]))
    d = torch.einsum("kh,nwho->nkwo", gh_adjoint, torch.complex(du[:, 0::2], du[:, 1::2]))
    return torch.view_as_real(torch.einsum("nkwc,nkwo->kwco", z.conj(), d).resolve_conj())


def _linear_weight_grad(x, g, out_major):
    return g.detach().t() @ x.detach(), g.detach().sum(0)


@pytest.fixture
def kernels(monkeypatch):
    for name, stand_in in (("truncated_dft_rows_forward", _rows_forward), ("truncated_dft_rows_inverse", _rows_inverse),
                           ("spectral_modes_middle", _modes_middle), ("spectral_inverse_linear", _inverse_linear),
                           ("_spectral_weight_adjoint", _weight_adjoint), ("_spectral_weight_grad", _weight_grad),
                           ("_spectral_linear_input_grad_into", _input_grad_into), ("linear_weight_grad", _linear_weight_grad),
                           ("inverse_table_operand", lambda table: table)):
        monkeypatch.setattr(td, name, stand_in)
    monkeypatch.setattr(td, "_TABLES", {})


def _layer(cin, cout, r=10, m=3):
    g = torch.Generator().manual_seed(0)
    rand = lambda *s: torch.randn(*s, generator=g).requires_grad_()
    x, w1, w2, w, b = rand(2, r, r, cin), rand(m, m, cin, cout, 2), rand(m, m, cin, cout, 2), rand(cout, cin), rand(cout)
    plain = x @ w.t() + b
    z = torch.fft.rfft2(x, dim=(1, 2), norm="ortho")
    kept = [torch.einsum("nklc,klco->nklo", part, torch.view_as_complex(weight))
            for part, weight in ((z[:, :m, :m], w1), (z[:, r - m:, :m], w2))]
    full = torch.zeros(2, r, r // 2 + 1, cout, dtype=torch.complex64)
    full = torch.cat([torch.cat([kept[0], full[:, m:r - m, :m], kept[1]], dim=1), full[:, :, m:]], dim=2)
    plain = plain + torch.fft.irfft2(full, s=(r, r), dim=(1, 2), norm="ortho")
    return td.spectral_linear_train(x, w1, w2, m, w, b, w.detach().t().contiguous()), plain, [x, w1, w2, w, b]


@pytest.mark.parametrize("cin,cout", [(32, 32), (64, 64), (64, 32), (128, 32), (128, 64)])
@pytest.mark.parametrize("through", [0, 1, 3], ids=["input", "fourier_weight", "linear_weight"])
def test_second_derivatives_are_refused(kernels, cin, cout, through):
    """The kernels record nothing: gradients taken under create_graph are right, and differentiating them again raises at
    every width instead of giving a part of the answer, whether dy depends on the input or not."""
    out, plain, leaves = _layer(cin, cout)
    dy = torch.randn(out.shape, generator=torch.Generator().manual_seed(1))
    want = torch.autograd.grad(plain, leaves, dy, retain_graph=True)
    once = torch.autograd.grad(out, leaves, dy, retain_graph=True)
    for g, w in zip(once, want):
        assert (g - w).norm() < 1e-5 * w.norm()
    for variable_dy in (dy, dy.clone().requires_grad_()):
        grads = torch.autograd.grad(out, leaves, variable_dy, create_graph=True)
        for g, w in zip(grads, want):
            assert (g - w).norm() < 1e-5 * w.norm()
        with pytest.raises(RuntimeError, match="twice"):
            (grads[through].square().sum() + plain.sum()).backward(retain_graph=True)
        # ... also where only some sources are asked for, and where another path leads to them
        for leaf in leaves[:4] + [variable_dy] * variable_dy.requires_grad:
            for value in (grads[through].square().sum(), grads[through].square().sum() + plain.sum()):
                with pytest.raises(RuntimeError, match="twice"):
                    torch.autograd.grad(value, leaf, allow_unused=True, retain_graph=True)


class _Recorder(torch.utils._python_dispatch.TorchDispatchMode):
    """The operators that ran on the device `kind`."""

    def __init__(self, kind):
        super().__init__()
        self.kind, self.seen = kind, []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if any(isinstance(a, torch.Tensor) and a.device.type == self.kind for a in args):
            self.seen.append(str(func))
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("r,m", [(10, 3), (43, 20)])
def test_tables_come_from_the_host_all_at_once(monkeypatch, r, m):
    """Kept tables are formed on the host and copied over, which waits for them: a kernel that formed one would be ordered
    on the stream of the first call alone, and belong to a graph if that call was captured.  The first pass in either
    direction brings those of the other along."""
    from spgt_amd.extension.bind import datamove
    monkeypatch.setattr(td, "_TABLES", {})
    monkeypatch.setattr(datamove, "_PADDED", {})
    host = td.dft_tables(r, m, "cpu")
    with _Recorder("meta") as recorder, torch.device("meta"), torch.inference_mode():
        fw, gh, ghi, fwi = td.dft_tables(r, m, "meta")
        td._operand_table(r, m, "meta")
        adjoint = td._adjoint_tables(r, m, "meta")
        padded = [datamove._padded(t, inverse) for t in (fw, fwi) for inverse in (False, True)]
    assert recorder.seen == [] and not fw.is_inference()
    assert all(t.device.type == "meta" for t in (fw, gh, ghi, fwi, *adjoint, *padded))
    # the same values as formed from the tables
    fw, gh, ghi, fwi = host
    for got, want in zip(td._adjoint_tables(r, m, "cpu"), (ghi.conj().t(), gh.conj().t(), datamove.inverse_table_operand(fw))):
        assert got.is_contiguous() and not got.is_conj() and torch.equal(got, want)
    assert torch.equal(td._operand_table(r, m, "cpu"), datamove.inverse_table_operand(fwi))
    for t in (fw, fwi):
        for inverse in (False, True):
            assert torch.equal(datamove._padded(t, inverse), datamove.pad_dft_table(t, inverse))
    count = lambda: [len(cache) for cache in (td._TABLES, datamove._PADDED)]
    before = count()
    td._adjoint_tables(r, m, "meta"), td._operand_table(r, m, "meta")
    assert count() == before


@pytest.mark.parametrize("query", ["spgt_spectral_linear_input_grad_supported", "spgt_spectral_weight_grad_supported"])
def test_training_asks_for_the_backward_kernels(monkeypatch, query):
    """The route is taken for the sizes that it was, and not where one of the backward's kernels has no form."""
    from spgt_amd import _lib
    lib = _lib.load()

    class Without:
        def __getattr__(self, name):
            return (lambda *sizes: 0) if name == query else getattr(lib, name)

    widths = [(32, 32), (64, 64), (64, 32), (128, 32), (128, 64)]
    sizes = [(r, cin, cout, m) for r in (8, 43, 64, 512) for m in (1, 4, 21, 32) if 2 * m <= r for cin, cout in widths]
    assert all(td.spectral_linear_trainable(*s) for s in sizes)
    assert not any(td.spectral_linear_trainable(*s) for s in ((64, 96, 32, 4), (64, 32, 64, 4), (64, 64, 64, 33), (1025, 32, 32, 4)))
    monkeypatch.setattr(_lib, "load", Without)
    assert not any(td.spectral_linear_trainable(*s) for s in sizes)
