"""custom_kernel's native call (csrc/fp8bs_torch.cpp) against its Python path, over the forms of data that both see: what one
accepts the other accepts with the same bits, what one refuses the other refuses with the same type of exception."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


class _Sub(torch.Tensor):
    pass


def _kmajor(t):
    return t.t().contiguous().t()


def _data(m, n, k, dev, seed=5):
    gen = torch.Generator().manual_seed(seed)
    def f8(r):
        return _kmajor(torch.randn(r, k, generator=gen).to(torch.float8_e4m3fn)).to(dev)
    def scale(r):
        return _kmajor(torch.rand(r, k // 128, generator=gen) + 0.5).to(dev)
    return [f8(m), f8(n), scale(m), scale((n + 127) // 128), torch.zeros(m, n, dtype=torch.bfloat16, device=dev)]


def _with(i, change):
    def form(d):
        d[i] = change(d[i])
        return tuple(d)
    return form


FORMS = {
    "tuple": tuple, "list": list, "four": lambda d: tuple(d[:4]), "subclass": _with(4, lambda t: t.as_subclass(_Sub)), "parameter": _with(2, lambda t: torch.nn.Parameter(t)),
    "a row-major": _with(0, lambda t: t.contiguous()), "b row-major": _with(1, lambda t: t.contiguous()), "a_scale row-major": _with(2, lambda t: t.contiguous()),
    "b_scale row-major": _with(3, lambda t: t.contiguous()), "c transposed": _with(4, lambda t: torch.zeros_like(t).t().contiguous().t()), "c float": _with(4, lambda t: t.float()),
    "c padded": _with(4, lambda t: torch.zeros(t.shape[0], t.shape[1] + 8, dtype=t.dtype, device=t.device)[:, :t.shape[1]]),
    "c short": _with(4, lambda t: t[:-1]), "a bytes": _with(0, lambda t: t.view(torch.uint8)), "a_scale half": _with(2, lambda t: t.half()), "b_scale short": _with(3, lambda t: t[:-1]),
    "b_scale short in k": _with(3, lambda t: t[:, :-1]), "b short in k": _with(1, lambda t: t[:, :-128]), "a offset by a byte": _with(0, lambda t: torch.empty(t.numel() + 1, dtype=torch.uint8, device=t.device)[1:]
        .view(t.shape[1], t.shape[0]).copy_(t.t().view(torch.uint8)).view(t.dtype).t()), "a on the CPU": _with(0, lambda t: t.cpu()), "c 3-D": _with(4, lambda t: t[None]),
    "none": _with(3, lambda t: None),
}


# (96 x 384 x 512: no workspace.  64 x 1536 x 7168: one.  The rest: dimensions of one element, and of one block, whose strides may be any)
@pytest.mark.parametrize("m,n,k", [(96, 384, 512), (64, 1536, 7168), (1, 384, 512), (96, 128, 512), (96, 1, 512), (96, 384, 128), (2, 129, 256)])
def test_forms(pkg, dev, m, n, k, monkeypatch):
    lib = importlib.import_module("amd-developer-challenge-2025_amd._lib")
    native = lib.dense()
    assert native is not None, "build() builds it"

    def outcome(form, fn):
        monkeypatch.setattr(lib, "_dense", fn)
        data = form(_data(m, n, k, dev))
        try:
            out = pkg.custom_kernel(data)
        except Exception as ex:
            return type(ex), None
        assert out is data[4]
        return None, out.as_subclass(torch.Tensor).cpu().view(torch.int16)

    taken = []
    def counted(*args):
        taken.append(native(*args))
        return taken[-1]

    for name, form in FORMS.items():
        want, bits = outcome(form, None)                          # (this plans the size too)
        if name == "tuple" and want is not None:
            pytest.fail("%s" % want)
        got, same = outcome(form, counted)
        assert got is want, (name, got, want)
        assert want is not None or torch.equal(bits, same), name
        if name in ("tuple", "list", "parameter", "a offset by a byte"):
            assert taken[-1] == 0, (name, taken)                                           # who took it


def test_goes_to_the_current_stream(pkg, dev):
    """An operand written on a side stream behind a long kernel is seen by a call on that stream."""
    data = tuple(_data(64, 384, 512, dev))
    want = pkg.custom_kernel(data).clone()
    a = data[0].clone(memory_format=torch.preserve_format)
    big = torch.randn(4096, 4096, device=dev)
    data[0].view(torch.uint8).zero_()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        for _ in range(20):
            big = big @ big * 1e-4
        data[0].copy_(a)
        got = pkg.custom_kernel(data).clone()
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_traced_tensors_are_refused(pkg, dev):
    """A tensor that vmap wraps has no storage: the error of the Python path, and the next call is well."""
    data = _data(96, 384, 512, dev)
    pkg.custom_kernel(tuple(data))
    with pytest.raises((RuntimeError, ValueError)):
        torch.func.vmap(lambda s: pkg.custom_kernel((data[0], data[1], s, data[3], data[4])))(torch.stack([data[2].t(), data[2].t()]).transpose(1, 2))
    pkg.custom_kernel(tuple(data))
