"""The native layout key of launch plans (csrc/layout.cpp): it changes exactly
when the attribute-by-attribute key (``_lib.layout_key``) does."""

import sys
import types

import pytest
import torch

from triton_muon_adamw import _build, _lib


def _params():
    ps = [torch.nn.Parameter(torch.randn(4, 6)), torch.nn.Parameter(torch.randn(3)), torch.zeros(()),
          torch.nn.Parameter(torch.randn(5, 2, 2)), torch.nn.Parameter(torch.randn(7))]
    for p in ps[:4]:
        p.grad = torch.randn_like(p)
    return ps


def test_layout_follows_every_attribute():
    ps = _params()
    active, key = _lib.layout(ps)
    assert isinstance(key, bytes)  # the native path
    assert [id(p) for p in active] == [id(p) for p in ps[:4]]
    assert _lib.layout(list(ps))[1] == key
    ps[0].data.add_(1.0)  # values do not matter
    ps[1].grad.zero_()
    assert _lib.layout(ps)[1] == key
    other = torch.nn.Parameter(ps[1].data)  # another parameter over the same memory
    other.grad = ps[1].grad
    data, grad = ps[0].data, ps[0].grad

    def swap(d, g):
        ps[0].grad = None
        ps[0].data = d
        ps[0].grad = g

    base = [_lib.layout_key(p) for p in ps[:4]]
    changes = [
        lambda: swap(data.clone(), grad),                              # parameter address
        lambda: swap(data, grad.clone()),                              # gradient address
        lambda: swap(data.view(6, 4), grad.view(6, 4)),                # shape, same address
        lambda: swap(data.as_strided((4, 6), (1, 4)), grad),           # strides
        lambda: swap(data, grad.as_strided((4, 6), (1, 4))),           # gradient strides
        lambda: swap(data.view(torch.int32)[:, :6].view(torch.float32)[:3], grad[:3]),  # fewer rows
        lambda: ps.append(other),                                      # one more
        lambda: ps.__setitem__(1, other),                              # another object
        lambda: ps.reverse(),                                          # order
        lambda: setattr(ps[1], "grad", None),                          # one less
    ]
    for i, change in enumerate(changes):
        change()
        got = _lib.layout(ps)
        assert got[1] != key, i
        assert [_lib.layout_key(p) for p in got[0]] != base, i
        ps[:] = ps[:5] if i == 6 else ps
        if i == 7:
            ps[1] = active[1]
        if i == 8:
            ps.reverse()
        if i < 6:
            swap(data, grad)
        if i < 9:
            assert _lib.layout(ps)[1] == key, i
    half = torch.nn.Parameter(torch.zeros(4, dtype=torch.bfloat16))  # element type, same address and shape
    half.grad = torch.zeros(4, dtype=torch.bfloat16)
    before = _lib.layout([half])[1]
    bits, gbits = half.data, half.grad
    half.grad = None
    half.data = bits.view(torch.float16)
    half.grad = gbits.view(torch.float16)
    assert _lib.layout([half])[1] != before


def test_layout_of_other_sequences_and_subclasses():
    class Sub(torch.Tensor):
        pass

    ps = _params()
    ref = tuple(_lib.layout_key(p) for p in ps[:4])
    assert _lib.layout(tuple(ps)) == (ps[:4], ref)
    sub = torch.zeros(3).as_subclass(Sub)
    sub.grad = torch.zeros(3)
    assert _lib.layout([*ps, sub]) == ([*ps[:4], sub], (*ref, _lib.layout_key(sub)))
    assert _lib.layout([]) [0] == []


def test_layout_of_a_subclass_gradient():
    """A gradient of a subclass is read through its own attributes, also on a plain parameter."""
    class Moved(torch.Tensor):
        offset = 0

        def data_ptr(self):
            return super().data_ptr() + self.offset

    ps = _params()
    ps[1].grad = torch.zeros(3).as_subclass(Moved)
    active, key = _lib.layout(ps)
    assert active == ps[:4] and key == tuple(_lib.layout_key(p) for p in ps[:4])
    ps[1].grad.offset = 4
    assert _lib.layout(ps)[1] != key
    ps[1].grad = torch.nn.Parameter(torch.zeros(3))  # as plain as a tensor
    assert isinstance(_lib.layout(ps)[1], bytes)


@pytest.mark.parametrize("module", [None, types.SimpleNamespace(torch_version="0.0.1", layout=lambda params: 1 / 0)],
                         ids=["missing", "of_another_torch"])
def test_layout_without_the_native_module(monkeypatch, module):
    """Built for another Python or torch, or not built: the same parameters and
    keys that follow the same changes, after one warning."""
    import triton_muon_adamw

    monkeypatch.setattr(_lib, "_layout", None)
    monkeypatch.setitem(sys.modules, "triton_muon_adamw._layout", module)  # None: the import fails
    monkeypatch.delattr(triton_muon_adamw, "_layout", raising=False)
    if module is not None:
        monkeypatch.setattr(triton_muon_adamw, "_layout", module, raising=False)
    ps = _params()
    with pytest.warns(RuntimeWarning, match="launch plans are compared in Python") as seen:
        active, key = _lib.layout(ps)
        assert _lib.layout(ps)[1] == key
    assert len(seen) == 1
    assert [id(p) for p in active] == [id(p) for p in ps[:4]] and key == tuple(_lib.layout_key(p) for p in ps[:4])
    ps[0].grad = ps[0].grad.clone()
    assert _lib.layout(ps)[1] != key


def test_build_without_a_compiler_for_the_native_module(monkeypatch, tmp_path):
    """The kernels' build goes on, and no module of an older build is left to be loaded."""
    stale = tmp_path / "_layout.so"
    stale.write_bytes(b"")
    monkeypatch.setattr(_build, "LAYOUT_PATH", stale)
    for cxx in (str(tmp_path / "no-such-compiler"), "false"):
        monkeypatch.setenv("CXX", cxx)
        with pytest.warns(RuntimeWarning, match="was not built"):
            _build._build_layout(verbose=False)
        assert not stale.exists()
