"""Forms of the layer and its modules that the fused forward accepts, on the CPU:
bare objects with the same attributes, and which modules the two gate
projections leave to their own calls (no kernel runs here; the host extension
is a stand-in that takes every call)."""
import types

import pytest
import torch
import torch.utils._python_dispatch

from engine.kernels import _lib, gdn_layer
from engine.kernels.gdn_layer import _gate_projections

TAKEN = ("b from the kernel", "a from the kernel")


def layer():
    lins = [torch.nn.Linear(8, 4, bias=False, dtype=torch.bfloat16).requires_grad_(False) for _ in range(2)]
    return types.SimpleNamespace(in_proj_b=lins[0], in_proj_a=lins[1])


class Doubles(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        y = func(*args, **(kwargs or {}))
        return y * 2 if func is torch.nn.functional.linear else y


class Observes(torch.utils._python_dispatch.TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def own_hook(lay, monkeypatch):
    lay.in_proj_a.register_forward_hook(lambda m, a, y: y + 1)


def backward_hook(lay, monkeypatch):
    lay.in_proj_b.register_full_backward_hook(lambda m, gi, go: None)


def own_forward(lay, monkeypatch):
    forward = lay.in_proj_b.forward
    lay.in_proj_b.forward = lambda x: forward(x) + 1


def class_forward(lay, monkeypatch):
    forward = torch.nn.Linear.forward
    monkeypatch.setattr(torch.nn.Linear, "forward", lambda self, x: forward(self, x) + 1)


def every_module(register):
    def set_up(lay, monkeypatch):
        return register()
    return set_up


nn_module = torch.nn.modules.module
FORMS = {
    "own hook": own_hook, "backward hook": backward_hook, "own forward": own_forward, "class forward": class_forward,
    "hook of all modules": every_module(lambda: nn_module.register_module_forward_hook(lambda m, a, y: y + 1)),
    "pre-hook of all modules": every_module(
        lambda: nn_module.register_module_forward_pre_hook(lambda m, a: (a[0] + 1,))),
}


def check(lay, taken):
    x = torch.randn(2, 3, 8).bfloat16()
    got = _gate_projections(lay, x)
    if taken:
        assert got == TAKEN
    else:
        for y, want in zip(got, (lay.in_proj_b(x), lay.in_proj_a(x))):
            assert torch.equal(y, want)


@pytest.fixture
def takes_all(monkeypatch):
    monkeypatch.setattr(_lib, "host", lambda: types.SimpleNamespace(gate_proj=lambda *a: TAKEN))


def test_plain_gate_projections_take_the_kernel(takes_all):
    check(layer(), True)


@pytest.mark.parametrize("form", FORMS)
def test_gate_projections_that_do_more_than_their_product_run_as_modules(takes_all, monkeypatch, form):
    lay = layer()
    handle = FORMS[form](lay, monkeypatch)
    try:
        check(lay, False)
    finally:
        if handle is not None:
            handle.remove()
    if handle is not None:
        check(lay, True)


@pytest.mark.parametrize("mode", [Doubles, Observes])
def test_gate_projections_under_a_mode_run_as_modules(takes_all, mode):
    lay = layer()
    with mode():
        check(lay, False)
    check(lay, True)


def plain_objects(kind, k=1024):
    """A layer's projections as bare objects that hold a weight and a bias, in a bare layer object or a module."""
    def lin(*shape):
        return types.SimpleNamespace(weight=torch.zeros(*shape, dtype=torch.bfloat16), bias=None)

    lay = types.SimpleNamespace() if kind == "layer" else torch.nn.Module()
    lay.in_proj_qkv, lay.in_proj_z, lay.in_proj_b, lay.in_proj_a = lin(1024, k), lin(512, k), lin(4, k), lin(4, k)
    lay.conv1d = lin(1024, 1, 4)
    lay.activation = "silu"
    return lay


@pytest.mark.parametrize("kind", ["layer", "projections"])
def test_layers_and_projections_need_not_be_modules(monkeypatch, kind):
    lay = plain_objects(kind)
    windows = torch.zeros(3, 1024, 4, dtype=torch.bfloat16)
    assert gdn_layer._fused_decode_fits(lay, torch.zeros(2, 1, 1024).bfloat16(), windows)
    assert not gdn_layer._fused_decode_fits(lay, torch.zeros(2, 1, 512).bfloat16(), windows)
    seen = []
    monkeypatch.setattr(gdn_layer, "gdn_in_proj_decode", lambda *a: seen.append(a))
    gdn_layer._fused_decode(lay, "x", windows, "slots")
    names = ("in_proj_qkv", "in_proj_z", "in_proj_b", "in_proj_a")
    assert all(a is getattr(lay, n).weight for a, n in zip(seen[0][1:5], names))
    assert seen[0][5] is lay.conv1d.weight and seen[0][6] is None
    # between the projections such a layer goes the general way
    assert gdn_layer._native_core(types.SimpleNamespace(), *(None,) * 6) is None
