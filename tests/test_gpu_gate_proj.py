"""The two gate projections of the GDN layer in one kernel (csrc/gdn_gate_proj.hip)."""
import types

import pytest
import torch

from engine.kernels import _lib
from engine.kernels.gdn_layer import _gate_projections

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs an MI355X")]

DEV = "cuda"


def randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device=DEV).bfloat16()


# one row, the edges of a row tile, and the last / first rows of each tile rule
@pytest.mark.parametrize("k,n", [(2048, 32), (2048, 16), (1024, 32), (1024, 16)])
@pytest.mark.parametrize("m", [1, 15, 17, 333, 1024, 1025, 2048, 2049, 4096, 4097, 8192, 8193, 8256])
def test_rows_and_tiles(m, k, n):
    gen = torch.Generator(device=DEV).manual_seed(m + k + n)
    x, w = randn(gen, m, k), [randn(gen, n, k) for _ in range(2)]
    out = _lib.host().gate_proj(x, *w)
    for y, wi in zip(out, w):
        ref = x.double() @ wi.double().t()
        # one rounding to bf16 (half an ulp: 2^-8 of the value), and fp32 sums of k products
        bound = ref.abs() * 2.0 ** -8 + k * 2.0 ** -24 * (x.double().abs() @ wi.double().abs().t())
        assert y.shape == (m, n) and y.dtype == torch.bfloat16 and ((y.double() - ref).abs() <= bound).all()


def layer(k=2048, n=32, bias=False, dtype=torch.bfloat16):
    lins = [torch.nn.Linear(k, n, bias=bias, device=DEV, dtype=dtype) for _ in range(2)]
    return types.SimpleNamespace(in_proj_b=lins[0], in_proj_a=lins[1])


def test_which_calls_take_the_kernel(monkeypatch):
    """Every form gives what the modules give; the kernel is taken by the plain one only."""
    host, took = _lib.host(), []
    spy = types.SimpleNamespace(gate_proj=lambda *a: took.append(r := host.gate_proj(*a)) or r)
    monkeypatch.setattr(_lib, "host", lambda: spy)
    x = torch.randn(3, 5, 2048, device=DEV).bfloat16()

    def check(lay, x, kernel, ctx=torch.no_grad):
        took.clear()
        with ctx():
            got = _gate_projections(lay, x)
            want = lay.in_proj_b(x), lay.in_proj_a(x)
        assert bool([t for t in took if t is not None]) == kernel
        for y, z in zip(got, want):
            assert y.shape == z.shape and y.dtype == z.dtype and y.requires_grad == z.requires_grad
            # both are fp32 sums rounded to bf16: at most one ulp apart, but for sums that cancel
            assert torch.allclose(y.float(), z.float(), rtol=2.0 ** -7, atol=1e-4 * z.float().abs().max().item())

    plain = layer()
    check(plain, x, True)
    check(plain, x[:, 1:], False)                                             # strided rows
    check(plain, x, False, torch.enable_grad)                                 # weights that record gradients
    check(plain, x, False, lambda: torch.autocast("cuda", torch.float16))
    check(layer(bias=True), x, False)
    check(layer(n=4), x, False)
    check(layer(k=512), x[..., :512].contiguous(), False)
    check(layer(dtype=torch.float32), x.float(), False)
    hooked = layer()
    hooked.in_proj_a.register_forward_hook(lambda m, a, y: y + 1)
    check(hooked, x, False)
