"""The native host path (csrc/gdn_host.cpp) against the wrappers' general way.

Both launch the same kernels, so every form of call that the native path
takes must give the same bits as the general way (forced here by a host
object that declines every call), and every form that it leaves must still
run.  Forms: strides (contiguous, views of a packed projection, swapped
axes), one token or one sequence, each dtype, pools with ids, packed
sequences, snapshots, final states; the layer step on pools.
"""
import itertools
import types

import pytest
import torch

import layer_cases as lc
from engine.kernels import (_lib, causal_conv1d_fn, chunk_gated_delta_rule, chunk_gated_delta_rule_from_projections,
                            fused_recurrent_gated_delta_rule, fused_recurrent_gated_delta_rule_from_projections,
                            gated_delta_net_forward, gdn_in_proj_decode, gdn_out_proj_decode, rms_norm_gated)

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs an MI355X")]

DEV = "cuda"


class Declines:
    def __getattr__(self, name):
        return lambda *a: None


class Counts:
    """The host extension, counting the calls it took and naming them."""

    def __init__(self):
        self.host, self.took, self.names = _lib.host(), 0, set()

    def __getattr__(self, name):
        def call(*a):
            r = getattr(self.host, name)(*a)
            self.took += r is not None
            if r is not None:
                self.names.add(name)
            return r
        return call


def both(monkeypatch, make, call, native=True, names=None):
    """call(make()) natively and the general way: the same bits; whether the native path took it (and, with
    ``names``, which of its functions did)."""
    outs = []
    for host in (Counts(), Declines()):
        monkeypatch.setattr(_lib, "host", lambda h=host: h)
        a = make()
        r = call(a)
        outs.append([x for x in (r if isinstance(r, tuple) else (r,)) if x is not None] + [a.get("pool")])
        if isinstance(host, Counts):
            assert (host.took > 0) == native
            assert names is None or host.names == names
    monkeypatch.undo()
    for x, y in zip(*outs):
        if x is not None:
            assert x.shape == y.shape and x.dtype == y.dtype and x.stride() == y.stride() and torch.equal(x, y)


def qkv(gen, b, t, hk, hv, dt, form):
    if form == "packed":
        x = torch.randn(b, t, (2 * hk + hv) * 128, generator=gen).to(dt).to(DEV)
        q, k, v = torch.split(x, [hk * 128, hk * 128, hv * 128], -1)
        return q.unflatten(-1, (hk, 128)), k.unflatten(-1, (hk, 128)), v.unflatten(-1, (hv, 128))
    if form == "heads first":  # swapped axes: copied by the general way
        return tuple(torch.randn(b, h, t, 128, generator=gen).to(dt).to(DEV).transpose(1, 2) for h in (hk, hk, hv))
    return tuple(torch.randn(b, t, h, 128, generator=gen).to(dt).to(DEV) for h in (hk, hk, hv))


@pytest.mark.parametrize("dt,form", itertools.product((torch.bfloat16, torch.float16, torch.float32),
                                                      ("contiguous", "packed", "heads first")))
def test_recurrent_and_chunk_calls(monkeypatch, dt, form):
    hk, hv = 2, 4
    for n, (b, t, mode) in enumerate([(1, 1, "none"), (3, 1, "pool"), (2, 5, "states"), (1, 70, "cu"), (2, 3, "snap"),
                                      (1, 2, "bf16 beta"), (2, 65, "final")]):
        def make():
            gen = torch.Generator().manual_seed(n)
            q, k, v = qkv(gen, b, t, hk, hv, dt, form)
            g, beta = -torch.rand(b, t, hv, generator=gen).to(DEV), torch.rand(b, t, hv, generator=gen).to(DEV)
            a = dict(q=q, k=k, v=v, g=g, beta=beta, kw={})
            if mode == "bf16 beta":
                a["beta"] = beta.bfloat16()
            if mode in ("pool", "states", "snap"):
                a["pool"] = torch.randn(5 if mode == "pool" else b, hv, 128, 128, generator=gen).to(DEV)
                a["kw"] = dict(initial_state=a["pool"])
            if mode == "pool":
                a["kw"].update(ssm_state_indices=torch.tensor([4, 1, 4], device=DEV), inplace_final_state=True)
            if mode == "cu":
                a["kw"] = dict(cu_seqlens=torch.tensor([0, 3, 3, 70], dtype=torch.int32, device=DEV), output_final_state=True)
            if mode in ("states", "final"):
                a["kw"].update(output_final_state=True)
            return a

        regular = form != "heads first" or t == 1  # (one token: the axes' order is no matter)
        args = lambda a: (a["q"], a["k"], a["v"], a["g"], a["beta"])  # noqa: E731
        print(f"B={b} T={t} {mode}", flush=True)
        if mode == "snap":
            both(monkeypatch, make, lambda a: fused_recurrent_gated_delta_rule(
                *args(a), snapshots=(s := torch.empty(b, t, hv, 128, 128, device=DEV)), **a["kw"]) + (s,), regular)
            continue
        both(monkeypatch, make, lambda a: fused_recurrent_gated_delta_rule(*args(a), use_qk_l2norm_in_kernel=True, **a["kw"]),
             regular)
        both(monkeypatch, make, lambda a: chunk_gated_delta_rule(*args(a), use_qk_l2norm_in_kernel=True, scale=0.1, **a["kw"]),
             regular)
        alog, dtb = torch.linspace(-1, 1, hv, device=DEV), torch.linspace(-1, 0, hv, device=DEV).bfloat16()
        for f in (fused_recurrent_gated_delta_rule_from_projections, chunk_gated_delta_rule_from_projections):
            both(monkeypatch, make, lambda a: f(a["q"], a["k"], a["v"], a["g"].to(dt), a["g"].flip(1).to(dt), alog, dtb,
                                                **a["kw"]), regular)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
def test_conv_norm_and_projection_calls(monkeypatch, dt):
    def gen():
        return torch.Generator().manual_seed(3)

    for b, t, c, mode in [(1, 9, 64, "tokens"), (2, 5, 64, "bct"), (3, 1, 64, "pool"), (1, 9, 64, "cu"), (2, 5, 64, "ctb")]:
        def make():
            g = gen()
            x = torch.randn(b, t, c, generator=g).to(dt).to(DEV)
            x = x[0] if mode in ("tokens", "cu") else x.transpose(1, 2) if mode != "ctb" else x.transpose(1, 2).contiguous()
            a = dict(x=x, w=torch.randn(c, 4, generator=g).to(dt).to(DEV), bias=torch.randn(c, generator=g).to(dt).to(DEV), kw={})
            if mode in ("pool", "cu"):
                a["pool"] = torch.randn(6, c, 4, generator=g).to(dt).to(DEV)
                a["kw"] = dict(conv_states=a["pool"], cache_indices=torch.tensor([5, -1, 2][:3 if mode == "pool" else 2], device=DEV))
            if mode == "cu":
                a["kw"]["cu_seqlens"] = torch.tensor([0, 4, 9], dtype=torch.int32, device=DEV)
            return a
        both(monkeypatch, make, lambda a: causal_conv1d_fn(a["x"], a["w"], a["bias"], "silu", **a["kw"]), mode != "ctb")

    def rows():
        g = gen()
        return dict(x=torch.randn(3, 2, 4, 128, generator=g).to(dt).to(DEV), z=torch.randn(3, 2, 4, 128, generator=g).to(dt).to(DEV),
                    w=torch.randn(128, generator=g).to(DEV))
    both(monkeypatch, rows, lambda a: rms_norm_gated(a["x"], a["z"], a["w"], 1e-5))
    both(monkeypatch, rows, lambda a: rms_norm_gated(a["x"][:, :, :2], a["z"][:, :, :2], a["w"]), False)
    if dt != torch.bfloat16:
        return

    def proj():
        g = gen()
        r = lambda *s: torch.randn(*s, generator=g).to(dt).to(DEV)  # noqa: E731
        return dict(x=r(5, 1, 1024), w=[r(n, 1024) for n in (1024, 512, 4, 4)], cw=r(1024, 1, 4), pool=r(8, 1024, 4),
                    idx=torch.tensor([3, 0, 3, -1, 7], device=DEV), wo=r(128, 1024))
    both(monkeypatch, proj, lambda a: gdn_in_proj_decode(a["x"], *a["w"], a["cw"], None, a["pool"], a["idx"], "silu"))
    both(monkeypatch, proj, lambda a: gdn_in_proj_decode(a["x"], *a["w"], a["cw"], None, a["pool"], a["idx"].int(), None), False)
    both(monkeypatch, proj, lambda a: gdn_out_proj_decode(a["x"], a["wo"]))
    both(monkeypatch, proj, lambda a: gdn_out_proj_decode(a["x"][:, 0, ::2].repeat(1, 2)[:, ::1], a["wo"]))
    both(monkeypatch, proj, lambda a: gdn_out_proj_decode(a["x"].transpose(0, 2).contiguous().transpose(0, 2), a["wo"]), False)


@pytest.mark.parametrize("rows,prefill,t", [(3, False, 1), (1, False, 1), (2, True, 70), (2, False, 5), (2, False, 40)])
def test_layer_on_pools(monkeypatch, rows, prefill, t):
    from engine.runtime import GDNSlotPools
    _, layer = lc.gpu_layer("w1024", lc.load_golden())

    def make():
        gen = torch.Generator().manual_seed(rows)
        conv = {0: torch.randn(6, 2 * 2 * 128 + 4 * 128, 4, generator=gen).bfloat16().to(DEV)}
        rec = {0: torch.randn(6, 4, 128, 128, generator=gen).to(DEV)}
        pools = GDNSlotPools(conv, rec)
        pools.bind(torch.tensor([4, 4, 9][:rows]), is_prefill=prefill)  # a repeated and an unknown slot
        return dict(pool=rec[0], pools=pools, x=torch.randn(rows, t, 1024, generator=gen).bfloat16().to(DEV))

    def call(a):
        with torch.no_grad():
            y = gated_delta_net_forward(layer, a["x"], cache_params=types.SimpleNamespace(gdn_slot_pools=a["pools"]))
        return y, a["pools"].layer(0)[0]
    # (the fixture layer's 4 heads: its b and a stay modules in longer steps)
    names = {"in_proj", "core_decode", "out_proj"} if t == 1 else {"conv", "chunk" if t > 16 else "recurrent", "rms_norm"}
    both(monkeypatch, make, call, names=names)
