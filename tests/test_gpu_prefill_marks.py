"""A prefill's rows that continue from their slots: rows marked in
``GDNSlotPools.has_state()`` after ``bind`` (a prompt prefilled in pieces
beside a fresh one) on the MI355X, eagerly and in a captured graph.  A marked
row gives the bits of the same tokens bound as a continued (decode) batch."""
import types

import pytest
import torch

import layer_cases as lc
from engine.kernels import gated_delta_net_forward
from engine.runtime import GDNSlotPools

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs an MI355X")]

DEV = "cuda"
T = 20  # above the step length that takes the recurrence: conv and chunk kernels in every form


def test_marked_rows_continue_from_their_slots():
    _, layer = lc.gpu_layer("tiny", lc.load_golden())
    gen = torch.Generator().manual_seed(5)
    pools = GDNSlotPools.allocate([0], 6, conv_dim=2 * 2 * 128 + 4 * 128, num_v_heads=4, device=torch.device(DEV))
    cache = types.SimpleNamespace(gdn_slot_pools=pools)
    conv, rec = pools.layer(0)
    slots, x = torch.tensor([4, 1]), lc.bf16_inputs(gen, 2, T, 64).to(DEV, torch.bfloat16)

    def forward():
        with torch.no_grad():
            return gated_delta_net_forward(layer, x, cache_params=cache)

    pools.bind(slots[:1], is_prefill=True)
    with torch.no_grad():
        gated_delta_net_forward(layer, lc.bf16_inputs(gen, 1, 33, 64).to(DEV, torch.bfloat16), cache_params=cache)
    conv0, rec0 = conv.clone(), rec.clone()

    def reset():
        conv.copy_(conv0)
        rec.copy_(rec0)

    def want(prefill):  # slot 1 holds zeros: continuing it is the fresh row
        reset()
        pools.bind(slots, is_prefill=prefill)
        y = forward().clone()
        return y, conv.clone(), rec.clone()

    fresh, continued = want(True), want(False)
    assert not torch.equal(fresh[0][0], continued[0][0]) and torch.equal(fresh[0][1], continued[0][1])
    reset()
    pools.bind(slots, is_prefill=True)
    pools.has_state()[0] = True
    y = forward()
    for got, ref in zip((y, conv, rec), continued):
        assert torch.equal(got, ref)

    pools.bind(slots, is_prefill=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        static = forward()
    for marked in (True, False, True):
        reset()
        pools.bind(slots, is_prefill=True)
        pools.has_state()[0] = marked
        graph.replay()
        torch.cuda.synchronize()
        for got, ref in zip((static, conv, rec), continued if marked else fresh):
            assert torch.equal(got, ref), marked
