"""Which rows of a bound batch start from their slot, on the CPU: the rows'
marks (``has_state``) decide what the layer forward hands to the conv and the
chunk kernels (``read_slots``)."""
import types

import pytest
import torch

from engine.kernels import gdn_layer
from engine.runtime import GDN_PAD_SLOT, GDNSlotPools

PAD = GDN_PAD_SLOT


def pools(num_slots=6, max_batch=5):
    return GDNSlotPools.allocate([0], num_slots, conv_dim=16, num_v_heads=2, head_k_dim=4, head_v_dim=4,
                                 device=torch.device("cpu"), max_batch=max_batch)


def test_decode_rows_start_from_their_slots_and_prefill_rows_from_nothing():
    p = pools()
    p.bind(torch.tensor([3, 1, 3, 7]), is_prefill=False)  # a repeated and an unknown slot
    assert p.read_slots().tolist() == [3, 1, PAD, PAD]
    p.bind(torch.tensor([2, 5]), is_prefill=True)
    assert p.read_slots().tolist() == [PAD, PAD]
    p.bind(torch.tensor([4]), is_prefill=False, verify_tokens=2)
    assert p.read_slots().tolist() == [4] and p.read_slots().dtype == torch.int64


def test_marked_rows_of_a_prefill_continue_from_their_slots():
    """An engine marks single rows in has_state()'s persistent buffer (a prompt continued in pieces)."""
    p = pools()
    p.bind(torch.tensor([2, 5, 2, 0]), is_prefill=True)
    marks = p.has_state()
    marks[1:].fill_(True)
    assert p.read_slots().tolist() == [PAD, 5, PAD, 0]  # the repeat of slot 2 still has none
    marks[3] = False
    assert p.read_slots().tolist() == [PAD, 5, PAD, PAD]
    p.bind(torch.tensor([1, 2]), is_prefill=True)  # the next bind starts over
    assert p.read_slots().tolist() == [PAD, PAD]
    p.bind(torch.tensor([1, 2]), is_prefill=False)
    p.has_state()[0] = False
    assert p.read_slots().tolist() == [PAD, 2]


def test_rows_follow_the_batch_size():
    p = pools()
    assert p.slots().tolist() == [] and p.read_slots().tolist() == []
    for ids in ([1, 2, 3], [4], [5, 0, 2], [3, 1, 0]):
        p.bind(torch.tensor(ids), is_prefill=False)
        assert p.slots().tolist() == ids and p.has_state().tolist() == [True] * len(ids)
        assert p.slots().data_ptr() == p._slots.data_ptr() and p.has_state().data_ptr() == p._has_state.data_ptr()


@pytest.mark.parametrize("inference", [False, True])
def test_marks_count_in_inference_mode(inference):
    with torch.inference_mode(inference):
        p = pools()
        p.bind(torch.tensor([2, 5]), is_prefill=True)
    with torch.inference_mode():
        p.has_state()[1] = True
        assert p.read_slots().tolist() == [PAD, 5]


def test_the_forward_hands_the_marked_rows_to_conv_and_chunk(monkeypatch):
    p = pools()
    p.bind(torch.tensor([2, 5]), is_prefill=True)
    p.has_state()[1] = True
    read = []

    def conv(x, *a, read_indices, **kw):
        read.append(read_indices.tolist())
        return x

    def chunk(q, k, v, *a, read_indices, **kw):
        read.append(read_indices.tolist())
        return v, None

    monkeypatch.setattr(gdn_layer, "_conv1d_fn", conv)
    monkeypatch.setattr(gdn_layer, "_from_projections", chunk)
    monkeypatch.setattr(gdn_layer, "rms_norm_gated", lambda core, *a: core)

    class Layer(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.layer_idx, self.activation = 0, "silu"
            self.key_dim, self.value_dim, self.head_k_dim, self.head_v_dim = 4, 8, 4, 4
            self.in_proj_qkv, self.in_proj_z = torch.nn.Linear(8, 16), torch.nn.Linear(8, 8)
            self.in_proj_b, self.in_proj_a = torch.nn.Linear(8, 2), torch.nn.Linear(8, 2)
            self.conv1d = types.SimpleNamespace(weight=torch.zeros(16, 1, 4), bias=None)
            self.norm = types.SimpleNamespace(weight=torch.zeros(4), variance_epsilon=1e-6)
            self.A_log, self.dt_bias = torch.zeros(2), torch.zeros(2)
            self.out_proj = torch.nn.Linear(8, 8)

    Layer.__module__ = __name__
    gdn_layer._forward_on_pools(Layer(), torch.randn(2, 3, 8), p, None)
    assert read == [[PAD, 5], [PAD, 5]]


def apply_mask_to_padding_states(hidden_states, attention_mask):
    return hidden_states
