"""GPU parity at the edges of the gates, through every prefill path and the
decode recurrence, against the token recurrence of the CPU oracle (fp64).

Gates per (token, v-head) drawn from a mix of the values a model produces at
its limits: no decay (g = 0), a decay strong enough that e^g, and every
product of it with the chunk's cumulative sums, underflows fp32 (g = -40:
e^{-40} = 4e-18, a chunk's cumsum reaches -2560), and ordinary decays;
beta exactly 0 (no update), exactly 1 and in between.  The chunk form exps
only non-positive differences of the cumsum, so nothing overflows; entries
that underflow are zero in fp32 and negligible in fp64 alike.

Paths: one sequence (prep + scan), three sequences (the column scan),
six packed sequences (the per-pair kernel, 192 (sequence, v-head) pairs).
Tolerances as everywhere: bf16 outputs max abs error 2e-2, fp32 final
states relative error 1e-3 norm-wise per (sequence, head); the fp32
recurrence 1e-4 / 1e-5.  One exception, with its reason: the final states
of the chunk paths when no token decays and every token writes in full
(test_chunk_prefill_with_full_updates).
"""
import numpy as np
import pytest
import torch

from engine.kernels import chunk_gated_delta_rule, fused_recurrent_gated_delta_rule
from oracle import gdn

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs an MI355X")]

DEV = "cuda"
HK, HV, D = 16, 32, 128


def np64(t):
    return t.detach().float().cpu().numpy().astype(np.float64)


def extreme_gates(shape, gen):
    """g in {0, -40, -U(0, 3)} and beta in {0, 1, U(0, 1)}, each a third of the entries."""
    pick_g = torch.randint(0, 3, shape, generator=gen)
    g = torch.where(pick_g == 0, torch.zeros(shape),
                    torch.where(pick_g == 1, torch.full(shape, -40.0), -3.0 * torch.rand(shape, generator=gen)))
    pick_b = torch.randint(0, 3, shape, generator=gen)
    beta = torch.where(pick_b == 0, torch.zeros(shape),
                       torch.where(pick_b == 1, torch.ones(shape), torch.rand(shape, generator=gen)))
    return g, beta


def packed_inputs(lens, seed):
    gen = torch.Generator().manual_seed(seed)
    t = sum(lens)
    q = torch.randn(1, t, HK, D, generator=gen).bfloat16()
    k = torch.randn(1, t, HK, D, generator=gen).bfloat16()
    v = torch.randn(1, t, HV, D, generator=gen).bfloat16()
    g, beta = extreme_gates((1, t, HV), gen)
    h0 = torch.randn(len(lens), HV, D, D, generator=gen) * 0.1
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    return q, k, v, g, beta, h0, cu


@pytest.mark.parametrize("lens,seed", [([300], 1), ([200, 77, 130], 2), ([150, 64, 1, 90, 200, 33], 3)],
                         ids=["prep_scan", "column_scan", "per_pair"])
def test_chunk_prefill_at_extreme_gates(lens, seed):
    q, k, v, g, beta, h0, cu = packed_inputs(lens, seed)
    o_ref, s_ref = gdn.recurrent_gated_delta_rule_varlen(
        *(x.float().numpy() for x in (q, k, v, g, beta)), cu, initial_state=h0.numpy())
    kw = {} if len(lens) == 1 else {"cu_seqlens": torch.tensor(cu, dtype=torch.int32, device=DEV)}
    o, s = chunk_gated_delta_rule(*(x.to(DEV) for x in (q, k, v, g, beta)), initial_state=h0.to(DEV),
                                  output_final_state=True, use_qk_l2norm_in_kernel=True, **kw)
    assert torch.isfinite(o).all() and torch.isfinite(s).all()
    assert np.abs(np64(o) - o_ref).max() < 2e-2
    assert gdn.state_rel_err(np64(s), s_ref) < 1e-3


@pytest.mark.parametrize("g_val,s_tol", [(-0.05, 1e-3), (0.0, 3e-3)], ids=["slow_decay", "no_decay"])
@pytest.mark.parametrize("b", [1, 3, 6], ids=["prep_scan", "column_scan", "per_pair"])
def test_chunk_prefill_with_full_updates(b, g_val, s_tol):
    """beta = 1 on every token and a uniform decay, 300 tokens per sequence.

    The chunk form's V' = U - W S cancels heavily when the state already
    holds the values (U and W S nearly equal), and its W and S are single
    bf16 MFMA operands (as in fla's chunk kernel): without decay the final
    states end 2.0e-3 from the recurrence at 300 tokens (2.4e-3 at 1024; a
    numpy emulation of the operand rounding gives the same figures), so the
    no-decay case is held to 3e-3, not the 1e-3 of the configurations.
    From a decay of 0.01 per token the error is back under 1e-3 (9.7e-4;
    1.5e-4 at 0.05, checked here).  Outputs stay within 2e-3 throughout."""
    gen = torch.Generator().manual_seed(4)
    t = 300
    q = torch.randn(1, b * t, HK, D, generator=gen).bfloat16()
    k = torch.randn(1, b * t, HK, D, generator=gen).bfloat16()
    v = torch.randn(1, b * t, HV, D, generator=gen).bfloat16()
    g, beta = torch.full((1, b * t, HV), g_val), torch.ones(1, b * t, HV)
    cu = np.arange(b + 1, dtype=np.int64) * t
    o_ref, s_ref = gdn.recurrent_gated_delta_rule_varlen(*(x.float().numpy() for x in (q, k, v, g, beta)), cu)
    kw = {} if b == 1 else {"cu_seqlens": torch.tensor(cu, dtype=torch.int32, device=DEV)}
    o, s = chunk_gated_delta_rule(*(x.to(DEV) for x in (q, k, v, g, beta)), output_final_state=True,
                                  use_qk_l2norm_in_kernel=True, **kw)
    assert np.abs(np64(o) - o_ref).max() < 2e-2
    assert gdn.state_rel_err(np64(s), s_ref) < s_tol


def test_recurrence_at_extreme_gates():
    """fp32 multi-token recurrence and a bf16 decode step on a slot pool."""
    gen = torch.Generator().manual_seed(5)
    b, t = 3, 40
    q, k = torch.randn(b, t, HK, D, generator=gen), torch.randn(b, t, HK, D, generator=gen)
    v = torch.randn(b, t, HV, D, generator=gen)
    g, beta = extreme_gates((b, t, HV), gen)
    h0 = torch.randn(b, HV, D, D, generator=gen) * 0.1
    o_ref, s_ref = gdn.recurrent_gated_delta_rule(*(x.numpy() for x in (q, k, v, g, beta)), initial_state=h0.numpy())
    o, s = fused_recurrent_gated_delta_rule(*(x.to(DEV) for x in (q, k, v, g, beta)), initial_state=h0.to(DEV),
                                            output_final_state=True, use_qk_l2norm_in_kernel=True)
    assert np.abs(np64(o) - o_ref).max() < 1e-4
    assert gdn.state_rel_err(np64(s), s_ref) < 1e-5

    bsz = 24
    q, k = (torch.randn(bsz, 1, HK, D, generator=gen).bfloat16() for _ in range(2))
    v = torch.randn(bsz, 1, HV, D, generator=gen).bfloat16()
    g, beta = extreme_gates((bsz, 1, HV), gen)
    pool0 = torch.randn(32, HV, D, D, generator=gen) * 0.1
    slots = torch.randperm(32, generator=gen)[:bsz]
    o_ref, pool_ref = gdn.slot_recurrent_step(pool0.numpy(), slots.numpy(),
                                              *(x.float().numpy() for x in (q, k, v, g, beta)))
    pool = pool0.to(DEV)
    o, _ = fused_recurrent_gated_delta_rule(*(x.to(DEV) for x in (q, k, v, g, beta)), initial_state=pool,
                                            ssm_state_indices=slots.to(DEV), inplace_final_state=True,
                                            use_qk_l2norm_in_kernel=True)
    assert np.abs(np64(o) - o_ref).max() < 2e-2
    assert gdn.state_rel_err(np64(pool[slots]), pool_ref[slots.numpy()]) < 1e-3
