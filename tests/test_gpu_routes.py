"""Which kernel a call takes, at the lines of the dispatch rules (both sides
of a line are right; the rules say which one is faster).  A recurrence with
snapshots always runs the per-token kernel, so a call without them that takes
that kernel too gives its bits, and one that takes the token-block kernel
gives others (sums in another order)."""
import pytest
import torch

from engine.kernels import fused_recurrent_gated_delta_rule

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs an MI355X")]

DEV = "cuda"
FP32, BF16 = torch.float32, torch.bfloat16


# k and v head dims, type, sequences, v-heads, tokens, whether in token blocks
@pytest.mark.parametrize("kd,vd,dt,n,hv,t,blocks", [
    (256, 128, FP32, 24, 4, 4, True), (256, 256, BF16, 12, 4, 4, True),   # up to 12,288 state columns
    (256, 256, FP32, 16, 4, 4, False), (256, 256, BF16, 16, 4, 7, False), (256, 256, BF16, 16, 4, 8, True),
    (256, 128, BF16, 32, 4, 7, False), (256, 128, BF16, 32, 4, 8, True),
    (128, 256, BF16, 16, 4, 4, True),                                     # 16,384
    (128, 256, BF16, 13, 5, 5, False), (128, 256, FP32, 13, 5, 6, True),
    (128, 256, BF16, 33, 4, 11, False), (128, 256, BF16, 33, 4, 12, True),  # over 32,768
    (128, 128, BF16, 32, 4, 4, True), (128, 128, BF16, 33, 4, 7, False), (128, 128, BF16, 33, 4, 8, True),
    (128, 128, FP32, 65, 4, 15, False), (128, 128, FP32, 65, 4, 16, True),
    (64, 64, BF16, 256, 4, 16, True),                                     # 65,536
    (64, 64, BF16, 205, 5, 23, False), (64, 64, BF16, 205, 5, 24, True), (64, 64, FP32, 205, 5, 16, True),
])
def test_short_recurrences_take_the_faster_kernel(kd, vd, dt, n, hv, t, blocks):
    gen = torch.Generator(device=DEV).manual_seed(n + t)
    q, k = (torch.randn(n, t, hv, kd, generator=gen, device=DEV).to(dt) for _ in range(2))
    v = torch.randn(n, t, hv, vd, generator=gen, device=DEV).to(dt)
    g, beta = -torch.rand(n, t, hv, generator=gen, device=DEV), torch.rand(n, t, hv, generator=gen, device=DEV)
    h0 = torch.randn(n, hv, kd, vd, generator=gen, device=DEV)
    print(f"K={kd} V={vd} {dt} {n}x{t} Hv={hv}", flush=True)

    def last(**kw):
        return fused_recurrent_gated_delta_rule(q, k, v, g, beta, initial_state=h0, output_final_state=True,
                                                use_qk_l2norm_in_kernel=True, **kw)[1]
    one, other = last(), last(snapshots=torch.empty(n, t, hv, kd, vd, device=DEV))
    assert torch.equal(one, other) == (not blocks)
    assert (one - other).norm() <= 1e-5 * other.norm()
