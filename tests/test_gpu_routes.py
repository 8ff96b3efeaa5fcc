"""Which kernels a call takes, at the lines of the dispatch rules (both sides
of a line are right; the rules say which one is faster).  A recurrence with
snapshots always runs the per-token kernel, so a call without them that takes
that kernel too gives its bits, and one that takes the token-block kernel
gives others (sums in another order).  Other routes are read off the launches that a
call records into a graph."""
import ctypes

import pytest
import torch

from engine.kernels import _lib, causal_conv1d_fn, chunk_gated_delta_rule, fused_recurrent_gated_delta_rule

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


class Dim3(ctypes.Structure):
    _fields_ = [(n, ctypes.c_uint32) for n in "xyz"]


class KernelNode(ctypes.Structure):  # hipKernelNodeParams
    _fields_ = [("block", Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", Dim3),
                ("params", ctypes.c_void_p), ("shared", ctypes.c_uint32)]


def grids_of(call):
    """The grids of the kernels that ``call`` records into a graph."""
    call()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        call()
    with open("/proc/self/maps") as f:  # the runtime that torch loaded
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64.so" in line))
    count, raw = ctypes.c_size_t(), ctypes.c_void_p(graph.raw_cuda_graph())
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(count)) == 0
    nodes, grids = (ctypes.c_void_p * count.value)(), []
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(count)) == 0
    for node in nodes:
        k = KernelNode()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(k)) == 0
        grids.append((k.grid.x, k.grid.y, k.grid.z))
    return grids


def chunk_args(n, t, hv):
    gen = torch.Generator(device=DEV).manual_seed(n + t)
    q, k, v = (torch.randn(n, t, h, 128, generator=gen, device=DEV).to(BF16) for h in (hv // 2, hv // 2, hv))
    g, beta = -torch.rand(n, t, hv, generator=gen, device=DEV), torch.rand(n, t, hv, generator=gen, device=DEV)
    return q, k, v, g, beta, torch.randn(n, hv, 128, 128, generator=gen, device=DEV)


# sequences, v-heads, tokens, segments (a prep and a scan launch each): one up to 80 chunks in all; windows
# in 64 slots, in 80 where those save a segment; one sequence
@pytest.mark.parametrize("n,hv,t,segments", [
    (10, 4, 512, 1), (10, 4, 513, 2), (4, 8, 1400, 2), (17, 4, 300, 2), (24, 4, 300, 2), (32, 4, 300, 3),
    (33, 4, 300, 3), (33, 4, 1300, 11), (39, 4, 450, 4), (48, 2, 200, 4), (1, 4, 5120, 1), (1, 4, 5121, 2)])
def test_segments_of_dense_batches(n, hv, t, segments):
    q, k, v, g, beta, h0 = chunk_args(n, t, hv)
    assert len(grids_of(lambda: chunk_gated_delta_rule(q, k, v, g, beta, initial_state=h0, output_final_state=True,
                                                       use_qk_l2norm_in_kernel=True))) == 2 * segments


def test_a_workspace_of_64_chunks_still_serves():
    """33 sequences in windows of two chunks use 66 slots where the workspace has them, one chunk where not."""
    n, t, hv = 33, 300, 4
    q, k, v, g, beta, h0 = chunk_args(n, t, hv)
    lib, out = _lib.load(), []
    full = lib.gdn_chunk_workspace_bytes(n, n * t, hv, 128, 128)
    slot = hv * (25 + 32) * 1024  # a chunk's operands: 25 blocks and U per v-head
    ws = torch.empty(full, dtype=torch.uint8, device=DEV)

    def call(bytes_):
        o, s = torch.empty_like(v), torch.empty_like(h0)
        st = lib.gdn_chunk_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), _lib.GDN_DTYPE[BF16], hv // 2 * 128, hv // 2 * 128,
                               hv * 128, g.data_ptr(), beta.data_ptr(), 0, h0.data_ptr(), None, n, s.data_ptr(), None, n,
                               o.data_ptr(), _lib.GDN_DTYPE[BF16], None, n, t, hv // 2, hv, 128, 128, 128 ** -0.5, 1,
                               ws.data_ptr(), bytes_, _lib.stream_of(q))
        out.append((o, s))
        return st

    assert call(full - 17 * slot) != 0  # 63 slots: refused
    for bytes_, launches in ((full, 6), (full - 15 * slot, 10)):
        assert len(grids_of(lambda: call(bytes_))) == launches
    (o, s), (o2, s2) = out[1], out[3]  # (out[2], out[4]: captured, not run)
    assert torch.equal(o, o2) and torch.equal(s, s2)


# channels, type, tokens, tokens per tile
@pytest.mark.parametrize("c,dt,t,tile", [
    (2048, FP32, 2048, 8), (2048, FP32, 3600, 16), (2048, FP32, 3906, 16),  # 16 up to 32 million bytes of x
    (2048, FP32, 3907, 32), (2048, FP32, 4096, 32), (8192, FP32, 1024, 32), (1024, FP32, 4096, 16), (2048, BF16, 4096, 16),
    (2048, BF16, 4097, 32), (8192, BF16, 1024, 16)])
def test_conv_tiles(c, dt, t, tile):
    gen = torch.Generator(device=DEV).manual_seed(t)
    x, w = torch.randn(t, c, generator=gen, device=DEV).to(dt), torch.randn(c, 4, generator=gen, device=DEV).to(dt)
    assert grids_of(lambda: causal_conv1d_fn(x, w, None, "silu")) == [((c // 8 + 255) // 256, (t + tile - 1) // tile, 1)]
