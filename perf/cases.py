"""What a user of this framework has it do, as cases that can be timed and checked.

The shapes are the Qwen3.5-35B-A3B Gated DeltaNet layer's (``engine.configs``): 16 q/k heads,
32 v-heads, head dim 128, conv width 4 over the 8192-wide q|k|v projection, hidden size 2048.
Each case is one call (or the short chain of calls that a step makes) through the public entry
points of ``engine.kernels`` / ``engine.runtime``:

* ``decode``         one token for each of ``batch`` sequences, states in a slot pool, in place;
* ``verify``         a speculative-verify step of ``tokens`` drafts per row and the commit of
                     the accepted prefix;
* ``prefill``        the chunk prefill of ``batch`` equal sequences in bf16, fp16 or fp32, from
                     zero or given states, q/k at their own heads or repeated to the v-heads;
* ``varlen``         packed sequences: the causal conv over the projection with its window
                     pool, then the chunk prefill on the state pool, both in place;
* ``layer_decode``   a whole layer's decode step on slot pools;
* ``layer_prefill``  a whole layer's prefill on slot pools.
"""
import math
import os
import random
import sys
from types import SimpleNamespace

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "paris-hackathon-2026-inference_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

from engine.configs import CONV_DIM, CONV_WIDTH, D, HK, HV  # noqa: E402
from engine.kernels import (causal_conv1d_fn, chunk_gated_delta_rule, fused_recurrent_gated_delta_rule,  # noqa: E402
                            gated_delta_net_forward, gdn_state_commit)
from engine.runtime import GDNSlotPools  # noqa: E402

DEV = "cuda"
HIDDEN = 2048
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
STATE_BYTES = HV * D * D * 4
WEIGHTS = HIDDEN * (CONV_DIM + HV * D + 2 * HV) + HV * D * HIDDEN  # the layer's projections


def listed():
    return [
        # a single user's next token: latency and launches
        {"name": "decode_b1", "kind": "decode", "batch": 1, "rows": 8},
        # a full serving batch's next tokens: the state stream
        {"name": "decode_b64", "kind": "decode", "batch": 64, "rows": 128},
        # a verify step of speculative decoding with three drafts and the last real token
        {"name": "verify_b32_t4", "kind": "verify", "batch": 32, "tokens": 4, "rows": 64},
        # a short odd-length prompt of one user
        {"name": "prefill_b1_t333", "kind": "prefill", "batch": 1, "tokens": 333, "dtype": "bf16", "h0": False,
         "repeat": False},
        # a long prompt of one user
        {"name": "prefill_b1_t4096", "kind": "prefill", "batch": 1, "tokens": 4096, "dtype": "bf16", "h0": False,
         "repeat": False},
        # a few prompts continued from cached prefixes
        {"name": "prefill_b4_t1038", "kind": "prefill", "batch": 4, "tokens": 1038, "dtype": "bf16", "h0": True,
         "repeat": False},
        # the microbatch that the reference engine was profiled on, q/k repeated to the v-heads by the caller
        {"name": "prefill_b16_t1038", "kind": "prefill", "batch": 16, "tokens": 1038, "dtype": "bf16", "h0": False,
         "repeat": True},
        # a model kept in fp32 (a parity or evaluation run)
        {"name": "prefill_fp32_b1_t1024", "kind": "prefill", "batch": 1, "tokens": 1024, "dtype": "fp32", "h0": False,
         "repeat": False},
        # continuous batching: prompts of mixed lengths packed into one call
        {"name": "varlen_n16", "kind": "varlen", "seqs": 16, "lo": 128, "hi": 2048, "spread": 3,
         "rows": 32},
        # the whole layer, one user's next token
        {"name": "layer_decode_b1", "kind": "layer_decode", "batch": 1, "rows": 8},
        # the whole layer, a full batch's next tokens
        {"name": "layer_decode_b64", "kind": "layer_decode", "batch": 64, "rows": 128},
        # the whole layer, one prompt
        {"name": "layer_prefill_b1_t2000", "kind": "layer_prefill", "batch": 1, "tokens": 2000,
         "rows": 8},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    kind = rng.choice(["decode", "verify", "prefill", "prefill", "prefill", "varlen", "layer_decode", "layer_prefill"])
    if kind in ("decode", "layer_decode", "verify"):
        c = {"kind": kind, "batch": _log_int(rng, 1, 32 if kind == "verify" else 64)}
        if kind == "verify":
            c["tokens"] = rng.randint(2, 5)
        return {**c, "rows": c["batch"] + rng.randint(0, 64)}
    if kind == "prefill":
        dtype = rng.choice(["bf16", "bf16", "bf16", "bf16", "fp16", "fp32"])
        batch = _log_int(rng, 1, 16)
        total = _log_int(rng, 20, 16384) if dtype == "bf16" else _log_int(rng, 20, 1024)
        return {"kind": kind, "batch": batch, "tokens": max(1, total // batch), "dtype": dtype,
                "h0": rng.random() < 0.5, "repeat": rng.random() < 0.3}
    if kind == "varlen":
        seqs = _log_int(rng, 1, 16)
        hi = _log_int(rng, 16, 2048)
        return {"kind": kind, "seqs": seqs, "lo": max(1, hi // 16), "hi": hi, "spread": rng.randint(0, 1 << 20),
                "rows": seqs + rng.randint(0, 16)}
    batch = _log_int(rng, 1, 8)
    return {"kind": kind, "batch": batch, "tokens": max(2, _log_int(rng, 20, 4096) // batch),
            "rows": batch + rng.randint(0, 16)}


def _lens(case):
    """A packed batch's sequence lengths (of the case, not of the seed: the work stays the same)."""
    r = random.Random(case["spread"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["seqs"])]


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(gen, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=gen, device=DEV).to(dtype)


def _uniform(gen, lo, hi, *shape):
    return torch.rand(*shape, generator=gen, device=DEV) * (hi - lo) + lo


def _gates(gen, *shape):
    """log-decay and write strength as the layer forms them: mostly slow decay, some fast."""
    g = -F.softplus(_randn(gen, *shape)) * torch.exp(_uniform(gen, -2.0, 0.0, *shape))
    return g, torch.sigmoid(_randn(gen, *shape))


def _packed(gen, b, t, dtype):
    """q, k, v as the views of one packed [b, t, 8192] activation that the conv leaves (silu of N(0, 1))."""
    x = F.silu(_randn(gen, b, t, CONV_DIM)).to(dtype)
    q, k, v = torch.split(x, [HK * D, HK * D, HV * D], dim=-1)
    return q.unflatten(-1, (HK, D)), k.unflatten(-1, (HK, D)), v.unflatten(-1, (HV, D))


def _slots(gen, rows, n):
    """The batch's n slots in a pool of ``rows``, in no order."""
    return torch.randperm(rows, generator=gen, device=DEV)[:n].contiguous()


class GatedDeltaNet(torch.nn.Module):
    """The layer's parameters under the names the patched forward reads."""

    def __init__(self, gen):
        super().__init__()

        def lin(n_in, n_out):
            m = torch.nn.Linear(n_in, n_out, bias=False, device="meta")
            m.weight = torch.nn.Parameter(_randn(gen, n_out, n_in).mul_(n_in ** -0.5).to(torch.bfloat16), False)
            return m

        def vec(x, dtype=torch.bfloat16):
            return torch.nn.Parameter(x.to(dtype), False)

        self.layer_idx = 0
        self.activation = "silu"
        self.conv_kernel_size = CONV_WIDTH
        self.key_dim, self.value_dim = HK * D, HV * D
        self.head_k_dim = self.head_v_dim = D
        self.in_proj_qkv, self.in_proj_z = lin(HIDDEN, CONV_DIM), lin(HIDDEN, HV * D)
        self.in_proj_b, self.in_proj_a = lin(HIDDEN, HV), lin(HIDDEN, HV)
        self.out_proj = lin(HV * D, HIDDEN)
        self.conv1d = torch.nn.Module()
        self.conv1d.weight = vec(_uniform(gen, -0.5, 0.5, CONV_DIM, 1, CONV_WIDTH))
        self.conv1d.bias = None
        self.norm = torch.nn.Module()
        self.norm.weight = vec(_uniform(gen, 0.75, 1.25, D))
        self.norm.variance_epsilon = 1e-6
        self.A_log = vec(_uniform(gen, -2.0, 1.0, HV))
        self.dt_bias = vec(_uniform(gen, -2.0, 1.0, HV))


def apply_mask_to_padding_states(hidden_states, attention_mask):
    """The transformers hook of the layer's module (there is no padding here)."""
    return hidden_states


def prepare(case, seed):
    gen = _gen(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind in ("decode", "verify"):
        b, t = case["batch"], case.get("tokens", 1)
        rows = case["rows"]
        s["slots"] = _slots(gen, rows, b)
        s["q"], s["k"], s["v"] = _packed(gen, b, t, torch.bfloat16)
        s["g"], s["beta"] = _gates(gen, b, t, HV)
        s["pool"] = _randn(gen, rows, HV, D, D).mul_(0.1)
        if kind == "verify":
            s["snapshots"] = torch.empty(b, t, HV, D, D, device=DEV)
            s["accepted"] = torch.randint(1, t + 1, (b,), generator=gen, device=DEV, dtype=torch.int32)
    elif kind == "prefill":
        b, t = case["batch"], case["tokens"]
        q, k, s["v"] = _packed(gen, b, t, DTYPES[case["dtype"]])
        if case["repeat"]:
            q, k = q.repeat_interleave(HV // HK, dim=2), k.repeat_interleave(HV // HK, dim=2)
        s["q"], s["k"] = q, k
        s["g"], s["beta"] = _gates(gen, b, t, HV)
        s["h0"] = _randn(gen, b, HV, D, D).mul_(0.1) if case["h0"] else None
    elif kind == "varlen":
        lens = _lens(case)
        n, total = len(lens), sum(lens)
        rows = case["rows"]
        s["slots"] = _slots(gen, rows, n)
        s["cu"] = torch.tensor([sum(lens[:i]) for i in range(n + 1)], dtype=torch.int32, device=DEV)
        s["x"] = _randn(gen, total, CONV_DIM, dtype=torch.bfloat16)
        s["conv_w"] = _uniform(gen, -0.5, 0.5, CONV_DIM, CONV_WIDTH).to(torch.bfloat16)
        s["windows"] = _randn(gen, rows, CONV_DIM, CONV_WIDTH, dtype=torch.bfloat16)
        s["g"], s["beta"] = _gates(gen, 1, total, HV)
        s["pool"] = _randn(gen, rows, HV, D, D).mul_(0.1)
    else:
        b, t = case["batch"], case.get("tokens", 1)
        rows = case["rows"]
        slots = _slots(gen, rows, b)
        s["layer"] = GatedDeltaNet(gen)
        s["hidden"] = _randn(gen, b, t, HIDDEN, dtype=torch.bfloat16)
        conv = {0: _randn(gen, rows, CONV_DIM, CONV_WIDTH, dtype=torch.bfloat16)}
        rec = {0: _randn(gen, rows, HV, D, D).mul_(0.1)}
        s["pools"] = GDNSlotPools(conv, rec, b)
        s["pools"].bind(slots, is_prefill=kind == "layer_prefill")
        s["cache"] = SimpleNamespace(gdn_slot_pools=s["pools"])
        s["slots"] = slots
    return s


# ------------------------------------------------------------------ one pass

def run(s):
    kind = s["case"]["kind"]
    if kind == "decode":
        o, pool = fused_recurrent_gated_delta_rule(
            s["q"], s["k"], s["v"], s["g"], s["beta"], initial_state=s["pool"], ssm_state_indices=s["slots"],
            inplace_final_state=True, use_qk_l2norm_in_kernel=True)
        return {"o": o, "state": pool}
    if kind == "verify":
        o, _ = fused_recurrent_gated_delta_rule(
            s["q"], s["k"], s["v"], s["g"], s["beta"], initial_state=s["pool"], ssm_state_indices=s["slots"],
            snapshots=s["snapshots"], use_qk_l2norm_in_kernel=True)
        gdn_state_commit(s["pool"], s["slots"], s["snapshots"], s["accepted"])
        return {"o": o, "state": s["pool"]}
    if kind == "prefill":
        o, last = chunk_gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"], initial_state=s["h0"],
                                         output_final_state=True, use_qk_l2norm_in_kernel=True)
        return {"o": o, "state": last}
    if kind == "varlen":
        y = causal_conv1d_fn(s["x"], s["conv_w"], None, "silu", cu_seqlens=s["cu"], conv_states=s["windows"],
                             cache_indices=s["slots"])
        q, k, v = torch.split(y.unsqueeze(0), [HK * D, HK * D, HV * D], dim=-1)
        o, pool = chunk_gated_delta_rule(
            q.unflatten(-1, (HK, D)), k.unflatten(-1, (HK, D)), v.unflatten(-1, (HV, D)), s["g"], s["beta"],
            initial_state=s["pool"], ssm_state_indices=s["slots"], inplace_final_state=True,
            use_qk_l2norm_in_kernel=True, cu_seqlens=s["cu"])
        return {"o": o, "state": pool, "windows": s["windows"]}
    with torch.no_grad():
        y = gated_delta_net_forward(s["layer"], s["hidden"], cache_params=s["cache"])
    conv, rec = s["pools"].layer(0)
    return {"y": y, "state": rec, "windows": conv}


# ------------------------------------------------------------------ what a pass cannot do without

def _core(tokens, states_read, states_written, size, hk=HK):
    """Bytes and operations of the gated delta rule itself: q, k, v in and o out at ``size`` bytes, the
    gates, the states; per token and v-head k^T S, the rank-1 update and q^T S."""
    return (tokens * ((2 * hk + 2 * HV) * D * size + HV * 8) + (states_read + states_written) * STATE_BYTES,
            tokens * HV * 6 * D * D)


def work(case):
    kind = case["kind"]
    if kind == "decode":
        nbytes, flops = _core(case["batch"], case["batch"], case["batch"], 2)
    elif kind == "verify":
        # the kept states are what must be written; per-token snapshots are this path's way to them
        nbytes, flops = _core(case["batch"] * case["tokens"], case["batch"], case["batch"], 2)
    elif kind == "prefill":
        b = case["batch"]
        nbytes, flops = _core(b * case["tokens"], b if case["h0"] else 0, b, DTYPES[case["dtype"]].itemsize,
                              HV if case["repeat"] else HK)
    elif kind == "varlen":
        n, total = case["seqs"], sum(_lens(case))
        nbytes, flops = _core(total, n, n, 2)
        # the conv: x in and y out (the core's q, k, v reads above are of y), windows in and out
        nbytes += 2 * total * CONV_DIM * 2 + 2 * n * CONV_DIM * CONV_WIDTH * 2
        flops += total * CONV_DIM * 2 * CONV_WIDTH
    else:
        b, tokens = case["batch"], case["batch"] * case.get("tokens", 1)
        _, core = _core(tokens, b, b, 2)
        nbytes = (WEIGHTS * 2 + 2 * tokens * HIDDEN * 2 + (2 if kind == "layer_decode" else 1) * b *
                  (STATE_BYTES + CONV_DIM * CONV_WIDTH * 2))
        flops = core + 2 * tokens * WEIGHTS + tokens * CONV_DIM * 2 * CONV_WIDTH
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the error against 64 bits that was measured, or that the other exact form of the
    rule has (fp32: the recurrence 1e-7, the chunk form in fp32 5.5e-7)."""
    kind = case["kind"]
    if kind in ("decode", "verify"):
        return {"rel": 7e-3}  # bf16 outputs, 1.7e-3
    if kind == "prefill":  # bf16: 2.7e-3, bf16 operands and outputs; fp16: the outputs' rounding, 2.5e-4
        return {"rel": {"bf16": 1.1e-2, "fp16": 1e-3, "fp32": 2.2e-6}[case["dtype"]]}
    if kind == "varlen":
        return {"rel": 1.5e-2}  # 3.7e-3
    return {"rel": 2.3e-2}  # bf16 between the layer's parts, 5.7e-3


# ------------------------------------------------------------------ the same in 64 bits

def _l2n(x):
    return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def _rule(q, k, v, g, beta, state, lens=None, keep=None):
    """The gated delta rule token by token in fp64: q, k [N, T, Hk, D] (any Hk that divides the v-heads),
    v [N, T, Hv, D], gates [N, T, Hv], state [N, Hv, D, D]; sequence n stops after lens[n] tokens.
    Returns o and the state, or the state after keep[n] tokens."""
    n, t, hv = v.shape[:3]
    r = hv // q.shape[2]
    q = (_l2n(q.double()) * D ** -0.5).repeat_interleave(r, 2)
    k = _l2n(k.double()).repeat_interleave(r, 2)
    v, decay, beta = v.double(), torch.exp(g.double()), beta.double()
    state = state.double().clone()
    kept = state.clone()
    o = torch.zeros(n, t, hv, D, dtype=torch.float64, device=v.device)
    if lens is not None:  # past its end a sequence neither decays nor writes
        live = torch.arange(t, device=v.device)[None, :] < torch.tensor(lens, device=v.device)[:, None]
        decay = torch.where(live[:, :, None], decay, torch.ones_like(decay))
        beta = beta * live[:, :, None]
    for i in range(t):
        state *= decay[:, i, :, None, None]
        ki = k[:, i].unsqueeze(-2)
        delta = beta[:, i, :, None] * (v[:, i] - torch.matmul(ki, state).squeeze(-2))
        state += ki.transpose(-1, -2) * delta.unsqueeze(-2)
        o[:, i] = torch.matmul(q[:, i].unsqueeze(-2), state).squeeze(-2)
        if keep is not None:
            kept = torch.where((keep == i + 1)[:, None, None, None], state, kept)
    return o, (state if keep is None else kept)


def _conv(x, w, windows):
    """silu of the causal depthwise conv of x [N, T, C] after its windows [N, C, W], and the windows
    after each prefix: all in fp64."""
    h = torch.cat([windows.double(), x.double().transpose(1, 2)], dim=-1)  # [N, C, W + T]
    y = F.silu(sum(h[:, :, 1 + i: 1 + i + x.shape[1]] * w.double()[:, i, None] for i in range(CONV_WIDTH)))
    return y.transpose(1, 2), h


def _put(pool, slots, rows):
    out = pool.double()
    out[slots] = rows
    return out


def _split(y):
    q, k, v = torch.split(y, [HK * D, HK * D, HV * D], dim=-1)
    return q.unflatten(-1, (HK, D)), k.unflatten(-1, (HK, D)), v.unflatten(-1, (HV, D))


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind in ("decode", "verify"):
        o, rows = _rule(s["q"], s["k"], s["v"], s["g"], s["beta"], s["pool"][s["slots"]],
                        keep=s.get("accepted"))
        return {"o": o, "state": _put(s["pool"], s["slots"], rows)}
    if kind == "prefill":
        h0 = s["h0"] if s["h0"] is not None else torch.zeros(case["batch"], HV, D, D, device=DEV)
        o, last = _rule(s["q"], s["k"], s["v"], s["g"], s["beta"], h0)
        return {"o": o, "state": last}
    if kind == "varlen":
        lens, slots = _lens(case), s["slots"]
        n, longest = len(lens), max(lens)
        where = torch.cat([torch.arange(x, device=DEV) + i * longest for i, x in enumerate(lens)])

        def pad(x):
            out = torch.zeros(n * longest, *x.shape[1:], dtype=torch.float64, device=DEV)
            out[where] = x.double()
            return out.unflatten(0, (n, longest))

        y, h = _conv(pad(s["x"]), s["conv_w"], s["windows"][slots])
        windows = torch.stack([h[i, :, x: x + CONV_WIDTH] for i, x in enumerate(lens)])
        o, rows = _rule(*_split(y), pad(s["g"][0]), pad(s["beta"][0]), s["pool"][slots], lens=lens)
        return {"o": o.flatten(0, 1)[where].unsqueeze(0), "state": _put(s["pool"], slots, rows),
                "windows": _put(s["windows"], slots, windows)}
    layer, slots, x = s["layer"], s["slots"], s["hidden"].double()
    conv, rec = s["pools"].layer(0)
    start, windows = rec[slots].double(), conv[slots].double()
    if kind == "layer_prefill":  # prefill rows start from nothing
        start, windows = torch.zeros_like(start), torch.zeros_like(windows)

    def lin(m, x):
        return torch.matmul(x, m.weight.double().t())

    y, h = _conv(lin(layer.in_proj_qkv, x), layer.conv1d.weight.squeeze(1), windows)
    g = -torch.exp(layer.A_log.double()) * F.softplus(lin(layer.in_proj_a, x) + layer.dt_bias.double())
    o, rows = _rule(*_split(y), g, torch.sigmoid(lin(layer.in_proj_b, x)), start)
    o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + layer.norm.variance_epsilon) * layer.norm.weight.double()
    out = lin(layer.out_proj, (o * F.silu(lin(layer.in_proj_z, x).unflatten(-1, (HV, D)))).flatten(-2))
    return {"y": out, "state": _put(rec, slots, rows), "windows": _put(conv, slots, h[:, :, -CONV_WIDTH:])}
