"""What the framework is used for, as cases that can be timed: the operator's forward and backward, the Phalanx layer in
training and in inference, prompts and tokens served through a layer, and the streaming form on gated operands.

``listed()`` names the fixed cases, ``draw(rng)`` gives one more case of the same ranges, ``prepare(case, seed)`` makes
what a program has in hand before the call, ``run(state)`` makes one pass through the public entry points, ``work(case)``
counts the bytes and operations the pass cannot do without, and ``tolerance(case)`` says how far two correct
implementations at the same precision may lie apart.
"""

from __future__ import annotations

import math

import torch

from spear_amd import Phalanx, btp, btp_qkv
from spear_amd.nn.phalanx.inference import (
    PhalanxStepState,
    parallel_jagged,
    phalanx_prefill,
    phalanx_step,
)

_DEVICE = "cuda"
_TYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def listed():
    return [
        # The operator at the batch of the smallest configuration (8 sequences of 128 steps, 32 heads), with its default
        # fp32 result: what one call costs when launches and host work count.
        dict(name="op_small", path="op", B=8, H=32, L=128, dtype="bf16", out="f32", train=True),
        # The headline configuration: 1024 sequences of 128 steps, dim 512, 16-bit in and out, forward and backward.
        dict(name="op_headline", path="op", B=1024, H=32, L=128, dtype="bf16", out="same", train=True),
        # Inference on long sequences of a length that is no whole number of cache lines, fp16, default fp32 result.
        dict(name="op_ragged_infer", path="op", B=64, H=128, L=2032, dtype="f16", out="f32", train=False),
        # The long-sequence configuration (16 x 8192 steps, dim 1024) in q/k/v/gate terms with fp32 log-space gates and
        # q/k heads shared by groups of four value heads, as grouped layers have them.
        dict(name="qkv_long", path="qkv", B=16, H=64, kv_heads=16, L=8192, dtype="bf16", train=True),
        # One training step of a layer as the reference builds it, at the size of its headline shape.
        dict(name="layer_train", path="layer", B=1024, L=128, dim=512, kv_heads=32, method="default", train=True),
        # The same layer on the smallest configuration's batch: fine-tuning and debugging runs, bound by the host.
        dict(name="layer_train_small", path="layer", B=8, L=128, dim=512, kv_heads=32, method="default", train=True),
        # A wide layer on the stability configuration's sequences, kv heads shared by four: the largest training step.
        dict(name="layer_train_wide", path="layer", B=64, L=2048, dim=2048, kv_heads=32, method="fused", train=True),
        # Scoring long documents: the forward alone.
        dict(name="layer_infer_long", path="layer", B=16, L=8192, dim=1024, kv_heads=64, method="fused", train=False),
        # Prompts of a length as it comes through a layer, leaving the state that decoding continues from.
        dict(name="prefill_prompt", path="prefill", B=64, L=1003, dim=512, kv_heads=32),
        # One token for 1024 sequences at different positions through a layer.
        dict(name="decode_token", path="token", B=1024, dim=512, kv_heads=32),
        # Streaming form on operands that are already gated: prompts of odd length in bf16 with the state kept in fp32.
        dict(name="stream_odd", path="stream", B=1024, H=32, D=16, L=127, block_len=16, dtype="bf16", state="f32"),
        # The same in fp32, the type of the reference's own streaming examples.
        dict(name="stream_f32", path="stream", B=64, H=32, D=16, L=1000, block_len=16, dtype="f32", state="same"),
    ]


def _spread(rng, lo, hi):
    """A whole number in [lo, hi], spread over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _group(rng, heads):
    """kv heads for `heads` heads: as many in half of the cases, else shared by a divisor."""
    if rng.random() < 0.5:
        return heads
    return heads // rng.choice([g for g in range(1, min(heads, 32) + 1) if heads % g == 0])


def draw(rng):
    path = rng.choices(("op", "qkv", "layer", "prefill", "token", "stream"), (3, 2, 3, 1, 1, 2))[0]
    while True:
        if path == "op":
            c = dict(path=path, B=_spread(rng, 1, 1024), H=_spread(rng, 1, 128), L=16 * _spread(rng, 1, 512),
                     dtype=rng.choice(("bf16", "bf16", "f16")), out=rng.choice(("same", "f32")), train=rng.random() < 0.7)
            size, lo, hi = c["B"] * c["H"] * c["L"], 1 << 14, 64 * 128 * 2048
        elif path == "qkv":
            H = _spread(rng, 1, 128)
            c = dict(path=path, B=_spread(rng, 1, 1024), H=H, kv_heads=_group(rng, H), L=16 * _spread(rng, 1, 512),
                     dtype=rng.choice(("bf16", "bf16", "f16")), train=rng.random() < 0.8)
            size, lo, hi = c["B"] * H * c["L"], 1 << 14, 64 * 128 * 2048
        elif path == "layer":
            H = _spread(rng, 8, 128)
            c = dict(path=path, B=_spread(rng, 1, 1024), L=16 * _spread(rng, 1, 512), dim=16 * H, kv_heads=_group(rng, H),
                     method=rng.choice(("default", "fused")), train=rng.random() < 0.7)
            size, lo, hi = c["B"] * c["L"] * c["dim"], 1 << 17, 1024 * 128 * (1024 if c["method"] == "fused" else 512)
        elif path == "prefill":
            H = _spread(rng, 8, 128)
            c = dict(path=path, B=_spread(rng, 1, 256), L=_spread(rng, 17, 8192), dim=16 * H, kv_heads=_group(rng, H))
            size, lo, hi = c["B"] * c["L"] * c["dim"], 1 << 17, 64 * 2048 * 512
        elif path == "token":
            H = _spread(rng, 8, 128)
            c = dict(path=path, B=_spread(rng, 1, 1024), dim=16 * H, kv_heads=_group(rng, H))
            size, lo, hi = 1, 1, 1
        else:
            c = dict(path=path, B=_spread(rng, 1, 1024), H=_spread(rng, 1, 64), D=rng.choice((16, 16, 16, 32, 64)),
                     L=_spread(rng, 9, 4096), block_len=rng.choice((16, 16, 16, 32, 64)),
                     dtype=rng.choice(("bf16", "f16", "f32")), state=rng.choice(("same", "f32")))
            size, lo, hi = c["B"] * c["H"] * c["D"] * c["L"], 1 << 18, 1024 * 32 * 16 * 128
        if lo <= size <= hi:
            return c


def _normal(gen, shape, dtype, std=1.0):
    return torch.randn(shape, generator=gen, device=_DEVICE, dtype=torch.float32).mul_(std).to(dtype)


def _log_decay(gen, shape):
    """fp32 log-decay gates -softplus(N(0, 1)), the benchmark configurations' distribution."""
    return -torch.nn.functional.softplus(torch.randn(shape, generator=gen, device=_DEVICE))


def _layer(case, seed, method):
    torch.manual_seed(seed)
    with torch.device(_DEVICE):
        return Phalanx(dim=case["dim"], length=case.get("L", 2048), method=method, dtype=torch.bfloat16,
                       kv_heads=case["kv_heads"])


def prepare(case, seed):
    gen = torch.Generator(device=_DEVICE).manual_seed(seed)
    path, B = case["path"], case["B"]
    state = dict(case=case)
    if path == "op":
        H, L, dtype = case["H"], case["L"], _TYPES[case["dtype"]]
        out = dtype if case["out"] == "same" else torch.float32
        state.update(coeff=_log_decay(gen, (B, H, L)).exp_().to(dtype), x=_normal(gen, (B, H, 16, L), dtype, 0.25), out=out)
        if case["train"]:
            state["coeff"].requires_grad_(True)
            state["x"].requires_grad_(True)
            state["dy"] = _normal(gen, (B, H, 16, L), out)
    elif path == "qkv":
        H, Hkv, L, dtype = case["H"], case["kv_heads"], case["L"], _TYPES[case["dtype"]]
        state.update(q=_normal(gen, (B, L, Hkv, 16), dtype, 0.25), k=_normal(gen, (B, L, Hkv, 16), dtype, 0.25),
                     v=_normal(gen, (B, L, H, 16), dtype, 0.25), gate=_log_decay(gen, (B, L, H)))
        if case["train"]:
            for name in ("q", "k", "v", "gate"):
                state[name].requires_grad_(True)
            state["dy"] = _normal(gen, (B, L, H, 16), dtype)
    elif path == "layer":
        state["layer"] = _layer(case, seed, case["method"])
        state["x"] = _normal(gen, (B, case["L"], case["dim"]), torch.bfloat16)
        if case["train"]:
            state["x"].requires_grad_(True)
            state["dy"] = _normal(gen, (B, case["L"], case["dim"]), torch.bfloat16)
    elif path == "prefill":
        state["layer"] = _layer(case, seed, "fused")
        state["x"] = _normal(gen, (B, case["L"], case["dim"]), torch.bfloat16)
    elif path == "token":
        H = case["dim"] // 16
        state["layer"] = _layer(case, seed, "fused")
        state["x"] = _normal(gen, (B, case["dim"]), torch.bfloat16)
        # a state in the middle of decoding: every sequence somewhere in its block
        state["decoding"] = PhalanxStepState(
            h_loc=_normal(gen, (B, H, 16), torch.float32, 0.25), r_pref=torch.rand((B, H), generator=gen, device=_DEVICE),
            c_prev_loc=_normal(gen, (B, H, 16), torch.float32, 0.25),
            pos=torch.randint(0, 16, (B,), generator=gen, device=_DEVICE, dtype=torch.int32))
    else:
        H, D, L, dtype = case["H"], case["D"], case["L"], _TYPES[case["dtype"]]
        state.update(A=_log_decay(gen, (B, H, L)).exp_().to(dtype), X=_normal(gen, (B, H, D, L), dtype, 0.5),
                     C=_normal(gen, (B, H, D, L), dtype), V=_normal(gen, (B, H, D, L), dtype),
                     state_dtype=torch.float32 if case["state"] == "f32" else None)
    return state


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "op":
        coeff, x = state["coeff"], state["x"]
        if not case["train"]:
            with torch.no_grad():
                return btp(coeff, x, output_dtype=state["out"])
        coeff.grad = x.grad = None
        y = btp(coeff, x, output_dtype=state["out"])
        y.backward(state["dy"])
        return y.detach(), coeff.grad, x.grad
    if path == "qkv":
        operands = [state[name] for name in ("q", "k", "v", "gate")]
        if not case["train"]:
            with torch.no_grad():
                return btp_qkv(*operands)
        for t in operands:
            t.grad = None
        y = btp_qkv(*operands)
        y.backward(state["dy"])
        return [y.detach()] + [t.grad for t in operands]
    if path == "layer":
        layer, x = state["layer"], state["x"]
        if not case["train"]:
            with torch.no_grad():
                return layer(x)
        layer.zero_grad(set_to_none=True)
        x.grad = None
        y = layer(x)
        y.backward(state["dy"])
        return [y.detach(), x.grad] + [p.grad for p in layer.parameters()]
    if path == "prefill":
        with torch.no_grad():
            y, st = phalanx_prefill(state["layer"], state["x"])
        return y, st.h_loc, st.r_pref, st.c_prev_loc, st.pos
    if path == "token":
        st = state["decoding"]
        y = phalanx_step(state["layer"], state["x"], st)
        return y, st.h_loc, st.r_pref, st.c_prev_loc, st.pos
    y, st = parallel_jagged(state["A"], state["X"], state["C"], state["V"], block_len=case["block_len"],
                            state_dtype=state["state_dtype"])
    return y, st.h_loc, st.r_pref, st.c_prev_loc


def _columns(case):
    """Columns of the four input projections of a layer together."""
    return case["dim"] + 2 * 16 * case["kv_heads"] + case["dim"] // 16


def work(case):
    path, B = case["path"], case["B"]
    if path == "op":
        units, o = B * case["H"] * case["L"], 2 if case["out"] == "same" else 4
        nbytes = units * (2 + 32 + 16 * o)                       # coeff, x -> y
        flops = units * 16 * 4
        if case["train"]:
            nbytes += units * (16 * o + 2 + 32)                  # dy -> d coeff, dx (in the leaves' types)
            flops += units * 16 * 12
        return dict(bytes=nbytes, flops=flops)
    if path == "qkv":
        units, kv = B * case["H"] * case["L"], B * case["kv_heads"] * case["L"]
        nbytes = units * (4 + 64) + kv * 64                      # gate, v, q, k -> out
        flops = units * 16 * 6
        if case["train"]:
            nbytes += units * (32 + 4 + 32) + kv * 64            # dout -> dgate, dv, dq, dk
            flops += units * 16 * 18
        return dict(bytes=nbytes, flops=flops)
    if path == "stream":
        n, o = B * case["H"] * case["L"], 4 if case["dtype"] == "f32" else 2
        return dict(bytes=n * o * (1 + 4 * case["D"]) + B * case["H"] * (2 * case["D"] + 1) * 4, flops=n * case["D"] * 8)
    # the layer: five projections around the mixing stage
    tokens, dim, cols = B * case.get("L", 1), case["dim"], _columns(case)
    weights = dim * (cols + dim)
    nbytes, flops = 2 * (2 * tokens * dim + weights), 2 * tokens * weights
    if path == "token":
        nbytes += 2 * 4 * tokens * (2 * dim + dim // 16)         # the state, read and written
    if path == "layer" and case["train"]:
        nbytes += 2 * (2 * tokens * dim + weights)               # dy -> dx, weight gradients
        flops *= 3
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    """About four times the distance to the same path in 64 bits, measured over the listed cases and 14 drawn ones."""
    rounding = {"bf16": 6.6e-3, "f16": 8.3e-4, "f32": 1e-6}  # of the results' type: 1.66e-3 and 2.08e-4; sums: below 1e-7
    path = case["path"]
    if path == "op" and not case["train"]:
        return {"rel": rounding["f32" if case["out"] == "f32" else case["dtype"]]}
    if path in ("op", "qkv", "stream"):
        return {"rel": rounding[case["dtype"]]}
    # the layer in bf16: every stage rounds. Outputs 2.9e-3 to 3.2e-3 off, gradients up to 5.8e-3 (9e-3 where many
    # heads share a kv head)
    return {"rel": 0.025 if path == "layer" and case["train"] else 0.0125}
