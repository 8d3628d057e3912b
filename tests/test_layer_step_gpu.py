"""The layer-layout decode step (spear_phalanx_mix_step, phalanx_step / phalanx_prefill): one token of the
Phalanx mixing stage on the projections' [B, features] outputs with the fp32 streaming state, against the
float64 oracle (oracle.jagged_oracle.layer_step), against the layer's own forward, and as a HIP graph that is
replayed once per token."""

import numpy as np
import pytest
import torch

from helpers import BF16_ATOL, BF16_RTOL, F32_ATOL, F32_RTOL, assert_close, f64
from oracle import jagged_oracle as jag

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def token_inputs(B, H, Hkv, n, seed, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    return [(torch.randn(B, H, generator=g).to(dtype), torch.randn(B, Hkv * 16, generator=g).to(dtype),
             torch.randn(B, Hkv * 16, generator=g).to(dtype), torch.randn(B, H * 16, generator=g).to(dtype)) for _ in range(n)]


@pytest.mark.parametrize("B,H,Hkv,n", [(1, 4, 4, 35), (3, 8, 2, 20), (2, 32, 32, 18), (5, 12, 3, 33), (2, 64, 8, 17)])
@pytest.mark.parametrize("device_positions", [True, False], ids=["pos_on_device", "host_boundary"])
def test_step_kernel_matches_oracle_over_block_boundaries(B, H, Hkv, n, device_positions):
    from spear_amd import _btp

    toks = token_inputs(B, H, Hkv, n, seed=9000 + H + n)
    h = torch.zeros(B, H, 16, device=DEV)
    r = torch.ones(B, H, device=DEV)
    cp = torch.zeros(B, H, 16, device=DEV)
    pos = torch.zeros(B, device=DEV, dtype=torch.int32) if device_positions else None
    ref = jag.zero_state(B, H, 16, 16)
    print(f"layer step B={B} H={H} Hkv={Hkv} n={n} device_positions={device_positions}", flush=True)
    for t, (a, b, c, v) in enumerate(toks):
        out = torch.full((B, H * 16), float("nan"), device=DEV, dtype=torch.bfloat16)
        _btp.mix_step(a.to(DEV), b.to(DEV), c.to(DEV), v.to(DEV), out, h, r, cp, pos, (t + 1) % 16 == 0, 16, H, Hkv)
        want, ref = jag.layer_step(f64(a), f64(b), f64(c), f64(v), ref, H, Hkv)
        assert_close(f64(out), want, BF16_ATOL, BF16_RTOL, f"out[{t}]")
        # the state is fp32 and never rounded to 16 bits: it follows the oracle at the fp32 bound
        assert_close(f64(h), ref.h_loc, F32_ATOL, F32_RTOL, f"h[{t}]")
        assert_close(f64(r), ref.r_pref, F32_ATOL, F32_RTOL, f"r[{t}]")
        assert_close(f64(cp), ref.c_prev_loc, F32_ATOL, F32_RTOL, f"c_prev[{t}]")
        if pos is not None:
            assert pos.tolist() == [(t + 1) % 16] * B


def test_batch_rows_at_different_block_positions():
    """With positions on the device every batch row closes its block when its own position says so."""
    from spear_amd import _btp

    B, H = 4, 8
    offsets = [0, 5, 15, 9]
    toks = token_inputs(B, H, H, 20, seed=9100)
    h = torch.zeros(B, H, 16, device=DEV)
    r = torch.ones(B, H, device=DEV)
    cp = torch.zeros(B, H, 16, device=DEV)
    pos = torch.tensor(offsets, device=DEV, dtype=torch.int32)
    refs = [jag.zero_state(1, H, 16, 16) for _ in range(B)]
    for b_, off in enumerate(offsets):
        refs[b_].i = off
    for t, (a, b, c, v) in enumerate(toks):
        out = torch.empty(B, H * 16, device=DEV, dtype=torch.bfloat16)
        _btp.mix_step(a.to(DEV), b.to(DEV), c.to(DEV), v.to(DEV), out, h, r, cp, pos, False, 16, H, H)
        for b_ in range(B):
            want, refs[b_] = jag.layer_step(f64(a[b_:b_ + 1]), f64(b[b_:b_ + 1]), f64(c[b_:b_ + 1]), f64(v[b_:b_ + 1]), refs[b_], H, H)
            assert_close(f64(out[b_:b_ + 1]), want, BF16_ATOL, BF16_RTOL, f"out[{t}][{b_}]")
    assert pos.tolist() == [(o + 20) % 16 for o in offsets]


def _layer(dim=128, kv_heads=None, seed=3):
    from spear_amd import Phalanx

    torch.manual_seed(seed)
    return Phalanx(dim=dim, length=64, method="fused", dtype=torch.bfloat16, kv_heads=kv_heads).to(DEV)


# (dim 64, B 1) and (dim 192, B 3): the rows a[t] of the tail's [tokens, B, H] logits start on 8- and 2-byte
# boundaries there (B * H * 2 bytes per token is not a multiple of 16)
@pytest.mark.parametrize("L,kv_heads,dim,B", [(48, None, 128, 3), (37, 2, 128, 3), (16, None, 128, 3), (5, None, 128, 3),
                                              (37, None, 64, 1), (37, None, 192, 3), (29, 6, 192, 1)])
def test_stepping_a_layer_equals_its_forward_and_prefill_hands_over(L, kv_heads, dim, B):
    """Token t of phalanx_step equals position t of the layer's forward on the whole sequence (both run the same
    projections; the mixing stage is the fused kernel there and the step kernel here), and prefill(first part) +
    steps continues exactly like stepping from the start."""
    from spear_amd.nn.phalanx.inference import PhalanxStepState, phalanx_prefill, phalanx_step

    layer = _layer(dim=dim, kv_heads=kv_heads)
    n_more = 21
    x = torch.randn(B, L + n_more, dim, generator=torch.Generator().manual_seed(L)).bfloat16().to(DEV)
    Lw = ((L + n_more) // 16) * 16
    with torch.no_grad():
        whole = layer(x[:, :Lw]).float()                     # forward needs whole blocks
    state = PhalanxStepState.zeros(B, layer.heads, DEV)
    stepped = torch.stack([phalanx_step(layer, x[:, t], state) for t in range(L + n_more)], dim=1).float()
    # two bf16 roundings apart at most (the mixing stage's output, then proj_out): the bf16 bound on the output scale
    scale = float(whole.abs().max())
    assert float((stepped[:, :Lw] - whole).abs().max()) <= 2e-2 * scale

    y, st = phalanx_prefill(layer, x[:, :L])
    assert y.shape == (B, L, dim)
    assert float((y.float() - stepped[:, :L]).abs().max()) <= 2e-2 * scale
    # the prefill projects the prompt as one matrix product and stepping projects token by token: the library may
    # sum those in another order, so the two states agree to the 16-bit rounding of the projections, not bit for bit
    ref_state = PhalanxStepState.zeros(B, layer.heads, DEV)
    for t in range(L):
        phalanx_step(layer, x[:, t], ref_state)
    assert st.pos.tolist() == ref_state.pos.tolist() == [L % 16] * B
    for name in ("h_loc", "r_pref", "c_prev_loc"):
        got, want = getattr(st, name), getattr(ref_state, name)
        assert float((got - want).abs().max()) <= 2e-2 * max(1.0, float(want.abs().max())), name
    cont = torch.stack([phalanx_step(layer, x[:, t], st) for t in range(L, L + n_more)], dim=1).float()
    assert float((cont - stepped[:, L:]).abs().max()) <= 2e-2 * scale


@pytest.mark.parametrize("B,H,Hkv,L", [(2, 4, 4, 16), (3, 8, 2, 48), (1, 32, 32, 128), (2, 12, 3, 272), (1, 64, 8, 2048),
                                       (2, 6, 2, 80), (1, 3, 1, 48), (2, 16, 1, 64)])
def test_prefill_kernel_leaves_the_state_that_stepping_reaches(B, H, Hkv, L):
    """spear_phalanx_mix_prefill on [B, L, features] against L calls of the step kernel on the same tensors: the
    hand-over state is the same fp32 arithmetic in the same order, so it is equal bit for bit; the outputs agree
    with the float64 oracle, and the forward entry point (no state) gives the same output."""
    from spear_amd import _btp

    g = torch.Generator().manual_seed(9200 + L + H)
    a = torch.randn(B, L, H, generator=g).bfloat16().to(DEV)
    b = torch.randn(B, L, Hkv * 16, generator=g).bfloat16().to(DEV)
    c = torch.randn(B, L, Hkv * 16, generator=g).bfloat16().to(DEV)
    v = torch.randn(B, L, H * 16, generator=g).bfloat16().to(DEV)
    out, plain = torch.empty_like(v), torch.empty_like(v)
    tail = torch.full((B, H, 16), float("nan"), device=DEV)
    print(f"mix prefill B={B} H={H} Hkv={Hkv} L={L}", flush=True)
    _btp.mix_forward(a, b, c, v, out, H, Hkv, c_prev_tail=tail)
    _btp.mix_forward(a, b, c, v, plain, H, Hkv)
    assert torch.equal(out, plain)

    h = torch.zeros(B, H, 16, device=DEV)
    r = torch.ones(B, H, device=DEV)
    cp = torch.zeros(B, H, 16, device=DEV)
    pos = torch.zeros(B, device=DEV, dtype=torch.int32)
    stepped = torch.empty_like(v)
    # stepped[:, t] is a strided view: step into a dense row and copy
    row = torch.empty(B, H * 16, device=DEV, dtype=torch.bfloat16)
    for t in range(L):
        _btp.mix_step(a[:, t].contiguous(), b[:, t].contiguous(), c[:, t].contiguous(), v[:, t].contiguous(), row,
                      h, r, cp, pos, False, 16, H, Hkv)
        stepped[:, t] = row
    assert torch.equal(tail, cp), "hand-over state"
    assert float(h.abs().max()) == 0.0 and torch.equal(r, torch.ones_like(r)) and pos.tolist() == [0] * B
    assert_close(f64(out), f64(stepped), BF16_ATOL, BF16_RTOL, "prefill output vs stepping")
    if L <= 272:
        ref = jag.zero_state(B, H, 16, 16)
        for t in range(L):
            want, ref = jag.layer_step(f64(a[:, t]), f64(b[:, t]), f64(c[:, t]), f64(v[:, t]), ref, H, Hkv)
            assert_close(f64(out[:, t]), want, BF16_ATOL, BF16_RTOL, f"out[{t}]")
        assert_close(f64(tail), ref.c_prev_loc, F32_ATOL, F32_RTOL, "c_prev_tail")


def test_prefill_entry_point_refuses_the_qkv_form_and_a_wrong_state():
    from spear_amd import _btp

    B, H, L = 1, 4, 16
    a = torch.zeros(B, L, H, device=DEV, dtype=torch.bfloat16)
    kv = torch.zeros(B, L, H * 16, device=DEV, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="float32"):
        _btp.mix_forward(a, kv, kv, kv, torch.empty_like(kv), H, H, c_prev_tail=torch.zeros(B, H, 16, device=DEV).bfloat16())
    with pytest.raises(RuntimeError, match="layer form"):
        _btp.mix_forward(a.float(), kv, kv, kv, torch.empty_like(kv), H, H, qkv_gate=True, c_prev_tail=torch.zeros(B, H, 16, device=DEV))


def test_one_graph_replayed_per_token_reproduces_eager_decoding():
    """The whole layer step (projections, step kernel, position update, output projection) recorded once and
    replayed for every token, across block boundaries, with eager work between the replays."""
    from spear_amd.nn.phalanx.inference import PhalanxStepState, phalanx_step

    layer = _layer(dim=256, seed=5)
    B, n = 4, 40
    xs = torch.randn(n, B, 256, generator=torch.Generator().manual_seed(77)).bfloat16().to(DEV)
    eager_state = PhalanxStepState.zeros(B, layer.heads, DEV)
    eager = [phalanx_step(layer, xs[t], eager_state).clone() for t in range(n)]

    state = PhalanxStepState.zeros(B, layer.heads, DEV)
    x_buf = torch.zeros(B, 256, device=DEV, dtype=torch.bfloat16)
    y_buf = torch.zeros(B, 256, device=DEV, dtype=torch.bfloat16)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):                             # warm-up on the capture stream, on scratch state
        phalanx_step(layer, x_buf, PhalanxStepState.zeros(B, layer.heads, DEV), out=y_buf)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        phalanx_step(layer, x_buf, state, out=y_buf)
    # the capture itself does not run the step: the state is still the zero state
    assert float(state.h_loc.abs().max()) == 0.0 and state.pos.tolist() == [0] * B
    for t in range(n):
        x_buf.copy_(xs[t])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y_buf, eager[t]), f"replay {t}"
        _ = (xs[t].float() @ xs[t].float().T).sum().item()    # unrelated eager work between replays
    assert state.pos.tolist() == [n % 16] * B
    assert torch.equal(state.h_loc, eager_state.h_loc) and torch.equal(state.c_prev_loc, eager_state.c_prev_loc)


def test_step_rejects_bad_arguments():
    from spear_amd import _btp

    B, H = 2, 4
    a, b, c, v = (t.to(DEV) for t in token_inputs(B, H, H, 1, seed=1)[0])
    out = torch.empty_like(v)
    h, r, cp = torch.zeros(B, H, 16, device=DEV), torch.ones(B, H, device=DEV), torch.zeros(B, H, 16, device=DEV)
    with pytest.raises(RuntimeError, match="state must be float32"):
        _btp.mix_step(a, b, c, v, out, h.bfloat16(), r, cp, None, False, 16, H, H)
    with pytest.raises(RuntimeError, match="pos must be int32"):
        _btp.mix_step(a, b, c, v, out, h, r, cp, torch.zeros(B, device=DEV), False, 16, H, H)
    with pytest.raises(RuntimeError, match="shape"):
        _btp.mix_step(a, b, c, v, out, h, r[:1], cp, None, False, 16, H, H)
    with pytest.raises(RuntimeError, match="block_len must be positive"):
        _btp.mix_step(a, b, c, v, out, h, r, cp, None, False, 0, H, H)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("B,H,Hkv,L", [(3, 4, 4, 1), (2, 8, 2, 15), (2, 3, 3, 17), (2, 32, 32, 63), (2, 5, 1, 65), (3, 12, 4, 129),
                                       (2, 8, 8, 513), (2, 24, 3, 1003), (2, 16, 16, 64)])
def test_prefill_of_any_length_is_one_launch_with_the_state_that_stepping_reaches(B, H, Hkv, L, dtype):
    """The prompt kernel at lengths that end inside a block (and, last case, at a block's end): its output is that of the
    forward kernel on the prompt filled up to a whole block, and its state the one the step kernel reaches, bit for bit."""
    from spear_amd import _btp

    g = torch.Generator().manual_seed(77 + L)
    a, b, c, v = (torch.randn(B, L, w, generator=g).to(dtype).to(DEV) for w in (H, Hkv * 16, Hkv * 16, H * 16))
    print(f"prefill of any length B={B} H={H} Hkv={Hkv} L={L} {dtype}", flush=True)
    out, h, r, c_prev, pos = _btp.load_extension().mix_prefill(a, b, c, v, H, Hkv)
    torch.cuda.synchronize()
    whole = [torch.nn.functional.pad(t, (0, 0, 0, -L % 16)).contiguous() for t in (a, b, c, v)]
    want = torch.empty_like(whole[3])
    _btp.mix_forward(*whole, want, H, Hkv)
    assert torch.equal(out, want[:, :L])
    sh, sr, sc = torch.zeros(B, H, 16, device=DEV), torch.ones(B, H, device=DEV), torch.zeros(B, H, 16, device=DEV)
    sp = torch.zeros(B, device=DEV, dtype=torch.int32)
    y = torch.empty(B, H * 16, device=DEV, dtype=dtype)
    for t in range(L):
        _btp.mix_step(*(q[:, t].contiguous() for q in (a, b, c, v)), y, sh, sr, sc, sp, False, 16, H, Hkv)
    for name, got, ref in (("h", h, sh), ("r", r, sr), ("c_prev", c_prev, sc), ("pos", pos, sp)):
        assert torch.equal(got, ref), name


# (B, H, kv heads): one, two and four token tiles per wavefront and the tile kernel, tiles and head groups that are not full, K = 16 H that ends inside
# a matrix instruction's 32 columns and inside a chunk of loads
@pytest.mark.parametrize("B,H,Hkv", [(1, 1, 1), (16, 3, 1), (17, 5, 5), (33, 32, 8), (200, 24, 8), (1024, 17, 17), (700, 33, 11), (1000, 72, 9)])
def test_layer_token_kernel_against_the_oracle(B, H, Hkv):
    from spear_amd import _btp

    K, g = 16 * H, torch.Generator().manual_seed(31 + B)
    bf = lambda *s, std=1.0: (std * torch.randn(*s, generator=g)).bfloat16()
    w = [bf(n, K, std=K ** -0.5) for n in (H, Hkv * 16, Hkv * 16, H * 16)]
    bias = [bf(n, std=0.3) for n in (H, Hkv * 16, Hkv * 16)]
    x = bf(B, 2 * K)[:, :K]  # rows of a wider buffer
    h, cp = torch.randn(B, H, 16, generator=g), torch.randn(B, H, 16, generator=g)
    r, pos = torch.rand(B, H, generator=g), torch.randint(0, 16, (B,), generator=g, dtype=torch.int32)
    dev = [t.to(DEV) for t in (h, r, cp, pos)]
    xd = torch.zeros(B, 2 * K, device=DEV, dtype=torch.bfloat16)[:, :K].copy_(x)
    wd, bd = [t.to(DEV) for t in w], [t.to(DEV) for t in bias]
    print(f"layer token B={B} H={H} Hkv={Hkv}", flush=True)
    out = _btp.load_extension().layer_token(xd, wd[0], bd[0], wd[1], bd[1], wd[2], bd[2], wd[3], *dev, 16, H, Hkv)
    torch.cuda.synchronize()
    a, b, c, v = (x.double() @ w_.double().T + (0 if b_ is None else b_.double()) for w_, b_ in zip(w, [*bias, None]))
    expand = lambda t: t.view(B, Hkv, 16).repeat_interleave(H // Hkv, 1)
    gate, v = torch.sigmoid(a), v.view(B, H, 16)
    h2 = gate[..., None] * h.double() + torch.sigmoid(expand(b)) * v
    r2 = gate * r.double()
    want = (h2 + r2[..., None] * cp.double()) * expand(c) + v
    done = (pos == 15)[:, None]
    # fp32 sums of K products of about unit total: K roundings of 2^-24 at most, and the hardware's exp and reciprocal
    tol = K * 2.0 ** -24 + 1e-5
    assert_close(f64(out), want.reshape(B, K).numpy(), 2.0 ** -8, 2.0 ** -8, "out")
    assert_close(f64(dev[0]), torch.where(done[..., None], 0.0, h2).numpy(), tol, tol, "h")
    assert_close(f64(dev[1]), torch.where(done, 1.0, r2).numpy(), tol, tol, "r")
    assert_close(f64(dev[2]), torch.where(done[..., None], h2, cp.double()).numpy(), tol, tol, "c_prev")
    assert dev[3].tolist() == ((pos + 1) % 16).tolist()


def test_hooked_projections_are_called_and_give_the_same_step():
    from spear_amd.nn.phalanx.inference import PhalanxStepState, phalanx_step

    layer = _layer(dim=256, seed=6)
    x = torch.randn(5, 256, generator=torch.Generator().manual_seed(8)).bfloat16().to(DEV)
    one, two = PhalanxStepState.zeros(5, 16, DEV), PhalanxStepState.zeros(5, 16, DEV)
    y = phalanx_step(layer, x, one)
    calls = []
    handle = layer.param.proj_b.register_forward_hook(lambda *a: calls.append(1))
    y_hooked = phalanx_step(layer, x, two)
    handle.remove()
    assert calls == [1]
    assert_close(f64(y), f64(y_hooked), 2e-2, 2e-2, "y")
    assert_close(f64(one.h_loc), f64(two.h_loc), 2e-2, 2e-2, "h")


def test_prefill_refuses_an_empty_prompt_and_takes_an_empty_batch():
    from spear_amd.nn.phalanx.inference import phalanx_prefill

    layer = _layer(dim=64, seed=7)
    x = torch.zeros(2, 3, 64, device=DEV, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="at least one token"):
        phalanx_prefill(layer, x[:, :0])
    y, st = phalanx_prefill(layer, x[:0])
    assert y.shape == (0, 3, 64) and st.h_loc.shape == (0, 4, 16) and st.pos.shape == (0,)


@pytest.mark.parametrize("B", [1, 5, 64])
@pytest.mark.parametrize("layout", ["expanded", "overlapping", "wide_rows", "unaligned", "columns", "odd_stride"])
def test_step_takes_tokens_in_any_layout(layout, B):
    """Rows that are one row, that overlap, that lie apart, that start off the 16-byte grid, that are columns: the step of the same
    values laid out densely, up to the roundings of the projections to 16 bits that the general path makes."""
    from spear_amd.nn.phalanx.inference import PhalanxStepState, phalanx_step

    dim, layer = 128, _layer(dim=128, seed=9)
    g = torch.Generator().manual_seed(10)
    base = torch.randn(B + 1, 2 * dim, generator=g).bfloat16().to(DEV)
    x = {"expanded": lambda: base[0, :dim].expand(B, dim),
         "overlapping": lambda: base.view(-1).as_strided((B, dim), (8, 1)),
         "wide_rows": lambda: base[:B, dim:],
         "unaligned": lambda: base.view(-1)[1:1 + B * dim].view(B, dim),
         "columns": lambda: base.view(-1)[:B * dim].view(dim, B).t(),
         "odd_stride": lambda: base.view(-1).as_strided((B, dim), (dim + 1, 1))}[layout]()
    one, two = PhalanxStepState.zeros(B, dim // 16, DEV), PhalanxStepState.zeros(B, dim // 16, DEV)
    for _ in range(2):
        y, want = phalanx_step(layer, x, one), phalanx_step(layer, x.contiguous(), two)
    assert_close(f64(y), f64(want), 2e-2, 2e-2, "y")
    assert_close(f64(one.h_loc), f64(two.h_loc), 2e-2, 2e-2, "h")
    assert one.pos.tolist() == [2] * B


def _steps_equal_the_modules(B, dim):
    from spear_amd.nn.phalanx.inference import PhalanxStepState, phalanx_step

    layer = _layer(dim=dim, seed=12)
    x = torch.randn(20, B, dim, generator=torch.Generator().manual_seed(13)).bfloat16().to(DEV)
    one, two = PhalanxStepState.zeros(B, dim // 16, DEV), PhalanxStepState.zeros(B, dim // 16, DEV)
    one.pos += torch.arange(B, device=DEV, dtype=torch.int32) % 16
    two.pos += one.pos
    for t in range(20):
        y = phalanx_step(layer, x[t], one)
        handle = layer.param.proj_a.register_forward_hook(lambda *a: None)  # the projections as modules
        want = phalanx_step(layer, x[t], two)
        handle.remove()
        assert_close(f64(y), f64(want), 2e-2, 2e-2, f"y[{t}]")
        assert one.pos.tolist() == two.pos.tolist() == [(b + t + 1) % 16 for b in range(B)]


@pytest.mark.parametrize("B,dim", [(73300, 64), (54, 3072)])
def test_step_with_the_output_projection_of_the_library(B, dim):
    """More narrow sequences than the output projection's kernel takes, and some of a wide layer, whose output projection the library has in less time: the
    token kernel moves the block positions on itself, also past a block's end."""
    _steps_equal_the_modules(B, dim)


@pytest.mark.parametrize("B,dim", [(17, 528), (1030, 784)])
def test_a_step_is_two_launches(B, dim):
    """The output projection moves the block positions on, also past a block's end, in its kernel for few rows and in 128 x 128 tiles."""
    from spear_amd.nn.phalanx.inference import PhalanxStepState, phalanx_step

    _steps_equal_the_modules(B, dim)
    layer, state = _layer(dim=dim, seed=12), PhalanxStepState.zeros(B, dim // 16, DEV)
    x = torch.zeros(B, dim, device=DEV, dtype=torch.bfloat16)
    phalanx_step(layer, x, state)
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as profile:
        phalanx_step(layer, x, state)
        torch.cuda.synchronize()
    kernels = [e.name for e in profile.events() if e.device_type == torch.autograd.DeviceType.CUDA]
    assert len(kernels) == 2, kernels


@pytest.mark.parametrize("B,H,Hkv", [(1030, 65, 65), (700, 100, 25)])
def test_steps_of_many_wide_sequences_equal_the_modules(B, H, Hkv):
    """Between 2^26 and 3 2^26 of batch x heads x dim, where the compiled step runs the projections in tiles."""
    from spear_amd import Phalanx
    from spear_amd.nn.phalanx.inference import PhalanxStepState, phalanx_step

    torch.manual_seed(16)
    layer = Phalanx(dim=16 * H, length=128, method="fused", dtype=torch.bfloat16, kv_heads=Hkv).to(DEV)
    x = torch.randn(18, B, 16 * H, generator=torch.Generator().manual_seed(17)).bfloat16().to(DEV)
    one, two = PhalanxStepState.zeros(B, H, DEV), PhalanxStepState.zeros(B, H, DEV)
    for t in range(18):
        print(f"step {t} B={B} H={H} Hkv={Hkv}", flush=True)
        y = phalanx_step(layer, x[t], one)
        handle = layer.param.proj_a.register_forward_hook(lambda *a: None)  # the projections as modules
        want = phalanx_step(layer, x[t], two)
        handle.remove()
        assert_close(f64(y), f64(want), 2e-2, 2e-2, f"y[{t}]")
        assert torch.equal(one.pos, two.pos)
    assert_close(f64(one.h_loc), f64(two.h_loc), 2e-2, 2e-2, "h")


@pytest.mark.parametrize("B,L,dim", [(2, 48, 64), (1, 33, 1040)])
def test_prompts_off_the_16_byte_grid_and_on_another_stream(B, L, dim):
    from spear_amd.nn.phalanx.inference import phalanx_prefill

    layer = _layer(dim=dim, seed=14)
    x = torch.randn(B, L, dim, generator=torch.Generator().manual_seed(15)).bfloat16().to(DEV)
    shifted = torch.cat([x.new_zeros(1), x.view(-1)])[1:].view(x.shape)
    y, st = phalanx_prefill(layer, x)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ys, sts = phalanx_prefill(layer, x)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(y, ys) and all(torch.equal(getattr(st, n), getattr(sts, n)) for n in ("h_loc", "r_pref", "c_prev_loc", "pos"))
    yu, stu = phalanx_prefill(layer, shifted)  # the library's products for the projections
    assert_close(f64(yu), f64(y), 2e-2, 2e-2, "y")
    assert_close(f64(stu.h_loc), f64(st.h_loc), 2e-2, 2e-2, "h")
    assert torch.equal(stu.pos, st.pos)
