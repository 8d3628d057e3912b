"""The layer's projections through spear_layer_linear, up to four of them on the same rows, its weight gradients and a decode token's projections in tiles,
against float64 products of the same bf16 operands at the edges of the kernels' tiles."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def assert_product(got, x, w, bias, label):
    """|got - x w^T - b| <= half a step of the result (bf16 has 8 significant bits: up to 2^-8 of it) and the fp32 sum's error, K 2^-24 of the terms' sum."""
    x, w = x.double(), w.double()
    want = x @ w.t()
    terms = x.abs() @ w.abs().t()
    if bias is not None:
        want = want + bias.double()
        terms = terms + bias.double().abs()
    bound = want.abs() * 2.0**-8 + terms * (x.shape[1] + 1) * 2.0**-24 * (1 + 2.0**-8)
    over = (got.double() - want).abs() - bound
    assert over.max().item() <= 0, f"{label}: {over.max().item():.3e} over the bound"


def kernel_of(M, K, columns, extra=0):
    """Which kernel spear_layer_linear takes: 0 for few rows, 1 tiles of 128 x 128, 2 of 256 x 256."""
    import ctypes

    from spear_amd import _btp

    return _btp.load_library().spear_layer_linear_choice(len(columns), ctypes.c_longlong(K + extra), M, K, (ctypes.c_int * len(columns))(*columns))


# Kernel, M, K, columns of the projections (bias on all but every third). Remainders of rows, of columns, of 64 columns of K; widths of 128 and
# less (half of the larger tiles) and not a multiple of 8 (element stores).
SHAPES = [
    # 256 x 256 tiles, several per workgroup, ending in another projection and in the last rows; results stored at once (K up to 1024) or not; two
    # and three steps of K, so that the requests of one tile reach into the next
    (2, 33027, 520, (592, 592, 257, 37)),
    (2, 33027, 1032, (1040, 129, 128, 127)),
    (2, 131077, 72, (1024, 130)),
    (2, 40007, 1000, (640,)),
    (2, 65541, 136, (1024, 130)),
    (2, 50000, 328, (256, 272, 16, 5)),
    (2, 16500, 1288, (520, 24, 136)),
    (2, 8192, 2048, (2048, 512, 512, 128)),
    # 128 x 128 tiles, more and fewer of them than compute units, in one chain over K and in quarters
    (1, 4099, 520, (592, 592, 257, 37)),
    (1, 4096, 512, (512, 512, 512, 32)),
    (1, 2305, 1032, (1040, 129, 128, 127)),
    (1, 16400, 136, (256, 272, 16, 5)),
    (1, 20000, 72, (1024, 130)),
    (1, 9000, 1000, (640,)),
    (1, 1003, 592, (592, 592, 592, 37)),
    (1, 700, 1000, (1040, 130, 129, 24)),
    (1, 2048, 72, (1024, 1024, 1024, 64)),
    (1, 2049, 1032, (1032, 1040, 1041, 5)),
    (0, 129, 1000, (1040, 130, 129, 24)),
]


@pytest.mark.parametrize("kernel,M,K,columns", SHAPES)
@pytest.mark.parametrize("extra", [0, 24], ids=["dense", "strided"])
def test_large_projections_against_float64(kernel, M, K, columns, extra):
    from spear_amd import _btp

    assert kernel_of(M, K, columns, extra) == kernel

    g = torch.Generator(device=DEV).manual_seed(M + K + extra)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=DEV).bfloat16()

    x = normal(M, K + extra)[:, :K]
    weights = [(normal(n, K) * K**-0.5).bfloat16() for n in columns]
    biases = [None if i % 3 == 2 else normal(n) for i, n in enumerate(columns)]
    print(f"projections M={M} K={K} columns={columns} row stride {K + extra}", flush=True)
    out = _btp.load_extension().linears(x, weights, biases)
    for i, (y, w, b) in enumerate(zip(out, weights, biases)):
        assert_product(y, x, w, b, f"M={M} K={K} projection {i} of {len(columns)}")


@pytest.mark.parametrize("kernel,M", [(1, 4096), (2, 33028)])
def test_large_projections_keep_rows_apart(kernel, M):
    """What lies beside a row (the next row's first columns, read with a step that K does not fill) must not reach its result."""
    from spear_amd import _btp

    K, N = 520, 1040
    assert kernel_of(M, K, [N]) == kernel
    x = torch.randn(M, K, device=DEV).bfloat16()
    x[1::2] = float("nan")
    w = torch.randn(N, K, device=DEV).bfloat16()
    y, = _btp.load_extension().linears(x, [w], [None])
    torch.cuda.synchronize()
    assert torch.isfinite(y[::2]).all() and torch.isnan(y[1::2]).all()


@pytest.mark.parametrize("kernel,M", [(1, 4096), (2, 32768)])
def test_large_projections_in_a_graph_follow_their_inputs(kernel, M):
    from spear_amd import _btp

    K, N = 512, 1024
    assert kernel_of(M, K, [N, N]) == kernel
    x, w = torch.randn(M, K, device=DEV).bfloat16(), torch.randn(N, K, device=DEV).bfloat16()
    run = lambda: _btp.load_extension().linears(x, [w, w], [None, None])
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = run()
    for seed in range(3):
        x.copy_(torch.randn(M, K, generator=torch.Generator().manual_seed(seed)).to(DEV))
        graph.replay()
        torch.cuda.synchronize()
        for got, want in zip(y, run()):
            assert torch.equal(got, want)


@pytest.mark.parametrize("M,dim,heads,kv_heads", [(33, 592, 37, 37), (5, 128, 8, 2), (1, 2048, 128, 32), (70, 1040, 65, 5)])
def test_transposed_weights_and_padding(M, dim, heads, kv_heads):
    import ctypes

    from spear_amd import _btp

    lib = _btp.load_library()
    lib.spear_layer_transpose.argtypes = [ctypes.c_void_p] * 8 + [ctypes.c_longlong] + [ctypes.c_int] * 5 + [ctypes.c_void_p]
    F, Fkv = 16 * heads, 16 * kv_heads
    used = 2 * Fkv + F + heads
    ld = -(-used // 64) * 64
    w_a, w_b, w_c, w_v = (torch.randn(n, dim, device=DEV).bfloat16() for n in (heads, Fkv, Fkv, F))
    w_out = torch.randn(dim, F, device=DEV).bfloat16()
    stacked, out_t = torch.full((dim, ld), 7.0, device=DEV).bfloat16(), torch.full((F, dim), 7.0, device=DEV).bfloat16()
    packed = torch.full((M, ld), 7.0, device=DEV).bfloat16()
    print(f"transpose M={M} dim={dim} heads={heads} kv_heads={kv_heads} ld={ld}", flush=True)
    rc = lib.spear_layer_transpose(*(t.data_ptr() for t in (w_a, w_b, w_c, w_v, w_out, stacked, out_t, packed)), M, ld, dim, heads, Fkv, F,
                                   torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    assert torch.equal(stacked[:, :used], torch.cat([w_b, w_c, w_v, w_a]).t()) and (stacked[:, used:] == 0).all()
    assert torch.equal(out_t, w_out.t())
    assert (packed[:, :used] == 7).all() and (packed[:, used:] == 0).all()


# tokens, (columns of dy, its row length, columns of x) per product, splits (0: as modelled). Remainders of 32 tokens, of 256 and 128 columns;
# one step per split and fewer steps than stages; units of both products on one workgroup; splits that differ by a step.
WGRADS = [
    (1, [(8, 8, 8)], [1]),
    (33, [(40, 64, 72), (300, 304, 136)], [2, 1]),
    (1000, [(1813, 1856, 592), (592, 592, 592)], [0, 0]),
    (4099, [(257, 264, 264), (129, 136, 520)], [7, 128]),
    (16384, [(1568, 1600, 512), (512, 512, 512)], [0, 0]),
    (9000, [(3136, 3136, 1024)], [3]),
]


@pytest.mark.parametrize("M,products,splits", WGRADS)
def test_weight_gradients_over_splits_against_float64(M, products, splits):
    import ctypes

    from spear_amd import _btp

    lib, n = _btp.load_library(), len(products)
    g = torch.Generator(device=DEV).manual_seed(M)
    dys = [torch.randn(M, ld, generator=g, device=DEV).bfloat16() for _, ld, _ in products]
    xs = [torch.randn(M, K, generator=g, device=DEV).bfloat16() for _, _, K in products]
    splits = [s or lib.spear_layer_wgrad_splits(ctypes.c_longlong(M), N, K) for s, (N, _, K) in zip(splits, products)]
    units = sum(-(-N // 256) * -(-K // 256) * s for (N, _, K), s in zip(products, splits))
    parts = torch.full((units * 65536,), float("nan"), device=DEV)
    dws = [torch.full((N + 1, K), 7.0, device=DEV).bfloat16() for N, _, K in products]
    tall = torch.randn(70, 24, generator=g, device=DEV)
    sums = torch.empty(24, device=DEV).bfloat16()
    print(f"weight gradients M={M} {products} splits={splits}", flush=True)
    ints, pointers = ctypes.c_int * n, ctypes.c_void_p * n
    of = lambda ts: pointers(*(t.data_ptr() for t in ts))
    lds, Ns, Ks, sp = (ints(*v) for v in ([p[1] for p in products], [p[0] for p in products], [p[2] for p in products], splits))
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.spear_layer_wgrad(n, of(dys), lds, lds, Ns, of(xs), Ks, sp, ctypes.c_longlong(M), ctypes.c_void_p(parts.data_ptr()), stream) == 0
    one = lambda t: (ctypes.c_void_p * 1)(t.data_ptr())
    assert lib.spear_layer_wgrad_sums(n, ctypes.c_void_p(parts.data_ptr()), Ns, Ks, sp, of(dws), 1, one(tall), one(sums), (ctypes.c_longlong * 1)(70),
                                      (ctypes.c_longlong * 1)(24), _btp._BF16, stream) == 0
    torch.cuda.synchronize()
    for dy, x, dw, (N, _, K) in zip(dys, xs, dws, products):
        assert_product(dw[:N], dy[:, :N].t(), x.t(), None, f"M={M} [{N}, {K}]")
        assert (dw[N] == 7).all()
    # 70 fp32 additions, then half a step of the result
    want = tall.double().sum(0)
    assert ((sums.double() - want).abs() <= want.abs() * 2.0**-8 + tall.double().abs().sum(0) * 71 * 2.0**-24).all()


# Rows of tokens and pairs of heads that end inside a tile, an odd number of heads, shared kv heads and a remainder of the steps of 64 columns, where the
# tiles are taken (the first seven; the last two of them have one step of 64 columns), and sizes past 512 (head, 16 tokens) pairs at which the other kernel with four token tiles per wavefront is.
# The last case's rows of tokens lie so far apart that 64 of them reach past the tiles' 32-bit offsets: it stays with the other kernel.
@pytest.mark.parametrize("B,H,Hkv,K,ldx", [(700, 37, 37, 592, 592), (4090, 8, 2, 128, 128), (700, 33, 11, 528, 552), (700, 32, 32, 520, 520),
                                           (16333, 3, 3, 1032, 1032), (16380, 2, 1, 32, 32),
                                           (8190, 3, 3, 48, 56), (1030, 37, 37, 592, 592), (333, 33, 11, 528, 528), (2049, 8, 2, 128, 128), (200, 48, 12, 768, 768),
                                           (5000, 2, 1, 96, 96), (20000, 1, 1, 16, 16), (80, 128, 128, 128, 1 << 24)])
def test_token_tiles_against_float64(B, H, Hkv, K, ldx):
    from spear_amd import _btp

    g = torch.Generator(device=DEV).manual_seed(B + H)
    normal = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    x = torch.empty((B - 1) * ldx + K, device=DEV, dtype=torch.bfloat16).as_strided((B, K), (ldx, 1))
    x.copy_(normal(B, K))
    w_a, w_b, w_c, w_v = ((normal(n, K) * K**-0.5).bfloat16() for n in (H, 16 * Hkv, 16 * Hkv, 16 * H))
    b_a, b_b, b_c = (normal(n).bfloat16() for n in (H, 16 * Hkv, 16 * Hkv))
    h, r, c_prev = normal(B, H, 16), torch.rand(B, H, generator=g, device=DEV), normal(B, H, 16)
    pos = torch.randint(0, 16, (B,), generator=g, device=DEV, dtype=torch.int32)
    state = [t.clone() for t in (h, r, c_prev, pos)]
    print(f"token tiles B={B} H={H} Hkv={Hkv} K={K} ldx={ldx}", flush=True)
    out = _btp.load_extension().layer_token(x, w_a, b_a, w_b, b_b, w_c, b_c, w_v, *state, 16, H, Hkv, False)
    # products in float64, and what K + 1 fp32 additions may be off by
    xd = x.double()
    per_head = lambda t: t.view(B, Hkv, 1, 16).expand(B, Hkv, H // Hkv, 16).reshape(B, H, 16)

    def product(w, b):
        y, e = xd @ w.double().t(), (xd.abs() @ w.double().abs().t()) * (K + 1) * 2.0**-24
        return (y, e) if b is None else (y + b.double(), e + (y + b.double()).abs() * 2.0**-24)

    (a, ea), (b, eb), (c, ec), (v, ev) = product(w_a, b_a), product(w_b, b_b), product(w_c, b_c), product(w_v, None)
    b, eb, c, ec = per_head(b), per_head(eb), per_head(c), per_head(ec)
    v, ev, a, ea = v.view(B, H, 16), ev.view(B, H, 16), torch.sigmoid(a)[..., None], ea[..., None]
    gate = torch.sigmoid(b)
    fast = 2.0**-20  # exp and reciprocal of the hardware, relative, some roundings of the step with it
    new = a * h.double() + gate * v
    e_new = (ea / 4 + fast) * h.double().abs() + (eb / 4 + fast) * v.abs() + ev + new.abs() * 2.0**-22
    r_new = a[..., 0] * r.double()
    e_r = (ea[..., 0] / 4 + fast) * r.double()
    sum_ = new + r_new[..., None] * c_prev.double()
    e_sum = e_new + e_r[..., None] * c_prev.double().abs() + sum_.abs() * 2.0**-22
    want = sum_ * c + v
    e_out = e_sum * (c.abs() + ec) + sum_.abs() * ec + ev + (sum_ * c).abs() * 2.0**-22
    end = (pos == 15)[:, None]
    got_h, got_r, got_c, got_pos = (t.double() for t in state)
    zero = torch.zeros_like(new)

    def within(got, want, error, name):
        assert ((got - want).abs() <= error).all(), f"{name}: {((got - want).abs() - error).max().item():.3e} over the bound"

    within(out.double().view(B, H, 16), want, e_out + (want.abs() + e_out) * 2.0**-8, "out")
    within(got_h, torch.where(end[..., None], zero, new), e_new, "h")
    within(got_r, torch.where(end, torch.ones_like(r_new), r_new), e_r, "r")
    within(got_c, torch.where(end[..., None], new, c_prev.double()), e_new, "c_prev")
    assert torch.equal(state[3], pos)


# Sizes of the tiles (the first eight; quarters of K that end inside a step of 64 columns, of one instruction, of one step, and no columns in the last quarter)
# and of four token tiles per wavefront.
@pytest.mark.parametrize("B,H,Hkv,K", [(1024, 32, 32, 512), (700, 37, 37, 592), (200, 64, 16, 1024), (4090, 8, 2, 128), (8001, 4, 4, 64), (3200, 10, 10, 160), (16380, 2, 1, 32),
                                       (8190, 3, 3, 48),
                                       (10007, 1, 1, 16), (5003, 3, 1, 48), (3001, 5, 5, 80)])
def test_a_token_is_the_same_whatever_number_comes_with_it(B, H, Hkv, K):
    """The tiles add up a token's products as the kernel for few tokens does: the state, which is kept in fp32, and the result are equal."""
    from spear_amd import _btp

    g = torch.Generator(device=DEV).manual_seed(B)
    normal = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    x = normal(B, K).bfloat16()
    weights = [(normal(n, K) * K**-0.5).bfloat16() for n in (H, 16 * Hkv, 16 * Hkv, 16 * H)]
    b_a, b_b, b_c = (normal(n).bfloat16() for n in (H, 16 * Hkv, 16 * Hkv))
    state = [normal(B, H, 16), torch.rand(B, H, generator=g, device=DEV), normal(B, H, 16),
             torch.randint(0, 16, (B,), generator=g, device=DEV, dtype=torch.int32)]

    def step(rows):
        of = [t[rows].clone() for t in state]
        out = _btp.load_extension().layer_token(x[rows], weights[0], b_a, weights[1], b_b, weights[2], b_c, weights[3], *of, 16, H, Hkv, False)
        return out, *of

    print(f"tokens B={B} H={H} Hkv={Hkv} K={K}", flush=True)
    all_at_once = step(slice(0, B))
    for first in (0, 16 * (B // 32), B - B % 16 if B % 16 else B - 16):
        few = step(slice(first, min(B, first + 16)))
        for got, want in zip(all_at_once, few):
            assert torch.equal(got[first:first + 16], want)


@pytest.mark.parametrize("B,H,tiles", [(33, 256, False), (64, 256, False), (65, 256, True), (33, 272, True)])
def test_up_to_64_tokens_of_256_heads_stay_with_the_kernel_without_tiles(B, H, tiles):
    from spear_amd import _btp

    K, g = 4096, torch.Generator(device=DEV).manual_seed(B)
    normal = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    x, weights = normal(B, K).bfloat16(), [normal(n, K).bfloat16() for n in (H, 16 * H, 16 * H, 16 * H)]
    b_a, b_b, b_c = (normal(n).bfloat16() for n in (H, 16 * H, 16 * H))
    state = [normal(B, H, 16), torch.rand(B, H, generator=g, device=DEV), normal(B, H, 16), torch.zeros(B, device=DEV, dtype=torch.int32)]
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as profile:
        _btp.load_extension().layer_token(x, weights[0], b_a, weights[1], b_b, weights[2], b_c, weights[3], *state, 16, H, H, False)
        torch.cuda.synchronize()
    kernel, = [e.name for e in profile.events() if e.device_type == torch.autograd.DeviceType.CUDA]
    assert ("layer_token_tile_kernel" in kernel) == tiles, kernel


# Sizes that 128 x 128 tiles take up to which K is added up in quarters: quarters that end inside a step of 64 columns, and of one instruction.
@pytest.mark.parametrize("M,K,columns", [(1024, 512, (512, 512, 512, 32)), (1003, 592, (592, 592, 257, 37)), (700, 1040, (1040, 130, 129, 24)), (1500, 72, (1024, 130))])
def test_a_row_is_the_same_whatever_number_comes_with_it(M, K, columns):
    """The tiles add up a row's products as the kernel for few rows does: the results are equal."""
    from spear_amd import _btp

    assert (kernel_of(M, K, columns), kernel_of(16, K, columns)) == (1, 0)

    g = torch.Generator(device=DEV).manual_seed(M)
    normal = lambda *shape: torch.randn(*shape, generator=g, device=DEV).bfloat16()
    x, weights, biases = normal(M, K), [normal(n, K) for n in columns], [normal(n) for n in columns]
    print(f"rows M={M} K={K} columns={columns}", flush=True)
    out = _btp.load_extension().linears(x, weights, biases)
    for first in (0, 16 * (M // 32), M - 16):
        for y, few in zip(out, _btp.load_extension().linears(x[first:first + 16], weights, biases)):
            assert torch.equal(y[first:first + 16], few)


# The kernel for few rows and 128 x 128 tiles, in each of which one workgroup of a panel of rows moves their positions.
@pytest.mark.parametrize("M,K,N", [(17, 528, 528), (129, 1024, 1024), (1003, 1040, 1040), (5000, 768, 768), (40000, 136, 136)])
def test_positions_move_on_with_a_projection(M, K, N):
    import ctypes

    from spear_amd import _btp

    lib = _btp.load_library()
    g = torch.Generator(device=DEV).manual_seed(M)
    x, w = torch.randn(M, K, generator=g, device=DEV).bfloat16(), (torch.randn(N, K, generator=g, device=DEV) * K**-0.5).bfloat16()
    y = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    pos = torch.randint(0, 16, (M + 1,), generator=g, device=DEV, dtype=torch.int32)
    was = pos.clone()
    one = lambda t: (ctypes.c_void_p * 1)(t.data_ptr())
    print(f"positions with a projection M={M} K={K} N={N}", flush=True)
    assert lib.spear_layer_linear(1, ctypes.c_void_p(x.data_ptr()), ctypes.c_longlong(K), M, K, one(w), (ctypes.c_void_p * 1)(None), one(y), (ctypes.c_int * 1)(N),
                                  ctypes.c_void_p(pos.data_ptr()), 16, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    assert_product(y, x, w, None, f"M={M} K={K}")
    assert torch.equal(pos[:M], (was[:M] + 1) % 16) and pos[M] == was[M]


# The kernel for few rows in each of its tiles (rows by columns of a workgroup): 16 x 16, 16 x 32, 32 x 32, 16 x 64, 32 x 64, 64 x 64; rows and
# columns that end inside a tile, a result narrower than one, K that ends inside an instruction's 32 columns and with a quarter that has none.
@pytest.mark.parametrize("M,K,columns", [(1, 8, (1,)), (17, 520, (513, 16, 7, 130)), (256, 40, (256,)), (40, 264, (1500, 37)), (100, 136, (2000,)), (13, 72, (8300,)),
                                         (300, 64, (1000,)), (1000, 40, (999, 3))])
def test_few_rows_against_float64(M, K, columns):
    from spear_amd import _btp

    g = torch.Generator(device=DEV).manual_seed(M + K)
    normal = lambda *shape: torch.randn(*shape, generator=g, device=DEV).bfloat16()
    x, weights, biases = normal(M, K + 8)[:, :K], [normal(n, K) for n in columns], [None if i % 3 == 2 else normal(n) for i, n in enumerate(columns)]
    print(f"few rows M={M} K={K} columns={columns}", flush=True)
    for i, y in enumerate(_btp.load_extension().linears(x, weights, biases)):
        assert_product(y, x, weights[i], biases[i], f"M={M} K={K} projection {i}")


# Products of one split, which are rounded where they are made: alone, beside one with parts in either place; results narrower than a half tile, that
# end inside one, and several units per workgroup.
@pytest.mark.parametrize("M,products,splits", [(1, [(8, 8, 8)], [1]), (33, [(300, 304, 136), (40, 64, 72)], [1, 1]), (1000, [(1813, 1856, 592), (592, 592, 592)], [1, 3]),
                                               (97, [(257, 264, 264), (1040, 1040, 520)], [3, 1]), (64, [(6272, 6272, 2048), (2048, 2048, 2048)], [1, 1])])
def test_weight_gradients_of_one_split_against_float64(M, products, splits):
    import ctypes

    from spear_amd import _btp

    lib, n = _btp.load_library(), len(products)
    g = torch.Generator(device=DEV).manual_seed(M)
    dys = [torch.randn(M, ld, generator=g, device=DEV).bfloat16() for _, ld, _ in products]
    xs = [torch.randn(M, K, generator=g, device=DEV).bfloat16() for _, _, K in products]
    dws = [torch.full((N + 1, K), 7.0, device=DEV).bfloat16() for N, _, K in products]
    parted = [i for i in range(n) if splits[i] > 1]
    units = sum(-(-products[i][0] // 256) * -(-products[i][2] // 256) * splits[i] for i in parted)
    parts = torch.full((units * 65536,), float("nan"), device=DEV)
    print(f"weight gradients without parts M={M} {products} splits={splits}", flush=True)
    ints = lambda values: (ctypes.c_int * len(values))(*values)
    of = lambda ts: (ctypes.c_void_p * len(ts))(*(t.data_ptr() for t in ts))
    whole = (ctypes.c_void_p * n)(*(dw.data_ptr() if s == 1 else None for dw, s in zip(dws, splits)))
    lds, Ns, Ks = (ints([p[k] for p in products]) for k in (1, 0, 2))
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.spear_layer_wgrad_to(n, of(dys), lds, lds, Ns, of(xs), Ks, ints(splits), ctypes.c_longlong(M), ctypes.c_void_p(parts.data_ptr() if parted else None),
                                    whole, stream) == 0
    if parted:
        pick = lambda k: ints([products[i][k] for i in parted])
        assert lib.spear_layer_wgrad_sums(len(parted), ctypes.c_void_p(parts.data_ptr()), pick(0), pick(2), ints([splits[i] for i in parted]), of([dws[i] for i in parted]),
                                          0, None, None, None, None, _btp._BF16, stream) == 0
    torch.cuda.synchronize()
    for dy, x, dw, (N, _, K) in zip(dys, xs, dws, products):
        assert_product(dw[:N], dy[:, :N].t(), x.t(), None, f"M={M} [{N}, {K}]")
        assert (dw[N] == 7).all()


def test_backward_of_few_tokens_of_a_wide_layer_needs_little_room():
    """No fp32 array of the size of the weight gradients: beside what is left afterwards, the transposed weights and arrays of the tokens."""
    from spear_amd import Phalanx

    torch.manual_seed(0)
    layer = Phalanx(dim=2048, length=64, method="fused", dtype=torch.bfloat16).to(DEV)
    x = torch.randn(1, 64, 2048, device=DEV).bfloat16()
    layer(x).backward(x)
    layer.zero_grad(set_to_none=True)
    y = layer(x)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    y.backward(x)
    torch.cuda.synchronize()
    weights = sum(p.numel() * p.element_size() for p in layer.parameters())
    assert torch.cuda.max_memory_allocated() - torch.cuda.memory_allocated() < 1.25 * weights


@pytest.mark.parametrize("M,N,K", [(65536, 1568, 512), (16384, 6272, 2048)])
def test_weight_gradients_lose_no_precision_against_the_library_in_slices(M, N, K):
    """The layer's backward takes splits of no more tokens than the library's slices: as many of the results are the nearest 16-bit value to the sum in
    64 bits, up to five standard deviations of that number."""
    import ctypes

    from spear_amd import _btp
    from spear_amd.nn.phalanx.projections import slice_count

    lib, slices = _btp.load_library(), slice_count(M, N, K)
    splits = lib.spear_layer_wgrad_splits_from(ctypes.c_longlong(M), N, K, slices)
    assert slices > 1 and splits >= slices
    g = torch.Generator(device=DEV).manual_seed(M)
    dy, x = (torch.randn(M, n, generator=g, device=DEV).bfloat16() for n in (N, K))
    parts, dw, sliced = torch.empty(-(-N // 256) * -(-K // 256) * splits * 65536, device=DEV), torch.empty(N, K, device=DEV).bfloat16(), torch.empty(N, K, device=DEV).bfloat16()
    one, of = lambda v: (ctypes.c_int * 1)(v), lambda t: (ctypes.c_void_p * 1)(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    print(f"weight gradients M={M} [{N}, {K}] splits={splits} slices={slices}", flush=True)
    assert lib.spear_layer_wgrad(1, of(dy), one(N), one(N), one(N), of(x), one(K), one(splits), ctypes.c_longlong(M), ctypes.c_void_p(parts.data_ptr()), stream) == 0
    assert lib.spear_layer_wgrad_sums(1, ctypes.c_void_p(parts.data_ptr()), one(N), one(K), one(splits), of(dw), 0, None, None, None, None, _btp._BF16, stream) == 0
    of_slices = torch.bmm(dy.view(slices, M // slices, N).transpose(1, 2).contiguous(), x.view(slices, M // slices, K), out_dtype=torch.float32)
    _btp.load_extension().layer_sums([of_slices.view(slices, N * K)], [sliced])
    want = sum(dy[i:i + 8192].double().t() @ x[i:i + 8192].double() for i in range(0, M, 8192)).bfloat16()
    off, off_sliced = ((t != want).sum().item() for t in (dw, sliced))
    assert off <= off_sliced + 5 * off_sliced**0.5
