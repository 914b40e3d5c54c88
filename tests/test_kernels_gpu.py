"""Each HIP kernel alone against its plain torch twin, at sizes other than the tiny models'."""

import ctypes
import math

import pytest
import torch

from twins import TwinKernels

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DTYPES = [torch.float32, torch.bfloat16]


@pytest.fixture(scope="module")
def hip():
    from simple_inference_amd.kernels import HipKernels
    return HipKernels()


twin = TwinKernels()


def tol(dtype):
    return dict(rtol=1e-5, atol=1e-5) if dtype == torch.float32 else dict(rtol=1.6e-2, atol=1e-2)


def rnd(*shape, dtype=torch.float32, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


class Ctx:
    """The fields of a step context that the kernels read."""

    def __init__(self, q_lens, kv_lens):
        pos, sot, cu = [], [], [0]
        for s, (q, kv) in enumerate(zip(q_lens, kv_lens)):
            pos += list(range(kv - q, kv))
            sot += [s] * q
            cu.append(cu[-1] + q)
        i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
        self.positions, self.seq_of_token, self.cu_q, self.kv_len = i32(pos), i32(sot), i32(cu), i32(kv_lens)
        self.n_tokens, self.n_seqs = len(pos), len(q_lens)
        self.max_q_len, self.max_kv_len = max(q_lens), max(kv_lens)
        self.q_lens, self.kv_bound = list(q_lens), 0
        self.n_decode_seqs = next((i for i, q in enumerate(q_lens) if q != 1), len(q_lens))


class Cache:
    def __init__(self, n_pages, n_kv, page_size, head_dim, dtype, kv_lens, seed=0):
        self.page_size = page_size
        self.k_pages = torch.zeros(n_pages, n_kv, page_size, head_dim, dtype=dtype, device=DEV)
        self.v_pages = torch.zeros(n_pages, n_kv, head_dim, page_size, dtype=dtype, device=DEV)
        g = torch.Generator().manual_seed(seed)
        perm = torch.randperm(n_pages, generator=g).tolist()  # pages in no particular order
        width = max(-(-kv // page_size) for kv in kv_lens)
        table = torch.full((len(kv_lens), width), -1, dtype=torch.int32)
        for s, kv in enumerate(kv_lens):
            for i in range(-(-kv // page_size)):
                table[s, i] = perm.pop()
        self.block_table = table.to(DEV)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hidden", [72, 1000, 3072])
def test_embed(hip, dtype, hidden):
    table = rnd(517, hidden, dtype=dtype)
    ids = torch.tensor([0, 516, 3, 3, 100], dtype=torch.int32, device=DEV)
    assert torch.equal(hip.embed(ids, table), twin.embed(ids, table))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [1, 33, 4096, 70000])
def test_take_rows(hip, dtype, width):
    """Rows of every width and alignment; a matrix of one row, whose stride is that of the wider matrix it comes from."""
    x = rnd(9, width, dtype=dtype, seed=1)
    rows = torch.tensor([8, 0, 3, 3], dtype=torch.int32, device=DEV)
    assert torch.equal(hip.take_rows(x, rows), x[rows.long()])
    assert hip.take_rows(x, rows[:0]).shape == (0, width)
    one = rnd(1, 3 * width, dtype=dtype, seed=2)[:, :width]
    assert one.is_contiguous() and one.stride(0) == 3 * width
    assert torch.equal(hip.take_rows(one, rows[1:2].repeat(2)), one.repeat(2, 1))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hidden", [40, 1000, 3072, 5000])
def test_add_rmsnorm(hip, dtype, hidden):
    res = rnd(7, hidden, seed=1, scale=3.0)
    delta = rnd(7, hidden, dtype=dtype, seed=2)
    w = 1 + 0.1 * rnd(hidden, seed=3)
    r1, r2 = res.clone(), res.clone()
    out = hip.add_rmsnorm(r1, delta, w, 1e-5, dtype)
    ref = twin.add_rmsnorm(r2, delta, w, 1e-5, dtype)
    torch.testing.assert_close(out.float(), ref.float(), **tol(dtype))
    torch.testing.assert_close(r1, r2, rtol=0, atol=0)
    # no delta; selected rows leave the residual alone
    rows = torch.tensor([6, 0, 3], dtype=torch.int32, device=DEV)
    r3 = res.clone()
    out = hip.add_rmsnorm(r3, delta, w, 1e-5, dtype, rows)
    ref = twin.add_rmsnorm(res.clone(), delta, w, 1e-5, dtype, rows)
    torch.testing.assert_close(out.float(), ref.float(), **tol(dtype))
    assert torch.equal(r3, res)
    out = hip.add_rmsnorm(r3, None, w, 1e-5, dtype)
    torch.testing.assert_close(out.float(), twin.add_rmsnorm(res.clone(), None, w, 1e-5, dtype).float(), **tol(dtype))


def test_rmsnorm_eps_is_inside_the_root(hip):
    x = torch.full((1, 64), 1e-4, device=DEV)
    w = torch.ones(64, device=DEV)
    out = hip.add_rmsnorm(x.clone(), None, w, 1e-2, torch.float32)
    assert abs(out[0, 0].item() - 1e-4 / math.sqrt(1e-8 + 1e-2)) < 1e-8


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("inter", [24, 37, 1000, 8192])
def test_swiglu(hip, dtype, inter):
    gu = rnd(5, 2 * inter, dtype=dtype, scale=3.0)
    torch.testing.assert_close(hip.swiglu(gu).float(), twin.swiglu(gu).float(), **tol(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", [(1, 37, 50), (5, 130, 77), (70, 64, 256), (130, 3, 1000)])
def test_gemm_generic(hip, dtype, shape):
    M, N, K = shape
    x, w = rnd(M, K, dtype=dtype, seed=1), rnd(N, K, dtype=dtype, seed=2)
    ref = x.double() @ w.double().T
    out = hip.gemm_generic(x, w, out_float32=True)
    torch.testing.assert_close(out.double(), ref, rtol=1e-5, atol=1e-4)
    if dtype == torch.bfloat16:
        out = hip.gemm_generic(x, w)
        assert out.dtype == torch.bfloat16
        torch.testing.assert_close(out.double(), ref, **tol(dtype))


def test_gemm_generic_in_float32_has_the_tiles_workspace(hip):
    x, w, seen, real = rnd(303, 512, seed=1), rnd(4096, 512, seed=2), [], hip.core.sia_gemm_f32
    hip.core.sia_gemm_f32 = lambda *a: seen.append(a[3]) or real(*a)
    try:
        assert torch.equal(hip.gemm_generic(x, w), hip.linear(x, w))
    finally:
        hip.core.sia_gemm_f32 = real
    assert len(seen) == 2 and all(seen)


@pytest.mark.parametrize("shape", [(1, 48, 64), (8, 5120, 3072), (16, 3072, 8192), (3, 16, 320), (11, 1008, 1024),
                                   (7, 203, 192), (2, 1, 64), (9, 4099, 128), (16, 16384, 576)])
def test_gemm_skinny(hip, shape):
    """bfloat16 products with few rows: this package's kernel against a float64 product and the library."""
    M, N, K = shape
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(N, K, dtype=torch.bfloat16, seed=2)
    ref = x.double() @ w.double().T
    out = hip.linear(x, w, out_float32=True)
    assert out.dtype == torch.float32
    torch.testing.assert_close(out.double(), ref, rtol=1e-4, atol=1e-3 * math.sqrt(K / 64))
    out16 = hip.linear(x, w)
    assert out16.dtype == torch.bfloat16
    torch.testing.assert_close(out16.double(), ref, rtol=1e-2, atol=1e-2 * math.sqrt(K / 64))
    hip.use_skinny_gemm = False
    try:
        lib = hip.linear(x, w)
    finally:
        hip.use_skinny_gemm = True
    torch.testing.assert_close(out16.float(), lib.float(), rtol=2e-2, atol=2e-2 * math.sqrt(K / 64))
    # a row's result does not depend on the other rows
    assert torch.equal(hip.linear(x[:1].contiguous(), w), out16[:1])


@pytest.mark.parametrize("M", [1, 8, 9, 16])
@pytest.mark.parametrize("N, K", [(1, 64), (9, 128), (2048, 1984), (2049, 2112), (8192, 192), (33000, 64)])
def test_few_row_product_at_the_edges_of_its_tiles(hip, M, N, K):
    """Tiles of 8 rows (up to 8 rows of x have one, and so have blocks of at most 8 weight rows: N = 2,048), a last block
    that is short, half a chunk of k at the end, waves without a step, two blocks a workgroup (N = 33,000); and an input
    that starts inside another tensor, not at a multiple of 16 bytes.  Errors of the float sums: K products of values
    around 1, each rounded by 2^-24, in an order of the kernel's own: below 1e-6 K."""
    flat = rnd(M * K + 3, dtype=torch.bfloat16, seed=1)
    w = rnd(N, K, dtype=torch.bfloat16, seed=2)
    x = flat[:M * K].view(M, K)
    want = x.double() @ w.double().T
    out = hip.linear(x, w, out_float32=True)
    assert float((out.double() - want).abs().max()) <= 1e-6 * K
    aside = flat[3:3 + M * K].view(M, K)
    assert aside.data_ptr() % 16
    assert torch.equal(hip.linear(aside, w, out_float32=True), hip.linear(aside.clone(), w, out_float32=True))
    gated = hip.gated_linear(aside, torch.cat([w, w]))
    assert torch.equal(gated, hip.gated_linear(aside.clone(), torch.cat([w, w])))


@pytest.mark.parametrize("M", [1, 8, 9, 16])
@pytest.mark.parametrize("N", [9216, 11008, 12288, 12352, 14336, 18432])
def test_few_row_products_of_many_columns_are_cut_by_whole_rounds(hip, M, N):
    """A compute unit gets its share of the columns in at most two rounds of the workgroups that it holds at a time (by the
    rows alone it was five rounds of one workgroup of 10 for 12,352 columns), and at most a quarter more of them than that."""
    cut = (ctypes.c_int * 4)()
    for K in (1024, 3072, 4096):
        assert hip.core.sia_gemm_skinny_cut(M, N, K, cut) == 0
        blocks, height, grid, at_a_time = cut
        assert grid == -(-N // (blocks * height))
        units = torch.cuda.get_device_properties(0).multi_processor_count
        on_unit = -(-grid // units)
        assert -(-on_unit // at_a_time) <= 2, (K, list(cut))
        assert on_unit * blocks * height <= 1.25 * N / units, (K, list(cut))


@pytest.mark.parametrize("N, K", [(9217, 64), (9216, 1984), (12352, 3072), (16390, 512), (70001, 192)])
def test_few_row_products_of_four_blocks_a_workgroup(hip, N, K):
    """9 to 16 rows beside many columns take four blocks a workgroup; up to 8 rows never do.  A row's sums are the same bit for
    bit, in the plain product (short last workgroup and block, half a chunk of k at the end), with an activation and in groups."""
    x, w = rnd(16, K, dtype=torch.bfloat16, seed=1), rnd(N, K, dtype=torch.bfloat16, seed=2, scale=K ** -0.5)
    cut = (ctypes.c_int * 4)()
    halves = (x[:8].contiguous(), x[8:].contiguous())
    for M in (9, 11, 16):
        assert hip.core.sia_gemm_skinny_cut(M, N, K, cut) == 0 and cut[0] == 4
        some = x[:M].contiguous()
        for call in (lambda a: hip.linear(a, w, out_float32=True), lambda a: hip.linear(a, w),
                     lambda a: hip.activated_linear(a, w, "relu2")):
            assert torch.equal(call(some), torch.cat([call(h) for h in halves])[:M])
        rows = N // 3 - 5
        main, low = hip.grouped_linear(torch.stack([some, some.flip(0), 2 * some]), w, rows)
        assert torch.equal(main[0], hip.linear(some, w[:rows]))
        assert torch.equal(main[1], hip.linear(some.flip(0), w[rows:2 * rows]))
        assert torch.equal(low, hip.linear(2 * some, w[2 * rows:]))
    want = x.double() @ w.double().T    # K roundings of 2^-24 of a sum that stays below 8
    assert float((hip.linear(x, w, out_float32=True).double() - want).abs().max()) <= 5e-7 * K


@pytest.mark.parametrize("shape", [(1, 32, 64), (8, 8192, 3072), (16, 1008, 512), (5, 96, 320), (40, 128, 256),
                                   (3, 1, 64), (12, 333, 192), (16, 14336, 256)])
def test_gated_linear(hip, shape):
    """The product with the SwiGLU activation in its epilogue (few rows) or after it, against the twin."""
    M, inter, K = shape
    x = rnd(M, K, dtype=torch.bfloat16, seed=1)
    w = rnd(2 * inter, K, dtype=torch.bfloat16, seed=2, scale=1 / math.sqrt(K))
    gu = x.double() @ w.double().T
    ref = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
    out = hip.gated_linear(x, w)
    assert out.shape == (M, inter) and out.dtype == torch.bfloat16
    torch.testing.assert_close(out.double(), ref, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("heads, kv, D, K", [(3, 1, 32, 192), (24, 8, 128, 320), (32, 8, 64, 2048), (5, 5, 96, 3072)])
def test_products_of_17_to_64_rows(hip, M, heads, kv, D, K):
    """This package's products of more than 16 rows: a row's sums are those of a product of up to 16 rows, bit for bit, and
    the forms with an activation or with rotation and cache write give the bits of the plain product and the kernel behind
    it (runs of several tokens, pages that a run shares with the next).  The widths take one, two and four blocks of weight
    rows a workgroup and blocks of up to 8 and up to 16 rows, the lengths of k half a chunk at the end."""
    dtype, ps = torch.bfloat16, 16
    width = (heads + 2 * kv) * D
    x = rnd(M, K, dtype=dtype, seed=1)
    w = rnd(width, K, dtype=dtype, seed=2, scale=K ** -0.5)

    def own(w, out_float32=False):
        y = torch.empty((M, w.shape[0]), dtype=torch.float32 if out_float32 else dtype, device=DEV)
        assert hip.core.sia_gemm_skinny(x.data_ptr(), w.data_ptr(), y.data_ptr(), M, w.shape[0], K, int(out_float32),
                                        hip._stream()) == 0
        return y

    few = [x[i:i + 16].contiguous() for i in range(0, M, 16)]
    for tall in (w, rnd(16390, K, dtype=dtype, seed=3, scale=K ** -0.5)):
        assert torch.equal(own(tall), torch.cat([hip.linear(a, tall) for a in few]))
        assert torch.equal(own(tall, True), torch.cat([hip.linear(a, tall, out_float32=True) for a in few]))
    for inter in (width // 2, 8200):
        gate_up = rnd(2 * inter, K, dtype=dtype, seed=4, scale=K ** -0.5)
        assert torch.equal(hip.gated_linear(x, gate_up), hip.swiglu(own(gate_up)))

    lens = [M // 2, 1, M - M // 2 - 1]
    ctx = Ctx(lens, [n + past for n, past in zip(lens, (0, 37, 9))])
    pages = sum(-(-int(n) // ps) for n in ctx.kv_len.tolist()) + 2
    caches = [Cache(pages, kv, ps, D, dtype, ctx.kv_len.tolist(), seed=5) for _ in range(2)]
    ang = torch.outer(torch.arange(128, dtype=torch.float32), 1.0 / (10000.0 ** (torch.arange(0, D, 2, dtype=torch.float32) / D)))
    cos, sin = ang.cos().to(DEV), ang.sin().to(DEV)
    apart = own(w)
    hip.rope_kv_write(apart, heads, kv, D, D, cos, sin, ctx, caches[0])
    at_once, c = torch.empty_like(apart), caches[1]
    assert hip.core.sia_gemm_skinny_rope(
        x.data_ptr(), w.data_ptr(), at_once.data_ptr(), M, K, cos.data_ptr(), sin.data_ptr(), ctx.positions.data_ptr(),
        ctx.seq_of_token.data_ptr(), c.block_table.data_ptr(), c.block_table.shape[1], c.k_pages.data_ptr(),
        c.v_pages.data_ptr(), heads, kv, D, ps, None, 0, 0.0, hip._stream()) == 0
    assert torch.equal(apart[:, :heads * D], at_once[:, :heads * D])
    assert torch.equal(caches[0].k_pages, c.k_pages) and torch.equal(caches[0].v_pages, c.v_pages)


@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("inter, K, takes", [(1024, 2048, (17, 64)), (1024, 2112, (17, 32)), (1024, 5184, ()), (2560, 3072, (17, 64)),
                                             (2560, 5120, (17, 48)), (4607, 8192, ()), (4608, 8192, (17, 64)), (8704, 3072, (17, 64)),
                                             (8705, 3072, (17, 48)), (10241, 1088, (17, 32)), (10241, 2048, (17, 64))])
def test_gated_products_of_17_to_64_rows_go_where_they_are_made_faster(hip, M, inter, K, takes):
    """The few-row kernel with the activation inside, or product and activation: the same rows either way (the product
    rounds first in both; its sums' order may differ: a rounding of bfloat16 in gate and up and one of the result)."""
    own = bool(takes) and takes[0] <= M <= takes[1]
    assert bool(hip.core.sia_gemm_skinny_takes_swiglu(M, inter, K)) == own
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(2 * inter, K, dtype=torch.bfloat16, seed=2, scale=K ** -0.5)
    launched, real = [], hip.core.sia_gemm_skinny_swiglu
    hip.core.sia_gemm_skinny_swiglu = lambda *a: launched.append(1) or real(*a)
    try:
        out = hip.gated_linear(x, w)
    finally:
        hip.core.sia_gemm_skinny_swiglu = real
    assert bool(launched) == own
    gu = x.double() @ w.double().T
    ref = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
    bound = 2.0 ** -8 * (ref.abs() + gu[:, inter:].abs() * (gu[:, :inter].abs() * 1.1 + 1e-3) + gu[:, :inter].abs() * gu[:, inter:].abs()) + 1e-5
    assert bool(((out.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("M, inter, K, inside", [
    (65, 8192, 2048, False), (128, 8192, 2048, True), (512, 8192, 3072, True), (512, 8192, 3136, False), (128, 8192, 4096, False),
    (192, 8192, 4096, True), (256, 8192, 4096, True), (257, 8192, 4096, False), (256, 5120, 8192, True), (192, 2560, 4096, False),
    (512, 1024, 14336, False), (1024, 8192, 2048, True), (1025, 8192, 2048, False)])
def test_gated_tiles_are_taken_where_their_undivided_k_pays(hip, M, inter, K, inside):
    """The borders of the rule, and either way the same rows: three roundings of bfloat16 (gate, up, result) on top of sums of
    K products in any order."""
    assert bool(hip.core.sia_gemm_tiles_takes_swiglu(M, inter, K)) == inside
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(2 * inter, K, dtype=torch.bfloat16, seed=2, scale=K ** -0.5)
    launched, real = [], hip.core.sia_gemm_tiles_swiglu
    hip.core.sia_gemm_tiles_swiglu = lambda *a: launched.append(1) or real(*a)
    try:
        out = hip.gated_linear(x, w)
    finally:
        hip.core.sia_gemm_tiles_swiglu = real
    assert bool(launched) == inside
    gate, up = (x.float() @ w.float().T).double().split(inter, 1)
    ref = torch.nn.functional.silu(gate) * up
    bound = 2.0 ** -8 * (ref.abs() + up.abs() * (gate.abs() * 1.1 + 1e-3) + gate.abs() * up.abs()) + 1e-5
    assert bool(((out.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("M, N, K, route", [
    (16, 8192, 8192, "own"), (20, 8192, 8192, "own"), (21, 8192, 8192, "library"), (48, 8192, 4096, "own"), (49, 8192, 4096, "library"),
    (32, 20480, 1088, "own"), (32, 20484, 1088, "library"), (32, 20484, 2048, "own"), (33, 10240, 1088, "own"), (33, 10244, 1088, "library"),
    (20, 4096, 14336, "own"), (21, 4096, 14336, "tiles"), (32, 4096, 12288, "own"), (33, 4096, 12288, "tiles"),
    (33, 1024, 8192, "library"), (33, 1536, 6144, "tiles"), (33, 1532, 5184, "library"), (33, 1532, 5120, "own"), (33, 2560, 6208, "tiles"),
    (48, 1024, 4096, "own"), (49, 1536, 5120, "tiles"), (49, 1532, 4096, "own"), (49, 6144, 4096, "own"), (49, 6144, 5120, "library"),
    (64, 6140, 5120, "own"), (64, 5120, 8256, "library"), (64, 512, 11008, "tiles"), (64, 512, 9216, "library"),
    (33, 64, 11008, "tiles"), (33, 64, 10240, "library"), (21, 40, 14336, "tiles"), (20, 40, 14336, "own"), (300, 64, 65536, "tiles"),
    (80, 1536, 8192, "library"), (81, 1536, 8192, "tiles"), (80, 2048, 8192, "tiles"), (128, 1536, 6144, "library"), (256, 1024, 9216, "tiles"),
    (256, 2048, 4096, "library"), (257, 2048, 5120, "tiles"), (1024, 1024, 6144, "tiles"), (1025, 2048, 8192, "library"),
    (257, 2048, 4096, "library"), (65, 5120, 3072, "tiles"), (65, 5116, 3072, "library"), (160, 8192, 2048, "library"),
    (161, 8192, 2048, "tiles"), (128, 8192, 5120, "tiles"), (128, 8192, 8192, "library"), (129, 8192, 5120, "library"), (65, 8192, 8256, "tiles"),
    (256, 8196, 3072, "library"), (257, 5120, 3072, "library")])
def test_products_go_where_they_are_made_fastest(hip, M, N, K, route):
    """The borders of the rules by which a bfloat16 product goes to the few-row kernels, the tiles or the library, and its
    result on either side: K products of values around 1, below 1e-6 K, and a rounding of 2^-8 at most."""
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(N, K, dtype=torch.bfloat16, seed=2)
    names = {"sia_gemm_skinny": "own", "sia_gemm_tiles": "tiles"}
    real, went = {n: getattr(hip.core, n) for n in names}, []
    for n in names:
        setattr(hip.core, n, lambda *a, n=n: went.append(names[n]) or real[n](*a))
    try:
        out = hip.linear(x, w)
    finally:
        for n in names:
            setattr(hip.core, n, real[n])
    assert went == ([route] if route != "library" else [])
    want = (x.float() @ w.float().T).double()   # (in float32: another rounding of 1e-6 K at most)
    assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2e-6 * K).all())


@pytest.mark.parametrize("M", [21, 32, 33, 48, 64, 65, 96, 97, 128, 129, 200, 257, 300, 513])
@pytest.mark.parametrize("N, K", [(64, 64), (136, 320), (1032, 1088), (2048, 8192), (5120, 3072), (16384, 192)])
def test_tiles_of_a_product_of_many_rows(hip, M, N, K):
    """The tiles of products between the few-row kernels and the library: row blocks and column blocks that are short at
    the end, one slice of k and several, slices of unequal length, the gated form.  Errors of the float sums: K products
    of values around 1, below 1e-6 K, and a rounding to bfloat16 of the result (2^-8 of it at most)."""
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(N, K, dtype=torch.bfloat16, seed=2)
    want = x.double() @ w.double().T
    splits = hip.core.sia_gemm_tiles_splits(M, N, K)
    assert splits >= 1
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    slices = torch.full((splits, M, N), float("nan"), device=DEV)
    assert hip.core.sia_gemm_tiles(x.data_ptr(), w.data_ptr(), y.data_ptr(), slices.data_ptr(), M, N, K, hip._stream()) == 0
    if splits > 1:
        assert float((slices.double().sum(0) - want).abs().max()) <= 1e-6 * K
        hip.sum_slices(slices, splits, y)
    assert bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-6 * K).all())
    gated = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert hip.core.sia_gemm_tiles_swiglu(x.data_ptr(), w.data_ptr(), gated.data_ptr(), M, N // 2, K, hip._stream()) == 0
    ref = torch.nn.functional.silu(want[:, :N // 2]) * want[:, N // 2:]
    scale = K ** 0.5        # of a gate or an up value; three roundings of 2^-9 each, the activation's slope below 1.1
    assert bool(((gated.double() - ref).abs() <= 2.0 ** -7 * ref.abs() + 2.0 ** -8 * scale * (want[:, N // 2:].abs() + scale)).all())


@pytest.mark.parametrize("M, N, K, gated", [(511, 16384, 2048, True), (821, 16384, 2048, True), (1023, 16384, 3072, True),
                                            (1024, 16384, 3072, True), (450, 3072, 8192, False), (769, 3072, 8192, False),
                                            (1023, 4096, 14336, False), (600, 4096, 14336, False)])
def test_the_largest_tiles_over_long_k(hip, M, N, K, gated):
    """Tiles of 128 x 256 and 256 x 256 through many rounds of their shallow rings, the gated form in one slice and the plain
    one in several, rows that are no multiple of a tile.  Bounds as below (values around 1 in K products)."""
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(N, K, dtype=torch.bfloat16, seed=2, scale=K ** -0.5)
    want = x.double() @ w.double().T
    if gated:
        out = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device=DEV)
        assert hip.core.sia_gemm_tiles_swiglu(x.data_ptr(), w.data_ptr(), out.data_ptr(), M, N // 2, K, hip._stream()) == 0
        gate, up = want.split(N // 2, 1)
        ref = torch.nn.functional.silu(gate) * up
        bound = 2.0 ** -8 * (ref.abs() + up.abs() * (gate.abs() * 1.1 + 1e-3) + gate.abs() * up.abs()) + 1e-5
        assert bool(((out.double() - ref).abs() <= bound).all())
        return
    splits = hip.core.sia_gemm_tiles_splits(M, N, K)
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    slices = torch.full((splits, M, N), float("nan"), device=DEV)
    assert hip.core.sia_gemm_tiles(x.data_ptr(), w.data_ptr(), out.data_ptr(), slices.data_ptr(), M, N, K, hip._stream()) == 0
    if splits > 1:      # K roundings of 2^-24 of a sum that stays below 8
        assert float((slices.double().sum(0) - want).abs().max()) <= 5e-7 * K
        hip.sum_slices(slices, splits, out)
    assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 5e-7 * K).all())


@pytest.mark.parametrize("M", [17, 32, 33, 64, 65, 128])
@pytest.mark.parametrize("N, K", [(32768, 64), (32900, 192), (40004, 1088)])
def test_tiles_of_an_output_head(hip, M, N, K):
    """Float results of whole k in each of the three shapes, the last columns' tile short; errors as above."""
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(N, K, dtype=torch.bfloat16, seed=2)
    assert hip.core.sia_gemm_tiles_takes_head(M, N, K)
    y = hip.linear(x, w, out_float32=True)
    assert y.dtype == torch.float32
    assert float((y.double() - x.double() @ w.double().T).abs().max()) <= 1e-6 * K


@pytest.mark.parametrize("M, hidden, splits", [(1, 8, 2), (65, 64, 1), (70, 2048, 3), (128, 3080, 16), (300, 8192, 5)])
def test_the_norm_that_adds_a_product_s_slices(hip, M, hidden, splits):
    """The same bits as the slices' sum and the norm behind it in launches of their own."""
    slices = rnd(splits, M, hidden, seed=1)
    res, gain = rnd(M, hidden, seed=2, scale=3.0), rnd(hidden, seed=3) + 1.0
    delta = hip.sum_slices(slices, splits, torch.empty((M, hidden), dtype=torch.bfloat16, device=DEV))
    a, b = res.clone(), res.clone()
    want = hip.add_rmsnorm(a, delta, gain, 1e-5, torch.bfloat16)
    got = torch.empty_like(want)
    assert hip.core.sia_add_rmsnorm_slices(b.data_ptr(), slices.data_ptr(), splits, gain.data_ptr(), got.data_ptr(), M, hidden,
                                           1e-5, hip._stream()) == 0
    assert torch.equal(a, b) and torch.equal(got, want)


@pytest.mark.parametrize("rows", [1, 8, 9, 16])
@pytest.mark.parametrize("N, K", [(64, 64), (1000, 1984), (4100, 3136), (9216, 320)])
def test_few_row_products_of_weights_that_begin_anywhere(hip, rows, N, K):
    """A weight inside another tensor is read where it lies, with the bits of a copy that begins at a multiple of 16 bytes: in
    the plain product, with an activation or a gate, in groups, into the residual, with rotation and cache write."""
    from simple_inference_amd.kernels import PendingProduct
    flat = rnd(N * K + 5, dtype=torch.bfloat16, seed=2, scale=K ** -0.5)
    w = flat[5:].view(N, K)
    assert w.data_ptr() % 16
    copy, x = w.clone(), rnd(rows, K, dtype=torch.bfloat16, seed=1)
    y = torch.empty(rows, N, dtype=torch.bfloat16, device=DEV)
    assert hip.core.sia_gemm_skinny(x.data_ptr(), w.data_ptr(), y.data_ptr(), rows, N, K, 0, hip._stream()) == 0
    assert torch.equal(y, hip.linear(x, copy))
    many = torch.stack([x, x.flip(0), -x])
    gain, residual = (rnd(N, seed=3) + 1.0).contiguous(), rnd(rows, N, seed=4)

    def into_residual(w):
        r = residual.clone()
        scaled = hip.linear_into_residual(PendingProduct(x, w, hip), r, gain, 1e-5)
        return r, scaled.rows, scaled.partials[:, :rows]

    for call in (lambda w: [hip.linear(x, w, out_float32=True)], lambda w: [hip.activated_linear(x, w, "gelu_tanh")],
                 lambda w: [hip.gated_linear(x, w)],
                 lambda w: hip.grouped_linear(many, w, N // 3), into_residual):
        assert all(torch.equal(a, b) for a, b in zip(call(w), call(copy)))
    if N in (64, 9216):
        heads, kv, D = {64: (2, 1, 16), 9216: (24, 24, 128)}[N]
        ctx = Ctx([1] * rows, [7 + i for i in range(rows)])
        ang = torch.outer(torch.arange(64, dtype=torch.float32), 1.0 / (10000.0 ** (torch.arange(0, D, 2, dtype=torch.float32) / D)))
        outs = []
        for weight in (w, copy):
            cache = Cache(2 * rows + 1, kv, 16, D, torch.bfloat16, ctx.kv_len.tolist(), seed=6)
            outs.append((hip.qkv_to_cache(x, weight, heads, kv, D, D, ang.cos().to(DEV), ang.sin().to(DEV), ctx, cache)[:, :heads * D],
                         cache.k_pages, cache.v_pages))
        assert all(torch.equal(a, b) for a, b in zip(*outs))


@pytest.mark.parametrize("rows", [17, 40, 64, 100, 300])
def test_products_of_more_rows_of_weights_that_begin_anywhere_are_the_library_s(hip, rows):
    """Neither copied nor given to kernels that bring whole pieces to LDS: one product by the library, where it lies."""
    N, K = 2048, 8192
    flat = rnd(N * K + 5, dtype=torch.bfloat16, seed=2, scale=K ** -0.5)
    w, x = flat[5:].view(N, K), rnd(rows, K, dtype=torch.bfloat16, seed=1)
    went, real = [], {n: getattr(hip.core, n) for n in ("sia_gemm_skinny", "sia_gemm_tiles", "sia_gemm_skinny_swiglu", "sia_gemm_tiles_swiglu")}
    for n in real:
        setattr(hip.core, n, lambda *a, n=n: went.append(n) or real[n](*a))
    try:
        out, gated = hip.linear(x, w), hip.gated_linear(x, w)
    finally:
        for n in real:
            setattr(hip.core, n, real[n])
    assert not went
    assert torch.equal(out, hip._library_product(x, w, False))
    want = x.double() @ w.double().T    # K roundings of 2^-24 of a sum that stays below 8, and one to bfloat16
    assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 5e-7 * K).all())
    assert torch.equal(gated, hip.swiglu(out))


@pytest.mark.parametrize("dtype", DTYPES)
def test_a_residual_read_itself_takes_a_product_left_in_slices(hip, dtype):
    """``ResidualStream.lower`` behind a block that left its last product in slices: as behind one that left the rows."""
    from simple_inference_amd.kernels import SlicedProduct
    from simple_inference_amd.parts.context import ResidualStream
    slices, residual = rnd(3, 70, 64, seed=1), rnd(70, 64, seed=2)
    out = torch.empty(70, 64, dtype=torch.bfloat16, device=DEV)
    ways = []
    for delta in (SlicedProduct(slices, 3, out, hip), hip.sum_slices(slices, 3, torch.empty_like(out))):
        stream = ResidualStream(residual.clone(), delta)
        if dtype == torch.float32:
            stream.settle(hip)
        ways.append((stream.lower(hip, dtype), stream.residual))
    assert all(torch.equal(a, b) for a, b in zip(*ways))


@pytest.mark.parametrize("shape", [(17, 3072, 3072), (512, 5120, 3072), (2048, 16384, 3072), (130, 3072, 8192),
                                   (33, 1008, 200), (64, 320, 96)])
def test_library_product_called_directly(hip, shape):
    """Products of many rows go to the BLAS library without a tensor library between: same results as through torch
    (it is the same library), against a float64 product, bfloat16 and float results, again on a second call (the
    kept algorithm)."""
    M, N, K = shape
    assert hip.blas is not None, "the direct way to the BLAS library was not built or did not initialise"
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(N, K, dtype=torch.bfloat16, seed=2)
    ref = x.double() @ w.double().T
    for _ in range(2):
        out = hip.linear(x, w)
        assert out.dtype == torch.bfloat16
        torch.testing.assert_close(out.double(), ref, rtol=1e-2, atol=1e-2 * math.sqrt(K / 64))
        torch.testing.assert_close(out.float(), torch.mm(x, w.t()).float(), rtol=2e-2, atol=2e-2 * math.sqrt(K / 64))
        wide = hip.linear(x, w, out_float32=True)
        assert wide.dtype == torch.float32
        torch.testing.assert_close(wide.double(), ref, rtol=1e-2, atol=1e-2 * math.sqrt(K / 64))


@pytest.mark.parametrize("shape", [(64, 3072, 3072), (33, 1008, 200), (256, 320, 512), (300, 128, 64)])
def test_library_product_with_candidates_tried_out(hip, shape):
    """Inside ``recurring_shapes`` the library's candidate algorithms are timed on the call's own operands and one is
    kept: the product is right on that call and on those after it, inside and outside, also for a shape that had an
    algorithm before."""
    M, N, K = shape
    assert hip.blas is not None
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=3), rnd(N, K, dtype=torch.bfloat16, seed=4)
    ref = x.double() @ w.double().T
    outs = [hip.linear(x, w)]
    with hip.recurring_shapes():
        outs += [hip.linear(x, w), hip.linear(x, w, out_float32=True)]
    outs += [hip.linear(x, w)]
    for out in outs:
        torch.testing.assert_close(out.double(), ref, rtol=1e-2, atol=1e-2 * math.sqrt(K / 64))
    assert torch.equal(outs[1], outs[3])   # the kept algorithm is used from then on


@pytest.mark.parametrize("bits", [8, 24])
@pytest.mark.parametrize("N, K", [(1, 4), (15, 31), (97, 129), (1000, 333), (520, 1056), (3072, 260), (8200, 2048), (12290, 192), (33000, 40)])
def test_float32_products_of_parts(hip, N, K, bits):
    """Few rows and tiles, whole k and slices, empty slices too, short last chunks, tiles and columns, rows on 16 bytes or not, against 64 bits,
    weights of one part and of three, one row of three parts among others of one; a row has the same bits whatever
    rows are beside it.  A chunk's sum is at most 192 roundings of 2^-24 of sums below sum |x w|, the chunks' and slices' sums
    K / 32 + 8 more, and what is left out of the parts' products 2^-32 of each.  (Far from what the products give; the next test's bound is near.)"""
    w = rnd(N, K, seed=2)
    if bits == 8:
        w = w.bfloat16().float()
        w[N // 2] = rnd(K, seed=3)
    x = rnd(700, K, seed=1)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    all_rows = hip.linear(x, w)
    assert bool(((all_rows.double() - want).abs() <= (201 + K / 32) * 2.0 ** -24 * size + 1e-30).all())
    for M in (1, 8, 9, 16, 17, 32, 33, 64, 65, 130, 303):
        assert torch.equal(hip.linear(x[700 - M:].contiguous(), w), all_rows[700 - M:]), M
    few = torch.empty(33, N, device=DEV)      # without a workspace: the few-row kernel
    assert hip.core.sia_gemm_f32(x.data_ptr(), w.data_ptr(), few.data_ptr(), None, 33, N, K, hip._stream()) == 0
    assert torch.equal(few, all_rows[:33])
    flat = torch.empty(N * K + 1, device=DEV)
    flat[1:] = w.flatten()
    for M in (5, 40, 303):
        assert torch.equal(hip.linear(x[:M].contiguous(), flat[1:].view(N, K)), all_rows[:M]), M


# (rows, columns, k, way):  2 * shape of the tiles + 1 where slices of k are apart, or blocks of rows and columns of the few-row kernel.  Each way of
# the tiles with one slice, two and eight where there are some, k that is a multiple of four and not; last tiles and chunks in part.
FLOAT_WAYS = [
    (65, 32770, 2052, 0), (259, 20002, 2052, 0), (65, 20002, 1028, 1), (259, 2050, 2052, 1),
    (303, 32770, 260, 2), (40, 32770, 1027, 2), (259, 12290, 260, 2), (193, 14337, 131, 2), (385, 8195, 260, 2), (385, 8195, 131, 2),
    (303, 16385, 2052, 3), (40, 16385, 2049, 3), (193, 3074, 2052, 3), (65, 4100, 1027, 3),
    (97, 14337, 1028, 4), (97, 12290, 261, 4), (385, 4100, 260, 4), (385, 4100, 131, 4), (33, 12290, 1027, 5), (40, 3074, 2049, 5),
    (193, 12290, 64, 6), (17, 12290, 63, 6), (65, 14337, 516, 6), (700, 2050, 260, 6), (259, 2050, 131, 6),
    (193, 14337, 516, 8), (97, 16385, 517, 8), (513, 4100, 516, 8), (513, 4100, 517, 8), (65, 12290, 2052, 9), (65, 2050, 2049, 9),
    (8, 32800, 256, -14), (12, 32800, 256, -11), (12, 14337, 131, -11), (5, 130, 260, -11), (20, 32800, 256, -24), (40, 14337, 132, -42),
    (17, 12290, 132, -22), (17, 12290, 131, -22), (33, 8195, 132, -22), (40, 130, 260, -21), (40, 130, 261, -21)]


def test_the_ways_of_float32_products_are_all_tested():
    """Way 7 is never taken: tiles of 32 x 64 have no slices apart."""
    assert {way for *_, way in FLOAT_WAYS} == set(range(10)) - {7} | {-11, -14, -21, -22, -24, -42}


@pytest.mark.parametrize("M, N, K, way", FLOAT_WAYS)
def test_float32_products_every_way(hip, M, N, K, way):
    """The bits of the few-row kernel without a workspace, with weights of one part, of three and of both; a 2-norm error against 64 bits of at most
    2e-7 (measured up to 9e-8; any of the products above 2^-24 of the whole left out gives 1e-6 and more); rows and columns that
    are not finite or have no three parts made again like the floats' product, in the last rows and columns too."""
    assert hip.core.sia_gemm_f32_way(None, None, M, N, K) == way
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    few = torch.empty(M, N, device=DEV)

    def same_as_few(x, w):
        y = hip.linear(x, w)
        assert hip.core.sia_gemm_f32(x.data_ptr(), w.data_ptr(), few.data_ptr(), None, M, N, K, hip._stream()) == 0
        assert torch.equal(torch.nan_to_num(y, nan=1.5), torch.nan_to_num(few, nan=1.5))
        return y

    for mixed in (False, True):
        if mixed:
            w[N // 3:] = w[N // 3:].bfloat16().float()
        y, want = same_as_few(x, w), x.double() @ w.double().T
        assert float((y.double() - want).norm() / want.norm()) <= 2e-7
    x[M - 1, 0], x[M // 2] = float("nan"), x[M // 2] * 2.0 ** -125
    w[N - 1, K - 1], w[N // 2, 0], w[N // 4] = float("inf"), 3.3999e38, w[N // 4] * 2.0 ** -120
    y, want = same_as_few(x, w), x.double() @ w.double().T
    assert torch.equal(y.isnan(), want.isnan()) and bool(y[:M - 1, N - 1].isinf().all())
    there = want.abs() < 1e38
    size = torch.nan_to_num(x.double(), nan=0.0).abs() @ torch.nan_to_num(w.double(), posinf=0.0).abs().T
    assert bool(((y.double() - want).abs() <= (24 + K / 4) * 2.0 ** -24 * size + K * 2.0 ** -149)[there].all())


# Tiles of 160 rows:  whole k and slices of 2 and 8, rows behind a tile and last tiles in part, columns that are no multiple of 4.
TALL_FLOAT_WAYS = [(129, 28674, 128, 10), (160, 50003, 224, 10), (259, 14337, 128, 10), (145, 14337, 768, 11), (129, 12290, 1024, 11), (160, 14337, 1024, 11),
                   (129, 32770, 224, 12), (150, 40961, 160, 12), (311, 2050, 2048, 13), (129, 5123, 1536, 13), (606, 16386, 1536, 13)]


@pytest.mark.parametrize("M, N, K, way", [(303, 14337, 1536, 11), (150, 40961, 160, 12), (311, 2050, 2048, 13)])
def test_tall_tiles_whose_waves_find_weights_of_24_bits_at_different_chunks(hip, M, N, K, way):
    """Weights are bfloat16 numbers but for some from a chunk on, another for each of some rows: waves of a workgroup go on with all parts of the weights from
    different chunks, with their sums and places in the rings.  A value under 2^-110 in a late chunk among them.  The few-row kernel's bits."""
    assert hip.core.sia_gemm_f32_way(None, None, M, N, K) == way
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2).bfloat16().float()
    whole = rnd(N, K, seed=3)
    chunks = K // 32
    for row, chunk in ((0, 0), (17, 1), (40, chunks // 2), (50, chunks // 2 + 1), (100, chunks - 1), (131, 3), (N // 2, chunks // 3), (N - 1, chunks - 1)):
        w[row, 32 * chunk:] = whole[row, 32 * chunk:]
    few = torch.empty(M, N, device=DEV)
    for small in (False, True):
        if small:
            w[70, K - 5], w[N // 3, K - 33] = 2.0 ** -120 * 1.2345678, 2.0 ** -115 * 1.2345678
        y = hip.linear(x, w)
        assert hip.core.sia_gemm_f32(x.data_ptr(), w.data_ptr(), few.data_ptr(), None, M, N, K, hip._stream()) == 0
        assert torch.equal(y, few)
        want = x.double() @ w.double().T
        assert float((y.double() - want).norm() / want.norm()) <= 2e-7


# The tall tiles take products of a float32 model's steps, and none that the smaller tiles or the few-row kernel take as long or less for:  us, theirs and the
# tall ones', weights of 8 bits:  768 x 12,288 x 3,072 263 and 327;  1,280 x 8,192 x 4,096 366 and 446;  640 x 1,024 x 1,536 21.4 and 26.1;  160 x 3,072 x
# 2,048 24.3 and 26.1;  303 x 128,256 x 2,048 691 and 594.
@pytest.mark.parametrize("M, N, K, way", [
    (303, 128256, 2048, 12), (303, 16384, 2048, 11), (303, 3072, 2048, 13), (303, 2048, 8192, 11), (303, 2048, 2048, 11),
    (768, 12288, 3072, 2), (1280, 8192, 4096, 2), (640, 1024, 1536, -21), (129, 3072, 2048, -21), (160, 3072, 2048, -21),
    (1024, 6144, 4096, 2), (256, 2048, 2048, 3)])
def test_tall_tiles_take_the_float32_products_that_they_are_the_faster_for(hip, M, N, K, way):
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    assert hip.core.sia_gemm_f32_way(None, None, M, N, K) == way


@pytest.mark.parametrize("M, N, K, way", TALL_FLOAT_WAYS)
def test_float32_products_in_tall_tiles(hip, M, N, K, way):
    """As every other way: the few-row kernel's bits, and its bound against 64 bits."""
    test_float32_products_every_way(hip, M, N, K, way)


@pytest.mark.parametrize("N, K", [(7, 1), (130, 35), (2050, 1056), (1000, 334), (16388, 2047), (33000, 258)])
def test_float32_products_of_rows_that_begin_anywhere(hip, N, K):
    """Either operand, or both, one to three floats behind a multiple of 16 bytes, rows of any length: the bits of operands that are not, and a
    last k whose neighbours in W are not finite.  Nothing is copied for it: W does not count in the workspace, whatever its size."""
    x, w = rnd(303, K, seed=1), rnd(N, K, seed=2)
    want = x.double() @ w.double().T
    want32 = hip.linear(x, w)
    assert bool(((want32.double() - want).abs() <= (24 + K / 4) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 1e-30).all())

    def shifted(t, by):
        flat = torch.full((t.numel() + 8,), float("nan"), device=DEV)
        flat[by:by + t.numel()] = t.flatten()
        return flat[by:by + t.numel()].view(t.shape)

    for M in (1, 8, 9, 17, 40, 130, 303):
        for bx, bw in ((1, 0), (0, 2), (3, 1), (2, 2)):
            assert torch.equal(hip.linear(shifted(x[:M], bx), shifted(w, bw)), want32[:M]), (M, bx, bw)
    assert 0 < hip.core.sia_gemm_f32_workspace(x.data_ptr(), w.data_ptr() + 4, 303, 40000, 2049) < 40000 * 2049


@pytest.mark.parametrize("M, N, K", [(3, 96, 64), (40, 520, 333), (100, 2048, 512), (70, 40000, 64), (40, 12800, 256)])
def test_float32_products_that_are_not_finite(hip, M, N, K):
    """Infinities, NaN, products of an infinity with zero and the largest finite numbers give what floats give."""
    largest = torch.finfo(torch.float32).max
    for where, value in (("x", float("inf")), ("x", float("nan")), ("w", float("-inf")), ("x", largest), ("w", largest)):
        for bits in (8, 24):
            x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
            if bits == 8:
                w = w.bfloat16().float()
            if abs(value) == largest:
                x[:, 1:], w[:, 1:] = 0.0, 0.0
                x[:, 0], w[:, 0] = 1.0, 1.0
            (x if where == "x" else w)[1, 0] = value
            w[2, 0] = 0.0
            want, got = (x.double() @ w.double().T).float(), hip.linear(x, w)
            assert torch.equal(torch.isnan(want), torch.isnan(got)) and torch.equal(torch.isinf(want), torch.isinf(got))
            odd = ~torch.isfinite(want) & ~torch.isnan(want) | (want.abs() == largest)
            assert torch.equal(want[odd], got[odd])


@pytest.mark.parametrize("M, N, K", [(1, 33000, 2048), (40, 12800, 2048), (303, 16384, 2048), (303, 2048, 2048), (303, 33000, 1024)])
def test_float32_products_that_are_not_finite_keep_a_step_s_pace(hip, M, N, K):
    """A row of NaN is made again by whole blocks: eight times the product's own time is far from one thread after the other's walks (12 to
    90 times) and from what it takes (under four).  What is made again has the same bits whoever makes it."""
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    huge = x.clone()
    huge[M // 2, 5::7] = 3.3999e38      # rounds to an infinite part: the floats' product, finite
    some = w * 1e-30
    got = hip.linear(huge, some)
    assert bool(torch.isfinite(got).all()) and torch.equal(got[M // 2:M // 2 + 1], hip.linear(huge[M // 2:M // 2 + 1], some))
    want, size = huge.double() @ some.double().T, huge.double().abs() @ some.double().abs().T
    assert bool(((got.double() - want).abs() <= (24 + K / 4) * 2.0 ** -24 * size).all())

    def us(x):
        times = []
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            a.record()
            hip.linear(x, w)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b) * 1e3)
        return min(times)

    plain = us(x)
    x[M // 2, 3] = float("nan")
    odd = us(x)
    assert bool(torch.isnan(hip.linear(x, w)[M // 2]).all())
    assert odd <= 8 * plain + 20, (odd, plain)


@pytest.mark.parametrize("M, N, K", [(3, 96, 64), (40, 520, 333), (100, 2048, 512), (303, 2050, 2048), (70, 40000, 64)])
def test_float32_products_of_small_numbers(hip, M, N, K):
    """Operands whose last bits lie below what bfloat16 holds, rows and columns of them among others, keep all their bits: a row's or column's
    sums are then those of floats, at most K / 4 + 24 roundings, and others' as ever (tested above).  Results below 2^-126 are known to
    a rounding of their own unit a term."""
    for sx, sw, bits in ((-112, 0, 8), (-120, 0, 24), (-126, 30, 24), (0, -115, 24), (-60, -60, 24), (-137, 8, 8), (0, -130, 8), (-70, -70, 24)):
        x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
        if bits == 8:
            w = w.bfloat16().float()
        x[::2] *= 2.0 ** sx
        w[1::2] *= 2.0 ** sw
        want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
        assert bool(((hip.linear(x, w).double() - want).abs() <= (24 + K / 4) * 2.0 ** -24 * size + K * 2.0 ** -149).all()), (sx, sw, bits)
    # two operands whose only large product is of a small number
    x, w = torch.zeros(M, K, device=DEV), torch.zeros(N, K, device=DEV)
    x[:, 0], x[:, 1], w[:, 0], w[:, 1] = 1.0, rnd(M, seed=3) * 2.0 ** -120, rnd(N, seed=4) * 2.0 ** -120, 1.0
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    assert bool(((hip.linear(x, w).double() - want).abs() <= 4 * 2.0 ** -24 * size).all())


@pytest.mark.parametrize("bits", [8, 24])
@pytest.mark.parametrize("M, N, K", [(8, 2050, 1), (303, 2048, 2048), (100, 300, 70), (40, 40000, 64), (300, 16388, 512)])
def test_float32_results_of_one_product_are_rounded_once(hip, M, N, K, bits):
    """One product a result, among zeros: the rounding to float (2^-24), and what the products of the smallest parts leave (2^-31)."""
    x, w = torch.zeros(M, K, device=DEV), rnd(N, K, seed=2)
    if bits == 8:
        w = w.bfloat16().float()
    x[:, K // 3] = rnd(M, seed=1)
    want = x[:, K // 3:K // 3 + 1].double() @ w[:, K // 3:K // 3 + 1].double().T
    error = ((hip.linear(x, w).double() - want).abs() / want.abs()).max()
    assert float(error) <= 2.0 ** -24 + 2.0 ** -31, float(error) * 2.0 ** 24


def test_float32_product_has_no_reduced_precision(hip):
    """An operand bit below bfloat16 (8 bits) and tf32 (10 bits) resolution must reach the product."""
    K = 8
    x = torch.ones(1, K, device=DEV)
    w = torch.ones(2, K, device=DEV)
    w[1, 3] += 2.0 ** -12
    y = hip.linear(x, w)
    assert y.dtype == torch.float32
    assert y[0, 0].item() == 8.0
    assert y[0, 1].item() - 8.0 == 2.0 ** -12


# edges of blocks of 16 rows and columns, of tiles and of chunks of 32 k; the one of 50 rows is misaligned.  Most go to the few-row
# kernel, (300, 16500), (129, 8320) and (303, 3070) to tiles; test_float32_products_every_way reaches all of either
@pytest.mark.parametrize("shape", [(1, 1, 1), (16, 17, 4), (17, 16, 60), (33, 33, 64), (64, 63, 68), (65, 130, 130), (40, 4100, 80),
                                   (129, 8320, 192), (300, 16500, 76), (50, 257, 128), (303, 3070, 76), (64, 16383, 66)])
def test_float32_product(hip, shape):
    """Against float64: a result is the sum of K / 32 chunks, each cut by the matrix cores (2^-23 of it) and rounded when it is added, and of small
    products with a sum of their own, 2^-8 of that, so it errs by less than (K / 4 + 8) times 2^-24 of the sum of the products' sizes; and
    whichever kernel a number of rows goes to, a row's bits are the same."""
    M, N, K = shape
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    if shape[0] == 50:
        x = rnd(M * K + 1, seed=1)[1:].view(M, K)
    y = hip.linear(x, w)
    wide = x.double().abs() @ w.double().abs().T
    assert ((y.double() - x.double() @ w.double().T).abs() <= 2.0 ** -24 * (K / 4 + 8) * wide).all()
    for rows in (1, 16, 17, 48):
        if rows < M:
            assert torch.equal(hip.linear(x[:rows].contiguous(), w), y[:rows]), rows


def test_linear_rows_do_not_depend_on_the_batch(hip):
    x, w = rnd(67, 300, seed=1), rnd(130, 300, seed=2)
    whole = hip.linear(x, w)
    assert torch.equal(whole[13:14], hip.linear(x[13:14].contiguous(), w))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("geom", [
    # heads, kv heads, head_dim, rotary_dim, page_size
    (4, 2, 16, 16, 4), (3, 1, 32, 32, 8), (6, 3, 80, 80, 16), (8, 8, 128, 64, 32), (2, 1, 256, 256, 64),
    (5, 5, 48, 0, 2),
])
def test_rope_kv_write_and_attention(hip, dtype, geom):
    n_heads, n_kv, D, rd, ps = geom
    q_lens, kv_lens = [1, 7, 64, 3], [130, 7, 64 + 37, 66]
    ctx = Ctx(q_lens, kv_lens)
    pages = sum(-(-kv // ps) for kv in kv_lens) + 3
    c_hip = Cache(pages, n_kv, ps, D, dtype, kv_lens, seed=4)
    c_twin = Cache(pages, n_kv, ps, D, dtype, kv_lens, seed=4)
    # earlier tokens' keys and values already in the pages (same in both)
    c_hip.k_pages.copy_(rnd(*c_hip.k_pages.shape, dtype=dtype, seed=5)); c_twin.k_pages.copy_(c_hip.k_pages)
    c_hip.v_pages.copy_(rnd(*c_hip.v_pages.shape, dtype=dtype, seed=6)); c_twin.v_pages.copy_(c_hip.v_pages)
    qkv = rnd(ctx.n_tokens, (n_heads + 2 * n_kv) * D, dtype=dtype, seed=7)
    q1, q2 = qkv.clone(), qkv.clone()
    pos = torch.arange(256, dtype=torch.float32)
    inv = 1.0 / (10000.0 ** (torch.arange(0, max(rd, 2), 2, dtype=torch.float32) / max(rd, 2)))
    ang = torch.outer(pos, inv)
    cos, sin = ang.cos().to(DEV), ang.sin().to(DEV)
    hip.rope_kv_write(q1, n_heads, n_kv, D, rd, cos, sin, ctx, c_hip)
    twin.rope_kv_write(q2, n_heads, n_kv, D, rd, cos, sin, ctx, c_twin)
    torch.testing.assert_close(q1.float(), q2.float(), **tol(dtype))
    torch.testing.assert_close(c_hip.k_pages.float(), c_twin.k_pages.float(), **tol(dtype))
    assert torch.equal(c_hip.v_pages, c_twin.v_pages)
    for window in (None, 19):
        out = hip.paged_attention(q2, n_heads, n_kv, D, 1 / math.sqrt(D), window, ctx, c_twin)
        ref = twin.paged_attention(q2, n_heads, n_kv, D, 1 / math.sqrt(D), window, ctx, c_twin)
        torch.testing.assert_close(out.float(), ref.float(), **tol(dtype))


@pytest.mark.parametrize("geom", [(24, 8, 128, 128, 16), (5, 1, 48, 32, 8), (3, 3, 12, 8, 4), (4, 2, 64, 64, 16)])
@pytest.mark.parametrize("tokens", [3, 130])
def test_the_rotation_s_rounding(hip, geom, tokens):
    """A rotated pair is fma(a, c, -(b s)) and fma(b, c, a s), bit for bit: what prompts and decoded tokens of any step get,
    so that their outputs stay what they were.  Inputs of 8 bits make the fused products exact in 64 bits."""
    n_heads, n_kv, D, rot, ps = geom
    ctx = Ctx([tokens], [tokens + 100])
    x = rnd(tokens, (n_heads + 2 * n_kv) * D, dtype=torch.bfloat16, seed=1).float()
    ang = torch.outer(torch.arange(tokens + 100, dtype=torch.float32), 1.0 / (10000.0 ** (torch.arange(0, rot, 2, dtype=torch.float32) / rot)))
    cos, sin = ang.cos().to(DEV), ang.sin().to(DEV)
    cache = Cache(-(-(tokens + 100) // ps) + 1, n_kv, ps, D, torch.float32, [tokens + 100])
    out = x.clone()
    hip.rope_kv_write(out, n_heads, n_kv, D, rot, cos, sin, ctx, cache)
    heads = x[:, :n_heads * D].view(tokens, n_heads, D)
    a, b = heads[..., :rot // 2], heads[..., rot // 2:rot]
    c, s = (t[ctx.positions.long()][:, None] for t in (cos, sin))
    want = torch.cat([(a.double() * c.double() - (b * s).double()).float(), (b.double() * c.double() + (a * s).double()).float(),
                      heads[..., rot:]], -1)
    assert torch.equal(out[:, :n_heads * D].view(tokens, n_heads, D), want)
    keys = x[:, n_heads * D:(n_heads + n_kv) * D].view(tokens, n_kv, D)
    a, b = keys[..., :rot // 2], keys[..., rot // 2:rot]
    want = torch.cat([(a.double() * c.double() - (b * s).double()).float(), (b.double() * c.double() + (a * s).double()).float(),
                      keys[..., rot:]], -1)
    for t, pos in enumerate(ctx.positions.tolist()):
        page = int(cache.block_table[0, pos // ps])
        assert torch.equal(cache.k_pages[page, :, pos % ps], want[t])


@pytest.mark.parametrize("geom", [(24, 8, 128, 128, 16), (5, 1, 48, 32, 8), (3, 3, 64, 64, 4)])
def test_rope_kv_write_of_a_long_step(hip, geom):
    """More than a thousand tokens in one step (the kernel then gives a thread several items): two prompt portions,
    one from the start of its sequence and one that begins in the middle of a page, and a single decoded token."""
    n_heads, n_kv, D, rd, ps = geom
    q_lens, kv_lens = [1, 700, 450], [77, 700, 450 + 21]
    ctx = Ctx(q_lens, kv_lens)
    pages = sum(-(-kv // ps) for kv in kv_lens) + 2
    c_hip = Cache(pages, n_kv, ps, D, torch.bfloat16, kv_lens, seed=14)
    c_twin = Cache(pages, n_kv, ps, D, torch.bfloat16, kv_lens, seed=14)
    c_hip.k_pages.copy_(rnd(*c_hip.k_pages.shape, dtype=torch.bfloat16, seed=15)); c_twin.k_pages.copy_(c_hip.k_pages)
    c_hip.v_pages.copy_(rnd(*c_hip.v_pages.shape, dtype=torch.bfloat16, seed=16)); c_twin.v_pages.copy_(c_hip.v_pages)
    qkv = rnd(ctx.n_tokens, (n_heads + 2 * n_kv) * D, dtype=torch.bfloat16, seed=17)
    q1, q2 = qkv.clone(), qkv.clone()
    ang = torch.outer(torch.arange(720, dtype=torch.float32), 1.0 / (500000.0 ** (torch.arange(0, rd, 2, dtype=torch.float32) / rd)))
    cos, sin = ang.cos().to(DEV), ang.sin().to(DEV)
    hip.rope_kv_write(q1, n_heads, n_kv, D, rd, cos, sin, ctx, c_hip)
    twin.rope_kv_write(q2, n_heads, n_kv, D, rd, cos, sin, ctx, c_twin)
    torch.testing.assert_close(q1.float(), q2.float(), **tol(torch.bfloat16))
    torch.testing.assert_close(c_hip.k_pages.float(), c_twin.k_pages.float(), **tol(torch.bfloat16))
    assert torch.equal(c_hip.v_pages, c_twin.v_pages)


@pytest.mark.parametrize("geom", [
    # heads, kv heads, head_dim, page_size, hidden, rows
    (24, 8, 128, 64, 3072, 8), (3, 1, 32, 8, 192, 16), (5, 5, 96, 16, 1088, 1), (2, 1, 256, 32, 64, 5),
    (7, 7, 64, 4, 2048, 13), (5, 1, 48, 16, 320, 9), (32, 8, 64, 16, 2048, 4), (1, 1, 16, 2, 64, 3), (24, 24, 128, 16, 320, 7),
])
def test_qkv_product_that_rotates_and_writes_the_pages(hip, geom):
    """Few rows: one kernel multiplies, rotates q and k and writes k and v into the pages.  Compared with the
    product, rotation and write done one after the other on float sums (the twin rounds the product first, so
    its result is a rounding away)."""
    n_heads, n_kv, D, ps, hidden, rows = geom
    dtype = torch.bfloat16
    kv_lens = [3 + 41 * i for i in range(rows)]
    kv_lens[-1] = 2 * ps  # a token in the last slot of a page
    if rows > 1:
        kv_lens[0] = ps + 1  # and one in the first
    ctx = Ctx([1] * rows, kv_lens)
    pages = sum(-(-kv // ps) for kv in kv_lens) + 3
    c_hip = Cache(pages, n_kv, ps, D, dtype, kv_lens, seed=4)
    c_ref = Cache(pages, n_kv, ps, D, torch.float32, kv_lens, seed=4)  # float pages: rounded once, at the comparison
    c_hip.k_pages.copy_(rnd(*c_hip.k_pages.shape, dtype=dtype, seed=5)); c_ref.k_pages.copy_(c_hip.k_pages)
    c_hip.v_pages.copy_(rnd(*c_hip.v_pages.shape, dtype=dtype, seed=6)); c_ref.v_pages.copy_(c_hip.v_pages)
    x = rnd(rows, hidden, dtype=dtype, seed=7)
    w = rnd((n_heads + 2 * n_kv) * D, hidden, dtype=dtype, seed=8, scale=hidden ** -0.5)
    pos = torch.arange(max(kv_lens) + 1, dtype=torch.float32)
    inv = 1.0 / (10000.0 ** (torch.arange(0, D, 2, dtype=torch.float32) / D))
    ang = torch.outer(pos, inv)
    cos, sin = ang.cos().to(DEV), ang.sin().to(DEV)
    launched = []
    real = hip.core.sia_gemm_skinny_rope
    hip.core.sia_gemm_skinny_rope = lambda *a: launched.append(1) or real(*a)
    try:
        qkv = hip.qkv_to_cache(x, w, n_heads, n_kv, D, D, cos, sin, ctx, c_hip)
    finally:
        hip.core.sia_gemm_skinny_rope = real
    assert launched, "the fused kernel did not run"
    # reference: float product, rotated in float, rounded once
    ref = (x.float() @ w.float().T)
    twin.rope_kv_write(ref, n_heads, n_kv, D, D, cos, sin, ctx, c_ref)
    nq = n_heads * D
    torch.testing.assert_close(qkv[:, :nq].float(), ref[:, :nq], **tol(dtype))
    torch.testing.assert_close(c_hip.k_pages.float(), c_ref.k_pages, **tol(dtype))
    torch.testing.assert_close(c_hip.v_pages.float(), c_ref.v_pages, **tol(dtype))
    # nothing but the tokens' own slots has changed
    before = rnd(*c_hip.k_pages.shape, dtype=dtype, seed=5)
    changed = (c_hip.k_pages != before).any(dim=-1)            # [page, kv head, offset]
    assert int(changed.any(dim=1).sum()) <= rows
    # and the separate path gives the same within the rounding of the product
    qkv2 = hip.linear(x, w)
    c_two = Cache(pages, n_kv, ps, D, dtype, kv_lens, seed=4)
    c_two.k_pages.copy_(before); c_two.v_pages.copy_(rnd(*c_hip.v_pages.shape, dtype=dtype, seed=6))
    hip.rope_kv_write(qkv2, n_heads, n_kv, D, D, cos, sin, ctx, c_two)
    torch.testing.assert_close(qkv[:, :nq].float(), qkv2[:, :nq].float(), rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(c_hip.k_pages.float(), c_two.k_pages.float(), rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(c_hip.v_pages.float(), c_two.v_pages.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("shape", [
    # rows, hidden, inner (the K of the product into the residual), intermediate of the gated product after it
    (8, 3072, 8192, 8192), (1, 3072, 3072, 8192), (16, 192, 64, 96), (5, 5120, 1024, 5120), (13, 1088, 2048, 320),
    (4, 4160, 128, 1001), (16, 4096, 14336, 1024),
])
def test_norm_shared_out_between_the_products_around_it(hip, shape):
    """Few rows: the product before a norm adds into the residual and leaves gain * x and sums of squares; the product
    after it divides its rows by the root mean square.  Compared with product, add + norm and product one by one."""
    from simple_inference_amd.kernels import PendingProduct, ScaledRows
    rows, hidden, inner, inter = shape
    eps = 1e-5
    x = rnd(rows, inner, dtype=torch.bfloat16, seed=1)
    w = rnd(hidden, inner, dtype=torch.bfloat16, seed=2, scale=inner ** -0.5)
    res = rnd(rows, hidden, seed=3, scale=3.0)
    res[0] *= 40.0   # rows of very different size: each needs its own scale
    gain = (rnd(hidden, seed=4, scale=0.3) + 1.0).contiguous()
    w_gu = rnd(2 * inter, hidden, dtype=torch.bfloat16, seed=5, scale=hidden ** -0.5)

    pending = hip.pending_linear(x, w)
    assert isinstance(pending, PendingProduct)
    res_fused = res.clone()
    scaled = hip.linear_into_residual(pending, res_fused, gain, eps)
    assert isinstance(scaled, ScaledRows)

    res_plain = res.clone()
    normed = hip.add_rmsnorm(res_plain, hip.linear(x, w), gain, eps, torch.bfloat16, None)
    # the residual: same sum unless the plain product went to the library, then a rounding of the delta apart
    torch.testing.assert_close(res_fused, res_plain, rtol=0, atol=2 ** -7)
    want = res.double() + (x.double() @ w.double().T)
    torch.testing.assert_close(res_fused.double(), want, rtol=0, atol=2 ** -6)
    # what it leaves for the product after it: gain * x rounded once, and the sums of squares
    assert torch.equal(scaled.rows, (res_fused * gain).to(torch.bfloat16))
    assert scaled.partials.shape[1] == 16 and hidden / 16 <= scaled.partials.shape[0] <= hidden / 8 + 4   # blocks of 8 to 16 columns
    sums = scaled.partials[:, :rows].double().sum(0)
    torch.testing.assert_close(sums, res_fused.double().pow(2).sum(-1), rtol=1e-5, atol=0)
    rs = torch.rsqrt(sums / hidden + eps)[:, None]
    normed_rows = scaled.rows.double() * rs   # the rows that the fused products multiply, exactly
    torch.testing.assert_close(hip.finish_rows(scaled).double(), normed_rows, **tol(torch.bfloat16))
    torch.testing.assert_close(normed.double(), normed_rows, **tol(torch.bfloat16))

    def mean_error(got, ref):
        return float((got.double() - ref).abs().mean())

    # the gated product: exact given the rows it multiplies, and as near the exact norm as the plain path is
    gu = normed_rows @ w_gu.double().T
    fused = hip.gated_linear(scaled, w_gu)
    torch.testing.assert_close(fused.double(), torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:],
                               **tol(torch.bfloat16))
    exact = want * torch.rsqrt(want.pow(2).mean(-1, keepdim=True) + eps) * gain.double()
    gu = exact @ w_gu.double().T
    ref = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
    assert mean_error(fused, ref) <= 1.25 * mean_error(hip.gated_linear(normed, w_gu), ref) + 1e-5
    torch.testing.assert_close(hip.linear(scaled, w_gu).double(), normed_rows @ w_gu.double().T, **tol(torch.bfloat16))

    # and into the q/k/v product that rotates and writes the pages
    D, n_kv, ps = 32, 2, 16
    n_heads = 4
    w_qkv = rnd((n_heads + 2 * n_kv) * D, hidden, dtype=torch.bfloat16, seed=6, scale=hidden ** -0.5)
    kv_lens = [7 + 19 * i for i in range(rows)]
    ctx = Ctx([1] * rows, kv_lens)
    pages = sum(-(-kv // ps) for kv in kv_lens) + 2
    c1 = Cache(pages, n_kv, ps, D, torch.bfloat16, kv_lens, seed=4)
    c2 = Cache(pages, n_kv, ps, D, torch.float32, kv_lens, seed=4)
    ang = torch.outer(torch.arange(max(kv_lens) + 1, dtype=torch.float32),
                      1.0 / (10000.0 ** (torch.arange(0, D, 2, dtype=torch.float32) / D)))
    cos, sin = ang.cos().to(DEV), ang.sin().to(DEV)
    q1 = hip.qkv_to_cache(scaled, w_qkv, n_heads, n_kv, D, D, cos, sin, ctx, c1)
    q2 = (normed_rows @ w_qkv.double().T).float()
    twin.rope_kv_write(q2, n_heads, n_kv, D, D, cos, sin, ctx, c2)
    torch.testing.assert_close(q1[:, :n_heads * D].float(), q2[:, :n_heads * D], **tol(torch.bfloat16))
    torch.testing.assert_close(c1.k_pages.float(), c2.k_pages, **tol(torch.bfloat16))
    torch.testing.assert_close(c1.v_pages.float(), c2.v_pages, **tol(torch.bfloat16))


@pytest.mark.parametrize("geom", [
    # heads, kv heads, head size, value size, page size, window, block, sinks, cap, kept first
    (32, 8, 64, 64, 16, 0, 0, False, 0.0, 0), (24, 8, 128, 128, 16, 0, 0, False, 0.0, 0), (5, 5, 36, 20, 4, 0, 0, True, 0.0, 0),
    (10, 2, 16, 16, 64, 70, 0, False, 5.0, 3), (6, 2, 100, 128, 128, 0, 96, True, 0.0, 0), (4, 2, 64, 65, 8, 1, 0, False, 0.0, 130),
    (8, 1, 4, 1, 32, 200, 0, True, 2.0, 65),
])
@pytest.mark.parametrize("more", [0, 700, 1500])
def test_float32_attention_is_the_plain_kernels(hip, geom, more):
    """The kernel whose workgroups share keys and values computes what the plain kernel does, with its order of sums:
    the same bits, in every form, for runs that cross the eights of tokens and the chunks of keys, in steps of few tokens
    (a workgroup each) and of many.  Values that a row does not see do not reach it, whatever they are."""
    n_heads, n_kv, D, Dv, ps, window, block, with_sinks, cap, keep = geom
    q_lens, kv_lens = [1, 1, 1, 13, 2, 150, 9], [1, 64, 500, 13, 129, 150, 300]
    if more:
        q_lens, kv_lens = q_lens + [more], kv_lens + [more]
    ctx = Ctx(q_lens, kv_lens)
    pages = sum(-(-kv // ps) for kv in kv_lens) + 2
    cache = Cache(pages, n_kv, ps, D, torch.float32, kv_lens, seed=3)
    cache.k_pages.copy_(rnd(*cache.k_pages.shape, seed=4))
    cache.v_pages = rnd(pages, n_kv, Dv, ps, seed=5)
    qkv = rnd(ctx.n_tokens, (n_heads + n_kv) * D, seed=6)
    sinks = rnd(n_heads, seed=7) if with_sinks else None
    whole = hip.paged_attention(qkv, n_heads, n_kv, D, 0.3, window or None, ctx, cache, value_dim=Dv, chunk=block or None, sinks=sinks,
                                softcap=cap or None, keep_first=keep)
    plain = torch.empty_like(whole)
    ptr = lambda t: None if t is None else t.data_ptr()
    for v in (False, True):
        if v:      # the last token of the long prompt: no other row may see its value
            at = sum(q_lens[:6]) - 1
            page = cache.block_table[5, 149 // ps]
            cache.v_pages[page, :, :, 149 % ps] = float("inf")
        got = hip.paged_attention(qkv, n_heads, n_kv, D, 0.3, window or None, ctx, cache, value_dim=Dv, chunk=block or None, sinks=sinks,
                                  softcap=cap or None, keep_first=keep)
        rc = hip.core.sia_attention_generic(
            ptr(qkv), qkv.shape[1], ptr(cache.k_pages), ptr(cache.v_pages), ptr(cache.block_table), cache.block_table.shape[1],
            ptr(ctx.seq_of_token), ptr(ctx.positions), ptr(plain), ctx.n_tokens, n_heads, n_kv, D, Dv, ps, 0.3, window, block,
            ptr(sinks), cap, keep, 0, torch.cuda.current_stream().cuda_stream)
        assert rc == 0 and torch.equal(got.isnan(), plain.isnan()) and torch.equal(got.nan_to_num(7.0), plain.nan_to_num(7.0)), v
        if v:
            assert torch.equal(got[:at], whole[:at]) and torch.equal(got[at + 1:], whole[at + 1:])


@pytest.mark.parametrize("n_heads,n_kv,D", [(32, 8, 64), (24, 8, 128), (6, 6, 32)])
@pytest.mark.parametrize("q_lens,kv_lens", [([16], [16]), ([17], [17]), ([1, 1, 3], [16, 2, 16]), ([3] * 16, [300] * 16), ([2] * 70, [40] * 70),
                                            ([1, 40], [70, 40]), ([1, 40], [30, 40]), ([64], [264]), ([65], [265])])
def test_float32_attention_has_the_same_bits_whichever_way_it_goes(hip, n_heads, n_kv, D, q_lens, kv_lens):
    """Few keys (the plain kernel), short runs (a workgroup a token), more (16 rows a workgroup): the plain kernel's bits."""
    ctx, ps = Ctx(q_lens, kv_lens), 16
    cache = Cache(sum(-(-kv // ps) for kv in kv_lens), n_kv, ps, D, torch.float32, kv_lens, seed=3)
    cache.k_pages.copy_(rnd(*cache.k_pages.shape, seed=4))
    cache.v_pages.copy_(rnd(*cache.v_pages.shape, seed=5))
    qkv = rnd(ctx.n_tokens, (n_heads + n_kv) * D, seed=6)
    out = hip.paged_attention(qkv, n_heads, n_kv, D, 0.3, None, ctx, cache)
    plain = torch.empty_like(out)
    rc = hip.core.sia_attention_generic(
        qkv.data_ptr(), qkv.shape[1], cache.k_pages.data_ptr(), cache.v_pages.data_ptr(), cache.block_table.data_ptr(),
        cache.block_table.shape[1], ctx.seq_of_token.data_ptr(), ctx.positions.data_ptr(), plain.data_ptr(), ctx.n_tokens, n_heads,
        n_kv, D, D, ps, 0.3, 0, 0, None, 0.0, 0, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and torch.equal(out, plain)


def plain_float_attention(hip, qkv, n_heads, n_kv, D, ctx, cache, window=0):
    out = torch.empty(ctx.n_tokens, n_heads * D, device=DEV)
    assert hip.core.sia_attention_generic(
        qkv.data_ptr(), qkv.shape[1], cache.k_pages.data_ptr(), cache.v_pages.data_ptr(), cache.block_table.data_ptr(),
        cache.block_table.shape[1], ctx.seq_of_token.data_ptr(), ctx.positions.data_ptr(), out.data_ptr(), ctx.n_tokens, n_heads, n_kv, D, D,
        cache.page_size, 0.3, window, 0, None, 0.0, 0, 0, hip._stream()) == 0
    return out


def float_attention_step(n_heads, n_kv, D, q_lens, kv_lens):
    ctx, ps = Ctx(q_lens, kv_lens), 16
    cache = Cache(sum(-(-kv // ps) for kv in kv_lens), n_kv, ps, D, torch.float32, kv_lens, seed=3)
    cache.k_pages.copy_(rnd(*cache.k_pages.shape, seed=4))
    cache.v_pages.copy_(rnd(*cache.v_pages.shape, seed=5))
    return ctx, cache, rnd(ctx.n_tokens, (n_heads + 2 * n_kv) * D, seed=6)


# Rows of one query head a key/value head: a workgroup's 16 rows hold one of a decoded token, or those of several short runs, 16, 8 or 4 of them;
# with few keys the plain kernel's.  Heads of up to 32, 64 and 128 have kernels of their own.
@pytest.mark.parametrize("n_heads,n_kv,D", [(6, 6, 32), (16, 16, 64), (5, 5, 100), (8, 4, 24)])
@pytest.mark.parametrize("n,q,kv", [(256, 1, 17), (256, 1, 41), (100, 1, 65), (200, 4, 64), (90, 3, 130), (64, 2, 40), (17, 9, 70)])
@pytest.mark.parametrize("window", [0, 30])
def test_float32_attention_of_a_query_head_a_key_head_has_the_plain_kernels_bits(hip, n_heads, n_kv, D, n, q, kv, window):
    """Whatever lies in a page behind the last position, or in front of a window, reaches no row; a value that is not finite reaches the rows that see it."""
    ctx, cache, qkv = float_attention_step(n_heads, n_kv, D, [q] * n, [kv - i % 3 for i in range(n)])
    attend = lambda: hip.paged_attention(qkv, n_heads, n_kv, D, 0.3, window or None, ctx, cache)
    whole = attend()
    assert torch.equal(whole, plain_float_attention(hip, qkv, n_heads, n_kv, D, ctx, cache, window))
    page, ps = cache.block_table[1, (kv - 2) // 16], 16      # of the second sequence's last position, kv - 2
    cache.v_pages[page, :, :, (kv - 2) % ps + 1:] = float("nan")
    cache.v_pages[cache.block_table[1, 0], :, :, 0] = float("nan") if window else 1.0
    unseen = attend()
    if window and kv - 1 - q >= window:
        assert torch.equal(unseen, whole)
    cache.v_pages[page, :, :, (kv - 2) % ps] = float("inf")
    got, want = attend(), plain_float_attention(hip, qkv, n_heads, n_kv, D, ctx, cache, window)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))
    assert not bool(got[2 * q - 1].isfinite().any()) and bool(got[2 * q:].isfinite().all())


@pytest.mark.parametrize("n,n_heads,D", [(512, 40, 96), (1024, 16, 128)])
def test_float32_attention_over_few_keys_takes_no_longer_than_the_plain_kernel(hip, n, n_heads, D):
    """Decoded tokens over 17 keys, a query head for each key/value head.  (256 of 40 heads of 96: 70 us by the plain kernel, 161 with a row of 16 a
    workgroup; here enough that the host is ahead.)"""
    ctx, cache, qkv = float_attention_step(n_heads, n_heads, D, [1] * n, [17] * n)

    def us(f):
        best = math.inf
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            f()
            torch.cuda.synchronize()
            a.record()
            for _ in range(40):
                f()
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) * 25)
        return best

    got = us(lambda: hip.paged_attention(qkv, n_heads, n_heads, D, 0.3, None, ctx, cache))
    assert got <= 1.4 * us(lambda: plain_float_attention(hip, qkv, n_heads, n_heads, D, ctx, cache)) + 5


# gate and up in slices and in one, the same of the second product, rows and columns that are no multiples of a tile; one product by tiles, and none
@pytest.mark.parametrize("K,inter,N,M,tiles", [
    (2048, 8192, 2048, 70, 2), (2048, 8192, 2048, 303, 2), (1024, 2816, 1000, 530, 2), (4096, 1056, 4096, 303, 2),
    (4096, 1056, 4096, 530, 2), (512, 4128, 1028, 303, 2), (2048, 8192, 2048, 33, 1), (1024, 2816, 1000, 303, 1),
    (512, 4128, 1028, 17, 0), (50, 37, 21, 3, 0), (50, 37, 21, 1, 0)])
@pytest.mark.parametrize("whole_weights", [False, True])
def test_float_feed_forward_in_one_call_has_the_bits_of_its_parts(hip, K, inter, N, M, tiles, whole_weights):
    """Both products and the activation between them, numbers that are not finite and numbers whose sums are made again among the rows'."""
    x, w, down = rnd(M, K, seed=1), rnd(2 * inter, K, seed=2, scale=K ** -0.5), rnd(N, inter, seed=3, scale=inter ** -0.5)
    if whole_weights:
        w, down = w.bfloat16().float(), down.bfloat16().float()
    for odd in (False, True):
        if odd:
            x[M // 3, 5], x[M - 1, K - 1], x[M // 2, 7], w[inter + 9, 3] = float("nan"), float("inf"), 3.39e38, 1e-39
        want = hip.linear(hip.swiglu(hip.linear(x, w)), down)
        got = hip.float_feed_forward(x, w, down)
        way = lambda t, m, n, k: hip.core.sia_gemm_f32_way(t.data_ptr(), t.data_ptr(), m, n, k) >= 0
        assert way(w, M, 2 * inter, K) + way(down, M, N, inter) == tiles
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0)), odd


# both by tiles and rows of the activation that are no chunks (in fours, and not);  the activation between, and a result whose rows are no fours
@pytest.mark.parametrize("K,inter,N,M", [(512, 4132, 1028, 303), (512, 4131, 1029, 303), (512, 4128, 1029, 303), (2048, 8192, 2047, 303)])
def test_float_feed_forward_of_odd_sizes_in_one_call(hip, K, inter, N, M):
    test_float_feed_forward_in_one_call_has_the_bits_of_its_parts(hip, K, inter, N, M, 2, False)


@pytest.mark.parametrize("which", ["input", "gate/up", "down"])
def test_float_feed_forward_of_operands_that_begin_anywhere(hip, which):
    """A float behind a multiple of 16 bytes: the same bits, by the products' general forms."""
    K, inter, N, M = 512, 4128, 1028, 303
    x, w, down = rnd(M, K, seed=1), rnd(2 * inter, K, seed=2, scale=K ** -0.5), rnd(N, inter, seed=3, scale=inter ** -0.5)
    want = hip.float_feed_forward(x, w, down)

    def shifted(t):
        flat = torch.full((t.numel() + 8,), float("nan"), device=DEV)
        flat[1:1 + t.numel()] = t.flatten()
        return flat[1:1 + t.numel()].view(t.shape)

    got = hip.float_feed_forward(shifted(x) if which == "input" else x, shifted(w) if which == "gate/up" else w, shifted(down) if which == "down" else down)
    assert torch.equal(got, want)


@pytest.mark.parametrize("M,K,inter", [(40000, 256, 1056), (3000, 1024, 8192), (300, 512, 4128), (2500, 512, 4100), (64, 2048, 8192)])
def test_a_float_feed_forward_holds_no_more_memory_than_its_parts(hip, M, K, inter):
    """At most 64 MiB beside what the products and the activation by themselves have in use at a time, in steps of any number of rows.  (The first two, fused
    whatever they need: 200 to 270 MB more.)"""
    from types import SimpleNamespace

    from simple_inference_amd.parts.swiglu import SwiGLU
    part = SwiGLU({"hidden_size": K, "intermediate_size": inter}, SimpleNamespace(kernels=hip))
    x = rnd(M, K, seed=1)
    gate, up, down = (rnd(*shape, seed=i, scale=K ** -0.5) for i, shape in enumerate(((inter, K), (inter, K), (K, inter))))
    part.bind({"gate": gate, "up": up, "down": down})

    def peak(f):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        y = f()
        return torch.cuda.max_memory_allocated() - before, y

    apart, want = peak(lambda: hip.pending_linear(hip.gated_linear(x, part.w_gate_up), part.w_down))
    whole, got = peak(lambda: part.forward(x, None))
    assert torch.equal(got, want) and whole <= apart + (64 << 20) + (1 << 20), (whole, apart)


# 16 rows that are several sequences' (two, six and sixteen of them), a part of one token's heads, and tokens that have workgroups of their own
@pytest.mark.parametrize("n_heads,n_kv,D,Dv", [(8, 8, 64, 64), (12, 4, 20, 36), (40, 2, 128, 100), (17, 1, 64, 64)])
@pytest.mark.parametrize("q_lens", [[1, 1, 30, 2, 1, 1, 70], [2] * 40, [3] * 400])
def test_float32_attention_keeps_sequences_apart(hip, n_heads, n_kv, D, Dv, q_lens):
    """Sequences that share a workgroup's rows: a value that is not finite reaches its own sequence's later rows only."""
    kv_lens, ps = [q + 64 * (i % 3) + i % 5 for i, q in enumerate(q_lens)], 16
    ctx = Ctx(q_lens, kv_lens)
    cache = Cache(sum(-(-kv // ps) for kv in kv_lens), n_kv, ps, D, torch.float32, kv_lens, seed=3)
    cache.k_pages.copy_(rnd(*cache.k_pages.shape, seed=4))
    cache.v_pages = rnd(cache.v_pages.shape[0], n_kv, Dv, ps, seed=5)
    qkv = rnd(ctx.n_tokens, (n_heads + n_kv) * D, seed=6)
    attend = lambda: hip.paged_attention(qkv, n_heads, n_kv, D, 0.3, None, ctx, cache, value_dim=Dv)
    whole = attend()
    plain = torch.empty_like(whole)
    for seq in (None, 2):
        if seq is not None:      # the first key that the sequence's last row alone sees
            at, j = sum(q_lens[:seq + 1]) - 1, kv_lens[seq] - 1
            cache.v_pages[cache.block_table[seq, j // ps], :, :, j % ps] = float("nan")
        got = attend()
        rc = hip.core.sia_attention_generic(
            qkv.data_ptr(), qkv.shape[1], cache.k_pages.data_ptr(), cache.v_pages.data_ptr(), cache.block_table.data_ptr(),
            cache.block_table.shape[1], ctx.seq_of_token.data_ptr(), ctx.positions.data_ptr(), plain.data_ptr(), ctx.n_tokens, n_heads,
            n_kv, D, Dv, ps, 0.3, 0, 0, None, 0.0, 0, 0, torch.cuda.current_stream().cuda_stream)
        assert rc == 0 and torch.equal(got.isnan(), plain.isnan()) and torch.equal(got.nan_to_num(7.0), plain.nan_to_num(7.0)), seq
    assert bool(got[at].isnan().all()) and torch.equal(got[:at], whole[:at]) and torch.equal(got[at + 1:], whole[at + 1:])


# kept positions that end inside a four, at its end, and in the second and third chunk of keys
@pytest.mark.parametrize("keep", [3, 4, 61, 64, 130])
def test_float32_attention_leaves_out_values_between_the_kept_positions_and_the_window(hip, keep):
    """What lies in the pages between the kept first positions and a row's window does not reach the row: with infinities
    and values that are no numbers there, every result has the bits that it has without."""
    n_heads, n_kv, D, ps, window = 8, 2, 64, 16, 50
    q_lens, kv_lens = [1, 1, 40], [300, 500, 260]
    ctx = Ctx(q_lens, kv_lens)
    cache = Cache(sum(-(-kv // ps) for kv in kv_lens), n_kv, ps, D, torch.float32, kv_lens, seed=3)
    cache.k_pages.copy_(rnd(*cache.k_pages.shape, seed=4))
    cache.v_pages.copy_(rnd(*cache.v_pages.shape, seed=5))
    qkv = rnd(ctx.n_tokens, (n_heads + n_kv) * D, seed=6)
    attend = lambda: hip.paged_attention(qkv, n_heads, n_kv, D, 0.3, window, ctx, cache, keep_first=keep)
    want = attend()
    for s, (q, kv) in enumerate(zip(q_lens, kv_lens)):
        for j in range(keep, kv - q - window + 1):      # what no row of the sequence sees
            cache.v_pages[cache.block_table[s, j // ps], :, :, j % ps] = float("inf") if j % 2 else float("nan")
    assert want.isfinite().all() and torch.equal(attend(), want)


@pytest.mark.parametrize("geom", [
    # heads, kv heads, head_dim, page_size, window
    (24, 8, 128, 16, None), (32, 8, 64, 64, None), (16, 1, 32, 8, None), (6, 2, 48, 16, 100), (5, 5, 112, 32, 700),
    (34, 2, 16, 16, None),
])
def test_matrix_core_attention_decode_and_mixed(hip, geom):
    """Many single-token sequences of different lengths (so that splits differ), alone and beside longer runs."""
    n_heads, n_kv, D, ps, window = geom
    dtype = torch.bfloat16
    for q_lens, kv_lens in (([1] * 7, [1, 63, 64, 65, 300, 1027, 2500]),
                            ([1, 1, 1, 130, 5, 257], [513, 17, 2048, 130, 900, 300])):
        ctx = Ctx(q_lens, kv_lens)
        pages = sum(-(-kv // ps) for kv in kv_lens) + 5
        cache = Cache(pages, n_kv, ps, D, dtype, kv_lens, seed=8)
        cache.k_pages.copy_(rnd(*cache.k_pages.shape, dtype=dtype, seed=9))
        cache.v_pages.copy_(rnd(*cache.v_pages.shape, dtype=dtype, seed=10))
        qkv = rnd(ctx.n_tokens, (n_heads + 2 * n_kv) * D, dtype=dtype, seed=11)
        out = hip.paged_attention(qkv, n_heads, n_kv, D, 1 / math.sqrt(D), window, ctx, cache)
        ref = twin.paged_attention(qkv, n_heads, n_kv, D, 1 / math.sqrt(D), window, ctx, cache)
        torch.testing.assert_close(out.float(), ref.float(), **tol(dtype))
        hip.use_mfma_attention = False
        try:
            plain_kernel = hip.paged_attention(qkv, n_heads, n_kv, D, 1 / math.sqrt(D), window, ctx, cache)
        finally:
            hip.use_mfma_attention = True
        torch.testing.assert_close(plain_kernel.float(), ref.float(), **tol(dtype))


@pytest.mark.parametrize("geom", [(24, 8, 128, 16, None), (6, 2, 48, 16, 700), (32, 8, 64, 64, None)])
def test_decode_attention_of_a_sequence_does_not_depend_on_its_batch(hip, geom):
    """How a sequence's keys are split between workgroups and merged follows from its own length: alone, beside
    others, beside many, and under a larger bound on the length (as replayed graphs have it) its result is the
    same bit for bit.  Lengths on both sides of every number of splits (1, 2, 4, 8, 16 from 512 keys a split)."""
    n_heads, n_kv, D, ps, window = geom
    dtype = torch.bfloat16
    kv_lens = [1, 63, 511, 512, 1023, 1024, 1500, 2048, 2500, 4095, 4097, 9000]
    pages = sum(-(-kv // ps) for kv in kv_lens) + 5
    cache = Cache(pages, n_kv, ps, D, dtype, kv_lens, seed=8)
    cache.k_pages.copy_(rnd(*cache.k_pages.shape, dtype=dtype, seed=9))
    cache.v_pages.copy_(rnd(*cache.v_pages.shape, dtype=dtype, seed=10))
    qkv = rnd(len(kv_lens), (n_heads + 2 * n_kv) * D, dtype=dtype, seed=11)
    scale = 1 / math.sqrt(D)

    def run(which, bound=0, repeat=1):
        """Attention of the sequences ``which`` (each ``repeat`` times in the batch) as one decode step."""
        ids = [i for i in which for _ in range(repeat)]
        ctx = Ctx([1] * len(ids), [kv_lens[i] for i in ids])
        ctx.kv_bound = bound
        sub = Cache.__new__(Cache)
        sub.page_size, sub.k_pages, sub.v_pages = ps, cache.k_pages, cache.v_pages
        sub.block_table = cache.block_table[ids].contiguous()
        out = hip.paged_attention(qkv[ids].contiguous(), n_heads, n_kv, D, scale, window, ctx, sub)
        return {i: out[j * repeat] for j, i in enumerate(which)}

    everyone = list(range(len(kv_lens)))
    together = run(everyone)
    ref = twin.paged_attention(qkv, n_heads, n_kv, D, scale, window, Ctx([1] * len(kv_lens), kv_lens), cache)
    torch.testing.assert_close(torch.stack([together[i] for i in everyone]).float(), ref.float(), **tol(dtype))
    bounded = run(everyone, bound=16384)
    many = run(everyone, repeat=6)                    # 72 sequences: more workgroups than compute units
    # so many that one workgroup takes all the splits of a (sequence, kv head) in turn and merges them itself
    crowd = run(everyone, repeat=-(-600 // (n_kv * len(everyone))))
    crowd_bounded = run(everyone, bound=16384, repeat=-(-600 // (n_kv * len(everyone))))
    for i in everyone:
        alone = run([i])[i]
        assert torch.equal(alone, together[i]), kv_lens[i]
        assert torch.equal(alone, bounded[i]), kv_lens[i]
        assert torch.equal(alone, many[i]), kv_lens[i]
        assert torch.equal(alone, crowd[i]), kv_lens[i]
        assert torch.equal(alone, crowd_bounded[i]), kv_lens[i]
    pair = run([3, 9])
    assert torch.equal(pair[3], together[3]) and torch.equal(pair[9], together[9])


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("sinks", [False, True])
def test_decode_attention_takes_nothing_from_splits_that_a_sequence_does_not_have(hip, D, sinks):
    """Sequences of 1 to 32 splits in one launch with a second that combines them: whatever the workspaces held before, the bits are the same.
    (The states of up to all splits are asked for before it is known how many there are.)"""
    n_heads, n_kv, ps = 16, 8, 16
    kv_lens = [40, 20000, 700, 1100, 2100, 1600, 5000, 9000]
    ctx = Ctx([1] * len(kv_lens), kv_lens)
    cache = Cache(sum(-(-kv // ps) for kv in kv_lens), n_kv, ps, D, torch.bfloat16, kv_lens, seed=8)
    cache.k_pages.copy_(rnd(*cache.k_pages.shape, dtype=torch.bfloat16, seed=9))
    cache.v_pages.copy_(rnd(*cache.v_pages.shape, dtype=torch.bfloat16, seed=10))
    qkv = rnd(len(kv_lens), (n_heads + 2 * n_kv) * D, dtype=torch.bfloat16, seed=11)
    sink = rnd(n_heads, seed=12) if sinks else None
    attend = lambda: hip.paged_attention(qkv, n_heads, n_kv, D, D ** -0.5, None, ctx, cache, sinks=sink)
    attend()
    (_, max_splits, ws_acc, ws_ml, _, _), = ctx.attention_plans.values()
    assert max_splits == 32 and hip._attn_lib(D).sia_attn_decode_mode(len(kv_lens), n_heads, n_kv, max_splits) == 0
    results = []
    for value in (0.0, float("nan"), float("inf"), -3e38):
        ws_acc.fill_(value)
        ws_ml.fill_(value)
        results.append(attend())
    assert bool(results[0].isfinite().all()) and all(torch.equal(r, results[0]) for r in results)
    ref = twin.paged_attention(qkv, n_heads, n_kv, D, D ** -0.5, None, ctx, cache, sinks=sink)
    torch.testing.assert_close(results[0].float(), ref.float(), **tol(torch.bfloat16))


def test_few_row_products_do_not_depend_on_the_number_of_rows(hip):
    """Up to 16 rows every product (plain, gated, into the residual, with the norm's row scale, with rotation and
    cache write) sums k in an order that K alone fixes: a row's result is the same bit for bit whether it runs
    alone, among 4, among 5 (another kernel shape from 5 rows on) or among 16."""
    from simple_inference_amd.kernels import ScaledRows
    dtype = torch.bfloat16
    for N, K in ((3072, 8192), (5120, 3072), (16384, 3072), (1008, 1024), (48, 192)):
        x, w = rnd(16, K, dtype=dtype, seed=1), rnd(N, K, dtype=dtype, seed=2, scale=K ** -0.5)
        full = hip.linear(x, w)
        full32 = hip.linear(x, w, out_float32=True)
        for m in (1, 4, 5, 11):
            assert torch.equal(hip.linear(x[:m].contiguous(), w), full[:m]), (N, K, m)
            assert torch.equal(hip.linear(x[:m].contiguous(), w, out_float32=True), full32[:m]), (N, K, m)
            assert torch.equal(hip.linear(x[m - 1:m].contiguous(), w), full[m - 1:m]), (N, K, m)
    for inter, K in ((8192, 3072), (96, 320), (5120, 1024)):
        x = rnd(16, K, dtype=dtype, seed=3)
        w = rnd(2 * inter, K, dtype=dtype, seed=4, scale=K ** -0.5)
        full = hip.gated_linear(x, w)
        for m in (1, 4, 5, 11):
            assert torch.equal(hip.gated_linear(x[:m].contiguous(), w), full[:m]), (inter, K, m)
    # into the residual, and out of it again through the row scale of the products that follow
    hidden, inner, inter = 3072, 8192, 8192
    x = rnd(16, inner, dtype=dtype, seed=5)
    w = rnd(hidden, inner, dtype=dtype, seed=6, scale=inner ** -0.5)
    w_gu = rnd(2 * inter, hidden, dtype=dtype, seed=7, scale=hidden ** -0.5)
    res = rnd(16, hidden, seed=8, scale=2.0)
    gain = (rnd(hidden, seed=9, scale=0.3) + 1.0).contiguous()

    def through(m):
        r = res[:m].clone()
        scaled = hip.linear_into_residual(hip.pending_linear(x[:m].contiguous(), w), r, gain, 1e-5)
        assert isinstance(scaled, ScaledRows)
        return r, scaled.rows, hip.gated_linear(scaled, w_gu), hip.linear(scaled, w_gu)
    full = through(16)
    for m in (1, 4, 5, 11):
        for got, want in zip(through(m), full):
            assert torch.equal(got, want[:m]), m


@pytest.mark.parametrize("N, K", [(3072, 3072), (3070, 8192), (2048, 2048), (4099, 192)])
def test_the_product_into_the_residual_reads_the_weight_as_it_is(hip, N, K):
    """Residual, scaled rows and sums of squares against the product in 64 bits, also where the last block of rows is short
    (3,070 and 4,099 rows), and again when the weight has been changed in place: nothing of it is kept."""
    dtype = torch.bfloat16
    x = rnd(16, K, dtype=dtype, seed=1)
    w = rnd(N, K, dtype=dtype, seed=2, scale=K ** -0.5)
    res = rnd(16, N, seed=3, scale=2.0)
    gain = (rnd(N, seed=4, scale=0.3) + 1.0).contiguous()
    for _ in range(2):
        product = x.double() @ w.double().T
        for m in (1, 7, 16):
            r = res[:m].clone()
            scaled = hip.linear_into_residual(hip.pending_linear(x[:m].contiguous(), w), r, gain, 1e-5)
            # the product is rounded to bfloat16 (2^-9 of it, and what its float sums leave), the sum to 32 bits
            want = res[:m].double() + product[:m]
            assert bool(((r.double() - want).abs() <= 2.0 ** -8 * product[:m].abs() + 5e-7 * K).all())
            assert torch.equal(scaled.rows, (r * gain).to(dtype))
            torch.testing.assert_close(scaled.partials[:, :m].double().sum(0), r.double().square().sum(1), rtol=1e-5, atol=0)
        w.mul_(2.0)


SPLIT, PAIRED, WIDE, LONG = range(4)      # of sia_attn_prefill_shape


def prefill_shape(hip, D, n_heads, q_lens, kv_lens, window=None, chunk=None, forms=False):
    """The workgroup shape that a step of these portions takes, decoded tokens apart."""
    lib = hip._attn_lib(D, forms=forms)
    tiles = [sum(-(-q // rows()) for q in q_lens)
             for rows in (lib.sia_attn_prefill_rows, lib.sia_attn_prefill_rows_split, lib.sia_attn_prefill_rows_long)]
    return lib.sia_attn_prefill_shape(*tiles, max(q_lens), max(kv_lens), n_heads, window or 0, chunk or 0)


# One prompt from its start, of 15/8 to 18/8 and of 30/8 to 36/8 workgroups of 128 tokens a compute unit, and what is none: through a window, in
# blocks, over earlier tokens, several.
@pytest.mark.parametrize("D, n_heads, q_lens, past, window, chunk, shape", [
    (64, 24, [3067], 0, None, None, PAIRED), (64, 24, [3067], 0, 1024, None, WIDE), (64, 24, [3067], 0, None, 1024, WIDE),
    (64, 24, [3067], 0, 4096, 8192, PAIRED), (64, 24, [3067], 1536, None, None, WIDE), (64, 32, [700] * 3, 0, None, None, WIDE),
    (64, 32, [1100] * 2, 0, None, None, PAIRED), (64, 32, [2043], 510, None, None, PAIRED), (64, 32, [2043], 0, 1600, None, PAIRED),
    (64, 32, [2171], 500, None, None, WIDE), (64, 24, [3000], 8192, None, None, WIDE), (32, 32, [2299], 0, 256, None, WIDE),
    (128, 24, [3067], 0, None, None, PAIRED), (128, 24, [3067], 0, 1024, None, WIDE), (128, 24, [3067], 1536, None, None, WIDE),
    (80, 24, [2939], 0, None, None, PAIRED), (80, 24, [3067], 0, None, None, WIDE), (112, 24, [3067], 0, None, None, WIDE),
    (128, 32, [4091], 0, None, None, LONG), (128, 32, [4091], 0, 256, None, WIDE), (128, 32, [4091], 0, None, 300, WIDE),
    (128, 32, [4091], 1000, None, None, LONG), (128, 32, [4347], 1000, None, None, WIDE), (128, 32, [2043] * 2, 0, None, None, WIDE),
    (64, 32, [4091], 0, None, None, WIDE), (80, 32, [4091], 0, None, None, WIDE), (112, 32, [4091], 0, None, None, WIDE),
    (80, 32, [4603], 0, None, None, LONG), (80, 32, [4603], 0, 256, None, LONG), (64, 32, [7001], 0, None, None, WIDE)])
def test_prefill_shapes_follow_what_the_row_tiles_see(hip, D, n_heads, q_lens, past, window, chunk, shape):
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    assert prefill_shape(hip, D, n_heads, q_lens, [q + past for q in q_lens], window, chunk) == shape


@pytest.mark.parametrize("q_len, kv_len, window, shape", [(130, 130, None, SPLIT), (900, 1000, None, PAIRED), (1900, 1900, None, PAIRED),
                                                         (1900, 2100, 300, WIDE), (2900, 2900, None, WIDE)])
def test_matrix_core_prefill_in_each_workgroup_shape(hip, q_len, kv_len, window, shape):
    """The prefill kernel picks one of four workgroup shapes, three for heads of 16: with 34 heads, 130
    tokens take the split shape (64 tokens, even and odd key tiles on two sets of waves, merged at the end),
    900 and 1,900 the paired one of 8 waves, and 1,900 through a window and 2,900 the wide one.  Lengths are no multiples of a tile."""
    n_heads, n_kv, D, ps = 34, 2, 16, 16
    dtype = torch.bfloat16
    ctx = Ctx([q_len, 3], [kv_len, 40])
    assert prefill_shape(hip, D, n_heads, [q_len, 3], [kv_len, 40], window) == shape
    cache = Cache(-(-kv_len // ps) + 8, n_kv, ps, D, dtype, [kv_len, 40], seed=31)
    cache.k_pages.copy_(rnd(*cache.k_pages.shape, dtype=dtype, seed=32))
    cache.v_pages.copy_(rnd(*cache.v_pages.shape, dtype=dtype, seed=33))
    qkv = rnd(ctx.n_tokens, (n_heads + 2 * n_kv) * D, dtype=dtype, seed=34, scale=2.0)
    out = hip.paged_attention(qkv, n_heads, n_kv, D, 1 / math.sqrt(D), window, ctx, cache)
    ref = twin.paged_attention(qkv, n_heads, n_kv, D, 1 / math.sqrt(D), window, ctx, cache)
    torch.testing.assert_close(out.float(), ref.float(), **tol(dtype))


def test_matrix_core_prefill_in_workgroups_of_256_tokens(hip):
    """Very many workgroups (128 heads of 80, 2,500 tokens) take the shape of 8 waves of 32 tokens; a second and a third
    run in the same launch, shorter than a workgroup and a little longer than one, and a window."""
    n_heads, n_kv, D, ps = 128, 8, 80, 16
    dtype = torch.bfloat16
    q_lens, kv_lens = [2500, 40, 300], [2700, 40, 555]
    ctx = Ctx(q_lens, kv_lens)
    cache = Cache(sum(-(-kv // ps) for kv in kv_lens) + 8, n_kv, ps, D, dtype, kv_lens, seed=41)
    cache.k_pages.copy_(rnd(*cache.k_pages.shape, dtype=dtype, seed=42))
    cache.v_pages.copy_(rnd(*cache.v_pages.shape, dtype=dtype, seed=43))
    qkv = rnd(ctx.n_tokens, (n_heads + 2 * n_kv) * D, dtype=dtype, seed=44, scale=2.0)
    assert hip._attn_lib(D).sia_attn_prefill_rows_long() == 256
    for window in (None, 700):
        assert prefill_shape(hip, D, n_heads, q_lens, kv_lens, window) == LONG
        out = hip.paged_attention(qkv, n_heads, n_kv, D, 1 / math.sqrt(D), window, ctx, cache)
        ref = twin.paged_attention(qkv, n_heads, n_kv, D, 1 / math.sqrt(D), window, ctx, cache)
        torch.testing.assert_close(out.float(), ref.float(), **tol(dtype))


# Every shape of workgroup with every form of mask and score.  Lengths are no multiples of a tile.
@pytest.mark.parametrize("q_len, shape", [(130, SPLIT), (900, PAIRED), (2600, WIDE), (4300, LONG)])
@pytest.mark.parametrize("form", [{}, {"window": 333}, {"chunk": 500}, {"sinks": True}, {"softcap": 2.0}, {"window": 333, "keep_first": 75}])
def test_matrix_core_prefill_shapes_in_every_form(hip, q_len, shape, form):
    n_heads, n_kv, D, ps, dtype = 34, 2, 80, 16, torch.bfloat16
    q_lens, kv_lens = [q_len, 3], [q_len + 50, 40]
    forms = "softcap" in form or "keep_first" in form
    assert prefill_shape(hip, D, n_heads, q_lens, kv_lens, form.get("window"), form.get("chunk"), forms) == shape
    ctx = Ctx(q_lens, kv_lens)
    cache = Cache(-(-kv_lens[0] // ps) + 8, n_kv, ps, D, dtype, kv_lens, seed=31)
    cache.k_pages.copy_(rnd(*cache.k_pages.shape, dtype=dtype, seed=32))
    cache.v_pages.copy_(rnd(*cache.v_pages.shape, dtype=dtype, seed=33))
    qkv = rnd(ctx.n_tokens, (n_heads + 2 * n_kv) * D, dtype=dtype, seed=34, scale=2.0)
    more = {k: v for k, v in form.items() if k != "window"}
    if "sinks" in more:
        more["sinks"] = rnd(n_heads, seed=35) + 1.0
    args = (qkv, n_heads, n_kv, D, 1 / math.sqrt(D), form.get("window"), ctx, cache)
    torch.testing.assert_close(hip.paged_attention(*args, **more).float(), twin.paged_attention(*args, **more).float(), **tol(dtype))


def test_matrix_core_attention_runs_longer_than_a_block_table_window(hip, monkeypatch):
    """A wave holds 64 block-table entries at a time.  With pages of 64, runs of more than 4,096 keys that
    start in the middle of a page (tiles are 32 keys) must reload the entries at a page's edge: one decoded
    token over 17,500 keys (four runs of about 4,380 keys), and a prompt portion under a window of 5,000."""
    n_heads, n_kv, D, ps = 2, 1, 16, 64
    dtype = torch.bfloat16
    # one workgroup per (sequence, kv head), whatever the length: a wave's run of keys is then longer than a window
    monkeypatch.setattr(hip._attn_lib(D), "sia_attn_decode_max_splits", lambda kv_bound, window: 1)
    for q_lens, kv_lens, window in (([1], [17500], None), ([1], [17500], 9001), ([70], [9000], 5000)):
        ctx = Ctx(q_lens, kv_lens)
        cache = Cache(-(-kv_lens[0] // ps) + 3, n_kv, ps, D, dtype, kv_lens, seed=21)
        cache.k_pages.copy_(rnd(*cache.k_pages.shape, dtype=dtype, seed=22))
        cache.v_pages.copy_(rnd(*cache.v_pages.shape, dtype=dtype, seed=23))
        qkv = rnd(ctx.n_tokens, (n_heads + 2 * n_kv) * D, dtype=dtype, seed=24, scale=3.0)
        out = hip.paged_attention(qkv, n_heads, n_kv, D, 1 / math.sqrt(D), window, ctx, cache)
        ref = twin.paged_attention(qkv, n_heads, n_kv, D, 1 / math.sqrt(D), window, ctx, cache)
        torch.testing.assert_close(out.float(), ref.float(), **tol(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("q_len", [1, 40])
def test_attention_finds_one_key_at_every_kind_of_edge(hip, dtype, q_len):
    """One key among hundreds is made to stand out; the output must be its value row.  The key is put at
    the edges where an indexing fault would lose it: first and last offset of a page, of a 32- and
    64-key tile, the first key, the newest key, and both sides of a window's edge.  (700 keys are 22 tiles, which
    the decode kernel does not split; longer sequences and their splits have a test of their own below.)"""
    n_heads, n_kv, D, ps = 4, 2, 64, 16
    kv = 700
    ctx = Ctx([q_len], [kv])
    last = kv - 1                       # the position of the last query
    direction = torch.nn.functional.normalize(rnd(D, seed=3), dim=0)
    base_k = 0.01 * rnd(64, n_kv, ps, D, seed=1)
    values = rnd(64, n_kv, D, ps, seed=2)
    qkv = torch.zeros(q_len, (n_heads + 2 * n_kv) * D)
    qkv[:, :n_heads * D] = (30.0 * direction).repeat(n_heads)
    qkv = qkv.to(dtype).to(DEV)
    cache = Cache(64, n_kv, ps, D, dtype, [kv])
    cache.v_pages.copy_(values.to(dtype))
    window = 300
    edge = last - window + 1            # oldest key the last query sees through the window
    for far, win, seen in [(0, None, True), (15, None, True), (16, None, True), (31, None, True), (32, None, True),
                           (63, None, True), (64, None, True), (255, None, True), (256, None, True),
                           (511, None, True), (512, None, True), (last - q_len, None, True), (last, None, True),
                           (edge, window, True), (edge - 1, window, False), (edge + 1, window, True)]:
        cache.k_pages.copy_(base_k.to(dtype))
        page = int(cache.block_table[0, far // ps])
        cache.k_pages[page, :, far % ps] = (30.0 * direction).to(dtype)
        out = hip.paged_attention(qkv, n_heads, n_kv, D, 1 / math.sqrt(D), win, ctx, cache).float()
        row = out[-1].view(n_heads, D)      # the last query sees every key up to ``last``
        for h in range(n_heads):
            want = cache.v_pages[page, h // 2, :, far % ps].float()
            close = torch.allclose(row[h], want, rtol=2e-2, atol=2e-2)
            assert close == seen, (far, win, h)


def _decode_splits(n_tiles):
    """How many workgroups share a sequence of that many visible key tiles (the kernel's own rule, written down a
    second time so that the test knows where the runs of tiles begin)."""
    s = 1
    while s < 32 and 2 * s * 16 <= n_tiles:
        s *= 2
    return s


@pytest.mark.parametrize("kv, window", [(1100, None), (2500, None), (9000, None), (9000, 5000)])
def test_decode_attention_finds_one_far_key_however_its_runs_are_spread(hip, kv, window):
    """A decoding sequence of 1,100 to 9,000 keys is cut into 2 to 16 splits of four runs of tiles each, and the
    runs are spread over workgroups in three ways: a workgroup a run (few sequences), a workgroup a split (some),
    one workgroup for all of a sequence's runs (a crowd).  One key is made to stand out and the output must be its
    value row, with the key at the first and the last position of runs in the middle of a split, at a split's
    edge, in the very first and the very last run, and on either side of a window's edge; in each of the three ways,
    and in a grid sized for a longer sequence than the step holds."""
    n_heads, n_kv, D, ps = 4, 2, 64, 16
    dtype = torch.bfloat16
    lib = hip._attn_lib(D)
    last = kv - 1
    lo_all = max(0, last - window + 1) if window else 0
    t_first, n_tiles = lo_all // 32, last // 32 - lo_all // 32 + 1
    n_splits = _decode_splits(n_tiles)
    n_runs = 4 * n_splits
    assert n_splits >= 2
    begin = lambda run: (t_first + run * n_tiles // n_runs) * 32         # first key of a run
    runs = sorted({1, 2, 4, 5, n_runs // 2, n_runs - 4, n_runs - 1})
    places = {max(lo_all, begin(run)) for run in runs} | {begin(run) - 1 for run in runs if begin(run) - 1 >= lo_all}
    cases = [(p, True) for p in sorted(places | {lo_all, last})]
    if window:
        cases += [(lo_all - 1, False), (lo_all + 1, True)]
    n_pages = -(-kv // ps)
    direction = torch.nn.functional.normalize(rnd(D, seed=3), dim=0)
    base_k = (0.01 * rnd(n_pages, n_kv, ps, D, seed=1)).to(dtype)
    cache = Cache(n_pages, n_kv, ps, D, dtype, [kv], seed=5)
    cache.v_pages.copy_(rnd(n_pages, n_kv, D, ps, seed=2).to(dtype))
    row = cache.block_table[0].clone()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    crowd = -(-cus // n_kv) + 3                                            # a (sequence, kv head) pair a compute unit
    some = -(-cus // (n_kv * n_splits)) + 1                                # more splits than compute units
    seen_modes = set()
    for n_seqs, bound, want_mode in ((1, 0, 2), (some, 0, 0), (crowd, 0, 1), (1, 4 * kv, 2), (crowd, 2 * kv, 1)):
        ctx = Ctx([1] * n_seqs, [kv] * n_seqs)
        ctx.kv_bound = bound
        max_splits = lib.sia_attn_decode_max_splits(bound or kv, window or 0)
        if some * n_kv >= cus and want_mode == 0:
            continue                                                       # two splits only: no step takes that way
        assert lib.sia_attn_decode_mode(n_seqs, n_heads, n_kv, max_splits) == want_mode, (n_seqs, bound)
        seen_modes.add(want_mode)
        cache.block_table = row.repeat(n_seqs, 1).contiguous()             # every sequence reads the same pages
        qkv = torch.zeros(n_seqs, (n_heads + 2 * n_kv) * D)
        qkv[:, :n_heads * D] = (30.0 * direction).repeat(n_heads)
        qkv = qkv.to(dtype).to(DEV)
        for far, seen in cases:
            cache.k_pages.copy_(base_k)
            page = int(row[far // ps])
            cache.k_pages[page, :, far % ps] = (30.0 * direction).to(dtype)
            out = hip.paged_attention(qkv, n_heads, n_kv, D, 1 / math.sqrt(D), window, ctx, cache).float()
            for s in sorted({0, n_seqs // 2, n_seqs - 1}):
                got = out[s].view(n_heads, D)
                for h in range(n_heads):
                    want = cache.v_pages[page, h // 2, :, far % ps].float()
                    assert torch.allclose(got[h], want, rtol=2e-2, atol=2e-2) == seen, (n_seqs, bound, far, s, h)
    assert {1, 2} <= seen_modes


@pytest.mark.parametrize("vocab", [16, 1000, 128256])
def test_sample_matches_twin(hip, vocab):
    rows = 12
    logits = rnd(rows, vocab, seed=1, scale=2.0)
    temperature = torch.tensor([0, 0, 1, 1, 0.7, 0.7, 1.3, 1, 1, 0.5, 1, 2], dtype=torch.float32, device=DEV)
    top_k = torch.tensor([0, 5, 0, 0, 5, 0, 50, 1, 0, 3, vocab, 7], dtype=torch.int32, device=DEV)
    top_p = torch.tensor([1, 1, 1, 1, 1, 0.9, 0.5, 1, 0.0, 0.8, 1, 0.3], dtype=torch.float32, device=DEV)
    for seed in range(4):
        u = torch.rand(rows, generator=torch.Generator().manual_seed(seed)).to(DEV)
        got = hip.sample(logits, temperature, top_k, top_p, u)
        ref = twin.sample(logits, temperature, top_k, top_p, u)
        assert got.tolist() == ref.tolist(), (seed, got.tolist(), ref.tolist())


@pytest.mark.parametrize("vocab", [7, 331, 50257])
def test_sample_filters_at_their_edges(hip, vocab):
    """Rows made so that a filter's edge shows: equal values (kept or dropped together), a k that is one short
    of everything, a p so small that only the top stays, a single dominant token, values of both signs far
    apart, and draws at both ends of the unit interval.  The hints of which filters exist must not matter."""
    g = torch.Generator().manual_seed(vocab)
    rows = []
    flat = torch.zeros(vocab)                                        # all equal
    steps = torch.arange(vocab, dtype=torch.float32).flip(0) * 0.25   # strictly falling
    pairs = (torch.arange(vocab) // 2).float().flip(0) * 0.5          # equal pairs
    spike = torch.randn(vocab, generator=g); spike[vocab // 3] = 30.0
    wide = torch.randn(vocab, generator=g) * 40.0
    shuffled = steps[torch.randperm(vocab, generator=g)]
    cases = []
    for base in (flat, steps, pairs, spike, wide, shuffled):
        ties = base is flat or base is pairs   # a sort splits equal values as it likes: no top-p oracle for them
        for k, p in ((0, 1.0), (1, 1.0), (3, 1.0), (vocab - 1, 1.0), (0, 1e-6), (0, 0.5), (4, 0.7), (0, 0.999)):
            if not (ties and p < 1.0):
                cases.append((base, 0.8, k, p))
    logits = torch.stack([c[0] for c in cases]).to(DEV)
    temperature = torch.tensor([c[1] for c in cases], dtype=torch.float32, device=DEV)
    top_k = torch.tensor([c[2] for c in cases], dtype=torch.int32, device=DEV)
    top_p = torch.tensor([c[3] for c in cases], dtype=torch.float32, device=DEV)
    for u_value in (1e-6, 0.37, 0.999999):
        u = torch.full((len(cases),), u_value, dtype=torch.float32, device=DEV)
        got = hip.sample(logits, temperature, top_k, top_p, u)
        ref = twin.sample(logits, temperature, top_k, top_p, u)
        assert got.tolist() == ref.tolist(), (u_value, [i for i, (a, b) in enumerate(zip(got.tolist(), ref.tolist())) if a != b])
    # equal values are kept or dropped together: under any top-p, all of a row of equal values can be drawn
    n = 5
    flat_rows = flat.repeat(n, 1).to(DEV)
    u = torch.linspace(0.01, 0.99, n, device=DEV)
    got = hip.sample(flat_rows, torch.full((n,), 0.8, device=DEV), torch.zeros(n, dtype=torch.int32, device=DEV),
                     torch.full((n,), 0.3, device=DEV), u)
    assert got.tolist() == [min(vocab - 1, int(x * vocab)) for x in u.tolist()]
    # rows without a filter, sampled with the hint that there is none
    plain_rows = [i for i, c in enumerate(cases) if c[2] == 0 and c[3] == 1.0]
    sel = torch.tensor(plain_rows, device=DEV)
    u = torch.full((len(plain_rows),), 0.61, dtype=torch.float32, device=DEV)
    args = (logits[sel].contiguous(), temperature[sel].contiguous(), top_k[sel].contiguous(), top_p[sel].contiguous(), u)
    assert hip.sample(*args, filters=0).tolist() == hip.sample(*args).tolist() == twin.sample(*args).tolist()


def test_sample_does_not_care_what_its_workspace_held(hip):
    """The sampler sets to zero what it needs at zero: a workspace full of ones gives the tokens of a zeroed one,
    and the kernels object's own workspace, used by every call before this one, gives them too."""
    rows, vocab = 6, 3001
    logits = rnd(rows, vocab, seed=8, scale=2.5)
    temperature = torch.tensor([0.9, 0.0, 1.1, 0.6, 1.0, 0.8], dtype=torch.float32, device=DEV)
    top_k = torch.tensor([40, 0, 0, 7, 0, 2999], dtype=torch.int32, device=DEV)
    top_p = torch.tensor([0.9, 1.0, 0.6, 1.0, 1.0, 0.95], dtype=torch.float32, device=DEV)
    u = torch.tensor([0.11, 0.5, 0.93, 0.42, 0.77, 0.3], dtype=torch.float32, device=DEV)
    want = hip.sample(logits, temperature, top_k, top_p, u).tolist()
    assert want == twin.sample(logits, temperature, top_k, top_p, u).tolist()
    size = hip.core.sia_sample_workspace_bytes(rows)
    for fill in (0, 255, 1):
        out = torch.full((rows,), -1, dtype=torch.int32, device=DEV)
        workspace = torch.full((size,), fill, dtype=torch.uint8, device=DEV)
        code = hip.core.sia_sample(logits.data_ptr(), temperature.data_ptr(), top_k.data_ptr(), top_p.data_ptr(),
                                   u.data_ptr(), out.data_ptr(), workspace.data_ptr(), rows, vocab, 7,
                                   torch.cuda.current_stream().cuda_stream)
        assert code == 0
        assert out.tolist() == want, fill


@pytest.mark.parametrize("vocab", [5, 1001, 4096, 128256])
def test_argmax_of_all_greedy_steps(hip, vocab):
    rows = 9
    logits = rnd(rows, vocab, seed=3, scale=3.0)
    logits[1] = 0.0                                   # all equal: index 0
    logits[2, vocab - 1] = 50.0                       # the last element
    logits[3, [vocab // 2, vocab - 2 if vocab > 2 else 0]] = 60.0   # a tie across chunks: the lower index
    z = lambda dt, v: torch.full((rows,), v, dtype=dt, device=DEV)
    args = (logits, z(torch.float32, 0.0), z(torch.int32, 0), z(torch.float32, 1.0), z(torch.float32, 0.5))
    spread = hip.sample(*args, all_greedy=True)
    assert spread.tolist() == hip.sample(*args).tolist()
    library = torch.argmax(logits, -1).tolist()
    assert [t for i, t in enumerate(spread.tolist()) if i not in (1, 3)] == [t for i, t in enumerate(library) if i not in (1, 3)]
    assert spread[1].item() == 0 and spread[2].item() == vocab - 1
    assert spread[3].item() == min(vocab // 2, vocab - 2 if vocab > 2 else 0)


def test_sample_greedy_is_argmax_with_lowest_index_on_ties(hip):
    logits = torch.zeros(3, 5000, device=DEV)
    logits[0, 4321] = 1.0
    logits[1, [17, 4000]] = 2.0
    z = lambda dt, v: torch.full((3,), v, dtype=dt, device=DEV)
    got = hip.sample(logits, z(torch.float32, 0.0), z(torch.int32, 0), z(torch.float32, 1.0), z(torch.float32, 0.5))
    assert got.tolist() == [4321, 17, 0]


@pytest.mark.parametrize("vocab", [1, 40, 511, 8192, 8193, 16 * 513, 128256, 131072, 131073])
def test_sampling_among_few_tokens_is_the_series_of_launches(hip, vocab):
    """The two launches for rows that all keep few tokens by top-k give the token of the series of launches, bit for bit:
    over random rows, rows of equal values (more than fit a chunk's places), rows with few finite values, infinities and
    values that are no numbers; any temperature, top-p and number; greedy rows beside them."""
    g = torch.Generator().manual_seed(vocab)
    rows = [torch.randn(vocab, generator=g) * s for s in (1.0, 4.0, 0.01, 30.0)]
    rows += [torch.zeros(vocab), torch.randint(0, 3, (vocab,), generator=g).float(), torch.full((vocab,), -float("inf"))]
    few = torch.full((vocab,), -float("inf"))
    few[torch.randint(0, vocab, (7,), generator=g)] = torch.randn(7, generator=g)
    high = torch.randn(vocab, generator=g)
    high[: vocab // 3] += 80.0
    odd = torch.randn(vocab, generator=g)
    odd[torch.randint(0, vocab, (3,), generator=g)] = float("nan")
    endless = torch.randn(vocab, generator=g)
    endless[vocab // 2] = float("inf")
    rows += [few, high, odd, endless]
    cases = [(t, k, p, u) for t in (1.0, 0.7, 1e-3, 0.0, 5.0) for k, p, u in ((1, 1.0, 0.3), (50, 0.9, 0.77), (256, 0.5, 0.999),
                                                                              (50, 0.0, 0.2), (7, 1.0, 0.0), (255, 0.99, 0.5))]
    logits = torch.stack(rows).repeat_interleave(len(cases), 0).to(DEV)
    column = lambda i, dtype: torch.tensor([c[i] for c in cases] * len(rows), dtype=dtype, device=DEV)
    args = (logits, column(0, torch.float32), column(1, torch.int32), column(2, torch.float32), column(3, torch.float32))
    for filters in (3, 1):
        assert torch.equal(hip.sample(*args, filters=filters, few=True), hip.sample(*args, filters=filters)), filters
