"""Every HIP kernel alone against a plain torch float32 reference of the same
operation, at sizes other than the tiny models' (widths and vocabularies that are
no power of two, odd head counts, head sizes in steps of 16, page sizes that do not
divide the lengths). Pure data movement must be bit-exact."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]


def tol(dtype):
    # float32: rounding of a few float operations; bfloat16: one rounding to 8 bits (2^-9 relative) of
    # values of size about 1-4
    return dict(rtol=1e-5, atol=1e-5) if dtype == torch.float32 else dict(rtol=1.6e-2, atol=1.6e-2)


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from nanohybrid_vlm_amd.native import ops as o
    assert o.backend().name == "hip"
    return o


def rnd(*shape, dtype=torch.float32, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).cuda()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,H,V", [(1, 80, 301), (37, 1000, 77), (300, 4096, 1000)])
def test_embed_and_gather_are_exact(ops, dtype, T, H, V):
    table = rnd(V, H, dtype=dtype)
    ids = torch.randint(0, V, (T,), dtype=torch.int32, device="cuda")
    out = ops.embed(ids, table)
    assert torch.equal(out, table[ids.long()])
    rows = torch.randint(0, T, (5,), dtype=torch.int32, device="cuda")
    assert torch.equal(ops.gather_rows(out, rows), out[rows.long()])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,H,eps", [(3, 80, 1e-5), (17, 1000, 1e-6), (5, 4096, 1e-6), (2, 12288, 1e-3), (4, 1001, 1e-5),
                                     (1, 8192, 1e-6), (300, 5120, 1e-6), (2, 16368, 1e-6)])
def test_rmsnorm(ops, dtype, T, H, eps):
    x = rnd(T, H, dtype=dtype, seed=1, scale=3.0)
    w = (1 + 0.1 * torch.randn(H)).to(dtype).cuda()
    y = ops.rmsnorm(x, w, eps)
    xf = x.float()
    ref = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps) * w.float()
    torch.testing.assert_close(y.float(), ref, **tol(dtype))
    # with a residual: the carried sum is the rounded sum; the norm is of the unrounded one
    res = rnd(T, H, dtype=dtype, seed=2, scale=3.0)
    res_before = res.clone()
    y2 = ops.rmsnorm(x, w, eps, residual=res)
    s = x.float() + res_before.float()
    assert torch.equal(res, s.to(dtype))
    ref2 = s * torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + eps) * w.float()
    torch.testing.assert_close(y2.float(), ref2, **tol(dtype))


def test_rmsnorm_float32_residual_with_bfloat16_rows(ops):
    """The residual carried in float32: started from x exactly, then sums are not rounded."""
    x = rnd(6, 200, dtype=torch.bfloat16, seed=1)
    w = (1 + 0.1 * torch.randn(200)).bfloat16().cuda()
    y, res = ops.rmsnorm(x, w, 1e-6, start_residual=True)
    assert res.dtype == torch.float32 and torch.equal(res, x.float())
    torch.testing.assert_close(y.float(), ops.rmsnorm(x, w, 1e-6).float(), rtol=0, atol=0)
    x2 = rnd(6, 200, dtype=torch.bfloat16, seed=2)
    y2 = ops.rmsnorm(x2, w, 1e-6, residual=res)
    s = x.float() + x2.float()
    assert torch.equal(res, s)
    ref = s * torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + 1e-6) * w.float()
    torch.testing.assert_close(y2.float(), ref, **tol(torch.bfloat16))
    # the residual in the rows' own type: it starts as x itself, and a sum is rounded when it is stored
    y3, res3 = ops.rmsnorm(x, w, 1e-6, start_residual=True, residual_float32=False)
    assert res3 is x and torch.equal(y3, y)
    before = x.clone()
    y4 = ops.rmsnorm(x2, w, 1e-6, residual=res3)
    assert torch.equal(res3, (before.float() + x2.float()).bfloat16())
    torch.testing.assert_close(y4.float(), ref, **tol(torch.bfloat16))


def test_rmsnorm_float32_weight_with_bfloat16_rows(ops):
    x = rnd(4, 96, dtype=torch.bfloat16)
    w = (1 + 0.1 * torch.randn(96)).cuda()
    y = ops.rmsnorm(x, w, 1e-6)
    xf = x.float()
    ref = (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6)).bfloat16().float() * w
    torch.testing.assert_close(y.float(), ref, **tol(torch.bfloat16))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,I", [(1, 112), (33, 1001), (64, 12288)])
def test_silu_mul(ops, dtype, T, I):
    gu = rnd(T, 2 * I, dtype=dtype, seed=3, scale=2.0)
    out = ops.silu_mul(gu)
    g, u = gu[:, :I].float(), gu[:, I:].float()
    torch.testing.assert_close(out.float(), torch.nn.functional.silu(g) * u, **tol(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,N,K", [(1, 301, 80), (7, 389, 96), (65, 130, 1000), (128, 256, 512), (3, 1000, 4104)])
def test_linear(ops, dtype, M, N, K):
    x = rnd(M, K, dtype=dtype, seed=4)
    w = rnd(N, K, dtype=dtype, seed=5, scale=K ** -0.5)
    b = rnd(N, dtype=dtype, seed=6)
    ref = x.double() @ w.double().T
    t = dict(rtol=1e-5, atol=2e-5) if dtype == torch.float32 else tol(dtype)
    torch.testing.assert_close(ops.linear(x, w).double(), ref, **t)
    torch.testing.assert_close(ops.linear(x, w, b).double(), ref + b.double(), **t)
    if dtype == torch.bfloat16:
        # float32 output from bfloat16 inputs (the logits): only the accumulation rounds
        torch.testing.assert_close(ops.linear(x, w, out_dtype=torch.float32).double(), ref, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("residual_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("norm_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,H,N", [(1, 4096, 6144), (8, 4096, 1536), (16, 1024, 389), (5, 96, 80), (16, 12288, 512), (7, 5120, 4096),
                                   (3, 72, 40), (16, 1000, 24), (12, 2056, 130)])      # widths that end inside a tile of 16
def test_products_that_take_over_the_addition_and_the_norm(ops, M, H, N, norm_dtype, residual_dtype):
    """``linear(x, w, add_to=AddTo(residual, norm weight, eps))`` of few rows adds its result to the residual stream
    in its own kernel and leaves the sum times the norm's weight, rounded, and the tiles' shares of the rows' sums
    of squares (``Summed``); what is left of the norm, the scaling of the rows, is done by the product that reads
    ``Normed(summed)``, on its finished sums. Both against the same steps in float64: residual += x w1^T;
    y = rmsnorm(residual) w2^T (plain and gated)."""
    K1 = 256
    x = rnd(M, K1, dtype=torch.bfloat16, seed=31)
    w1 = rnd(H, K1, dtype=torch.bfloat16, seed=32, scale=K1 ** -0.5)
    residual = rnd(M, H, dtype=residual_dtype, seed=33)
    before = residual.clone()
    norm_w = (1 + 0.1 * torch.randn(H)).to(norm_dtype).cuda()
    w2 = rnd(N, H, dtype=torch.bfloat16, seed=34, scale=H ** -0.5)
    w3 = rnd(2 * (N // 2), H, dtype=torch.bfloat16, seed=35, scale=H ** -0.5)
    bias = rnd(N, dtype=torch.bfloat16, seed=37)
    eps = 1e-5
    summed = ops.linear(x, w1, add_to=ops.AddTo(residual, norm_w, eps))
    assert isinstance(summed, ops.Summed) and summed.residual is residual and summed.norm_weight is norm_w
    want_sum = before.double() + x.double() @ w1.double().T
    torch.testing.assert_close(residual.double(), want_sum, **(dict(rtol=1e-5, atol=1e-5) if residual_dtype == torch.float32 else tol(torch.bfloat16)))
    torch.testing.assert_close(summed.weighted.double(), want_sum * norm_w.double(), **tol(torch.bfloat16))
    assert summed.squares.shape == (M, (H + 15) // 16)
    torch.testing.assert_close(summed.squares.double().sum(-1), want_sum.pow(2).sum(-1), rtol=1e-4, atol=1e-4)
    torch.testing.assert_close(summed.squares[:, 3].double(), want_sum[:, 48:64].pow(2).sum(-1), rtol=1e-4, atol=1e-4)
    # the scaling left to the products that read it
    normed = ops.Normed(summed)
    scale = torch.rsqrt(want_sum.pow(2).mean(-1, keepdim=True) + eps)
    want_normed = want_sum * scale * norm_w.double()
    torch.testing.assert_close(normed.tensor().double(), want_normed, **tol(torch.bfloat16))
    # (the products are compared with products of the weighted sum as it was rounded, scaled afterwards: what is left
    # is the order of the sums)
    rows = summed.weighted.double()
    y = ops.linear(normed, w2, bias)
    torch.testing.assert_close(y.double(), rows @ w2.double().T * scale + bias.double(), **tol(torch.bfloat16))
    torch.testing.assert_close(y.double(), want_normed @ w2.double().T + bias.double(), rtol=3e-2, atol=3e-2)
    g = rows @ w3.double().T * scale
    half = w3.shape[0] // 2
    torch.testing.assert_close(ops.gated_linear(normed, w3).double(),
                               torch.nn.functional.silu(g[:, :half]) * g[:, half:], **tol(torch.bfloat16))
    # and one product that does both: the scaling of its rows and the addition of its result
    res2 = rnd(M, N, dtype=residual_dtype, seed=36)
    before2 = res2.clone()
    next_w = (1 + 0.1 * torch.randn(N)).to(norm_dtype).cuda()
    both = ops.linear(normed, w2, add_to=ops.AddTo(res2, next_w, eps))
    assert isinstance(both, ops.Summed)
    torch.testing.assert_close(both.weighted.double(), (before2.double() + rows @ w2.double().T * scale) * next_w.double(),
                               **tol(torch.bfloat16))
    # switched off, the same calls give tensors and leave the residual alone
    backend = ops.backend()
    backend.fuse_norms = False
    try:
        res3 = before.clone()
        plain = ops.linear(x, w1, add_to=ops.AddTo(res3, norm_w, eps))
        assert isinstance(plain, torch.Tensor) and torch.equal(res3, before)
        torch.testing.assert_close(plain.double(), x.double() @ w1.double().T, **tol(torch.bfloat16))
        torch.testing.assert_close(ops.linear(normed, w2).double(), want_normed @ w2.double().T, rtol=3e-2, atol=3e-2)
    finally:
        backend.fuse_norms = True


@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (8, 1000, 12288), (16, 389, 96), (17, 301, 80), (33, 6144, 1024),
                                   (48, 50, 2048), (64, 151936, 256), (64, 4096, 12288)])
def test_skinny_linear_bfloat16(ops, M, N, K):
    """Few rows in bfloat16 (a decoding step): own MFMA kernel, K split over waves."""
    x = rnd(M, K, dtype=torch.bfloat16, seed=14)
    w = rnd(N, K, dtype=torch.bfloat16, seed=15, scale=K ** -0.5)
    ref = x.double() @ w.double().T
    torch.testing.assert_close(ops.linear(x, w, out_dtype=torch.float32).double(), ref, rtol=1e-4, atol=2e-4)
    torch.testing.assert_close(ops.linear(x, w).double(), ref, **tol(torch.bfloat16))
    # inside a HIP graph no library is called: the own kernel also takes 17 to 64 rows with bfloat16 output
    backend = ops.backend()
    backend.own_kernels_only = True
    try:
        torch.testing.assert_close(ops.linear(x, w).double(), ref, **tol(torch.bfloat16))
    finally:
        backend.own_kernels_only = False
    # a row's result does not depend on how many other rows there are, beyond the rounding of the float sums
    # (the number of waves that split K changes with the number of rows)
    if M > 1:
        torch.testing.assert_close(ops.linear(x[:1].contiguous(), w, out_dtype=torch.float32),
                                   ops.linear(x, w, out_dtype=torch.float32)[:1], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("M,N,K", [
    # every way the kernel for up to 16 rows cuts the work: one or two tiles of 16 outputs per block, 4 or 8 waves
    (1, 6144, 264), (2, 5000, 4096), (5, 7168, 72), (8, 6100, 1032), (12, 5120, 520), (16, 151936, 64), (9, 10240, 40),
    (16, 16, 8), (3, 17, 25608),
    # x too large for LDS at once, up to 256 tiles: it comes in pieces (K off 256: the others go by lines)
    (16, 4000, 12296), (7, 272, 12288), (11, 4096, 25608),
    # x too large for LDS at once and more than 256 tiles: two pieces, every tile walked over twice
    (16, 7168, 5128), (10, 5136, 8200), (5, 4112, 17416),
    # K a multiple of 256: by lines
    (11, 4096, 25600), (16, 7168, 5120), (5, 4112, 17408),
])
def test_few_rows_linear_bfloat16_in_all_its_variants(ops, M, N, K):
    x = rnd(M, K, dtype=torch.bfloat16, seed=34)
    w = rnd(N, K, dtype=torch.bfloat16, seed=35, scale=K ** -0.5)
    b = rnd(N, dtype=torch.bfloat16, seed=36)
    ref = x.double() @ w.double().T
    torch.testing.assert_close(ops.linear(x, w, out_dtype=torch.float32).double(), ref, rtol=1e-4, atol=2e-4)
    torch.testing.assert_close(ops.linear(x, w, b).double(), ref + b.double(), **tol(torch.bfloat16))
    # the same call twice gives the same bits: the sums are added in a fixed order
    assert torch.equal(ops.linear(x, w, out_dtype=torch.float32), ops.linear(x, w, out_dtype=torch.float32))


@pytest.mark.parametrize("M,N,K", [
    # one tile a block: of 4 rows, of 16, the last one cut off; a K of one piece, of part of the waves, of steps that do not come out even
    (1, 4, 8), (3, 20, 40), (16, 1020, 520), (5, 1036, 1000), (2, 4096, 3592), (9, 4092, 4608), (16, 512, 9728),
    # several tiles a block, even and not, and blocks at the end whose last tile lies beyond the matrix
    (1, 4100, 264), (7, 6144, 3584), (16, 8200, 2560), (4, 9732, 1544), (3, 20484, 72),
    # x beside w, and just not (LDS)
    (8, 4096, 12288), (6, 3076, 16392), (4, 4092, 18440),
    # a residual of more than 256 tiles: x beside w in LDS and not, and one row of many columns
    (4, 5136, 4104), (8, 4112, 17416), (1, 4100, 20488),
    # chunks of whole lines: one tile a block and two, ends inside a tile, as few chunks as the ring has places and fewer, the
    # fewest outputs at every bound of rows
    (1, 4096, 2048), (3, 4100, 2816), (16, 6148, 3072), (5, 8196, 2048), (8, 2560, 2304), (12, 2048, 4352), (16, 16388, 2304),
    # a round of blocks and a bit: by lines with a residual only, and where x is too large or K small; K of 8,192
    (8, 8448, 2304), (16, 9220, 3072), (16, 11264, 4096), (2, 10000, 2048), (4, 5120, 8192), (5, 4100, 8192),
])
def test_tiles_of_few_rows_products(ops, M, N, K):
    """Plain, activated, gated, with rows that lack their scales and added to a residual (bounds: float32 sums of K products of
    size K^-1/2; one rounding to 8 bits, of values up to 8 where a residual is added)."""
    b = ops.backend()
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=71), rnd(2 * N, K, dtype=torch.bfloat16, seed=72, scale=K ** -0.5)
    bias, squares, eps = rnd(2 * N, dtype=torch.bfloat16, seed=73), rnd(M, 270, seed=74).abs() + 0.5, 1e-6
    both = x.double() @ w.double().T
    plain, wn = both[:, :N], w[:N].contiguous()
    b.own_kernels_only = True
    try:
        torch.testing.assert_close(ops.linear(x, wn, out_dtype=torch.float32).double(), plain, rtol=1e-4, atol=2e-4)
        torch.testing.assert_close(ops.linear(x, wn, bias[:N].contiguous()).double(), plain + bias[:N].double(), **tol(torch.bfloat16))
        gated = lambda g, u: g * torch.sigmoid(g) * u
        if 2 * N * K < 120_000_000:
            torch.testing.assert_close(ops.gated_linear(x, w).double(), gated(plain, both[:, N:]), **tol(torch.bfloat16))
    finally:
        b.own_kernels_only = False
    scale = torch.rsqrt(squares.double().sum(-1, keepdim=True) / K + eps)
    out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    b.fused_linear(x, wn, bias[:N].contiguous(), out, row_scales=(squares, eps))
    torch.testing.assert_close(out.double(), plain * scale + bias[:N].double(), **tol(torch.bfloat16))
    b.fused_linear(x, w, bias, out, gated=True, row_scales=(squares, eps))
    want = both * scale + bias.double()
    torch.testing.assert_close(out.double(), gated(want[:, :N], want[:, N:]), **tol(torch.bfloat16))
    for dtype in DTYPES:
        residual, next_w = rnd(M, N, dtype=dtype, seed=75), rnd(N, dtype=dtype, seed=76, scale=0.1) + 1
        want = residual.double() + plain + bias[:N].double()
        left = torch.empty(M, (N + 15) // 16, device="cuda")
        b.fused_linear(x, wn, bias[:N].contiguous(), None, residual=residual, sum_out=out, ss_out=left, next_w=next_w)
        torch.testing.assert_close(residual.double(), want, **(dict(rtol=1e-4, atol=2e-4) if dtype == torch.float32 else tol(dtype)))
        torch.testing.assert_close(out.double(), want * next_w.double(), **tol(torch.bfloat16))
        tiles = torch.nn.functional.pad(want, (0, -N % 16)).view(M, -1, 16).pow(2).sum(-1)
        torch.testing.assert_close(left.double(), tiles, rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("M,N,K,rows", [(1, 1024, 1024, 4), (16, 1024, 3072, 4), (5, 40, 1032, 4), (3, 1028, 1080, 8), (16, 2040, 2048, 8), (9, 2052, 1096, 12),
                                        (2, 2556, 2056, 12), (7, 3084, 1048, 16), (4, 2560, 2048, 16), (8, 2564, 2304, 16), (1, 1024, 1016, 16)])
def test_sums_of_squares_by_the_blocks_outputs(ops, M, N, K, rows):
    """A product that is added to the residual stream leaves its blocks' shares of the rows' sums of squares, of fewer than 16 outputs where these
    give every unit a block; the norm and the product that read them (bounds: float32 sums of K products of size K^-1/2, one rounding to 8 bits)."""
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=81), rnd(N, K, dtype=torch.bfloat16, seed=82, scale=K ** -0.5)
    w2 = rnd(64, N, dtype=torch.bfloat16, seed=85, scale=N ** -0.5) if N % 8 == 0 else None
    for dtype in DTYPES:
        residual, next_w = rnd(M, N, dtype=dtype, seed=83), rnd(N, dtype=torch.float32, seed=84, scale=0.1) + 1
        want = residual.double() + x.double() @ w.double().T
        summed = ops.linear(x, w, add_to=ops.AddTo(residual, next_w, 1e-6))
        assert isinstance(summed, ops.Summed) and summed.squares.shape == (M, -(-N // rows))
        torch.testing.assert_close(residual.double(), want, **(dict(rtol=1e-4, atol=2e-4) if dtype == torch.float32 else tol(dtype)))
        torch.testing.assert_close(summed.weighted.double(), want * next_w.double(), **tol(torch.bfloat16))
        tiles = torch.nn.functional.pad(want, (0, -N % rows)).view(M, -1, rows).pow(2).sum(-1)
        torch.testing.assert_close(summed.squares.double(), tiles, rtol=1e-3, atol=1e-3)
        scale = torch.rsqrt(want.pow(2).mean(-1, keepdim=True) + 1e-6)
        torch.testing.assert_close(ops.Normed(summed).tensor().double(), want * next_w.double() * scale, **tol(torch.bfloat16))
        if w2 is not None:
            torch.testing.assert_close(ops.linear(ops.Normed(summed), w2).double(), summed.weighted.double() @ w2.double().T * scale, **tol(torch.bfloat16))


@pytest.mark.parametrize("M", [1, 2, 3, 7, 8, 9])
@pytest.mark.parametrize("N,K", [(2560, 2048), (4100, 2304), (9000, 2560)])
def test_few_rows_by_lines_whose_other_rows_are_not_there(ops, M, N, K):
    """Up to 8 rows only the waves that have some bring x: against float64, and where more rows take the same tiles, the bits that these give."""
    x, w = rnd(16, K, dtype=torch.bfloat16, seed=86), rnd(N, K, dtype=torch.bfloat16, seed=87, scale=K ** -0.5)
    b = ops.backend()
    rows, more = torch.empty(M, N, dtype=torch.bfloat16, device="cuda"), torch.empty(16, N, dtype=torch.bfloat16, device="cuda")
    b.fused_linear(x[:M].contiguous(), w, None, rows)
    b.fused_linear(x, w, None, more)
    torch.testing.assert_close(rows.double(), x[:M].double() @ w.double().T, **tol(torch.bfloat16))
    if M < 9 and N == 2560:
        assert torch.equal(rows, more[:M])


@pytest.mark.parametrize("M", [4, 7, 8, 11, 16])
@pytest.mark.parametrize("N,K", [(1025, 2048), (1532, 4352), (2044, 5120), (2048, 6144)])
def test_few_rows_by_lines_of_eight_rows_of_weights(ops, M, N, K):
    """Blocks of 8 outputs, whose other columns are not there: against float64, with a bias; values that are no numbers in a row of x or
    of w reach their outputs alone."""
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=108), rnd(N, K, dtype=torch.bfloat16, seed=109, scale=K ** -0.5)
    bias = rnd(N, dtype=torch.bfloat16, seed=110)
    want = x.double() @ w.double().T
    torch.testing.assert_close(ops.linear(x, w).double(), want, **tol(torch.bfloat16))
    torch.testing.assert_close(ops.linear(x, w, bias).double(), want + bias.double(), **tol(torch.bfloat16))
    x[1, 3], w[9, 5], w[N - 1, 7] = float("nan"), float("inf"), float("nan")
    out, hit = ops.linear(x, w), torch.zeros(M, N, dtype=torch.bool, device="cuda")
    hit[1], hit[:, 9], hit[:, N - 1] = True, True, True
    assert not torch.isfinite(out[hit]).any()
    torch.testing.assert_close(out[~hit].double(), want[~hit], **tol(torch.bfloat16))


@pytest.mark.parametrize("M,N,K", [(4, 2048, 2048), (16, 2048, 2048), (5, 1536, 3072), (6, 1536, 3072), (11, 1040, 3072), (12, 1040, 3072), (7, 1040, 4096),
                                   (8, 1040, 4096), (12, 1025, 6144), (6, 2044, 5120), (6, 2048, 2816), (12, 1040, 2816), (16, 1028, 4608), (15, 1028, 4608),
                                   (1, 2560, 2048), (7, 3068, 2048), (2, 2940, 2560), (3, 2940, 2560), (7, 3072, 2048)])
def test_products_that_scale_their_rows_on_either_side_of_the_blocks_of_eight(ops, M, N, K):
    """A reader of a norm, by tiles and by blocks of 8 outputs (1,025 to 2,048 outputs) or of 16: against float64 (bound: one rounding to 8 bits)."""
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=151), rnd(N, K, dtype=torch.bfloat16, seed=152, scale=K ** -0.5)
    squares = rnd(M, K // 16, seed=153).abs() + 0.1
    scale = torch.rsqrt(squares.double().sum(-1, keepdim=True) / K + 1e-6)
    got = ops.linear(ops.Normed(ops.Summed(x, squares, rnd(M, K, seed=154), rnd(K, dtype=torch.bfloat16, seed=155), 1e-6)), w)
    torch.testing.assert_close(got.double(), x.double() @ w.double().T * scale, rtol=1.6e-2, atol=1.6e-2 * float(scale.max()))


@pytest.mark.parametrize("M,N,K", [(1, 2560, 2048), (7, 3068, 2048), (8, 2560, 2048), (1, 3072, 2048), (3, 2816, 4096), (3, 2816, 2304)])
def test_float_results_of_few_rows_by_tiles_and_by_lines(ops, M, N, K):
    """On either side of where they go by lines: against float64 (bound: float sums of K products of size K^-1/2), and alike for equal rows of w."""
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=156), rnd(N, K, dtype=torch.bfloat16, seed=157, scale=K ** -0.5)
    w[N - 1], w[N // 2] = w[1], w[1]
    got = ops.linear(x, w, out_dtype=torch.float32)
    torch.testing.assert_close(got.double(), x.double() @ w.double().T, rtol=1e-4, atol=2e-4)
    if K % 2048 == 0:
        assert torch.equal(got[:, 1], got[:, N - 1]) and torch.equal(got[:, 1], got[:, N // 2])


@pytest.mark.parametrize("M,I,K", [(1, 112, 80), (5, 1001, 96), (16, 12288, 4096), (17, 160, 96), (64, 300, 1024),
                                   (4, 17408, 136), (16, 25600, 72), (13, 25000, 264), (16, 9000, 5120), (15, 520, 5384)])
def test_gated_linear(ops, M, I, K):
    """silu(x Wg^T) * (x Wu^T): the fused kernel for few rows, the two-kernel way for many; float32 as well."""
    for dtype in DTYPES:
        x = rnd(M, K, dtype=dtype, seed=24)
        w = rnd(2 * I, K, dtype=dtype, seed=25, scale=K ** -0.5)
        g, u = x.double() @ w[:I].double().T, x.double() @ w[I:].double().T
        ref = g * torch.sigmoid(g) * u
        t = dict(rtol=1e-5, atol=2e-5) if dtype == torch.float32 else tol(dtype)
        torch.testing.assert_close(ops.gated_linear(x, w).double(), ref, **t)
        backend = ops.backend()
        backend.own_kernels_only = True                      # as inside a HIP graph: fused up to 64 rows
        try:
            torch.testing.assert_close(ops.gated_linear(x, w).double(), ref, **t)
        finally:
            backend.own_kernels_only = False


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("M,N,K", [(1, 8, 128), (255, 136, 256), (256, 256, 128), (257, 1000, 384), (300, 264, 1152), (2049, 520, 256), (4400, 2200, 128), (700, 9728, 640)])
def test_gates_and_activations_of_many_rows(ops, M, N, K, gated):
    """Edges of the tiles of 256 x 256, two pieces of 64 columns and more, one tile a block and several, more than eight tiles of rows, every gate with and
    without biases and every activation: against float64. A float sum of K products is off by K^(1/2) roundings of 2^-24 of its size at most,
    which rounding the result to 8 bits (2^-9 of it) hides. Nothing behind the last row is written."""
    b = ops.backend()
    x = rnd(M, K, dtype=torch.bfloat16, seed=131)
    w = rnd((2 if gated else 1) * N, K, dtype=torch.bfloat16, seed=132, scale=2 * K ** -0.5)
    sums = x.double() @ w.double().T
    bias = rnd(2 * N, dtype=torch.bfloat16, seed=133)
    for act in range(3):
        for with_bias in ((False, True) if gated else (False,)):
            gate = ops.Gate(act, 1.5, 1.702, 1.0)
            out = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device="cuda")
            b._call("nhv_gemm_phases_bf16", ops._ptr(x), ops._ptr(w), ops._ptr(bias if with_bias else None), ops._ptr(out), M, N, K, int(gated),
                    *gate.args(), ops._stream())
            z = sums + bias.double() if with_bias else sums
            g = z[:, :N]
            if gated and act == 2:
                g = g.clamp(max=1.5)
                want = g * torch.sigmoid(1.702 * g) * (z[:, N:].clamp(-1.5, 1.5) + 1.0)
            else:
                silu, gelu = g * torch.sigmoid(g), torch.nn.functional.gelu(g, approximate="tanh")
                want = (silu, gelu, g.clamp(min=0).square())[act] * (z[:, N:] if gated else 1.0)
            torch.testing.assert_close(out[:M].double(), want, rtol=2.0 ** -8, atol=1e-4)
            assert bool((out[M] == 7.0).all())


def test_many_rows_take_the_kernel_that_gates_them_where_it_pays(ops):
    """By the share of the tiles' rounds that are outputs; a bias goes with it; a step of the same rows gives the same bits."""
    pays = ops.backend().lib.nhv_gemm_phases_pays
    assert [pays(*size) for size in ((2048, 12288, 4096, 1), (1866, 12288, 4096, 1), (600, 12288, 4096, 1), (97, 12288, 4096, 1), (2048, 12288, 4096 + 64, 1),
                                     (2048, 12284, 4096, 1), (1925, 6144, 2048, 0), (1000, 6144, 2048, 0))] == [1, 1, 0, 0, 0, 0, 1, 0]
    x, w = rnd(1300, 512, dtype=torch.bfloat16, seed=134), rnd(2 * 8192, 512, dtype=torch.bfloat16, seed=135, scale=512 ** -0.5)
    bias = rnd(2 * 8192, dtype=torch.bfloat16, seed=136)
    sums = x.double() @ w.double().T
    # (against float64: gates of rounded rows are off by more, 2^-9 (|h'(g) g u| + 2 |y|), 0.1 at the largest of these)
    bound = dict(rtol=2.0 ** -8, atol=1e-4)
    for gate, b in (("silu", None), ("gelu_tanh", bias), (ops.Gate(2, 7.0, 1.702, 1.0), bias)):
        assert ops.backend().gated_linear(x, w, torch.empty(1300, 8192, dtype=torch.bfloat16, device="cuda"), ops.gate_of(gate), b)
        y = ops.gated_linear(x, w, gate, b)
        g, u = (sums if b is None else sums + b.double()).chunk(2, dim=1)
        if gate == "silu":
            want = g * torch.sigmoid(g) * u
        elif gate == "gelu_tanh":
            want = torch.nn.functional.gelu(g, approximate="tanh") * u
        else:
            want = g.clamp(max=7.0) * torch.sigmoid(1.702 * g.clamp(max=7.0)) * (u.clamp(-7.0, 7.0) + 1.0)
        torch.testing.assert_close(y.double(), want, **bound)
        assert torch.equal(y, ops.gated_linear(x, w, gate, b))
    torch.testing.assert_close(ops.activated_linear(x, w[:8192], "gelu_tanh").double(), torch.nn.functional.gelu(sums[:, :8192], approximate="tanh"), **bound)


@pytest.mark.parametrize("N,K", [(1, 1), (17, 130), (48, 16), (130, 20), (65, 516), (300, 2064), (16400, 36), (24000, 7), (2500, 68), (2100, 331)])
def test_float32_linear_in_all_its_tiles(ops, N, K):
    """Every tile that the number of rows and columns can choose, K below and beyond eight blocks of 16, ends inside a block of
    16, rows off 16-byte boundaries: against float64 (a sum of K products of size 1 is off by K^(1/2) roundings of its own size,
    K^(1/2), at most), and the same row bit for bit whatever the number of rows."""
    x, w, b = rnd(520, K, seed=51), rnd(N, K, seed=52), rnd(N, seed=53)
    ref = x.double() @ w.double().T + b.double()
    last = None
    for M in (520, 65, 64, 33, 17, 16, 1):
        y = ops.linear(x[520 - M:].contiguous(), w, b)
        torch.testing.assert_close(y.double(), ref[520 - M:], rtol=1e-6, atol=K * 2.0 ** -23 + 1e-6)
        assert last is None or torch.equal(y, last[-M:])
        last = y


@pytest.mark.parametrize("M,N,K,taken", [(300, 8000, 192, 1), (300, 7970, 224, 1), (417, 6144, 544, 1), (517, 6100, 288, 1),
                                         (517, 6144, 1024, 1), (577, 4130, 256, 1),
                                         (1000, 6268, 352, 1), (1049, 3072, 1056, 1), (1100, 14400, 256, 1), (128, 20000, 256, 1),
                                         (300, 8000, 160, 0), (517, 7168, 288, 0), (300, 8000, 1200, 0), (545, 4130, 256, 0), (150, 2000, 256, 0)])
def test_float32_linear_in_tiles_of_128_rows(ops, M, N, K, taken):
    """Tiles of 128 x 128 in one round of blocks, two and four, and sizes that just do not take them: segments of one piece of 32 columns and
    of several, rows and columns that end inside a tile, plain and gated, an infinite row: the rows that few rows alone give, bit for bit."""
    big = ops.backend().lib.nhv_gemm_float32_big_tiles
    assert big(M, N, K, 0) == taken and big(M, N // 2, K, 1) == taken
    x, w, b = rnd(M, K, seed=141), rnd(N, K, seed=142), rnd(N, seed=143)
    x[M - 3, K // 2] = float("inf")
    y, g = ops.linear(x, w[:N], b[:N]), ops.gated_linear(x, w[:N], "silu", b[:N])
    for rows in (slice(0, 16), slice(M - 5, M), slice(124, 134)):
        some = x[rows].contiguous()
        for got, want in ((y[rows], ops.linear(some, w[:N], b[:N])), (g[rows], ops.act_mul(ops.linear(some, w[:N]), "silu", b[:N]))):
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(1.5, 2.5, 3.5), want.nan_to_num(1.5, 2.5, 3.5))


@pytest.mark.parametrize("M,N,K", [(1090, 4100, 64), (1090, 4100, 70), (545, 4130, 256), (577, 4130, 33), (321, 4096, 1000), (190, 6150, 256), (200, 3080, 288),
                                   (250, 2047, 768), (700, 3072, 1024)])
def test_float32_linear_in_tiles_of_64_rows(ops, M, N, K):
    """Tiles of 64 x 64 and 64 x 128, whole pieces of 32 columns and not, plain and gated (halved or not): the rows that few rows alone give, bit for bit."""
    x, w, b = rnd(M, K, seed=121), rnd(2 * N, K, seed=122), rnd(2 * N, seed=123)
    y, g = ops.linear(x, w[:N], b[:N]), ops.gated_linear(x, w, "silu", b)
    for rows in (slice(0, 16), slice(M - 5, M), slice(60, 70)):
        some = x[rows].contiguous()
        assert torch.equal(y[rows], ops.linear(some, w[:N], b[:N]))
        assert torch.equal(g[rows], ops.act_mul(ops.linear(some, w), "silu", b))


@pytest.mark.parametrize("M,N,K", [(1, 64, 512), (6, 1024, 3072), (16, 1024, 544), (16, 2560, 3104), (17, 72, 1312), (65, 1000, 2080), (150, 2056, 2048),
                                   (517, 1024, 768), (256, 1536, 1024), (49, 8200, 2048), (193, 6104, 2080), (65, 16360, 2048)])
def test_float32_parts_through_the_norm(ops, M, N, K):
    """The norm that adds up a product's parts gives the bits of the norm that takes the finished product, and leaves the same sums in the
    residual; so does the kernel that only adds them up. With sums beyond 2^96 and entries that are no numbers as well."""
    norm_w = 1 + 0.1 * rnd(N, seed=133)
    for odd in (False, True):
        x, w, r = rnd(M, K, seed=131), rnd(N, K, seed=132), rnd(M, N, seed=134)
        if odd:
            x[M // 2] *= 1e16
            w[N // 3] *= 1e16
            w[5, K - 1], x[0, K // 2] = float("inf"), float("nan") if M > 1 else 1.0
        rows = ops.linear(x, w)
        want_r = r.clone()
        want = ops.rmsnorm(rows, norm_w, 1e-6, residual=want_r)
        made = ops.linear(x, w, add_to=ops.AddTo(r, norm_w, 1e-6, None, takes_parts=True))
        assert isinstance(made, ops.Parts) and made.shape == (M, N)
        same = lambda a, b: torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(1.5, 2.5, 3.5), b.nan_to_num(1.5, 2.5, 3.5))
        assert same(made.tensor(), rows)
        got = ops.rmsnorm(made, norm_w, 1e-6, residual=r)
        assert same(got, want) and same(r, want_r)


def test_which_float32_products_come_in_parts(ops):
    """For the norm that adds to the residual alone, few outputs, whole pieces of 32 columns on 16-byte boundaries; and only where what is
    saved by cutting K outweighs the parts' way to the norm (517 rows of 2,048 outputs: of 512 columns in parts 1.2 times as long, of 2,048 0.74 times)."""
    def parts(M, N, K, off=0, takes=True):
        x, w = rnd(M * K + off, seed=1)[off:].view(M, K), rnd(N, K, seed=2)
        return isinstance(ops.linear(x, w, add_to=ops.AddTo(rnd(M, N, seed=3), rnd(N, seed=4), 1e-6, None, takes_parts=takes)), ops.Parts)

    assert parts(6, 1024, 2048) and parts(16, 2048, 768) and parts(16, 2560, 3072) and parts(17, 4096, 8192)
    assert parts(517, 2048, 2048) and parts(256, 1536, 1024) and parts(150, 2056, 1536)
    assert not parts(517, 2048, 512) and not parts(257, 1280, 1024) and not parts(17, 4096, 4096) and not parts(16, 2560, 1312) and not parts(16, 2048, 512)
    assert not parts(6, 4096, 2048) and not parts(1500, 2048, 2048) and not parts(6, 1024, 500) and not parts(6, 1024, 256)
    assert not parts(6, 1024, 2048, off=1) and not parts(6, 1024, 2048, takes=False)
    assert not isinstance(ops.linear(rnd(6, 1024, seed=1), rnd(1024, 1024, seed=2), parts=True), ops.Parts)


@pytest.mark.parametrize("M,N,K", [(1, 16, 33), (6, 40, 300), (30, 600, 1024), (70, 4096, 64), (130, 9000, 96)])
def test_float32_linear_at_the_ends_of_its_range(ops, M, N, K):
    """Infinities, no numbers, numbers that round up to infinity in 8 bits and numbers whose parts are tiny: in their own rows and
    columns what float multiply-adds give, everywhere else what the product without them gives, bit for bit."""
    x, w = rnd(M, K, seed=61), rnd(N, K, seed=62)
    clean = ops.linear(x, w)
    odd, columns = [0] if M == 1 else [0, M // 2, M - 1], [0, 3, N // 2, N - 1]
    top = 3.4e38                                             # (rounds to infinity in 8 bits)
    x[odd[0], K // 3] = top
    if M > 1:
        x[odd[1], 0], x[odd[2], K - 1] = float("inf"), float("nan")
    w[columns[0], K // 2], w[columns[1], 1], w[columns[2], K - 1] = float("-inf"), float("nan"), top
    w[columns[3]] *= 1e-30
    y = ops.linear(x, w)
    rows, cols = [i for i in range(M) if i not in odd], [i for i in range(N) if i not in columns]
    assert torch.equal(y[rows][:, cols], clean[rows][:, cols])
    want = x.double().cpu() @ w.double().cpu().T
    want = torch.where(want.abs() > 3.4028235e38, torch.sign(want) * math.inf, want)
    got = y.double().cpu()
    sure = (want.abs() < 3.3e38) | ~torch.isfinite(want) | (want.abs() > 3.5e38)
    for row, column in ((odd[0], columns[2]), (odd[0], columns[0]), (odd[len(odd) // 2], columns[2])):
        sure[row, column] = False                            # a term that overflows beside an infinite or another large one
    assert torch.equal(torch.isnan(got)[sure], torch.isnan(want)[sure]) and torch.equal(torch.isinf(got)[sure], torch.isinf(want)[sure])
    near = sure & torch.isfinite(want)
    # K roundings of the sum of the terms' sizes at most
    size = x.double().cpu().abs() @ w.double().cpu().abs().T
    assert ((got - want).abs()[near] <= (K * 2.0 ** -24 * size)[near]).all()


@pytest.mark.parametrize("M,N,K", [(1, 16, 32), (6, 512, 96), (70, 300, 64), (130, 2000, 36)])
@pytest.mark.parametrize("of_x,of_w", [(1e-34, 1.0), (1e-36, 1.0), (1.0, 1e-37), (1e-40, 1.0), (1e-36, 1e36), (1e-38, 1e20), (1e-19, 1e-19), (1e-21, 1e-20)])
def test_float32_linear_of_tiny_entries(ops, M, N, K, of_x, of_w):
    """Operands down to the denormals, one of them and both, lose none of their bits (bound: an output's roundings, six an inner
    block of 32 and a few at the ends, of the sum of its terms' sizes, and the last place of a denormal), and the same gated."""
    x, w = rnd(M, K, seed=111) * of_x, rnd(2 * N, K, seed=112) * of_w
    want = x.double().cpu() @ w.double().cpu().T
    size = x.double().cpu().abs() @ w.double().cpu().abs().T
    bound = (6 * -(-K // 32) + 10) * 2.0 ** -24 * size + 2.0 ** -149
    assert ((ops.linear(x, w).double().cpu() - want).abs() <= bound).all()
    if 1e-2 < of_x * of_w < 1e2:
        g, u = want.split(N, dim=1)
        got = ops.gated_linear(x, w).double().cpu()
        # (SiLU's slope is at most 1.1, its own float arithmetic a few roundings)
        slack = 1.1 * bound[:, :N] * u.abs() + torch.nn.functional.silu(g).abs() * bound[:, N:] + 2.0 ** -21 * (g * u).abs() + 2.0 ** -60
        assert ((got - torch.nn.functional.silu(g) * u).abs() <= slack).all()


def test_float32_linear_of_entries_whose_smallest_parts_are_largest(ops):
    """1 + 2^-8 - 2^-17, whose products lose most by the part products that are not made (2^-24 of a term), and its negative."""
    a = 1 + 2.0 ** -8 - 2.0 ** -17
    for M, N, K in ((1, 16, 32), (5, 40, 256), (70, 300, 1024)):
        x, w = torch.full((M, K), a, device="cuda"), torch.full((N, K), a, device="cuda")
        w[N // 2:] *= -1
        want = x.double().cpu() @ w.double().cpu().T
        assert ((ops.linear(x, w).double().cpu() - want).abs() <= (6 * -(-K // 32) + 10) * 2.0 ** -24 * want.abs()).all()


@pytest.mark.parametrize("M,N,K", [(1, 40, 33), (7, 300, 1000), (40, 600, 260), (150, 4100, 70)])
def test_float32_linear_of_sums_that_the_parts_cannot_hold(ops, M, N, K):
    """Sums beyond 2^96, rows and columns with several infinities or entries that are no numbers side by side, and entries beyond 2^112:
    what float64 gives (bound: K roundings of the sum of the terms' sizes), plain and gated, in every row and column."""
    x, w = rnd(M, K, seed=115), rnd(2 * N, K, seed=116)
    x[::3] *= 1e15
    w[::2] *= 1e16
    w[1::4] *= 1e20
    if M > 6:
        x[2, K // 2], x[3, 1], x[3, K - 1], x[5] = float("nan"), float("inf"), float("-inf"), 2e34
    w[3, K - 1], w[6, 0], w[7, 5], w[11] = float("nan"), float("inf"), float("inf"), -3e35
    want = x.double().cpu() @ w.double().cpu().T
    size = x.double().cpu().abs().nan_to_num(0, 0, 0) @ w.double().cpu().abs().nan_to_num(0, 0, 0).T
    got = ops.linear(x, w).double().cpu()
    sure = torch.isnan(want) | (size < 3e38)                 # (terms or sums on the way beyond the largest float: either way)
    assert torch.equal(torch.isnan(got)[sure], torch.isnan(want)[sure]) and torch.equal(torch.isposinf(got)[sure], torch.isposinf(want)[sure])
    near = torch.isfinite(want) & sure
    assert near.any() and ((got - want).abs()[near] <= (K * 2.0 ** -24 * size + 2.0 ** -149)[near]).all()
    gated, packed = ops.gated_linear(x, w), ops.act_mul(ops.linear(x, w), "silu")
    assert torch.equal(gated.isnan(), packed.isnan()) and torch.equal(gated.nan_to_num(1.5, 2.5, 3.5), packed.nan_to_num(1.5, 2.5, 3.5))


@pytest.mark.parametrize("M,N,K", [(1, 151936, 1024), (6, 1024, 3072), (517, 4096, 1024)])
def test_a_row_that_is_no_number_does_not_hold_up_a_float32_product(ops, M, N, K):
    """Twice the product's time and 20 us at most (each output of such a row by one thread took 3 to 14 times as long)."""
    x, w = rnd(M, K, seed=117), rnd(N, K, seed=118)

    def shortest():
        times = []
        for _ in range(12):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            ops.linear(x, w)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    clean = shortest()
    x[M // 2, K // 3] = float("nan")
    assert shortest() <= 2 * clean + 0.02


@pytest.mark.parametrize("N,K", [(1, 7), (40, 516), (520, 1024), (3072, 64), (9000, 36)])
def test_float32_gated_linear_in_all_its_tiles(ops, N, K):
    """A gate of two products in one kernel: the bits of the packed product and the gate's own kernel, for every tile that the
    sizes can choose, with and without biases, and with an infinite row."""
    x, w, b = rnd(300, K, seed=64), rnd(2 * N, K, seed=65), rnd(2 * N, seed=66)
    for M in (300, 130, 70, 40, 17, 16, 3):
        rows = x[300 - M:].contiguous()
        if M == 40:
            rows[M // 2, K // 2] = float("inf")
        for gate, bias in (("silu", None), (ops.Gate(2, 3.0, 1.702, 1.0), b)):
            packed = ops.linear(rows, w)
            got, want = ops.gated_linear(rows, w, gate, bias), ops.act_mul(packed, gate, bias)
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(1.5, 2.5, 3.5), want.nan_to_num(1.5, 2.5, 3.5)), (M, gate)


@pytest.mark.parametrize("M,N,K,fused", [
    (1, 3072, 1024, True), (6, 2560, 2560, True), (300, 512, 4096, True), (16, 512, 512, True), (70, 1000, 1001, True),
    (1, 512, 8192, False), (17, 1024, 3072, False), (16, 2048, 2048, False), (1, 1000, 1001, False),
])
def test_which_float32_gates_are_made_in_the_products_kernel(ops, M, N, K, fused):
    """Not where the packed product's blocks are twice as many and the chip is not full: the same bits either way."""
    x, w = rnd(M, K, seed=67), rnd(2 * N, K, seed=68)
    out = torch.full((M, N), float("nan"), device="cuda")
    assert ops.backend().gated_linear(x, w, out) == fused
    want = ops.act_mul(ops.linear(x, w), "silu")
    assert torch.equal(ops.gated_linear(x, w), want)
    by_product = ops.backend().lib.nhv_gemm_float32_gated
    assert by_product(ops._ptr(x), ops._ptr(w), ops._ptr(None), ops._ptr(out), M, N, K, *ops.Gate().args(), ops._stream()) == 0
    assert torch.equal(out, want)


def test_linear_rows_do_not_depend_on_the_batch_in_float32(ops):
    x = rnd(70, 200, seed=7)
    w = rnd(150, 200, seed=8)
    full = ops.linear(x, w)
    for rows in ([0], [69], [3, 4, 5], list(range(64, 70))):
        part = ops.linear(x[rows].contiguous(), w)
        assert torch.equal(part, full[rows])


def _rope_reference(x, positions, base, rot):
    inv = 1.0 / (base ** (torch.arange(0, rot, 2, dtype=torch.float32) / rot))
    ang = positions.float()[:, None] * inv[None, :]
    cos, sin = ang.cos()[:, None, :], ang.sin()[:, None, :]
    x1, x2 = x[..., :rot // 2], x[..., rot // 2:rot]
    return torch.cat((x1 * cos - x2 * sin, x2 * cos + x1 * sin, x[..., rot:]), dim=-1)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("Hq,Hkv,D,rot,norm,bias", [
    (4, 2, 16, 16, True, False), (6, 1, 32, 32, True, False), (5, 5, 48, 48, False, True),
    (3, 3, 80, 40, True, False), (32, 8, 128, 128, True, False), (2, 1, 256, 0, False, False),
])
def test_qk_rope_write(ops, dtype, Hq, Hkv, D, rot, norm, bias):
    from nanohybrid_vlm_amd.parts.positions import RotaryEmbedding
    T, page, pages, eps, base = 23, 8, 9, 1e-5, 10000.0
    width = (Hq + 2 * Hkv) * D
    qkv = rnd(T, width, dtype=dtype, seed=9, scale=2.0)
    b = rnd(width, dtype=dtype, seed=10) if bias else None
    qw = (1 + 0.1 * torch.randn(D)).to(dtype).cuda() if norm else None
    kw = (1 + 0.1 * torch.randn(D)).to(dtype).cuda() if norm else None
    table = RotaryEmbedding(rot, 300, base).table.cuda() if rot else None
    positions = torch.randint(0, 300, (T,), dtype=torch.int32, device="cuda")
    slots = torch.randperm(page * pages)[:T].to(torch.int32).cuda()
    slots[5] = -1                                     # a token that is not stored
    k_cache = torch.zeros(pages, page, Hkv, D, dtype=dtype, device="cuda")
    v_cache = torch.zeros_like(k_cache)
    q = ops.qk_rope_write(qkv, b, qw, kw, eps, table, positions, slots, k_cache, v_cache, Hq, Hkv, D)

    x = qkv.float()
    if bias:
        x = (x + b.float()).to(dtype).float()
    qr = x[:, :Hq * D].reshape(T, Hq, D)
    kr = x[:, Hq * D:(Hq + Hkv) * D].reshape(T, Hkv, D)
    vr = x[:, (Hq + Hkv) * D:].reshape(T, Hkv, D)
    if norm:
        qr = qr * torch.rsqrt(qr.pow(2).mean(-1, keepdim=True) + eps) * qw.float()
        kr = kr * torch.rsqrt(kr.pow(2).mean(-1, keepdim=True) + eps) * kw.float()
    if rot:
        qr = _rope_reference(qr.cpu(), positions.cpu(), base, rot).cuda()
        kr = _rope_reference(kr.cpu(), positions.cpu(), base, rot).cuda()
    t = tol(dtype) if dtype == torch.bfloat16 else dict(rtol=1e-5, atol=2e-5)
    torch.testing.assert_close(q.float(), qr, **t)
    stored = slots >= 0
    kf, vf = k_cache.view(-1, Hkv, D), v_cache.view(-1, Hkv, D)
    torch.testing.assert_close(kf[slots[stored].long()].float(), kr[stored], **t)
    assert torch.equal(vf[slots[stored].long()], vr[stored].to(dtype))      # values are only moved
    untouched = torch.ones(page * pages, dtype=torch.bool, device="cuda")
    untouched[slots[stored].long()] = False
    assert not kf[untouched].any() and not vf[untouched].any()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("Hq,Hkv,D,rot,axes", [(4, 2, 16, 16, 2), (3, 1, 48, 24, 3), (8, 2, 128, 128, 2), (2, 2, 32, 8, 1)])
def test_qk_rope_write_over_several_position_axes(ops, dtype, Hq, Hkv, D, rot, axes):
    """positions [axes, T]: pair j of a head turns by the angle that the table holds at the coordinate of axis
    pair_axes[j] (without pair_axes: of the first axis)."""
    from nanohybrid_vlm_amd.parts.positions import RotaryEmbedding
    T, base = 19, 10000.0
    width = (Hq + 2 * Hkv) * D
    qkv = rnd(T, width, dtype=dtype, seed=19, scale=2.0)
    table = RotaryEmbedding(rot, 200, base).table.cuda()
    positions = torch.randint(0, 200, (axes, T), dtype=torch.int32, device="cuda")
    pair_axes = (torch.arange(rot // 2) * 5 % axes).to(torch.int32).cuda() if axes > 1 else None
    slots = torch.arange(T, dtype=torch.int32, device="cuda")
    k_cache = torch.zeros(4, 8, Hkv, D, dtype=dtype, device="cuda")
    v_cache = torch.zeros_like(k_cache)
    q = ops.qk_rope_write(qkv, None, None, None, 0.0, table, positions, slots, k_cache, v_cache, Hq, Hkv, D, pair_axes=pair_axes)
    # the angle of pair j at position p is p * base^(-2j/rot): here p differs from pair to pair
    j = torch.arange(rot // 2)
    at = positions.cpu().long()[pair_axes.cpu().long() if pair_axes is not None else torch.zeros(rot // 2, dtype=torch.long)].T   # [T, rot/2]
    ang = at.double() * (base ** (-2.0 * j.double() / rot))
    cos, sin = ang.cos()[:, None, :], ang.sin()[:, None, :]

    def turned(x):
        x = x.double().cpu()
        x1, x2 = x[..., :rot // 2], x[..., rot // 2:rot]
        return torch.cat((x1 * cos - x2 * sin, x2 * cos + x1 * sin, x[..., rot:]), -1)

    x = qkv.float()
    t = dict(rtol=1.6e-2, atol=1.6e-2) if dtype == torch.bfloat16 else dict(rtol=1e-4, atol=1e-4)
    torch.testing.assert_close(q.double().cpu(), turned(x[:, :Hq * D].reshape(T, Hq, D)), **t)
    torch.testing.assert_close(k_cache.view(-1, Hkv, D)[:T].double().cpu(), turned(x[:, Hq * D:(Hq + Hkv) * D].reshape(T, Hkv, D)), **t)


@pytest.mark.parametrize("dtype", DTYPES)
def test_embed_scale_and_soft_cap(ops, dtype):
    table = rnd(301, 200, dtype=dtype, seed=21)
    ids = torch.randint(0, 301, (13,), dtype=torch.int32, device="cuda")
    assert torch.equal(ops.embed(ids, table, 1.0), table[ids.long()])
    assert torch.equal(ops.embed(ids, table, 1.75), (table[ids.long()].float() * 1.75).to(dtype))
    logits = rnd(7, 1001, seed=22, scale=6.0)
    want = 4.0 * torch.tanh(logits / 4.0)
    assert ops.soft_cap_(logits, 4.0) is logits
    torch.testing.assert_close(logits, want, rtol=1e-5, atol=1e-5)
    assert float(logits.abs().max()) <= 4.0


def _paged_setup(dtype, lens, q_lens, Hq, Hkv, D, page, seed=0, scale=1.0):
    """Requests with ``lens`` keys each whose last ``q_lens`` tokens are this step's queries; pages handed out
    in a shuffled order. Returns the pieces for ops.paged_attention and the dense keys and values."""
    from nanohybrid_vlm_amd.native.ops import AttentionBatch
    g = torch.Generator().manual_seed(seed)
    B = len(lens)
    n_pages = sum(-(-n // page) for n in lens) + 3
    order = torch.randperm(n_pages, generator=g).tolist()
    k_cache = torch.full((n_pages, page, Hkv, D), float("nan"), dtype=dtype)
    v_cache = torch.full((n_pages, page, Hkv, D), float("nan"), dtype=dtype)
    width = max(-(-n // page) for n in lens)
    bt = torch.full((B, width), -1, dtype=torch.int32)
    ks, vs, qs, token_req, positions = [], [], [], [], []
    for r, (n, nq) in enumerate(zip(lens, q_lens)):
        k = (torch.randn(n, Hkv, D, generator=g) * scale).to(dtype)
        v = torch.randn(n, Hkv, D, generator=g).to(dtype)
        ks.append(k)
        vs.append(v)
        for lp in range(-(-n // page)):
            pid = order.pop()
            bt[r, lp] = pid
            m = min(page, n - lp * page)
            k_cache[pid, :m] = k[lp * page:lp * page + m]
            v_cache[pid, :m] = v[lp * page:lp * page + m]
        qs.append((torch.randn(nq, Hq, D, generator=g) * scale).to(dtype))
        token_req += [r] * nq
        positions += list(range(n - nq, n))
    cu = torch.tensor([0] + list(torch.tensor(q_lens).cumsum(0)), dtype=torch.int32)
    batch = AttentionBatch(num_tokens=sum(q_lens), num_requests=B,
                           token_req=torch.tensor(token_req, dtype=torch.int32).cuda(),
                           positions=torch.tensor(positions, dtype=torch.int32).cuda(),
                           cu_seqlens_q=cu.cuda(), context_lens=torch.tensor(lens, dtype=torch.int32).cuda(),
                           max_q_len=max(q_lens), max_context_len=max(lens))
    return torch.cat(qs).cuda(), k_cache.cuda(), v_cache.cuda(), batch, bt.cuda(), ks, vs, qs


def _attention_reference(qs, ks, vs, lens, q_lens, scale, window):
    outs = []
    for q, k, v, n, nq in zip(qs, ks, vs, lens, q_lens):
        Hq, Hkv = q.shape[1], k.shape[1]
        kk = k.double().repeat_interleave(Hq // Hkv, dim=1)
        vv = v.double().repeat_interleave(Hq // Hkv, dim=1)
        s = torch.einsum("qhd,khd->hqk", q.double(), kk) * scale
        qpos = torch.arange(n - nq, n)[:, None]
        kpos = torch.arange(n)[None, :]
        ok = kpos <= qpos
        if window:
            ok &= kpos > qpos - window
        s = s.masked_fill(~ok[None], float("-inf"))
        outs.append(torch.einsum("hqk,khd->qhd", torch.softmax(s, dim=-1), vv))
    return torch.cat(outs)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("Hq,Hkv,D,page,window", [
    (4, 2, 16, 4, None), (6, 1, 32, 8, None), (5, 5, 48, 7, None), (3, 1, 80, 16, 9),
    (8, 2, 128, 64, None), (32, 8, 128, 256, None), (2, 2, 64, 5, 64), (7, 7, 112, 3, None),
])
def test_paged_attention(ops, dtype, Hq, Hkv, D, page, window):
    # whole prompts, portions with earlier keys, single decoded tokens, a length of one, page edges
    lens = [1, 64, 65, 300, 17, 128, 5, 257]
    q_lens = [1, 64, 1, 43, 2, 1, 5, 1]
    scale = D ** -0.5
    q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(dtype, lens, q_lens, Hq, Hkv, D, page, seed=11, scale=1.5)
    out = ops.paged_attention(q, kc, vc, batch, bt, scale, window)
    ref = _attention_reference(qs, ks, vs, lens, q_lens, scale, window)
    t = dict(rtol=1e-5, atol=1e-5) if dtype == torch.float32 else tol(dtype)
    torch.testing.assert_close(out.double().cpu(), ref, **t)


@pytest.mark.parametrize("Hq,Hkv,D,E,page,reach,cap,sinks,slopes,gated", [
    (2, 2, 64, 64, 16, None, None, None, False, False), (3, 1, 16, 64, 5, ("window", 70), None, "each", False, True),
    (8, 1, 128, 128, 64, ("chunk", 50), 3.0, "one", False, False), (34, 2, 48, 192, 256, None, None, None, True, True),
    (4, 4, 256, 256, 7, ("window", 1), None, "each", True, False), (2, 1, 240, 128, 8, ("chunk", 64), None, None, False, False),
])
def test_float32_attention_of_whole_tiles(ops, Hq, Hkv, D, E, page, reach, cap, sinks, slopes, gated):
    """The kernel on the float matrix cores with every option: row tiles that end inside a token's heads, rounds of eight blocks of
    keys and their rests, against float64; the same bits for a token alone; and a value that is no number, which reaches the
    rows that read it and no others."""
    import dataclasses
    lens, q_lens = [1, 64, 65, 300, 17, 513, 5, 257], [1, 64, 1, 43, 2, 30, 5, 1]
    q, kc, _, batch, bt, ks, _, qs = _paged_setup(torch.float32, lens, q_lens, Hq, Hkv, D, page, seed=61)
    g = torch.Generator().manual_seed(62)
    vc = torch.full((*kc.shape[:3], E), float("nan"))
    vs = [torch.randn(n, Hkv, E, generator=g) for n in lens]
    for r, v in enumerate(vs):
        for p in range(len(v)):
            vc[bt[r, p // page], p % page] = v[p]
    vc = vc.cuda()
    rows = torch.randn(q.shape[0], Hq + 3, generator=g)
    slope = torch.rand(Hq, generator=g) * 0.1 if slopes else None
    sink = {None: None, "one": 0.7, "each": torch.randn(Hq, generator=g)}[sinks]
    options = {"softcap": cap, "slopes": None if slope is None else slope.cuda(), "sink": sink.cuda() if sinks == "each" else sink,
               "gate": (rows.cuda(), 2) if gated else None, **({reach[0]: reach[1]} if reach else {})}
    out = ops.paged_attention(q, kc, vc, batch, bt, D ** -0.5, **options)
    want, reads, at = [], [], 0
    for r, (n, nq) in enumerate(zip(lens, q_lens)):
        group = Hq // Hkv
        pos, key = torch.arange(n - nq, n)[:, None], torch.arange(n)[None]
        ok = key <= pos
        if reach:
            ok &= key > pos - reach[1] if reach[0] == "window" else key // reach[1] == pos // reach[1]
        s = torch.einsum("qhd,khd->hqk", qs[r].double(), ks[r].double().repeat_interleave(group, 1)) * D ** -0.5
        s = cap * torch.tanh(s / cap) if cap else s
        s = s - slope.double()[:, None, None] * (pos - key) if slopes else s
        s = s.masked_fill(~ok, float("-inf"))
        if sinks:
            s = torch.cat((s, torch.as_tensor(sink, dtype=torch.float64).expand(Hq)[:, None, None].expand(Hq, nq, 1)), -1)
        o = torch.einsum("hqk,khd->qhd", torch.softmax(s, -1)[..., :n], vs[r].double().repeat_interleave(group, 1))
        want.append(o * torch.sigmoid(rows[at:at + nq, 2:2 + Hq].double())[..., None] if gated else o)
        reads.append(ok[:, n - 2:n - 1].any(-1) if n > 1 else torch.zeros(nq, dtype=torch.bool))
        at += nq
    torch.testing.assert_close(out.double().cpu(), torch.cat(want), rtol=1e-5, atol=1e-5)
    last = dataclasses.replace(batch, num_tokens=1, num_requests=1, token_req=torch.zeros(1, dtype=torch.int32, device="cuda"),
                               positions=batch.positions[-1:], cu_seqlens_q=torch.tensor([0, 1], dtype=torch.int32, device="cuda"),
                               context_lens=batch.context_lens[-1:], max_q_len=1)
    if gated:
        options["gate"] = (rows[-1:].cuda(), 2)
    alone = ops.paged_attention(q[-1:].contiguous(), kc, vc, last, bt[7:8].contiguous(), D ** -0.5, **options)
    assert torch.equal(alone, out[-1:])
    if gated:
        options["gate"] = (rows.cuda(), 2)
    for r, n in enumerate(lens):
        if n > 1:
            vc[bt[r, (n - 2) // page], (n - 2) % page] = float("inf")
    spoilt = ops.paged_attention(q, kc, vc, batch, bt, D ** -0.5, **options)
    hit = torch.cat(reads)
    assert not torch.isfinite(spoilt[hit.cuda()]).any()
    torch.testing.assert_close(spoilt[~hit.cuda()], out[~hit.cuda()], rtol=1e-5, atol=1e-5)

@pytest.mark.parametrize("sink", [None, 0.3])
@pytest.mark.parametrize("dtype,D", [(torch.float32, 64), (torch.float32, 192), (torch.float32, 20)])
def test_attention_hides_no_score_that_is_no_number(ops, dtype, D, sink):
    """A key or a query that is no number: what reads it is no number either, also where it is the only one of its block of keys
    (33, 65 and 257 keys) or where a sink would stand in for the rest; everything else keeps its bits."""
    lens, q_lens = [33, 65, 257, 1, 40, 300], [33, 1, 2, 1, 7, 60]
    q, kc, vc, batch, bt, *_ = _paged_setup(dtype, lens, q_lens, 4, 2, D, 16, seed=63)
    options = {} if sink is None else {"sink": sink}
    clean = ops.paged_attention(q, kc, vc, batch, bt, D ** -0.5, **options)
    assert torch.isfinite(clean).all()
    bad = kc.clone()
    for r, n in enumerate(lens):
        bad[bt[r, (n - 1) // 16], (n - 1) % 16, 1, D // 2] = float("nan")       # the last key, read by the last token's heads 2 and 3
    out = ops.paged_attention(q, bad, vc, batch, bt, D ** -0.5, **options)
    hit = torch.zeros(q.shape[:2], dtype=torch.bool, device="cuda")
    hit[batch.cu_seqlens_q[1:].long() - 1, 2:] = True
    assert torch.isnan(out[hit]).all() and torch.equal(out[~hit], clean[~hit])
    spoilt, hit = q.clone(), torch.zeros_like(hit)
    for t in (0, 32, 33, 34, 36, 44, 80):
        spoilt[t, 3, 0], hit[t, 3] = float("nan"), True
    out = ops.paged_attention(spoilt, kc, vc, batch, bt, D ** -0.5, **options)
    assert torch.isnan(out[hit]).all() and torch.equal(out[~hit], clean[~hit])


@pytest.mark.parametrize("Hq,Hkv,D,page,reach", [(16, 8, 128, 16, {}), (16, 8, 128, 256, {"window": 70}), (4, 4, 64, 7, {}),
                                                 (16, 1, 64, 5, {"chunk": 50}), (6, 2, 128, 8, {"window": 33, "softcap": 3.0})])
def test_float32_attention_of_one_tile_of_rows(ops, Hq, Hkv, D, page, reach):
    """Where 16 rows hold a request's portion, a block of keys is asked for at once, the first one before it is known which of its
    keys are read: the bits of the same tokens among longer portions, also beside keys and values that are no numbers and pages
    that no request holds (-1 in the table)."""
    import dataclasses
    lens = [1, 31, 32, 33, 64, 255, 256, 257, 300, 530, 40]
    q_lens = [1, 1, 2, 1, 1, 1, 1, 1, 1, 1, 40]
    q, kc, vc, batch, bt, *_ = _paged_setup(torch.float32, lens, q_lens, Hq, Hkv, D, page, seed=95)
    vc[bt[8, 3 // page], 3 % page, 0, 1] = float("inf")
    vc[bt[9, 500 // page], 500 % page, Hkv - 1, 2] = float("nan")
    kc[bt[7, 256 // page], 256 % page, 0, 3] = float("nan")
    together = ops.paged_attention(q, kc, vc, batch, bt, D ** -0.5, **reach)
    n = len(lens) - 1
    few = dataclasses.replace(batch, num_tokens=n + 1, num_requests=n, token_req=batch.token_req[:n + 1], positions=batch.positions[:n + 1],
                              cu_seqlens_q=batch.cu_seqlens_q[:n + 1], context_lens=batch.context_lens[:n], max_q_len=2, max_context_len=530)
    if 2 * (Hq // Hkv) > 16:                   # (only single tokens are one tile)
        few = dataclasses.replace(few, num_tokens=2, num_requests=2, token_req=batch.token_req[:2], positions=batch.positions[:2],
                                  cu_seqlens_q=batch.cu_seqlens_q[:3], context_lens=batch.context_lens[:2], max_q_len=1, max_context_len=31)
        n = 1
    alone = ops.paged_attention(q[:few.num_tokens].contiguous(), kc, vc, few, bt[:few.num_requests].contiguous(), D ** -0.5, **reach)
    assert torch.equal(alone.view(torch.int32), together[:few.num_tokens].view(torch.int32))


def test_float32_attention_of_rows_that_begin_anywhere(ops):
    """Queries that begin 4, 8 and 12 bytes off a boundary of 16: the bits of those that begin on one."""
    lens, q_lens = [33, 257, 70], [33, 1, 20]
    q, kc, vc, batch, bt, *_ = _paged_setup(torch.float32, lens, q_lens, 4, 2, 64, 16, seed=88)
    want = ops.paged_attention(q, kc, vc, batch, bt, 0.125)
    for off in (1, 2, 3):
        rows = torch.empty(q.numel() + off, device="cuda")[off:].view_as(q).copy_(q)
        assert rows.data_ptr() % 16 == 4 * off and torch.equal(ops.paged_attention(rows, kc, vc, batch, bt, 0.125), want)


@pytest.mark.parametrize("Hq,Hkv,D,page,window", [
    (4, 2, 16, 4, None), (6, 1, 32, 8, None), (5, 5, 48, 7, None), (3, 1, 80, 16, 9), (8, 2, 128, 64, None),
    (32, 8, 128, 256, None), (16, 1, 64, 5, 70), (7, 7, 112, 3, None), (2, 1, 256, 32, None), (12, 2, 96, 16, 300),
])
def test_decode_attention_bfloat16(ops, Hq, Hkv, D, page, window):
    """Single tokens of several requests in bfloat16: the split-key kernel (lengths around the edges of
    tiles of 16, of splits and of pages)."""
    lens = [1, 15, 16, 17, 31, 32, 33, 64, 65, 300, 257, 1000, 1024, 1025]
    q_lens = [1] * len(lens)
    scale = D ** -0.5
    q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, lens, q_lens, Hq, Hkv, D, page, seed=21, scale=1.5)
    out = ops.paged_attention(q, kc, vc, batch, bt, scale, window)
    ref = _attention_reference(qs, ks, vs, lens, q_lens, scale, window)
    torch.testing.assert_close(out.double().cpu(), ref, **tol(torch.bfloat16))
    # the same tokens one at a time (other split lengths are chosen then): same result up to rounding
    one = ops.paged_attention(q[9:10].contiguous(), kc, vc,
                              type(batch)(1, 1, torch.zeros(1, dtype=torch.int32).cuda(), batch.positions[9:10].contiguous(),
                                          torch.tensor([0, 1], dtype=torch.int32).cuda(), batch.context_lens[9:10].contiguous(),
                                          1, lens[9]), bt[9:10].contiguous(), scale, window)
    torch.testing.assert_close(one.float(), out[9:10].float(), rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("Hq,Hkv,D,page,window", [(4, 2, 64, 16, None), (8, 1, 128, 64, 40), (2, 2, 256, 32, None), (3, 1, 48, 7, 700)])
def test_decode_attention_over_infinite_values(ops, Hq, Hkv, D, page, window):
    """The last key's value, and the first one's that a window leaves, hold an infinity each: the entry is infinite for the heads
    that read it, whatever keys beside it in its round are masked, and no other entry changes a bit."""
    lens = [1, 2, 15, 31, 32, 33, 65, 257, 300, 500, 1000, 1025]
    q, kc, vc, batch, bt, *_ = _paged_setup(torch.bfloat16, lens, [1] * len(lens), Hq, Hkv, D, page, seed=87, scale=0.4)
    scale, bad = D ** -0.5, vc.clone()
    clean = ops.paged_attention(q, kc, vc, batch, bt, scale, window)
    for r, n in enumerate(lens):
        lo = max(0, n - window) if window else 0
        bad[bt[r, (n - 1) // page], (n - 1) % page, Hkv - 1, 3] = float("inf")
        bad[bt[r, lo // page], lo % page, Hkv - 1, D - 1] = float("-inf")
    out = ops.paged_attention(q, kc, bad, batch, bt, scale, window)
    mine = slice(Hq // Hkv * (Hkv - 1), Hq)
    assert (out[:, mine, 3] == float("inf")).all() and (out[:, mine, D - 1] == float("-inf")).all()
    out[:, mine, 3], out[:, mine, D - 1] = clean[:, mine, 3], clean[:, mine, D - 1]
    assert torch.equal(out, clean)


@pytest.mark.parametrize("Hq,Hkv,D,page,window", [(8, 2, 128, 256, None), (6, 1, 48, 16, None), (4, 4, 64, 64, 3000)])
def test_decode_attention_of_few_tokens_over_many_splits(ops, Hq, Hkv, D, page, window):
    """One or two requests of thousands of keys: the splits that the engine chooses, which four waves merge."""
    for lens in ([5000], [4097, 2100]):
        q_lens = [1] * len(lens)
        scale = D ** -0.5
        q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, lens, q_lens, Hq, Hkv, D, page, seed=27, scale=1.5)
        out = ops.paged_attention(q, kc, vc, batch, bt, scale, window)
        ref = _attention_reference(qs, ks, vs, lens, q_lens, scale, window)
        torch.testing.assert_close(out.double().cpu(), ref, **tol(torch.bfloat16))


@pytest.mark.parametrize("T,Hq,Hkv,D,page,window", [(16, 4, 2, 128, 16, None), (64, 2, 1, 64, 8, None), (63, 2, 2, 128, 32, 40),
                                                    (41, 1, 1, 256, 16, None), (30, 1, 1, 32, 7, None), (300, 1, 1, 16, 64, None)])
def test_decode_attention_of_many_tokens_with_one_split(ops, T, Hq, Hkv, D, page, window):
    """Blocks take the tokens in the order of their numbers of keys (equal ones among them), up to 64, and as they come beyond;
    contexts from one key to some rounds of all waves; every token's result is its own."""
    g = torch.Generator().manual_seed(81)
    lens = torch.randint(1, 700 if T < 100 else 90, (T,), generator=g).tolist()
    lens[0], lens[-1], lens[T // 2] = 1, max(lens), max(lens)
    scale = D ** -0.5
    q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, lens, [1] * T, Hq, Hkv, D, page, seed=82)
    out = ops.paged_attention(q, kc, vc, batch, bt, scale, window)
    ref = _attention_reference(qs, ks, vs, lens, [1] * T, scale, window)
    torch.testing.assert_close(out.double().cpu(), ref, **tol(torch.bfloat16))


@pytest.mark.parametrize("T,n_splits", [(32, 1), (33, 3), (44, 3), (45, 2), (52, 2), (53, 1)])
def test_decode_attention_of_a_little_over_one_block_a_unit(ops, T, n_splits):
    """257 to 416 blocks: three splits, two, and one on either side, of contexts that end in any of them."""
    from nanohybrid_vlm_amd.native.ops import decode_split_length
    assert -(-700 // decode_split_length(T * 8, 700, 700, 0)) == n_splits
    g = torch.Generator().manual_seed(83)
    lens = [700, 1] + torch.randint(2, 700, (T - 2,), generator=g).tolist()
    q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, lens, [1] * T, 8, 8, 64, 16, seed=84)
    out = ops.paged_attention(q, kc, vc, batch, bt, 0.125, None)
    torch.testing.assert_close(out.double().cpu(), _attention_reference(qs, ks, vs, lens, [1] * T, 0.125, None), **tol(torch.bfloat16))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("W", [8, 1000, 2048, 2056, 4104, 8192, 8200, 50])
def test_depth_mix_in_all_its_widths(ops, dtype, W):
    """Rows in one, two and four passes of 2,048 entries and what does not fit them; layers that read none to five results."""
    T, eps = 5, 1e-5
    x, gain = rnd(T, W, seed=91), torch.tensor(0.7, device="cuda")
    results = torch.zeros(8, T, W, device="cuda")
    want = [x.double()]
    for i in range(6):
        a, b, c = (rnd(T, W, dtype=dtype, seed=92 + 3 * i + j) for j in range(3))
        wa, wb, w = rnd(W, seed=93, scale=0.1) + 1, rnd(W, seed=94, scale=0.1) + 1, rnd(i + 2, seed=95 + i, scale=0.5)
        pair = i % 2 == 1
        first = ops.NormedPairMean(a, wa, c, wb, eps) if pair else a
        got, normed = ops.depth_mix(x, first, None if i == 2 else b, results, i, w, gain=gain, eps=eps)
        unit = lambda t: t / torch.sqrt(t.pow(2).mean(-1, keepdim=True) + eps)
        add = 0.5 * (unit(a.double()) * wa + unit(c.double()) * wb) if pair else a.double()
        want.append(x.double() + add + (0 if i == 2 else b.double()))
        ref = sum(w[j].double() * want[j] for j in range(i + 2))
        torch.testing.assert_close(got.double(), ref, rtol=1e-5, atol=1e-5)
        torch.testing.assert_close(results[i + 1].double(), want[-1], rtol=1e-5, atol=1e-5)
        torch.testing.assert_close(normed.double(), unit(ref) * 0.7, **tol(dtype))
        x = got


@pytest.mark.parametrize("rows_dtype,result_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("W", [4, 1000, 1028, 2048, 2052, 4100, 8192, 8196, 16384, 16388, 1001])
def test_sandwich_step_in_all_its_widths(ops, W, rows_dtype, result_dtype):
    """One, two and four passes, full and not, and what is not read four at a time; both halves and either alone."""
    T, ea, eb = 3, 1e-5, 1e-3
    x, y, wa, wb = rnd(T, W, seed=81), rnd(T, W, dtype=result_dtype, seed=82), rnd(W, seed=83) + 1, rnd(W, seed=84) + 1
    unit = lambda t, eps: t / torch.sqrt(t.pow(2).mean(-1, keepdim=True) + eps)
    want = x.double() + unit(y.double(), eb) * wb.double()
    stream = x.clone()
    read = ops.sandwich_step(stream, read=(wa, ea), rows_dtype=rows_dtype)
    torch.testing.assert_close(read.double(), unit(x.double(), ea) * wa.double(), **tol(rows_dtype))
    assert torch.equal(stream, x)
    both = ops.sandwich_step(stream, add=(y, wb, eb), read=(wa, ea), rows_dtype=rows_dtype)
    torch.testing.assert_close(stream.double(), want, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(both.double(), unit(want, ea) * wa.double(), **tol(rows_dtype))
    alone = x.clone()
    assert ops.sandwich_step(alone, add=(y, wb, eb)) is None
    assert torch.equal(alone, stream)
    # a token's result is its own, whatever the batch
    one = x[1:2].clone()
    assert torch.equal(ops.sandwich_step(one, add=(y[1:2].contiguous(), wb, eb), read=(wa, ea), rows_dtype=rows_dtype)[0], both[1])


@pytest.mark.parametrize("D,split_len,n_splits,window", [
    (128, 64, 5, None),      # one wave, four splits a lane
    (128, 64, 20, None),     # four waves, four splits a lane; the last waves' splits lie past every position but one
    (128, 64, 40, 900),      # four waves, eight a lane, a window that leaves the first splits out
    (128, 64, 100, None),    # four waves, sixteen a lane
    (128, 64, 140, None),    # past the at-once kernels: the kernel that loops, four waves
    (64, 128, 9, None), (256, 64, 3, None), (256, 64, 30, 500), (48, 64, 33, None), (16, 64, 70, None),
])
def test_merge_of_splits_in_all_its_forms(ops, D, split_len, n_splits, window):
    """The decode kernel called with the split length and the number of splits named: every form of the merge (one
    wave or four, 4 to 16 splits a lane, and the looping kernel), with more splits than most positions reach and the
    buffers of the splits' results full of NaN beforehand, so that a split read without having been written shows."""
    import ctypes
    from nanohybrid_vlm_amd.native.ops import _ptr, _stream
    Hq, Hkv, page = 8, 2, 64
    longest = n_splits * split_len
    lens = [longest, 1, split_len, split_len + 1, longest // 2 + 3, longest - 1, 77]
    lens = [n for n in lens if n <= longest]
    q_lens = [1] * len(lens)
    scale = D ** -0.5
    q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, lens, q_lens, Hq, Hkv, D, page, seed=61, scale=1.5)
    backend = ops.backend()
    T = len(lens)
    out = torch.full((T, Hq, D), float("nan"), dtype=torch.bfloat16, device="cuda")
    part_o = torch.full((T, Hq, n_splits, D), float("nan"), dtype=torch.float32, device="cuda")
    part_ml = torch.full((T, Hq, n_splits, 2), float("nan"), dtype=torch.float32, device="cuda")
    backend._call("nhv_decode_attention_bf16", _ptr(q), _ptr(kc), _ptr(vc), _ptr(out), _ptr(part_o), _ptr(part_ml),
                  _ptr(batch.token_req), _ptr(batch.positions), _ptr(bt), bt.shape[1], T, Hq, Hkv, page,
                  ctypes.c_float(scale), window or 0, split_len, n_splits, _stream(), lib=backend.attention_lib(D))
    ref = _attention_reference(qs, ks, vs, lens, q_lens, scale, window)
    torch.testing.assert_close(out.double().cpu(), ref, **tol(torch.bfloat16))


@pytest.mark.parametrize("D,split_len,n_splits", [(128, 64, 1), (128, 64, 5), (128, 64, 20), (64, 64, 100), (128, 64, 140), (256, 32, 3)])
@pytest.mark.parametrize("sink", [None, 0.3])
def test_merge_of_splits_hides_no_score_that_is_no_number(ops, D, split_len, n_splits, sink):
    """A key that is no number and the only one of its split, in every form of the merge, also beside a sink: the result of what
    reads it is no number; the other heads keep their bits."""
    import ctypes
    from nanohybrid_vlm_amd.native.ops import _ptr, _stream
    Hq, Hkv, page = 4, 2, 32
    lens = [n_splits * split_len] + [s * split_len + 1 for s in range(1, n_splits, 3)] + [1, 2]
    q, kc, vc, batch, bt, *_ = _paged_setup(torch.bfloat16, lens, [1] * len(lens), Hq, Hkv, D, page, seed=64)
    T, backend = len(lens), ops.backend()

    def call(keys):
        out = torch.full((T, Hq, D), 7.0, dtype=torch.bfloat16, device="cuda")
        part_o, part_ml = torch.zeros(T, Hq, n_splits, D, device="cuda"), torch.zeros(T, Hq, n_splits, 2, device="cuda")
        backend._call("nhv_decode_attention_bf16_more", _ptr(q), _ptr(keys), _ptr(vc), _ptr(out), _ptr(part_o), _ptr(part_ml),
                      _ptr(batch.token_req), _ptr(batch.positions), _ptr(bt), bt.shape[1], T, Hq, Hkv, page, ctypes.c_float(D ** -0.5), 0,
                      split_len, n_splits, ctypes.c_float(0.0), int(sink is not None), ctypes.c_float(sink or 0.0), None, None, None,
                      ctypes.c_longlong(0), _stream(), lib=backend.attention_lib(D))
        return out

    clean, bad = call(kc), kc.clone()
    for r, n in enumerate(lens):
        bad[bt[r, (n - 1) // page], (n - 1) % page, 1, 5] = float("nan")
    out = call(bad)
    assert torch.isfinite(clean).all() and torch.equal(out[:, :2], clean[:, :2]) and torch.isnan(out[:, 2:]).all()


def _decode_in_splits(ops, q, kc, vc, batch, bt, scale, window, split_len, n_splits, cap=0.0, sink=None, sinks=None, slopes=None, gate=None):
    """The decode kernel with the splits named; the buffers of the splits' results are full of NaN beforehand."""
    import ctypes
    from nanohybrid_vlm_amd.native.ops import _gate_args, _ptr, _stream
    T, Hq, D = q.shape
    out = torch.full((T, Hq, D), float("nan"), dtype=torch.bfloat16, device="cuda")
    part_o = torch.full((T, Hq, n_splits, D), float("nan"), device="cuda")
    part_ml = torch.full((T, Hq, n_splits, 2), float("nan"), device="cuda")
    ops.backend()._call("nhv_decode_attention_bf16_more", _ptr(q), _ptr(kc), _ptr(vc), _ptr(out), _ptr(part_o), _ptr(part_ml), _ptr(batch.token_req),
                        _ptr(batch.positions), _ptr(bt), bt.shape[1], T, Hq, kc.shape[2], kc.shape[1], ctypes.c_float(scale), window, split_len, n_splits,
                        ctypes.c_float(cap), int(sink is not None), ctypes.c_float(sink or 0.0), _ptr(sinks), _ptr(slopes), *_gate_args(gate), _stream(),
                        lib=ops.backend().attention_lib(D))
    return out


@pytest.mark.parametrize("options", ["cap", "sink", "sinks", "slopes", "gate", "cap sinks gate", "slopes sink gate", "cap slopes"])
@pytest.mark.parametrize("D,split_len,n_splits,window", [(64, 640, 1, 0), (128, 128, 5, 0), (64, 64, 20, 900), (128, 64, 100, 0), (128, 64, 140, 0)])
def test_options_of_decoded_tokens_over_splits(ops, options, D, split_len, n_splits, window):
    """What a layer may ask for besides, where one block writes the result and in every form of the merge."""
    Hq, Hkv = 6, 2
    longest = n_splits * split_len
    lens = [longest, 1, split_len, min(longest, split_len + 1), longest // 2 + 3]
    q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, lens, [1] * len(lens), Hq, Hkv, D, 64, seed=65, scale=1.2)
    given, scale, T = set(options.split()), D ** -0.5, len(lens)
    rows = rnd(T, Hq + 3, dtype=torch.bfloat16, seed=66)
    args = {"cap": 3.0, "sink": 0.7, "sinks": rnd(Hq, seed=67), "slopes": rnd(Hq, seed=68).abs() * 0.02, "gate": (rows, 2)}
    args = {name: value for name, value in args.items() if name in given}
    out = _decode_in_splits(ops, q, kc, vc, batch, bt, scale, window, split_len, n_splits, **args)
    heads = torch.arange(Hq) // (Hq // Hkv)
    for t, n in enumerate(lens):
        keys = torch.arange(max(0, n - window) if window else 0, n)
        s = torch.einsum("hd,khd->hk", qs[t][0].double(), ks[t].double()[keys][:, heads]) * scale
        if "cap" in given:
            s = 3.0 * torch.tanh(s / 3.0)
        if "slopes" in given:
            s = s - args["slopes"].double().cpu()[:, None] * (n - 1 - keys)[None]
        more = torch.full((Hq, 1), 0.7, dtype=torch.float64) if "sink" in given else args["sinks"].double().cpu()[:, None] if "sinks" in given else None
        p = torch.softmax(s if more is None else torch.cat([s, more], dim=1), dim=1)[:, :len(keys)]
        want = torch.einsum("hk,khd->hd", p, vs[t].double()[keys][:, heads])
        if "gate" in given:
            want = want * torch.sigmoid(rows[t, 2:2 + Hq].double().cpu())[:, None]
        torch.testing.assert_close(out[t].double().cpu(), want, **tol(torch.bfloat16))


@pytest.mark.parametrize("T,D,split_len,n_splits,window", [(16, 64, 128, 5, 0), (17, 256, 64, 4, 0), (33, 128, 32, 9, 70), (63, 64, 96, 3, -50), (64, 128, 64, 6, 0),
                                                           (64, 48, 224, 2, 0), (65, 64, 96, 3, 0), (15, 64, 96, 3, 0)])
def test_decoded_tokens_in_any_order_over_splits(ops, T, D, split_len, n_splits, window):
    """Of each split's blocks the ones with the most keys come first, from 16 to 64 tokens, and tokens without a key there have none:
    every (token, split) is done once, in whatever order the contexts come, and a token's bits are those it has alone."""
    g = torch.Generator().manual_seed(85)
    longest = split_len * n_splits
    lens = [longest, 1, split_len, split_len + 1, longest - 1] + torch.randint(1, longest + 1, (T - 5,), generator=g).tolist()
    lens = [lens[i] for i in torch.randperm(T, generator=g).tolist()]
    scale = D ** -0.5
    q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, lens, [1] * T, 2, 1, D, 16, seed=86)
    out = _decode_in_splits(ops, q, kc, vc, batch, bt, scale, window, split_len, n_splits)
    if window >= 0:
        torch.testing.assert_close(out.double().cpu(), _attention_reference(qs, ks, vs, lens, [1] * T, scale, window), **tol(torch.bfloat16))
    for t in range(0, T, 5):
        alone = type(batch)(1, 1, torch.zeros(1, dtype=torch.int32).cuda(), batch.positions[t:t + 1].contiguous(), torch.tensor([0, 1], dtype=torch.int32).cuda(),
                            batch.context_lens[t:t + 1].contiguous(), 1, lens[t])
        one = _decode_in_splits(ops, q[t:t + 1].contiguous(), kc, vc, alone, bt[t:t + 1].contiguous(), scale, window, split_len, n_splits)
        assert torch.equal(one[0], out[t]), t


def test_merge_of_splits_of_many_tokens(ops):
    """More than 1,024 (token, head) pairs with more splits than the at-once kernels take: the looping kernel with
    one wave."""
    import ctypes
    from nanohybrid_vlm_amd.native.ops import _ptr, _stream
    Hq, Hkv, D, page, split_len, n_splits = 16, 2, 128, 64, 64, 140
    lens = [8960] + [40 + 3 * i for i in range(69)]
    q_lens = [1] * len(lens)
    scale = D ** -0.5
    q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, lens, q_lens, Hq, Hkv, D, page, seed=62, scale=1.5)
    backend = ops.backend()
    T = len(lens)
    assert T * Hq > 1024
    out = torch.full((T, Hq, D), float("nan"), dtype=torch.bfloat16, device="cuda")
    part_o = torch.full((T, Hq, n_splits, D), float("nan"), dtype=torch.float32, device="cuda")
    part_ml = torch.full((T, Hq, n_splits, 2), float("nan"), dtype=torch.float32, device="cuda")
    backend._call("nhv_decode_attention_bf16", _ptr(q), _ptr(kc), _ptr(vc), _ptr(out), _ptr(part_o), _ptr(part_ml),
                  _ptr(batch.token_req), _ptr(batch.positions), _ptr(bt), bt.shape[1], T, Hq, Hkv, page,
                  ctypes.c_float(scale), 0, split_len, n_splits, _stream(), lib=backend.attention_lib(D))
    ref = _attention_reference(qs, ks, vs, lens, q_lens, scale, None)
    torch.testing.assert_close(out.double().cpu(), ref, **tol(torch.bfloat16))


@pytest.mark.parametrize("Hq,Hkv,D,page,window", [
    (4, 1, 128, 256, None), (8, 2, 64, 16, None), (6, 1, 32, 8, 100), (3, 3, 48, 5, None), (16, 1, 16, 64, None),
    (5, 1, 256, 32, None), (32, 8, 128, 64, 700),
])
def test_prefill_attention_bfloat16(ops, Hq, Hkv, D, page, window):
    """Long portions with and without earlier keys in bfloat16: the matrix-core kernel (tiles of 64 keys and of
    16 tokens; portions that end inside a tile; a single token beside them)."""
    lens = [700, 300, 64, 1500, 17, 129]
    q_lens = [300, 300, 1, 1025, 16, 65]
    scale = D ** -0.5
    q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, lens, q_lens, Hq, Hkv, D, page, seed=31, scale=1.5)
    out = ops.paged_attention(q, kc, vc, batch, bt, scale, window)
    ref = _attention_reference(qs, ks, vs, lens, q_lens, scale, window)
    torch.testing.assert_close(out.double().cpu(), ref, **tol(torch.bfloat16))


@pytest.mark.parametrize("B,new,Hq,Hkv,keys", [
    # few blocks, larger groups; many, with two row tiles a wave; groups that the other way gives several blocks
    (5, 75, 32, 8, 256), (8, 1000, 32, 8, 256), (16, 901, 32, 8, 256), (61, 100, 32, 8, 256), (61, 20, 32, 2, 256), (200, 20, 64, 4, 256),
    # many blocks of one row tile a wave, or two of which one is without any; few of groups of one beside longer portions
    (14, 50, 32, 8, None), (14, 100, 32, 8, None), (31, 33, 32, 8, None), (14, 75, 40, 8, None), (46, 20, 16, 8, None), (14, 500, 16, 8, None),
    (6, 500, 8, 8, None), (6, 20, 8, 8, 448), (8, 64, 16, 8, 448), (9, 64, 16, 8, None),
])
def test_which_short_requests_share_their_keys_out(ops, B, new, Hq, Hkv, keys):
    """Where that was measured to be the faster way for a request of a few tokens beside portions (else another 4 to 26 % slower)."""
    for D, most in ((128, keys), (64, keys), (96, None), (256, None)):
        assert ops.backend().attention_lib(D).nhv_prefill_attention_one_tile_from(B, new, Hq, Hkv) == (most or 2 ** 31 - 1)


@pytest.mark.parametrize("Hq,Hkv,D,page,portion,two,reach,cap,sinks,slopes,gated", [
    (32, 8, 128, 16, 900, True, None, None, None, False, False), (8, 2, 128, 256, 60, False, ("window", 70), None, "each", False, True),
    (16, 1, 128, 64, 60, False, ("chunk", 50), 3.0, "one", False, False), (5, 5, 48, 7, 60, False, None, None, None, True, True),
    (6, 2, 48, 32, 60, False, ("window", 1), None, "each", True, False), (3, 1, 16, 8, 60, False, None, 2.0, None, False, True),
    (4, 4, 64, 48, 60, False, ("chunk", 33), None, "each", True, False), (7, 1, 112, 128, 60, False, ("window", 333), None, None, False, False),
    # tables of more than 1,024 entries: of single tokens, of pages; and with two row tiles a wave, plain, capped and biased
    (8, 2, 64, 1, 60, False, None, None, None, False, False), (8, 1, 64, 32, 60, False, None, None, "one", False, True),
    (16, 4, 64, 1, 700, True, ("window", 600), None, None, True, False), (32, 4, 128, 32, 700, True, ("window", 500), 5.0, "each", False, True),
    (12, 3, 32, 1, 900, True, None, None, None, False, False),
])
def test_prefill_attention_of_one_tile_beside_prompts(ops, Hq, Hkv, D, page, portion, two, reach, cap, sinks, slopes, gated):
    """Requests whose rows are one tile, whose keys four waves share, beside a longer portion: one to four tokens, from the last length that goes
    the portions' way over the edges of a wave's 32 and the four waves' 128 on, every option, one and two row tiles a wave, tables in LDS and in
    memory, and an infinite value that only its readers see."""
    G = Hq // Hkv
    start = 256 if G >= 4 else 448
    some = min(4, 16 // G)
    lens = [31, start, start + 1, start + 31, start + 32, start + 33, start + 127, start + 128, start + 129, start + 300, 1700, start + 129, portion + 140]
    q_lens = [1, 1, 1, 1, some, 1, some, 1, 1, min(2, some), 1, 16 // G, portion]
    if G == 1:
        lens, q_lens = lens[1:], q_lens[1:]
    if page == 32 and G >= 8:                                # (a table of 1,026 pages)
        lens[2] = 32 * 1024 + 40
    assert (G * -(-portion // 16) + 7) // 8 * Hkv * len(lens) >= 512 if two else (G * -(-portion // 16) + 7) // 8 * Hkv * len(lens) < 512
    assert ops.backend().attention_lib(D).nhv_prefill_attention_one_tile_from(len(lens), portion, Hq, Hkv) == start
    at_1700 = lens.index(1700)
    q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, lens, q_lens, Hq, Hkv, D, page, seed=97, scale=1.5)
    g = torch.Generator().manual_seed(98)
    rows = torch.randn(q.shape[0], Hq + 3, generator=g).to(torch.bfloat16)
    slope = torch.rand(Hq, generator=g) * 0.1 if slopes else None
    sink = {None: None, "one": 0.7, "each": torch.randn(Hq, generator=g)}[sinks]
    options = {"softcap": cap, "slopes": None if slope is None else slope.cuda(), "sink": sink.cuda() if sinks == "each" else sink,
               "gate": (rows.cuda(), 2) if gated else None, **({reach[0]: reach[1]} if reach else {})}
    out = ops.paged_attention(q, kc, vc, batch, bt, D ** -0.5, **options)
    want, at = [], 0
    for r, (n, nq) in enumerate(zip(lens, q_lens)):
        pos, key = torch.arange(n - nq, n)[:, None], torch.arange(n)[None]
        ok = key <= pos
        if reach:
            ok &= key > pos - reach[1] if reach[0] == "window" else key // reach[1] == pos // reach[1]
        s = torch.einsum("qhd,khd->hqk", qs[r].double(), ks[r].double().repeat_interleave(Hq // Hkv, 1)) * D ** -0.5
        s = cap * torch.tanh(s / cap) if cap else s
        s = s - slope.double()[:, None, None] * (pos - key) if slopes else s
        s = s.masked_fill(~ok, float("-inf"))
        if sinks:
            s = torch.cat((s, torch.as_tensor(sink, dtype=torch.float64).expand(Hq)[:, None, None].expand(Hq, nq, 1)), -1)
        o = torch.einsum("hqk,khd->qhd", torch.softmax(s, -1)[..., :n], vs[r].double().repeat_interleave(Hq // Hkv, 1))
        want.append(o * torch.sigmoid(rows[at:at + nq, 2:2 + Hq].double())[..., None] if gated else o)
        at += nq
    torch.testing.assert_close(out.double().cpu(), torch.cat(want), **tol(torch.bfloat16))
    vc[bt[at_1700, 1690 // page], 1690 % page, Hkv - 1, D - 1] = float("inf")
    spoilt = ops.paged_attention(q, kc, vc, batch, bt, D ** -0.5, **options)
    row = sum(q_lens[:at_1700])
    reads = not reach or (1690 > 1699 - reach[1] if reach[0] == "window" else 1690 // reach[1] == 1699 // reach[1])
    assert bool(torch.isfinite(spoilt[row, Hq - 1, D - 1])) is not reads
    hit = torch.zeros_like(out, dtype=torch.bool)
    hit[row, Hq - Hq // Hkv:, D - 1] = reads
    assert torch.equal(spoilt[~hit], out[~hit])


@pytest.mark.parametrize("scale", [1.0, 3.0])
@pytest.mark.parametrize("n", [257, 300, 1000, 2000])
def test_a_token_is_as_exact_alone_beside_a_portion_as_inside_one(ops, n, scale):
    """Requests' last tokens where four waves share the keys and at the end of portions, against float64 and each other: rounding the weights and the
    result to 8 bits is 2^-9 of the result each at most, either way."""
    Hq, Hkv, D = 32, 4, 128
    assert ops.backend().attention_lib(D).nhv_prefill_attention_one_tile_from(7, 60, Hq, Hkv) < n
    q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, [n] * 6 + [60], [40] * 6 + [60], Hq, Hkv, D, 64, seed=n, scale=scale)
    inside = ops.paged_attention(q, kc, vc, batch, bt, D ** -0.5).double().cpu()
    last = [40 * i + 39 for i in range(6)]
    alone, _, _, batch, *_ = _paged_setup(torch.bfloat16, [n] * 6 + [60], [1] * 6 + [60], Hq, Hkv, D, 64, seed=n, scale=scale)
    alone[:6], alone[6:] = q[last], q[240:]
    alone = ops.paged_attention(alone, kc, vc, batch, bt, D ** -0.5).double().cpu()[:6]
    want = _attention_reference([x[-1:] for x in qs[:6]], ks[:6], vs[:6], [n] * 6, [1] * 6, D ** -0.5, None)
    off = lambda x, y: float((x - y).norm() / want.norm())
    assert off(alone, want) < 2.0 ** -8 and off(inside[last], want) < 2.0 ** -8
    assert off(alone, want) < 1.1 * off(inside[last], want) and off(alone, inside[last]) < 2.0 ** -7


@pytest.mark.parametrize("far", [3, 650, 1290])
def test_prefill_attention_scores_that_outgrow_their_reference(ops, far):
    """The prompt kernel takes a row's exponentials against a reference point that stays while they stay far below
    float's range. Here one key's scores stand 110 powers of two above all others, for every query of one head: an
    early key (everything after it is tiny against the reference), a key in the middle of the portion and one near
    its end (the sums so far have to be scaled down by 2^-110 when it comes). Against the float64 computation."""
    Hq, Hkv, D, page = 4, 2, 128, 64
    scale = D ** -0.5
    lens, q_lens = [1300, 200], [700, 200]
    q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, lens, q_lens, Hq, Hkv, D, page, seed=71, scale=1.0)
    g = torch.Generator().manual_seed(6)
    direction = torch.randn(D, generator=g)
    direction = (direction / direction.norm()).to(torch.bfloat16)
    ks[0][far, 0] = 30.0 * direction                              # heads 0 and 1 read key/value head 0
    kc[int(bt[0, far // page]), far % page, 0] = ks[0][far, 0].cuda()
    qs[0][:, 1] = qs[0][:, 1] + 29.0 * direction                  # 30 x 29 / sqrt(128) = 77 = 111 powers of two
    q[:q_lens[0], 1] = qs[0][:, 1].cuda()
    out = ops.paged_attention(q, kc, vc, batch, bt, scale, None)
    ref = _attention_reference(qs, ks, vs, lens, q_lens, scale, None)
    torch.testing.assert_close(out.double().cpu(), ref, **tol(torch.bfloat16))
    # (the input does what it is meant to: a query of head 1 that sees the key puts all of its weight on it)
    first_q = lens[0] - q_lens[0]
    row = max(far - first_q, 0) + 5
    torch.testing.assert_close(ref[row, 1], vs[0][far, 0].double(), rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("window", [None, 5000])
def test_attention_over_32768_keys(ops, window):
    """Both bfloat16 attention kernels at 32,768 keys on pages of 256 (128 pages a request, the engine's splits to
    merge, block tables past what a block keeps in LDS at smaller pages), against the float64 computation: a single
    token at the end of 32,768 keys beside one after 9,001; and portions of 130 and 64 tokens that end at 32,768
    and 20,000 keys. In every request one early key is made to stand out for one head's queries, so that a key lost
    far from the end shows."""
    Hq, Hkv, D, page = 8, 2, 128, 256
    scale = D ** -0.5
    for lens, q_lens in ([[32768, 9001], [1, 1]], [[32768, 20000], [130, 64]]):
        q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, lens, q_lens, Hq, Hkv, D, page, seed=41, scale=1.0)
        # key 777 (and key n - 4100, inside a window of 5,000) of every request points where head 3's queries point
        g = torch.Generator().manual_seed(5)
        direction = torch.randn(D, generator=g)
        direction = (direction / direction.norm()).to(torch.bfloat16)
        row = 0
        for r, (n, nq) in enumerate(zip(lens, q_lens)):
            for far in (777, n - 4100):
                ks[r][far, 0] = ks[r][far, 0] + 14.0 * direction          # head 3 reads key/value head 0
                pid = int(bt[r, far // page])
                kc[pid, far % page, 0] = ks[r][far, 0].cuda()
            qs[r][:, 3] = qs[r][:, 3] + 14.0 * direction
            q[row:row + nq, 3] = qs[r][:, 3].cuda()
            row += nq
        out = ops.paged_attention(q, kc, vc, batch, bt, scale, window)
        ref = _attention_reference(qs, ks, vs, lens, q_lens, scale, window)
        torch.testing.assert_close(out.double().cpu(), ref, **tol(torch.bfloat16))
        # (the input does what it is meant to: nearly all of the softmax's weight of head 3's last query lies on the
        # keys that stand out, so an output that agrees with the reference has found them)
        for r, n in enumerate(lens):
            scores = (ks[r][:, 0].double() @ qs[r][-1, 3].double()) * scale
            if window:
                scores[:n - window] = float("-inf")
            weight = torch.softmax(scores, 0)
            far = [n - 4100] if window else [777, n - 4100]
            assert weight[far].sum() > 0.95


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("page", [8, 64, 256])
def test_attention_finds_one_far_key(ops, dtype, page):
    """One key is made to stand out (score far above the rest): the output must be that key's value,
    wherever the key lies: first of the sequence, last of a page, first of a page, the query's own position."""
    Hq, Hkv, D, n = 8, 2, 64, 700
    for far in [0, page - 1, page, 2 * page - 1, n // 2, n - 2, n - 1]:
        g = torch.Generator().manual_seed(far)
        k = torch.randn(n, Hkv, D, generator=g) * 0.1
        v = torch.randn(n, Hkv, D, generator=g)
        q = torch.randn(1, Hq, D, generator=g) * 0.1
        direction = torch.randn(D, generator=g)
        direction = direction / direction.norm()
        k[far] += 10.0 * direction
        q[0] += 10.0 * direction                    # score of `far` is about 100 * D^-0.5 = 12.5 above the others
        from nanohybrid_vlm_amd.native.ops import AttentionBatch
        n_pages = -(-n // page)
        perm = torch.randperm(n_pages, generator=g)
        kc = torch.full((n_pages, page, Hkv, D), float("nan"))
        vc = torch.full((n_pages, page, Hkv, D), float("nan"))
        for lp in range(n_pages):
            m = min(page, n - lp * page)
            kc[perm[lp], :m] = k[lp * page:lp * page + m]
            vc[perm[lp], :m] = v[lp * page:lp * page + m]
        batch = AttentionBatch(1, 1, torch.zeros(1, dtype=torch.int32).cuda(),
                               torch.tensor([n - 1], dtype=torch.int32).cuda(),
                               torch.tensor([0, 1], dtype=torch.int32).cuda(),
                               torch.tensor([n], dtype=torch.int32).cuda(), 1, n)
        out = ops.paged_attention(q.to(dtype).cuda(), kc.to(dtype).cuda(), vc.to(dtype).cuda(), batch,
                                  perm.to(torch.int32)[None].cuda(), D ** -0.5)
        ref = _attention_reference([q.to(dtype)], [k.to(dtype)], [v.to(dtype)], [n], [1], D ** -0.5, None)
        torch.testing.assert_close(out.double().cpu(), ref, **tol(dtype))
        if far < n - 1:
            # the same query once more as the second-to-last token of a portion of two (the portion kernel)
            q2 = torch.cat((q, q)).to(dtype).cuda()
            batch2 = AttentionBatch(2, 1, torch.zeros(2, dtype=torch.int32).cuda(),
                                    torch.tensor([n - 2, n - 1], dtype=torch.int32).cuda(),
                                    torch.tensor([0, 2], dtype=torch.int32).cuda(),
                                    torch.tensor([n], dtype=torch.int32).cuda(), 2, n)
            out2 = ops.paged_attention(q2, kc.to(dtype).cuda(), vc.to(dtype).cuda(), batch2,
                                       perm.to(torch.int32)[None].cuda(), D ** -0.5)
            torch.testing.assert_close(out2[1:].double().cpu(), ref, **tol(dtype))
        # and it is mostly that one value
        kvh = torch.arange(Hq) // (Hq // Hkv)
        assert (out.float().cpu()[0] - v[far, kvh]).abs().max() < 0.5, f"far key {far} not found"


@pytest.mark.parametrize("V", [301, 389, 5000, 151936])
def test_sampling(ops, V):
    import plain_qwen3 as plain
    g = torch.Generator().manual_seed(V)
    n = 6
    logits = (torch.randn(n, V, generator=g) * 3).cuda()
    logits[0, 17] = logits[0, 200] = 50.0                # a tie: the first index wins
    temps = torch.tensor([0.0, 0.0, 0.8, 1.0, 0.3, 2.5]).cuda()
    keys = torch.tensor([0, 0, 1234567, -99, 2**62 + 5, 42], dtype=torch.int64).cuda()
    tokens = ops.sample(logits, temps, keys).cpu()
    assert tokens[0] == 17
    assert tokens[1] == logits[1].argmax().item()
    if V <= 5000:
        mask = (1 << 64) - 1
        for r in range(2, n):
            key = int(keys[r]) & mask
            # the noise of plain_qwen3.sample_noise for an already mixed key
            noise = torch.tensor([plain.noise_of_bits(_mix(key ^ i) >> 40) for i in range(V)])
            assert tokens[r] == plain.sample_token(logits[r].cpu(), float(temps[r]), noise)


def _mix(z):
    mask = (1 << 64) - 1
    z = (z + 0x9E3779B97F4A7C15) & mask
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
    return z ^ (z >> 31)


def test_noise_of_every_bit_pattern(ops):
    """All 2^24 patterns through the kernel's own noise function: the values are those of the plain formula, none is
    0 or infinite, and the share of patterns below x is the Exp(1) distribution's 1 - exp(-x) to within one and a
    half patterns, from the smallest values (3e-8) up. A noise of 1e-10 once in 2^24 draws would fail both."""
    import ctypes
    import numpy as np
    n = 1 << 24
    bits = torch.arange(n, dtype=torch.int32, device="cuda")
    out = torch.empty(n, dtype=torch.float32, device="cuda")
    lib = ops.backend().lib
    assert lib.nhv_noise_of_bits(ctypes.c_void_p(bits.data_ptr()), ctypes.c_void_p(out.data_ptr()), n,
                                 ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    got = out.cpu().numpy().astype(np.float64)
    want = -np.log((np.arange(n, dtype=np.float64) + 0.5) / n)
    assert np.isfinite(got).all() and got.min() > 2.9e-8
    assert np.abs(got / want - 1).max() < 1e-6
    ordered = np.sort(got)
    share = np.arange(1, n + 1) / n                       # share of patterns at or below each value
    # (half a pattern by construction, and up to as much again from rounding the larger values to float)
    assert np.abs(share - (1 - np.exp(-ordered))).max() <= 1.5 / n


def test_sampling_follows_the_distribution(ops):
    """Empirical frequencies of 4000 draws against softmax(logits / T) (chi-square, fixed keys)."""
    V, draws, temp = 12, 4000, 0.7
    logits = torch.tensor([[2.0, 1.0, 0.5, 0.0, -0.5, -1.0, 1.5, 0.2, -2.0, 0.7, 0.1, -0.3]])
    p = torch.softmax(logits[0] / temp, dim=0)
    rows = logits.repeat(draws, 1).cuda()
    keys = torch.arange(draws, dtype=torch.int64).cuda() * 7919 + 13
    tokens = ops.sample(rows, torch.full((draws,), temp).cuda(), keys).cpu()
    counts = torch.bincount(tokens.long(), minlength=V).float()
    chi2 = ((counts - draws * p) ** 2 / (draws * p)).sum().item()
    assert chi2 < 31.3, f"chi-square {chi2:.1f} with 11 degrees of freedom (0.999 quantile is 31.3)"


def test_refusals(ops):
    from nanohybrid_vlm_amd.native.ops import KernelError
    x = rnd(2, 64)
    with pytest.raises(KernelError, match="columns"):
        ops.linear(x, rnd(8, 32))
    with pytest.raises(KernelError, match="element type"):
        ops.linear(x.half(), rnd(8, 64).half())
    with pytest.raises(KernelError, match="limit"):
        ops.rmsnorm(rnd(1, 20000), rnd(20000), 1e-6)
    with pytest.raises(KernelError, match="contiguous"):
        ops.rmsnorm(rnd(4, 128)[:, ::2], rnd(64), 1e-6)
    with pytest.raises(KernelError, match="device"):
        ops.rmsnorm(torch.zeros(2, 8), torch.ones(8), 1e-6)


def test_products_of_few_rows_are_done_the_fastest_way_measured(ops):
    """While ``measure_linears`` is set a shape not seen before is timed by the own kernel and by every algorithm
    of the library, and the answer kept; whichever way a product goes, it is the same product."""
    from nanohybrid_vlm_amd.native.ops import OWN
    backend = ops.backend()
    N, K = 512, 1024
    for M in (8, 40):                                       # the own kernel is among the ways / the library's ways only
        x = rnd(M, K, dtype=torch.bfloat16, seed=51)
        w = rnd(N, K, dtype=torch.bfloat16, seed=52, scale=K ** -0.5)
        w2 = rnd(2 * N, K, dtype=torch.bfloat16, seed=53, scale=K ** -0.5)
        ref = x.double() @ w.double().T
        g, u = x.double() @ w2[:N].double().T, x.double() @ w2[N:].double().T
        keys = [(M, N, K, False, False), (M, N, K, True, False)] + ([(M, 2 * N, K, False, True)] if M <= 16 else [])
        every = keys + [(M, 2 * N, K, False, False)]
        saved = {k: backend.chosen.pop(k, None) for k in every}
        try:
            assert ops.linear(x, w) is not None and keys[0] not in backend.chosen      # not measured unasked
            backend.measure_linears = True
            try:
                ops.linear(x, w)
                ops.linear(x, w, out_dtype=torch.float32)
                ops.gated_linear(x, w2)
            finally:
                backend.measure_linears = False
                backend.end_measurements()
            assert all(isinstance(backend.chosen[k], int) for k in keys)
            assert M <= 16 or all(backend.chosen[k] != OWN for k in keys)
            _, count = backend._library_plan(M, N, K, False)
            assert count > 0
            for how in [OWN] + list(range(min(count, 3))):
                for k in every:
                    backend.chosen[k] = how
                torch.testing.assert_close(ops.linear(x, w).double(), ref, **tol(torch.bfloat16))
                torch.testing.assert_close(ops.linear(x, w, out_dtype=torch.float32).double(), ref, rtol=1e-4, atol=1e-4)
                torch.testing.assert_close(ops.gated_linear(x, w2).double(), g * torch.sigmoid(g) * u, **tol(torch.bfloat16))
        finally:
            for k, v in saved.items():
                backend.chosen.pop(k, None)
                if v is not None:
                    backend.chosen[k] = v


def test_a_shape_of_many_rows_is_measured_in_the_third_step_that_meets_it(ops):
    """Prompt portions: only a shape that comes step after step is timed (against ``torch.mm``, which stays
    unless one of the library's algorithms is clearly faster); the product is the same product either way."""
    from nanohybrid_vlm_amd.native.ops import RULE
    backend = ops.backend()
    M, N, K = 200, 384, 512
    x = rnd(M, K, dtype=torch.bfloat16, seed=61)
    w = rnd(N, K, dtype=torch.bfloat16, seed=62, scale=K ** -0.5)
    ref = x.double() @ w.double().T
    key = (M, N, K, False, False)
    saved = backend.chosen.pop(key, None), backend._met.pop(key, None)
    try:
        for step in range(3):
            backend.step_number += 1
            for _ in range(4):                               # layers of one step count once
                torch.testing.assert_close(ops.linear(x, w).double(), ref, **tol(torch.bfloat16))
            assert (key in backend.chosen) == (step == 2)
        assert backend.chosen[key] == RULE or backend.chosen[key] >= 0
        _, count = backend._library_plan(M, N, K, False)
        for how in [RULE] + list(range(min(count, 3))):
            backend.chosen[key] = how
            torch.testing.assert_close(ops.linear(x, w).double(), ref, **tol(torch.bfloat16))
    finally:
        backend.chosen.pop(key, None)
        backend._met.pop(key, None)
        if saved[0] is not None:
            backend.chosen[key] = saved[0]
        if saved[1] is not None:
            backend._met[key] = saved[1]


def test_library_products_refuse_what_they_cannot_do(ops):
    """The wrapper of the vendor's matrix library names what is wrong: an algorithm the plan does not have, a
    workspace smaller than the plan's, a plan that was never made."""
    import ctypes
    from nanohybrid_vlm_amd.native.ops import KernelError
    backend = ops.backend()
    plan, count = backend._library_plan(8, 256, 512, False)
    assert count > 0 and backend._library_plan(8, 256, 512, False) == (plan, count)      # a shape has one plan
    x = rnd(8, 512, dtype=torch.bfloat16, seed=71)
    w = rnd(256, 512, dtype=torch.bfloat16, seed=72)
    out = torch.empty(8, 256, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(KernelError, match="algorithms"):
        backend._library_product(x, w, out, count)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    with pytest.raises(KernelError, match="no plan"):
        backend._call("nhv_library_gemm", 10 ** 6, 0, ptr(x), ptr(w), ptr(out), None, ctypes.c_size_t(0), None, lib=backend.blas_lib())
    with pytest.raises(KernelError, match="result type"):
        backend._call("nhv_library_gemm_plan", 8, 256, 512, 7, 4, ctypes.c_size_t(0), ctypes.byref(ctypes.c_int()),
                      ctypes.byref(ctypes.c_int()), lib=backend.blas_lib())
    backend._library_product(x, w, out, 0)
    torch.testing.assert_close(out.double(), x.double() @ w.double().T, **tol(torch.bfloat16))


# ---------------------------------------------------------------- sizes drawn at random (seeded)
# The kernels choose waves, loads in flight, tiles a block and split lengths from the sizes by rules; these cases walk
# over the rules' borders at sizes nobody picked by hand.

@pytest.mark.parametrize("M,N,K", [
    # one and two tiles past 16 rows, every number of row tiles up to 8, the last one cut off; outputs that end inside a tile, a
    # chunk and two chunks of columns, chunks that do not divide by the parts
    (17, 64, 256), (32, 1000, 384), (33, 4096, 4096), (49, 6144, 2560), (64, 4096, 12288), (79, 2560, 1152), (80, 1033, 3072), (96, 333, 9728),
    (97, 512, 512), (112, 2048, 6144), (128, 1024, 3072),
    # wider than the 8B shape
    (31, 5120, 17408), (64, 10240, 5120),
])
def test_products_by_lines(ops, M, N, K):
    """As float parts and as a gate of two products, with biases and without (float sums of K products of size K^-1/2)."""
    x = rnd(M, K, dtype=torch.bfloat16, seed=81)
    w = rnd(2 * N, K, dtype=torch.bfloat16, seed=82, scale=K ** -0.5)
    b = rnd(2 * N, dtype=torch.bfloat16, seed=83)
    both = x.double() @ w.double().T
    wn = w[:N].contiguous()
    got = ops.linear(x, wn, parts=True)
    assert isinstance(got, ops.Parts) and got.shape == (M, N)
    torch.testing.assert_close(got.parts.double().sum(0), both[:, :N], rtol=1e-4, atol=2e-4)
    assert torch.equal(got.parts, ops.linear(x, wn, parts=True).parts)
    total = got.parts[0].clone()
    for part in got.parts[1:]:
        total += part
    assert torch.equal(ops.dense(got), total.bfloat16())
    if M <= 96:                                              # (also where the library's way is the faster one)
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        by_lines = ops.backend().lib.nhv_gemm_lines_bf16
        assert by_lines(ops._ptr(x), ops._ptr(w), ops._ptr(None), ops._ptr(out), M, N, K, 1, *ops.Gate().args(), ops._stream()) == 0
        torch.testing.assert_close(out.double(), torch.nn.functional.silu(both[:, :N]) * both[:, N:], **tol(torch.bfloat16))
        gate = ops.Gate(2, 1.5, 1.702, 1.0)
        g, u = (both + b.double()).split(N, dim=1)
        g, u = g.clamp(max=1.5), u.clamp(-1.5, 1.5)
        assert by_lines(ops._ptr(x), ops._ptr(w), ops._ptr(b), ops._ptr(out), M, N, K, 1, *gate.args(), ops._stream()) == 0
        torch.testing.assert_close(out.double(), g * torch.sigmoid(1.702 * g) * (u + 1), **tol(torch.bfloat16))


@pytest.mark.parametrize("M,N,K,parts,gated", [
    # the 0.6B to 8B shapes' products; gated ones of one round of blocks and of two, of few blocks over few columns and many
    (17, 4096, 1024, True, True), (96, 3072, 1024, True, True), (64, 4096, 12288, True, True), (64, 12288, 4096, True, True),
    (32, 17408, 5120, False, False), (96, 13824, 5120, False, False), (64, 25600, 1024, False, False), (79, 1024, 4096, True, False),
    (48, 512, 1024, True, True), (17, 2040, 9344, True, False),
    # more outputs than the plain ones are taken for, more blocks, more rows, the smallest
    (32, 12296, 1024, False, False), (96, 8832, 28672, False, False), (112, 8704, 9216, False, False), (112, 5120, 17408, True, False),
    (79, 376, 384, False, True), (64, 376, 384, True, True),
])
def test_which_products_go_by_lines(ops, M, N, K, parts, gated):
    """As parts and as a gate, where that was measured to be the faster way; elsewhere rows that the library (or torch) makes."""
    x, w = (torch.zeros(r, K, dtype=torch.bfloat16, device="cuda") for r in (M, 2 * N))
    assert isinstance(ops.linear(x, w[:N], parts=True), ops.Parts) == parts
    out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    assert ops.backend().gated_linear(x, w, out) == gated


def test_what_goes_by_lines_hangs_on_the_shape_and_on_a_table_that_is_read(ops):
    """A library algorithm measured for the same shape's rows changes nothing; a table from a file that names one is followed, unless it
    says that the own kernel made the product where its reader took parts, or the gate."""
    backend = ops.backend()
    M, N, K = 40, 2048, 1024
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=121), rnd(2 * N, K, dtype=torch.bfloat16, seed=122, scale=K ** -0.5)
    out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")

    def ways():
        return isinstance(ops.linear(x, w[:N], parts=True), ops.Parts), backend.gated_linear(x, w, out)

    saved, allowed, chosen = dict(backend.shared_chosen), backend.measuring_allowed, backend.chosen
    try:
        backend.shared_chosen.clear()
        backend.use_choices(None, True)
        assert ways() == (True, True)
        written = backend.choices_table()
        assert written == {f"{M},{N},{K},0,2": -1, f"{M},{2 * N},{K},0,1": -1}
        algorithms = {f"{M},{N},{K},0,0": 0, f"{M},{2 * N},{K},0,0": 0}
        backend.shared_chosen.update(backend.parse_choices(algorithms))        # (as if measured for a plain product)
        assert ways() == (True, True)
        for table, want in (({}, (True, True)), (algorithms, (False, False)), ({**algorithms, **written}, (True, True))):
            backend.use_choices(backend.parse_choices(table), False)
            assert ways() == want and backend.choices_table() == table
    finally:
        backend.shared_chosen.clear()
        backend.shared_chosen.update(saved)
        backend.chosen, backend.measuring_allowed = chosen, allowed


def test_results_off_their_boundaries_are_not_the_kernel_of_many_rows_ones(ops):
    """Rows of results that do not begin on 8 bytes: left to the product and the kernel behind it, untouched."""
    backend = ops.backend()
    M, N, K = 1300, 8192, 512
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=134), rnd(2 * N, K, dtype=torch.bfloat16, seed=135, scale=K ** -0.5)
    room = torch.full((M * N + 8,), 7.0, dtype=torch.bfloat16, device="cuda")
    for off in (1, 2, 3, 4):
        out, taken = room[off:off + M * N].view(M, N), off == 4
        assert backend.gated_linear(x, w, out) is taken and (taken or bool((room == 7.0).all()))
    assert torch.equal(room[4:4 + M * N].view(M, N), ops.gated_linear(x, w)) and bool((room[:4] == 7.0).all())
    room.fill_(7.0)
    assert not backend.activated_linear(x, w[:N], room[1:1 + M * N].view(M, N), 1) and bool((room == 7.0).all())


@pytest.mark.parametrize("how", [-2, 0])
def test_many_rows_are_gated_the_way_that_a_table_which_is_read_names(ops, how):
    """A gated and an activated product of many rows: a table from a file that names torch.mm or a library algorithm for the shape is followed,
    whether or not other shapes may be timed, unless it says that the own kernel joined the gate; what was measured for the same shape's
    plain products in this process changes nothing, also where an engine's own table comes to hold it."""
    backend = ops.backend()
    M, N, K = 1300, 8192, 512
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=134), rnd(2 * N, K, dtype=torch.bfloat16, seed=135, scale=K ** -0.5)
    out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")

    def ways():
        done = backend.gated_linear(x, w, out), backend.activated_linear(x, w[:N], out, 1)
        assert torch.equal(ops.gated_linear(x, w), ops.act_mul(ops.linear(x, w), "silu")) is not done[0]
        return done

    saved, allowed, chosen, many = dict(backend.shared_chosen), backend.measuring_allowed, backend.chosen, backend.measure_many_rows
    try:
        backend.measure_many_rows = False
        backend.shared_chosen.clear()
        backend.use_choices(None, True)
        assert ways() == (True, True)
        written = backend.choices_table()
        assert written == {f"{M},{N},{K},0,1": -1, f"{M},{2 * N},{K},0,1": -1}
        apart = {f"{M},{N},{K},0,0": how, f"{M},{2 * N},{K},0,0": how}
        backend.shared_chosen.update(backend.parse_choices(apart))             # (as if measured for plain products)
        assert ways() == (True, True)
        for measuring in (False, True):
            for table, want in (({}, True), (apart, False), ({**apart, **written}, True)):
                backend.use_choices(backend.parse_choices(table), measuring)
                assert ways() == (want, want) and backend.choices_table() == ({**written, **table} if measuring and want else table)
        backend.use_choices({}, True)
        assert ways() == (True, True)
        backend.chosen.update(backend.parse_choices(apart))
        assert ways() == (True, True)
    finally:
        backend.shared_chosen.clear()
        backend.shared_chosen.update(saved)
        backend.chosen, backend.measuring_allowed, backend.measure_many_rows = chosen, allowed, many


@pytest.mark.parametrize("M,N,K", [(3, 4096, 2048), (16, 4100, 2304), (17, 2048, 1024), (40, 3000, 1280), (90, 4096, 2048)])
def test_products_by_lines_keep_rows_and_columns_apart(ops, M, N, K):
    """Rows of x and of w that are infinite or no numbers: their own rows and columns are what float64 says of them, all others the same bits as
    without them, as rows, parts and a gate."""
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=141), rnd(2 * N, K, dtype=torch.bfloat16, seed=142, scale=K ** -0.5)

    def results():
        made = [ops.linear(x, w[:N]), ops.gated_linear(x, w)]
        if M <= 16:
            return made + [ops.linear(x, w[:N], out_dtype=torch.float32)]
        return made + list(ops.linear(x, w[:N], parts=True).parts)

    clean = [r.clone() for r in results()]
    x[0, K // 2], x[M - 1, 7] = float("nan"), float("inf")
    w[5, K - 1], w[N - 1, 0], w[N + 9, 3] = float("-inf"), float("nan"), float("inf")
    rows = [i for i in range(M) if i not in (0, M - 1)]
    columns = [j for j in range(N) if j not in (5, N - 1, 9)]
    want = x.double() @ w[:N].double().T
    got = results()
    for before, now in zip(clean, got):
        assert torch.equal(now[rows][:, columns], before[rows][:, columns])
    for odd in [got[0]] + ([got[2]] if M <= 16 else [sum(got[2:])]):
        odd = odd.double()
        assert torch.equal(odd.isnan(), want.isnan()) and torch.equal(odd.isposinf(), want.isposinf()) and torch.equal(odd.isneginf(), want.isneginf())


@pytest.mark.parametrize("M,band,last,K", [(1, 1024, 32, 2048), (16, 2048, 5, 2304), (7, 1056, 1100, 2048)])
def test_products_in_bands_by_lines(ops, M, band, last, K):
    """Five sets of rows against a matrix's bands, where the kernel by lines takes them (float sums of K products of size K^-1/2)."""
    x = rnd(5, M, K, dtype=torch.bfloat16, seed=92)
    w = rnd(4 * band + last, K, dtype=torch.bfloat16, seed=93, scale=K ** -0.5)
    want = torch.cat([x[i].double() @ w[i * band:(4 * band + last if i == 4 else (i + 1) * band)].double().T for i in range(5)], dim=1)
    torch.testing.assert_close(torch.cat(list(ops.banded_linear(x, w, band)), dim=1).double(), want, **tol(torch.bfloat16))


@pytest.mark.parametrize("M", [1, 3, 8, 12])
@pytest.mark.parametrize("band,last,K", [(512, 512, 2048), (640, 704, 2304), (960, 250, 2304), (512, 512, 4096), (512, 544, 4096)])
def test_products_in_bands_of_few_outputs(ops, M, band, last, K):
    """Four sets of rows against the bands of 2,048 to 3,130 outputs, in both result types: on either side of where they go by lines (by blocks of 8
    outputs for 12 rows of 2,048), each band's rows of a size of their own (float sums of K products of that size times K^-1/2, and one rounding)."""
    sizes = torch.tensor([1.0, 4.0, 16.0, 64.0], device="cuda").view(4, 1, 1)
    x = (rnd(4, M, K, seed=94) * sizes).to(torch.bfloat16)
    w = rnd(3 * band + last, K, dtype=torch.bfloat16, seed=95, scale=K ** -0.5)
    out = torch.empty(M, 3 * band + last, dtype=torch.bfloat16, device="cuda")
    assert ops.backend().banded_linear(x, w, out, band)
    for i, got in enumerate(ops.banded_linear(x, w, band)):
        of = slice(i * band, (i + 1) * band if i < 3 else None)
        want = x[i].double() @ w[of].double().T
        torch.testing.assert_close(got.double(), want, rtol=1e-4, atol=2e-4 * float(sizes[i]))
        torch.testing.assert_close(out[:, of].double(), want, rtol=8e-3, atol=2e-4 * float(sizes[i]))


@pytest.mark.parametrize("splits", [1, 2, 4, 8])
def test_parts_of_a_product_through_the_norm_and_the_rotation(ops, splits):
    """Parts whose sum is a bfloat16 number give the bits that this number gives: the norm that adds to the residual stream (in
    both types, for widths in one piece and in two) and the kernel that turns queries and keys."""
    def parts_of(t):
        share = t.float() / splits                           # (a power of two: exact)
        return ops.Parts(share.expand(splits, *t.shape).contiguous(), torch.bfloat16)

    for width in (8, 520, 4096, 9216):
        x = rnd(5, width, dtype=torch.bfloat16, seed=84)
        for res_dtype in DTYPES:
            for w_dtype in DTYPES:
                w, r = rnd(width, dtype=w_dtype, seed=85) + 1, rnd(5, width, dtype=res_dtype, seed=86)
                r2 = r.clone()
                want = ops.rmsnorm(x, w, 1e-6, residual=r)
                assert torch.equal(ops.rmsnorm(parts_of(x), w, 1e-6, residual=r2), want) and torch.equal(r, r2)
    # a width that is no multiple of 8, a residual and a weight off 16 bytes: the parts are summed first
    for width, off, w_off in ((20, 0, 0), (520, 1, 0), (520, 0, 1)):
        x, space, w_space = rnd(5, width, dtype=torch.bfloat16, seed=84), rnd(5 * width + 1, seed=86), rnd(width + 1, seed=85)
        w, r = w_space[w_off:w_off + width], space[off:off + 5 * width].view(5, width)
        r2 = space.clone()[off:off + 5 * width].view(5, width)
        want = ops.rmsnorm(x, w, 1e-6, residual=r)
        assert torch.equal(ops.rmsnorm(parts_of(x), w, 1e-6, residual=r2), want) and torch.equal(r, r2)
    T, Hq, Hkv = 7, 6, 2
    for D in (16, 64, 128, 512, 48):                         # (48: no power of two, the parts are summed first)
        qkv, bias = rnd(T, (Hq + 2 * Hkv) * D, dtype=torch.bfloat16, seed=87), rnd((Hq + 2 * Hkv) * D, dtype=torch.bfloat16, seed=88)
        nq, nk = rnd(D, dtype=torch.bfloat16, seed=89) + 1, rnd(D, dtype=torch.bfloat16, seed=90) + 1
        table = rnd(40, D, seed=91)
        positions = torch.arange(3, 3 + T, dtype=torch.int32, device="cuda")
        slots = torch.tensor([4, -1, 0, 9, 10, 3, 7], dtype=torch.int32, device="cuda")
        for norms, b in (((nq, nk), None), ((None, None), bias)):
            results = []
            for rows in (qkv, parts_of(qkv)):
                k, v = (torch.zeros(3, 4, Hkv, D, dtype=torch.bfloat16, device="cuda") for _ in range(2))
                q = ops.qk_rope_write(rows, b, *norms, 1e-6, table, positions, slots, k, v, Hq, Hkv, D)
                results.append((q, k, v))
            assert all(torch.equal(a, c) for a, c in zip(*results)), D


@pytest.mark.parametrize("N,K", [(5000, 2048), (9000, 4096), (4112, 6144), (4100, 2304), (700, 1024), (2600, 2560)])
def test_equal_rows_of_a_head_give_equal_logits(ops, N, K):
    """Whichever block makes them: between equal rows the first is chosen, not one that rounding favours. In float32 from bfloat16, few
    rows, against float64 (float sums of K products of size K^-1/2)."""
    w = rnd(N, K, dtype=torch.bfloat16, seed=131, scale=K ** -0.5)
    equal = sorted({3, 16, 40, N // 3, N // 2, N - 17, N - 1})
    w[equal] = w[3].clone()
    for M in (1, 5, 8, 12, 16):
        x = rnd(M, K, dtype=torch.bfloat16, seed=132 + M)
        y = ops.linear(x, w, out_dtype=torch.float32)
        assert torch.equal(y[:, equal], y[:, [3]].expand(M, len(equal)))
        torch.testing.assert_close(y.double(), x.double() @ w.double().T, rtol=1e-4, atol=2e-4)


def _random_product_sizes(seed, count, max_rows):
    import random
    rnd_ = random.Random(seed)
    sizes = []
    while len(sizes) < count:
        M = rnd_.randint(1, max_rows)
        N = rnd_.choice([rnd_.randint(1, 600), rnd_.randint(600, 9000), rnd_.randint(9000, 40000)])
        K = 8 * rnd_.choice([rnd_.randint(1, 64), rnd_.randint(64, 1000), rnd_.randint(1000, 3300)])
        if N * K <= 48_000_000:
            sizes.append((M, N, K))
    return sizes


@pytest.mark.parametrize("M,N,K", _random_product_sizes(1, 40, 16) + _random_product_sizes(2, 12, 64))
def test_products_of_few_rows_at_random_sizes(ops, M, N, K):
    x = rnd(M, K, dtype=torch.bfloat16, seed=44)
    w = rnd(N, K, dtype=torch.bfloat16, seed=45, scale=K ** -0.5)
    ref = x.double() @ w.double().T
    backend = ops.backend()
    backend.own_kernels_only = True                          # the own kernels, whatever a measurement would choose
    try:
        got = ops.linear(x, w, out_dtype=torch.float32)
        torch.testing.assert_close(got.double(), ref, rtol=1e-4, atol=2e-4)
        assert torch.equal(got, ops.linear(x, w, out_dtype=torch.float32))
        torch.testing.assert_close(ops.linear(x, w).double(), ref, **tol(torch.bfloat16))
        if N % 2 == 0:
            g, u = ref[:, :N // 2], ref[:, N // 2:]
            torch.testing.assert_close(ops.gated_linear(x, w).double(), g * torch.sigmoid(g) * u, **tol(torch.bfloat16))
    finally:
        backend.own_kernels_only = False


def _random_attention_cases(seed, count):
    import random
    rnd_ = random.Random(seed)
    cases = []
    for _ in range(count):
        Hkv = rnd_.choice([1, 2, 3, 8])
        G = rnd_.choice([1, 2, 3, 4, 5, 8, 16])
        D = 16 * rnd_.randint(1, 8) if rnd_.random() < 0.8 else 256
        page = rnd_.choice([3, 8, 16, 48, 64, 256])
        window = rnd_.choice([None, None, rnd_.randint(1, 40), rnd_.randint(41, 900)])
        cases.append((Hkv * G, Hkv, D, page, window, rnd_.randint(0, 10 ** 6)))
    return cases


@pytest.mark.parametrize("Hq,Hkv,D,page,window,seed", _random_attention_cases(3, 16))
def test_attention_kernels_at_random_sizes(ops, Hq, Hkv, D, page, window, seed):
    """Both bfloat16 attention kernels (single tokens; portions beside single tokens) at head counts, group sizes,
    head sizes, page sizes, windows and lengths drawn at random."""
    import random
    rnd_ = random.Random(seed)
    scale = D ** -0.5
    # single tokens: the split-key kernel
    lens = [rnd_.choice([rnd_.randint(1, 70), rnd_.randint(70, 700), rnd_.randint(700, 2600)]) for _ in range(rnd_.randint(1, 9))]
    q_lens = [1] * len(lens)
    q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, lens, q_lens, Hq, Hkv, D, page, seed=seed, scale=1.5)
    out = ops.paged_attention(q, kc, vc, batch, bt, scale, window)
    torch.testing.assert_close(out.double().cpu(), _attention_reference(qs, ks, vs, lens, q_lens, scale, window),
                               **tol(torch.bfloat16))
    # portions with and without earlier keys beside single tokens: the matrix-core kernel for prompts
    lens = [rnd_.randint(1, 1200) for _ in range(rnd_.randint(1, 5))]
    q_lens = [rnd_.choice([1, n, rnd_.randint(1, n)]) for n in lens]
    q_lens[0] = max(2, min(lens[0], q_lens[0])) if lens[0] > 1 else 1
    if max(q_lens) == 1:
        lens.append(300)
        q_lens.append(77)
    q, kc, vc, batch, bt, ks, vs, qs = _paged_setup(torch.bfloat16, lens, q_lens, Hq, Hkv, D, page, seed=seed + 1, scale=1.5)
    out = ops.paged_attention(q, kc, vc, batch, bt, scale, window)
    torch.testing.assert_close(out.double().cpu(), _attention_reference(qs, ks, vs, lens, q_lens, scale, window),
                               **tol(torch.bfloat16))


@pytest.fixture
def sixteen_at_a_time(ops, monkeypatch):
    """The delta rule takes sixteen tokens at a time also where there are few tokens in all."""
    monkeypatch.setattr(ops, "DELTA_CHUNK_WORK", 0)


def test_delta_rule_of_few_tokens_goes_token_by_token(ops, monkeypatch):
    """Which kernels a step's portions take, and that both ways give the same state."""
    backend, taken = ops.backend(), []
    chunks = backend.delta_chunks
    monkeypatch.setattr(backend, "delta_chunks", lambda *a: (taken.append(1), chunks(*a))[1])
    g = torch.Generator().manual_seed(83)
    H, G, D, E = 2, 1, 32, 16
    args = lambda n: (torch.randn(n, 2 * G * D + H * E + H, generator=g), torch.randn(n, H * D, generator=g), torch.randn(n, H * E, generator=g),
                      torch.randn(2 * G * D + H * E, 4, generator=g), torch.zeros(H * D), torch.zeros(H), torch.ones(E), H, G, D, E, False)
    for n in (15, 16, 45, 46, 200):
        del taken[:]
        inputs = args(n)
        state = _delta_rule_once(ops, *inputs)[1]
        assert len(taken) == (n >= 46), n
        with monkeypatch.context() as m:
            m.setattr(ops, "DELTA_CHUNK_WORK", 0 if n < 46 else 10 ** 9)
            torch.testing.assert_close(_delta_rule_once(ops, *inputs)[1], state, rtol=1e-5, atol=2e-6)
            assert len(taken) == (n >= 16), n


@pytest.mark.usefixtures("sixteen_at_a_time")
@pytest.mark.parametrize("H,G,D,E,taps,per_head,packed,lengths", [
    (2, 1, 16, 16, 4, False, False, [16, 17]), (3, 3, 20, 5, 1, False, False, [40, 1, 31]), (2, 2, 128, 128, 4, False, False, [100]),
    (4, 2, 72, 40, 5, True, True, [15, 33, 2]), (1, 1, 200, 24, 4, False, False, [64, 3]), (2, 1, 256, 100, 3, True, True, [19]),
    (1, 1, 3, 3, 16, False, False, [50]),
])
def test_delta_rule_sixteen_tokens_at_a_time(ops, H, G, D, E, taps, per_head, packed, lengths):
    """Portions that end inside a chunk and on its edge, beside requests of fewer tokens; a second portion goes on from the state
    and the kept inputs of the first; weak and very strong decays. State and result against the recurrence token by token in
    float64. The state is 32 bits: sums of 16 products a chunk of entries below 1 are off by some 16 roundings of 2^-24 each,
    and a chunk's error decays or stays; the result is one bfloat16 rounding of what follows from it."""
    import plain_pevazen as plain
    from nanohybrid_vlm_amd.native.ops import AttentionBatch
    g = torch.Generator().manual_seed(71)
    C, Dd, B = 2 * G * D + H * E, 1 if per_head else D, len(lengths)
    total = [n + 18 for n in lengths]                      # a portion of 18 more for every request
    proj = [torch.randn(n, C + H, generator=g) for n in total]
    a_lin = [3.0 * torch.randn(n, H * Dd, generator=g) for n in total]
    a_lin[0][5:8] = 60.0                                   # decays that are zero in 32 bits
    gates = [torch.randn(n, H * E, generator=g) for n in total]
    tap, dt_bias = 0.6 * torch.randn(C, taps, generator=g), torch.randn(H * Dd, generator=g) - 0.5
    a_log, norm = 0.5 * torch.randn(H, generator=g) - 0.5, 1.0 + 0.2 * torch.randn(E, generator=g)
    kept = torch.full((B + 1, C, taps - 1), float("nan")).cuda()
    state = torch.full((B + 1, H, E, D), float("nan")).cuda()
    slots = torch.arange(B, 0, -1).to(torch.int32)
    got = [[] for _ in lengths]
    for lo, hi in (([0] * B, lengths), (lengths, total)):
        at = [torch.arange(a, b) for a, b in zip(lo, hi)]
        batch = AttentionBatch(num_tokens=sum(map(len, at)), num_requests=B,
                               token_req=torch.repeat_interleave(torch.arange(B), torch.tensor([len(a) for a in at])).to(torch.int32).cuda(),
                               positions=torch.cat(at).to(torch.int32).cuda(),
                               cu_seqlens_q=torch.tensor([0] + [len(a) for a in at]).cumsum(0).to(torch.int32).cuda(),
                               context_lens=torch.tensor(hi, dtype=torch.int32).cuda(), max_q_len=max(map(len, at)), max_context_len=max(hi))
        rows = lambda x: torch.cat([t[a] for t, a in zip(x, at)]).cuda()
        p, a, z = rows(proj), rows(a_lin), rows(gates)
        y = ops.gated_delta_rule(torch.cat((p, a, z), 1) if packed else p, None if packed else a, None if packed else z, tap.cuda(),
                                 dt_bias.cuda(), a_log.cuda(), norm.cuda(), 1e-5, kept, state, batch, slots.cuda(), H, G, D, E,
                                 torch.bfloat16, decay_per_head=per_head)
        for i, part in enumerate(y.float().cpu().split([len(a) for a in at])):
            got[i].append(part)
    for i, n in enumerate(total):
        x = proj[i].double()
        act = plain.silu(plain.causal_taps(x[:, :C], tap.double()))
        unit = lambda t: t / torch.sqrt(t.pow(2).sum(-1, keepdim=True) + 1e-6)
        q = unit(act[:, :G * D].view(n, G, D)).repeat_interleave(H // G, dim=1) * D ** -0.5
        k = unit(act[:, G * D:2 * G * D].view(n, G, D)).repeat_interleave(H // G, dim=1)
        v, beta = act[:, 2 * G * D:].view(n, H, E), torch.sigmoid(x[:, C:])
        decay = torch.exp(-torch.exp(a_log.double())[None, :, None] * plain.softplus((a_lin[i] + dt_bias).double()).view(n, H, Dd)).expand(n, H, D)
        S = torch.zeros(H, D, E, dtype=torch.float64)
        want = []
        for t in range(n):
            S = decay[t][..., None] * S
            u = beta[t][:, None] * (v[t] - torch.einsum("hde,hd->he", S, k[t]))
            S = S + k[t][..., None] * u[:, None]
            want.append(torch.einsum("hde,hd->he", S, q[t]))
        torch.testing.assert_close(state[int(slots[i])].double().cpu(), S.transpose(1, 2), rtol=1e-5, atol=2e-6)
        want = (plain.unit_rms(torch.stack(want), 1e-5) * norm * torch.sigmoid(gates[i].double()).view(n, H, E)).reshape(n, H * E)
        torch.testing.assert_close(torch.cat(got[i]).double(), want, rtol=1e-2, atol=2e-3)
    assert state[0].isnan().all()                          # a slot that no request holds is left alone


def _delta_rule_once(ops, proj, a_lin, gates, tap, dt_bias, a_log, norm, H, G, D, E, per_head):
    """One portion of one request from the start: (result in bfloat16, state)."""
    from nanohybrid_vlm_amd.native.ops import AttentionBatch
    n = len(proj)
    ints = lambda *v: torch.tensor(v, dtype=torch.int32).cuda()
    batch = AttentionBatch(num_tokens=n, num_requests=1, token_req=torch.zeros(n, dtype=torch.int32).cuda(), positions=ints(*range(n)),
                           cu_seqlens_q=ints(0, n), context_lens=ints(n), max_q_len=n, max_context_len=n)
    kept, state = torch.zeros(1, 2 * G * D + H * E, tap.shape[1] - 1).cuda(), torch.zeros(1, H, E, D).cuda()
    y = ops.gated_delta_rule(proj.cuda(), a_lin.cuda(), gates.cuda(), tap.cuda(), dt_bias.cuda(), a_log.cuda(), norm.cuda(), 1e-5, kept, state,
                             batch, ints(0), H, G, D, E, torch.bfloat16, decay_per_head=per_head)
    return y.cpu(), state[0].cpu()


@pytest.mark.usefixtures("sixteen_at_a_time")
@pytest.mark.parametrize("per_head", [False, True])
@pytest.mark.parametrize("rate,strong", [(0.6, 1.0), (4.0, 60.0), (16.0, 300.0), (0.6, float("inf")), (3e38, 5.0), (16.0, 3.0)])
@pytest.mark.parametrize("D", [64, 256])
def test_delta_rule_after_strong_decays(ops, D, rate, strong, per_head):
    """Weak decays after strong and infinite ones, within sixteen tokens: the state is as far from float64 as sixteen products of decays
    rounded to 2^-24 each (1e-6 of its largest entry; token by token 1e-7), not as the rounding of a sum of logarithms that a
    strong decay has made large, and a decay of zero leaves zeros."""
    import plain_pevazen as plain
    g = torch.Generator().manual_seed(73)
    H, G, E, n, taps = 2, 1, 32, 41, 4
    C, Dd = 2 * G * D + H * E, 1 if per_head else D
    proj, gates = torch.randn(n, C + H, generator=g), torch.randn(n, H * E, generator=g)
    a_lin = torch.randn(n, H * Dd, generator=g) - (0.0 if rate < 1 else 8.0 if rate < 100 else 200.0)
    for t in (2, 3, 4, 20, 37):
        a_lin[t] = strong
    tap, dt_bias, norm = 0.6 * torch.randn(C, taps, generator=g), 0.1 * torch.randn(H * Dd, generator=g), torch.ones(E)
    a_log = torch.full((H,), rate).log()
    y, state = _delta_rule_once(ops, proj, a_lin, gates, tap, dt_bias, a_log, norm, H, G, D, E, per_head)
    act = plain.silu(plain.causal_taps(proj[:, :C].double(), tap.double()))
    unit = lambda t: t / torch.sqrt(t.pow(2).sum(-1, keepdim=True) + 1e-6)
    k = unit(act[:, G * D:2 * G * D].view(n, G, D)).repeat_interleave(H // G, dim=1)
    v, beta = act[:, 2 * G * D:].view(n, H, E), torch.sigmoid(proj[:, C:].double())
    z = (a_lin + dt_bias).double()
    decay = torch.exp(-a_log.double().exp()[None, :, None] * torch.logaddexp(z, torch.zeros_like(z)).view(n, H, Dd)).expand(n, H, D)
    S = torch.zeros(H, D, E, dtype=torch.float64)
    for t in range(n):
        S = decay[t][..., None] * S
        S = S + k[t][..., None] * (beta[t][:, None] * (v[t] - torch.einsum("hde,hd->he", S, k[t])))[:, None]
    off = (state.transpose(1, 2).double() - S).abs().max() / S.abs().max()
    assert off < 1e-6, off
    assert torch.isfinite(y).all()


@pytest.mark.usefixtures("sixteen_at_a_time")
@pytest.mark.parametrize("per_head", [False, True])
@pytest.mark.parametrize("strong", [float("inf"), 3e38, 1e30, 700.0])
def test_delta_rule_after_decays_beyond_any_number_at_many_rates(ops, strong, per_head):
    """Infinite and huge decays at rates whose product with log2(e) is rounded up and down, a head each: what lies before them
    is gone, what comes after is there, within sixteen roundings of 2^-24 of the largest entry."""
    import plain_pevazen as plain
    g = torch.Generator().manual_seed(83)
    a_log = torch.cat((torch.linspace(-6.0, 4.0, 51), torch.tensor([20.0, 40.0, 60.0, 80.0])))
    H, G, D, E, n, taps = len(a_log), 1, 16, 16, 37, 4
    C, Dd = 2 * G * D + H * E, 1 if per_head else D
    proj, gates = torch.randn(n, C + H, generator=g), torch.randn(n, H * E, generator=g)
    a_lin = torch.randn(n, H, Dd, generator=g) - (a_log.clamp(min=0.0) + 1.0)[:, None]
    a_lin[[2, 3, 20, 33]] = strong
    tap, dt_bias = 0.6 * torch.randn(C, taps, generator=g), 0.1 * torch.randn(H * Dd, generator=g)
    y, state = _delta_rule_once(ops, proj, a_lin.view(n, H * Dd), gates, tap, dt_bias, a_log, torch.ones(E), H, G, D, E, per_head)
    act = plain.silu(plain.causal_taps(proj[:, :C].double(), tap.double()))
    k = act[:, G * D:2 * G * D]
    k = k / torch.sqrt(k.pow(2).sum(-1, keepdim=True) + 1e-6)
    v, beta = act[:, 2 * G * D:].view(n, H, E), torch.sigmoid(proj[:, C:].double())
    z = (a_lin + dt_bias.view(H, Dd)).double()
    decay = torch.exp(-a_log.double().exp()[:, None] * torch.logaddexp(z, torch.zeros_like(z)))
    S = torch.zeros(H, D, E, dtype=torch.float64)
    for t in range(n):
        S = decay[t][..., None] * S
        S = S + k[t][:, None] * (beta[t][:, None] * (v[t] - torch.einsum("hde,d->he", S, k[t])))[:, None]
    assert torch.isfinite(y).all() and torch.isfinite(state).all(), a_log[~torch.isfinite(state).flatten(1).all(1)]
    off = (state.transpose(1, 2).double() - S).abs().amax((1, 2)) / S.abs().amax((1, 2))
    assert off.max() < 1e-6, (off.max(), a_log[off.argmax()])


@pytest.mark.usefixtures("sixteen_at_a_time")
@pytest.mark.parametrize("per_head", [False, True])
@pytest.mark.parametrize("D,E", [(64, 32), (20, 5), (112, 128)])
def test_delta_rule_lets_no_token_reach_the_ones_before_it(ops, D, E, per_head):
    """A value, a key or a decay that is infinite or no number: the tokens before it, also those of the same sixteen, and the
    heads that do not read it keep their bits."""
    g = torch.Generator().manual_seed(79)
    H, G, n, taps = 2, 2, 53, 3
    C, Dd = 2 * G * D + H * E, 1 if per_head else D
    proj, gates, a_lin = torch.randn(n, C + H, generator=g), torch.randn(n, H * E, generator=g), torch.randn(n, H * Dd, generator=g)
    rest = (gates, 0.6 * torch.randn(C, taps, generator=g), torch.zeros(H * Dd), torch.zeros(H), torch.ones(E), H, G, D, E, per_head)
    clean, state = _delta_rule_once(ops, proj, a_lin, *rest)
    assert torch.isfinite(clean).all() and torch.isfinite(state).all()
    for t, column, value in ((22, 2 * G * D + 1, float("inf")), (37, G * D, float("nan")), (31, 0, float("nan")), (40, C + 0, float("nan")),
                             (9, None, float("nan"))):
        p, a = proj.clone(), a_lin.clone()
        if column is None:
            a[t, 0] = value
        else:
            p[t, column] = value
        out, left = _delta_rule_once(ops, p, a, *rest)
        assert torch.equal(out[:t], clean[:t]), (t, column)
        assert torch.equal(out[:, E:], clean[:, E:]) and torch.equal(left[1], state[1]), (t, column)
        assert not torch.isfinite(out[t, :E]).all(), (t, column)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,Hq,Hkv,D,E,rot,of_values,more", [(1, 1, 1, 16, 8, 16, None, ()), (513, 1, 1, 16, 8, 16, None, ()), (190, 5, 2, 24, 40, 16, None, ("bias",)),
                                                             (140, 16, 8, 128, 128, 128, "turned", ()), (48, 16, 8, 128, 128, 128, "turned", ()),
                                                             (70, 33, 11, 128, 64, 48, "mixed", ("temperature",)),
                                                             (360, 6, 3, 64, 64, 64, "keys", ("bias", "columns")),
                                                             (300, 7, 3, 32, 16, 0, "turned", ("bias",)),
                                                             (171, 12, 4, 80, 48, 80, "none", ("columns",))])
def test_heads_turned_in_pieces_of_eight_pairs(ops, dtype, T, Hq, Hkv, D, E, rot, of_values, more):
    """Against the kernel of one wave to a head, which takes the same rows where they start one entry off a piece: the same
    expressions of the same angles, whose products a compiler may contract one way or the other (half a float's last place,
    which can become one of bfloat16's); up to 1,536 heads of all tokens (2,048 that are turned back) both take that kernel. Rows without a slot store nothing; so the caches keep what they held."""
    kv = of_values != "none"
    width = Hq * D + (Hkv * D + (0 if of_values == "keys" else Hkv * E) if kv else 0) + (8 if "columns" in more else 0)
    bias = rnd(width - (8 if "columns" in more else 0), dtype=dtype, seed=91) if "bias" in more else None
    rows = rnd(T * width, dtype=dtype, seed=92)
    off = torch.cat((rows[:1], rows))[1:].view(T, width)
    rows = rows.view(T, width)
    assert rows.data_ptr() % 16 == 0 and off.data_ptr() % 16 != 0
    freqs = None if rot == 0 else torch.rand(rot // 2, device="cuda")
    v_freqs = torch.rand(E // 2, device="cuda") if of_values == "turned" else None
    positions = torch.randint(0, 20000, (T,), dtype=torch.int32, device="cuda")
    slots = torch.randperm(T + 3, device="cuda")[:T].int()
    slots[T // 2 + 1:T // 2 + 3] = -1
    options = {"temperature": (0.1, 100.0)} if "temperature" in more else {}
    if of_values == "mixed":
        options["mix"] = ((rnd(T, Hkv * E + 16, dtype=dtype, seed=93), 8), torch.tensor([0.3], device="cuda"))
    got = []
    for x in (rows, off):
        k_cache, v_cache = (torch.full((T + 3, 1, Hkv, n), 7.0, dtype=dtype, device="cuda") for n in (D, E))
        q = ops.rotary_split_write(x, bias, freqs, v_freqs, positions, slots if kv else None, k_cache if kv else None,
                                   v_cache if kv else None, Hq, Hkv, D, E, with_kv=kv,
                                   more_columns=8 if "columns" in more else 0, values_from_keys=of_values == "keys", **options)
        got.append((q, k_cache, v_cache))
    for a, b in zip(*got):
        torch.testing.assert_close(a, b, rtol=2.0 ** -7 if dtype == torch.bfloat16 else 0.0, atol=2.0 ** -20)
    if kv and T > 1:
        empty = torch.ones(T + 3, dtype=torch.bool, device="cuda")
        empty[slots[slots >= 0].long()] = False
        assert (got[0][1][empty] == 7).all() and (got[0][2][empty] == 7).all() and empty.sum() >= 4
    if E % 16 == 0:
        o = rnd(T * Hq * E, dtype=dtype, seed=94)
        o_off = torch.cat((o[:1], o))[1:].view(T, Hq, E)
        f = torch.rand(E // 2, device="cuda")
        a, b = ops.turn_back_(o.view(T, Hq, E), f, positions), ops.turn_back_(o_off, f, positions)
        torch.testing.assert_close(a, b, rtol=2.0 ** -7 if dtype == torch.bfloat16 else 0.0, atol=2.0 ** -20)


@pytest.mark.parametrize("Hq,Hkv,D,page,window,norm,bias,parts", [
    (16, 8, 128, 16, None, "float", False, 0), (6, 2, 64, 5, 70, None, True, 4), (20, 1, 32, 7, None, "rows", True, 0),
    (32, 2, 128, 256, 300, "rows", False, 8), (4, 4, 64, 64, None, "turn nothing", False, 0),
    (16, 8, 128, 16, None, "in 32 bits", False, 0), (6, 2, 64, 5, 70, "in 32 bits", True, 0), (16, 1, 128, 256, 33, "in 32 bits", True, 0),
    (4, 4, 64, 7, None, "in 32 bits, turn nothing", False, 0),
])
@pytest.mark.parametrize("lens", [[150], [1, 2, 31, 32, 33, 64, 65, 300, 17], [40, 3, 2000, 500, 501] * 4, [300] * 40])
def test_single_tokens_turned_stored_and_read_in_one_launch(ops, monkeypatch, Hq, Hkv, D, page, window, norm, bias, parts, lens):
    """Against the two launches, bit for bit: what is read, and the whole cache afterwards (keys and values that are stored, rows
    without a slot, a slot that is not where the token's position lies); also beside values that are no numbers and over
    several splits."""
    T, dtype = len(lens), torch.float32 if norm and "32" in norm else torch.bfloat16
    _, k, v, batch, bt, *_ = _paged_setup(dtype, lens, [1] * T, Hq, Hkv, D, page, seed=96)
    width = (Hq + 2 * Hkv) * D
    rows = rnd(T, width, dtype=dtype, seed=97)
    if parts:
        rows = ops.Parts(rnd(parts, T, width, seed=98), torch.bfloat16)
    b = rnd(width, dtype=dtype, seed=99) if bias else None
    norms = (None, None) if norm is None or "nothing" in norm else tuple(
        rnd(D, dtype=torch.float32 if norm == "float" else dtype, seed=i) + 1 for i in (100, 101))
    table = None if norm and "nothing" in norm else rnd(max(lens), D, seed=102)
    t = torch.arange(T, device="cuda")
    pos = batch.positions.long()
    slots = (bt[t, pos // page] * page + pos % page).int()
    spare = k.shape[0]
    k, v = (torch.cat((c, c[:1])) for c in (k, v))            # (a page that no request holds)
    if T > 4:
        slots[1], slots[3] = -1, spare * page + page - 1
        k[bt[1, (lens[1] - 1) // page], (lens[1] - 1) % page] = 0.5
        v[bt[1, (lens[1] - 1) // page], (lens[1] - 1) % page] = 0.25
        v[bt[4, 0], 0, 0, 1] = float("inf")
    k[bt[t, pos // page].long()[2:3], (pos % page)[2:3]] = float("nan")          # (what a token's own place held before is not read)
    arguments = (rows, b, *norms, 1e-6, table, batch.positions, slots)
    k1, v1, k2, v2 = k.clone(), v.clone(), k.clone(), v.clone()
    q = ops.qk_rope_write(*arguments, k1, v1, Hq, Hkv, D)
    want = ops.paged_attention(q, k1, v1, batch, bt, D ** -0.5, window)
    monkeypatch.setattr(ops, "ROTATED_BLOCKS", 1 << 20)
    monkeypatch.setattr(ops, "qk_rope_write", None)
    got = ops.rotated_attention(*arguments, k2, v2, Hq, Hkv, D, batch, bt, D ** -0.5, window)
    for a, c in ((got, want), (k2, k1), (v2, v1)):
        assert torch.equal(a.view(torch.uint8), c.view(torch.uint8))


@pytest.mark.parametrize("T,window", [(3, None), (20, None), (3, 40)])
@pytest.mark.parametrize("splits", [1, 2])
def test_single_tokens_beyond_what_the_splits_cover_are_stored_and_read(ops, monkeypatch, T, window, splits):
    """A launch whose splits end before the tokens' positions (as many keys a split, and splits, as are asked for here): the last split takes the
    keys that are left, so that the token's own key and value lie in the cache afterwards. Against the two launches: the cache bit for bit, the
    result within one rounding to 8 bits."""
    Hq, Hkv, D, page = 8, 2, 64, 16
    lens = [200 - 7 * i for i in range(T)]
    _, k, v, batch, bt, *_ = _paged_setup(torch.bfloat16, lens, [1] * T, Hq, Hkv, D, page, seed=161)
    rows, table = rnd(T, (Hq + 2 * Hkv) * D, dtype=torch.bfloat16, seed=162), rnd(256, D, seed=163)
    t, pos = torch.arange(T, device="cuda"), batch.positions.long()
    slots = (bt[t, pos // page] * page + pos % page).int()
    arguments = (rows, None, None, None, 0.0, table, batch.positions, slots)
    k1, v1, k2, v2 = k.clone(), v.clone(), k.clone(), v.clone()
    want = ops.paged_attention(ops.qk_rope_write(*arguments, k1, v1, Hq, Hkv, D), k1, v1, batch, bt, D ** -0.5, window)
    parts = [torch.zeros((T, Hq, splits, n), device="cuda") if splits > 1 else None for n in (D, 2)]
    monkeypatch.setattr(ops.backend(), "_decode_splits", lambda *args: (*parts, 32, splits), raising=False)
    got = ops.rotated_attention(*arguments, k2, v2, Hq, Hkv, D, batch, bt, D ** -0.5, window)
    assert torch.equal(k1.view(torch.int16), k2.view(torch.int16)) and torch.equal(v1.view(torch.int16), v2.view(torch.int16))
    torch.testing.assert_close(got, want, rtol=1.6e-2, atol=1.6e-2)


@pytest.mark.parametrize("H, N, K, rot, rows, in_lds", [
    # the matrix in LDS: full tiles, small heads, many blocks; once and in pieces, rows that end inside a block and a wave
    (16, 192, 128, 64, 2100, 1), (16, 128, 192, 0, 2050, 1), (1, 520, 256, 64, 16500, 1), (3, 8, 40, 16, 65, 1), (5, 56, 264, 32, 129, 1), (2, 64, 512, 0, 257, 1),
    (40, 72, 40, 16, 1170, 1), (64, 88, 512, 0, 700, 1), (128, 200, 8, 16, 330, 1), (7, 128, 480, 0, 191, 1), (2, 600, 128, 16, 66, 1),
    # outputs over the rows in LDS
    (3, 8, 8, 16, 65, 0), (2, 130, 40, 6, 257, 0), (5, 330, 168, 32, 129, 0), (2, 72, 512, 16, 191, 0), (40, 33, 264, 0, 1030, 0), (16, 300, 64, 0, 2038, 0),
    (5, 368, 288, 32, 512, 0), (40, 100, 24, 6, 1200, 0)])
def test_a_matrix_per_head_of_many_rows(ops, H, N, K, rot, rows, in_lds):
    """Products with a matrix per head of more than 64 rows at the edges of a block's rows, of the pieces of the matrix that
    are in LDS at a time and of the outputs that a lane writes at once, with and without gates and a turned part; rows of results that
    begin anywhere, of the same bits."""
    assert ops.backend().lib.nhv_head_gemm_rows_pays(rows, H, N, K) == in_lds
    g = torch.Generator(device="cuda").manual_seed(rows)
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda").to(torch.bfloat16)
    pad = -(K + rot) % 8
    x, w = rand(rows, H, K + rot + pad), rand(H, N, K)
    pos = torch.randint(0, 5000, (rows,), generator=g, device="cuda", dtype=torch.int32)
    want = torch.stack([x[:, h, :K].double() @ w[h].double().T for h in range(H)], dim=1)
    # one rounding to bfloat16, and the sums' own in float
    bound = want.abs() * 2.0 ** -8 + 2.0 ** -22 * K ** 0.5 * float(want.std())
    for off in (0, 1):
        for halves in ((True, False) if rot else (None,)):
            freqs = 10000.0 ** (-2.0 * torch.arange(rot // 2, dtype=torch.float64, device="cuda") / max(rot, 1))
            width = -(-(N + rot + off) // 8) * 8 + 8
            out = torch.full((rows, H, width), 7.0, dtype=torch.bfloat16, device="cuda")
            at = -(-(N + off) // 8) * 8 if off == 0 and N + rot <= width - 8 and N % 8 == 0 else N + off
            turn = (rot, K, at, freqs, 1.0, pos, halves) if rot else None
            ops.head_gemm(x, w.view(H * N, K), False, N, K, out=out, out_off=off, turn=turn)
            assert bool(((out[:, :, off:off + N].double() - want).abs() <= bound).all()), (off, halves)
            got = out[:, :, off:off + N].clone()
            assert off == 0 or torch.equal(got, first)
            first = got
            mask = torch.ones(width, dtype=torch.bool)
            mask[off:off + N] = False
            if rot:
                mask[at:at + rot] = False
                angle = (pos.double()[:, None] * freqs)[:, None]
                t = x[:, :, K:K + rot].double()
                u, v = (t[..., :rot // 2], t[..., rot // 2:]) if halves else (t[..., 0::2], t[..., 1::2])
                a, b = u * angle.cos() - v * angle.sin(), v * angle.cos() + u * angle.sin()
                turned = torch.cat((a, b), dim=-1) if halves else torch.stack((a, b), dim=-1).flatten(-2)
                # one rounding to bfloat16; the hardware's sine and cosine to 2^-16
                limit = turned.abs() * 2.0 ** -8 + 2.0 ** -16 * float(t.abs().max())
                assert bool(((out[:, :, at:at + rot].double() - turned).abs() <= limit).all()), (off, halves)
            assert bool((out[:, :, mask.to(out.device)] == 7.0).all())
    for gate, per in ((rand(rows, H * N + 4), "per entry"), (torch.randn(rows, H + 2, generator=g, device="cuda"), "per head")):
        for col in (0, 1):
            got = ops.head_gemm(x, w.view(H * N, K), False, N, K, gate=(gate, col, per))
            s = torch.sigmoid(gate.double())[:, col:col + (H * N if per == "per entry" else H)].reshape(rows, H, -1)
            assert bool(((got.double() - want * s).abs() <= (want * s).abs() * 2.0 ** -8 + 2.0 ** -20 * K ** 0.5 * float(want.std())).all()), (per, col)


@pytest.mark.parametrize("H", [8, 24, 511, 520, 2048, 2056, 4096, 8192, 8200])
def test_rows_in_pieces_of_eight(ops, H):
    """Embeddings, scaled sums and norms by one number where a row is a whole number of pieces, one or several a thread, and where
    it is not or does not begin on 16 bytes: the same as entry by entry."""
    g = torch.Generator(device="cuda").manual_seed(H)
    backend = ops.backend()
    for dtype in (torch.float32, torch.bfloat16):
        flat = torch.randn(40 * H + 1, generator=g, device="cuda").to(dtype)
        for table in (flat[:-1].view(40, H), flat[1:].view(40, H)):
            ids = torch.tensor([0, 39, 7, -1, 40, 12], dtype=torch.int32, device="cuda")
            want = table[ids.long().clamp(0, 39)] * ((ids >= 0) & (ids < 40))[:, None].to(dtype)
            for scale in (1.0, 1.75):
                out = torch.empty(6, H, dtype=dtype, device="cuda")
                backend.embed(ids, table, out, scale)
                assert torch.equal(out, (want.float() * scale).to(dtype))
                out = torch.empty(6, H, device="cuda")
                backend.embed_float(ids, table, out, scale)
                assert torch.equal(out, want.float() * scale)
            gain = torch.tensor([1.3], device="cuda")
            for to in (torch.float32, torch.bfloat16):
                got = ops.scalar_rmsnorm(table, gain, 1e-5, to)
                exact = table.double() * (1.3 / (table.double().square().mean(-1, keepdim=True) + 1e-5).sqrt())
                # float sums of H squares: H^0.5 2^-24 of the mean, half of that of the root; and one rounding
                assert bool(((got.double() - exact).abs() <= exact.abs() * (2.0 ** -8 if to == torch.bfloat16 else 2.0 ** -21)).all())
    for tiles in (1, 128, 300):
        x, squares = torch.randn(5, H, generator=g, device="cuda").to(torch.bfloat16), torch.rand(5, tiles, generator=g, device="cuda")
        out = torch.empty_like(x)
        backend.scale_rows(x, squares, 1e-5, out)
        exact = x.double() / (squares.double().sum(-1, keepdim=True) / H + 1e-5).sqrt()
        assert bool(((out.double() - exact).abs() <= exact.abs() * (2.0 ** -8 + 2.0 ** -20)).all())


@pytest.mark.parametrize("B, H, D, rank", [(200, 1, 40, 7), (70, 2, 64, 64), (70, 1, 128, 100), (40, 3, 80, 129), (60, 1, 160, 16), (40, 1, 256, 65)])
def test_recurrences_of_many_requests_at_once(ops, B, H, D, rank):
    """More chains than two a compute unit, of one to four chunks, which are asked for otherwise than few chains are: the bits that each
    request gives alone, and zeros from states of others nowhere."""
    g = torch.Generator(device="cuda").manual_seed(D)
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    lens = [1 + (17 * i) % 50 for i in range(B)]
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    T, n = cu[-1], H * D
    r, k, v, gate = (rand(T, n).to(torch.bfloat16) for _ in range(4))
    z, w2, w0, u = 2.0 * rand(T, rank), (rand(n, rank) * rank ** -0.5).to(torch.bfloat16), rand(n) - 1.0, rand(H, D)
    start = rand(B, H, D, D)
    ints = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")

    def run(first, last):
        at, end = cu[first], cu[last]
        batch = ops.AttentionBatch(num_tokens=end - at, num_requests=last - first, token_req=ints([i - first for i in range(first, last) for _ in range(lens[i])]),
                                   positions=ints([7 + j for i in range(first, last) for j in range(lens[i])]), cu_seqlens_q=ints([c - at for c in cu[first:last + 1]]),
                                   context_lens=ints([7 + m for m in lens[first:last]]), max_q_len=50, max_context_len=57)
        state = start.clone()
        y = ops.linear_recurrence(ops.WKV(z[at:end], w2, w0, u), r[at:end], k[at:end], v[at:end], gate[at:end], state, 1e-5, batch, ints(list(range(first, last))), torch.bfloat16)
        return y, state

    y, state = run(0, B)
    assert bool(torch.isfinite(y).all()) and bool(torch.isfinite(state).all())
    for i in range(0, B, 7):
        alone, left = run(i, i + 1)
        assert torch.equal(y[cu[i]:cu[i + 1]], alone) and torch.equal(state[i], left[i])
