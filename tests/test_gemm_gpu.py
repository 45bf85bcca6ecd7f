"""Projection GEMM parity (y = x W^T) against a plain PyTorch reference.

f16: compared with the f32-accumulated product rounded to half, within one
half ulp plus 1e-3 (the reference's rule, neural.rs:466-480).  f32: compared
with an f64 product, relative to the norm of the terms.  SwiGLU: compared with
the reference's half rounding steps, and with the unfused kernels.
"""
import pytest
import torch

gpu = pytest.mark.gpu


@pytest.fixture(scope="module")
def clef():
    import clef_hip
    clef_hip.lib()
    return clef_hip


def _inputs(seed, M, N, K, dtype):
    import workloads
    return workloads.gemm_inputs(seed, M, N, K, dtype=dtype)


def _check_f16(y, x, w):
    ref = (x.float() @ w.float().T)
    exp = ref.half().float()
    err = (y.float() - exp).abs()
    tol = 1e-3 + exp.abs() * 2.0 ** -10
    assert (err <= tol).all(), f"max err {err.max().item():.3e}"


def _check_f32(y, x, w):
    ref = x.double() @ w.double().T
    scale = x.double().abs() @ w.double().abs().T
    err = (y.double() - ref).abs()
    assert (err <= 1e-5 * scale + 1e-6).all(), f"max rel err {(err / (scale + 1e-30)).max().item():.3e}"


SHAPES = [(1, 1, 1), (17, 73, 65), (139, 129, 128), (17, 73, 4096), (513, 137, 65), (1025, 257, 128),
          (4096, 3000, 256)]  # the last: 192-wide tiles, ragged last column


@gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_gemm_reference_shapes(clef, M, N, K, dtype):
    """neural.rs:439-480 shapes, including ragged tiles and unaligned K."""
    x, w = _inputs(7, M, N, K, dtype)
    y = clef.gemm(x, w)
    (_check_f16 if dtype == torch.float16 else _check_f32)(y, x, w)


@gpu
@pytest.mark.parametrize("N", [8192, 2048, 6144, 12352, 9216])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_gemm_projection_shapes(clef, N, dtype):
    """M = 2048 tokens, K = 2048 hidden; x ~ N(0,1), W ~ N(0,0.02), seed 1."""
    x, w = _inputs(1, 2048, N, 2048, dtype)
    y = clef.gemm(x, w)
    (_check_f16 if dtype == torch.float16 else _check_f32)(y, x, w)


@gpu
@pytest.mark.parametrize("M,N,K", [(2100, 12300, 128), (2100, 12300, 2048), (2048, 9216, 2048), (4096, 12288, 192),
                                   (2100, 2100, 256),  # 289 tiles of 128 x 128
                                   # 256 x 128 tiles on four waves: one whole round, and
                                   # ragged rows and columns
                                   (4096, 2048, 512), (4000, 1900, 320)])
def test_gemm_persistent_launches(clef, M, N, K):
    """More tiles than CUs: one work-group per CU runs several tiles, the
    next tile's first stages requested during the current one's last.
    Ragged rows and columns, two K stages, a partial last round, 192-wide
    tiles, 128 x 128 tiles (three-slot rings); the f32 output (one tile per
    work-group) must agree bit for bit once rounded."""
    x, w = _inputs(9, M, N, K, torch.float16)
    y = clef.gemm(x, w)
    _check_f16(y, x, w)
    assert torch.equal(clef.gemm(x, w, out_dtype=torch.float32).half(), y)


@gpu
@pytest.mark.parametrize("M,N,K", [(2100, 6150, 128), (2048, 6144, 2048)])
def test_swiglu_persistent_launches(clef, M, N, K):
    gen = torch.Generator(device="cuda").manual_seed(15)
    x = torch.randn((M, K), generator=gen, device="cuda").half()
    wg = (torch.randn((N, K), generator=gen, device="cuda") * 0.05).half()
    wu = (torch.randn((N, K), generator=gen, device="cuda") * 0.05).half()
    y = clef.gemm_swiglu(x, wg, wu)
    assert torch.equal(y, clef.silu_mul(clef.gemm(x, wg), clef.gemm(x, wu)))


@gpu
@pytest.mark.parametrize("M,N,K", [(4096, 2048, 4096), (4096, 2048, 6144), (20, 16, 8), (300, 203, 128),
                                   (4096, 3000, 256),
                                   # residual tiles read during the last eight K stages: full and
                                   # partial tiles in one launch, exactly eight stages, an odd row
                                   # pitch (no vector access), 128 x 128 tiles
                                   (1000, 2000, 1024), (768, 2048, 512), (600, 2001, 1024),
                                   (256, 1024, 768)])
def test_gemm_residual_epilogue(clef, M, N, K):
    x, w = _inputs(3, M, N, K, torch.float16)
    h = torch.randn((M, N), device="cuda")
    h0 = h.clone()
    clef.gemm(x, w, residual=h, out_dtype=torch.float16)
    prod = (x.float() @ w.float().T).half().float()
    exp = h0 + prod
    err = (h - exp).abs()  # one half ulp of the product, plus the f32 add
    assert (err <= 1e-3 + prod.abs() * 2.0 ** -10 + exp.abs() * 2.0 ** -23).all(), \
        f"max err {err.max().item():.3e}"


@gpu
@pytest.mark.parametrize("M,N,K", [(512, 256, 256), (300, 203, 128), (1024, 1024, 1024)])
def test_gemm_residual_epilogue_unrounded(clef, M, N, K):
    """Residual add of the f32 accumulator itself (no half rounding), aligned
    and ragged rows, and residual tiles read during the last K stages."""
    x, w = _inputs(8, M, N, K, torch.float16)
    h = torch.randn((M, N), device="cuda")
    h0 = h.clone()
    clef.gemm(x, w, residual=h, out_dtype=torch.float32)
    prod = x.double() @ w.double().T
    scale = x.double().abs() @ w.double().abs().T
    err = (h.double() - (h0.double() + prod)).abs()
    assert (err <= 1e-5 * scale + 2e-6 * (h0.double().abs() + 1)).all(), f"max err {err.max().item():.3e}"


@gpu
def test_gemm_f16_output_from_f32_accumulator_rounds_once(clef):
    x, w = _inputs(4, 300, 200, 512, torch.float16)
    y32 = clef.gemm(x, w, out_dtype=torch.float32)
    y16 = clef.gemm(x, w)
    assert torch.equal(y32.half(), y16)


@gpu
@pytest.mark.parametrize("M,N,K", [(2048, 6144, 2048), (600, 6144, 2048), (20, 32, 16), (513, 137, 64)])
def test_swiglu_matches_half_rounding_steps_and_unfused_kernels(clef, M, N, K):
    import workloads
    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn((M, K), generator=gen, device="cuda").half()
    wg = (torch.randn((N, K), generator=gen, device="cuda") * 0.02).half()
    wu = (torch.randn((N, K), generator=gen, device="cuda") * 0.02).half()
    y = clef.gemm_swiglu(x, wg, wu)
    g16, u16 = clef.gemm(x, wg), clef.gemm(x, wu)
    # the reference's rule: the fused kernel equals the unfused kernels
    assert torch.equal(y, clef.silu_mul(g16, u16))
    # the half-rounding steps with an exactly rounded SiLU: the hardware SiLU
    # moves the rounded silu by one ulp in rare cases, which the product
    # carries to at most two ulps of the output
    g, u = g16.float(), u16.float()
    s = (g / (1.0 + torch.exp(-g))).half().float()
    unfused = (s * u).half()
    diff = (y.float() - unfused.float()).abs()
    ulp = unfused.float().abs().clamp(min=2.0 ** -14) * 2.0 ** -10
    assert (diff <= 2 * ulp).all()
    assert (diff == 0).float().mean() > 0.999
    gr = (x.float() @ wg.float().T).half().float()
    ur = (x.float() @ wu.float().T).half().float()
    ref = ((gr / (1 + torch.exp(-gr))).half().float() * ur).half().float()
    err = (y.float() - ref).abs()
    assert (err <= 1e-3 + ref.abs() * 2.0 ** -9).all(), f"max err {err.max().item():.3e}"


@gpu
def test_swiglu_f32(clef):
    gen = torch.Generator(device="cuda").manual_seed(6)
    x = torch.randn((333, 256), generator=gen, device="cuda")
    wg = torch.randn((500, 256), generator=gen, device="cuda") * 0.05
    wu = torch.randn((500, 256), generator=gen, device="cuda") * 0.05
    y = clef.gemm_swiglu(x, wg, wu)
    g = x.double() @ wg.double().T
    ref = torch.nn.functional.silu(g) * (x.double() @ wu.double().T)
    assert (y.double() - ref).abs().max().item() < 1e-4


@gpu
def test_swiglu_f32_projection_shape(clef):
    """The f32 SwiGLU the bench times: M = K = 2048, N = 6144 gate and up,
    x ~ N(0,1), W ~ N(0,0.02) (seeds 1 and 2), against an f64 product; the
    bound carries each projection's f32 accumulation error (relative to its
    terms' magnitudes) through silu(g) u."""
    x, wg = _inputs(1, 2048, 6144, 2048, torch.float32)
    _, wu = _inputs(2, 2048, 6144, 2048, torch.float32)
    y = clef.gemm_swiglu(x, wg, wu).double()
    xd = x.double()
    g, u = xd @ wg.double().T, xd @ wu.double().T
    sg, su = xd.abs() @ wg.double().abs().T, xd.abs() @ wu.double().abs().T
    sil = torch.nn.functional.silu(g)
    ref = sil * u
    tol = 1e-5 * (1.1 * sg * u.abs() + sil.abs() * su) + 2e-6 * ref.abs() + 1e-7
    err = (y - ref).abs()
    assert (err <= tol).all(), f"max err {err.max().item():.3e}, worst ratio {(err / tol).max().item():.2f}"


@gpu
@pytest.mark.parametrize("dt", [torch.float16, torch.float32])
def test_silu_mul_matches_the_formula(clef, dt):
    """clef_silu_mul: f32 as silu(g) * u; f16 with the SwiGLU's half roundings,
    the SiLU within one f16 ulp of the exactly rounded one."""
    gen = torch.Generator(device="cuda").manual_seed(12)
    g = (4 * torch.randn(100_003, generator=gen, device="cuda")).to(dt)
    u = torch.randn(100_003, generator=gen, device="cuda").to(dt)
    y = clef.silu_mul(g, u).float()
    gf, uf = g.float(), u.float()
    if dt == torch.float32:
        torch.testing.assert_close(y, gf / (1 + torch.exp(-gf)) * uf, rtol=1e-6, atol=1e-7)
    else:
        ref = ((gf / (1 + torch.exp(-gf))).half().float() * uf).half().float()
        ulp = ref.abs().clamp(min=2.0 ** -14) * 2.0 ** -10
        assert ((y - ref).abs() <= 2 * ulp).all()
        assert (y == ref).float().mean() > 0.999


def test_silu_mul_rejects_bad_arguments(clef):
    """Validation before any launch (no GPU needed)."""
    assert clef.lib().clef_silu_mul(None, None, None, 16, 1, None) < 0
    assert clef.lib().clef_silu_mul(1, 1, 1, 0, 1, None) < 0
    assert clef.lib().clef_silu_mul(1, 1, 1, 16, 7, None) < 0


# launches on small tiles (32 x 16, 64 x 32, 64 x 64, 128 x 64): one row, tile
# edges and remainders in rows and columns, odd row pitches, one K stage,
# partial stages (K = 320, 192), a request-sized call of each projection.  With
# 12288 rows N = 1000 and more takes 128- or 256-row tiles of the other kernels,
# N = 100 and 73 still 128 x 64 (their columns' edges; the order of their sums is
# that of N = 1000 with the same K)
SMALL = [(1, 2048, 6144), (33, 2048, 6144), (31, 100, 64), (31, 1000, 64), (64, 1000, 320), (65, 73, 192),
         (65, 1000, 192), (200, 2048, 4096), (129, 2047, 1024), (1, 12288, 2048), (37, 12288, 2048),
         (100, 12288, 2048), (300, 2048, 2048), (500, 2000, 512), (1000, 2048, 6144)]


@gpu
@pytest.mark.parametrize("M,N,K", SMALL)
def test_gemm_small_tiles(clef, M, N, K):
    """Each epilogue against the reference, and equal bit for bit to the same
    rows of a call of 12288 rows (one summation order on all tiles)."""
    x, w = _inputs(21, M, N, K, torch.float16)
    _, u = _inputs(22, 1, N, K, torch.float16)
    rows = 4096 * 3
    xl = torch.cat([x, torch.zeros((rows - M, K), dtype=x.dtype, device="cuda")])
    y = clef.gemm(x, w)
    _check_f16(y, x, w)
    assert torch.equal(y, clef.gemm(xl, w)[:M])
    assert torch.equal(clef.gemm(x, w, out_dtype=torch.float32).half(), y)
    h0 = torch.randn((M, N), device="cuda")
    h = clef.gemm(x, w, residual=h0.clone(), out_dtype=torch.float16)
    assert torch.equal(h, h0 + y.float())
    s = clef.gemm_swiglu(x, w, u)
    assert torch.equal(s, clef.silu_mul(y, clef.gemm(x, u)))
    assert torch.equal(s, clef.gemm_swiglu(xl, w, u)[:M])


@gpu
def test_gemm_small_tiles_write_only_their_rows(clef):
    """Strided operands and outputs (views into wider buffers): nothing outside
    the output's rows and columns is written."""
    M, N, K = 45, 90, 128
    xb, wb = _inputs(23, M, N, 2 * K, torch.float16)
    x, w = xb[:, K:], wb[:, :K]
    buf = torch.full((M + 3, N + 30), 7.0, device="cuda").half()
    clef.gemm(x, w, out=buf[:M, 8:8 + N])
    _check_f16(buf[:M, 8:8 + N], x, w)
    assert (buf[M:] == 7).all() and (buf[:, :8] == 7).all() and (buf[:, 8 + N:] == 7).all()


# a few rows past whole rounds of large tiles: one call as two launches (one
# row, a partial small tile, most of a tile row; N off the tile edges)
SPLIT_ROWS = [(1281, 12288, 2048), (1400, 12288, 1024), (1296, 12281, 1536), (1801, 9216, 2048), (2600, 6144, 2048)]


@gpu
@pytest.mark.parametrize("M,N,K", SPLIT_ROWS)
def test_gemm_split_rows(clef, M, N, K):
    """Every row equals the same row of calls of 700 and fewer rows, which are
    single launches on other tiles; rows of a wider buffer, nothing else written."""
    x, w = _inputs(24, M, N, K, torch.float16)
    _, u = _inputs(25, 1, N, K, torch.float16)
    parts = [slice(i, min(i + 700, M)) for i in range(0, M, 700)]
    buf = torch.full((M + 2, N + 16), 7.0, device="cuda").half()
    y = clef.gemm(x, w, out=buf[:M, 8:8 + N])
    _check_f16(y, x, w)
    assert torch.equal(y, torch.cat([clef.gemm(x[r], w) for r in parts]))
    assert (buf[M:] == 7).all() and (buf[:, :8] == 7).all() and (buf[:, 8 + N:] == 7).all()
    assert torch.equal(clef.gemm(x, w, out_dtype=torch.float32).half(), y)
    h0 = torch.randn((M, N), device="cuda")
    assert torch.equal(clef.gemm(x, w, residual=h0.clone(), out_dtype=torch.float16), h0 + y.float())
    s = clef.gemm_swiglu(x, w, u)
    assert torch.equal(s, clef.silu_mul(y.contiguous(), clef.gemm(x, u)))
    assert torch.equal(s, torch.cat([clef.gemm_swiglu(x[r], w, u) for r in parts]))


# f32 operands with 16-byte rows: each tile shape (32 x 32 .. 256 x 128), edges
# and remainders in rows and columns, K of one float4, below one step, ragged
# steps and stages
F32_SPLIT = [(1, 16, 4), (31, 33, 28), (33, 100, 196), (1, 2048, 6144), (65, 2047, 132), (300, 2048, 1028),
             (500, 8192, 96), (129, 4099, 64), (2048, 8192, 256), (1100, 9216, 100)]


def _f32_split_bound(K):
    return ((1 + 2.0 ** -10) + 2 * -(-K // 32) + -(-K // 128) + 1) * 2.0 ** -24


@gpu
@pytest.mark.parametrize("signs", [False, True])
@pytest.mark.parametrize("M,N,K", [(33, 2048, 4), (33, 2048, 32), (300, 2000, 100), (2048, 8192, 64)])
def test_gemm_f32_split_worst_significands(clef, M, N, K, signs):
    """The significands whose split drops most (2^-24.01 of a product; found over all 2^23),
    of one sign, where the dropped parts add up, and of both."""
    bits = torch.tensor([0x3f807fc0, 0x3f808040, 0x3f807f40, 0x3f8080c0], dtype=torch.int32, device="cuda")
    worst = bits.view(torch.float32)
    gen = torch.Generator(device="cuda").manual_seed(45)

    def draw(*shape):
        v = worst[torch.randint(4, shape, generator=gen, device="cuda")]
        v = v * 2.0 ** torch.randint(-3, 4, shape, generator=gen, device="cuda").float()
        return v * (1 - 2 * torch.randint(2, shape, generator=gen, device="cuda").float()) if signs else v

    x, w = draw(M, K), draw(N, K)
    y = clef.gemm(x, w).double()
    err = (y - x.double() @ w.double().T).abs()
    assert (err <= _f32_split_bound(K) * (x.double().abs() @ w.double().abs().T)).all()


@gpu
@pytest.mark.parametrize("M,N,K", F32_SPLIT)
def test_gemm_f32_split_tiles(clef, M, N, K):
    """The split drops at most (1 + 2^-10) 2^-24 of a term (mid lo + lo mid + lo lo, mid <=
    2^-8 and lo <= 2^-17 of the value) and rounds a sum twice per 32 columns, once more per
    128 and at the end: |err| <= ((1 + 2^-10) + 2 ceil(K / 32) + ceil(K / 128) + 1) 2^-24 sum|x w|."""
    x, w = _inputs(31, M, N, K, torch.float32)
    _, u = _inputs(32, 1, N, K, torch.float32)
    ref, scale = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    bound = _f32_split_bound(K) * scale
    y = clef.gemm(x, w)
    assert ((y.double() - ref).abs() <= bound).all()
    # in the 2-norm the error of a random sum is far smaller: below that of the
    # f32 MFMA kernel (1.0e-7 at K = 36, 2.7e-7 at K = 6144)
    assert (y.double() - ref).norm() <= 2e-7 * ref.norm()
    h0 = torch.randn((M, N), device="cuda")
    assert torch.equal(clef.gemm(x, w, residual=h0.clone()), h0 + y)
    assert torch.equal(clef.gemm(x, w, out_dtype=torch.float16), y.half())
    g, v = y, clef.gemm(x, u)
    s = clef.gemm_swiglu(x, w, u)
    assert torch.allclose(s, g / (1 + torch.exp(-g)) * v, rtol=2e-6, atol=1e-30)
    # a row does not depend on how many share the call
    xl = torch.cat([x, torch.zeros((4096, K), device="cuda")])
    assert torch.equal(clef.gemm(xl, w)[:M], y)


@gpu
@pytest.mark.parametrize("M", [20, 150, 300, 2048])
def test_gemm_f32_split_special_values(clef, M):
    """Infinities, NaN, values next to the largest float and far below 2^-100
    give what an f32 product gives."""
    N, K = 8192, 64
    x, w = _inputs(33, M, N, K, torch.float32)
    x[3, 5], x[7, 9], x[11, 2], x[12] = float("inf"), float("nan"), 3.4e38, 0.0
    w[100, 30] = -float("inf")
    x[13] *= 1e-32
    x[14] = torch.randn(K, device="cuda") * 1e-38  # subnormal parts
    w[200] *= 1e20
    y = clef.gemm(x, w).double()
    ref = x.double() @ w.double().T
    ok = ref.abs() <= 3.0e38
    scale = x.double().abs() @ w.double().abs().T
    assert ((y - ref).abs()[ok] <= (1e-6 * scale + 2.0 ** -145)[ok]).all()
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    big = ref.abs() > 3.5e38
    assert torch.isinf(y[big]).all() and torch.equal(y[big].sign(), ref[big].sign())


@gpu
@pytest.mark.parametrize("M,N,K", [(33, 2048, 6144), (33, 8192, 100), (200, 8192, 64), (500, 2048, 260)])
def test_gemm_f32_rows_do_not_depend_on_their_neighbours(clef, M, N, K):
    """A call's rows equal those of a call on larger tiles bit for bit with values below
    2^-100, infinities and NaN in other rows and columns as well as their own, for each
    epilogue; rows and columns without such values equal those of a call without any."""
    x, w = _inputs(41, M, N, K, torch.float32)
    _, u = _inputs(42, 1, N, K, torch.float32)
    plain = clef.gemm(x, w)
    x[3, 5], x[7, 9], x[11, 2] = 1e-33, float("inf"), 1e-40
    w[0, 0], w[70, 1], w[200, 3] = 1e-31, float("nan"), -1e-38
    u[1, 2] = 1e-35
    xl = torch.cat([x, _inputs(43, 4096 - M, 1, K, torch.float32)[0]])
    xl[M + 1, 0], xl[-1, 1] = 1e-32, float("nan")

    def same(a, b):
        return torch.equal(torch.nan_to_num(a, nan=1e30), torch.nan_to_num(b, nan=1e30))

    y = clef.gemm(x, w)
    assert same(y, clef.gemm(xl, w)[:M])
    assert same(clef.gemm_swiglu(x, w, u), clef.gemm_swiglu(xl, w, u)[:M])
    h0 = torch.randn((4096, N), device="cuda")
    assert same(clef.gemm(x, w, residual=h0[:M].clone()), clef.gemm(xl, w, residual=h0.clone())[:M])
    assert same(clef.gemm(x, w, residual=h0[:M].clone()), h0[:M] + y)
    assert same(clef.gemm(x, w, out_dtype=torch.float16), y.half())
    rows = torch.ones(M, dtype=torch.bool)
    cols = torch.ones(N, dtype=torch.bool)
    rows[[3, 7, 11]] = False
    cols[[0, 70, 200]] = False
    assert torch.equal(y[rows][:, cols], plain[rows][:, cols])
    # strided outputs: the repeated elements go where they belong and nowhere else
    buf = torch.full((M + 2, N + 15), 7.0, device="cuda")
    clef.gemm(x, w, out=buf[:M, 5:5 + N])
    assert same(buf[:M, 5:5 + N], y)
    assert (buf[M:] == 7).all() and (buf[:, :5] == 7).all() and (buf[:, 5 + N:] == 7).all()


@gpu
@pytest.mark.parametrize("M", [33, 300, 2048])
def test_gemm_f32_small_terms_alone_keep_their_precision(clef, M):
    """Rows and columns whose products are all far below 2^-100: each term is one product,
    rounded once (and the other terms of those rows and columns as usual)."""
    N, K = 8192, 96
    x, w = _inputs(44, M, N, K, torch.float32)
    x[5], w[9] = 0.0, 0.0
    x[5, 40], w[9, 7] = 1.2345678e-34, -7.654321e-33
    y = clef.gemm(x, w).double()
    row, col = x[5, 40].double() * w[:, 40].double(), w[9, 7].double() * x[:, 7].double()
    row[9] = col[5] = 0.0
    assert ((y[5] - row).abs() <= 2.0 ** -23 * row.abs() + 2.0 ** -149).all()
    assert ((y[:, 9] - col).abs() <= 2.0 ** -23 * col.abs() + 2.0 ** -149).all()


@gpu
@pytest.mark.parametrize("M,N,K", [(1000, 6144, 128), (700, 6144, 64), (1024, 6100, 192), (3000, 6144, 64)])
def test_swiglu_192_wide_tiles(clef, M, N, K):
    """256 x 192 tiles (96 outputs): whole and ragged rows and columns, one to
    three K stages; equal to the unfused products."""
    x, wg = _inputs(25, M, N, K, torch.float16)
    _, wu = _inputs(26, 1, N, K, torch.float16)
    y = clef.gemm_swiglu(x, wg, wu)
    assert torch.equal(y, clef.silu_mul(clef.gemm(x, wg), clef.gemm(x, wu)))
