"""Each kernel alone against a plain fp32/fp64 reference of the same operation, at sizes other than the engine's
tiny configurations: sizes that are no power of two, head sizes in steps of 16, any number of heads and groups."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from jllm_serve_amd.kernels import ops
    ops.library()
    return ops


def bf16_close(got, want, ulps=1.0):
    """got (bf16 or f32 tensor) against a float64 reference: within `ulps` bf16 roundings of the reference."""
    want = want.double()
    err = (got.double() - want).abs()
    tol = ulps * (2.0 ** -8) * want.abs() + 1e-6 * want.abs().max()
    return bool((err <= tol).all()), float((err / (want.abs() + 1e-3 * want.abs().max())).max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_embed(ops, dtype):
    table = torch.randn(301, 80, device=DEV).to(dtype)
    ids = torch.tensor([0, 300, 7, 7, 150], dtype=torch.int32, device=DEV)
    out = ops.embed(table, ids, 1.0)
    assert out.dtype == torch.float32 and torch.equal(out, table[ids.long()].float())
    assert torch.equal(ops.embed(table, ids, 2.0), table[ids.long()].float() * 2.0)


@pytest.mark.parametrize("d", [16, 80, 96, 4096, 5000])
@pytest.mark.parametrize("gdt,odt", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16)])
def test_rmsnorm(ops, d, gdt, odt):
    x = torch.randn(7, d, device=DEV) * 3
    x[2] = 0  # an all-zero row gives zeros, not NaN
    g = (torch.rand(d, device=DEV) + 0.5).to(gdt)
    eps = 1e-5
    ref = (x.double() * torch.rsqrt((x.double() ** 2).mean(-1, keepdim=True) + eps)) * g.double()
    out = ops.rmsnorm(x, g, eps, odt)
    if odt == torch.float32:
        assert torch.allclose(out.double(), ref, rtol=2e-6, atol=1e-6)
    else:
        assert bf16_close(out, ref)[0]
    rows = torch.tensor([5, 0, 5], dtype=torch.int32, device=DEV)
    assert torch.equal(ops.rmsnorm(x, g, eps, odt, rows), out[rows.long()])


@pytest.mark.parametrize("d", [4, 1020, 1024, 4096, 8192])
@pytest.mark.parametrize("gdt", [torch.float32, torch.bfloat16])
def test_rmsnorm_has_the_same_bits_at_any_alignment(ops, d, gdt):
    """Rows and gains that begin anywhere in a 16-byte piece (pieces of a larger tensor) against those that begin with one."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(d)
    x = torch.randn(9, d, device=DEV, generator=gen) * 3
    g = (torch.rand(d, device=DEV, generator=gen) + 0.5).to(gdt)
    want = ops.rmsnorm(x, g, 1e-5, torch.float32)
    for at in (1, 2, 3, 5):
        gains = torch.zeros(d + 8, device=DEV, dtype=gdt)[at:at + d]
        gains.copy_(g)
        rows = torch.zeros(9 * d + 8, device=DEV)[at:at + 9 * d].view(9, d)
        rows.copy_(x)
        assert gains.data_ptr() % 16 and rows.data_ptr() % 16
        assert torch.equal(ops.rmsnorm(x, gains, 1e-5, torch.float32), want) and torch.equal(ops.rmsnorm(rows, g, 1e-5, torch.float32), want)


GEMM_SHAPES = [(1, 16, 128), (5, 48, 384), (16, 4096, 128), (17, 80, 256), (33, 16, 1024), (64, 304, 640), (50, 144, 2176),
               (20, 4112, 512),
               (8, 6144, 256), (3, 6144, 128), (16, 6144, 1152),  # 24 weight rows per workgroup (N / 24 = 256 of them)
               (8, 5120, 256), (1, 5120, 1152), (13, 7168, 384), (16, 10240, 128),  # 20 weight rows per workgroup for N = 5120
               (5, 32768, 128), (16, 32800, 256),  # thousands of 16-row tiles
               (100, 256, 64), (70, 200, 192), (90, 136, 320),  # one, three and five stages of the tiled kernel's rings
               (3, 50, 70), (65, 96, 128), (200, 130, 96), (128, 256, 512), (300, 384, 4096), (1000, 192, 136)]


@pytest.mark.parametrize("M,N,K", GEMM_SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gemm_epilogues(ops, M, N, K, dtype):
    torch.manual_seed(M * 7 + N)
    a = torch.randn(M, K, device=DEV).to(dtype)
    w = (torch.randn(N, K, device=DEV) / math.sqrt(K)).to(dtype)
    w2 = (torch.randn(N, K, device=DEV) / math.sqrt(K)).to(dtype)
    bias = torch.randn(N, device=DEV)
    ref = a.double() @ w.double().T
    exact = dtype == torch.float32
    # store, fp32 out (the output head)
    out = ops.gemm(a, w, out_dtype=torch.float32, exact=exact)
    assert torch.allclose(out.double(), ref, rtol=1e-5, atol=2e-5 * ref.abs().max())
    # store in the activations' type with a bias, from a strided input view
    wide = torch.cat([a, a], dim=1)
    out = ops.gemm(wide[:, K:], w, bias=bias, exact=exact)
    assert out.dtype == dtype
    if exact:
        assert torch.allclose(out.double(), ref + bias.double(), rtol=1e-5, atol=2e-5 * ref.abs().max())
    else:
        assert bf16_close(out, ref + bias.double())[0]
    # add into the fp32 residual
    res = torch.randn(M, N, device=DEV)
    want = res.double() + ref
    ops.gemm(a, w, out=res, epilogue=ops.EPI_ADD, exact=exact)
    assert torch.allclose(res.double(), want, rtol=1e-5, atol=2e-5 * want.abs().max())
    # gated: silu(a w^T) * (a w2^T)
    g, u = ref, a.double() @ w2.double().T
    want = (g / (1 + torch.exp(-g))) * u
    out = ops.gemm(a, w, w2=w2, epilogue=ops.EPI_GATED, exact=exact)
    if exact:
        assert torch.allclose(out.double(), want, rtol=1e-5, atol=2e-5 * want.abs().max())
    else:
        assert bf16_close(out, want, ulps=1.01)[0]


def test_gemm_large_tile(ops, monkeypatch):
    """Products of many tiles in tiles of 256 rows, whatever the choice between tiles makes of so short a K: all three epilogues at sizes that
    leave partial tiles in both directions, and the same bits as the smaller tiles give for the same rows."""
    own = ops._tiled_choice
    monkeypatch.setattr(ops, "_tiled_choice", lambda m, *rest: (256, 1) if m > 128 else own(m, *rest))
    torch.manual_seed(5)
    M, N, K = 530, 43800, 192
    a = torch.randn(M, K, device=DEV).bfloat16()
    w = (torch.randn(N, K, device=DEV) / math.sqrt(K)).bfloat16()
    bias = torch.randn(N, device=DEV)
    ref = a.double() @ w.double().T
    ops.reset_stats()
    out = ops.gemm(a, w, out_dtype=torch.float32)
    assert torch.allclose(out.double(), ref, rtol=1e-5, atol=2e-5 * ref.abs().max())
    small = ops.gemm(a[:100].contiguous(), w, out_dtype=torch.float32)
    assert torch.equal(small, out[:100])
    assert ops.stats()["ran"] == {"jllm_gemm_pingpong_bf16": 1, "jllm_gemm_mfma_bf16": 1}
    assert bf16_close(ops.gemm(a, w, bias=bias), ref + bias.double())[0]
    res = torch.randn(M, N, device=DEV)
    want = res.double() + ref
    ops.gemm(a, w, out=res, epilogue=ops.EPI_ADD)
    assert torch.allclose(res.double(), want, rtol=1e-5, atol=2e-5 * want.abs().max())
    del out, res, want, ref, small
    N = 21900
    w = (torch.randn(N, K, device=DEV) / math.sqrt(K)).bfloat16()
    w2 = (torch.randn(N, K, device=DEV) / math.sqrt(K)).bfloat16()
    g, u = a.double() @ w.double().T, a.double() @ w2.double().T
    want = (g / (1 + torch.exp(-g))) * u
    out = ops.gemm(a, w, w2=w2, epilogue=ops.EPI_GATED)
    assert bf16_close(out, want, ulps=1.01)[0]
    assert torch.equal(ops.gemm(a[:100].contiguous(), w, w2=w2, epilogue=ops.EPI_GATED), out[:100])
    # 200 large tiles: one round that fills most of the compute units also takes the large tile
    M, N = 1990, 6300
    a = torch.randn(M, K, device=DEV).bfloat16()
    w = (torch.randn(N, K, device=DEV) / math.sqrt(K)).bfloat16()
    ref = a.double() @ w.double().T
    out = ops.gemm(a, w, out_dtype=torch.float32)
    assert torch.allclose(out.double(), ref, rtol=1e-5, atol=2e-5 * ref.abs().max())
    assert torch.equal(ops.gemm(a[:100].contiguous(), w, out_dtype=torch.float32), out[:100])


@pytest.mark.parametrize("M,N,K,plan", [(1500, 8200, 160, (256, 1)), (2048, 6144, 1024, (256, 1)), (300, 25000, 128, (256, 1)),
                                        (520, 16400, 4096, (256, 1)), (2000, 4096, 8192, (256, 2)), (1024, 6140, 8256, (256, 2)),
                                        (1000, 4100, 8192, (256, 2)), (640, 4100, 8192, (256, 4)), (1024, 6144, 4096, (256, 2))])
def test_gemm_two_group_kernel(ops, monkeypatch, M, N, K, plan):
    """The large tiles' kernel (loads straight to LDS, a ring of half stages) with its tile of 256
    rows, whatever the choice between tiles makes of these sizes: every epilogue, with a bias, partial tiles in both directions, K from four stages to many, inputs and
    outputs whose rows are not contiguous, K cut in two or four with partial sums (also an odd number of stages per half);
    against float64."""
    assert ops._pingpong_plan(M, N, K, False) == plan
    monkeypatch.setattr(ops, "_tiled_plan", lambda m, n, k, gated: (256, 1) if gated else plan)
    torch.manual_seed(M + N + K)
    a = torch.randn(M, K, device=DEV).bfloat16()
    w = (torch.randn(N, K, device=DEV) / math.sqrt(K)).bfloat16()
    bias = torch.randn(N, device=DEV)
    ref = a.double() @ w.double().T
    ops.reset_stats()
    out = ops.gemm(a, w, out_dtype=torch.float32)
    assert ops.stats()["ran"].get("jllm_gemm_pingpong_bf16") == 1, ops.stats()
    assert torch.allclose(out.double(), ref, rtol=1e-5, atol=2e-5 * ref.abs().max())
    wide = torch.cat([a, a], dim=1)
    assert bf16_close(ops.gemm(wide[:, K:], w, bias=bias), ref + bias.double())[0]
    res = torch.randn(M, N, device=DEV)
    want = res.double() + ref + bias.double()
    ops.gemm(a, w, bias=bias, out=res, epilogue=ops.EPI_ADD)
    assert torch.allclose(res.double(), want, rtol=1e-5, atol=2e-5 * want.abs().max())
    if ops._pingpong_plan(M, N // 2, K, True)[0]:
        w1, w2 = w[:N // 2], w[N // 2:2 * (N // 2)]
        g, u = ref[:, :N // 2], ref[:, N // 2:2 * (N // 2)]
        want = (g / (1 + torch.exp(-g))) * u
        out = ops.gemm(a, w1.contiguous(), w2=w2.contiguous(), epilogue=ops.EPI_GATED)
        assert bf16_close(out, want, ulps=1.01)[0]
    assert ops.stats()["ran"].get("jllm_gemm_pingpong_bf16") >= 3 and not ops.stats()["general"], ops.stats()


@pytest.mark.parametrize("M,N,K,cut", [(193, 520, 160, 1), (600, 2500, 128, 1), (575, 1300, 2048, 2), (577, 700, 4224, 4)])
def test_gemm_two_group_kernel_with_tiles_of_192_rows(ops, monkeypatch, M, N, K, cut):
    """The 192-row tile (waves of one group load four chunks of a stage, the other's three) against the 256-row tile, bit
    for bit: one row beyond a tile and one short of it, K from four stages on and cut in two and four, every epilogue."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(M + K)
    a = torch.randn(M, K, device=DEV, generator=gen).bfloat16()
    w, w2 = ((torch.randn(N, K, device=DEV, generator=gen) * K ** -0.5).bfloat16() for _ in range(2))
    bias = torch.randn(N, device=DEV, generator=gen)

    def outputs(rows):
        monkeypatch.setattr(ops, "_tiled_plan", lambda m, n, k, gated: (rows, 1 if gated else cut))
        ops.reset_stats()
        res = torch.ones(M, N, device=DEV)
        ops.gemm(a, w, bias=bias, out=res, epilogue=ops.EPI_ADD)
        got = [res, ops.gemm(a, w, out_dtype=torch.float32), ops.gemm(a, w, bias=bias), ops.gemm(a, w, w2=w2, epilogue=ops.EPI_GATED)]
        assert ops.stats()["ran"] == {"jllm_gemm_pingpong_bf16": 4}
        return got

    tall, got = outputs(256), outputs(192)
    assert all(torch.equal(x, y) for x, y in zip(got, tall))
    ref = a.double() @ w.double().T  # fp32 sums of K rounded products: K 2^-24 of the sum of magnitudes at most
    assert bool(((got[1].double() - ref).abs() <= K * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)).all())


@pytest.mark.parametrize("M,N,K,cut", [(257, 520, 128, 1), (320, 131, 160, 1), (321, 1300, 192, 1), (640, 700, 3200, 3), (512 + 60, 2500, 5376, 5)])
def test_gemm_two_group_kernel_with_wide_last_rows(ops, monkeypatch, M, N, K, cut):
    """The last 1 to 64 or 65 to 128 rows in tiles of twice the columns against tiles of 256 rows throughout: both edges of either
    kind, an odd number of column tiles (the last wide one is half beyond the end), K from four stages on and in parts of unequal
    length, every epilogue. Sums that are stored or added have the same bits. The gated epilogue takes the hardware's exponential and
    reciprocal in tiles that lie inside the output and the library's in others, and which rows that are differs between the
    tilings: some 2^-22 of the value, so neighbouring bf16 numbers at most."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(M + K)
    a = torch.randn(M, K, device=DEV, generator=gen).bfloat16()
    w, w2 = ((torch.randn(N, K, device=DEV, generator=gen) * K ** -0.5).bfloat16() for _ in range(2))
    bias = torch.randn(N, device=DEV, generator=gen)

    def outputs(rows):
        monkeypatch.setattr(ops, "_tiles", lambda m, n, k, gated, *plan: (rows, 1 if gated else cut))
        ops.reset_stats()
        res = torch.ones(M, N, device=DEV)
        ops.gemm(a, w, bias=bias, out=res, epilogue=ops.EPI_ADD)
        got = [res, ops.gemm(a, w, out_dtype=torch.float32), ops.gemm(a, w, bias=bias), ops.gemm(a, w, w2=w2, epilogue=ops.EPI_GATED)]
        assert ops.stats()["ran"] == {"jllm_gemm_pingpong_bf16": 4}
        return got

    monkeypatch.setattr(ops, "_wide_plan", lambda *_: None)
    tall, got = outputs(256), outputs(ops.WIDE_LAST)
    assert all(torch.equal(x, y) for x, y in zip(got[:3], tall[:3]))
    x, y = got[3].double(), tall[3].double()
    assert bool(((x - y).abs() <= 2.0 ** -7 * torch.maximum(x.abs(), y.abs())).all())
    ref = a.double() @ w.double().T  # fp32 sums of K rounded products: K 2^-24 of the sum of magnitudes at most
    assert bool(((got[1].double() - ref).abs() <= K * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)).all())


@pytest.mark.parametrize("M,N,K,cut", [(65, 68, 64, 1), (129, 131, 128, 1), (255, 260, 320, 2), (257, 516, 448, 3), (300, 1028, 1088, 5),
                                       (300, 260, 1088, 1), (129, 131, 1024, 1), (257, 516, 2176, 3), (200, 324, 704, 1), (70, 200, 960, 2)])
def test_gemm_small_tiles(ops, monkeypatch, M, N, K, cut):
    """Every tile of the small kernel against every other and against the tile of 256 x 256, bit for bit, and float64: one row beyond a tile
    and one short of it, odd numbers of column tiles, K of one stage, shorter than the rings (of three to five stages), and so long that
    every slot of every ring is filled again, an even and an odd number of stages, whole and in parts of unequal length, every epilogue. (Gated:
    tiles that lie inside the output take the hardware's exponential and reciprocal, others the library's, some 2^-22 of the value.)"""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(M + K)
    a = torch.randn(M, K, device=DEV, generator=gen).bfloat16()
    w, w2 = ((torch.randn(N, K, device=DEV, generator=gen) * K ** -0.5).bfloat16() for _ in range(2))
    bias = torch.randn(N, device=DEV, generator=gen)
    monkeypatch.setattr(ops, "_wide_plan", lambda *_: None)
    got = []
    for tile in ops.SMALL_TILES:
        monkeypatch.setattr(ops, "_tiled_choice", lambda m, n, k, gated, normed: (128128 if gated and tile == 64064 else tile, 1 if gated else cut))
        ops.reset_stats()
        res = torch.ones(M, N, device=DEV)
        ops.gemm(a, w, bias=bias, out=res, epilogue=ops.EPI_ADD)
        got.append([res, ops.gemm(a, w, out_dtype=torch.float32), ops.gemm(a, w, bias=bias), ops.gemm(a, w, w2=w2, epilogue=ops.EPI_GATED)])
        assert ops.stats()["ran"] == {"jllm_gemm_mfma_bf16": 4}
    if K // cut >= 128:
        monkeypatch.setattr(ops, "_tiled_choice", lambda m, n, k, gated, normed: (256, 1 if gated else cut))
        ops.reset_stats()
        res = torch.ones(M, N, device=DEV)
        ops.gemm(a, w, bias=bias, out=res, epilogue=ops.EPI_ADD)
        got.append([res, ops.gemm(a, w, out_dtype=torch.float32), ops.gemm(a, w, bias=bias), ops.gemm(a, w, w2=w2, epilogue=ops.EPI_GATED)])
        assert ops.stats()["ran"] == {"jllm_gemm_pingpong_bf16": 4}
    for other in got[1:]:
        assert all(torch.equal(x, y) for x, y in zip(got[0][:3], other[:3]))
        x, y = got[0][3].double(), other[3].double()
        assert bool(((x - y).abs() <= 2.0 ** -7 * torch.maximum(x.abs(), y.abs())).all())
    ref = a.double() @ w.double().T  # fp32 sums of K rounded products: K 2^-24 of the sum of magnitudes at most
    assert bool(((got[0][1].double() - ref).abs() <= K * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)).all())
    u = a.double() @ w2.double().T
    assert bf16_close(got[0][3], ref / (1 + torch.exp(-ref)) * u, ulps=1.01)[0]


@pytest.mark.parametrize("M,N,K,cut", [(256, 256, 128, 1), (257, 300, 160, 1), (320, 700, 288, 2), (300, 516, 1056, 3), (330, 260, 2080, 5)])
def test_gemm_ring_of_half_stages(ops, monkeypatch, M, N, K, cut):
    """A ring of halves of stages of 64: K of two stages, of whole ones and with a last one of 32, alone and as the end of the last of
    several parts of unequal length, shorter than the ring and longer, in all three tilings, which give the same bits."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(M + K)
    a = torch.randn(M, K, device=DEV, generator=gen).bfloat16()
    w = (torch.randn(N, K, device=DEV, generator=gen) * K ** -0.5).bfloat16()
    monkeypatch.setattr(ops, "_wide_plan", lambda *_: None)
    got = []
    for rows in (256, 192) + ((ops.WIDE_LAST,) if 1 <= M % 256 <= 128 else ()):
        monkeypatch.setattr(ops, "_tiles", lambda m, n, k, gated, *plan: (rows, cut))
        ops.reset_stats()
        got.append(ops.gemm(a, w, out_dtype=torch.float32))
        assert ops.stats()["ran"] == {"jllm_gemm_pingpong_bf16": 1}
    assert all(torch.equal(got[0], x) for x in got[1:])
    ref = a.double() @ w.double().T  # fp32 sums of K rounded products: K 2^-24 of the sum of magnitudes at most
    assert bool(((got[0].double() - ref).abs() <= K * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)).all())


@pytest.mark.parametrize("M,N,K,stride", [(66, 72, 128, (1 << 22) + 8), (130, 72, 192, (1 << 23) + 8), (65, 24, (1 << 23) + 64, (1 << 23) + 64)])
def test_gemm_of_very_long_rows(ops, M, N, K, stride):
    """Rows 8 and 16 MB and more apart, beyond the 32-bit offsets of a tile: still the tiled kernel. Small whole numbers, so that every sum
    is exact, at the ends of K and in between."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(M)
    at = sorted({0, 1, 63, 64, K // 2 - 1, K // 2, K - 65, K - 64, K - 1} & set(range(K)))
    whole = torch.zeros(M * stride, dtype=torch.bfloat16, device=DEV)
    a = whole.as_strided((M, K), (stride, 1))
    a[:, at] = torch.randint(-3, 4, (M, len(at)), device=DEV, generator=gen).bfloat16()
    w, w2 = (torch.zeros(N, K, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    for x in (w, w2):
        x[:, at] = torch.randint(-3, 4, (N, len(at)), device=DEV, generator=gen).bfloat16()
    g, u = (a[:, at].double() @ x[:, at].double().T for x in (w, w2))
    ops.reset_stats()
    assert torch.equal(ops.gemm(a, w, out_dtype=torch.float32).double(), g)
    res = torch.ones(M, N, device=DEV)
    ops.gemm(a, w, out=res, epilogue=ops.EPI_ADD)
    assert torch.equal(res.double(), g + 1)
    assert bf16_close(ops.gemm(a, w, w2=w2, epilogue=ops.EPI_GATED), g / (1 + torch.exp(-g)) * u, ulps=1.01)[0]
    assert ops.stats()["ran"] == {"jllm_gemm_mfma_bf16": 3} and not ops.stats()["general"], ops.stats()


@pytest.mark.parametrize("M,N,K", [(65, 520, 128), (130, 516, 192), (256, 1024, 256), (385, 131, 576)])
def test_the_small_tile_gives_the_bits_of_the_two_group_kernel(ops, monkeypatch, M, N, K):
    """Tiles of 128 x 128 (fragments of a whole stage in registers) against tiles of 256 x 256 (of half a stage): every
    epilogue at whole tiles, at edges and at rows that cannot be stored eight at a time, bit for bit."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(M + N)
    a = torch.randn(M, K, device=DEV, generator=gen).bfloat16()
    w, w2 = ((torch.randn(N, K, device=DEV, generator=gen) * K ** -0.5).bfloat16() for _ in range(2))
    bias = torch.randn(N, device=DEV, generator=gen)
    got = []
    for rows, kernel in ((256, "jllm_gemm_pingpong_bf16"), (0, "jllm_gemm_mfma_bf16")):
        monkeypatch.setattr(ops, "_tiled_plan", lambda m, n, k, gated, rows=rows: (rows, 1))
        monkeypatch.setattr(ops, "_k_splits", lambda m, n, k, gated: 1)
        ops.reset_stats()
        res = torch.ones(M, N, device=DEV)
        ops.gemm(a, w, bias=bias, out=res, epilogue=ops.EPI_ADD)
        got.append([res, ops.gemm(a, w, out_dtype=torch.float32), ops.gemm(a, w, bias=bias), ops.gemm(a, w, w2=w2, epilogue=ops.EPI_GATED)])
        assert ops.stats()["ran"] == {kernel: 4}
    assert all(torch.equal(x, y) for x, y in zip(*got))


@pytest.mark.parametrize("M,N,K,N2", [(1, 128, 256, 48), (5, 4096, 384, 4112), (8, 640, 4096, 304), (16, 304, 128, 16), (13, 5120, 1024, 640),
                                      (40, 1024, 1024, 512), (64, 2048, 2048, 768), (17, 1024, 4096, 256),
                                      # few rows, N / 16 just above the compute units: 20 weight rows per workgroup
                                      (8, 5120, 3072, 5120), (16, 5120, 4096, 640), (3, 5120, 3072, 5120), (11, 5120, 128, 7168),
                                      # few rows, few columns and a long K
                                      (8, 1024, 8192, 512), (3, 1280, 8192, 1024),
                                      # the consuming product with 24 weight rows per workgroup, and with thousands of tiles
                                      (8, 1024, 512, 6144), (13, 256, 256, 32768)])
@pytest.mark.parametrize("gdt", [torch.bfloat16, torch.float32])
def test_norm_between_two_products(ops, M, N, K, N2, gdt):
    """residual += a w^T (+ bias); h = RMSNorm(residual) w2^T without a norm launch: the first product leaves
    bf16(residual * gain) and partial sums of squares, the second scales its sums at the end (both weight-streaming
    kernels: up to 16 rows, and 17 to 64 rows with K cut in parts). Against float64, and
    against the same roundings in float64 (only fp32 summation is left). One residual entry is huge, so a norm over
    the wrong columns or rows shows."""
    torch.manual_seed(M * N + K)
    if N == 5120 and M <= 16:
        assert ops._skinny_second_rows(N, False) == 4, "this case is meant for workgroups with 20 weight rows"
    a = torch.randn(M, K, device=DEV).bfloat16()
    w = (torch.randn(N, K, device=DEV) / math.sqrt(K)).bfloat16()
    bias = torch.randn(N, device=DEV)
    res = torch.randn(M, N, device=DEV) * 2
    res[M // 2, N - 3] = 200.0
    gain = (torch.rand(N, device=DEV) + 0.5).to(gdt)
    w2 = (torch.randn(N2, N, device=DEV) / math.sqrt(N)).bfloat16()
    w3 = (torch.randn(N2, N, device=DEV) / math.sqrt(N)).bfloat16()
    eps = 1e-3
    want_res = res.double() + a.double() @ w.double().T + bias.double()
    promise = ops.gemm_add_then_norm(a, w, res, gain, eps, torch.bfloat16, bias=bias)
    assert promise.scaled is not None and promise.partials is not None, "the few-row product did not prepare the norm"
    assert torch.allclose(res.double(), want_res, rtol=1e-5, atol=2e-5 * want_res.abs().max())
    scale = torch.rsqrt((res.double() ** 2).mean(-1, keepdim=True) + eps)
    assert torch.allclose(promise.partials.double().sum(-1, keepdim=True), (res.double() ** 2).sum(-1, keepdim=True), rtol=1e-5)
    assert torch.equal(promise.scaled, (res * gain.float()).bfloat16())
    xn = res.double() * scale * gain.double()
    rounded = promise.scaled.double()
    fused = N % 128 == 0  # what the consuming kernels take (and partial sums in fours); else the norm is a launch of its own
    ref = xn @ w2.double().T
    tol = 5 * 2.0 ** -9 * torch.sqrt((xn ** 2) @ (w2.double() ** 2).T) + 1e-6
    if fused:
        out = ops.gemm(promise, w2, w2=w3, epilogue=ops.EPI_GATED, out_dtype=torch.float32)
        g_, u_ = (rounded @ w2.double().T) * scale, (rounded @ w3.double().T) * scale
        same = torch.nn.functional.silu(g_) * u_
        assert torch.allclose(out.double(), same, rtol=2e-4, atol=2e-5 * same.abs().max())
    out = ops.gemm(promise, w2, out_dtype=torch.float32)
    if fused:
        same = (rounded @ w2.double().T) * scale
        fp32_sum = 4e-6 * (rounded.abs() @ w2.double().abs().T) * scale + 1e-6
        assert bool(((out.double() - same).abs() <= fp32_sum).all())
    assert bool(((out.double() - ref).abs() <= tol).all())
    assert (promise._rows is None) == fused, "the norm ran as a launch of its own exactly when it had to"
    # the long way gives the same within bf16 rounding; many rows and 32-bit runs take it by themselves
    long_way = ops.gemm(ops.rmsnorm(res, gain, eps, torch.bfloat16), w2, out_dtype=torch.float32)
    assert bool(((out.double() - long_way.double()).abs() <= 2 * tol).all())
    big_a, big_res = torch.randn(100, K, device=DEV).bfloat16(), torch.randn(100, N, device=DEV)
    p2 = ops.gemm_add_then_norm(big_a, w, big_res, gain, eps, torch.bfloat16)
    assert p2.scaled is None
    assert torch.equal(ops.gemm(p2, w2), ops.gemm(ops.rmsnorm(big_res, gain, eps, torch.bfloat16), w2))


@pytest.mark.parametrize("rows", [1, 4, 7, 8, 9, 12, 16, 17, 20, 24, 31, 32])
@pytest.mark.parametrize("M,N,K", [(1, 96, 128), (8, 4112, 384), (9, 272, 1152), (16, 48, 2560), (5, 8192, 640), (9, 16448, 256), (3, 16400, 1920)])
def test_few_row_products_at_any_weight_rows_per_workgroup(ops, monkeypatch, M, N, K, rows):
    """The kernel for up to 16 rows with any number of weight rows per workgroup: last workgroups with fewer rows than the
    others, loads of eight rows that are not all there, fewer blocks of K than waves and than the ring holds, one and
    two loads of activations, one to three workgroups a compute unit. Against float64: an fp32 sum of K products, whatever its order, is within
    K 2^-24 of the sum of their sizes (and twice that for what is summed before the add), the bf16 rows for a norm exactly
    what the new residual gives. Without the gate the split of K knows nothing of the rows per workgroup: the same bits."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(M * N + K + rows)
    rnd = lambda *shape: torch.randn(*shape, device=DEV, generator=gen)
    a, w, w2 = rnd(M, K).bfloat16(), (rnd(N, K) / math.sqrt(K)).bfloat16(), (rnd(N, K) / math.sqrt(K)).bfloat16()
    bias, gain, res0 = rnd(N), rnd(N).abs() + 0.5, rnd(M, N)
    monkeypatch.setattr(ops, "_skinny_rows", lambda n, k, gated: min(rows, 16) if gated else rows)
    ops.reset_stats()
    exact, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    bound = 2 * K * 2.0 ** -24 * size + 1e-6
    out = ops.gemm(a, w, bias=bias, out_dtype=torch.float32)
    assert bool(((out.double() - exact - bias.double()).abs() <= bound + 2.0 ** -23 * (exact.abs() + bias.abs())).all())
    res = res0.clone()
    promise = ops.gemm_add_then_norm(a, w, res, gain, 1e-3, torch.bfloat16)
    assert bool(((res.double() - exact - res0.double()).abs() <= bound + 2.0 ** -23 * (exact.abs() + res0.abs())).all())
    assert torch.equal(promise.scaled, (res * gain).bfloat16())
    want = (res.double() ** 2).sum(-1)
    assert bool(((promise.partials.double().sum(-1) - want).abs() <= 32 * 2.0 ** -24 * want).all())
    gated = ops.gemm(a, w, w2=w2, epilogue=ops.EPI_GATED, out_dtype=torch.float32)
    up = a.double() @ w2.double().T
    both = bound * (1.1 * up.abs() + 1) + 2 * K * 2.0 ** -24 * (a.double().abs() @ w2.double().abs().T) * exact.abs() + 1e-5 * (exact * up).abs()
    assert bool(((gated.double() - torch.nn.functional.silu(exact) * up).abs() <= both).all())
    assert set(ops.stats()["ran"]) == {"jllm_gemm_skinny_bf16", "jllm_gemm_skinny_norm_bf16"}
    if (N + rows - 1) // rows > ops.compute_units():  # four waves; the sums of eight differ from theirs
        return
    monkeypatch.setattr(ops, "_skinny_rows", lambda n, k, gated: 32)
    assert torch.equal(out, ops.gemm(a, w, bias=bias, out_dtype=torch.float32))


@pytest.mark.parametrize("M,N,K,rows", [(1, 160, 2048, 32), (9, 4096, 4096, 16), (8, 4112, 2048, 8), (16, 8192, 4096, 20), (3, 48, 8320, 4), (13, 272, 11008, 16),
                                        (5, 6144, 2048, 24), (16, 96, 16384, 12)])
def test_few_row_products_that_begin_at_different_blocks(ops, monkeypatch, M, N, K, rows):
    """Rows a multiple of 4 KB apart, and long ones: workgroups that begin anywhere in K, with as many blocks as a power of two
    and more, for every number of loads per block, one and two workgroups a compute unit. Against float64 within the bound of an
    fp32 sum of K products; a row has the same bits alone as beside others, and adding as storing."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(M * N + K + rows)
    rnd = lambda *shape: torch.randn(*shape, device=DEV, generator=gen)
    a, w, res0 = rnd(M, K).bfloat16(), (rnd(N, K) / math.sqrt(K)).bfloat16(), rnd(M, N)
    monkeypatch.setattr(ops, "_skinny_rows", lambda *_: rows)
    ops.reset_stats()
    out = ops.gemm(a, w, out_dtype=torch.float32)
    bound = 2 * K * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T) + 1e-6
    assert bool(((out.double() - a.double() @ w.double().T).abs() <= bound).all())
    res = res0.clone()
    promise = ops.gemm_add_then_norm(a, w, res, torch.ones(N, device=DEV), 1e-5, torch.bfloat16)
    assert torch.equal(res, res0 + out) and torch.equal(promise.scaled, res.bfloat16())
    for r in {0, M // 2, M - 1}:
        assert torch.equal(ops.gemm(a[r:r + 1].contiguous(), w, out_dtype=torch.float32), out[r:r + 1])
    assert set(ops.stats()["ran"]) == {"jllm_gemm_skinny_bf16", "jllm_gemm_skinny_norm_bf16"}


@pytest.mark.parametrize("rows", [32, 64, 96, 128])
@pytest.mark.parametrize("M,N,K,parts", [(17, 160, 128, 1), (33, 1040, 640, 2), (64, 2064, 1152, 3), (1, 336, 2560, 6), (48, 4112, 256, 1),
                                         (25, 9728, 384, 1), (64, 192, 4096, 8)])
def test_products_of_17_to_64_rows_at_any_plan(ops, monkeypatch, M, N, K, rows, parts):
    """The kernel for 17 to 64 rows at every number of weight rows per workgroup: last column tiles with fewer columns than
    the others, ranges of K shorter than the ring and of unequal length, one to four tiles of rows, one workgroup a compute
    unit and two. Against float64 within the bound of an fp32 sum of K products in any order; a row's bits are the same alone as
    among the others, in the step's shared counters as in counters of its own; the rows for a norm are exactly what
    the new residual gives."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(M * N + K + rows)
    rnd = lambda *shape: torch.randn(*shape, device=DEV, generator=gen)
    a, w, w2 = rnd(M, K).bfloat16(), (rnd(N, K) / math.sqrt(K)).bfloat16(), (rnd(N, K) / math.sqrt(K)).bfloat16()
    bias, gain, res0 = rnd(N), rnd(N).abs() + 0.5, rnd(M, N)
    monkeypatch.setattr(ops, "SKINNY_MAX_ROWS", 0)  # up to 16 rows as well
    monkeypatch.setattr(ops, "_stream_plan", lambda *_: (rows, parts))
    ops.reset_stats()
    exact, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    bound = 2 * K * 2.0 ** -24 * size + 1e-6
    out = ops.gemm(a, w, bias=bias, out_dtype=torch.float32)
    assert bool(((out.double() - exact - bias.double()).abs() <= bound + 2.0 ** -23 * (exact.abs() + bias.abs())).all())
    res = res0.clone()
    with ops.step_scratch(M, a.device):
        for _ in range(2):  # the second launch finds the counters as the first one left them
            res = res0.clone()
            promise = ops.gemm_add_then_norm(a, w, res, gain, 1e-3, torch.bfloat16)
    assert bool(((res.double() - exact - res0.double()).abs() <= bound + 2.0 ** -23 * (exact.abs() + res0.abs())).all())
    assert torch.equal(promise.scaled, (res * gain).bfloat16())
    want = (res.double() ** 2).sum(-1)
    assert bool(((promise.partials.double().sum(-1) - want).abs() <= 128 * 2.0 ** -24 * want).all())
    gated = ops.gemm(a, w, w2=w2, epilogue=ops.EPI_GATED, out_dtype=torch.float32)
    up = a.double() @ w2.double().T
    both = bound * (1.1 * up.abs() + 1) + 2 * K * 2.0 ** -24 * (a.double().abs() @ w2.double().abs().T) * exact.abs() + 1e-5 * (exact * up).abs()
    assert bool(((gated.double() - torch.nn.functional.silu(exact) * up).abs() <= both).all())
    for r in {0, M // 2, M - 1}:
        assert torch.equal(ops.gemm(a[r:r + 1].contiguous(), w, bias=bias, out_dtype=torch.float32), out[r:r + 1])
        assert torch.equal(ops.gemm(a[r:r + 1].contiguous(), w, w2=w2, epilogue=ops.EPI_GATED, out_dtype=torch.float32), gated[r:r + 1])
    assert set(ops.stats()["ran"]) == {"jllm_gemm_stream_bf16"}


def test_counters_of_parts_belong_to_a_stream(ops, monkeypatch):
    """Products with K cut over workgroups inside one step's scope on two streams at once, and recorded into a graph on the other
    stream: only those in the stream of the first one share its counters, and every result has the same bits."""
    M, N, K = 40, 1024, 2048
    monkeypatch.setattr(ops, "_stream_plan", lambda *_: (32, 4))
    gen = torch.Generator(device=DEV)
    gen.manual_seed(3)
    a, w = torch.randn(M, K, device=DEV, generator=gen).bfloat16(), (torch.randn(N, K, device=DEV, generator=gen) / math.sqrt(K)).bfloat16()
    want = ops.gemm(a, w, out_dtype=torch.float32)
    torch.cuda.synchronize()
    side, graph, got = torch.cuda.Stream(), torch.cuda.CUDAGraph(), []
    with ops.step_scratch(M, a.device):
        for _ in range(4):
            got.append(ops.gemm(a, w, out_dtype=torch.float32))
            with torch.cuda.stream(side):
                got.append(ops.gemm(a, w, out_dtype=torch.float32))
        assert ops._step_scratch.shared[1] == torch.cuda.current_stream().cuda_stream
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            recorded = ops.gemm(a, w, out_dtype=torch.float32)
        with torch.cuda.stream(side):  # in front of the first replay, which clears what the capture counts in
            got.append(ops.gemm(a, w, out_dtype=torch.float32))
        torch.cuda.synchronize()
    for _ in range(3):
        graph.replay()
        got.append(recorded.clone())
        got.append(ops.gemm(a, w, out_dtype=torch.float32))
        torch.cuda.synchronize()
    assert all(torch.equal(g, want) for g in got)


@pytest.mark.parametrize("rows,tile", [(32, 64), (64, 64), (96, 64), (128, 64), (32, 128), (64, 128), (96, 128), (128, 128)])
@pytest.mark.parametrize("M,N,K,parts", [(128, 1024, 1024, 1), (129, 1040, 1152, 2), (200, 2048, 1024, 3), (321, 528, 3072, 4), (640, 4096, 1024, 1)])
def test_products_of_more_rows_at_any_plan(ops, monkeypatch, M, N, K, parts, rows, tile):
    """The same kernel for more than 64 rows in tiles of 64 and 128, the last one with a single row or more, rows with a
    stride: every epilogue and the norm on both sides, against float64 within the bound of an fp32 sum of K products."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(M * N + K + rows + tile)
    rnd = lambda *shape: torch.randn(*shape, device=DEV, generator=gen)
    a = ops.activation_rows(M, K, torch.bfloat16, torch.device(DEV))
    a.copy_(rnd(M, K))
    w, w2 = (rnd(N, K) / math.sqrt(K)).bfloat16(), (rnd(N, K) / math.sqrt(K)).bfloat16()
    w3 = (rnd(272, N) / math.sqrt(N)).bfloat16()
    bias, gain, res0 = rnd(N), rnd(N).abs() + 0.5, rnd(M, N)
    monkeypatch.setattr(ops, "_wide_plan", lambda m, n, k, gated, adds=False: (rows, tile, parts if k == K else 1))
    ops.reset_stats()
    exact, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    bound = 2 * K * 2.0 ** -24 * size + 1e-6
    out = ops.gemm(a, w, bias=bias, out_dtype=torch.float32)
    assert bool(((out.double() - exact - bias.double()).abs() <= bound + 2.0 ** -23 * (exact.abs() + bias.abs())).all())
    assert torch.equal(ops.gemm(a, w, bias=bias), out.bfloat16())
    res = res0.clone()
    with ops.step_scratch(M, a.device):
        promise = ops.gemm_add_then_norm(a, w, res, gain, 1e-3, torch.bfloat16)
        assert bool(((res.double() - exact - res0.double()).abs() <= bound + 2.0 ** -23 * (exact.abs() + res0.abs())).all())
        assert torch.equal(promise.scaled, (res * gain).bfloat16())
        if N % 128 == 0:  # what the consuming product takes as its K
            scale = torch.rsqrt((res.double() ** 2).mean(-1, keepdim=True) + 1e-3)
            got = ops.gemm(promise, w3, out_dtype=torch.float32)
            want = (promise.scaled.double() @ w3.double().T) * scale
            assert bool(((got.double() - want).abs() <= (2 * N + 256) * 2.0 ** -24 * (promise.scaled.double().abs() @ w3.double().abs().T) * scale + 1e-6).all())
        gated = ops.gemm(a, w, w2=w2, epilogue=ops.EPI_GATED, out_dtype=torch.float32)
    up = a.double() @ w2.double().T
    both = bound * (1.1 * up.abs() + 1) + 2 * K * 2.0 ** -24 * (a.double().abs() @ w2.double().abs().T) * exact.abs() + 1e-5 * (exact * up).abs()
    assert bool(((gated.double() - torch.nn.functional.silu(exact) * up).abs() <= both).all())
    assert set(ops.stats()["ran"]) == {"jllm_gemm_stream_bf16"} and promise._rows is None


@pytest.mark.parametrize("M,N,K,tile,cut", [(65, 1024, 2048, 0, 4), (631, 4096, 4096, 256, 2), (300, 2560, 4096, 192, 2), (130, 8192, 1024, 0, 2),
                                            (700, 96, 2048, 0, 8), (70, 1040, 1024, 0, 1), (600, 2560, 2176, 256, 3), (390, 1040, 2176, 192, 5),
                                            (560, 1296, 2176, 384, 3), (890, 1024, 2176, 384, 5)])  # 384: wide tiles for the last rows
@pytest.mark.parametrize("gdt", [torch.bfloat16, torch.float32])
def test_the_reduction_makes_the_norm(ops, monkeypatch, M, N, K, tile, cut, gdt):
    """An adding product of many rows with K cut, in odd and even numbers of parts, equal and not: the residual and the rows for the
    next product have the bits of the reduction and the norm as launches of their own, with and without a bias, in rows with a
    stride; with K whole the norm stays a launch."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(M + N + K)
    rnd = lambda *shape: torch.randn(*shape, device=DEV, generator=gen)
    a, w, res0, gain = rnd(M, K).bfloat16(), (rnd(N, K) / math.sqrt(K)).bfloat16(), rnd(M, N), (rnd(N).abs() + 0.5).to(gdt)
    monkeypatch.setattr(ops, "_wide_plan", lambda *_: None)
    monkeypatch.setattr(ops, "_tiled_plan", lambda *_: (tile, cut))
    monkeypatch.setattr(ops, "_k_splits", lambda *_: cut)
    for bias in (None, rnd(N), rnd(N).bfloat16()):
        want, got = res0.clone(), res0.clone()
        ops.gemm(a, w, bias=bias, out=want, epilogue=ops.EPI_ADD)
        promise = ops.gemm_add_then_norm(a, w, got, gain, 1e-5, torch.bfloat16, bias=bias)
        assert torch.equal(got, want) and promise.scaled is None and (promise._rows is not None) == (cut > 1)
        assert torch.equal(promise.tensor().view(torch.int16), ops.rmsnorm(want, gain, 1e-5, torch.bfloat16).view(torch.int16))


def test_gemm_rows_do_not_depend_on_the_batch(ops):
    """The result of a row is the same bits whether it is alone or among others, within one kernel family (the
    bfloat16 path has one kernel for up to 16 rows, one for up to 64 and one for more; between them results differ
    by rounding)."""
    torch.manual_seed(0)
    for dtype, K, full_rows, parts in ((torch.float32, 200, 64, (1, 2, 7, 16, 33)), (torch.float32, 203, 40, (1, 3, 16, 17)),
                                       (torch.bfloat16, 512, 16, (1, 7, 11)),
                                       (torch.bfloat16, 1024, 64, (17, 33, 48)), (torch.bfloat16, 512, 128, (65, 100)),
                                       (torch.bfloat16, 8192, 16, (1, 8)), (torch.bfloat16, 8192, 64, (17, 40)),  # with N = 1024
                                       (torch.bfloat16, 3072, 16, (1, 8, 11)),  # with N = 5120: 20 weight rows per workgroup
                                       (torch.bfloat16, 384, 16, (1, 5, 9))):  # with N = 6144: 24 weight rows per workgroup
        N = {8192: 1024, 3072: 5120, 384: 6144}.get(K, 96)
        a = torch.randn(full_rows, K, device=DEV).to(dtype)
        w = torch.randn(N, K, device=DEV).to(dtype)
        full = ops.gemm(a, w, out_dtype=torch.float32, exact=dtype == torch.float32)
        for rows in parts:
            part = ops.gemm(a[:rows].contiguous(), w, out_dtype=torch.float32, exact=dtype == torch.float32)
            assert torch.equal(part, full[:rows])
    # the 32-bit path has a kernel of its own for up to 16 rows: every epilogue and operand type gives the same bits
    a = torch.randn(40, 136, device=DEV)
    w, w2, bias = torch.randn(100, 136, device=DEV), torch.randn(100, 136, device=DEV), torch.randn(100, device=DEV)
    for wt in (torch.float32, torch.bfloat16):
        full = ops.gemm(a, w.to(wt), w2=w2.to(wt), epilogue=ops.EPI_GATED, out_dtype=torch.float32, exact=True)
        few = ops.gemm(a[:9].contiguous(), w.to(wt), w2=w2.to(wt), epilogue=ops.EPI_GATED, out_dtype=torch.float32, exact=True)
        assert torch.equal(few, full[:9])
        res_full, res_few = torch.ones(40, 100, device=DEV), torch.ones(9, 100, device=DEV)
        ops.gemm(a, w.to(wt), bias=bias, out=res_full, epilogue=ops.EPI_ADD, exact=True)
        ops.gemm(a[:9].contiguous(), w.to(wt), bias=bias, out=res_few, epilogue=ops.EPI_ADD, exact=True)
        assert torch.equal(res_few, res_full[:9])
    # and between the bfloat16 kernels: rounding only
    a = torch.randn(100, 1024, device=DEV).bfloat16()
    w = (torch.randn(256, 1024, device=DEV) / 32).bfloat16()
    few = ops.gemm(a[:16].contiguous(), w, out_dtype=torch.float32)
    some = ops.gemm(a[:40].contiguous(), w, out_dtype=torch.float32)[:16]
    many = ops.gemm(a, w, out_dtype=torch.float32)[:16]
    assert torch.allclose(few, many, rtol=1e-4, atol=1e-4) and torch.allclose(few, some, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (3, 100, 203), (16, 49, 772), (17, 33, 100), (65, 130, 192), (33, 1030, 36),
                                   (700, 1100, 68), (2041, 4090, 40)])
@pytest.mark.parametrize("wdt", [torch.float32, torch.bfloat16])
def test_float32_products_are_one_chain_of_multiply_adds(ops, M, N, K, wdt):
    """Every tile of the 32-bit products, at its edges: an output has the bits of one fp32 accumulator that takes its
    terms in ascending k. Operands of 12 (8) bits: a product and an accumulator then add without rounding in
    float64 (2^-44 .. 2^6), so the chain is restated there with one rounding to fp32 per step, exactly. (Products of so few
    bits are exact in fp32: that they are not rounded by themselves is the next test's.) The gated form
    gives, in any batch, the bits it gives its rows in batches of 16."""
    assert [ops.library().jllm_f32_tile(m, n, 0) for m, n in ((33, 1030), (700, 1100), (2041, 4090))] == [2, 1, 0]
    gen = torch.Generator(device=DEV)
    gen.manual_seed(M + N + K)

    def short(*shape):
        return ((torch.randn(*shape, device=DEV, generator=gen) * 512).round() / 512).to(wdt).float()

    a, w, w2 = short(M, K), short(N, K), short(N, K)
    want = torch.zeros(M, N, device=DEV)
    for k in range(K):
        want = (want.double() + a[:, k:k + 1].double() * w[:, k].double()).float()
    assert torch.equal(ops.gemm(a, w.to(wdt), exact=True), want)
    gated = ops.gemm(a, w.to(wdt), w2=w2.to(wdt), epilogue=ops.EPI_GATED, exact=True)
    for at in range(0, M, max(16, M // 4)):
        few = ops.gemm(a[at:at + 16].contiguous(), w.to(wdt), w2=w2.to(wdt), epilogue=ops.EPI_GATED, exact=True)
        assert torch.equal(few, gated[at:at + 16])


@pytest.mark.parametrize("N,K", [(1, 128), (16, 256), (17, 384), (40, 512), (300, 640), (4100, 1152)])
def test_float32_products_of_few_rows(ops, N, K):
    """Up to four rows, K in turns of 128 (one, fewer than the ring holds, exactly those, more, not a multiple of them), weight
    rows that end inside a workgroup, every epilogue: the bits of the same rows among six, which the other kernel takes, also with
    an infinity in one row; a stride between the rows."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(N + K)
    a = torch.randn(6, K + 4, device=DEV, generator=gen)[:, :K]
    w, w2 = (torch.randn(N, K, device=DEV, generator=gen) * K ** -0.5 for _ in range(2))
    a[1, K // 2] = float("inf")
    bias = torch.randn(N, device=DEV, generator=gen)
    res = torch.randn(6, N, device=DEV, generator=gen)
    add = ops.gemm(a, w, bias=bias, out=res.clone(), epilogue=ops.EPI_ADD, exact=True)
    many = [ops.gemm(a, w, bias=bias, exact=True), ops.gemm(a, w, w2=w2, epilogue=ops.EPI_GATED, exact=True), ops.gemm(a, w, out_dtype=torch.bfloat16, exact=True)]
    for first, rows in ((0, 1), (1, 2), (0, 3), (2, 4)):
        x, r = a[first:first + rows], res[first:first + rows].clone()
        few = [ops.gemm(x, w, bias=bias, exact=True), ops.gemm(x, w, w2=w2, epilogue=ops.EPI_GATED, exact=True), ops.gemm(x, w, out_dtype=torch.bfloat16, exact=True)]
        ops.gemm(x, w, bias=bias, out=r, epilogue=ops.EPI_ADD, exact=True)
        for got, want in zip(few + [r], many + [add]):
            assert torch.equal(torch.nan_to_num(got, nan=7.0), torch.nan_to_num(want[first:first + rows], nan=7.0)), (rows, first)
    tiny, small = a.nan_to_num(posinf=1.0) * 2.0 ** -68, w * 2.0 ** -68  # denormal products and sums
    assert torch.equal(ops.gemm(tiny[:3], small, exact=True), ops.gemm(tiny, small, exact=True)[:3])


@pytest.mark.parametrize("M,N,tile", [(17, 33, 2), (33, 1030, 2), (700, 1100, 1), (769, 1030, 1), (2041, 4090, 0), (1921, 4092, 0)])
@pytest.mark.parametrize("K", [32, 64, 96, 128, 352])
def test_float32_products_of_whole_lines(ops, M, N, tile, K):
    """Many rows, K in stages of 32 (one, fewer than a ring holds, exactly those, more), edges of tiles, every epilogue: the bits of
    the same rows in batches of 16, which another kernel takes, also with an infinity in one row; a stride between the rows."""
    assert [ops.library().jllm_f32_tile(M, N, gated) for gated in (0, 1)] == [tile, tile]
    gen = torch.Generator(device=DEV)
    gen.manual_seed(M + K)
    a = torch.randn(M, K + 4, device=DEV, generator=gen)[:, :K]
    w, w2 = (torch.randn(N, K, device=DEV, generator=gen) * K ** -0.5 for _ in range(2))
    a[1, K // 2] = float("inf")
    bias = torch.randn(N, device=DEV, generator=gen)
    res = torch.randn(M, N, device=DEV, generator=gen)

    def forms(x, r):
        r = r.clone()
        ops.gemm(x, w, bias=bias, out=r, epilogue=ops.EPI_ADD, exact=True)
        return [r, ops.gemm(x, w, bias=bias, exact=True), ops.gemm(x, w, out_dtype=torch.bfloat16, exact=True),
                ops.gemm(x, w, w2=w2, epilogue=ops.EPI_GATED, exact=True)]

    many = forms(a, res)
    for at in {0, min(16, M - 16), M // 2 if M > 100 else 0, M - 16}:
        for got, want in zip(many, forms(a[at:at + 16], res[at:at + 16])):
            assert torch.equal(torch.nan_to_num(got[at:at + 16], nan=7.0), torch.nan_to_num(want, nan=7.0)), at


@pytest.mark.parametrize("M,N,K,exponent", [(3, 17, 67, 0), (16, 20, 200, -70), (20, 33, 70, 0), (40, 35, 68, -71), (130, 40, 36, -70)])
def test_float32_products_round_once_per_multiply_add(ops, M, N, K, exponent):
    """The 32-bit products on operands of 24 bits, whose products a multiply-add must not round, against the C library's
    fmaf in ascending k, bit for bit; with magnitudes around 2^-70 products and sums are denormal."""
    import ctypes
    libm = ctypes.CDLL("libm.so.6")
    libm.fmaf.restype, libm.fmaf.argtypes = ctypes.c_float, [ctypes.c_float] * 3
    g = torch.Generator().manual_seed(M + N)
    a, w = (torch.randn(n, K, generator=g) * 2.0 ** exponent for n in (M, N))
    want = torch.zeros(M, N)
    for m, row in enumerate(a.tolist()):
        for n, col in enumerate(w.tolist()):
            x = 0.0
            for p, q in zip(row, col):
                x = libm.fmaf(p, q, x)
            want[m, n] = x
    if exponent:
        assert bool(((want != 0) & (want.abs() < 2.0 ** -126)).any())
    assert torch.equal(ops.gemm(a.to(DEV), w.to(DEV), exact=True).cpu(), want)


def test_gemm_refuses_bad_arguments(ops):
    a = torch.randn(4, 32, device=DEV)
    w = torch.randn(8, 31, device=DEV)
    with pytest.raises(ops.KernelError):
        ops.gemm(a, w)
    with pytest.raises(ops.KernelError):
        ops.gemm(a.cpu(), torch.randn(8, 32))
    with pytest.raises(ops.KernelError):
        ops.gemm(a, torch.randn(8, 32, device=DEV), epilogue=ops.EPI_ADD)
    with pytest.raises(ops.KernelError):
        ops.gemm(a.double(), torch.randn(8, 32, device=DEV).double())


# ------------------------------------------------------------------------------- q/k norm, rotation, cache store


ROPE_CASES = [  # H, Hkv, hd, rotary width (0: none), page, gains (None: no norm)
    (4, 2, 16, 16, 8, torch.bfloat16), (6, 2, 32, 32, 16, torch.float32), (5, 5, 48, 48, 32, torch.bfloat16),
    (3, 3, 24, 12, 4, torch.bfloat16), (8, 1, 64, 32, 4, None), (3, 3, 80, 64, 16, torch.float32),
    (32, 8, 128, 128, 16, torch.bfloat16), (2, 1, 256, 256, 16, torch.bfloat16), (7, 7, 96, 0, 2, torch.bfloat16),
    (2, 2, 20, 10, 8, torch.float32),
]


@pytest.mark.parametrize("H,Hkv,hd,rot,page,gdt", ROPE_CASES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_qk_norm_rope_store(ops, H, Hkv, hd, rot, page, gdt, dtype):
    """Per-head RMSNorm of q and k, rotation of pairs (i, i + rot/2) by the angles of each row's position, k and v
    into their pages, against float64. The angles differ for every position and pair, q and k have different gains,
    some rows store nothing (slot -1): a wrong pairing, sign, gain or row shows."""
    gen = torch.Generator().manual_seed(H * 131 + hd)
    T, n_pages, max_pos, eps = 37, 20, 50, 1e-4
    qkv = (torch.randn(T, (H + 2 * Hkv) * hd, generator=gen) * 1.5).to(dtype)
    positions = torch.randint(0, max_pos, (T,), generator=gen, dtype=torch.int32)
    slots = torch.randperm(n_pages * page, generator=gen)[:T].to(torch.int32)
    slots[5] = -1
    slots[T - 1] = -1
    gq = gk = None
    if gdt is not None:
        gq = (torch.rand(hd, generator=gen) + 0.5).to(gdt if dtype == torch.bfloat16 else torch.float32)
        gk = (torch.rand(hd, generator=gen) + 0.5).to(gdt if dtype == torch.bfloat16 else torch.float32)
    cos = sin = None
    if rot:
        ang = torch.rand(max_pos, rot // 2, generator=gen, dtype=torch.float64) * 6.28
        cos, sin = torch.cos(ang).float(), torch.sin(ang).float()

    def prepared(x, gain):  # [T, heads, hd] float64
        x = x.double()
        if gain is not None:
            x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * gain.double()
        if rot:
            c, s_ = cos[positions.long()].double()[:, None, :], sin[positions.long()].double()[:, None, :]
            a, b = x[..., :rot // 2].clone(), x[..., rot // 2:rot].clone()
            x[..., :rot // 2] = a * c - b * s_
            x[..., rot // 2:rot] = b * c + a * s_
        return x

    want_q = prepared(qkv[:, :H * hd].view(T, H, hd), gq)
    want_k = prepared(qkv[:, H * hd:(H + Hkv) * hd].view(T, Hkv, hd), gk)
    want_v = qkv[:, (H + Hkv) * hd:].view(T, Hkv, hd)
    dev = lambda x: None if x is None else x.to(DEV)
    for write_kv in (True, False):
        work = qkv.clone().to(DEV)
        kc = torch.full((n_pages, Hkv, page, hd), 7.0).to(dtype).to(DEV)
        vc = torch.full((n_pages, Hkv, page, hd), 7.0).to(dtype).to(DEV)
        ops.qk_norm_rope_store(work, dev(positions), dev(slots), dev(cos), dev(sin), dev(gq), dev(gk), eps, H, Hkv, hd, rot,
                               page, kc, vc, write_kv=write_kv)
        got_q = work[:, :H * hd].view(T, H, hd).cpu()
        if dtype == torch.float32:
            assert torch.allclose(got_q.double(), want_q, rtol=1e-5, atol=1e-5)
        else:
            assert bf16_close(got_q, want_q)[0]
        assert torch.equal(work[:, H * hd:].cpu(), qkv[:, H * hd:]), "k and v of the projection output stay as they are"
        stored = torch.zeros(n_pages, page, dtype=torch.bool)
        for t in range(T):
            sl = int(slots[t])
            if sl < 0 or not write_kv:
                continue
            pg, off = sl // page, sl % page
            stored[pg, off] = True
            gk_, gv_ = kc[pg, :, off].cpu(), vc[pg, :, off].cpu()
            if dtype == torch.float32:
                assert torch.allclose(gk_.double(), want_k[t], rtol=1e-5, atol=1e-5)
            else:
                assert bf16_close(gk_, want_k[t])[0]
            assert torch.equal(gv_, want_v[t])
        untouched = ~stored[:, None, :, None].expand(n_pages, Hkv, page, hd)
        assert bool((kc.cpu()[untouched] == 7.0).all()) and bool((vc.cpu()[untouched] == 7.0).all())


@pytest.mark.parametrize("H,Hkv,hd,rot", [(4, 2, 16, 16), (6, 2, 32, 32), (5, 5, 48, 24), (8, 2, 128, 128), (3, 1, 80, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rotation_comes_after_the_head_norm(ops, H, Hkv, hd, rot, dtype):
    """Scores depend only on the distance between query and key when the rotation is what happens last to q and k:
    with gains that differ within every rotated pair, the products q_i . k_j of the kernel's outputs are the same at
    positions p.. and p + 10.. . A kernel that rotated first and normalised afterwards would fail this by a wide
    margin (shown below on the same numbers in float64), whatever reference it was compared with."""
    gen = torch.Generator().manual_seed(hd + rot)
    T, page, eps, theta = 12, 4, 1e-6, 100.0
    G = H // Hkv
    qkv = (torch.randn(T, (H + 2 * Hkv) * hd, generator=gen) * 1.5).to(dtype)
    gdt = torch.float32 if dtype == torch.float32 else torch.bfloat16
    gq = (torch.rand(hd, generator=gen) * 2.5 + 0.25).to(gdt)
    gk = (torch.rand(hd, generator=gen) * 2.5 + 0.25).to(gdt)
    inv = 1.0 / theta ** (torch.arange(rot // 2, dtype=torch.float64) * 2 / rot)
    ang = torch.arange(64, dtype=torch.float64)[:, None] * inv[None, :]
    cos, sin = torch.cos(ang).float(), torch.sin(ang).float()
    slots = torch.arange(T, dtype=torch.int32)

    def scores(shift):
        work = qkv.clone().to(DEV)
        kc = torch.zeros(T // page, Hkv, page, hd, dtype=dtype, device=DEV)
        vc = torch.zeros_like(kc)
        pos = (torch.arange(T, dtype=torch.int32) + shift).to(DEV)
        ops.qk_norm_rope_store(work, pos, slots.to(DEV), cos.to(DEV), sin.to(DEV), gq.to(DEV), gk.to(DEV), eps, H, Hkv, hd,
                               rot, page, kc, vc)
        q = work[:, :H * hd].view(T, H, hd).cpu().double()
        k = kc.permute(0, 2, 1, 3).reshape(T, Hkv, hd).cpu().double()  # [page, kv head, row, :] -> [position, kv head, :]
        return torch.einsum("ihd,jhd->ijh", q, k.repeat_interleave(G, 1))

    a, b = scores(3), scores(13)
    span = float(a.abs().max())
    assert (a - b).abs().max() <= (2e-5 if dtype == torch.float32 else 3e-2) * span

    def wrong(shift):  # rotate, then normalise
        def prep(x, g):
            x = x.double().clone()
            c, s_ = cos[shift:shift + T].double()[:, None, :], sin[shift:shift + T].double()[:, None, :]
            u, v = x[..., :rot // 2].clone(), x[..., rot // 2:rot].clone()
            x[..., :rot // 2], x[..., rot // 2:rot] = u * c - v * s_, v * c + u * s_
            return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * g.double()
        q = prep(qkv[:, :H * hd].view(T, H, hd), gq)
        k = prep(qkv[:, H * hd:(H + Hkv) * hd].view(T, Hkv, hd), gk)
        return torch.einsum("ihd,jhd->ijh", q, k.repeat_interleave(G, 1))
    assert (wrong(3) - wrong(13)).abs().max() > 0.1 * span, "the case must tell the two orders apart"


def test_fused_decode_rotates_after_the_head_norm(ops):
    """The same invariant for the decode kernel that prepares q and k itself: a row at position p over keys
    p - 15 .. p (a window hides what lies before) gives the same output when the request sits ten positions
    further on, with the keys stored by the kernel for whole portions at their shifted positions."""
    H, Hkv, hd, page, eps, theta, W = 8, 2, 128, 16, 1e-6, 50.0, 16
    gen = torch.Generator().manual_seed(5)
    gq = (torch.rand(hd, generator=gen) * 2.5 + 0.25).bfloat16().to(DEV)
    gk = (torch.rand(hd, generator=gen) * 2.5 + 0.25).bfloat16().to(DEV)
    inv = 1.0 / theta ** (torch.arange(hd // 2, dtype=torch.float64) * 2 / hd)
    ang = torch.arange(64, dtype=torch.float64)[:, None] * inv[None, :]
    cos, sin = torch.cos(ang).float().to(DEV), torch.sin(ang).float().to(DEV)
    rows = (torch.randn(W, (H + 2 * Hkv) * hd, generator=gen) * 1.5).bfloat16()
    scale = 1.0 / math.sqrt(hd)
    outs = []
    for shift in (0, 10):
        n_pages = 3
        kc = torch.full((n_pages, Hkv, page, hd), float("nan")).bfloat16().to(DEV)  # what the window hides is NaN
        vc = kc.clone()
        table = torch.arange(n_pages, dtype=torch.int32, device=DEV).view(1, n_pages)
        pos = (torch.arange(W, dtype=torch.int32) + shift).to(DEV)
        work = rows.clone().to(DEV)
        ops.qk_norm_rope_store(work[:W - 1], pos[:W - 1], pos[:W - 1], cos, sin, gq, gk, eps, H, Hkv, hd, hd, page, kc, vc)
        meta = {"max_context": W + shift, "decode_only": True, "requests": 1}
        out = ops.decode_attention_fused(rows[W - 1:].to(DEV), kc, vc, table, torch.zeros(1, dtype=torch.int32, device=DEV),
                                         pos[W - 1:], pos[W - 1:], cos, sin, gq, gk, eps, H, Hkv, hd, hd, W, scale, meta)
        assert out is not None and not torch.isnan(out.float()).any()
        outs.append(out.float().cpu())
    assert (outs[0] - outs[1]).abs().max() <= 2e-2 * max(1.0, float(outs[0].abs().max()))
    assert outs[0].abs().max() > 0.1


# ------------------------------------------------------------------------------------------------ attention


def make_cache(R, ctx_lens, Hkv, hd, page, dtype, extra_pages=3, seed=0):
    """Random k/v for R requests in shuffled pages of a pool that also holds garbage pages."""
    g = torch.Generator().manual_seed(seed)
    blocks = [-(-c // page) for c in ctx_lens]
    n_pages = sum(blocks) + extra_pages
    perm = torch.randperm(n_pages, generator=g).tolist()
    kc = torch.full((n_pages, Hkv, page, hd), float("nan")).to(dtype)  # unused slots hold NaN: nothing may read them
    vc = torch.full((n_pages, Hkv, page, hd), float("nan")).to(dtype)
    width = max(blocks)
    table = torch.full((R, width), -1, dtype=torch.int32)
    ks, vs = [], []
    it = iter(perm)
    for r, c in enumerate(ctx_lens):
        k = torch.randn(c, Hkv, hd, generator=g).to(dtype)
        v = torch.randn(c, Hkv, hd, generator=g).to(dtype)
        ks.append(k); vs.append(v)
        for b in range(blocks[r]):
            pg = next(it)
            table[r, b] = pg
            n = min(page, c - b * page)
            kc[pg, :, :n] = k[b * page:b * page + n].transpose(0, 1)
            vc[pg, :, :n] = v[b * page:b * page + n].transpose(0, 1)
    return kc.to(DEV), vc.to(DEV), table.to(DEV), ks, vs


def attention_reference(qrow, k, v, pos, H, window, scale):
    """One row in float64: keys [max(0, pos+1-window), pos]."""
    Hkv = k.shape[1]
    first = max(0, pos + 1 - window) if window > 0 else 0
    out = []
    for h in range(H):
        kk, vv = k[first:pos + 1, h // (H // Hkv)].double(), v[first:pos + 1, h // (H // Hkv)].double()
        p = torch.softmax((kk @ qrow[h].double()) * scale, 0)
        out.append(p @ vv)
    return torch.stack(out)


ATT_CASES = [  # H, Hkv, hd, page, window
    (4, 2, 16, 8, 0), (6, 2, 32, 16, 0), (5, 5, 48, 32, 20), (8, 1, 64, 4, 0), (3, 3, 80, 16, 300), (32, 8, 128, 16, 0),
    (16, 2, 128, 16, 100), (2, 1, 256, 16, 0), (9, 1, 64, 16, 0), (7, 7, 96, 1, 0), (4, 2, 192, 16, 0), (2, 2, 112, 8, 50),
    # head size 128 (the matrix-core decode kernel) with every group size it is instantiated for; 40 over 8 is the 14B shape
    (3, 3, 128, 16, 0), (6, 2, 128, 16, 0), (40, 8, 128, 16, 0), (6, 1, 128, 8, 300), (7, 1, 128, 16, 0), (4, 2, 128, 4, 0),
]


@pytest.mark.parametrize("H,Hkv,page,window", [(16, 8, 16, 0), (4, 4, 4, 70), (8, 2, 16, 100), (10, 2, 32, 0), (24, 3, 16, 300), (17, 1, 16, 0)])
def test_float32_attention_gives_the_general_kernels_bits(ops, H, Hkv, page, window):
    """Head size 128 in fp32: single rows and tiles of rows (requests that end inside a tile, one-row requests between
    portions, heads that fill 16 columns or leave some empty, more than 8 heads to a kv head) against the general kernel,
    bit for bit. One value is infinite: the rows in front of it must not feel it."""
    lens = [1, 200, 37, 64, 5, 333, 1]
    kc, vc, table, _, _ = make_cache(len(lens), lens, Hkv, 128, page, torch.float32, seed=H)
    vc[int(table[5, 100 // page]), 0, 100 % page, 77] = float("inf")
    g = torch.Generator().manual_seed(2)
    news = [1, 130, 37, 3, 1, 333, 1]  # the last rows of every request
    row_req = torch.tensor([r for r, n in enumerate(news) for _ in range(n)], dtype=torch.int32, device=DEV)
    positions = torch.tensor([p for c, n in zip(lens, news) for p in range(c - n, c)], dtype=torch.int32, device=DEV)
    q = (torch.randn(len(positions), H * 128, generator=g) * 1.5).to(DEV)
    zeros = torch.zeros(H, device=DEV)  # a bias of nothing: only the general kernel takes one

    def attend(rows, slopes=None):
        return ops.paged_attention(q[rows].contiguous(), kc, vc, table, row_req[rows].contiguous(), positions[rows].contiguous(), H,
                                   Hkv, 128, window, 128 ** -0.5, exact=True, slopes=slopes)

    every = torch.arange(len(positions), device=DEV)
    want = attend(every, zeros)
    forms = [(every, attend(every))] + [(every[a:a + n], attend(every[a:a + n])) for a, n in ((0, 7), (60, 20), (200, 27), (len(every) - 1, 1))]
    for rows, got in forms:
        ref = want[rows]
        fine = torch.isfinite(ref)  # (a row that does see the infinite value: infinite or NaN)
        assert torch.equal(torch.isfinite(got), fine) and torch.equal(got[fine], ref[fine])
    seen = (row_req == 5) & (positions >= 100) & ((positions < 100 + window) if window else True)
    assert bool(torch.isfinite(want[~seen]).all()) and not bool(torch.isfinite(want[seen]).all())


@pytest.mark.parametrize("H,Hkv,n_req,n,shuffled", [(16, 8, 64, 64, False),  # two heads to a workgroup of a row
                                                    (12, 4, 70, 70, False),  # the same with three heads of a kv head
                                                    (16, 8, 6, 25, False),   # a portion of few rows, row by row
                                                    (16, 8, 6, 41, False),   # single rows behind a portion, inside its last tile
                                                    (8, 8, 5, 300, True), (24, 3, 40, 1300, True)])  # requests in no order
def test_float32_attention_of_rows_in_any_order_gives_the_general_kernels_bits(ops, H, Hkv, n_req, n, shuffled):
    """Head size 128 in fp32 where a tile's rows belong to several requests, whose rows may lie anywhere in the step, and
    single rows of many requests, against the general kernel, bit for bit."""
    g = torch.Generator().manual_seed(n)
    lens = [int(x) for x in torch.randint(1, 200, (n_req,), generator=g)]
    kc, vc, table, _, _ = make_cache(n_req, lens, Hkv, 128, 16, torch.float32, seed=n)
    if shuffled:
        req = torch.randint(0, n_req, (n,), generator=g)
    else:
        req = torch.cat([torch.zeros(n - n_req, dtype=torch.int64), torch.arange(n_req)])
    pos = (torch.rand(n, generator=g) * torch.tensor(lens)[req]).long()
    q = torch.randn(n, H * 128, generator=g).to(DEV)

    def attend(slopes=None):
        return ops.paged_attention(q, kc, vc, table, req.int().to(DEV), pos.int().to(DEV), H, Hkv, 128, 0, 128 ** -0.5, exact=True, slopes=slopes)

    assert torch.equal(attend(), attend(torch.zeros(H, device=DEV)))


@pytest.mark.parametrize("H,Hkv,page,window", [(16, 8, 16, 0), (3, 3, 1, 0), (8, 1, 64, 300), (32, 8, 16, 65)])
def test_float32_rows_with_their_keys_by_way_of_lds(ops, H, Hkv, page, window):
    """float32 rows at head size 128 with more than 256 keys in the table and no more workgroups than compute units take their
    keys by way of LDS: bit for bit the general kernel (here by slopes of zero), at the edges of a wave's blocks and of a window."""
    lens = [1, 63, 64, 65, 257, 321, 1000]
    kc, vc, table, _, _ = make_cache(len(lens), lens, Hkv, 128, page, torch.float32, seed=H + page)
    q = torch.randn(len(lens), H * 128, generator=torch.Generator().manual_seed(H)).to(DEV)
    req = torch.arange(len(lens), dtype=torch.int32, device=DEV)
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=DEV)
    attend = lambda slopes: ops.paged_attention(q, kc, vc, table, req, pos, H, Hkv, 128, window, 128 ** -0.5, exact=True, slopes=slopes)
    got = attend(None)
    assert not torch.isnan(got).any() and torch.equal(got, attend(torch.zeros(H, device=DEV)))


@pytest.mark.parametrize("window", [0, 1, 65, 66, 128, 129, 257])
def test_float32_rows_of_a_wide_table_choose_by_their_own_keys(ops, window):
    """Rows of one to five blocks of keys in a table of many, as a captured step has them: up to two blocks the keys go into registers,
    beyond by way of LDS; on either side of that line, without a window and with ones that reach over two and three blocks."""
    lens = [1, 2, 64, 65, 127, 128, 129, 192, 193, 257, 1500]
    kc, vc, table, _, _ = make_cache(len(lens), lens, 2, 128, 16, torch.float32, seed=window)
    q = torch.randn(len(lens), 4 * 128, generator=torch.Generator().manual_seed(window)).to(DEV)
    req = torch.arange(len(lens), dtype=torch.int32, device=DEV)
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=DEV)
    attend = lambda slopes: ops.paged_attention(q, kc, vc, table, req, pos, 4, 2, 128, window, 128 ** -0.5, exact=True, slopes=slopes)
    got = attend(None)
    assert not torch.isnan(got).any() and torch.equal(got, attend(torch.zeros(4, device=DEV)))


@pytest.mark.parametrize("H,Hkv,hd,window", [(12, 3, 32, 0), (10, 2, 48, 70), (6, 3, 64, 0), (8, 8, 16, 0)])
def test_general_attention_gives_a_row_the_same_bits_in_any_step(ops, H, Hkv, hd, window):
    """The general kernel (the 32-bit path) takes up to four query heads of a kv head in one workgroup when the step
    has many rows, and one head per workgroup when it has few: a row's result is the same bits either way, and whatever
    the other rows of the step are (5 heads to a kv head: a workgroup of four and one that is nearly empty)."""
    page, n = 16, 420
    kc, vc, table, ks, vs = make_cache(1, [n], Hkv, hd, page, torch.float32, seed=H + hd)
    g = torch.Generator().manual_seed(2)
    q = (torch.randn(n, H * hd, generator=g) * 1.5).to(DEV)
    scale = 1.0 / math.sqrt(hd)
    positions = torch.arange(n, dtype=torch.int32, device=DEV)
    row_req = torch.zeros(n, dtype=torch.int32, device=DEV)
    whole = ops.paged_attention(q, kc, vc, table, row_req, positions, H, Hkv, hd, window, scale,
                                meta={"max_context": n, "decode_only": False, "requests": 1}, exact=True)
    for t in (0, 63, 64, 300, n - 1):
        alone = ops.paged_attention(q[t:t + 1].contiguous(), kc, vc, table, row_req[:1], positions[t:t + 1].contiguous(), H, Hkv,
                                    hd, window, scale, meta={"max_context": t + 1, "decode_only": True, "requests": 1},
                                    exact=True)
        assert torch.equal(alone[0], whole[t]), t
        ref = attention_reference(q[t].view(H, hd).cpu(), ks[0], vs[0], t, H, window, scale)
        assert torch.allclose(whole[t].view(H, hd).cpu().double(), ref, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("H,Hkv,hd,page,window", ATT_CASES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_decode_rows(ops, H, Hkv, hd, page, window, dtype):
    """One row per request at the end of contexts of very different lengths (1 key, a page's edge, several splits)."""
    ctx = [1, page, page + 1, 255, 256, 257, 700, 1500]
    kc, vc, table, ks, vs = make_cache(len(ctx), ctx, Hkv, hd, page, dtype, seed=H * hd)
    g = torch.Generator().manual_seed(1)
    q = (torch.randn(len(ctx), H, hd, generator=g) * 1.5).to(dtype)
    scale = 1.0 / math.sqrt(hd)
    positions = torch.tensor([c - 1 for c in ctx], dtype=torch.int32, device=DEV)
    row_req = torch.arange(len(ctx), dtype=torch.int32, device=DEV)
    meta = {"max_context": max(ctx), "decode_only": True, "requests": len(ctx)}
    out = ops.paged_attention(q.view(len(ctx), H * hd).to(DEV), kc, vc, table, row_req, positions, H, Hkv, hd, window,
                              scale, meta=meta, exact=dtype == torch.float32)
    assert not torch.isnan(out.float()).any(), "something read an unused cache slot"
    for r, c in enumerate(ctx):
        ref = attention_reference(q[r], ks[r], vs[r], c - 1, H, window, scale)
        got = out[r].view(H, hd).cpu().double()
        tol = 1e-5 if dtype == torch.float32 else 6e-3  # fp32 sums over up to 1500 keys
        assert (got - ref).abs().max() <= tol * max(1.0, ref.abs().max()), f"request {r} (context {c})"


@pytest.mark.parametrize("R", [12, 24, 40])
def test_decode_rows_with_longer_key_ranges(ops, R):
    """More rows make the decode attention cut the keys into ranges of 256 (12 rows here), 512 (24 rows) and 1,024 (40
    rows) instead of 128: contexts around every one of those edges."""
    H, Hkv, hd, page = 16, 8, 64, 16
    assert ops._decode_split(R, Hkv, 1500) == {12: 256, 24: 512, 40: 1024}[R]
    base = [1, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 1500]
    ctx = [base[i % len(base)] for i in range(R)]
    ctx[-1] = 1500
    kc, vc, table, ks, vs = make_cache(R, ctx, Hkv, hd, page, torch.bfloat16, seed=R)
    g = torch.Generator().manual_seed(R)
    q = (torch.randn(R, H, hd, generator=g) * 1.5).bfloat16()
    scale = 1.0 / math.sqrt(hd)
    positions = torch.tensor([c - 1 for c in ctx], dtype=torch.int32, device=DEV)
    row_req = torch.arange(R, dtype=torch.int32, device=DEV)
    meta = {"max_context": max(ctx), "decode_only": True, "requests": R}
    out = ops.paged_attention(q.view(R, H * hd).to(DEV), kc, vc, table, row_req, positions, H, Hkv, hd, 0, scale, meta=meta)
    assert not torch.isnan(out.float()).any()
    for r, c in enumerate(ctx):
        ref = attention_reference(q[r], ks[r], vs[r], c - 1, H, 0, scale)
        got = out[r].view(H, hd).cpu().double()
        assert (got - ref).abs().max() <= 6e-3 * max(1.0, ref.abs().max()), f"request {r} (context {c})"


def test_decode_rows_over_a_long_context(ops):
    """64 query heads over 8 key heads of 128 (the 32B shape) at contexts up to 16,500 keys: 17 key ranges of 1,024 to
    merge, and every range's edge."""
    H, Hkv, hd, page = 64, 8, 128, 16
    ctx = [16500, 16384, 16385, 9000, 1]
    R = len(ctx)
    kc, vc, table, ks, vs = make_cache(R, ctx, Hkv, hd, page, torch.bfloat16, seed=11)
    g = torch.Generator().manual_seed(12)
    q = (torch.randn(R, H, hd, generator=g) * 1.5).bfloat16()
    scale = 1.0 / math.sqrt(hd)
    positions = torch.tensor([c - 1 for c in ctx], dtype=torch.int32, device=DEV)
    row_req = torch.arange(R, dtype=torch.int32, device=DEV)
    meta = {"max_context": max(ctx), "decode_only": True, "requests": R}
    ops.reset_stats()
    out = ops.paged_attention(q.view(R, H * hd).to(DEV), kc, vc, table, row_req, positions, H, Hkv, hd, 0, scale, meta=meta)
    assert ops.stats()["ran"].get("jllm_decode_attention_bf16") == 1 and not ops.stats()["general"]
    assert not torch.isnan(out.float()).any()
    for r, c in enumerate(ctx):
        ref = attention_reference(q[r], ks[r], vs[r], c - 1, H, 0, scale)
        got = out[r].view(H, hd).cpu().double()
        assert (got - ref).abs().max() <= 6e-3 * max(1.0, ref.abs().max()), f"request {r} (context {c})"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_cache_addresses_beyond_four_gigabytes(ops, dtype):
    """A layer's cache of more than 2^32 bytes with the request's pages at its far end: the store of keys and
    values, the decode kernels (plain and fused), the portion kernel, the general kernel and the page copy all
    compute addresses in 64 bits (the reference checks the same arithmetic past 2^31 elements,
    cpu/LongContextTest.java:8-16)."""
    H, Hkv, hd, page = 8, 2, 128, 16
    esize = 4 if dtype == torch.float32 else 2
    page_bytes = Hkv * page * hd * esize
    n_pages = (5 << 30) // page_bytes
    assert (n_pages - 40) * page_bytes > 1 << 32
    storage = torch.empty((2, n_pages, Hkv, page, hd), dtype=dtype, device=DEV)  # keys and values as two runs of one tensor
    kc, vc = storage[0], storage[1]
    ctx, n_new = 300, 45  # 255 positions are in the cache, the step brings 45 more (it crosses pages)
    blocks = -(-ctx // page)
    gen = torch.Generator().manual_seed(3)
    pages = (n_pages - 1 - torch.randperm(blocks + 8, generator=gen)[:blocks]).to(torch.int32)
    kc[pages.long().to(DEV)] = float("nan")
    vc[pages.long().to(DEV)] = float("nan")
    table = pages.view(1, -1).to(DEV)
    k = torch.randn(ctx, Hkv, hd, generator=gen).to(dtype)
    v = torch.randn(ctx, Hkv, hd, generator=gen).to(dtype)
    old = ctx - n_new
    for b in range(-(-old // page)):
        n = min(page, old - b * page)
        kc[int(pages[b]), :, :n] = k[b * page:b * page + n].transpose(0, 1).to(DEV)
        vc[int(pages[b]), :, :n] = v[b * page:b * page + n].transpose(0, 1).to(DEV)
    q = (torch.randn(n_new, H, hd, generator=gen) * 1.5).to(dtype)
    qkv = torch.cat([q.view(n_new, -1), k[old:].reshape(n_new, -1), v[old:].reshape(n_new, -1)], dim=1).to(DEV)
    positions = torch.arange(old, ctx, dtype=torch.int32, device=DEV)
    slots = torch.tensor([int(pages[p // page]) * page + p % page for p in range(old, ctx)], dtype=torch.int32, device=DEV)
    row_req = torch.zeros(n_new, dtype=torch.int32, device=DEV)
    scale = 1.0 / math.sqrt(hd)
    tol = 1e-5 if dtype == torch.float32 else 8e-3
    # the store (no norm, no rotation: the bytes must arrive as they are) of all but the last new position
    ops.qk_norm_rope_store(qkv[:-1], positions[:-1], slots[:-1], None, None, None, None, 1e-6, H, Hkv, hd, 0, page, kc, vc)
    got_k = torch.stack([kc[int(pages[p // page]), :, p % page] for p in range(old, ctx - 1)]).cpu()
    assert torch.equal(got_k, k[old:ctx - 1]), "keys did not arrive at their far pages"
    # portions through the tiles
    meta = {"max_context": ctx - 1, "decode_only": False, "requests": 1, "n_tiles": 1,
            "segments_dev": torch.tensor([0, 0, n_new - 1, old], dtype=torch.int32, device=DEV)}
    ops.reset_stats()
    out = ops.paged_attention(qkv[:-1, :H * hd], kc, vc, table, row_req, positions, H, Hkv, hd, 0, scale, meta=meta,
                              exact=dtype == torch.float32)
    for t in (0, 17, n_new - 2):
        ref = attention_reference(q[t], k, v, old + t, H, 0, scale)
        assert (out[t].view(H, hd).cpu().double() - ref).abs().max() <= tol * max(1.0, ref.abs().max()), f"portion row {t}"
    # the last position as a decode step: fused (bf16) or store + single row
    meta = {"max_context": ctx, "decode_only": True, "requests": 1}
    last = None
    if dtype == torch.bfloat16:
        last = ops.decode_attention_fused(qkv[-1:], kc, vc, table, row_req[:1], positions[-1:], slots[-1:], None, None, None,
                                          None, 1e-6, H, Hkv, hd, 0, 0, scale, meta)
        assert last is not None
        assert not ops.stats()["general"], ops.stats()
    else:
        ops.qk_norm_rope_store(qkv[-1:], positions[-1:], slots[-1:], None, None, None, None, 1e-6, H, Hkv, hd, 0, page, kc, vc)
    again = ops.paged_attention(qkv[-1:, :H * hd], kc, vc, table, row_req[:1], positions[-1:], H, Hkv, hd, 0, scale, meta=meta,
                                exact=dtype == torch.float32)
    ref = attention_reference(q[-1], k, v, ctx - 1, H, 0, scale)
    for o in (last, again):
        if o is not None:
            assert (o.view(H, hd).cpu().double() - ref).abs().max() <= tol * max(1.0, ref.abs().max())
    # the page copy between two far pages
    src, dst = int(pages[0]), n_pages - 1 - (blocks + 8)
    ops.copy_page_rows(storage, src, dst, 5)
    assert torch.equal(kc[dst, :, :5], kc[src, :, :5]) and torch.equal(vc[dst, :, :5], vc[src, :, :5])
    del storage, kc, vc
    torch.cuda.empty_cache()


FUSED_CASES = [  # H, Hkv, hd, rotary width (0: no rotation), page, window, q/k norm gains (None: no norm)
    (4, 2, 16, 16, 8, 0, torch.bfloat16), (6, 2, 32, 32, 16, 0, torch.float32), (5, 5, 48, 48, 32, 20, torch.bfloat16),
    (8, 1, 64, 32, 4, 0, None), (3, 3, 80, 64, 16, 300, torch.bfloat16), (32, 8, 128, 128, 16, 0, torch.bfloat16),
    (16, 2, 128, 0, 16, 100, torch.float32), (2, 1, 256, 256, 16, 0, torch.bfloat16), (7, 7, 96, 96, 2, 0, torch.bfloat16),
    # head size 128, group sizes 1, 3, 5 (the 14B shape), 6, 7, 2
    (3, 3, 128, 128, 16, 0, torch.bfloat16), (6, 2, 128, 64, 16, 0, torch.bfloat16), (40, 8, 128, 128, 16, 0, torch.bfloat16),
    (6, 1, 128, 128, 8, 300, torch.float32), (7, 1, 128, 128, 16, 0, None), (4, 2, 128, 128, 4, 0, torch.bfloat16),
]


@pytest.mark.parametrize("H,Hkv,hd,rot,page,window,gdt", FUSED_CASES)
def test_decode_fused(ops, H, Hkv, hd, rot, page, window, gdt):
    """The fused decode attention (q/k norm, rotation, store of the new key and value and attention in one launch)
    against float64 and against the separate launches it replaces; and without the store, for a layer that reads
    another layer's cache."""
    ctx = [1, page, page + 1, 255, 256, 257, 700, 1500]
    R = len(ctx)
    kc0, vc0, table, ks, vs = make_cache(R, ctx, Hkv, hd, page, torch.bfloat16, seed=H * hd + 1)
    eps = 1e-4
    scale = 1.0 / math.sqrt(hd)
    gen = torch.Generator().manual_seed(7)
    positions = torch.tensor([c - 1 for c in ctx], dtype=torch.int32, device=DEV)
    row_req = torch.arange(R, dtype=torch.int32, device=DEV)
    slots = torch.tensor([int(table[r, (c - 1) // page]) * page + (c - 1) % page for r, c in enumerate(ctx)],
                         dtype=torch.int32, device=DEV)
    gq = gk = None
    if gdt is not None:
        gq = (torch.rand(hd, generator=gen) + 0.5).to(gdt).to(DEV)
        gk = (torch.rand(hd, generator=gen) + 0.5).to(gdt).to(DEV)
    cos = sin = None
    if rot:
        ang = torch.rand(max(ctx), rot // 2, generator=gen, dtype=torch.float64) * 6.28
        cos, sin = torch.cos(ang).float().to(DEV), torch.sin(ang).float().to(DEV)
    meta = {"max_context": max(ctx), "decode_only": True, "requests": R}

    def prepared(x, gain, pos):  # [heads, hd] float64: norm, rotation (half pairing), rounded to bf16 like the kernels
        x = x.double()
        if gain is not None:
            x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * gain.double().cpu()
        if rot:
            c, s_ = cos[pos].double().cpu(), sin[pos].double().cpu()
            a, b = x[:, :rot // 2].clone(), x[:, rot // 2:rot].clone()
            x[:, :rot // 2] = a * c - b * s_
            x[:, rot // 2:rot] = b * c + a * s_
        return x.float().bfloat16()

    for attempt in range(2):
        qkv = (torch.randn(R, (H + 2 * Hkv) * hd, generator=gen) * 1.5).bfloat16()
        kc, vc = kc0.clone(), vc0.clone()
        for r, c in enumerate(ctx):  # the new token's place holds NaN until the kernel stores it
            pg, off = int(slots[r]) // page, int(slots[r]) % page
            kc[pg, :, off] = float("nan")
            vc[pg, :, off] = float("nan")
        kc3, vc3, q3 = kc.clone(), vc.clone(), qkv.clone().to(DEV)
        out = ops.decode_attention_fused(qkv.to(DEV), kc, vc, table, row_req, positions, slots, cos, sin, gq, gk, eps, H,
                                         Hkv, hd, rot, window, scale, meta)
        assert out is not None, "the fused kernel declined a case it is meant to take"
        ops.qk_norm_rope_store(q3, positions, slots, cos, sin, gq, gk, eps, H, Hkv, hd, rot, page, kc3, vc3)
        out3 = ops.paged_attention(q3[:, :H * hd], kc3, vc3, table, row_req, positions, H, Hkv, hd, window, scale, meta=meta)
        assert not torch.isnan(out.float()).any()
        assert torch.equal(vc.view(torch.int16), vc3.view(torch.int16))
        kd = (kc.float() - kc3.float()).abs()
        assert not torch.isnan(kd[~torch.isnan(kc3.float())]).any()
        assert bool((kd[~torch.isnan(kc3.float())] <= 2.0 ** -7 * kc3.float().abs()[~torch.isnan(kc3.float())] + 1e-30).all())
        for r, c in enumerate(ctx):
            q = prepared(qkv[r, :H * hd].view(H, hd), gq, c - 1)
            k, v = ks[r].clone(), vs[r].clone()
            k[c - 1] = prepared(qkv[r, H * hd:(H + Hkv) * hd].view(Hkv, hd), gk, c - 1)
            v[c - 1] = qkv[r, (H + Hkv) * hd:].view(Hkv, hd)
            ref = attention_reference(q, k, v, c - 1, H, window, scale)
            got = out[r].view(H, hd).cpu().double()
            assert (got - ref).abs().max() <= 6e-3 * max(1.0, ref.abs().max()), f"request {r} (context {c}), attempt {attempt}"
            assert (got - out3[r].view(H, hd).cpu().double()).abs().max() <= 1.2e-2 * max(1.0, ref.abs().max())
    # a layer that reads another layer's cache: nothing is stored, the (complete) cache is only read
    before_k, before_v = kc3.clone(), vc3.clone()
    again = ops.decode_attention_fused(qkv.to(DEV), kc3, vc3, table, row_req, positions, slots, cos, sin, gq, gk, eps, H,
                                       Hkv, hd, rot, window, scale, meta, write_kv=False)
    assert torch.equal(kc3.view(torch.int16), before_k.view(torch.int16)) and torch.equal(vc3.view(torch.int16), before_v.view(torch.int16))
    assert (again.float() - out3.float()).abs().max() <= 1.2e-2 * max(1.0, float(out3.float().abs().max()))


@pytest.mark.parametrize("page", [1, 16])
@pytest.mark.parametrize("window", [0, 300, 385])
@pytest.mark.parametrize("order", [(0, 1, 2, 3, 4, 5), (5, 2, 0, 4, 1, 3), (1, 0)])
def test_decode_rows_of_one_range_and_of_several(ops, page, window, order):
    """Head size 128 takes rows of up to 384 keys (seen through the window) as one range and cuts longer ones: the rows on both
    sides of that line in one launch, rows that are the requests of their numbers (whose table entries are asked for ahead) and
    others, more requests in the table than rows, more entries in a range than threads (pages of one position). The bound: the
    probabilities that weight the values and the result are rounded to bf16 once each, by 2^-8 of their size at most; the sums
    are 32-bit (1e-4 covers them and the scores)."""
    H, Hkv, hd = 8, 2, 128
    ctx = [384, 385, 1, 383, 1100, 386]
    R = len(order)
    kc, vc, table, ks, vs = make_cache(len(ctx), ctx, Hkv, hd, page, torch.bfloat16, seed=page + window)
    gen = torch.Generator().manual_seed(R)
    positions = torch.tensor([ctx[r] - 1 for r in order], dtype=torch.int32, device=DEV)
    row_req = torch.tensor(order, dtype=torch.int32, device=DEV)
    slots = torch.tensor([int(table[r, (ctx[r] - 1) // page]) * page + (ctx[r] - 1) % page for r in order], dtype=torch.int32, device=DEV)
    qkv = (torch.randn(R, (H + 2 * Hkv) * hd, generator=gen) * 1.5).bfloat16()
    plain = ops.paged_attention(qkv[:, :H * hd].to(DEV), kc, vc, table, row_req, positions, H, Hkv, hd, window, hd ** -0.5,
                                meta={"max_context": max(ctx), "decode_only": True, "requests": R})
    meta = {"max_context": max(ctx), "decode_only": True, "requests": R, "arrivals": torch.zeros(R * Hkv, dtype=torch.int32, device=DEV)}
    fused = ops.decode_attention_fused(qkv.to(DEV), kc, vc, table, row_req, positions, slots, None, None, None, None, 1e-6, H, Hkv, hd,
                                       0, window, hd ** -0.5, meta)
    for i, r in enumerate(order):
        q, k, v = qkv[i, :H * hd].view(H, hd), ks[r].clone(), vs[r].clone()
        for got, name in ((plain, "plain"), (fused, "fused")):
            if name == "fused":
                k[-1], v[-1] = qkv[i, H * hd:(H + Hkv) * hd].view(Hkv, hd), qkv[i, (H + Hkv) * hd:].view(Hkv, hd)
            ref = attention_reference(q, k, v, ctx[r] - 1, H, window, hd ** -0.5)
            size = attention_reference(q, k, v.abs(), ctx[r] - 1, H, window, hd ** -0.5) + ref.abs()
            assert bool(((got[i].view(H, hd).cpu().double() - ref).abs() <= 2.0 ** -8 * size + 1e-4).all()), (name, r)
    assert int(meta["arrivals"].abs().max()) == 0


@pytest.mark.parametrize("H,Hkv,ctx,window,split", [(16, 8, (300, 1, 128, 129, 1024), 0, 128), (32, 8, (8000, 17, 5000), 0, 0),
                                                    (5, 1, (9100, 640), 0, 128), (8, 2, (3000, 700, 129), 300, 128), (64, 8, (2500,) * 9, 0, 0)])
def test_decode_attention_merged_by_its_last_workgroup(ops, monkeypatch, H, Hkv, ctx, window, split):
    """The splits of a row merged inside the launch by the workgroup that arrives last: bit for bit what the separate merge
    gives (same sums in the same order), for rows of one split, of up to eight, of more than eight and more than 64, through a
    window; over several launches that use the same counters, which are zero after each."""
    hd, page, R = 128, 16, len(ctx)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(H + sum(ctx))
    rnd = lambda *shape: torch.randn(*shape, device=DEV, generator=gen)
    width = -(-max(ctx) // page)
    table = torch.randperm(R * width, device=DEV, generator=gen).to(torch.int32).view(R, width)
    kc, vc = rnd(R * width, Hkv, page, hd).bfloat16(), rnd(R * width, Hkv, page, hd).bfloat16()
    rows = torch.arange(R, dtype=torch.int32, device=DEV)
    positions = torch.tensor([c - 1 for c in ctx], dtype=torch.int32, device=DEV)
    slots = torch.stack([table[r, (c - 1) // page] * page + (c - 1) % page for r, c in enumerate(ctx)]).to(torch.int32)
    if split:
        monkeypatch.setattr(ops, "_decode_split", lambda *_: split)
    arrivals = torch.zeros(R * Hkv, dtype=torch.int32, device=DEV)
    meta = {"max_context": max(ctx), "decode_only": True, "requests": R}
    for _ in range(3):
        qkv = rnd(R, (H + 2 * Hkv) * hd).bfloat16()
        run = lambda m: ops.decode_attention_fused(qkv, kc, vc, table, rows, positions, slots, None, None, None, None, 1e-6, H, Hkv, hd, 0,
                                                   window, hd ** -0.5, m)
        want, got = run(meta), run({**meta, "arrivals": arrivals})
        assert torch.equal(want.view(torch.int16), got.view(torch.int16)) and not torch.isnan(got.float()).any()
        assert int(arrivals.abs().max()) == 0


def _crafted_cache(ks, vs, table, ctx, page, dtype):
    """A cache tensor pair holding exactly the given keys and values of one request, NaN elsewhere."""
    n_pages = int(table.max()) + 2
    Hkv, hd = ks.shape[1], ks.shape[2]
    kc = torch.full((n_pages, Hkv, page, hd), float("nan")).to(dtype)
    vc = torch.full((n_pages, Hkv, page, hd), float("nan")).to(dtype)
    for b in range(-(-ctx // page)):
        pg = int(table[0, b])
        n = min(page, ctx - b * page)
        kc[pg, :, :n] = ks[b * page:b * page + n].transpose(0, 1).to(dtype)
        vc[pg, :, :n] = vs[b * page:b * page + n].transpose(0, 1).to(dtype)
    return kc.to(DEV), vc.to(DEV)


# how the rows of the crafted request reach the attention: one decoding row; the same through the fused decode kernel;
# a tile of 128 rows whose last row is the crafted one; a portion of two rows; a single row riding beside a portion of
# another request (a mixed step, which takes the single rows through the decode kernel)
FAR_FORMS = ["decode", "fused", "tile", "two", "mixed"]


@pytest.mark.parametrize("form", FAR_FORMS)
@pytest.mark.parametrize("hd,H,Hkv", [(64, 4, 2), (128, 8, 2), (128, 5, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_far_key_and_window_edge(ops, dtype, hd, H, Hkv, form):
    """Keys made so that a fault shows: one far key among 1200 carries all the weight; with a window, the key just
    outside it would dominate if it were read and the key just inside does dominate. The window's first key is put
    on a split's edge (a multiple of 128, 256 and 512), on a page's edge, and one key before and after them."""
    if form == "fused" and dtype == torch.float32:
        pytest.skip("the fused decode kernel is a bfloat16 kernel")
    page = 16
    ctx = 1200
    G = H // Hkv
    gen = torch.Generator().manual_seed(hd + H)
    blocks = -(-ctx // page)
    perm = torch.randperm(blocks + 3, generator=gen)
    table = perm[:blocks].to(torch.int32).view(1, -1)
    k = torch.randn(ctx, Hkv, hd, generator=gen) * 0.05
    v = torch.randn(ctx, Hkv, hd, generator=gen)
    scale = 1.0
    pos = ctx - 1

    def run(window, special, other=None):
        kk = k.clone()
        kk[special, :, 0] = 4.0  # score 32 against about 0 elsewhere
        if other is not None:
            kk[other, :, 0] = 6.0  # would win if it were visible
        kc, vc = _crafted_cache(kk, v, table, ctx, page, dtype)
        tab = table.to(DEV)
        qrow = torch.zeros(H, hd)
        qrow[:, 0] = 8.0
        if form in ("decode", "fused"):
            n, p0 = 1, pos
        elif form == "tile":
            n, p0 = 128, pos - 127
        elif form == "two":
            n, p0 = 2, pos - 1
        else:
            n, p0 = 1, pos
        q = torch.zeros(n, H, hd)
        q[-1] = qrow
        positions = torch.arange(p0, p0 + n, dtype=torch.int32)
        row_req = torch.zeros(n, dtype=torch.int32)
        meta = {"max_context": ctx, "decode_only": form in ("decode", "fused"), "requests": 1}
        if form == "fused":
            qkv = torch.zeros(1, (H + 2 * Hkv) * hd)
            qkv[0, :H * hd] = qrow.view(-1)
            qkv[0, H * hd:(H + Hkv) * hd] = kk[pos].view(-1)
            qkv[0, (H + Hkv) * hd:] = v[pos].view(-1)
            slot = int(table[0, pos // page]) * page + pos % page
            out = ops.decode_attention_fused(qkv.bfloat16().to(DEV), kc, vc, tab, row_req.to(DEV), positions.to(DEV),
                                             torch.tensor([slot], dtype=torch.int32, device=DEV), None, None, None, None,
                                             1e-6, H, Hkv, hd, 0, window, scale, meta)
            assert out is not None
            return out.view(H, hd).cpu().float()
        if form == "mixed":
            # another request brings a portion of 40 rows in the same step; its pages follow in the table's second row
            n2, ctx2 = 40, 40
            k2 = torch.randn(ctx2, Hkv, hd, generator=torch.Generator().manual_seed(5)) * 0.05
            tab2 = torch.zeros(2, table.shape[1], dtype=torch.int32)
            tab2[0] = table[0]
            extra = [int(perm[blocks]), int(perm[blocks + 1]), int(perm[blocks + 2])]
            tab2[1, :3] = torch.tensor(extra, dtype=torch.int32)
            for b in range(3):
                m = min(page, ctx2 - b * page)
                kc[extra[b], :, :m] = k2[b * page:b * page + m].transpose(0, 1).to(dtype).to(DEV)
                vc[extra[b], :, :m] = k2[b * page:b * page + m].transpose(0, 1).to(dtype).to(DEV)
            q = torch.cat([torch.randn(n2, H, hd, generator=torch.Generator().manual_seed(6)), qrow[None]])
            positions = torch.cat([torch.arange(n2, dtype=torch.int32), torch.tensor([pos], dtype=torch.int32)])
            row_req = torch.cat([torch.ones(n2, dtype=torch.int32), torch.zeros(1, dtype=torch.int32)])
            tiles = [1, 0, n2, 0, 0, n2, 1, pos]
            meta.update(requests=2, n_tiles=2, n_tiles_multi=1, single_rows=(n2, 1),
                        segments_dev=torch.tensor(tiles, dtype=torch.int32, device=DEV))
            tab = tab2.to(DEV)
        elif form in ("tile", "two"):
            meta.update(n_tiles=1, segments_dev=torch.tensor([0, 0, n, p0], dtype=torch.int32, device=DEV))
        out = ops.paged_attention(q.view(-1, H * hd).to(dtype).to(DEV), kc, vc, tab, row_req.to(DEV), positions.to(DEV), H,
                                  Hkv, hd, window, scale, meta=meta, exact=dtype == torch.float32)
        return out[-1].view(H, hd).cpu().float()

    ops.reset_stats()
    far = run(0, 37)
    for h in range(H):
        assert torch.allclose(far[h], v[37, h // G].float(), atol=2e-2), "the far key's value must come through"
    for first in (pos + 1 - 100, 1024, 1023, 1025, 512, 768, 1168, 1167, pos - 1, pos):
        w = pos + 1 - first  # the window whose oldest visible key, for the last row, is `first`
        edge = run(w, first, other=first - 1)
        for h in range(H):
            assert torch.allclose(edge[h], v[first, h // G].float(), atol=2e-2), \
                f"window edge at key {first}: the key inside must win, the one outside is unseen (head {h})"
    if dtype == torch.bfloat16:
        assert not ops.stats()["general"], f"a matrix-core or split-key kernel declined: {ops.stats()}"


@pytest.mark.parametrize("H,Hkv,hd,page,window", ATT_CASES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_portions(ops, H, Hkv, hd, page, window, dtype):
    """A batch of portions at different places of their requests (a whole prompt, a portion deep inside a long
    context, two tokens, one token) beside each other."""
    ctx = [130, 900, 40, 513, 7]        # keys held after this step
    ns = [130, 200, 2, 1, 7]            # rows of this step (the last ns positions of each request)
    R = len(ctx)
    kc, vc, table, ks, vs = make_cache(R, ctx, Hkv, hd, page, dtype, seed=hd + page)
    g = torch.Generator().manual_seed(2)
    T = sum(ns)
    q = (torch.randn(T, H, hd, generator=g) * 1.5).to(dtype)
    scale = 1.0 / math.sqrt(hd)
    pos, req, tiles = [], [], []
    row = 0
    for r in range(R):
        p0 = ctx[r] - ns[r]
        pos += list(range(p0, ctx[r]))
        req += [r] * ns[r]
        for a in range(0, ns[r], 128):
            tiles += [r, row + a, min(128, ns[r] - a), p0 + a]
        row += ns[r]
    positions = torch.tensor(pos, dtype=torch.int32, device=DEV)
    row_req = torch.tensor(req, dtype=torch.int32, device=DEV)
    meta = {"max_context": max(ctx), "decode_only": False, "requests": R,
            "segments_dev": torch.tensor(tiles, dtype=torch.int32, device=DEV), "n_tiles": len(tiles) // 4}
    wide = torch.zeros(T, H * hd + 2 * Hkv * hd, dtype=dtype)
    wide[:, :H * hd] = q.view(T, H * hd)
    wide = wide.to(DEV)
    out = ops.paged_attention(wide[:, :H * hd], kc, vc, table, row_req, positions, H, Hkv, hd, window, scale,
                              meta=meta, exact=dtype == torch.float32)
    assert not torch.isnan(out.float()).any(), "something read an unused cache slot"
    tol = 1e-5 if dtype == torch.float32 else 8e-3  # fp32 sums over hundreds of keys; the reference's 2e-6 is for 40
    for t in range(T):
        r = req[t]
        ref = attention_reference(q[t], ks[r], vs[r], pos[t], H, window, scale)
        got = out[t].view(H, hd).cpu().double()
        assert (got - ref).abs().max() <= tol * max(1.0, ref.abs().max()), f"row {t} (request {r}, position {pos[t]})"


@pytest.mark.parametrize("window", [0, 200])
def test_portions_in_a_small_and_in_a_large_step(ops, window):
    """The matrix-core kernel for portions has two forms: with few tiles in the step a workgroup cuts a tile's keys
    over two groups of waves and merges them, with many it does not. The same 300 rows deep inside a request, alone
    (3 tiles) and beside a 4,200-token prompt (36 tiles at 16 heads: more workgroups than two per compute unit),
    against the reference, and the two against each other."""
    H, Hkv, hd, page = 16, 4, 128, 16
    assert H * 36 > 2 * ops.compute_units() >= H * 3, "the sizes of this test assume about 256 compute units"
    ctx, ns = [900, 4200], [300, 4200]
    kc, vc, table, ks, vs = make_cache(2, ctx, Hkv, hd, page, torch.bfloat16, seed=77)
    g = torch.Generator().manual_seed(3)
    q = (torch.randn(sum(ns), H, hd, generator=g) * 1.5).bfloat16()
    scale = 1.0 / math.sqrt(hd)

    def run(requests):
        pos, req, tiles, rows = [], [], [], []
        row = 0
        for i, r in enumerate(requests):
            p0 = ctx[r] - ns[r]
            pos += list(range(p0, ctx[r]))
            req += [i] * ns[r]
            rows += list(range(sum(ns[:r]), sum(ns[:r]) + ns[r]))
            for a in range(0, ns[r], 128):
                tiles += [i, row + a, min(128, ns[r] - a), p0 + a]
            row += ns[r]
        order = sorted(range(len(tiles) // 4), key=lambda t: -(tiles[4 * t + 3] + tiles[4 * t + 2]))  # most keys first
        tiles = [x for t in order for x in tiles[4 * t:4 * t + 4]]
        meta = {"max_context": max(ctx[r] for r in requests), "decode_only": False, "requests": len(requests),
                "segments_dev": torch.tensor(tiles, dtype=torch.int32, device=DEV), "n_tiles": len(tiles) // 4}
        return ops.paged_attention(q[rows].view(len(rows), H * hd).to(DEV), kc, vc, table[requests].contiguous(),
                                   torch.tensor(req, dtype=torch.int32, device=DEV),
                                   torch.tensor(pos, dtype=torch.int32, device=DEV), H, Hkv, hd, window, scale, meta=meta)

    ops.reset_stats()
    small = run([0])[:300].float().cpu()
    large = run([0, 1])[:300].float().cpu()
    assert ops.stats()["ran"].get("jllm_prefill_attention_bf16") == 2 and not ops.stats()["general"], ops.stats()
    assert not torch.equal(small, large), "the two forms add in different orders: equal bits mean one form ran twice"
    for t in range(0, 300, 7):
        ref = attention_reference(q[t], ks[0], vs[0], ctx[0] - 300 + t, H, window, scale)
        for got in (small[t], large[t]):
            assert (got.view(H, hd).double() - ref).abs().max() <= 8e-3 * max(1.0, ref.abs().max()), f"row {t}"
    assert (small - large).abs().max() <= 8e-3 * max(1.0, small.abs().max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_copy_page_rows(ops, dtype):
    storage = torch.randn(3, 7, 2, 8, 48, device=DEV).to(dtype)  # [runs, pages, heads, page size, head size]
    before = storage.clone()
    ops.copy_page_rows(storage, 5, 2, 3)
    want = before.clone()
    want[:, 2, :, :3, :] = before[:, 5, :, :3, :]
    assert torch.equal(storage, want), "rows 0..2 of page 5 go to page 2 in every run and head; nothing else moves"
    odd = torch.randint(0, 255, (2, 4, 1, 4, 7), device=DEV).to(torch.uint8)  # 7 bytes per position: the byte path
    before = odd.clone()
    ops.copy_page_rows(odd, 0, 3, 2)
    want = before.clone()
    want[:, 3, :, :2] = before[:, 0, :, :2]
    assert torch.equal(odd, want)
    with pytest.raises(ops.KernelError):
        ops.copy_page_rows(storage, 5, 9, 3)
    with pytest.raises(ops.KernelError):
        ops.copy_page_rows(storage, 5, 2, 9)
