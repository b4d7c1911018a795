"""The small-tile product kernels and the rules that choose them, against the
kernels whose place they take: bit for bit."""
import numpy as np
import pytest

from decisive_amd import rocm
from gpu_util import bits_equal, dev, empty, host, launched
from tests import pplx_model
from tests.test_gpu_pplx import SMALL

pytestmark = pytest.mark.gpu

SMALL_W4A16 = ("small32x32", "small32x64", "small64x64", "small64x128", "pipe-auto")


@pytest.mark.parametrize("group", [32, 64])
@pytest.mark.parametrize("m,k,n", [
    (17, 8, 1), (33, 120, 63), (31, 128, 64), (32, 136, 65), (65, 256, 129),  # edges of tiles, one partial or whole block
    (64, 384, 128), (63, 640, 127), (129, 1000, 272),                          # fewer steps than the ring, ragged k
    (40, 4096, 4096), (200, 2568, 1040), (2100, 1688, 1063),                   # long rings; the ragged pipelined tiles
])
def test_w4a16_small_tiles_give_the_staged_kernels_bits(ctx, group, m, k, n):
    """Every small tile and the automatic choice against the register-staged
    kernel (pinned to the closed form elsewhere): the same MFMA per 32-k run in
    k order, so the same bits, in f32 and through each f16 epilogue."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(m + k + n + group)
    x = dev(rng.standard_normal((m, k)).astype(np.float16))
    w = ctx.quantize(dev((rng.standard_normal((n, k)) * 0.02).astype(np.float32)), rocm.F32, n, k, 4, group)
    res = dev(rng.standard_normal((m, n)).astype(np.float16))

    def outputs(name):
        ctx.select_variant("gemm_w4a16", name)
        y = empty((m, n), torch.float32)
        ctx.linear(w, x, rocm.F16, m, y, rocm.W4A16)
        outs = [host(ctx, y)]
        for epi in (rocm.EPI_NONE, rocm.EPI_GELU, rocm.EPI_RESIDUAL):
            h = empty((m, n), torch.float16)
            ctx.linear_f16(w, x, m, h, epi, res if epi == rocm.EPI_RESIDUAL else None)
            outs.append(host(ctx, h).view(np.uint16))
        return outs

    try:
        want = outputs("256x128w2x2")
        assert np.isfinite(want[0]).all()
        for name in SMALL_W4A16:
            got = outputs(name)
            assert bits_equal(got[0], want[0]), name
            assert all(np.array_equal(a, b) for a, b in zip(got[1:], want[1:])), name
    finally:
        ctx.select_variant("gemm_w4a16", "pipe-auto")


@pytest.mark.parametrize("m,k,n,kernel,tile", [
    (700, 1080, 4001, "gemm_w4a16_kernel", (128, 128)), (700, 1096, 4001, "w4a16_pipe_kernel", (128, 128)),    # short products
    (700, 1080, 4004, "w4a16_pipe_kernel", (128, 128)), (700, 1024, 4001, "w4a16_pipe_kernel", (128, 128)),    # whole vectors, k-blocks
    (4096, 136, 4096, "w4a16_pipe_kernel", (256, 256)), (4097, 136, 4096, "w4a16_pipe_kernel", (128, 128)),    # one 256x256 per unit
    (5120, 136, 4096, "w4a16_pipe_kernel", (128, 128)), (5121, 136, 4096, "w4a16_pipe_kernel", (256, 256)),    # one and a quarter
    (300, 1080, 4001, "w4a16_small_kernel", (64, 128)), (4100, 200, 4099, "gemm_w4a16_kernel", (128, 128)),    # small tiles first
])
def test_w4a16_rule_at_ragged_k_takes_the_measured_kernel(ctx, m, k, n, kernel, tile):
    """On both sides of the lines of the rule where k is not whole blocks (256
    units): the kernel that runs, for f32 and plain f16 outputs, and no staged
    one through the other epilogues."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(k)
    w = ctx.quantize(dev((rng.standard_normal((n, k)) * 0.02).astype(np.float32)), rocm.F32, n, k, 4, 32)
    x, y, h = dev(rng.standard_normal((m, k)).astype(np.float16)), empty((m, n), torch.float32), empty((m, n), torch.float16)
    forms = ["{}<{}, {},".format(kernel, *tile), "{}ILi{}ELi{}E".format(kernel, *tile)]  # demangled or not
    for run in (lambda: ctx.linear(w, x, rocm.F16, m, y, rocm.W4A16), lambda: ctx.linear_f16(w, x, m, h, rocm.EPI_NONE)):
        got = launched(ctx, run)
        assert any(f in g for g in got for f in forms), got
    got = launched(ctx, lambda: ctx.linear_f16(w, x, m, h, rocm.EPI_GELU))
    assert not any("gemm_w4a16_kernel" in g for g in got), got


@pytest.mark.parametrize("k", [1000, 4096])
def test_w4a16_rows_do_not_see_each_other(ctx, k):
    """A row of infinities beside finite ones: the chunks a partial block loads
    past a row's end are the next row's and must not reach it."""
    torch = pytest.importorskip("torch")
    m, n = 70, 96
    rng = np.random.default_rng(k)
    clean = rng.standard_normal((m, k)).astype(np.float16)
    dirty = clean.copy()
    dirty[1::2] = np.inf
    w = ctx.quantize(dev((rng.standard_normal((n, k)) * 0.02).astype(np.float32)), rocm.F32, n, k, 4, 32)
    try:
        for name in SMALL_W4A16 + ("128x128p2w4", "256x256p2w8-persist"):
            ctx.select_variant("gemm_w4a16", name)
            outs = []
            for v in (clean, dirty):
                y = empty((m, n), torch.float32)
                ctx.linear(w, dev(v), rocm.F16, m, y, rocm.W4A16)
                outs.append(host(ctx, y))
            assert bits_equal(outs[1][0::2], outs[0][0::2]), name
            assert not np.isfinite(outs[1][1::2]).any(), name
    finally:
        ctx.select_variant("gemm_w4a16", "pipe-auto")


@pytest.mark.parametrize("m,n,k", [
    (1, 1, 4), (16, 16, 64), (17, 33, 68), (32, 47, 508), (33, 64, 512),        # the few-row kernel's edges and chunk tails
    (64, 65, 20), (65, 129, 132), (300, 4096, 260), (129, 1000, 516),           # small tiles, partial words of a chunk
    (700, 2100, 1004), (40, 70, 30), (520, 300, 1001),                          # most 64x64 tiles; staged k
    (1000, 2000, 1004), (1100, 1900, 508),                                      # auto: ragged 128x128, eight and four steps
    (2100, 4100, 76), (2100, 4100, 132), (2100, 4100, 268), (2100, 4100, 396),  # auto: ragged 256x256, one to four steps
])
def test_i8_products_of_every_size_are_exact(ctx, m, n, k):
    """The automatic choice and the small kernels against float64 dots (exact
    below 2^53) over the whole code range, in raw int32 and through the f32
    epilogue, and nothing written past the output."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-127, 128, (m, k), dtype=np.int8)
    b = rng.integers(-127, 128, (n, k), dtype=np.int8)
    sa, sb = (rng.uniform(0.1, 2.0, s).astype(np.float32) for s in (m, n))
    dots = (a.astype(np.float64) @ b.astype(np.float64).T).astype(np.int32)
    want = ((dots.astype(np.float32) * sa[:, None]).astype(np.float32) * sb).astype(np.float32)
    da, db, dsa, dsb = dev(a), dev(b), dev(sa), dev(sb)
    try:
        for name in ("auto", "256x256p2w8", "rows", "64x64p4", "128x128p3w8"):
            ctx.select_variant("i8_gemm", name)
            r = torch.full((m * n + 64,), -7, dtype=torch.int32, device="cuda")
            y = torch.full((m * n + 64,), -7.0, dtype=torch.float32, device="cuda")
            torch.cuda.synchronize()
            ctx.i8_gemm(da, dsa, m, db, dsb, n, k, r, raw=True)
            ctx.i8_gemm(da, dsa, m, db, dsb, n, k, y, raw=False)
            raw, f = host(ctx, r), host(ctx, y)
            assert np.array_equal(raw[:m * n].reshape(m, n), dots), name
            assert bits_equal(f[:m * n].reshape(m, n), want), name
            assert (raw[m * n:] == -7).all() and (f[m * n:] == -7.0).all(), name
    finally:
        ctx.select_variant("i8_gemm", "auto")


@pytest.mark.parametrize("k", [4, 6, 1024, 1028, 2052, 4096, 8196, 16388, 32768])
def test_i8_row_quantizer_of_every_width(ctx, oracle, k):
    """The vector row quantizer's register counts and the scalar kernel (k % 4
    != 0) against the oracle, codes, scales and sums; a zero row and a row with
    an infinity among them."""
    torch = pytest.importorskip("torch")
    rows = 5
    x = np.random.default_rng(k).standard_normal((rows, k)).astype(np.float32)
    x[1] = 0.0
    q, s, sums = empty((rows, k), torch.int8), empty((rows,), torch.float32), empty((rows,), torch.int32)
    ctx.i8_quantize_rows(dev(x), rows, k, q, s, sums)
    wq, ws, wsum = oracle.i8_quantize_rows(x, rows, k)
    assert np.array_equal(host(ctx, q), wq) and bits_equal(host(ctx, s), ws) and np.array_equal(host(ctx, sums), wsum)
    x[2, k // 2] = np.inf
    ctx.i8_quantize_rows(dev(x), rows, k, q, s)
    assert np.isinf(host(ctx, s)[2]) and np.array_equal(host(ctx, q)[[0, 1, 3, 4]], wq[[0, 1, 3, 4]])
    assert not host(ctx, q)[2].any()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,k,n", [(17, 64, 16), (31, 320, 63), (33, 576, 65), (48, 192, 200), (129, 1088, 128)])
def test_grouped_four_group_tiles_give_the_one_wave_kernels_bits(ctx, bits, m, k, n):
    """The 16x64 and 32x64 tiles with four groups per step: one to seventeen
    groups (a last step of one, two or three), ragged rows and columns, no
    store past the output."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(m + n + k + bits)
    w = ctx.quantize(dev((rng.standard_normal((n, k)) * 0.05).astype(np.float32)), rocm.F32, n, k, bits, 64)
    x = dev(rng.standard_normal((m, k)).astype(np.float32))
    out = {}
    try:
        for name in ("wave16x16", "pipe32x64w4g4", "pipe16x64w4g4"):
            ctx.select_variant("grouped", name)
            y = torch.full((m * n + 64,), -7.0, dtype=torch.float32, device="cuda")
            torch.cuda.synchronize()
            ctx.linear(w, x, rocm.F32, m, y, rocm.W4A8)
            out[name] = host(ctx, y)
            assert (out[name][m * n:] == -7.0).all(), name
    finally:
        ctx.select_variant("grouped", "pipe-auto")
    for name in out:
        assert bits_equal(out[name], out["wave16x16"]), name


@pytest.mark.parametrize("layer,n", [(1, 17), (1, 37), (1, 130), (3, 77)])
def test_four_group_tiles_add_the_residual_in_their_store(ctx, oracle, layer, n):
    """out_proj, o_proj and down_proj onto the hidden rows, on the 32x64 and
    16x64 tiles and by the separate add of the one-wave kernel."""
    pytest.importorskip("torch")
    model = pplx_model.random_model(oracle, SMALL, seed=4)
    p = pplx_model.load(ctx, rocm, model)
    h = np.random.default_rng(n).standard_normal((n, SMALL["hidden"])).astype(np.float32)
    out = {}
    for name in ("wave16x16", "pipe32x64w4", "pipe32x64w4g4", "pipe16x64w4g4"):
        hd = dev(h)
        ctx.select_variant("grouped", name)
        try:
            p.layer(layer, hd, n)
        finally:
            ctx.select_variant("grouped", "pipe-auto")
        out[name] = host(ctx, hd)
    p.close()
    assert np.isfinite(out["wave16x16"]).all()
    for name in out:
        assert bits_equal(out[name], out["wave16x16"]), name


@pytest.mark.parametrize("bits,m,n,tile", [
    (4, 208, 2560, "16, 64, 1, 4"), (4, 240, 2560, "16, 64, 1, 4"), (4, 241, 2560, "32, 64, 1, 4"),  # 2.5 16x64 blocks per unit
    (4, 608, 2560, "32, 64, 1, 4"), (4, 640, 2560, "32, 128, 1, 8"), (4, 800, 2560, "32, 128, 1, 8"),  # three 32x64
    (4, 192, 8192, "32, 64, 1, 4"), (4, 193, 8192, "32, 128, 1, 8"), (8, 640, 2560, "32, 64, 1, 4"),
    (4, 48, 9520, "16, 64, 1, 4"), (4, 53, 9520, "32, 64, 1, 4"), (4, 454, 1183, "16, 64, 1, 4"), (4, 125, 4672, "16, 64, 1, 4"),
    (4, 503, 3869, "32, 64, 1, 4"),  # stored a value at a time, few groups
    (4, 3538, 128, "32, 128, 1, 8"), (4, 3000, 128, "16, 64, 1, 4"), (4, 2600, 128, "16, 64, 1, 4"),  # one column of 32x128
    (8, 4097, 128, "32, 128, 1, 8"), (8, 4096, 128, "16, 64, 1, 4"), (8, 4097, 129, "32, 64, 1, 4"),
    (8, 97, 4160, "16, 64, 1, 4"), (8, 113, 4160, "32, 64, 1, 4"), (8, 192, 2560, "16, 64, 1, 4"),   # Q8: two 16x64 per unit;
    (8, 208, 2560, "32, 64, 1, 4"), (8, 300, 4005, "32, 64, 1, 4"),                                # some grids not whole rounds
])
def test_grouped_rule_takes_the_measured_tile(ctx, bits, m, n, tile):
    """On both sides of the lines of the grouped rule for grids below two
    32x128 blocks per unit (256 units): the tile that runs, with four groups
    per step, and its bits."""
    torch = pytest.importorskip("torch")
    k = 192
    rng = np.random.default_rng(m + n + bits)
    w = ctx.quantize(dev((rng.standard_normal((n, k)) * 0.05).astype(np.float32)), rocm.F32, n, k, bits, 64)
    x = dev(rng.standard_normal((m, k)).astype(np.float32))
    y, want = empty((m, n), torch.float32), empty((m, n), torch.float32)
    got = launched(ctx, lambda: ctx.linear(w, x, rocm.F32, m, y, rocm.W4A8))
    assert any(f"grouped_pipe_kernel<{bits}, {tile}, false, 4>" in g for g in got), got
    try:
        ctx.select_variant("grouped", "wave16x16")
        ctx.linear(w, x, rocm.F32, m, want, rocm.W4A8)
    finally:
        ctx.select_variant("grouped", "pipe-auto")
    assert bits_equal(host(ctx, y), host(ctx, want))


@pytest.mark.parametrize("m,k,n", [(1, 64, 64), (3, 128, 64), (4, 192, 128), (63, 320, 64), (65, 1088, 192), (129, 576, 64)])
def test_mlp_64_row_blocks_give_the_one_wave_kernels_bits(ctx, m, k, n):
    """The fused MLP's 64x64 blocks: odd group counts, one group, ragged rows,
    and the rows where the choice of kernel turns."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(m + n + k)
    gate, up = (ctx.quantize(dev((rng.standard_normal((n, k)) * 0.05).astype(np.float32)), rocm.F32, n, k, 4, 64)
                for _ in range(2))
    x = dev((rng.standard_normal((m, k)) * 1.3).astype(np.float32))
    out = {}
    try:
        for name in ("wave16x64", "pipe64x64n4", "pipe-auto"):
            ctx.select_variant("mlp", name)
            q = torch.full((m * n + 64,), 99, dtype=torch.int8, device="cuda")
            s = torch.full((m * n // 64 + 16,), -7.0, dtype=torch.float32, device="cuda")
            torch.cuda.synchronize()
            ctx.mlp_requant(gate, up, x, m, q, s)
            out[name] = host(ctx, q), host(ctx, s)
            assert (out[name][0][m * n:] == 99).all() and (out[name][1][m * n // 64:] == -7.0).all(), name
    finally:
        ctx.select_variant("mlp", "pipe-auto")
    for name in out:
        assert np.array_equal(out[name][0], out["wave16x64"][0]) and bits_equal(out[name][1], out["wave16x64"][1]), name


@pytest.mark.parametrize("m,k,n,small", [
    (3, 640, 64, True), (4, 384, 64, False),                                    # rows
    (64, 320, 1024, True), (64, 384, 1024, False),                              # five groups
    (256, 320, 1024, True), (257, 320, 1024, False),                            # one block per unit
    (320, 192, 1024, True), (321, 192, 1024, False), (320, 256, 1024, False),   # one and a quarter, up to three groups
    (640, 64, 1024, True), (641, 64, 1024, False),                              # two and a half, at one group
])
def test_mlp_rule_takes_the_measured_blocks(ctx, m, k, n, small):
    """On both sides of the lines between the one-wave and the 64-row blocks
    (256 units): the kernel that runs."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(m + n + k)
    gate, up = (ctx.quantize(dev((rng.standard_normal((n, k)) * 0.05).astype(np.float32)), rocm.F32, n, k, 4, 64)
                for _ in range(2))
    x = dev(rng.standard_normal((m, k)).astype(np.float32))
    q, s = empty((m, n), torch.int8), empty((m, n // 64), torch.float32)
    got = launched(ctx, lambda: ctx.mlp_requant(gate, up, x, m, q, s))
    want = "mlp_requant_kernel" if small else "mlp_pipe_kernel<64, 4, 1>"
    assert any(want in g for g in got), got
