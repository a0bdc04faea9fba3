"""GPU parity: the MFMA dequant-GEMM (prefill) against the exact-fp32 oracle.

Tolerance stated by the task for the bf16-MFMA path: max relative error 2e-2 against the fp32 reference, measured
as |got - ref| / max(|ref|, 1e-2 * ||ref||_inf). The reference has no packed GEMM (m rows = m scalar GEMV calls,
PackedViewMatmulKernel.kt:99), which is exactly what the oracle does here.
"""
import numpy as np
import pytest

from oracle import golden as G
from oracle import lib as L
from gpu_util import ENCS, MORE_ENCS, dev, gaussian_weight, launches, normalized_err, random_valid_blocks

ALL_ENCS = ENCS + MORE_ENCS

pytestmark = pytest.mark.gpu
GEMM_TOL = 2e-2       # max |got - ref| / ||ref||_inf against the exact-fp32 oracle
GEMM_RMS_TOL = 1e-2   # RMS(err) / RMS(ref), the aggregate form the reference uses for its own reduced-precision path
                      # (NativeQ4KMatmulKernelParityTest.kt:84-103, bound 0.03 there)
EXACT_TOL = 2e-4      # against the same product with both operands rounded to bf16 first (what the kernel computes)


def check(got, want_fp32):
    """bf16-MFMA bound: operands carry 8 significant bits, so an output near zero has an unbounded per-element
    relative error; the bound is taken against the largest output (and in aggregate)."""
    err = normalized_err(got, want_fp32, eps=1.0)
    rms = float(np.sqrt(((got - want_fp32.astype(np.float64)) ** 2).mean()) / max(np.sqrt((want_fp32.astype(np.float64) ** 2).mean()), 1e-30))
    assert err <= GEMM_TOL and rms <= GEMM_RMS_TOL, (err, rms)
    return err


def bf16_round(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(torch.bfloat16).to(torch.float64).numpy()


def check_exact(torch, enc, got, x, packed, n):
    """The kernel's own arithmetic restated: decode (oracle, fp32) -> bf16, activations -> bf16, exact products, wide sums.
    Only the fp32 accumulation order is left, so a wrong fragment layout or a misplaced scale cannot hide."""
    w = bf16_round(torch, L.dequant(enc, packed).reshape(n, -1))
    want = bf16_round(torch, x) @ w.T
    assert normalized_err(got, want) <= EXACT_TOL, normalized_err(got, want)


def gpu_gemm(kernels, torch, enc, packed, n, k, x, kind=1):
    w = kernels.DeviceWeight.upload(enc, packed, n, k)
    m = x.shape[0]
    y = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda")
    w.matmul(dev(torch, x), m, y, kind)
    return y.cpu().numpy()


@pytest.mark.parametrize("enc", ALL_ENCS)
@pytest.mark.parametrize("m,n,k", [(9, 5, 256), (33, 130, 512), (256, 128, 1024), (300, 257, 768), (64, 1000, 2304), (1, 64, 256)])
def test_gemm_ragged_tiles(hip_backend, torch_cuda, enc, m, n, k):
    packed = gaussian_weight(hip_backend, enc, n, k, 200 + n)
    x = np.random.default_rng(m + k).standard_normal((m, k)).astype(np.float32)
    got = gpu_gemm(hip_backend, torch_cuda, enc, packed, n, k, x)
    want = L.gemv(enc, x, packed, n)
    assert not np.isnan(got).any()
    check(got, want)
    check_exact(torch_cuda, enc, got, x, packed, n)
    # the automatic choice (m > 8 -> GEMM, else GEMV) gives the same product
    auto = gpu_gemm(hip_backend, torch_cuda, enc, packed, n, k, x, kind=None)
    check(auto, want)
    # and so does the wide (256 x 256) tile, which the launcher would only pick for weights of many rows
    try:
        hip_backend.set_tuning("gemm_wide", 1)
        wide = gpu_gemm(hip_backend, torch_cuda, enc, packed, n, k, x)
        assert not np.isnan(wide).any()
        check(wide, want)
        check_exact(torch_cuda, enc, wide, x, packed, n)
    finally:
        hip_backend.set_tuning("gemm_wide", -1)


@pytest.mark.parametrize("enc", ALL_ENCS)
def test_gemm_on_random_valid_blocks_and_forced_k_splits(hip_backend, torch_cuda, enc):
    bs = G.PACKED[enc][0]
    m, n, k = 40, 200, 2048
    packed = random_valid_blocks(enc, n * k // bs, 300)
    x = np.random.default_rng(5).standard_normal((m, k)).astype(np.float32)
    want = L.gemv(enc, x, packed, n)
    try:
        for rows in (2, 4):                      # 128 / 256 activation rows per tile (40 rows would pick 128 by itself)
            hip_backend.set_tuning("gemm_rows", rows)
            for wide in (0, 1):
                hip_backend.set_tuning("gemm_wide", wide)
                for ks in (1, 2, 3, 8):
                    hip_backend.set_tuning("gemm_ksplit", ks)
                    got = gpu_gemm(hip_backend, torch_cuda, enc, packed, n, k, x)
                    check(got, want)
                    check_exact(torch_cuda, enc, got, x, packed, n)
    finally:
        hip_backend.set_tuning("gemm_ksplit", 0)
        hip_backend.set_tuning("gemm_wide", -1)
        hip_backend.set_tuning("gemm_rows", 0)


@pytest.mark.parametrize("m,n,k", [(192, 192, 256), (193, 385, 512), (385, 191, 768), (255, 257, 1024)])
@pytest.mark.parametrize("enc", ALL_ENCS)
def test_gemm_tiles_of_192_rows_or_columns_give_the_bits_of_the_others(hip_backend, torch_cuda, enc, m, n, k):
    """An output is one chain of matrix instructions over K whatever tile it lies in, so every tile gives the same bits."""
    packed = gaussian_weight(hip_backend, enc, n, k, 900 + n)
    x = np.random.default_rng(m + n).standard_normal((m, k)).astype(np.float32)
    try:
        hip_backend.set_tuning("gemm_ksplit", 1)
        hip_backend.set_tuning("gemm_rows", 2)
        hip_backend.set_tuning("gemm_wide", 0)
        want = gpu_gemm(hip_backend, torch_cuda, enc, packed, n, k, x)
        check_exact(torch_cuda, enc, want, x, packed, n)
        for rows, wide, tile in ((3, 0, "3, 2"), (3, 2, "3, 3"), (3, 1, "3, 4"), (4, 2, "4, 3")):
            hip_backend.set_tuning("gemm_rows", rows)
            hip_backend.set_tuning("gemm_wide", wide)
            got = []
            ran = launches(torch_cuda, lambda: got.append(gpu_gemm(hip_backend, torch_cuda, enc, packed, n, k, x)))
            assert sum(f"{tile}, false>" in name for name, _, _ in ran if "dequant_gemm_kernel<" in name) == 1, (tile, ran)
            assert np.array_equal(got[0].view(np.uint32), want.view(np.uint32)), (rows, wide)
    finally:
        hip_backend.set_tuning("gemm_ksplit", 0)
        hip_backend.set_tuning("gemm_wide", -1)
        hip_backend.set_tuning("gemm_rows", 0)


@pytest.mark.parametrize("m,n,k,kernel", [(300, 28672, 4096, "q4k_gemm_frag_kernel"), (300, 6144, 4096, "q4k_gemm_frag_kernel"),
                                          (528, 21086, 6656, "3, 4, false>"), (260, 5954, 13824, "3, 4, false>")])
def test_q4k_tiles_with_a_192_take_over_where_they_are_well_below(hip_backend, torch_cuda, m, n, k, kernel):
    """The fragment-order kernel keeps products on which the new tiles' estimate is less than 5 % below its own (the first is 2 % off, the
    second not below it): the choice changes the order of the sums. 23 and 15 % off, the tiles have them."""
    torch = torch_cuda
    gen = torch.Generator(device="cuda").manual_seed(n)
    packed = torch.randint(0, 120, (n * (k // 256) * 144,), generator=gen, dtype=torch.uint8, device="cuda")
    w = hip_backend.DeviceWeight.wrap("Q4_K", packed, n, k)
    x, got = torch.randn((m, k), generator=gen, device="cuda"), torch.empty((m, n), device="cuda")
    ran = launches(torch, lambda: w.matmul(x, m, got, 1))
    assert sum(kernel in name for name, _, _ in ran) == 1, ran


@pytest.mark.parametrize("m,n,k,ks", [(128, 128, 256, 1), (129, 131, 512, 1), (33, 257, 1024, 3), (300, 127, 2304, 2), (16, 16, 256, 1)])
@pytest.mark.parametrize("enc", ALL_ENCS)
def test_gemm_tile_on_fp32_rows_gives_the_bits_of_the_rounded_rows(hip_backend, torch_cuda, enc, m, n, k, ks):
    """The tile rounds the rows itself instead of a pass in front: the same values, so the same bits; also where the product lies over the
    rows, which then go through the pass."""
    torch = torch_cuda
    packed = gaussian_weight(hip_backend, enc, n, k, 700 + n)
    w = hip_backend.DeviceWeight.upload(enc, packed, n, k)
    x = torch.from_numpy(np.random.default_rng(m + k).standard_normal((m, k)).astype(np.float32)).cuda()
    got = {}

    def product(rows, out, f32):                               # the tile on fp32 rows alone, or behind the pass
        ran = [name for name, _, _ in launches(torch, lambda: w.matmul(rows, m, out, 1))]
        assert sum(f"2, 2, {str(f32).lower()}>" in name for name in ran if "dequant_gemm_kernel<" in name) == 1, ran
        assert any("prepass" in name for name in ran) != f32, ran
    try:
        for key, v in (("gemm_skinny", 0), ("gemm_frag", 0), ("gemm_ksw", 0), ("gemm_rows", 2), ("gemm_wide", 0), ("gemm_ksplit", ks)):
            hip_backend.set_tuning(key, v)
        for mode in (0, 2):
            hip_backend.set_tuning("gemm_f32", mode)
            both = torch.full((m * k + m * n,), float("nan"), device="cuda")
            xs, apart, over = both[:m * k].reshape(m, k).copy_(x), both[m * k:], both[:m * n]
            product(xs, apart, mode == 2)
            got[mode] = apart.clone()
            if n <= k:
                product(xs, over, False)
                assert torch.equal(over, got[mode])
    finally:
        for key, v in (("gemm_skinny", 1), ("gemm_frag", 1), ("gemm_ksw", 1), ("gemm_rows", 0), ("gemm_wide", -1), ("gemm_ksplit", 0), ("gemm_f32", 1)):
            hip_backend.set_tuning(key, v)
    assert not torch.isnan(got[0]).any() and torch.equal(got[0], got[2])
    check_exact(torch, enc, got[2].reshape(m, n).cpu().numpy(), x.cpu().numpy(), packed, n)


@pytest.mark.parametrize("enc,m,n,k,tile", [("Q6_K", 1000, 11008, 4096, "4, 3, false>"), ("Q5_K", 348, 1503, 2560, "2, 2, true>"), ("Q8_0", 400, 9000, 3072, "3, 2, false>")])
def test_gemm_tiles_that_the_rule_takes(hip_backend, torch_cuda, enc, m, n, k, tile):
    torch, (_, elems, size) = torch_cuda, hip_backend.ENCODINGS[enc]
    w = hip_backend.DeviceWeight.wrap(enc, torch.full((n * (k // elems) * size,), 17, dtype=torch.uint8, device="cuda"), n, k)
    x, out = torch.ones((m, k), device="cuda"), torch.empty((m, n), device="cuda")
    ran = launches(torch, lambda: w.matmul(x, m, out, 1))
    assert sum(tile in name for name, _, _ in ran if "dequant_gemm_kernel<" in name) == 1, ran


@pytest.mark.parametrize("k", [96, 192, 320, 448])
def test_gemm_q8_0_rows_that_are_not_whole_256_element_groups_fall_back_to_the_row_kernels(hip_backend, torch_cuda, k):
    """The tile kernel's K loop runs over whole 256-element groups; a Q8_0 row of 3, 6, 10 or 14 blocks takes the
    row kernels instead (exact fp32 products, so the one-row bound applies)."""
    m, n = 20, 50
    packed = gaussian_weight(hip_backend, "Q8_0", n, k, 7)
    x = np.random.default_rng(8).standard_normal((m, k)).astype(np.float32)
    got = gpu_gemm(hip_backend, torch_cuda, "Q8_0", packed, n, k, x)
    assert normalized_err(got, L.gemv("Q8_0", x, packed, n)) <= 1e-3


@pytest.mark.parametrize("enc,n,k", [("Q4_K", 4096, 4096), ("Q6_K", 32000, 4096), ("Q4_K", 14336, 4096), ("Q4_K", 4096, 14336)])
def test_gemm_at_config_sizes(hip_backend, torch_cuda, enc, n, k):
    """Prefill configuration: activations 512 x 4096 ~ N(0, 1). The oracle checks 6 sampled activation rows in full
    (each a scalar GEMV over the whole weight); linearity ties the rest of the batch to those rows."""
    m = 512
    packed = gaussian_weight(hip_backend, enc, n, k, 400)
    rng = np.random.default_rng(401)
    x = rng.standard_normal((m, k)).astype(np.float32)
    got = gpu_gemm(hip_backend, torch_cuda, enc, packed, n, k, x)
    rows = [0, 1, 255, 256, 300, 511]
    want = L.gemv(enc, x[rows], packed, n)
    err = check(got[rows], want)
    print(f"{enc} {m}x{n}x{k}: normalized max err {err:.2e}")
    check_exact(torch_cuda, enc, got[rows], x[rows], packed, n)
    # size-independent property over the whole batch: C is linear in A -- (P A) W^T == P (A W^T) for a mixing matrix P
    p = rng.standard_normal((8, m)).astype(np.float32) / np.sqrt(m)
    mixed = gpu_gemm(hip_backend, torch_cuda, enc, packed, n, k, (p.astype(np.float64) @ x).astype(np.float32))
    check(mixed, (p.astype(np.float64) @ got).astype(np.float32))
    # and the GEMM agrees with the fp32 row kernels on the same device
    few = gpu_gemm(hip_backend, torch_cuda, enc, packed, n, k, x[:4].copy(), kind=0)
    check(got[:4], few)


@pytest.mark.parametrize("m,n,k", [(512, 4096, 4096), (9, 64, 256), (130, 70, 512), (128, 129, 1024), (300, 1000, 2304), (40, 200, 14336),
                                   (257, 63, 768)])
def test_q4k_gemm_with_k_split_over_the_waves(hip_backend, torch_cuda, m, n, k):
    """The Q4_K kernel that gives every wave the whole 128 x 64 tile and a share of K, forced on shapes with ragged row
    and column tiles, one and many super-blocks per row, and the shape the launcher picks it for by itself; against the
    oracle (2e-2) and against the same product with both operands rounded to bf16 first (2e-4)."""
    packed = gaussian_weight(hip_backend, "Q4_K", n, k, 900 + n)
    x = np.random.default_rng(m * 7 + k).standard_normal((m, k)).astype(np.float32)
    want = L.gemv("Q4_K", x, packed, n)
    try:
        hip_backend.set_tuning("gemm_ksw", 2)
        got = gpu_gemm(hip_backend, torch_cuda, "Q4_K", packed, n, k, x)
        assert hip_backend.last_kernel() == "q4k_gemm_ksw_kernel"
        assert not np.isnan(got).any()
        check(got, want)
        check_exact(torch_cuda, "Q4_K", got, x, packed, n)
        # one team of four waves per workgroup instead of two (each team takes half of K where the super-blocks split
        # evenly), with the fewest and the most activation stages in LDS: same operands, another fp32 summation order
        for stages in (3, 7):
            hip_backend.set_tuning("gemm_ksw_teams", 1)
            hip_backend.set_tuning("gemm_ksw_stages", stages)
            one_team = gpu_gemm(hip_backend, torch_cuda, "Q4_K", packed, n, k, x)
            assert hip_backend.last_kernel() == "q4k_gemm_ksw_kernel"
            assert normalized_err(got, one_team) <= 1e-4
        hip_backend.set_tuning("gemm_ksw", 0)
        tiles = gpu_gemm(hip_backend, torch_cuda, "Q4_K", packed, n, k, x)
        assert hip_backend.last_kernel() == "dequant_gemm_kernel"
        assert normalized_err(got, tiles) <= 1e-4          # same operands, another fp32 summation order
    finally:
        hip_backend.set_tuning("gemm_ksw", 1)
        hip_backend.set_tuning("gemm_ksw_teams", 2)
        hip_backend.set_tuning("gemm_ksw_stages", 5)


@pytest.mark.parametrize("m,n,k", [(512, 4096, 4096), (9, 64, 256), (130, 70, 512), (128, 129, 1024), (300, 1000, 2304), (40, 200, 14336),
                                   (257, 63, 768), (64, 512, 11008), (384, 1024, 4096)])
def test_q4k_gemm_with_activations_in_fragment_order(hip_backend, torch_cuda, m, n, k):
    """The Q4_K kernel whose activations are laid out by the pass in front in the order the matrix instruction reads them
    (every wave: the whole 128 x 64 tile and whole super-blocks of K), in both of its forms (eight waves per workgroup,
    and four with two workgroups per CU), forced on shapes with ragged row and column tiles,
    fewer super-blocks than waves, uneven super-block counts per wave (43 and 56 super-blocks over 8 waves), tile counts
    that are and are not a multiple of the eight dies; against the oracle (2e-2), against the same product with both
    operands rounded to bf16 first (2e-4), and against the tile kernel."""
    packed = gaussian_weight(hip_backend, "Q4_K", n, k, 900 + n)
    x = np.random.default_rng(m * 7 + k).standard_normal((m, k)).astype(np.float32)
    want = L.gemv("Q4_K", x, packed, n)
    try:
        hip_backend.set_tuning("gemm_frag", 2)
        for waves in (8, 4):                       # one workgroup of eight waves per CU, or two of four
            hip_backend.set_tuning("gemm_frag_waves", waves)
            got = gpu_gemm(hip_backend, torch_cuda, "Q4_K", packed, n, k, x)
            assert hip_backend.last_kernel() == "q4k_gemm_frag_kernel"
            assert not np.isnan(got).any()
            check(got, want)
            check_exact(torch_cuda, "Q4_K", got, x, packed, n)
        hip_backend.set_tuning("gemm_frag", 0)
        hip_backend.set_tuning("gemm_ksw", 0)
        tiles = gpu_gemm(hip_backend, torch_cuda, "Q4_K", packed, n, k, x)
        assert hip_backend.last_kernel() == "dequant_gemm_kernel"
        assert normalized_err(got, tiles) <= 1e-4          # same operands, another fp32 summation order
    finally:
        hip_backend.set_tuning("gemm_frag", 1)
        hip_backend.set_tuning("gemm_frag_waves", 0)
        hip_backend.set_tuning("gemm_ksw", 1)
    if (m, n, k) == (512, 4096, 4096):
        gpu_gemm(hip_backend, torch_cuda, "Q4_K", packed, n, k, x)
        assert hip_backend.last_kernel() == "q4k_gemm_frag_kernel"     # the launcher's own choice for this shape


@pytest.mark.parametrize("enc", ALL_ENCS)
@pytest.mark.parametrize("m,n,k", [(9, 5, 256), (16, 16, 2048), (17, 33, 2304), (33, 130, 768), (64, 31, 4352), (100, 70, 512), (150, 40, 256)])
def test_gemm_of_few_rows(hip_backend, torch_cuda, enc, m, n, k):
    """The kernel whose lanes decode their own operands, forced at each of its tiles (1, 2 or 4 row tiles x 1 or 2 column
    tiles of 16) on ragged rows and columns, fewer super-blocks than waves and uneven counts per wave (1, 2, 8, 9, 17 over
    8 waves), Q6_K rows that start on odd half words; against the oracle (2e-2) and the product of bf16-rounded operands
    (2e-4); with RMSNorm, residual and SwiGLU against the same product finished in float64."""
    torch, kx = torch_cuda, hip_backend
    packed = gaussian_weight(kx, enc, n, k, 700 + n)
    rng = np.random.default_rng(m + n + k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    want = L.gemv(enc, x, packed, n)
    gain, res = (1 + 0.2 * rng.standard_normal(k)).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    try:
        for tile in (2, 11, 12, 21, 22, 41, 42):
            kx.set_tuning("gemm_skinny", tile)
            got = gpu_gemm(kx, torch, enc, packed, n, k, x)
            assert kx.last_kernel() == "packed_gemm_skinny_kernel"
            check(got, want)
            check_exact(torch, enc, got, x, packed, n)
        w = kx.DeviceWeight.upload(enc, packed, n, k)
        xn = (x.astype(np.float64) / np.sqrt((x.astype(np.float64) ** 2).mean(1, keepdims=True) + 1e-5) * gain).astype(np.float32)
        p = bf16_round(torch, xn) @ bf16_round(torch, L.dequant(enc, packed).reshape(n, -1)).T
        out = torch.full((m, n), float("nan"), device="cuda")
        w.matmul_fused(dev(torch, x), m, out, gain=dev(torch, gain), eps=1e-5, residual=dev(torch, res), epilogue=kx.EPI_RESIDUAL)
        # a normalised activation that two fp32 evaluations round to neighbouring bf16 values moves one product by 2^-8 of it,
        # at most 2^-8 * 4.5 * 0.08 = 1.4e-3 for these operands, against a largest output above 1
        assert normalized_err(out.cpu().numpy(), p + res, eps=1.0) <= 2e-3
        if n % 2 == 0:
            half = torch.full((m, n // 2), float("nan"), device="cuda")
            w.matmul_fused(dev(torch, x), m, half, gain=dev(torch, gain), eps=1e-5, epilogue=kx.EPI_SWIGLU)
            assert normalized_err(half.cpu().numpy(), p[:, 0::2] / (1 + np.exp(-p[:, 0::2])) * p[:, 1::2], eps=1.0) <= 4e-3
    finally:
        kx.set_tuning("gemm_skinny", 1)


@pytest.mark.parametrize("enc", ALL_ENCS)
@pytest.mark.parametrize("m,n,k", [(9, 5, 256), (16, 64, 2048), (17, 65, 512), (33, 130, 768), (40, 129, 4352), (150, 40, 1280)])
def test_gemm_of_few_rows_in_one_launch(hip_backend, torch_cuda, enc, m, n, k):
    """The forms that read their fp32 rows themselves, forced at each tile: ragged rows, columns and rounds, waves without a
    super-block, Q6_K rows on odd half words. `direct` has the tiles, operands and sums of the two-launch kernel: the same bits.
    `shared` sums K in two shares instead of eight: the product of bf16-rounded operands (2e-4). With a residual, and with an output
    that overlaps the rows, which is two launches again."""
    torch, kx = torch_cuda, hip_backend
    packed = gaussian_weight(kx, enc, n, k, 900 + n)
    rng = np.random.default_rng(m * n + k)
    x, res = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    w = kx.DeviceWeight.upload(enc, packed, n, k)
    try:
        for tile in (111, 112, 411, 422):
            kx.set_tuning("gemm_skinny", tile)
            got = gpu_gemm(kx, torch, enc, packed, n, k, x)
            assert kx.last_kernel() == ("packed_gemm_skinny_shared_kernel" if tile > 400 else "packed_gemm_skinny_direct_kernel")
            check_exact(torch, enc, got, x, packed, n)
            out = torch.full((m, n), float("nan"), device="cuda")
            w.matmul_fused(dev(torch, x), m, out, residual=dev(torch, res), epilogue=kx.EPI_RESIDUAL)
            assert np.array_equal(out.cpu().numpy(), got + res)
            if tile < 400:
                kx.set_tuning("gemm_skinny", tile - 100)
                assert np.array_equal(gpu_gemm(kx, torch, enc, packed, n, k, x), got)
        kx.set_tuning("gemm_skinny", 111)
        buf = torch.zeros(m * max(n, k), device="cuda")
        buf[:m * k] = dev(torch, x).reshape(-1)
        w.matmul(buf, m, buf)
        assert kx.last_kernel() == "packed_gemm_skinny_kernel"
        check_exact(torch, enc, buf[:m * n].cpu().numpy().reshape(m, n), x, packed, n)
    finally:
        kx.set_tuning("gemm_skinny", 1)


@pytest.mark.parametrize("enc,m,n,k,kernel", [("Q4_0", 18, 924, 1024, "direct"), ("Q5_K", 91, 8978, 512, "shared"), ("Q8_0", 24, 4096, 4096, "kernel"),
                                              ("Q4_0", 46, 1086, 9984, "kernel"), ("Q8_0", 100, 7267, 1024, "kernel"), ("Q4_K", 95, 668, 5888, "kernel")])
def test_small_products_of_few_rows_take_one_launch(hip_backend, torch_cuda, enc, m, n, k, kernel):
    packed = gaussian_weight(hip_backend, enc, n, k, 31)
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    got = []
    ran = launches(torch_cuda, lambda: got.append(gpu_gemm(hip_backend, torch_cuda, enc, packed, n, k, x)))
    ours = [name for name, _, _ in ran if "skinny" in name]
    assert len(ours) == (2 if kernel == "kernel" else 1) and f"packed_gemm_skinny_{kernel}" in ours[-1], ran
    check_exact(torch_cuda, enc, got[0], x, packed, n)


def test_the_few_rows_key_takes_what_names_a_form(hip_backend, torch_cuda):
    """2 to 10: wherever it fits; a value that names no form leaves the key as it is; the one-launch forms have a key of their own."""
    def ran(enc, m, n, k):
        gpu_gemm(hip_backend, torch_cuda, enc, gaussian_weight(hip_backend, enc, n, k, 31), n, k, np.ones((m, k), np.float32))
        return hip_backend.last_kernel()
    big, small = ("Q6_K", 1000, 2048, 1024), ("Q4_0", 18, 924, 1024)
    try:
        for value, kernel in ((1, "dequant_gemm_kernel"), (121, "dequant_gemm_kernel"), (13, "dequant_gemm_kernel"), (412, "dequant_gemm_kernel"),
                              (3, "packed_gemm_skinny_kernel"), (13, "packed_gemm_skinny_kernel"), (422, "packed_gemm_skinny_shared_kernel"), (0, "dequant_gemm_kernel")):
            hip_backend.set_tuning("gemm_skinny", value)
            assert ran(*big) == kernel, value
        hip_backend.set_tuning("gemm_skinny", 1)
        for value, kernel in ((0, "packed_gemm_skinny_kernel"), (1, "packed_gemm_skinny_direct_kernel")):
            hip_backend.set_tuning("gemm_skinny_direct", value)
            assert ran(*small) == kernel
    finally:
        hip_backend.set_tuning("gemm_skinny", 1)
        hip_backend.set_tuning("gemm_skinny_direct", 1)


@pytest.mark.parametrize("knob", ["gemm_frag", "gemm_ksw"])
def test_the_q4k_gemm_knobs_leave_other_formats_alone(hip_backend, torch_cuda, knob):
    """Either Q4_K kernel switched off: a product of few rows in another format takes the kernel it takes by rule, Q4_K one
    of those before the switched-off one."""
    m, n, k = 24, 4096, 4096
    x = np.random.default_rng(24).standard_normal((m, k)).astype(np.float32)
    try:
        hip_backend.set_tuning(knob, 0)
        for enc in ALL_ENCS:
            packed = gaussian_weight(hip_backend, enc, n, k, 24)
            got = gpu_gemm(hip_backend, torch_cuda, enc, packed, n, k, x)
            assert (hip_backend.last_kernel() == "packed_gemm_skinny_kernel") == (enc != "Q4_K")
            check(got[:2], L.gemv(enc, x[:2], packed, n))
    finally:
        hip_backend.set_tuning(knob, 1)


@pytest.mark.parametrize("enc,m,n,k", [("Q8_0", 129, 907, 13312), ("Q6_K", 229, 581, 14336), ("Q4_0", 256, 700, 9472), ("Q8_0", 250, 513, 13312), ("Q5_K", 385, 513, 14336)])
def test_gemm_of_few_tiles_with_more_than_eight_splits(hip_backend, torch_cuda, enc, m, n, k):
    """Few tiles over a long K: 9 to 24 splits, the last of them shorter than the rest or none at all, summed in split order."""
    packed = gaussian_weight(hip_backend, enc, n, k, 210 + n)
    x = np.random.default_rng(m + k).standard_normal((m, k)).astype(np.float32)
    try:
        hip_backend.set_tuning("gemm_skinny", 0)
        got = []
        ran = launches(torch_cuda, lambda: got.append(gpu_gemm(hip_backend, torch_cuda, enc, packed, n, k, x)))
    finally:
        hip_backend.set_tuning("gemm_skinny", 1)
    assert hip_backend.last_kernel() == "dequant_gemm_kernel"
    splits = [grid[2] for name, grid, _ in ran if "dequant_gemm_kernel<" in name]
    assert len(splits) == 1 and 9 <= splits[0] <= 24, ran
    assert not np.isnan(got[0]).any()
    check_exact(torch_cuda, enc, got[0], x, packed, n)
