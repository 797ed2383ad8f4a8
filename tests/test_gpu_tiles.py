"""Every 16-bit Primitive at the edges of its tiles, stages and store widths.

Integer inputs, so every product and partial sum is exact in fp32 (k * 16 < 2^24) and d must be the
exact result bit for bit: for a 16-bit d, its rounding to nearest even.  Operands lie in storages
padded with NaN, so a read past a row that feeds a result fails the comparison, and d in one filled
with a marker, so a store outside the matrix does too.
"""

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
MARK = 77.0


@pytest.fixture(scope="module")
def capi():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a visible device")
    from flash_train import capi as c

    return c


@pytest.fixture(scope="module")
def ops(capi):
    return capi.GemmOps()


def store(rows, cols, col_major, dtype, pad, shift, fill):
    """A rows x cols view, row- or column-major, `shift` elements into a storage with `pad` spare
    elements per leading dimension."""
    r, c = (cols, rows) if col_major else (rows, cols)
    whole = torch.full((r * (c + pad) + shift,), fill, dtype=dtype, device="cuda")
    view = whole[shift:].view(r, c + pad)[:, :c]
    return (view.t() if col_major else view), whole


def check(capi, ops, kind, cd, m, n, k, ta, tb, with_c, ab_pad=0, ab_shift=0, cd_pad=0, cd_shift=0, only=None):
    dtype, out = DT[kind], DT[cd]
    gen = torch.Generator(device="cuda").manual_seed(m * 7 + n * 5 + k)

    def ints(rows, cols):
        return torch.randint(-4, 5, (rows, cols), generator=gen, device="cuda")

    ai, bi, ci = ints(m, k), ints(k, n), ints(m, n)
    a, _ = store(m, k, ta, dtype, ab_pad, ab_shift, float("nan"))
    b, _ = store(k, n, tb, dtype, ab_pad, ab_shift, float("nan"))
    c, _ = store(m, n, False, out, cd_pad, cd_shift, float("nan"))
    d, whole = store(m, n, False, out, cd_pad, cd_shift, MARK)
    a.copy_(ai), b.copy_(bi), c.copy_(ci)
    want = 0.5 * (ai.double() @ bi.double()) + (2.0 * ci.double() if with_c else 0.0)
    want = want.float().to(out)
    outside = torch.ones_like(whole, dtype=torch.bool)
    outside[cd_shift:].view(m, n + cd_pad)[:, :n] = False
    plan = capi.plan_for(a, b, c if with_c else None, d, 0.5, 2.0, ops)
    names = plan.names()
    for i, name in enumerate(names):
        if only is not None and only not in name:
            continue
        d.fill_(float("nan"))
        plan.execute(i, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        where = f"{name} {kind} {cd} {m}x{n}x{k} ta={ta} tb={tb} c={with_c} pads {ab_pad} {ab_shift} {cd_pad} {cd_shift}"
        assert torch.equal(d, want), f"{where}: {int((d != want).sum())} wrong"
        assert bool((whole[outside] == MARK).all()), f"{where}: stored outside d"
    return names


# One, two, three and more stages of 64 k with and without a tail; one tile, a tile less and more a
# row, several tiles; c and d in 16-byte units, and not (odd leading dimension, unaligned base).
@pytest.mark.parametrize("kind,cd", [("bf16", "bf16"), ("bf16", "fp32"), ("fp16", "fp16")])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_half_tile_edges(capi, ops, kind, cd, ta, tb):
    for m, n, k in ((256, 256, 64), (248, 264, 128), (264, 248, 136), (512, 520, 328), (8, 520, 40), (136, 136, 704)):
        for with_c, pad, shift in ((False, 0, 0), (True, 0, 0), (True, 8, 8), (True, 3, 1), (False, 4, 4)):
            check(capi, ops, kind, cd, m, n, k, ta, tb, with_c, cd_pad=pad, cd_shift=shift)
    if not ta:  # rows free
        check(capi, ops, kind, cd, 255, 264, 200, ta, tb, True)
        check(capi, ops, kind, cd, 1, 264, 72, ta, tb, True)
    if tb:  # columns free
        check(capi, ops, kind, cd, 256, 255, 200, ta, tb, True)
        check(capi, ops, kind, cd, 264, 130, 1032, ta, tb, True)


def us_of(run, reps=20, rounds=5):
    """Median microseconds of a launch among others."""
    start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    got = []
    for _ in range(rounds + 1):
        start.record()
        for _ in range(reps):
            run()
        stop.record()
        torch.cuda.synchronize()
        got.append(start.elapsed_time(stop) / reps * 1e3)
    return sorted(got[1:])[rounds // 2]


def tile_us(capi, ops, name, dtype, out, m, n, k, tb, with_c):
    a = torch.zeros(m, k, dtype=dtype, device="cuda")
    b = torch.zeros(n, k, dtype=dtype, device="cuda").t() if tb else torch.zeros(k, n, dtype=dtype, device="cuda")
    c = torch.zeros(m, n, dtype=out, device="cuda") if with_c else None
    d = torch.empty(m, n, dtype=out, device="cuda")
    plan = capi.plan_for(a, b, c, d, 1.0, 0.5 if with_c else 0.0, ops)
    i = plan.names().index(name)
    return us_of(lambda: plan.execute(i, torch.cuda.current_stream().cuda_stream))


# Rows of d that start on odd 2-byte addresses: a tile's stores stay whole rows.  The two launches differ by
# the 5 columns (under 1%); stores of single elements took 2.6 times as long.
@pytest.mark.parametrize("with_c", [False, True])
def test_half_256_tile_cost_of_unaligned_rows(capi, ops, with_c):
    odd, even = (tile_us(capi, ops, "Fp16MfmaGemm_256x256_Dma", torch.float16, torch.float16, 4096, n, 1024, True, with_c)
                 for n in (2811, 2816))
    assert odd < 1.6 * even, (odd, even)


def test_half_256_tile_in_place(capi, ops):
    # c and d one matrix, rows on odd addresses and a last tile of 1 to 7 columns past a multiple of 8.
    for n, out in ((257, torch.float32), (262, torch.bfloat16), (519, torch.bfloat16)):
        a = torch.randint(-4, 5, (300, 136), device="cuda").bfloat16()
        b = torch.randint(-4, 5, (n, 136), device="cuda").bfloat16().t()
        c = torch.randint(-4, 5, (300, n), device="cuda").to(out)
        want = (0.5 * (a.double() @ b.double()) + 2.0 * c.double()).float().to(out)
        d = c.clone()
        plan = capi.plan_for(a, b, d, d, 0.5, 2.0, ops)
        i = plan.names().index("Bf16MfmaGemm_256x256_Dma")
        plan.execute(i, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(d, want), (n, out)


# Launches of at most one workgroup per CU (three stage buffers) and of more, 1 to 7 stages, whole-k.
@pytest.mark.parametrize("m,n", [(128, 128), (2048, 2048), (2048, 2176)])
def test_half_128_tile_stage_counts(capi, ops, m, n):
    for k in (40, 64, 128, 192, 200, 256, 320, 384, 456):
        names = check(capi, ops, "bf16", "fp32", m, n, k, False, True, False, only="128x128_Dma")
        assert "Bf16MfmaGemm_128x128_Dma" in names, names


# fp32 without 16-byte alignment: rows, columns and depths of every remainder by 4, one to several
# stages of 32 k, tile edges crossed by 1, 2 and 3 columns, unaligned bases and leading dimensions.
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("m,n,k", [(127, 97, 33), (128, 129, 31), (65, 130, 1), (129, 131, 64), (64, 4, 101), (3, 5, 7),
                                   (200, 255, 130), (257, 385, 1027), (64, 128, 2050)])
def test_fp32_unaligned_tiles(capi, ops, tb, m, n, k):
    for with_c, ab_pad, ab_shift, cd_pad, cd_shift in ((False, 0, 0, 0, 0), (True, 0, 0, 0, 0), (True, 1, 1, 3, 2),
                                                       (True, 4, 1, 0, 1), (False, 2, 3, 5, 3)):
        names = check(capi, ops, "fp32", "fp32", m, n, k, False, tb, with_c, ab_pad, ab_shift, cd_pad, cd_shift)
        assert "Fp32Mfma16Gemm_128x128_Dma_Unaligned" in names, names


def test_fp32_unaligned_in_place(capi, ops):
    # c and d one matrix, a last column tile of 1, 2 and 3 columns: every element read before it is written once.
    for n in (129, 130, 131):
        a = torch.randint(-4, 5, (200, 70), device="cuda").float()
        b = torch.randint(-4, 5, (70, n), device="cuda").float()
        c = torch.randint(-4, 5, (200, n), device="cuda").float()
        want = (0.5 * (a.double() @ b.double()) + 2.0 * c.double()).float()
        d = c.clone()
        plan = capi.plan_for(a, b, d, d, 0.5, 2.0, ops)
        for i, name in enumerate(plan.names()):
            d.copy_(c)
            plan.execute(i, torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            assert torch.equal(d, want), (name, n)


# 16-bit rows that are not multiples of 8 elements: problems on the per-element 64x64 tile and, from
# 128 rows or columns of a transposed operand on, on its 128x128 form, whose last tile moves inside the
# matrix; k tails of 1 to 63, unaligned bases and leading dimensions.
@pytest.mark.parametrize("kind,cd", [("bf16", "fp32"), ("fp16", "fp16")])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_half_unaligned_tiles(capi, ops, kind, cd, ta, tb):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    large = {}
    for m, n, k in ((129, 131, 1281), (128, 128, 1283), (255, 257, 1151), (255, 257, 1215), (300, 129, 1407),
                    (131, 300, 1344), (65, 66, 100), (127, 127, 1300), (66, 500, 1357), (300, 129, 639), (131, 300, 641),
                    (1500, 1601, 385)):
        for with_c, ab_pad, ab_shift, cd_pad in ((True, 0, 0, 0), (False, 3, 1, 1), (True, 1, 5, 3)):
            names = check(capi, ops, kind, cd, m, n, k, ta, tb, with_c, ab_pad, ab_shift, cd_pad, 1 if cd_pad else 0,
                          only="Unaligned")
            assert any("64x64_Unaligned" in nm for nm in names), names
            large[m, n, k, with_c] = capi.testing_lib().ftrainTestingTakes128(m, n, k, ta, tb, with_c, cd != "fp32", cus)
    # The Primitive ran both of its tiles, the 128x128 one with moved last tiles and shifted k-tail chunks among them.
    assert all(large[m, n, k, with_c] for m, n, k in ((129, 131, 1281), (128, 128, 1283), (255, 257, 1215), (300, 129, 1407),
                                                      (131, 300, 1344)) for with_c in (False, True)), large
    assert not all(large.values()), large


def test_half_unaligned_in_place(capi, ops):
    # c and d one matrix: the outputs that a moved last tile shares with its neighbour are written once.
    a = torch.randint(-4, 5, (300, 1325), device="cuda").bfloat16()
    b = torch.randint(-4, 5, (1325, 301), device="cuda").bfloat16()
    c = torch.randint(-4, 5, (300, 301), device="cuda").float()
    want = (0.5 * (a.double() @ b.double()) + 2.0 * c.double()).float()
    d = c.clone()
    plan = capi.plan_for(a, b, d, d, 0.5, 2.0, ops)
    for i, name in enumerate(plan.names()):
        d.copy_(c)
        plan.execute(i, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(d, want), name


# The one-pass skinny kernel with a column-major b: every row count, columns across a workgroup's 32 and
# a wave's 4, depths with and without whole groups of its steps, padded strides.
@pytest.mark.parametrize("m", range(1, 9))
def test_fp32_gemv_column_major_b(capi, ops, m):
    for n, k in ((32, 256), (36, 1024), (4, 4), (100, 516), (200, 2052), (64, 4096), (1000, 3076), (8196, 516),
                 (8192, 2308)):
        for with_c, ab_pad, cd_pad in ((False, 0, 0), (True, 4, 8)):
            names = check(capi, ops, "fp32", "fp32", m, n, k, False, True, with_c, ab_pad, 0, cd_pad, 0, only="Fp32Gemv")
            assert ("Fp32Gemv" in names) == (m <= 2 or n >= 8192 or (m <= 4 and k <= 2048)), names
