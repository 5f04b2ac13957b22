"""How the products say they will be computed, for knobs of any value: whole-number answers, no device needed."""
import pytest


@pytest.fixture
def knobs(hip):
    """set(name, value), undone afterwards."""
    seen = set()

    def put(name, value):
        seen.add(name)
        hip.set_tunable(name, value)
    yield put
    for name in seen:
        hip.set_tunable(name, 0)


@pytest.mark.parametrize("value", [-1, 2, 3, 9, 10, 12, 16, 20, 28, 34, 48, 64, 99, 18 + 2 ** 32])
def test_f32_direct_knob_of_no_variant_counts_as_zero(hip, knobs, value):
    """gemm_f32.direct names a variant by its digits; a number that names none (2: no rows at all; 34, 64: rows the kernel
    has no form for, and fewer tickets than its tiles draw) leaves the choice to the library."""
    shapes = [(1, 1, 1), (128, 128, 128), (68, 119, 3328), (153, 1216, 1920), (4096, 2048, 512), (2049, 4097, 3000)]
    for split_k in (0, 2, 16):
        knobs("gemm_f32.split_k", split_k)
        knobs("gemm_f32.direct", 0)
        own = [hip.gemm_f32_k_splits(*s) for s in shapes]
        knobs("gemm_f32.direct", value)
        assert [hip.gemm_f32_k_splits(*s) for s in shapes] == own


@pytest.mark.parametrize("m,n,k,room", [(200, 200, 40, False), (100, 64, 32, False), (200, 200, 63, False), (8192, 4096, 4096, False),
                                         (300, 520, 448, True), (200, 200, 64, False), (200, 200, 127, False)])
@pytest.mark.parametrize("forced", [2, 7])
def test_16_bit_pieces_forced_where_there_is_no_room(hip, knobs, m, n, k, room, forced):
    """A forced count of K pieces is cut to whole stages of 64 and to planes that fit the workspace, and to no less than the
    one piece that says K stays whole."""
    knobs("gemm16.tile", 128)
    knobs("gemm16.split_k", forced)
    assert hip.gemm16_k_splits(m, n, k) == (forced if room else 1)


@pytest.mark.parametrize("m,n,k,kernel", [(64, 27136, 2432, 128), (64, 20992, 4160, 128), (51, 7969, 5857, 128), (64, 29028, 2725, 128),
                                          (64, 31360, 2624, 128), (256, 1280, 191, 128), (723, 1702, 256, 128),
                                          (16, 30000, 4096, 128), (16, 30016, 4096, 64), (16, 27136, 2432, 64), (16, 8192, 8192, 64), (32, 4096, 4096, 64), (48, 4096, 1024, 64),
                                          (64, 1001, 1001, 64), (64, 576, 1064, 64), (62, 23936, 1305, 128), (60, 20992, 2483, 128),
                                          (35, 27888, 858, 128), (38, 24064, 2749, 128), (77, 2332, 1920, 64), (130, 4608, 140, 64)])
def test_16_bit_products_of_few_rows_go_where_they_are_faster(hip, m, n, k, kernel):
    """The few-rows kernel (64) or the 128 x 128 tile, whichever was measured to be the faster at these sizes."""
    assert hip.gemm16_tile(m, n, k) == kernel


@pytest.mark.parametrize("m,n,k,pieces", [(1561, 1280, 8121, 3), (522, 2053, 4672, 3), (114, 5824, 2687, 4), (110, 2048, 192, 1),
                                          (4096, 2048, 1000, 1), (128, 30000, 6000, 1), (1920, 4000, 8192, 1)])
def test_pieces_of_k_on_the_small_tile(hip, knobs, m, n, k, pieces):
    """The count with the lowest estimate: workgroups that fit the CUs twice over, planes that fit the workspace, a stage of 64 each;
    where the tile is asked for by name, K is whole unless it is long against C."""
    knobs("gemm16.rows", 1)
    tiles, seen = -(-m // 128) * -(-n // 128), hip.gemm16_k_splits(m, n, k)
    assert seen == pieces
    for longer in (k, 2 * k, 3 * k + 1, 8 * k):
        s = hip.gemm16_k_splits(m, n, longer)
        assert s == 1 or (s <= 16 and tiles * s <= 512 and 4 * m * n * s <= 64 << 20 and longer // s >= 64)
    if hip.gemm16_tile(m, n, k) == 128:
        knobs("gemm16.tile", 128)
        assert hip.gemm16_k_splits(m, n, k) == (pieces if k >= 1500 + 640 * m * n * 4e-6 else 1)


@pytest.mark.parametrize("m,n,k,pieces", [(64, 64, 1536, 4), (256, 256, 8192, 16), (16, 8192, 8192, 8), (100, 256, 1536, 1), (130, 520, 1600, 1)])
def test_pieces_of_k_on_a_tile_asked_for_by_name(hip, knobs, m, n, k, pieces):
    """A K that is long against C is cut there too, into half as many pieces at least as when they were powers of two (a sum in chunks
    is the more exact by more than that)."""
    knobs("gemm16.tile", 128)
    assert (hip.gemm16_k_splits(m, n, k) == 1) == (pieces == 1) and 2 * hip.gemm16_k_splits(m, n, k) >= pieces


@pytest.mark.parametrize("m,n,k,columns", [
    (2048, 8448, 4096, 8192), (2048, 8448, 128, 8192), (2048, 8448, 127, 8448), (2048, 50257, 1024, 49152), (2048, 12288, 4096, 12288),
    (7232, 13568, 82, 13568), (7232, 13568, 767, 13568), (7232, 13568, 768, 52 * 256), (3712, 39176, 768, 39176),
    (4160, 8000, 126, 8000), (4160, 8000, 256, 30 * 256), (4096, 4097, 4096, 4096), (8192, 8192, 8192, 8192), (100, 1, 64, 0),
    (16, 8192, 8192, 8192)])
def test_columns_past_whole_rounds_of_large_tiles(hip, knobs, m, n, k, columns):
    """The cut wants K to be 128 times the whole rounds of workgroups; gemm16.cut = 1 never cuts, a count cuts whatever K."""
    assert hip.gemm16_tile_columns(m, n, k) == columns
    knobs("gemm16.cut", 1)
    assert hip.gemm16_tile_columns(m, n, k) == (n if n not in (1, 4097) else n - 1)
    if (m, n) in ((2048, 8448), (4160, 8000), (7232, 13568)):
        knobs("gemm16.cut", 256)
        assert hip.gemm16_tile_columns(m, n, k) < n


@pytest.mark.parametrize("m,n,k,rows", [
    (8192, 6401, 64, 1), (8192, 6400, 64, 1), (8192, 6399, 64, 0), (6400, 8192, 1024, 1), (8192, 8191, 4096, 1), (8192, 8191, 4097, 0), (8192, 8192, 4096, 0),
    (2048, 50257, 625, 1), (2048, 50257, 1024, 1), (2048, 50272, 625, 1), (2048, 50272, 626, 0), (2048, 50256, 1024, 1),
    (4096, 4096, 256, 0), (16, 8192, 8192, 0), (128, 128, 128, 0)])
def test_c_stored_by_rows(hip, knobs, m, n, k, rows):
    """A C of 200 MiB and more (8192 x 6400), up to a K of 4096, and not where its rows are whole lines and B has more than 60 MiB
    (50272 columns: from a K of 626 on); never and always where asked, on the 256 x 256 tile alone."""
    assert hip.gemm16_by_rows(m, n, k) == rows
    knobs("gemm16.by_rows", 1)
    assert hip.gemm16_by_rows(m, n, k) == 0
    knobs("gemm16.by_rows", 2)
    assert hip.gemm16_by_rows(m, n, k) == (hip.gemm16_tile(m, n, k) == 256)


@pytest.mark.parametrize("m,n,k,columns", [
    (4096, 2048, 8192, 2048), (1921, 4095, 1200, 4095), (1921, 4095, 1199, 0), (392, 12497, 4079, 12497), (3072, 3072, 3072, 0),
    (2048, 2048, 2048, 0), (1921, 4099, 1200, 0), (2048, 12288, 4096, 4096), (2048, 11264, 1199, 0), (2048, 11264, 1200, 3072),
    (2880, 13120, 1799, 0), (2880, 13120, 1800, 2368), (2048, 8448, 4096, 0), (1920, 4097, 2048, 4097), (16, 8192, 8192, 0), (100, 1, 64, 0)])
def test_columns_of_the_half_tile(hip, knobs, m, n, k, columns):
    """The 128 x 256 tile: whole products of at most one such tile to a CU, and the columns past whole rounds of large tiles, from a
    K of 600 for each round and one more on; K is never cut beside it, and asking for pieces of K goes before it."""
    assert hip.gemm16_half_columns(m, n, k) == columns
    if columns:
        assert hip.gemm16_k_splits(m, n, k) == 1
    knobs("gemm16.split_k", 1)
    assert hip.gemm16_half_columns(m, n, k) == columns
    knobs("gemm16.split_k", 2)
    assert hip.gemm16_half_columns(m, n, k) == 0
    knobs("gemm16.split_k", 0)
    knobs("gemm16.half", 1)
    assert hip.gemm16_half_columns(m, n, k) == 0


@pytest.mark.parametrize("m,n,k,columns", [(2048, 11264, 64, 3072), (2048, 8448, 64, 256), (2048, 12288, 256, 4096), (4160, 8000, 126, 320),
                                           (3072, 3072, 64, 0), (256, 256, 4096, 256)])
def test_half_tile_wherever_a_workgroup_per_cu_takes_the_columns(hip, knobs, m, n, k, columns):
    """gemm16.half = 2: whatever K, and however few 128 x 128 tiles the columns would be; not against a cut that was asked for."""
    knobs("gemm16.half", 2)
    if hip.gemm16_tile(m, n, k) == 256:
        assert hip.gemm16_half_columns(m, n, k) == columns
        knobs("gemm16.cut", 1)
        assert hip.gemm16_half_columns(m, n, k) == 0
    else:
        assert hip.gemm16_half_columns(m, n, k) == columns and hip.gemm16_k_splits(m, n, k) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("value", [2, 34])
def test_f32_direct_knob_of_no_variant_computes_the_same_product(hip, torch_cuda, knobs, value):
    """The same bits as with the knob at 0, K left whole and cut, where the direct kernel is the library's choice."""
    torch = torch_cuda
    torch.manual_seed(value)
    a, b = torch.randn(153, 1921, device="cuda"), torch.randn(1921, 1217, device="cuda")
    for split_k in (0, 3):
        knobs("gemm_f32.split_k", split_k)
        knobs("gemm_f32.direct", 0)
        c = hip.gemm_f32(a, b)
        knobs("gemm_f32.direct", value)
        assert torch.equal(hip.gemm_f32(a, b), c)
