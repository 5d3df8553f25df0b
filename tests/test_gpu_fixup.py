"""The fix-up's tile counts: how many tiles a thread of ``fixup_kernel`` takes and how many blocks run follow from the
number of tiles of a launch.  Integer sums have one right answer, so every launch is compared exactly with torch's
``index_add_`` on the same data."""
import ctypes

import pytest

torch = pytest.importorskip("torch")

from flexspmv_amd.binding import DTYPE_CODES, load_named

pytestmark = pytest.mark.gpu

# one tile and two (one block folds and adds up); blocks of 256 tiles that fold carries beside the block that adds up,
# four to eight of them; blocks of 1 024 tiles; the most tiles of that shape and one more (17 blocks of 512
# tiles then, the last ticket adds their aggregator sums)
TILES = (1, 2, 1023, 1024, 1025, 2048, 2049, 4097, 8192, 8193, 12_300)


def tiles_of(ext, num_rows, ne):
    out = (ctypes.c_int32 * 6)()
    assert ext._lib.flexspmv_tiling(DTYPE_CODES["int64"], num_rows, ne, out) == 0
    return out[0]


def row_lengths(n):
    """Rows of four edges; now and then one that no tile boundary can step over (it carries), and one of several tiles."""
    length = torch.full((n,), 4, dtype=torch.int64, device="cuda")
    length[777::9_001] = 190
    length[30_000::70_001] = 9_000
    return length


@pytest.mark.parametrize("tiles", TILES)
def test_integer_sums_at_every_fixup_shape(tiles):
    ext = load_named("index_spmv", build_if_missing=False)
    ends = torch.cumsum(row_lengths(6_000_000), 0).cpu()
    lo, hi = 1, ends.numel()
    while lo < hi:                      # the fewest rows that make at least this many tiles
        mid = (lo + hi) // 2
        lo, hi = (lo, mid) if tiles_of(ext, mid, int(ends[mid - 1])) >= tiles else (mid + 1, hi)
    n, ne = lo, int(ends[lo - 1])
    print(f"case fixup {tiles}: {tiles_of(ext, n, ne)} tiles, {n} rows, {ne} edges", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(tiles)
    ptr = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
    ptr[1:] = ends[:n].cuda()
    w = torch.randint(-1000, 1000, (ne,), generator=gen, device="cuda")
    ids = torch.randint(-1000, 1000, (n,), generator=gen, device="cuda")
    col = torch.randint(0, n, (ne,), generator=gen, device="cuda", dtype=torch.int32)
    want = w * ids[col.long()]
    rows = torch.repeat_interleave(torch.arange(n, device="cuda"), row_lengths(6_000_000)[:n], output_size=ne)
    want_y = torch.zeros(n, dtype=torch.int64, device="cuda").index_add_(0, rows, want)
    for _ in range(3):                  # boundaries searched, then confirmed
        y, total = ext.merged_spmv_launch(w, ids, col, ptr, n, n)
        assert torch.equal(y, want_y)
        assert int(total) == int(want.sum())


# Without an aggregator: the reducer's last block up to 128 tiles, blocks of 256 tiles from there on
@pytest.mark.parametrize("tiles", (1, 2, 127, 128, 129, 256, 257, 513, 1024, 1025, 4097))
def test_carries_without_an_aggregator(tiles):
    ext = load_named("csr_spmv", build_if_missing=False)
    out = (ctypes.c_int32 * 6)()
    length = torch.full((max(2, tiles * 41),), 50, dtype=torch.int64)     # hardly a tile starts on a row of 50 entries
    length[tiles // 2] = 20 * 2048 if tiles > 30 else 50                  # ... and a row of 20 tiles
    ends = torch.cumsum(length, 0)
    lo, hi = 1, ends.numel()
    while lo < hi:                      # the fewest rows that make at least this many tiles
        mid = (lo + hi) // 2
        assert ext._lib.flexspmv_tiling(DTYPE_CODES["float32"], mid, int(ends[mid - 1]), out) == 0
        lo, hi = (lo, mid) if out[0] >= tiles else (mid + 1, hi)
    n, ne = lo, int(ends[lo - 1])
    print(f"case carries {tiles} tiles {n} rows {ne} edges", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(tiles)
    ptr = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
    ptr[1:] = ends[:n].cuda()
    col = torch.randint(0, n, (ne,), generator=gen, device="cuda", dtype=torch.int32)
    rows = torch.repeat_interleave(torch.arange(n), length[:n]).cuda()
    for dtype, top in ((torch.float32, 8), (torch.float64, 1 << 20)):
        # whole numbers whose sums the type holds exactly: one right answer in every order
        a = torch.randint(-top, top, (ne,), generator=gen, device="cuda").to(dtype)
        x = torch.randint(-top, top, (n,), generator=gen, device="cuda").to(dtype)
        (y,) = ext.merged_spmv_launch(a, x, col, ptr, n, n)
        (again,) = ext._launch_checked((a, x, col, ptr, n, n), {})
        want = torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, rows, a.double() * x.double()[col.long()])
        assert torch.equal(y.double(), want) and torch.equal(again, y)


# With an aggregator: the reducer's last block up to 256 tiles of 8-byte values, then blocks that fold beside one that adds
@pytest.mark.parametrize("tiles", (255, 256, 257, 511, 512, 513, 767))
def test_integer_sums_around_the_smallest_launches(tiles):
    test_integer_sums_at_every_fixup_shape(tiles)
