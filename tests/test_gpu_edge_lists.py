"""Edge-list sort at every number of bits per digit."""
import pytest

torch = pytest.importorskip("torch")

from flexspmv_amd import formats

pytestmark = pytest.mark.gpu


# digits of 5, 6, 6+6, 7, 7+6, 8, 8+7+7 and 8+8+8 bits; lists in tiles of 4 096 pairs (up to 64 of them
# without a scan kernel) and of 16 384
@pytest.mark.parametrize("ids", ["int32", "int64"])
@pytest.mark.parametrize("rows", [32, 64, 4_096, 128, 8_192, 256, 3_000_017, 1 << 24])
@pytest.mark.parametrize("n", [1, 40_961, 64 * 4_096, 64 * 4_096 + 1, (16 << 20) + 3])
def test_sort_at_every_digit_width(n, rows, ids):
    print(f"case sort {n} {rows} {ids}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n + rows)
    row = torch.randint(0, rows, (n,), generator=gen, device="cuda", dtype=getattr(torch, ids))
    got, perm = formats.sort_edges_by_row(row, rows)
    want, order = torch.sort(row, stable=True)
    assert torch.equal(got.to(row.dtype), want)
    assert torch.equal(perm.long(), order)
