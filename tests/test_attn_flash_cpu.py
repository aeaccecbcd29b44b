"""Which workgroups prompt attention takes (attn_flash.hip), from the sizes of a
step alone."""
import pytest

from bee2bee_amd import ops

pytestmark = pytest.mark.skipif(not ops.hip_available(),
                                reason="the extension is not built")


def _spread(n, longest):
    lo = max(1, longest // 8)
    return [longest - (longest - lo) * i // max(1, n - 1) for i in range(n)]


def _form(lens, nq, nkv, hd, page=0):
    return ops.require_hip().attn_flash_form(sum(lens), len(lens), nq, nkv, hd,
                                             max(lens), page)


@pytest.mark.parametrize("full,page,form", [
    (139, 256, 64), (140, 256, 257), (400, 64, 257), (139, 48, 64),
    (140, 48, 128), (300, 48, 128), (379, 16, 128), (380, 48, 256),
    (140, 96, 128)])
def test_turns_need_pages_of_whole_tiles(full, page, form):
    """The 256-row workgroups without turns are behind the 128-row ones up to
    350 (8000 cached 579 us and 545; 500 cached, 256: 90 and 78) and ahead at
    400 (605 and 655)."""
    assert _form([full * 8], 32, 8, 128, page) == form


# as measured: prompts of an eighth of the longest up to it, or of one length;
# the two shapes' times in us
@pytest.mark.parametrize("n,longest,nq,nkv,rows256,rows128", [
    (2, 1200, 32, 8, 31, 32), (3, 1090, 32, 8, 33, 31),
    (3, 2133, 24, 8, 76, 79), (4, 772, 28, 4, 26, 27),
    (4, 1218, 28, 4, 36, 41), (4, 1066, 32, 8, 50, 52),
    (9, 1580, 32, 8, 106, 99), (9, 2211, 32, 8, 170, 179),
    (9, 2528, 28, 4, 311, 285), (9, 3611, 28, 4, 590, 582),
    (9, 5056, 28, 4, 976, 1106), (9, 1106, 64, 8, 113, 107),
    (9, 2211, 64, 8, 346, 361), (30, 1327, 32, 8, 267, 263)])
def test_shapes_follow_what_was_measured(n, longest, nq, nkv, rows256, rows128):
    want = 257 if rows256 < rows128 else 128
    assert _form(_spread(n, longest), nq, nkv, 128) == want


@pytest.mark.parametrize("n,each,nq,nkv,rows256,rows128", [
    (2, 600, 32, 8, 21.7, 20.4), (2, 920, 32, 8, 29.3, 29.5),
    (4, 600, 32, 8, 25.9, 24.1), (4, 900, 32, 8, 41.6, 45.0),
    (9, 1422, 28, 4, 157.2, 161.9), (9, 711, 32, 8, 70.0, 64.8)])
def test_prompts_of_one_length(n, each, nq, nkv, rows256, rows128):
    want = 257 if rows256 < rows128 else 128
    assert _form([each] * n, nq, nkv, 128) == want


# us, row of tiles by row of tiles as the sequences stand / turned / by the number of
# keys; of prompts of an eighth of the longest up to it
@pytest.mark.parametrize("n,longest,nq,nkv,straight,turned,keys", [
    (2, 2500, 32, 8, 94.9, 67.7, 67.4), (4, 2500, 32, 8, 175, 106, 99),
    (6, 2500, 32, 8, 157, 149, 144), (8, 1000, 32, 8, 60.0, 46.6, 48.3),
    (12, 1600, 32, 8, 164, 140, 143), (9, 1600, 28, 4, 93, 137, 96),
    (7, 700, 28, 4, 27.3, 25.2, 26.0), (7, 2500, 12, 12, 71.6, 59.1, 57.6),
    (4, 64, 32, 8, 6.1, 6.2, 6.6), (2, 64, 12, 12, 4.5, 4.5, 4.8)])
def test_orders_follow_what_was_measured(n, longest, nq, nkv, straight, turned,
                                         keys):
    """The fastest, or within 4% of it."""
    order = ops.require_hip().attn_flash_order(
        sum(_spread(n, longest)), n, nq, nkv, longest, False)
    took = (straight, turned, turned, keys)[order]
    assert took <= 1.04 * min(straight, turned, keys)


def test_only_few_large_and_uneven_steps_search():
    """A workgroup's search costs 0.3 to 1 us."""
    order = ops.require_hip().attn_flash_order
    for n, each, pages in ((1, 4000, False), (2, 2000, False), (4, 1000, False),
                           (3, 20, True), (8, 64, True), (9, 1000, True)):
        assert order(n * each, n, 32, 8, each, pages) != 3
    assert order(4 * 1000, 4, 32, 8, 1000, True) == 3    # (histories may differ)
