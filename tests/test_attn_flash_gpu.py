"""The prompt-attention kernel (attn_flash.hip) at the edges of its tiles and
of its three workgroup shapes, against the fp32 reference.

Tolerance: a weight and an output element are rounded to bf16 once each (2^-8
relative at most), so an element is off by less than 2^-7 of the largest
value; half of that is asked for, since the weights' roundings do not all add
up. fp32 sums and exp2 add far less."""
import pytest
import torch

from bee2bee_amd import ops
from bee2bee_amd.ops import reference

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("needs a GPU", allow_module_level=True)

DEV = "cuda"


def _qkv(T, nq, nkv, hd, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    qkv = torch.randn(T, (nq + 2 * nkv) * hd, generator=g,
                      device=DEV).bfloat16()
    q, k, v = qkv.split([nq * hd, nkv * hd, nkv * hd], -1)
    return q.view(T, nq, hd), k.view(T, nkv, hd), v.view(T, nkv, hd)


def _cu(lens):
    return torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(),
                        dtype=torch.int32, device=DEV)


def _check(got, want, v):
    assert torch.isfinite(got).all()
    err = (got.float() - want.float()).abs().max().item()
    assert err <= v.float().abs().max().item() * 2 ** -8, err


@pytest.mark.parametrize("nq,nkv,hd,lens", [
    (4, 4, 64, [1]), (4, 1, 128, [1, 63, 64, 65]), (7, 1, 128, [9, 10, 37]),
    (32, 8, 64, [57, 0, 129]), (12, 12, 64, [31, 32, 33, 127, 128, 129]),
    (24, 8, 128, [255, 256, 257]), (16, 1, 64, [2, 100]),
    # 128- and 256-row workgroups
    (28, 4, 128, [700, 513, 64, 300]), (32, 8, 128, [512] * 7 + [1]),
    (12, 12, 64, [1000] * 6), (64, 8, 64, [513] * 8 + [63]),
    (32, 8, 128, [3300]), (32, 8, 128, [300, 1, 257]), (12, 12, 64, [7000]),
])
def test_whole_prompts(nq, nkv, hd, lens):
    q, k, v = _qkv(sum(lens), nq, nkv, hd, len(lens))
    cu, scale = _cu(lens), 0.7 * hd ** -0.5
    got = ops.attn_prefill(q, k, v, cu, max(lens), scale)
    want = reference.attn_prefill(q.float(), k.float(), v.float(), cu,
                                  max(lens), scale)
    _check(got, want, v)


# rows that are not 16-byte aligned, and rows 2^27 elements apart: 32 of them
# are 2^32
@pytest.mark.parametrize("lens,stride,offset", [
    ([700], 1024 + 16, 1), ([300, 600], 1024 + 3, 0), ([70], 1024 + 4, 4),
    ([40], 1 << 27, 0)])
def test_keys_of_any_stride_and_alignment(lens, stride, offset):
    nq, nkv, hd, T = 64, 8, 128, sum(lens)
    g = torch.Generator(device=DEV).manual_seed(T)
    q = torch.randn(T, nq, hd, generator=g, device=DEV).bfloat16()
    at = lambda: torch.empty(T * stride + offset, dtype=torch.bfloat16,
                             device=DEV)[offset:].as_strided(
        (T, nkv, hd), (stride, hd, 1))
    k, v = at(), at()
    for t in (k, v):
        t.copy_(torch.randn(T, nkv, hd, generator=g, device=DEV))
    cu, scale = _cu(lens), hd ** -0.5
    got = ops.attn_prefill(q, k, v, cu, max(lens), scale)
    want = reference.attn_prefill(q.float(), k.float(), v.float(), cu,
                                  max(lens), scale)
    _check(got, want, v)


def test_pages_that_are_not_aligned():
    nq, nkv, hd, bs, n = 64, 8, 128, 64, 700
    g = torch.Generator(device=DEV).manual_seed(1)
    q = torch.randn(n, nq, hd, generator=g, device=DEV).bfloat16()
    size = 16 * nkv * bs * hd
    kc, vc = (torch.randn(size + 4, generator=g, device=DEV).bfloat16()[4:]
              .view(16, nkv, bs, hd) for _ in range(2))
    table = torch.randperm(16, generator=g, device=DEV).int().view(1, 16)
    total = torch.tensor([n + 99], dtype=torch.int32, device=DEV)
    got = ops.attn_prefill_paged(q, kc, vc, table, total, _cu([n]), n,
                                 hd ** -0.5)
    want = reference.attn_decode_with_history(
        q.float(), kc.float(), vc.float(), table, total,
        torch.tensor([n], dtype=torch.int32, device=DEV), hd ** -0.5)
    _check(got, want, vc)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("nq,nkv,hd,lens,hist,bs", [
    (32, 8, 128, [5, 5, 1], [1500, 255, 0], 256),
    (28, 4, 128, [64, 40], [63, 64], 64), (32, 8, 64, [33, 2], [77, 1], 16),
    (6, 2, 128, [40, 9], [100, 300], 24), (12, 12, 64, [130], [1000], 256),
    (28, 4, 128, [2100], [500], 256), (32, 8, 128, [3600], [130], 256),
    # pages of no whole tiles: 128- and 256-row workgroups without turns
    (32, 8, 128, [1300], [200], 48), (28, 4, 128, [900, 1100], [70, 0], 16),
    (64, 8, 128, [1700], [30], 48),
])
def test_chunks_against_pages(nq, nkv, hd, lens, hist, bs, fp8):
    q, _, _ = _qkv(sum(lens), nq, nkv, hd, 3)
    total = [a + b for a, b in zip(lens, hist)]
    W = max(-(-n // bs) for n in total) + 1
    nb = W * len(lens) + 2
    g = torch.Generator(device=DEV).manual_seed(4)
    table = torch.randperm(nb, generator=g, device=DEV)[: W * len(lens)]
    table = table.int().view(len(lens), W)
    kc = torch.randn(nb, nkv, bs, hd, generator=g, device=DEV).bfloat16()
    vc = torch.randn(nb, nkv, bs, hd, generator=g, device=DEV).bfloat16()
    if fp8:
        kc = kc.to(torch.float8_e4m3fn).view(torch.uint8)
        vc = vc.to(torch.float8_e4m3fn).view(torch.uint8)
    cu, scale = _cu(lens), hd ** -0.5
    lens_t = torch.tensor(lens, dtype=torch.int32, device=DEV)
    total_t = torch.tensor(total, dtype=torch.int32, device=DEV)
    got = ops.attn_prefill_paged(q, kc, vc, table, total_t, cu, max(lens),
                                 scale)
    up = (lambda c: c.view(torch.float8_e4m3fn).float()) if fp8 else \
        (lambda c: c.float())
    want = reference.attn_decode_with_history(q.float(), up(kc), up(vc),
                                              table, total_t, lens_t, scale)
    _check(got, want, up(vc))


# 256-row workgroups whose waves take turns: 1 to 5 and more tiles of keys, last
# tiles of 1, 63 and 64, new pages within a workgroup's tiles; scores that climb
# along the keys raise the maximum in every tile
@pytest.mark.parametrize("pages", [None, "bf16", "fp8"])
@pytest.mark.parametrize("nq,nkv,lens,hist,bs", [
    (64, 64, [1, 65, 130, 1020], [0, 63, 62, 1], 64),
    (64, 8, [400, 400], [5, 700], 256), (28, 4, [1950], [191], 64),
    (64, 64, [900], [1], 128), (64, 4, [577, 600], [0, 40], 192),
])
def test_waves_in_turn(nq, nkv, lens, hist, bs, pages):
    hd, T = 128, sum(lens)
    assert ops.require_hip().attn_flash_form(
        T, len(lens), nq, nkv, hd, max(lens), bs if pages else 0) == 257
    g = torch.Generator(device=DEV).manual_seed(T)
    q, k, v = _qkv(T, nq, nkv, hd, 5)
    cu, scale = _cu(lens), hd ** -0.5
    if pages is None:
        k = k * torch.linspace(0.5, 3, T, device=DEV)[:, None, None].bfloat16()
        got = ops.attn_prefill(q, k, v, cu, max(lens), scale)
        want = reference.attn_prefill(q.float(), k.float(), v.float(), cu,
                                      max(lens), scale)
        _check(got, want, v)
        return
    total = [a + b for a, b in zip(lens, hist)]
    W = max(-(-n // bs) for n in total)
    table = torch.randperm(W * len(lens), generator=g, device=DEV).int()
    table = table.view(len(lens), W)
    kc, vc = (torch.randn(W * len(lens), nkv, bs, hd, generator=g,
                          device=DEV) for _ in range(2))
    for row in table.tolist():
        for at, page in enumerate(row):
            kc[page] *= 0.5 + 2.5 * at / W
    dt = torch.bfloat16 if pages == "bf16" else torch.float8_e4m3fn
    kc, vc = kc.to(dt), vc.to(dt)
    lens_t = torch.tensor(lens, dtype=torch.int32, device=DEV)
    total_t = torch.tensor(total, dtype=torch.int32, device=DEV)
    raw = (lambda c: c) if pages == "bf16" else (lambda c: c.view(torch.uint8))
    got = ops.attn_prefill_paged(q, raw(kc), raw(vc), table, total_t, cu,
                                 max(lens), scale)
    want = reference.attn_decode_with_history(
        q.float(), kc.float(), vc.float(), table, total_t, lens_t, scale)
    _check(got, want, vc)


def test_scores_that_climb():
    """Scores that grow along the keys raise the running maximum tile by
    tile, in steps below and above the kernel's slack."""
    T, hd = 400, 128
    q = torch.ones(T, 1, hd, device=DEV).bfloat16()
    ramp = torch.arange(T, device=DEV, dtype=torch.float32)
    for step in (0.02, 1.0):
        k = (ramp * step / hd)[:, None, None].expand(T, 1, hd).bfloat16()
        v = torch.randn(T, 1, hd, device=DEV).bfloat16()
        got = ops.attn_prefill(q, k, v, _cu([T]), T, 1.0)
        want = reference.attn_prefill(q.float(), k.float(), v.float(),
                                      _cu([T]), T, 1.0)
        _check(got, want, v)


def test_a_scale_that_is_not_positive():
    """Takes the plain kernel, as before."""
    q, k, v = _qkv(70, 2, 1, 64, 9)
    for scale in (0.0, -0.1):
        got = ops.attn_prefill(q, k, v, _cu([70]), 70, scale)
        want = reference.attn_prefill(q.float(), k.float(), v.float(),
                                      _cu([70]), 70, scale)
        _check(got, want, v)


@pytest.mark.parametrize("T", [300, 3000])
@pytest.mark.parametrize("hd", [64, 128])
def test_weights_add_up_to_one(hd, T):
    """Where all values are 1 the output is 1: the sum that divides is of the
    weights as they are multiplied. Key 70's weight is 2^7 and 0.98 of half a
    unit of bf16 above, within the kernel's slack."""
    q = torch.zeros(T, 8, hd, device=DEV).bfloat16()
    k = torch.zeros(T, 8, hd, device=DEV).bfloat16()
    q[..., :2] = 1.0
    k[70, :, 0], k[70, :, 1] = 7.0, 0.0055
    v = torch.ones_like(k)
    got = ops.attn_prefill(q, k, v, _cu([T]), T, 0.6931471805599453)
    assert (got == 1).all(), got.float().min().item()
    q, k, _ = _qkv(T, 8, 8, hd, 5)
    got = ops.attn_prefill(q, k, v, _cu([T]), T, hd ** -0.5)
    assert (got == 1).all(), got.float().min().item()


@pytest.mark.parametrize("nkv", [4, 8])
@pytest.mark.parametrize("lens", [
    [700, 90], [33, 0, 650, 1], [1, 600, 40, 300, 64, 65], [500, 20] * 4,
    [257, 1, 900], [150, 31, 400, 90, 7], [260, 30, 129] * 3 + [500],
    [90, 40, 128, 20, 300] * 4,
    # as many blocks of each, of one length and not; rows of tiles turned by their
    # dies; twelve sequences whose parts even out
    [300, 290, 310], [257] * 4, [200, 150, 40] * 2 + [700], [60, 200, 130] * 4])
@pytest.mark.parametrize("hd", [64, 128])
def test_blocks_of_every_sequence(hd, lens, nkv):
    """Every row of tiles of every sequence is taken, however many of them there
    are and whatever the lengths and histories."""
    nq = 4 * nkv
    q, k, v = _qkv(sum(lens), nq, nkv, hd, len(lens))
    cu, scale = _cu(lens), hd ** -0.5
    got = ops.attn_prefill(q, k, v, cu, max(lens), scale)
    want = reference.attn_prefill(q.float(), k.float(), v.float(), cu,
                                  max(lens), scale)
    _check(got, want, v)
    # portions: every second sequence has a history
    bs, old = 64, [(i % 2) * (40 + 97 * i) for i in range(len(lens))]
    total = [a + b for a, b in zip(old, lens)]
    counts = [-(-n // bs) for n in total]
    table = torch.zeros(len(lens), max(counts), dtype=torch.int32, device=DEV)
    pages = torch.randperm(sum(counts) + 1, device=DEV).int()
    at = 0
    for i, c in enumerate(counts):
        table[i, :c] = pages[at : at + c]
        at += c
    kc, vc = (torch.randn(sum(counts) + 1, nkv, bs, hd, device=DEV).bfloat16()
              for _ in range(2))
    sl = torch.tensor(total, dtype=torch.int32, device=DEV)
    got = ops.attn_prefill_paged(q, kc, vc, table, sl, cu, max(lens), scale)
    want = reference.attn_decode_with_history(
        q.float(), kc.float(), vc.float(), table, sl,
        torch.tensor(lens, dtype=torch.int32), scale)
    _check(got, want, vc)


def _check_portions(lens, old, nq, nkv, hd, bs=64):
    total = [a + b for a, b in zip(old, lens)]
    counts = [-(-n // bs) for n in total]
    table = torch.zeros(len(lens), max(counts), dtype=torch.int32, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(sum(total))
    pages = torch.randperm(sum(counts), generator=g, device=DEV).int()
    at = 0
    for i, c in enumerate(counts):
        table[i, :c] = pages[at : at + c]
        at += c
    kc, vc = (torch.randn(sum(counts), nkv, bs, hd, generator=g,
                          device=DEV).bfloat16() for _ in range(2))
    q = torch.randn(sum(lens), nq, hd, generator=g, device=DEV).bfloat16()
    sl = torch.tensor(total, dtype=torch.int32, device=DEV)
    scale = hd ** -0.5
    got = ops.attn_prefill_paged(q, kc, vc, table, sl, _cu(lens), max(lens),
                                 scale)
    want = reference.attn_decode_with_history(
        q.float(), kc.float(), vc.float(), table, sl,
        torch.tensor(lens, dtype=torch.int32), scale)
    _check(got, want, vc)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("lens,old", [
    ([300, 290, 310], [70, 100, 64]), ([520] * 2, [600] * 2),
    ([200, 193, 256, 250, 210, 256, 255, 199], [0] * 8)])
def test_portions_of_as_many_blocks(hd, lens, old):
    """Sequences whose blocks and histories count the same, their lengths do not."""
    order = ops.require_hip().attn_flash_order(sum(lens), len(lens), 32, 8,
                                               max(lens), True)
    assert order == 3
    _check_portions(lens, old, 32, 8, hd)


# (the last: rows of tiles of the longest, its history's among them)
@pytest.mark.parametrize("nq,nkv,hd,form,lens,old,levels", [
    (32, 8, 64, 64, [1024, 30], None, 64), (32, 8, 64, 64, [1025, 30], None, 65),
    (28, 4, 128, 257, [2341, 40], None, 65), (28, 4, 128, 257, [4681, 900], None,
                                              128),
    (28, 4, 128, 257, [4682, 30], None, 129),
    (32, 8, 64, 128, [2100, 20, 700, 1], None, 66),
    (32, 8, 64, 128, [2050, 0, 90, 800, 33, 64], None, 65),
    (28, 4, 128, 64, [64, 700], [5800, 0], 641),
    (32, 8, 128, 64, [300, 65, 300], [0, 4800, 1900], 305),
])
def test_blocks_found_in_two_passes(nq, nkv, hd, form, lens, old, levels):
    """The search by keys looks at 64 levels (rows of tiles) at a time."""
    hip = ops.require_hip()
    T, n, most = sum(lens), len(lens), max(lens)
    bs, G, rows = 64 if old else 0, nq // nkv, form & ~1
    assert max(-(-a * G // rows) + b * G // rows
               for a, b in zip(lens, old or [0] * n)) == levels
    assert hip.attn_flash_form(T, n, nq, nkv, hd, most, bs) == form
    assert hip.attn_flash_order(T, n, nq, nkv, most, bool(old)) == 3
    if old:
        return _check_portions(lens, old, nq, nkv, hd, bs)
    q, k, v = _qkv(T, nq, nkv, hd, n)
    got = ops.attn_prefill(q, k, v, _cu(lens), most, hd ** -0.5)
    want = reference.attn_prefill(q.float(), k.float(), v.float(), _cu(lens),
                                  most, hd ** -0.5)
    _check(got, want, v)


@pytest.mark.parametrize("nq,nkv,new,old,bs", [
    (32, 8, 2100, 4200, 256),       # 33 rows of blocks of 8 heads: 8 are shared
    (32, 8, 2049, 3991, 64), (28, 4, 2900, 6000, 256),
    (16, 1, 4200, 4300, 128),       # 7 blocks, 256 that share them
    (64, 16, 1090, 6001, 256), (24, 8, 2800, 100, 256),
])
def test_a_portion_whose_last_blocks_are_shared(nq, nkv, new, old, bs):
    """Blocks that are more than whole rounds of 256 are cut by keys and joined;
    blocks that no cut meets, and rows that see no key of a piece, among them."""
    hd, total = 128, new + old
    pages = -(-max(total, 6400) // bs)  # (room for more: the kernel finds out)
    g = torch.Generator(device=DEV).manual_seed(new)
    table = torch.randperm(pages, generator=g, device=DEV).int()[None]
    kc, vc = (torch.randn(pages, nkv, bs, hd, generator=g,
                          device=DEV).bfloat16() for _ in range(2))
    q = torch.randn(new, nq, hd, generator=g, device=DEV).bfloat16()
    sl = torch.tensor([total], dtype=torch.int32, device=DEV)
    got = ops.attn_prefill_paged(q, kc, vc, table, sl, _cu([new]), new, 0.1)
    at = torch.cat([torch.arange(0, 80), torch.randint(0, new, (200,)),
                    torch.arange(new - 80, new)]).to(DEV)
    k = kc[table[0].long()].transpose(1, 2).reshape(-1, nkv, hd)[:total].float()
    v = vc[table[0].long()].transpose(1, 2).reshape(-1, nkv, hd)[:total].float()
    k, v = (t.repeat_interleave(nq // nkv, 1).transpose(0, 1).contiguous()
            for t in (k, v))
    sc = q[at].float().transpose(0, 1) @ k.transpose(1, 2).contiguous() * 0.1
    ahead = torch.arange(total, device=DEV) > (old + at)[:, None]
    want = torch.softmax(sc.masked_fill(ahead, -torch.inf), -1) @ v
    _check(got[at], want.transpose(0, 1), vc)
    assert torch.isfinite(got).all()


def _portion(nq, nkv, new, total, bs=256):
    """A portion of `new` tokens of a sequence of `total`, on pages in order."""
    pages = -(-total // bs)
    kc, vc = (torch.randn(pages, nkv, bs, 128, device=DEV).bfloat16()
              for _ in range(2))
    table = torch.arange(pages, dtype=torch.int32, device=DEV)[None]
    sl = torch.tensor([total], dtype=torch.int32, device=DEV)
    q = torch.randn(new, nq, 128, device=DEV).bfloat16()
    cu = _cu([new])
    return lambda: ops.attn_prefill_paged(q, kc, vc, table, sl, cu, new, 0.1), vc


# (8 blocks that 256 workgroups share, and 92)
@pytest.mark.parametrize("nq,nkv,new,places", [(32, 8, 2100, 264),
                                               (28, 4, 3150, 348)])
def test_shared_blocks_without_memory_for_their_pieces(nq, nkv, new, places):
    """The pieces take the places that they need, and where there is no memory for
    these, blocks are taken whole."""
    call, v = _portion(nq, nkv, new, new + 8000)
    want = call()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    held = torch.cuda.memory_allocated()
    assert torch.equal(call(), want)
    room = (torch.cuda.max_memory_allocated() - held
            - want.numel() * want.element_size())
    assert 0 <= room - places * 256 * 130 * 4 < 2 << 20
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    limit = torch.cuda.memory_reserved() + (want.numel() * 2) + (8 << 20)
    whole = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.reset_peak_memory_stats()
    held = torch.cuda.memory_allocated()
    torch.cuda.set_per_process_memory_fraction(limit / whole)
    try:
        got = call()
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert (torch.cuda.max_memory_allocated() - held
            < want.numel() * want.element_size() + (8 << 20))
    # (each is off the exact result by up to _check's bound)
    assert ((got.float() - want.float()).abs().max()
            <= v.float().abs().max() * 2 ** -7)
