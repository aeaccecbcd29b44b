"""The one-pass paged attention of few query rows (attn_stream.hip) at the
edges of its tiles, row tiles and splits, against the fp32 reference.

Tolerance: a weight and an output element are rounded to bf16 once each (2^-8
relative at most), so an element is off by less than 2^-7 of the largest
value; half of that is asked for, since the weights' roundings do not all add
up. fp32 sums and exp2 add far less. 8-bit cache rows are exact in bf16."""
import pytest
import torch

from bee2bee_amd import ops
from bee2bee_amd.ops import reference

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("needs a GPU", allow_module_level=True)

DEV = "cuda"


def _pages(nkv, hd, bs, total, fp8, seed, width=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    counts = [-(-n // bs) for n in total]
    table = torch.zeros(len(total), max(counts + [width, 1]),
                        dtype=torch.int32, device=DEV)
    nb = sum(counts) + 1
    ids = torch.randperm(nb, generator=g, device=DEV).int()
    at = 0
    for i, c in enumerate(counts):
        table[i, :c] = ids[at : at + c]
        at += c
    caches = []
    for _ in range(2):
        c = torch.randn(nb, nkv, bs, hd, generator=g, device=DEV).bfloat16()
        caches.append(c.to(torch.float8_e4m3fn).view(torch.uint8) if fp8
                      else c)
    lens = torch.tensor(total, dtype=torch.int32, device=DEV)
    return caches[0], caches[1], table, lens


def _wide(c):
    return (c.view(torch.float8_e4m3fn) if c.dtype == torch.uint8
            else c).float()


def _check(got, want, v):
    assert torch.isfinite(got).all()
    err = (got.float() - want.float()).abs().max().item()
    assert err <= v.max().item() * 2 ** -8, err


# (heads, key heads, head size, contexts, page size, table width)
DECODE = [
    (4, 4, 64, [1], 256, 1), (8, 1, 128, [31, 32, 33, 127, 128, 129], 64, 0),
    (7, 1, 128, [1000, 1, 255, 256, 257], 256, 16), (12, 12, 64, [300], 16, 4),
    (6, 2, 128, [77, 129], 24, 0), (16, 1, 64, [3000, 40], 256, 32),
    (32, 8, 128, [5 + 37 * i for i in range(40)], 256, 0),
    (28, 4, 128, [9000, 200], 256, 64),
    # 2 to 4 splits, and some sequences short of them
    (16, 8, 128, [1 + 50 * i for i in range(20)], 256, 0),
    (16, 8, 128, [1 + 80 * i for i in range(9)], 256, 0),
    (12, 12, 64, [1 + 90 * i for i in range(7)], 16, 0),
    # long contexts among short ones: parts of limited length, and contexts
    # of one part that write their result beside them
    (16, 8, 128, [5000, 2048, 2049, 4096, 4097, 1] + [60] * 30, 256, 32),
    (16, 8, 128, [60] * 14 + [7000, 300, 2048, 128], 256, 32),
    (12, 12, 64, [2049, 33] + [33] * 20 + [4100], 64, 96),
]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("nq,nkv,hd,total,bs,width", DECODE)
def test_decode(nq, nkv, hd, total, bs, width, fp8):
    kc, vc, table, lens = _pages(nkv, hd, bs, total, fp8, 1, width)
    q = torch.randn(len(total), nq, hd, device=DEV).bfloat16()
    scale = 0.8 * hd ** -0.5
    got, ml = ops.attn_decode_lse(q, kc, vc, table, lens, scale)
    qf = q.float()
    if fp8:     # decode queries are rounded to the cache's type, scaled
        qf = (qf * scale).bfloat16().to(torch.float8_e4m3fn).float() / scale
    want, want_ml = reference.attn_decode_lse(
        qf, _wide(kc), _wide(vc), table, lens, scale)
    _check(got, want, _wide(vc))
    # the (m, l) pair that ranks merge: l e^m is the sum of e^score
    assert torch.allclose(ml[..., 0] + ml[..., 1].log(),
                          want_ml[..., 0] + want_ml[..., 1].log(), atol=2e-3)
    assert torch.equal(ops.attn_decode(q, kc, vc, table, lens, scale), got)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("nq,nkv,hd,new,old,bs", [
    (32, 8, 128, [5, 1, 4], [1500, 0, 251], 256),
    (32, 8, 64, [8, 3], [77, 1000], 16), (28, 4, 128, [8, 5, 2], [999, 3, 60],
                                          256),
    (6, 2, 128, [11, 0, 1], [100, 40, 300], 24),
    (12, 12, 64, [17, 33], [300, 31], 64), (32, 8, 128, [64], [2000], 256),
])
def test_chunks_of_a_few_tokens(nq, nkv, hd, new, old, bs, fp8):
    total = [a + b for a, b in zip(new, old)]
    kc, vc, table, lens = _pages(nkv, hd, bs, total, fp8, 2)
    q = torch.randn(sum(new), nq, hd, device=DEV).bfloat16()
    cu = torch.tensor([0] + torch.tensor(new).cumsum(0).tolist(),
                      dtype=torch.int32, device=DEV)
    scale = hd ** -0.5
    got = ops.attn_prefill_paged(q, kc, vc, table, lens, cu, max(new), scale)
    want = reference.attn_decode_with_history(
        q.float(), _wide(kc), _wide(vc), table, lens,
        torch.tensor(new, dtype=torch.int32), scale)
    _check(got, want, _wide(vc))


def test_the_last_verified_token_gets_the_sums_of_decoding():
    """On bf16 pages, beside as many sequences in a table as wide, the result
    of a sequence's last token is the same to the bit whether it is decoded or
    verified with others (16 rows in one tile either way)."""
    total, new = [700, 1300], 3
    kc, vc, table, lens = _pages(8, 128, 256, total, False, 3)
    q = torch.randn(2 * new, 32, 128, device=DEV).bfloat16()
    cu = torch.tensor([0, new, 2 * new], dtype=torch.int32, device=DEV)
    rows = ops.attn_prefill_paged(q, kc, vc, table, lens, cu, new, 0.1)
    last = ops.attn_decode(q[new - 1 :: new], kc, vc, table, lens, 0.1)
    assert torch.equal(rows[new - 1 :: new], last)


# (96, 192 and 320 (sequence, key head) pairs: three splits, two, none)
@pytest.mark.parametrize("nseq", [12, 24, 40])
def test_last_verified_tokens_of_many_sequences(nseq):
    """As above, whatever the number of sequences and the order in which decoding
    reads them."""
    total, new = [130 + 57 * i for i in range(nseq)], 4
    kc, vc, table, lens = _pages(8, 128, 256, total, False, 3)
    q = torch.randn(nseq * new, 32, 128, device=DEV).bfloat16()
    cu = torch.arange(nseq + 1, dtype=torch.int32, device=DEV) * new
    rows = ops.attn_prefill_paged(q, kc, vc, table, lens, cu, new, 0.1)
    last = q[new - 1 :: new].contiguous()
    _, order = ops.decode_plan(table, lens - 1, 256, lens, 8)
    for o in (None, order):
        got = ops.attn_decode(last, kc, vc, table, lens, 0.1, o)
        assert torch.equal(rows[new - 1 :: new], got)


def test_queries_at_odd_addresses_and_other_scales():
    kc, vc, table, lens = _pages(2, 64, 32, [70, 5], False, 4)
    flat = torch.randn(2 * (4 * 64 + 1) + 1, device=DEV).bfloat16()
    q = flat[1:].as_strided((2, 4, 64), (4 * 64 + 1, 64, 1), 1)
    for scale in (0.2, 0.0, -0.1):
        got = ops.attn_decode(q, kc, vc, table, lens, scale)
        want = reference.attn_decode(q.float(), kc.float(), vc.float(), table,
                                     lens, scale)
        _check(got, want, vc.float())


def test_an_empty_context_is_zero():
    kc, vc, table, lens = _pages(1, 64, 32, [40, 40], False, 5)
    lens[1] = 0
    q = torch.randn(2, 4, 64, device=DEV).bfloat16()
    out, ml = ops.attn_decode_lse(q, kc, vc, table, lens, 0.125)
    assert (out[1] == 0).all() and (ml[1, :, 1] == 0).all()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("nseq", [2, 40])      # contexts split, and not
def test_a_nan_reaches_the_output(nseq, fp8):
    """A NaN in a key takes the rows of its head, one in a value its
    coordinate, and nothing else, whatever the batch."""
    kc, vc, table, lens = _pages(8, 128, 256, [600] * nseq, fp8, 6)
    nan = 0x7F if fp8 else float("nan")
    kc[table[0, 0], 3, 5, 17] = nan
    vc[table[1, 2], 6, 600 - 512 - 1, 40] = nan
    q = torch.randn(nseq, 32, 128, device=DEV).bfloat16()
    got, ml = ops.attn_decode_lse(q, kc, vc, table, lens, 0.1)
    want, want_ml = reference.attn_decode_lse(q.float(), _wide(kc), _wide(vc),
                                              table, lens, 0.1)
    assert torch.equal(got.isnan(), want.isnan())
    assert got.isnan().sum() == 4 * 128 + 4
    assert torch.equal(ml[..., 1].isnan(), want_ml[..., 1].isnan())
    rows = ops.attn_prefill_paged(q, kc, vc, table, lens, torch.arange(
        nseq + 1, device=DEV, dtype=torch.int32), 1, 0.1)
    assert torch.equal(rows.isnan(), want.isnan())


def test_a_chunk_longer_than_said():
    """Rows past max_qlen have no place in the splits' workspaces: they are
    left out, and the rows before them are what they are without them."""
    kc, vc, table, lens = _pages(2, 64, 256, [1500, 905], False, 8)
    q = torch.randn(10, 8, 64, device=DEV).bfloat16()
    cu = torch.tensor([0, 5, 10], dtype=torch.int32, device=DEV)
    want = ops.attn_prefill_paged(q, kc, vc, table, lens, cu, 5, 0.125)
    got = ops.attn_prefill_paged(q, kc, vc, table, lens, cu, 3, 0.125)
    for at in (0, 5):
        assert torch.equal(got[at : at + 3], want[at : at + 3])


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("nseq", [1, 40])      # contexts split, and not
def test_weights_add_up_to_one(nseq, hd):
    """Where all values are 1 the output is 1: the sum that divides is of the
    weights as they are multiplied. One key of a wave's 32 at the maximum, the
    others where rounding to bf16 takes most (0.5 and 0.98 of half a unit), or
    anywhere."""
    for far in (True, False):
        kc, vc, table, lens = _pages(8, hd, 256, [1000] * nseq, False, 7)
        vc.fill_(1.0)
        q = torch.randn(nseq, 8, hd, device=DEV).bfloat16()
        scale = hd ** -0.5
        if far:
            q.zero_()
            q[..., :2] = 1.0
            kc.zero_()
            kc[..., 0], kc[..., 1] = -1.0, 0.0055
            kc[:, :, ::32, :2] = 0.0
            scale = 0.6931471805599453
        got = ops.attn_decode(q, kc, vc, table, lens, scale)
        assert (got == 1).all(), (far, got.float().min().item())


# contexts at the edges of a tile, of a workgroup's steps and of splits
EDGES = [0, 1, 31, 32, 33, 127, 128, 129, 255, 256, 257, 287, 288, 289, 383, 384,
         385, 511, 512, 513, 767, 768, 769, 900]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("nq,nkv,hd,total,bs,width", [
    (16, 8, 128, EDGES[:12], 256, 4),        # 288 workgroups, 3 splits
    (16, 8, 64, EDGES, 64, 0),               # 384, 2 splits
    (8, 4, 128, EDGES * 4, 128, 0),          # 384 of whole contexts
    (8, 8, 128, EDGES[1::2] * 6, 32, 64),    # 384, tables wider than contexts
    (8, 8, 64, EDGES[::3] + [2500], 256, 16),
    (8, 8, 128, EDGES[:12] * 2, 24, 0),      # pages that tiles cross
])
def test_decode_by_length(nq, nkv, hd, total, bs, width, fp8):
    """In the order of lengths and as the rows stand: the same to the bit."""
    kc, vc, table, lens = _pages(nkv, hd, bs, total, fp8, 4, width)
    q = torch.randn(len(total), nq, hd, device=DEV).bfloat16()
    pos = (lens - 1).clamp(0)
    slots, order = ops.decode_plan(table, pos, bs, lens, nkv)
    assert torch.equal(slots, ops.decode_slots(table, pos, bs))
    if 80 <= len(total) * nkv <= 2048:
        want = sorted(range(len(total)), key=lambda b: (-total[b], b))
        assert order.tolist() == want
    else:
        assert order is None
    got = ops.attn_decode(q, kc, vc, table, lens, 0.1, order)
    assert torch.equal(got, ops.attn_decode(q, kc, vc, table, lens, 0.1))
    qf = q.float()
    if fp8:
        qf = (qf * 0.1).bfloat16().to(torch.float8_e4m3fn).float() / 0.1
    keep = lens > 0
    assert not got[~keep].any()
    want = reference.attn_decode(qf[keep], _wide(kc), _wide(vc), table[keep],
                                 lens[keep], 0.1)
    _check(got[keep], want, _wide(vc))


@pytest.mark.parametrize("B", [10, 64, 65, 2048])
def test_rows_by_length(B):
    """Equal lengths stay as they stand; more lengths and tables than rows."""
    lens = torch.randint(0, 40, (B + 3,), device=DEV, dtype=torch.int32)
    table = torch.randint(0, 99, (B + 3, 2), device=DEV, dtype=torch.int32)
    pos = torch.randint(-1, 70, (B,), device=DEV, dtype=torch.int32)
    nkv = 8 if B < 100 else 1
    slots, order = ops.decode_plan(table, pos, 32, lens, nkv)
    assert torch.equal(slots, ops.decode_slots(table, pos, 32))
    assert torch.equal(order.long(), lens[:B].sort(descending=True,
                                                   stable=True).indices)


@pytest.mark.parametrize("fp8", [False, True])
def test_chunks_of_many_contexts(fp8):
    """Two and three row tiles of a chunk, in 12 and 13 contexts."""
    for new, old in ([4, 5, 1] * 4, [300, 0, 255] * 4), ([9] * 13, [600] * 13):
        total = [a + b for a, b in zip(new, old)]
        kc, vc, table, lens = _pages(8, 128, 256, total, fp8, 2)
        q = torch.randn(sum(new), 32, 128, device=DEV).bfloat16()
        cu = torch.tensor([0] + torch.tensor(new).cumsum(0).tolist(),
                          dtype=torch.int32, device=DEV)
        got = ops.attn_prefill_paged(q, kc, vc, table, lens, cu, max(new), 0.1)
        want = reference.attn_decode_with_history(
            q.float(), _wide(kc), _wide(vc), table, lens,
            torch.tensor(new, dtype=torch.int32), 0.1)
        _check(got, want, _wide(vc))
