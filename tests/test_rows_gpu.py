"""Projections of a few rows (linear_rows.hip) at the edges of their tiles, of
the waves' shares of K and of the kernel shapes, against fp32.

Tolerance: the normed input and the output are rounded to bf16 once each (2^-8
relative at most): an element is off by at most 2^-8 of the sum of its
products' magnitudes, carried through the activation (whose slope is below
1.13), and 2^-8 of itself."""
import types

import pytest
import torch
import torch.nn.functional as F

from bee2bee_amd import ops
from bee2bee_amd.ops import reference

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("needs a GPU", allow_module_level=True)

DEV = "cuda"


def _rand(*shape, std=1.0, mean=0.0):
    return (torch.randn(*shape, device=DEV) * std + mean).bfloat16()


def _norm(kind, K):
    if kind is None:
        return None
    b = _rand(K, std=0.1) if kind == "layer" else None
    return (_rand(K, std=0.1, mean=1.0), b, 1e-5)


def _f32(norm):
    return norm and (norm[0].float(),
                     None if norm[1] is None else norm[1].float(), norm[2])


def _products(x, w, norm):
    """fp32 product and the sum of its terms' magnitudes."""
    h = x.float()
    if norm is not None:
        n = _f32(norm)
        h = (reference.rmsnorm(h, n[0], n[2]) if n[1] is None
             else reference.layernorm(h, *n))
    return h @ w.float().t(), h.abs() @ w.float().abs().t()


@pytest.mark.parametrize("M", [1, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K", [
    (16, 32), (17, 64), (50257, 96), (768, 3072), (4096, 2048), (4112, 256),
    (4608, 3584), (1000, 4096 + 32), (9, 64), (2052, 576),
    (16384, 160), (16421, 96), (16400, 8192),
])
@pytest.mark.parametrize("kind", [None, "rms", "layer"])
def test_plain(M, N, K, kind):
    torch.manual_seed(M + N)
    x, w, b, r = _rand(M, K), _rand(N, K, std=0.05), _rand(N), _rand(M, N)
    norm = _norm(kind, K)
    got = ops.rows_linear(x, w, b, r, norm).float()
    y, mag = _products(x, w, norm)
    want = y + b.float() + r.float()
    assert ((got - want).abs() <= 2 ** -8 * (mag + want.abs()) + 1e-5).all()
    if N > 16:    # bare, and rows at an odd address
        flat = _rand(M * K + 1)
        xo = flat[1:].view(M, K)
        got = ops.rows_linear(xo, w).float()
        y, mag = _products(xo, w, None)
        assert ((got - y).abs() <= 2 ** -8 * (mag + y.abs()) + 1e-5).all()


@pytest.mark.parametrize("M", [1, 5, 6, 16])
@pytest.mark.parametrize("I,K", [(16, 64), (8192, 2048), (48, 3072 + 96)])
def test_activations(M, I, K):
    torch.manual_seed(M + I)
    x, w, norm = _rand(M, K), _rand(2 * I, K, std=0.03), _norm("rms", K)
    got = ops.rows_linear(x, w, norm=norm, act="swiglu").float()
    y, mag = _products(x, w, norm)
    (g, u), (mg, mu) = y.chunk(2, -1), mag.chunk(2, -1)
    want = F.silu(g) * u
    bound = 2 ** -8 * (1.13 * mg * u.abs() + F.silu(g).abs() * mu
                       + want.abs()) + 2 ** -16 * mg * mu
    assert ((got - want).abs() <= bound + 1e-5).all()
    norm, b = _norm("layer", K), _rand(2 * I)
    got = ops.rows_linear(x, w, b, norm=norm, act="gelu").float()
    y, mag = _products(x, w, norm)
    want = F.gelu(y + b.float(), approximate="tanh")
    assert ((got - want).abs()
            <= 2 ** -8 * (1.13 * mag + want.abs()) + 1e-5).all()


@pytest.mark.parametrize("N,K,act", [
    (2048, 576, None), (4096, 576, None), (4112, 256, None), (64, 96, None),
    (16384, 96, None), (16421, 416, None), (4100, 8192, None),
    (4096, 320, "swiglu"), (4096, 96, "swiglu"), (64, 256, "gelu"),
])
def test_rows_alone(N, K, act):
    """A row's result is the same to the bit whatever rows are beside it."""
    torch.manual_seed(N)
    x, w, norm = _rand(16, K), _rand(N, K, std=0.05), _norm("rms", K)
    b = _rand(N) if act == "gelu" else None
    rows = lambda n: ops.rows_linear(x[:n].contiguous(), w, b, norm=norm,
                                     act=act)
    one = rows(1)
    for n in (2, 8, 9, 16):
        assert torch.equal(rows(n)[:1], one)


# (sides up to 768 and 4096: loads without the streaming hint)
@pytest.mark.parametrize("M", [1, 9])
@pytest.mark.parametrize("N,K,act", [
    (768, 4096, None), (776, 4096, None), (768, 4160, None), (4096, 768, None),
    (2048, 768, "swiglu"), (2064, 768, "swiglu"), (2048, 832, "swiglu")])
def test_both_sides_of_the_streaming_hint(M, N, K, act):
    torch.manual_seed(N + K)
    x, w = _rand(M, K), _rand(2 * N if act else N, K, std=0.05)
    got = ops.rows_linear(x, w, act=act).float()
    want, mag = _products(x, w, None)
    if act:
        (g, u), (mg, mu) = want.chunk(2, -1), mag.chunk(2, -1)
        want = F.silu(g) * u
        mag = 1.13 * mg * u.abs() + F.silu(g).abs() * mu
    assert ((got - want).abs() <= 2 ** -8 * (mag + want.abs()) + 1e-5).all()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("M,nq,nkv,hd,K,kind", [
    (1, 32, 8, 128, 256, "rms"), (16, 7, 1, 64, 96, "rms"),
    (3, 12, 12, 64, 768, "layer"), (2, 2, 1, 32, 64, "rms"),
    (8, 24, 4, 128, 320, "rms"), (9, 24, 4, 128, 320, "rms"),
    (2, 32, 2, 128, 192, "layer"), (3, 32, 2, 128, 192, "rms"),
])
def test_qkv(M, nq, nkv, hd, K, kind, fp8):
    torch.manual_seed(M)
    N = (nq + 2 * nkv) * hd
    x, w, b, norm = _rand(M, K), _rand(N, K, std=0.1), _rand(N), \
        _norm(kind, K)
    cos, sin = reference.rope_tables(64, hd, 1e4, DEV)
    pos = torch.arange(M, device=DEV, dtype=torch.int32) * 3 + 1
    rope = kind == "rms"
    nb, bs = 3, 24
    dt = torch.uint8 if fp8 else torch.bfloat16
    kc = torch.zeros(nb, nkv, bs, hd, device=DEV, dtype=dt)
    vc = torch.zeros_like(kc)
    slots = torch.randperm(nb * bs, device=DEV)[:M].int()
    q = ops.rows_qkv(x, w, b, norm, nq, pos if rope else None, cos, sin, kc,
                     vc, slots)
    y, mag = _products(x, w, norm)
    y = (y + b.float()).view(M, -1, hd)
    # a rotated element mixes two products
    mag = mag.view(M, -1, hd) + y.abs()
    mag = mag + mag.roll(hd // 2, -1)
    wq, wk, wv = (t.clone() for t in y.split([nq, nkv, nkv], 1))
    if rope:
        reference.rope_inplace(wq, wk, pos, cos, sin)
    mq, mk, mv = mag.split([nq, nkv, nkv], 1)
    assert ((q.float() - wq).abs() <= 2 ** -8 * mq + 1e-5).all()
    s = slots.long()
    for cache, want, m in ((kc, wk, mk), (vc, wv, mv)):
        rows = cache[s // bs, :, s % bs]
        step = 2 ** -8
        if fp8:      # and one rounding to 3 mantissa bits
            rows, step = rows.view(torch.float8_e4m3fn), 2 ** -8 + 2 ** -4
        assert ((rows.float() - want).abs() <= step * m + 2 ** -9).all()
        rest = cache.clone()
        rest[s // bs, :, s % bs] = 0
        assert (rest == 0).all()


@pytest.mark.parametrize("M", [1, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(64, 32), (2048, 576), (2080, 192),
                                 (4104, 96), (4128, 64)])
def test_sum_and_next_norm(M, N, K):
    """The residual sum in fp32 and what the next RMS norm's projection takes
    of it, through that projection; and a layer norm of fp32 rows. Their norm
    stands at 256: rounded to bf16, rows would move in steps of 2."""
    torch.manual_seed(M + N)
    x, w, b = _rand(M, K), _rand(N, K, std=0.05), _rand(N)
    resid = 256 + torch.randn(M, N, device=DEV)
    then = _rand(N, std=0.1, mean=1.0)
    total, scaled, squares = ops.rows_linear(x, w, b, resid, keep32=True,
                                             then=then)
    want = x.double() @ w.double().t() + b.double() + resid.double()
    # fp32 sums of K exact products, and of values near 256
    assert ((total.double() - want).abs() <= 2 ** -23 * (K + 300)).all()
    t32 = total * then.float()
    assert ((scaled.float() - t32).abs() <= 2 ** -8 * t32.abs()).all()
    eights = total.double().square().view(M, -1, 8).sum(-1)
    assert ((squares.double() - eights).abs() <= 2 ** -21 * eights).all()
    if N % 32:
        return
    w2 = _rand(80, N, std=0.05)
    for norm in ((then, None, 1e-5), (then, b, 1e-5)):
        y, mag = _products(total, w2, norm)
        args = (scaled, w2), {"norm": (squares, 1e-5)}
        if norm[1] is not None:
            args = (total, w2), {"norm": norm}
            # mean and deviation of values near 256 from sums of fp32 squares:
            # 2^-24 of 2^16, a few times, of a variance near 1
            mag = mag * 1.5 + 2 ** -5 * y.abs()
        got = ops.rows_linear(*args[0], **args[1]).float()
        assert ((got - y).abs() <= 2 ** -8 * (mag + y.abs()) + 1e-5).all()


def test_a_row_does_not_depend_on_the_others():
    torch.manual_seed(0)
    x, w, norm = _rand(16, 4096), _rand(6144, 4096, std=0.02), \
        _norm("rms", 4096)
    full = ops.rows_linear(x, w, norm=norm)
    for rows in (slice(0, 1), slice(7, 12)):
        part = ops.rows_linear(x[rows].contiguous(), w, norm=norm)
        assert torch.equal(part, full[rows])


def test_refused():
    x, w = _rand(17, 64), _rand(32, 64)
    with pytest.raises(RuntimeError):
        ops.rows_linear(x, w)
    with pytest.raises(RuntimeError):
        ops.rows_linear(x[:4, :40].contiguous(), w[:, :40].contiguous())
    with pytest.raises(RuntimeError):       # fp32 rows without a layer norm
        ops.rows_linear(x[:4].float(), w)
    with pytest.raises(RuntimeError):       # squares of other rows
        ops.rows_linear(x[:4], w, norm=(torch.ones(4, 4, device=DEV), 1e-5))


# ------------------------------------------------- steps of some tens of rows


@pytest.mark.parametrize("M", [1, 17, 32, 33, 64, 65, 96, 97, 128, 129, 160,
                               161, 200, 256])
@pytest.mark.parametrize("N,K", [(64, 64), (68, 1088), (3584, 960),
                                 (4096, 2048), (512, 8192 + 64), (6148, 3072),
                                 (33004, 64)])
def test_parts_over_k(M, N, K):
    """Products of bf16 numbers are exact in fp32: only the order of the sums
    differs, at most K roundings of a partial sum."""
    torch.manual_seed(M + N)
    x, w = _rand(M, K), _rand(N, K, std=0.05)
    part = ops.mid_linear(x, w)
    want = x.double() @ w.double().t()
    mag = x.double().abs() @ w.double().abs().t()
    assert ((part.double().sum(0) - want).abs() <= 2 ** -24 * K * mag).all()


# (tiles a workgroup takes: 1 to 4, 5 to 8, 9 to 12, and several groups of
# them; steps of K fewer than the rings' slots, and more)
@pytest.mark.parametrize("M", [1, 17, 32, 33, 64, 65, 96, 97, 128, 129, 160,
                               161, 192, 193, 224, 225, 256])
@pytest.mark.parametrize("N,K,act", [
    (8, 64, "swiglu"), (2056, 1088, "swiglu"), (9000, 192, "swiglu"),
    (17000, 704, "swiglu"), (25000, 128, "swiglu"), (4, 64, None),
    (3072, 768, "gelu"), (8204, 320, "gelu"), (33004, 576, None),
    (32004, 320, None)])     # (eight tiles each, the last workgroup one)
def test_activated_rows(M, N, K, act):
    """Products are exact in fp32, their sums off by K roundings at most; an
    activation's slope is below 1.13, and the result is rounded to bf16."""
    torch.manual_seed(M + N)
    x, w = _rand(M, K), _rand(2 * N if act == "swiglu" else N, K, std=0.1)
    bias = _rand(N) if act == "gelu" else None
    got = ops.mid_rows_linear(x, w, bias, act).double()
    z = x.double() @ w.double().t()
    e = 2 ** -24 * K * (x.double().abs() @ w.double().abs().t())
    if act == "swiglu":
        g, u = z.chunk(2, -1)
        eg, eu = e.chunk(2, -1)
        want = F.silu(g) * u
        e = 1.13 * eg * u.abs() + F.silu(g).abs() * eu + 1.13 * eg * eu
    elif act == "gelu":
        want = F.gelu(z + bias.double(), approximate="tanh")
        e = 1.13 * (e + 2 ** -23 * (z.abs() + bias.double().abs()))
    else:
        want = z
    # (exp in fp32: 2^-20 covers its argument's rounding)
    assert ((got - want).abs() <= e + (2 ** -8 + 2 ** -20) * want.abs()
            + 1e-6).all()


# (five to eight tiles a workgroup)
@pytest.mark.parametrize("N,K,act", [
    (4096, 14336, None), (6144, 2048, None), (3588, 4160, None),
    (14336, 512, "swiglu"), (9000, 320, "swiglu")])
def test_sums_of_k_in_halves(N, K, act):
    """161 to 224 rows sum K in two chains as 65 to 96 do: a row is the same to the
    bit among them."""
    torch.manual_seed(N)
    x = _rand(224, K)
    w = _rand(2 * N if act else N, K, std=0.05)
    run = (lambda rows: ops.mid_rows_linear(x[:rows], w, None, act)) if act else (
        lambda rows: ops.mid_linear(x[:rows], w))
    want = run(96)
    for rows in (161, 192, 193, 224):
        assert torch.equal(run(rows)[..., :96, :], want)


@pytest.mark.parametrize("M", [1, 17, 57, 129, 256])
@pytest.mark.parametrize("N,K", [(8192, 704), (3588, 640), (512, 320)])
def test_rows_are_parts_rounded(N, K, M):
    """Rows of narrow projections (tails of many rows, gelu) and their parts, of
    which these have one, sum K in the same order."""
    torch.manual_seed(N + M)
    x, w = _rand(M, K), _rand(N, K, std=0.1)
    parts = ops.mid_linear(x, w)
    assert parts.shape[0] == 1
    assert torch.equal(ops.mid_rows_linear(x, w), parts[0].bfloat16())


# (tiles a workgroup: six, the last of 12 columns, fewer steps of K than the rings
# have slots; five and a second group, more steps; eight, and in the last workgroup
# one; eight and a second group)
@pytest.mark.parametrize("N,K", [(20492, 128), (40004, 960), (32004, 320),
                                 (65524, 192)])
def test_logits_of_few_rows(N, K):
    """As above without an activation; a row's logits are the same to the bit
    whatever rows are beside it."""
    torch.manual_seed(N)
    x, w = _rand(16, K), _rand(N, K, std=0.1)
    got = ops.mid_rows_linear(x, w)
    want = x.double() @ w.double().t()
    e = 2 ** -24 * K * (x.double().abs() @ w.double().abs().t())
    assert ((got.double() - want).abs() <= e + 2 ** -8 * want.abs()
            + 1e-6).all()
    for at in (slice(0, 1), slice(3, 5), slice(1, 16)):
        assert torch.equal(ops.mid_rows_linear(x[at].contiguous(), w), got[at])


# (a workgroup's tiles of 8 columns: up to 4, 8, 12, and two groups of 7)
@pytest.mark.parametrize("N,K", [(8192, 6144), (12560, 4096), (17008, 3008),
                                 (25008, 2048)])
def test_long_gated_projections_of_few_rows(N, K):
    """Rows that come with their sums of squares: 1 / rms in fp32 (a relative
    2^-20 of the products, with the slopes of the activation), a row's result
    the same to the bit whatever rows are beside it."""
    torch.manual_seed(N)
    x, w = _rand(16, K), _rand(2 * N, K, std=0.05)
    squares = torch.rand(16, K // 8, device=DEV) * 16 + 1
    rows = lambda at: ops.rows_linear(
        x[at].contiguous(), w, norm=(squares[at].contiguous(), 1e-5),
        act="swiglu")
    got = rows(slice(0, 16))
    inv = torch.rsqrt(squares.double().sum(-1, keepdim=True) / K + 1e-5)
    z = x.double() @ w.double().t() * inv
    mag = (x.double().abs() @ w.double().abs().t()) * inv
    e = (2 ** -24 * K + 2 ** -20) * mag
    (g, u), (eg, eu) = z.chunk(2, -1), e.chunk(2, -1)
    want = F.silu(g) * u
    bound = 1.13 * eg * u.abs() + F.silu(g).abs() * eu + 1.13 * eg * eu
    assert ((got.double() - want).abs() <= bound + (2 ** -8 + 2 ** -20)
            * want.abs() + 1e-6).all()
    for at in (slice(0, 1), slice(3, 5), slice(7, 16)):
        assert torch.equal(rows(at), got[at])


# (rows: edges of halves and of tiles of 128, 192 and 256; 256 columns a tile,
# 128 gated; 2 steps of K a part, the least, and more. The last four: more tiles
# than CUs at 2100 rows, so that a workgroup takes several, the loads of one
# under the last steps and the stores of another.)
@pytest.mark.parametrize("tall", [2, 3, 4])
@pytest.mark.parametrize("M", [1, 64, 97, 129, 256, 2100])
@pytest.mark.parametrize("N,K,act,S", [
    (8, 128, None, 1), (264, 256, None, 1), (2304, 1152, None, 1),
    (8, 256, "swiglu", 1), (136, 128, "swiglu", 1), (1160, 896, "swiglu", 1),
    (264, 256, None, 2), (512, 1152, None, 3), (1032, 4096, None, 8),
    (9000, 128, None, 1), (8712, 640, None, 1), (4616, 256, "swiglu", 1),
    (4104, 768, None, 2)])
def test_wide_products(M, N, K, act, S, tall):
    """As the activated rows and the parts above."""
    torch.manual_seed(M + N)
    x, w = _rand(M, K), _rand(2 * N if act else N, K, std=0.1)
    got = ops.wide_linear(x, w, tall + 8 * S, act).double()
    want = x.double() @ w.double().t()
    e = 2 ** -24 * K * (x.double().abs() @ w.double().abs().t())
    if S > 1:
        assert got.shape == (S, M, N)
        assert ((got.sum(0) - want).abs() <= e).all()
        return
    if act:
        (g, u), (eg, eu) = want.chunk(2, -1), e.chunk(2, -1)
        want = F.silu(g) * u
        e = 1.13 * eg * u.abs() + F.silu(g).abs() * eu + 1.13 * eg * eu
    bound = e + (2 ** -8 + 2 ** -20) * want.abs() + 1e-6
    assert ((got - want).abs() <= bound).all()
    if M > tall * 64:       # the rows past the last whole tile on their own
        got = ops.wide_linear(x, w, tall + 8 + 128, act).double()
        assert ((got - want).abs() <= bound).all()


# (tiles of 160 and 224 rows, whose halves differ: one row or one short of a tile
# past the last, rows that end in either half; several tiles a workgroup)
@pytest.mark.parametrize("M,N,K,act,S,tall", [
    (161, 264, 256, None, 1, 3), (449, 8712, 768, None, 1, 3),
    (2242, 1032, 768, None, 1, 3), (4559, 4104, 512, None, 1, 3),
    (321, 3072, 768, None, 2, 3), (2242, 264, 512, None, 2, 3),
    (449, 4104, 768, "swiglu", 1, 3), (4559, 3072, 512, "swiglu", 1, 3),
    (225, 264, 512, None, 1, 4), (1121, 1032, 512, None, 1, 4),
    (2241, 3072, 256, None, 1, 4), (4481, 4104, 256, None, 1, 4),
    (1345, 3072, 256, None, 2, 4), (321, 9000, 256, "swiglu", 1, 4),
    (3001, 3072, 256, "swiglu", 1, 4)])
def test_heights_between(M, N, K, act, S, tall):
    """As above, and to the bit what tiles of 128 rows give."""
    plan = tall + 8 * S
    hip = ops.require_hip()
    assert hip.wide_height(M, N, K, plan, bool(act)) == 64 * tall - 32
    assert hip.wide_height(M, N, K, 2 + 8 * S, bool(act)) == 128
    torch.manual_seed(M + N)
    x, w = _rand(M, K), _rand(2 * N if act else N, K, std=0.1)
    got = ops.wide_linear(x, w, plan, act)
    assert torch.equal(got, ops.wide_linear(x, w, 2 + 8 * S, act))
    if S == 1 and not act:
        want = x.double() @ w.double().t()
        e = 2 ** -24 * K * (x.double().abs() @ w.double().abs().t())
        bound = e + (2 ** -8 + 2 ** -20) * want.abs() + 1e-6
        assert ((got.double() - want).abs() <= bound).all()


def test_wide_plans_are_what_the_kernel_takes():
    """Whole pairs of steps a part, parts only for a reader that sums them, rows
    apart only beside whole tiles; sizes that the kernel does not take stay with
    the library."""
    for M in (1, 129, 257, 300, 1000, 1536, 4097, 9217, 16384):
        for N, K in ((8, 256), (768, 3072), (3584, 18944), (4608, 3584),
                     (14336, 4096), (128256, 4096), (4096, 14336)):
            for form in ("rows", "gated", "parts"):
                plan = ops.wide_plan(M, N, K, form)
                if plan == 0:
                    assert form != "gated"
                    continue
                tall, S, apart = plan % 8, plan // 8 % 16, plan >= 128
                assert 2 <= tall <= 4 and S in (1, 2, 4, 8) and plan < 256
                assert K % (128 * S) == 0 and (S == 1 or form == "parts")
                assert not apart or (S == 1 and 0 < M % (64 * tall) < M)
    for N, K in ((12, 4096), (4096, 4160), (4096, 128), (4096, 1 << 23)):
        for form in ("rows", "gated", "parts"):
            assert ops.wide_plan(4096, N, K, form) == 0


@pytest.mark.parametrize("S,M,H", [(1, 17, 64), (8, 128, 4096), (4, 20, 8192),
                                   (2, 33, 3592)])
@pytest.mark.parametrize("kind", [None, "rms", "layer"])
def test_add_norm_parts(S, M, H, kind):
    torch.manual_seed(S)
    part = torch.randn(S, M, H, device=DEV)
    bias, resid = _rand(H) if S > 1 else None, _rand(M, H)
    norm = _norm(kind, H)
    y, total = ops.add_norm_parts(part, bias, resid, norm)
    want_y, want = reference.add_norm_parts(
        part, None if bias is None else bias.float(), resid.float(),
        _f32(norm))
    assert ((total.float() - want).abs() <= 2 ** -8 * want.abs()
            + 1e-5).all()
    assert (y is None) == (norm is None)
    if y is not None:
        assert ((y.float() - want_y).abs() <= 2 ** -8 * want_y.abs()
                + 1e-4).all()


# (256 rows and more: another kernel; 2048 columns and more: another's threads)
@pytest.mark.parametrize("S,M,H", [(2, 256, 2048), (8, 9, 2056), (4, 257, 4096),
                                   (1, 300, 72)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_add_norm_parts_in_fp32(S, M, H, dtype):
    """A residual in fp32, as fp32 or bf16: fp32 sums of S + 2 numbers."""
    torch.manual_seed(S)
    part, resid = (torch.randn(*s, M, H, device=DEV) for s in ((S,), ()))
    norm = _norm("rms", H)
    y, total = ops.add_norm_parts(part, _rand(H), resid, norm, dtype)
    torch.manual_seed(S)
    part, resid = (torch.randn(*s, M, H, device=DEV) for s in ((S,), ()))
    norm = _norm("rms", H)
    want_y, want = reference.add_norm_parts(part, _rand(H).float(), resid,
                                            _f32(norm))
    assert total.dtype is dtype and y.dtype is torch.bfloat16
    step = 2 ** -8 if dtype is torch.bfloat16 else 0
    assert ((total.float() - want).abs() <= step * want.abs() + 1e-5).all()
    assert ((y.float() - want_y).abs() <= 2 ** -8 * want_y.abs() + 1e-4).all()


@pytest.mark.parametrize("parts", [0, 1, 4])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("T,nq,nkv,hd,rope,biased", [
    (1, 4, 2, 16, True, False), (57, 28, 4, 128, True, True),
    (33, 12, 12, 64, False, True), (300, 3, 1, 96, True, False),
    (65, 8, 8, 64, False, False),
])
def test_rope_store_qkv(T, nq, nkv, hd, rope, biased, parts, fp8):
    torch.manual_seed(T)
    N = (nq + 2 * nkv) * hd
    qkv = torch.randn(parts, T, N, device=DEV) if parts else _rand(T, N)
    bias = _rand(N) if biased else None
    cos, sin = reference.rope_tables(512, hd, 1e4, DEV)
    pos = torch.randint(0, 512, (T,), device=DEV, dtype=torch.int32)
    bs, nb = 24, T // 24 + 2
    dt = torch.uint8 if fp8 else torch.bfloat16
    kc = torch.zeros(nb, nkv, bs, hd, device=DEV, dtype=dt)
    vc = torch.zeros_like(kc)
    slots = torch.randperm(nb * bs, device=DEV)[:T].int()
    y = (qkv.sum(0) if parts else qkv.float().clone())
    if biased:
        y = y + bias.float()
    want = y.view(T, -1, hd).clone()
    wq, wk, _ = want.split([nq, nkv, nkv], 1)
    if rope:
        reference.rope_inplace(wq, wk, pos, cos, sin)
    got = ops.rope_store_qkv(qkv, bias, nq, pos if rope else None, cos, sin,
                             kc, vc, slots)
    if not parts:
        assert got.data_ptr() == qkv.data_ptr()
    got = got.view(T, -1, hd)
    # one rounding to bf16 (2^-8 relative at most) of a sum that fp32 holds to
    # 2^-20 of its terms
    mag = y.view(T, -1, hd).abs()
    mag = mag + mag.roll(hd // 2, -1)
    assert ((got.float() - want).abs()
            <= 2 ** -8 * want.abs() + 2 ** -20 * mag + 1e-6).all()
    s = slots.long()
    for cache, rows in ((kc, got[:, nq : nq + nkv]), (vc, got[:, nq + nkv :])):
        stored = cache[s // bs, :, s % bs]
        if fp8:
            rows = rows.float().to(torch.float8_e4m3fn).view(torch.uint8)
        assert torch.equal(stored, rows)
        rest = cache.clone()
        rest[s // bs, :, s % bs] = 0
        assert (rest == 0).all()


# ------------------------------------------------------ what a step starts with


@pytest.mark.parametrize("B,W,bs", [(1, 1, 16), (257, 5, 24), (3, 128, 256)])
def test_decode_slots(B, W, bs):
    torch.manual_seed(B)
    wide = torch.randint(0, 10000, (B + 1, W + 3), device=DEV,
                         dtype=torch.int32)
    table = wide[:, :W]           # rows at a stride, more of them than asked
    pos = torch.randint(0, W * bs, (B,), device=DEV, dtype=torch.int32)
    pos[0] = W * bs - 1
    got = ops.decode_slots(table, pos, bs)
    want = reference.decode_slots(table[:B], pos, bs)
    assert got.dtype == want.dtype and torch.equal(got, want)


@pytest.mark.parametrize("T,H", [(1, 8), (33, 768), (2, 2048)])
def test_embed_positions(T, H):
    torch.manual_seed(T)
    table, pos_table = _rand(50, H), _rand(40, H)
    ids = torch.randint(0, 50, (T,), device=DEV)
    pos = torch.randint(0, 40, (T,), device=DEV, dtype=torch.int32)
    got = ops.embed_positions(ids, table, pos, pos_table)
    assert torch.equal(got, table[ids] + pos_table[pos.long()])


def test_ids_and_positions_that_the_tables_do_not_have():
    """No slot and nothing stored, a row of NaN, keys of the pages alone; the
    rows beside them are what they are."""
    i32 = dict(device=DEV, dtype=torch.int32)
    table = torch.tensor([[1, 3], [2, 0], [4, 5], [3, 1]], **i32)
    pos = torch.tensor([31, 32, -1, 5], **i32)
    slots = ops.decode_slots(table, pos, 16)
    assert slots.tolist() == [63, -1, -1, 53]
    emb, pemb = _rand(50, 64), _rand(40, 64)
    ids = torch.tensor([3, 50, -1, 7, 8], device=DEV)
    at = torch.tensor([1, 2, 3, 40, 39], **i32)
    got = ops.embed_positions(ids, emb, at, pemb)
    assert torch.equal(got[[0, 4]], emb[[3, 8]] + pemb[[1, 39]])
    assert got[1:4].isnan().all()
    nkv, hd = 2, 64
    cos, sin = reference.rope_tables(64, hd, 1e4, DEV)
    pos = pos.clamp(0)
    for dt in (torch.bfloat16, torch.uint8):
        qkv, x = _rand(4, 4 * nkv * hd), _rand(4, 64)
        w, norm = _rand(4 * nkv * hd, 64), (_rand(64), None, 1e-5)
        k = qkv.view(4, -1, hd)[:, :nkv]
        for store in (
                lambda c, v: ops.rope_store_qkv(
                    qkv.clone(), None, 2 * nkv, pos, cos, sin, c, v, slots),
                lambda c, v: ops.rows_qkv(x, w, None, norm, 2 * nkv, pos, cos,
                                          sin, c, v, slots),
                lambda c, v: ops.kv_cache_store(k, k, c, v, slots)):
            # a page before the cache and one after it
            flat = torch.zeros(2, 8, nkv, 16, hd, device=DEV, dtype=dt)
            store(flat[0][1:7], flat[1][1:7])
            rows = flat.transpose(2, 3).reshape(2, 8 * 16, nkv * hd)
            used = (rows != 0).any(-1)
            assert used.nonzero().tolist() == [
                [c, 16 + s] for c in (0, 1) for s in (53, 63)]
    kc, vc = _rand(6, nkv, 16, hd), _rand(6, nkv, 16, hd)
    q = _rand(4, 4, hd)
    past = torch.tensor([32, 33, 1000, 6], **i32)
    assert torch.equal(ops.attn_decode(q, kc, vc, table, past, 0.1),
                       ops.attn_decode(q, kc, vc, table, past.clamp(max=32),
                                       0.1))


@pytest.mark.parametrize("hd", [64, 128])
def test_positions_that_the_rotation_has_not(hd):
    """Its first row for positions before the tables, its last for those behind
    them, in every kernel that rotates."""
    M, nq, nkv, K, rows = 6, 4, 2, 256, 40
    torch.manual_seed(hd)
    N = (nq + 2 * nkv) * hd
    x, w, norm = _rand(M, K), _rand(N, K, std=0.1), _norm("rms", K)
    qkv = _rand(M, N)
    cos, sin = (t[:rows] for t in reference.rope_tables(rows + 24, hd, 1e4, DEV))
    pos = torch.tensor([-1, 39, 40, 63, -2 ** 31, 2 ** 31 - 1],
                       dtype=torch.int32, device=DEV)
    table = torch.arange(M, dtype=torch.int32, device=DEV).view(M, 1)
    slots = table.view(-1) * 16
    wo, up, down = (_rand(*s, std=0.1) for s in ((K, nq * hd), (1024, K),
                                                 (K, 512)))
    layer = types.SimpleNamespace(
        wqkv=w, wo=wo, w_gate_up=up, w_down=down, attn_norm=norm[0],
        mlp_norm=norm[0], **{n + "_bias": None for n in (
            "wqkv", "wo", "w_gate_up", "w_down", "attn_norm", "mlp_norm")})

    def inplace(pos, k, v):
        y = qkv.clone().view(M, -1, hd)
        ops.rope_inplace(y[:, :nq], y[:, nq : nq + nkv], pos, cos, sin)
        return y

    for op in (
            lambda p, k, v: ops.rows_qkv(x, w, None, norm, nq, p, cos, sin, k,
                                         v, slots),
            lambda p, k, v: ops.rope_store_qkv(qkv.clone(), None, nq, p, cos,
                                               sin, k, v, slots),
            inplace,
            lambda p, k, v: ops.decode_stack(
                x, [layer], [(k, v)], nq, "swiglu", 1e-5, 0.125, p, cos, sin,
                slots, table, torch.ones_like(slots))):
        results = []
        for p in (pos, pos.clamp(0, rows - 1)):
            pages = [torch.zeros(M, nkv, 16, hd, device=DEV,
                                 dtype=torch.bfloat16) for _ in range(2)]
            results.append([op(p, *pages), *pages])
        for a, b in zip(*results):
            assert torch.equal(a, b)
