"""A decode step's layers in one launch (decode_stack.hip) against the reference
ops in fp64: sizes at the edges of its octets, waves and tiles, contexts that one
workgroup reads and such as are split, one row to the most, and fewer workgroups
than there are numbers.

Tolerance: what passes between the products is rounded to bf16 (2^-9 relative at
most each, independent of each other), about eight times a layer, into a residual
that is not: 1.5% of the result's norm, as the steps' tests ask for. 8-bit pages
round the step's own keys and values, and queries, to 3 mantissa bits: 5%."""
import types

import pytest
import torch

from bee2bee_amd import ops
from bee2bee_amd.ops import reference

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("needs a GPU", allow_module_level=True)

DEV = torch.device("cuda:0")


def _spec(H, nq, nkv, hd, I, kind):
    return types.SimpleNamespace(
        hidden_size=H, n_heads=nq, n_kv_heads=nkv, head_dim=hd,
        intermediate_size=I, norm_type=kind)


def _layer(s, biased, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)

    def rand(*shape, std=1.0, mean=0.0):
        t = torch.empty(*shape, device=DEV).normal_(mean, std, generator=g)
        return t.bfloat16()

    H, I, Q = s.hidden_size, s.intermediate_size, s.n_heads * s.head_dim
    gelu = s.norm_type == "layernorm"
    N = Q + 2 * s.n_kv_heads * s.head_dim
    up = I if gelu else 2 * I
    lw = types.SimpleNamespace(
        wo=rand(H, Q, std=2 * Q ** -0.5), w_gate_up=rand(up, H, std=H ** -0.5),
        w_down=rand(H, I, std=2 * I ** -0.5), wqkv=rand(N, H, std=H ** -0.5))
    for name in ("attn_norm", "mlp_norm"):
        setattr(lw, name, rand(H, std=0.2, mean=1.0))
        setattr(lw, name + "_bias", rand(H, std=0.2) if gelu else None)
    for name, n in (("wo_bias", H), ("w_gate_up_bias", up if gelu else 0),
                    ("w_down_bias", H), ("wqkv_bias", N)):
        setattr(lw, name, rand(n, std=0.5) if biased and n else None)
    return lw


def _wide(lw):
    return types.SimpleNamespace(**{
        k: None if v is None else v.double() for k, v in vars(lw).items()})


def _rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


class _Step:
    """A stack with its pages; `lens` counts the step's own tokens."""

    def __init__(self, spec, layers, lens, bs, biased=False, fp8=False, W=None):
        self.spec, self.fp8, M = spec, fp8, len(lens)
        self.layers = [_layer(spec, biased, i) for i in range(layers)]
        g = torch.Generator(device=DEV).manual_seed(M)
        W = W or max(-(-n // bs) for n in lens)
        nb, nkv, hd = M * W + 1, spec.n_kv_heads, spec.head_dim
        self.pages = []
        for _ in range(layers):
            kv = [torch.empty(nb, nkv, bs, hd, device=DEV).normal_(
                generator=g) for _ in range(2)]
            self.pages.append([
                t.to(torch.float8_e4m3fn).view(torch.uint8) if fp8
                else t.bfloat16() for t in kv])
        self.table = 1 + torch.randperm(M * W, generator=g, device=DEV).int(
            ).view(M, W)
        self.lens = torch.tensor(lens, dtype=torch.int32, device=DEV)
        self.pos, self.bs = self.lens - 1, bs
        self.place()
        self.x = torch.randn(M, spec.hidden_size, generator=g,
                             device=DEV).bfloat16()
        self.cos, self.sin = reference.rope_tables(max(lens), hd, 1e4, DEV)
        self.rope = spec.norm_type == "rmsnorm"
        self.act = "swiglu" if self.rope else "gelu"

    def place(self):
        """Slots of the positions."""
        at, bs = self.pos.long(), self.bs
        self.slots = (self.table.gather(1, (at // bs)[:, None]).squeeze(1) * bs
                      + at % bs).int()

    def run(self, rows=None, workgroups=256, pages=None, **more):
        rows = list(range(len(self.x))) if rows is None else rows
        pages = pages or [[t.clone() for t in kv] for kv in self.pages]
        s = self.spec
        out = ops.decode_stack(
            self.x[rows], self.layers, pages, s.n_heads, self.act, 1e-5,
            s.head_dim ** -0.5, self.pos[rows] if self.rope else None,
            self.cos, self.sin, self.slots[rows], self.table[rows],
            self.lens[rows], workgroups, **more)
        return out, pages

    def want(self):
        s, x = self.spec, self.x.double()
        pages = []
        for lw, kv in zip(self.layers, self.pages):
            lw = _wide(lw)
            kv = [(t.view(torch.float8_e4m3fn) if self.fp8 else t).double()
                  for t in kv]
            q = reference.rows_qkv(
                x, lw.wqkv, lw.wqkv_bias, (lw.attn_norm, lw.attn_norm_bias,
                                           1e-5), s.n_heads,
                self.pos if self.rope else None, self.cos.double(),
                self.sin.double(), *kv, self.slots)
            o = _attention(q, *kv, self.table, self.lens)
            x = reference.rows_linear(o, lw.wo, lw.wo_bias, x)
            z = reference.rows_linear(
                x, lw.w_gate_up, lw.w_gate_up_bias,
                norm=(lw.mlp_norm, lw.mlp_norm_bias, 1e-5), act=self.act)
            x = reference.rows_linear(z, lw.w_down, lw.w_down_bias, x)
            pages.append(kv)
        return x, pages


def _attention(q, kc, vc, table, lens):
    M, nq, hd = q.shape
    nkv, bs = kc.shape[1:3]
    out = []
    for m in range(M):
        k, v = (t[table[m].long()].transpose(0, 1).reshape(nkv, -1, hd)
                [:, : lens[m]].repeat_interleave(nq // nkv, 0)
                for t in (kc, vc))
        p = torch.softmax((k @ q[m][:, :, None])[..., 0] * hd ** -0.5, -1)
        out.append((p[:, None] @ v)[:, 0].reshape(-1))
    return torch.stack(out)


# H, query heads, key heads, head size, inner width, norm, biases, page size,
# contexts: one octet to several a workgroup, waves without a step of K, sizes
# that leave workgroups without an octet of some products; contexts of one key,
# at the ends of tiles and pages, and split ones
CASES = [
    (64, 1, 1, 64, 64, "rmsnorm", False, 16, [1]),
    (256, 4, 2, 64, 1024, "rmsnorm", True, 16, [33, 1, 16, 700, 32]),
    (256, 2, 1, 128, 704, "rmsnorm", False, 24, [1025, 31, 2000]),
    (768, 12, 12, 64, 3072, "layernorm", True, 256, [300]),
    (768, 12, 12, 64, 3072, "layernorm", True, 32, [64, 1500, 257, 1024]),
    (1024, 8, 8, 128, 704, "layernorm", False, 16, [5, 1030]),
    (2048, 32, 8, 64, 8192, "rmsnorm", False, 256, [1000]),
    (2048, 32, 8, 64, 2048, "rmsnorm", False, 256, [3000, 255, 256, 9, 1, 1024,
                                                    1025, 2100]),
    (3584, 28, 4, 128, 18944, "rmsnorm", True, 256, [5000, 8192]),
    (4160, 32, 2, 128, 1088, "rmsnorm", False, 256, [31, 4000, 97]),
]


@pytest.mark.parametrize("workgroups", [256, 100, 3])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[1]}-{c[8]}")
def test_stack(case, fp8, workgroups):
    H, nq, nkv, hd, I, kind, biased, bs, lens = case
    if workgroups == 3 and (H > 1024 or fp8):
        pytest.skip("long")
    spec = _spec(H, nq, nkv, hd, I, kind)
    assert len(lens) <= ops.stack_rows(spec)
    step = _Step(spec, 2, lens, bs, biased, fp8)
    got, pages = step.run(workgroups=workgroups)
    want, want_pages = step.want()
    limit = 0.05 if fp8 else 0.015
    error = _rel(got, want)
    assert error <= limit
    s = step.slots.long()
    for kv, kv_want, before in zip(pages, want_pages, step.pages):
        for t, w, b in zip(kv, kv_want, before):
            rows = (t.view(torch.float8_e4m3fn) if fp8 else t).double()
            error = _rel(rows[s // bs, :, s % bs], w[s // bs, :, s % bs])
            assert error <= limit
            t[s // bs, :, s % bs] = b[s // bs, :, s % bs]
            assert torch.equal(t, b)           # and nothing else


# contexts of one split, and of splits of 128 keys for any number of rows: 1000
# keys in 8 (8 rows of 4 key heads) or more
@pytest.mark.parametrize("lens", [[40, 255, 7, 256, 64, 1, 129, 200],
                                  [40, 1000, 7, 513, 64, 1, 300, 999]])
def test_rows_and_workgroups_do_not_change_a_row(lens):
    """Where a context's splits do not depend on the number of rows, a row is the
    same to the bit beside others, and whoever computes it."""
    spec = _spec(1024, 16, 4, 64, 2816, "rmsnorm")
    step = _Step(spec, 2, lens, 16)
    full, _ = step.run()
    for rows in ([3], [5, 2], [7, 0, 1, 4, 6]):
        assert torch.equal(step.run(rows)[0], full[rows])
        for workgroups in (77, 300, 512):
            assert torch.equal(step.run(rows, workgroups)[0], full[rows])


@pytest.mark.parametrize("kind", ["rmsnorm", "layernorm"])
def test_steps_side_by_side(kind):
    """Three streams whose steps want all CUs: each has some, its workgroups take
    over what the others' keep from starting, and those leave when they start."""
    spec = _spec(768, 12, 4, 64, 3072, kind)
    steps = [_Step(spec, 6, [300, 40], 16), _Step(spec, 6, [1500], 16),
             _Step(spec, 6, [7, 257, 64, 90], 16)]
    status = torch.zeros(1, dtype=torch.int32, pin_memory=True)
    want = [s.run() for s in steps]
    streams = [torch.cuda.Stream() for _ in steps]
    torch.cuda.synchronize()
    for _ in range(5):
        pages = [[[t.clone() for t in kv] for kv in s.pages] for s in steps]
        torch.cuda.synchronize()
        got = []
        for _ in range(4):                     # (the same tokens again)
            for s, p, stream in zip(steps, pages, streams):
                with torch.cuda.stream(stream):
                    got.append(s.run(pages=p, status=status)[0])
        torch.cuda.synchronize()
        assert status.item() == 0
        for i, x in enumerate(got):
            assert torch.equal(x, want[i % 3][0])
        for p, (_, w) in zip(pages, want):
            for kv, kv_want in zip(p, w):
                assert all(torch.equal(a, b) for a, b in zip(kv, kv_want))


def test_more_layers_than_a_launch_takes():
    spec = _spec(128, 2, 1, 64, 128, "rmsnorm")
    step = _Step(spec, 64, [70, 1], 16)
    for lw in step.layers:
        lw.wo *= 0.2
        lw.w_down *= 0.2
    got, want = step.run()[0], step.want()[0]
    error = _rel(got, want)
    assert error <= 0.03


def test_values_that_are_not_numbers_pass():
    """A NaN in one row is that row's alone, and nothing waits for it; so with
    all bits set, the mark of words that are not there yet."""
    spec = _spec(256, 4, 2, 64, 1024, "rmsnorm")
    step = _Step(spec, 2, [5, 1200, 40], 16)
    step.x.view(torch.int16)[1] = -1
    got = step.run()[0]
    assert got[1].isnan().all() and not got[[0, 2]].isnan().any()
    # in what a page holds behind the context's end
    step = _Step(spec, 2, [5, 1200, 40], 16)
    want = step.run()[0]
    for kv in step.pages:
        for t in kv:
            for m, n in enumerate(step.lens.tolist()):
                page = t[step.table[m, (n - 1) // 16].item()]
                page[:, (n - 1) % 16 :] = float("nan")
    assert torch.equal(step.run()[0], want)


def test_a_token_without_a_position():
    """Slot -1: nothing is stored, and attention reads what the pages hold, as
    the plain route does."""
    spec = _spec(256, 4, 2, 64, 1024, "rmsnorm")
    step = _Step(spec, 1, [48, 20], 16)
    step.slots[0] = -1
    step.lens[0] = 49                          # past its three pages
    got, pages = step.run()
    s = step.slots.clone()
    step.slots[0] = 0                          # (page 0 is nobody's)
    step.lens[0] = 48
    want = step.want()[0]
    error = _rel(got, want)
    assert error <= 0.015
    before = [[t.clone() for t in kv] for kv in step.pages]
    for kv, b in zip(pages, before):
        for t, old in zip(kv, b):
            t[s[1] // 16, :, s[1] % 16] = old[s[1] // 16, :, s[1] % 16]
            assert torch.equal(t, old)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hd,bs,lens", [(64, 32, [34, 34, 34, 7]),
                                        (128, 16, [254, 254, 254, 1000]),
                                        (64, 24, [1500, 1500, 1500, 300]),
                                        (128, 256, [2049, 2049, 2049, 20])])
def test_new_tokens_anywhere_in_the_contexts(hd, bs, lens, fp8):
    """Each row's attention has the step's own token of all rows whose pages it
    reads: of three that follow each other in one sequence, and of one that is
    stored inside its context; not behind a context's end."""
    spec = _spec(256, 4, 2, hd, 1024, "rmsnorm")
    step = _Step(spec, 2, lens, bs, fp8=fp8)
    step.table[1] = step.table[2] = step.table[0]
    for m in (0, 1):                           # row 2 has the last of the three
        step.lens[m] -= 2 - m
    step.pos = step.lens - 1
    step.pos[3] = lens[3] // 2
    step.place()
    got, pages = step.run()
    want, want_pages = step.want()
    limit = 0.05 if fp8 else 0.015
    for m in range(4):
        error = _rel(got[m], want[m])
        assert error <= limit, m
    s = step.slots.long()
    for kv, kv_want in zip(pages, want_pages):
        for t, w in zip(kv, kv_want):
            rows = (t.view(torch.float8_e4m3fn) if fp8 else t).double()
            assert _rel(rows[s // bs, :, s % bs], w[s // bs, :, s % bs]) <= limit


@pytest.mark.parametrize("length", [0, -3])
@pytest.mark.parametrize("at", [0, 1, 2])
def test_a_row_without_keys(at, length):
    """Beside contexts that are split: zeros from its attention, as the plain
    route gives, and the other rows as they are beside a row with keys."""
    spec = _spec(256, 4, 2, 64, 1024, "rmsnorm")
    step = _Step(spec, 2, [1500, 48, 2000], 16)
    beside = step.run()[0]
    step.lens[at] = length
    step.slots[at] = -1
    got = step.run()[0]
    others = [m for m in range(3) if m != at]
    assert torch.equal(got[others], beside[others])
    step.lens[at] = step.slots[at] = 0         # (page 0 is nobody's)
    assert _rel(got, step.want()[0]) <= 0.015


@pytest.mark.parametrize("kind", ["rmsnorm", "layernorm"])
@pytest.mark.parametrize("lens", [[40, 7], [1500, 2000, 300]])
@pytest.mark.parametrize("absent", [1, 30, 255])
def test_a_wait_that_ends(kind, lens, absent):
    """For shares that nobody has: the launch ends, the host is told, and the
    pages have what they had, or what a sound step stores."""
    inner = 1024 if kind == "rmsnorm" else 2048          # of 256 octets
    spec = _spec(256, 4, 2, 64, inner, kind)
    step = _Step(spec, 2, lens, 16)
    status = torch.zeros(1, dtype=torch.int32, pin_memory=True)
    want, sound = step.run(status=status)
    torch.cuda.synchronize()
    assert status.item() == 0
    _, pages = step.run(status=status, patience=256, absent=absent)
    torch.cuda.synchronize()
    assert status.item() == 1
    for layer in range(2):
        for t, good, before in zip(pages[layer], sound[layer],
                                   step.pages[layer]):
            same = (t == before) | ((t == good) & (layer == 0))
            assert same.all(), layer
    status.zero_()
    assert torch.equal(step.run(status=status)[0], want)
    assert status.item() == 0


def test_waits_last_while_others_get_on():
    """Three workgroups with some 85 numbers each, of which one takes up to 150 us
    of a product: a launch of 20 ms with a patience of a millisecond at most (of
    64 polls, it gives up now and then)."""
    spec = _spec(8192, 64, 8, 128, 28672, "rmsnorm")
    step = _Step(spec, 1, [300], 256)
    status = torch.zeros(1, dtype=torch.int32, pin_memory=True)
    want = step.run(status=status)[0]
    got = step.run(workgroups=3, status=status, patience=512)[0]
    torch.cuda.synchronize()
    assert status.item() == 0
    assert torch.equal(got, want)


@pytest.mark.parametrize("kind", ["rmsnorm", "layernorm"])
def test_slots_of_the_positions(kind):
    """No slots: where the table has the positions, and nowhere behind its end or
    before its start."""
    spec = _spec(256, 4, 2, 64, 1024, kind)
    step = _Step(spec, 2, [33, 1, 48, 300], 16, W=19)
    step.pos[1], step.pos[2] = -1, 19 * 16
    step.slots[1] = step.slots[2] = -1
    step.cos, step.sin = reference.rope_tables(400, 64, 1e4, DEV)
    step.rope, want = False, step.run() if kind == "layernorm" else None
    pages = [[t.clone() for t in kv] for kv in step.pages]
    cos = step.cos if kind == "rmsnorm" else None

    def run(slots, pages):
        return ops.decode_stack(
            step.x, step.layers, pages, 4, step.act, 1e-5, 0.125,
            step.pos.clamp(min=0) if slots is not None else step.pos, cos,
            step.sin, slots, step.table, step.lens)

    if want is None:
        step.pos[1] = 19 * 16 + 5              # (rotated by a row of the table)
        want = [[t.clone() for t in kv] for kv in step.pages]
        want = run(step.slots, want), want
    assert torch.equal(run(None, pages), want[0])
    for kv, kv_want in zip(pages, want[1]):
        for t, w in zip(kv, kv_want):
            assert torch.equal(t, w)


def test_refused():
    spec = _spec(256, 4, 2, 64, 1024, "rmsnorm")
    step = _Step(spec, 1, [5, 12], 16)
    ok = dict(x=step.x, table=step.table, lens=step.lens, slots=step.slots,
              layers=step.layers, pages=step.pages)

    def call(**change):
        a = {**ok, **change}
        return ops.decode_stack(a["x"], a["layers"], a["pages"], 4, "swiglu",
                                1e-5, 0.125, step.pos, step.cos, step.sin,
                                a["slots"], a["table"], a["lens"])

    call()
    narrow = types.SimpleNamespace(**{**vars(step.layers[0]),
                                      "wo": step.layers[0].wo[:, :128]})
    for bad in [dict(x=step.x[:1]), dict(x=step.x.float()),
                dict(x=step.x[:, :192]), dict(lens=step.lens.long()),
                dict(slots=step.slots[:1]), dict(table=step.table[:1]),
                dict(layers=[narrow]), dict(layers=[], pages=[]),
                dict(pages=[[t[:, :1] for t in step.pages[0]]])]:
        with pytest.raises((RuntimeError, TypeError, IndexError)):
            call(**bad)
    assert ops.stack_rows(_spec(2048, 2, 2, 64, 256, "layernorm")) == 0
    assert ops.stack_rows(_spec(256, 4, 2, 96, 256, "rmsnorm")) == 0
    assert ops.stack_rows(_spec(288, 4, 2, 64, 256, "rmsnorm")) == 0
    assert ops.stack_rows(_spec(256, 34, 2, 64, 256, "rmsnorm")) == 0
