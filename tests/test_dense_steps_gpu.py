"""Steps of dense stacks at the row counts where the Runner changes its route
(few rows, some tens, a few hundred, more), against the same steps in fp32 on
the CPU.

Tolerance: a layer rounds about eight tensors to bf16 (2^-9 relative at most,
independent of each other) and adds their effects to a residual that is rounded
once or twice; two layers and the head stay below 1% of the result's norm, and
1.5% is asked for. 8-bit pages round keys, values and, in decoding, queries
to 3 mantissa bits (2^-4 at most) on top: 5%."""
import pytest
import torch

from bee2bee_amd.engine.graphs import decode_slot_mapping
from bee2bee_amd.engine.kv import PagedKV
from bee2bee_amd.engine.runner import Runner
from bee2bee_amd.models.spec import ModelSpec
from bee2bee_amd.models.weights import ModelWeights

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("needs a GPU", allow_module_level=True)

DEV, CPU = torch.device("cuda:0"), torch.device("cpu")
SWIGLU = ModelSpec(name="t-swiglu", vocab_size=500, hidden_size=256,
                   intermediate_size=1024, n_layers=2, n_heads=4, n_kv_heads=2,
                   head_dim=64, max_seq_len=1024, qkv_bias=True)
GELU = ModelSpec(name="t-gelu", vocab_size=500, hidden_size=256,
                 intermediate_size=1024, n_layers=2, n_heads=4, n_kv_heads=4,
                 head_dim=64, max_seq_len=1024, qkv_bias=True, arch="gpt2",
                 norm_type="layernorm", act_type="gelu", pos_type="learned",
                 attn_out_bias=True, mlp_bias=True)


# long q|k|v and attention output, and rows longer than 4096: few parts of K, or
# one; from 129 rows on some of their products are the library's
WIDE = [ModelSpec(name="t-wide-qkv", vocab_size=500, hidden_size=128,
                  intermediate_size=256, n_layers=2, n_heads=64,
                  n_kv_heads=32, head_dim=64, max_seq_len=1024),
        ModelSpec(name="t-wide", vocab_size=500, hidden_size=6208,
                  intermediate_size=128, n_layers=2, n_heads=2, n_kv_heads=2,
                  head_dim=64, max_seq_len=1024)]


def _tensors(holder):
    names = getattr(holder, "__slots__", None) or list(vars(holder))
    pairs = [(n, getattr(holder, n, None)) for n in names]
    return [(n, t) for n, t in pairs if isinstance(t, torch.Tensor)]


def _weights(spec):
    """The same random weights, biases and norms on GPU and CPU."""
    W = ModelWeights(spec, CPU, torch.float32).random_init(seed=3)
    g = torch.Generator().manual_seed(4)
    W.embed.normal_(0.0, 1.0, generator=g)
    for holder in [W, *W.layers]:
        for name, t in _tensors(holder):
            if name == "embed":
                continue
            if name.endswith("bias"):
                t.normal_(0.0, 0.5, generator=g)
            elif name.endswith("norm"):
                t.normal_(1.0, 0.2, generator=g)
            elif t.dim() == 2:
                t.normal_(0.0, t.shape[1] ** -0.5, generator=g)
    G = ModelWeights(spec, DEV, torch.bfloat16).random_init(seed=3)
    for a, b in zip([W, *W.layers], [G, *G.layers]):
        for name, t in _tensors(a):
            t.copy_(t.bfloat16())
            getattr(b, name).copy_(t)
    return W, G


class _Side:
    """A stack with its pages on one device."""

    def __init__(self, spec, weights, device, dtype, kv_dtype):
        self.kv = PagedKV(spec, device, dtype, n_blocks=600, block_size=16,
                          kv_dtype=kv_dtype)
        self.runner = Runner(spec, weights, self.kv, device, dtype)
        self.device, self.seqs = device, 0

    def ints(self, x):
        return torch.tensor(x, dtype=torch.int32, device=self.device)

    def prompt(self, ids, lens, old=None):
        """ids of new sequences of these lengths, or, with `old`, the next
        portions of the last ones."""
        chunked = old is not None
        if not chunked:
            old = [0] * len(lens)
            self.rows = list(range(self.seqs, self.seqs + len(lens)))
            self.seqs += len(lens)
            for s in self.rows:
                self.kv.new_seq(s)
        pos, slots, cu = [], [], [0]
        for s, n, o in zip(self.rows, lens, old):
            self.kv.extend_seq(s, o + n)
            pos += range(o, o + n)
            slots += self.kv.slot_mapping(s, range(o, o + n))
            cu.append(cu[-1] + n)
        more = {}
        if chunked:
            more = {"block_table": self.kv.block_table(self.rows),
                    "seq_lens": self.ints([o + n for o, n in zip(old, lens)]),
                    "query_lens": self.ints(lens)}
        return self.runner.forward_prefill(
            ids.to(self.device), self.ints(pos), self.ints(slots),
            self.ints(cu), max(lens), **more)

    def decode(self, ids, n):
        """One token for each of the last sequences, which hold n."""
        for s in self.rows:
            self.kv.extend_seq(s, n + 1)
        table = self.kv.block_table(self.rows)
        pos = self.ints([n] * len(self.rows))
        return self.runner.forward_decode(
            ids.to(self.device), pos,
            decode_slot_mapping(table, pos, 16), table, pos + 1)


def _rel(got, want):
    got, want = got.double().cpu(), want.double().cpu()
    return ((got - want).norm() / want.norm()).item()


@pytest.mark.parametrize("spec,rows,kv_dtype", [
    (spec, rows, kv_dtype) for spec in (SWIGLU, GELU)
    for rows in (1, 9, 16, 17, 128, 129, 160, 161, 256, 257)
    for kv_dtype in ("native", "fp8")
] + [(spec, rows, "native") for spec in WIDE for rows in (17, 129, 200, 257)],
    ids=lambda v: getattr(v, "name", str(v)))
@torch.no_grad()
def test_steps(spec, rows, kv_dtype):
    W, G = _weights(spec)
    gpu = _Side(spec, G, DEV, torch.bfloat16, kv_dtype)
    cpu = _Side(spec, W, CPU, torch.float32, kv_dtype)
    g = torch.Generator().manual_seed(rows)
    ids = lambda n: torch.randint(0, 500, (n,), generator=g)
    lens = [n for n in (rows - rows // 3 - rows // 5, rows // 3, rows // 5)
            if n]
    steps = [("prompts", "prompt", ids(rows), lens),
             ("histories", "prompt", ids(3 * rows), [3] * rows),
             ("decode", "decode", ids(rows), 3),
             ("history", "prompt", ids(40), [40]),
             ("portion", "prompt", ids(rows), [rows], [40])]
    for name, call, *args in steps:
        got, want = (getattr(side, call)(*args) for side in (gpu, cpu))
        limit = 0.015 if kv_dtype == "native" else 0.05
        assert _rel(got, want) <= limit, (name, _rel(got, want))
        last = slice(-min(rows, 20), None)
        got, want = gpu.runner.lm_head(got[last]), cpu.runner.lm_head(
            want[last])
        assert _rel(got, want) <= limit, (name, _rel(got, want))


@pytest.mark.parametrize("hidden,rows,rings", [
    (3072, 11, False), (3072, 12, True), (4096, 8, False), (4096, 9, True),
    (4096, 16, True)])
def test_few_rows_of_wide_stacks(hidden, rows, rings):
    spec = ModelSpec(name="t-few", vocab_size=512, hidden_size=hidden,
                     intermediate_size=1024, n_layers=2, n_heads=8,
                     n_kv_heads=2, head_dim=64, max_seq_len=128)
    side = _Side(spec, ModelWeights(spec, DEV, torch.bfloat16).random_init(
        seed=3), DEV, torch.bfloat16, "native")
    assert side.runner._few_on_rings(rows) == rings
    test_steps(spec, rows, "native")


DEEP = ModelSpec(name="t-deep", vocab_size=500, hidden_size=256,
                 intermediate_size=14336, n_layers=2, n_heads=4, n_kv_heads=2,
                 head_dim=64, max_seq_len=1024)


@pytest.mark.parametrize("spec,rows,attention,one", [
    (SWIGLU, 1, False, True), (SWIGLU, 6, False, True), (SWIGLU, 7, False, False),
    (GELU, 6, False, True), (GELU, 8, False, False), (DEEP, 2, False, True),
    (DEEP, 3, False, False), (SWIGLU, 1, True, False)],
    ids=lambda v: getattr(v, "name", str(v)))
@torch.no_grad()
def test_which_steps_are_one_launch(spec, rows, attention, one, monkeypatch):
    from bee2bee_amd import ops

    W = ModelWeights(spec, DEV, torch.bfloat16).random_init(seed=3)
    side = _Side(spec, W, DEV, torch.bfloat16, "native")
    side.prompt(torch.arange(rows), [1] * rows)
    if attention:
        side.runner.decode_attn_fn = ops.attn_decode
    taken, op = [], ops.decode_stack
    monkeypatch.setattr(ops, "decode_stack", lambda *a, **k: (
        taken.append(1), op(*a, **k))[1])
    side.decode(torch.arange(rows), 1)
    assert len(taken) == one


@pytest.mark.parametrize("spec", [SWIGLU, GELU], ids=["swiglu", "gelu"])
@torch.no_grad()
def test_captured_steps_of_few_rows(spec, monkeypatch):
    """One capture, replayed at lengths around a tile, 256 keys (what is not
    split) and the table's end: as the same step is eagerly, to the bit, and as
    it is launch by launch (the tolerance above)."""
    from bee2bee_amd.engine.graphs import DecodeGraphs

    W = ModelWeights(spec, DEV, torch.bfloat16).random_init(seed=3)
    side = _Side(spec, W, DEV, torch.bfloat16, "native")
    kv, runner = side.kv, side.runner
    for t in [*kv.k_cache, *kv.v_cache]:
        t.normal_()
    graphs = DecodeGraphs(runner, 2, 64)
    graphs.block_table.copy_(torch.randperm(600)[:128].int().view(2, 64))
    held = [t.clone() for t in [*kv.k_cache, *kv.v_cache]]

    def step(run, lens):
        for t, h in zip([*kv.k_cache, *kv.v_cache], held):
            t.copy_(h)
        graphs.input_ids.copy_(torch.tensor([7, 11]))
        graphs.seq_lens.copy_(torch.tensor(lens))
        graphs.positions.copy_(torch.tensor(lens) - 1)
        logits = run().clone()
        return [logits, *(t.clone() for t in [*kv.k_cache, *kv.v_cache])]

    for lens in ([255, 1], [256, 32], [257, 33], [1000, 1024], [2, 256]):
        got = step(lambda: graphs.run(2), lens)
        for a, b in zip(got, step(lambda: graphs._run(2), lens)):
            assert torch.equal(a, b)
        with monkeypatch.context() as m:
            m.setattr(Runner, "_one_launch", lambda self, *a: False)
            want = step(lambda: graphs._run(2), lens)
        assert _rel(got[0], want[0]) <= 0.015
        assert _rel(torch.stack(got[1:]), torch.stack(want[1:])) <= 0.015


@torch.no_grad()
def test_what_few_rows_take_and_refuse():
    """As steps of more rows do: tables and lengths of more rows than there are;
    no contexts past 32768 tokens, and not every group of query heads."""
    W = ModelWeights(SWIGLU, DEV, torch.bfloat16).random_init(seed=3)
    side = _Side(SWIGLU, W, DEV, torch.bfloat16, "native")
    side.prompt(torch.arange(9), [1] * 9)
    table = side.kv.block_table(side.rows)
    lens = side.ints([2] * 9)

    def step(rows, table=table, lens=lens):
        pos = lens[:rows] - 1
        return side.runner.forward_decode(
            torch.ones(rows, dtype=torch.int64, device=DEV), pos,
            decode_slot_mapping(table[:rows], pos, 16), table, lens)

    for rows in (2, 7):
        assert torch.equal(step(rows), step(rows, table[:rows].contiguous(),
                                            lens[:rows]))
        wide = torch.zeros(rows, 2049, dtype=torch.int32, device=DEV)
        wide[:, 0] = table[:rows, 0]
        assert step(rows, wide[:, :2048].contiguous()).isfinite().all()
        with pytest.raises(RuntimeError, match="32768"):
            step(rows, wide)
        with pytest.raises(RuntimeError):
            step(rows, wide[:, :2048])         # (not contiguous)
    from bee2bee_amd import ops

    for heads, rows in ((8, 8), (9, 0), (15, 0), (16, 8)):
        spec = ModelSpec(name="t-group", vocab_size=64, hidden_size=576,
                         intermediate_size=128, n_layers=1, n_heads=heads,
                         n_kv_heads=1, head_dim=64, max_seq_len=64)
        assert ops.stack_rows(spec) == rows


def test_a_step_that_gave_up_is_told():
    """What such a launch leaves on the host (test_decode_stack_gpu.py): the next
    call raises, and the ones after it do not."""
    W = ModelWeights(SWIGLU, DEV, torch.bfloat16).random_init(seed=3)
    side = _Side(SWIGLU, W, DEV, torch.bfloat16, "native")
    side.prompt(torch.arange(3), [3])
    want = side.decode(torch.tensor([1]), 3)
    side.runner.step_status.fill_(1)
    with pytest.raises(RuntimeError, match="without all"):
        side.decode(torch.tensor([1]), 3)
    side.runner.check_steps()
    assert torch.equal(side.decode(torch.tensor([1]), 3), want)


def test_wide_specs_leave_products_to_the_library():
    """What WIDE above is for: each has one that is left, and one that is not."""
    from bee2bee_amd import ops

    for spec in WIDE:
        H, I, Q = spec.hidden_size, spec.intermediate_size, spec.q_size
        shapes = [(Q + 2 * spec.kv_size, H), (H, Q), (H, I)]
        assert len({ops.mid_shape(200, *s) for s in shapes}) == 2, spec.name
        assert all(ops.mid_shape(128, *s) for s in shapes)


# logits that are linear_wide's, the rings' (up to 160 rows) and the library's
@pytest.mark.parametrize("vocab,hidden,rows,wide", [
    (100000, 2048, 129, True), (100000, 2048, 200, True),
    (65536, 1024, 700, True), (65536, 1024, 160, False),
    (65536, 1024, 161, False)])
@torch.no_grad()
def test_output_heads_of_many_rows(vocab, hidden, rows, wide):
    from bee2bee_amd import ops

    spec = ModelSpec(name="t-head", vocab_size=vocab, hidden_size=hidden,
                     intermediate_size=128, n_layers=1, n_heads=2,
                     n_kv_heads=2, head_dim=64, max_seq_len=64)
    W = ModelWeights(spec, DEV, torch.bfloat16).random_init(seed=3)
    kv = PagedKV(spec, DEV, torch.bfloat16, n_blocks=4, block_size=16)
    runner = Runner(spec, W, kv, DEV, torch.bfloat16)
    g = torch.Generator(device=DEV).manual_seed(rows)
    x = torch.randn(rows, hidden, generator=g, device=DEV).bfloat16()
    assert bool(ops.wide_plan(rows, vocab, hidden, "rows")) == wide
    got = runner.lm_head(x).double()
    x, w = x.double(), W.lm_head.double()
    normed = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + spec.rms_eps)
    normed = normed * W.final_norm.double()
    want, mag = normed @ w.t(), normed.abs() @ w.abs().t()
    # the normed rows and the logits are rounded to bf16 once each
    assert ((got - want).abs() <= 2 ** -8 * (mag + want.abs()) + 1e-5).all()


@pytest.mark.parametrize("rows", [1, 9, 17])
@torch.no_grad()
def test_norms_see_the_unrounded_residual(rows):
    """Where the residual stands at 256, a bf16 one moves in steps of 2: the
    norm after a sum takes it before it is rounded."""
    spec = GELU
    W, G = _weights(spec)
    for w in (W, G):
        w.embed.fill_(256.0)
        w.pos_embed.zero_()
        for lw in w.layers:
            lw.wo.zero_()
            lw.w_down.copy_(100 * lw.w_down)
    gpu = _Side(spec, G, DEV, torch.bfloat16, "native")
    cpu = _Side(spec, W, CPU, torch.float32, "native")
    ids = torch.arange(rows) % 7
    got, want = (s.prompt(ids, [rows]) for s in (gpu, cpu))
    # the first layer's norm of 256 + bias, through gelu and 100 w_down
    assert _rel(got, want) <= 0.015, _rel(got, want)


def test_a_captured_step_ends_at_its_block_table():
    """48 positions in three pages of 16: a request that asks for more ends
    there, and the one beside it goes on."""
    from bee2bee_amd.engine.engine import GenerationRequest, InferenceEngine
    from bee2bee_amd.engine.sampler import SamplingParams

    eng = InferenceEngine("tiny", device="cuda:0", max_batch=2, max_seq_len=40,
                          kv_block_size=16, kv_blocks=12)
    try:
        assert eng.graphs is not None
        reqs = [eng.submit(GenerationRequest(
            prompt_ids=[1, 2, 3], max_new_tokens=n,
            sampling=SamplingParams(greedy=True))) for n in (1000, 30)]
        for r in reqs:
            while isinstance(r.out_queue.get(timeout=60), int):
                pass
            assert r.error is None
        assert [len(r.prompt_ids) + len(r.output_ids) for r in reqs] == [49,
                                                                         33]
    finally:
        eng.shutdown()
