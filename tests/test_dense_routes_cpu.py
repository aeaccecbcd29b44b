"""The Runner's routes for dense steps of few rows and of some tens, on the CPU
with the reference ops in the kernels' places, against the plain route."""
import dataclasses
import multiprocessing as mp
import pickle

import pytest
import torch

from bee2bee_amd import ops
from bee2bee_amd.engine.graphs import decode_slot_mapping
from bee2bee_amd.engine.kv import PagedKV
from bee2bee_amd.engine.runner import Runner
from bee2bee_amd.models.spec import PRESETS
from bee2bee_amd.models.weights import ModelWeights
from bee2bee_amd.ops import reference

CPU = torch.device("cpu")
TINY = dataclasses.replace(PRESETS["tiny"], qkv_bias=True, head_dim=32)
ROUTES = {"few": {"few_rows": True}, "mid": {"mid_rows": True},
          "deep": {"deep_rows": True}}


def _weights(spec):
    W = ModelWeights(spec, CPU, torch.float32).random_init(seed=3)
    g = torch.Generator().manual_seed(4)
    W.embed.normal_(0.0, 1.0, generator=g)
    for lw in W.layers:
        for name in lw.__slots__:
            t = getattr(lw, name, None)
            if isinstance(t, torch.Tensor):
                std = 0.5 if name.endswith("bias") else 0.2
                t.normal_(float(name.endswith("norm")), std, generator=g)
    return W


def _steps(spec, W):
    """Hidden rows of two prompts, a decode step and a portion."""
    kv = PagedKV(spec, CPU, torch.float32, n_blocks=16, block_size=16)
    r = Runner(spec, W, kv, CPU, torch.float32)
    ints = lambda x: torch.tensor(x, dtype=torch.int32)
    ids = torch.arange(30) * 7 % 500

    def chunk(lens, old, more):
        pos, slots, cu = [], [], [0]
        for s, (n, o) in enumerate(zip(lens, old)):
            if not o:
                kv.new_seq(s)
            kv.extend_seq(s, o + n)
            pos += range(o, o + n)
            slots += kv.slot_mapping(s, range(o, o + n))
            cu.append(cu[-1] + n)
        if more:
            more = {"block_table": kv.block_table([0, 1]),
                    "seq_lens": ints([a + b for a, b in zip(lens, old)]),
                    "query_lens": ints(lens)}
        return r.forward_prefill(ids[: cu[-1]], ints(pos), ints(slots),
                                 ints(cu), max(lens), **(more or {}))

    out = [chunk([5, 18], [0, 0], False)]
    for s, n in enumerate((6, 19)):
        kv.extend_seq(s, n)
    table, pos = kv.block_table([0, 1]), ints([5, 18])
    out.append(r.forward_decode(ids[:2], pos,
                                decode_slot_mapping(table, pos, 16), table,
                                pos + 1))
    out.append(chunk([4, 3], [6, 19], True))
    out.append(r.lm_head(out[-1]))
    return out


@pytest.mark.parametrize("route", list(ROUTES))
@pytest.mark.parametrize("spec", [TINY, PRESETS["tiny-gpt2"]],
                         ids=["swiglu", "gelu"])
@torch.no_grad()
def test_a_route_computes_what_the_plain_one_does(spec, route, monkeypatch):
    W = _weights(spec)
    want = _steps(spec, W)
    taken = []
    for name in ("few_rows", "mid_rows", "deep_rows"):
        on = ROUTES[route].get(name, False)
        monkeypatch.setattr(ops, name, lambda *a, on=on: on)
    for name in ("rows_linear", "rows_qkv", "mid_linear"):
        op = getattr(ops, name)
        monkeypatch.setattr(ops, name, lambda *a, op=op, name=name, **k: (
            taken.append(name), op(*a, **k))[1])
    got = _steps(spec, W)
    few = {"rows_linear"} | ({"rows_qkv"} if spec.head_dim == 32 else set())
    assert set(taken) == (few if route == "few" else {"mid_linear"})
    for a, b in zip(got, want):
        # fp32 sums in another order
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("spec", [TINY, PRESETS["tiny-gpt2"]],
                         ids=["swiglu", "gelu"])
@torch.no_grad()
def test_few_rows_on_the_rings(spec, monkeypatch):
    W = _weights(spec)
    want = _steps(spec, W)
    taken = []
    monkeypatch.setattr(ops, "few_rows", lambda x: True)
    monkeypatch.setattr(Runner, "_few_on_rings", lambda self, rows: True)
    op = ops.mid_linear
    monkeypatch.setattr(ops, "mid_linear", lambda *a: (
        taken.append(1), op(*a))[1])
    got = _steps(spec, W)
    assert len(taken) == 9 * spec.n_layers     # three steps of three
    for a, b in zip(got, want):
        # fp32 sums in another order
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-4)


# plans: left to the library, whole rows, 4 parts, rows past the last tile apart
@pytest.mark.parametrize("plan", [0, 12, 36, 140])
@pytest.mark.parametrize("spec", [TINY, PRESETS["tiny-gpt2"]],
                         ids=["swiglu", "gelu"])
@torch.no_grad()
def test_steps_of_many_rows_compute_what_the_plain_route_does(spec, plan,
                                                              monkeypatch):
    W = _weights(spec)
    want = _steps(spec, W)
    taken = []
    for name in ("few_rows", "mid_rows", "deep_rows"):
        monkeypatch.setattr(ops, name, lambda *a: False)
    monkeypatch.setattr(ops, "wide_rows", lambda x: True)
    for name in ("MID_MAX", "DEEP_MAX"):
        monkeypatch.setattr(ops, name, 0)
    monkeypatch.setattr(ops, "wide_plan", lambda rows, width, depth, form: (
        plan if form == "parts" or plan != 36 else 12))
    op = ops.wide_linear
    monkeypatch.setattr(ops, "wide_linear", lambda x, w, plan, act=None: (
        taken.append((plan, act)), op(x, w, plan, act))[1])
    got = _steps(spec, W)
    acts = {act for _, act in taken}
    assert taken if plan else not taken
    assert not plan or acts == {None} | (
        set() if spec.act_type == "gelu" else {"swiglu"})
    for a, b in zip(got, want):
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("fp8", [False, True])
def test_parts_beside_8_bit_pages(fp8):
    """Parts give rows of the pages' type, and bf16 beside 8-bit pages."""
    g = torch.Generator().manual_seed(1)
    parts = torch.randn(3, 4, 8 * 16, generator=g)
    dt = torch.uint8 if fp8 else torch.bfloat16
    kc, vc = torch.zeros(2, 2, 16, 16, dtype=dt), torch.zeros(2, 2, 16, 16,
                                                              dtype=dt)
    slots = torch.tensor([3, 17, 0, 31], dtype=torch.int32)
    got = reference.rope_store_qkv(parts, None, 4, None, None, None, kc, vc,
                                   slots)
    assert got.dtype == torch.bfloat16
    assert torch.equal(got, parts.sum(0).bfloat16())
    rows = kc[slots.long() // 16, :, slots.long() % 16]
    want = got.view(4, 8, 16)[:, 4:6]
    assert torch.equal(rows, reference._kv_quant_like(want, kc) if fp8
                       else want)


def _tp_worker(rank, world, port, few, out_path):
    import torch.distributed as dist

    from bee2bee_amd.parallel.tp import TPEngine

    dist.init_process_group(
        backend="gloo", init_method=f"tcp://127.0.0.1:{port}", rank=rank,
        world_size=world)
    try:
        if few:
            ops.few_rows = lambda x: x.dim() == 2 and x.shape[0] <= 16
        eng = TPEngine(TINY, device="cpu", max_batch=4, max_seq_len=64, seed=5)
        out, lm_head = [], eng.runner.lm_head
        eng.runner.lm_head = lambda h: (out.append(lm_head(h)), out[-1])[1]
        tokens = eng.generate([[5, 6, 7, 8, 9], [100, 101]], 4)
        # (a cycle would keep the engine, and so the process group's threads,
        # until the interpreter is gone)
        del eng.runner.lm_head
        if rank == 0:
            with open(out_path, "wb") as f:
                pickle.dump((tokens, out), f)
    finally:
        dist.destroy_process_group()


@pytest.mark.timeout(300)
def test_few_rows_under_tensor_parallelism(tmp_path):
    """Two ranks, each with its part of the inner dimensions: the reduced rows
    are added and normed as on the plain route."""
    results = []
    for few, port in ((False, 29741), (True, 29742)):
        path = str(tmp_path / f"tp{few}.pkl")
        ctx = mp.get_context("spawn")
        procs = [ctx.Process(target=_tp_worker, args=(r, 2, port, few, path))
                 for r in range(2)]
        for p in procs:
            p.start()
        for p in procs:
            p.join(timeout=140)
            assert p.exitcode == 0
        with open(path, "rb") as f:
            results.append(pickle.load(f))
    (t0, l0), (t1, l1) = results
    assert t0 == t1
    for a, b in zip(l0, l1):
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-4)


# rows, outputs, depth: measured with the norm that follows (us, the library's
# product, the best of linear_wide.hip's own)
@pytest.mark.skipif(not ops.hip_available(), reason="the extension is not built")
@pytest.mark.parametrize("M,N,K,library,own", [
    (300, 3072, 2048, 17.8, 20.3), (400, 2048, 2048, 15.1, 17.6),
    (700, 2048, 2048, 17.6, 19.0), (1024, 2048, 2048, 20.9, 23.4),
    (1536, 3072, 2048, 34.4, 37.4), (384, 2560, 2560, 19.9, 22.8),
    (560, 5120, 3072, 34.9, 36.9), (300, 4096, 11008, 67.9, 80.3),
    (330, 1536, 8960, 39.6, 64.7), (3000, 3072, 3072, 77.9, 65.5),
    (512, 2048, 8192, 39.6, 29.6), (1536, 4096, 14336, 184.7, 144.5),
    (800, 5120, 27648, 334.9, 248.7), (600, 1024, 4096, 21.8, 18.4),
    (9217, 5120, 3072, 395.3, 282.8), (650, 4096, 11008, 96.7, 80.6)])
def test_plans_follow_what_was_measured(M, N, K, library, own):
    assert bool(ops.wide_plan(M, N, K, "parts")) == (own < library)


@pytest.mark.skipif(not ops.hip_available(), reason="the extension is not built")
def test_small_products_keep_their_kernel():
    for M in (257, 600, 1023, 4096):
        for N, K in ((768, 768), (2304, 768), (768, 3072), (3072, 1024)):
            assert ops.wide_plan(M, N, K, "parts")


@pytest.mark.parametrize("rows,width,depth,own", [
    (129, 2304, 768, True), (160, 768, 768, True), (160, 2048, 2048, True),
    (161, 768, 768, False), (161, 768, 3072, True), (256, 1024, 4096, True),
    (129, 3072, 2048, False), (256, 2048, 2048, False), (128, 3072, 2048, True),
    (256, 4096, 14336, True), (200, 5120, 3072, False)])
def test_small_products_of_129_to_256_rows(rows, width, depth, own):
    """Steps of small stacks are bound by the host, which a library product
    costs three times as much."""
    assert ops.mid_shape(rows, width, depth) == own


# us as measured: the rings behind a norm, rows_linear
@pytest.mark.parametrize("rows,width,depth,rings,alone", [
    (1, 128256, 8192, 370, 363), (8, 128256, 8192, 371, 359),
    (12, 128256, 8192, 370, 376), (1, 152064, 8192, 454, 427),
    (12, 152064, 8192, 454, 459), (1, 152064, 5120, 244, 277),
    (8, 128256, 4096, 174, 187), (1, 32000, 4096, 48, 50)])
def test_output_heads_of_few_rows(rows, width, depth, rings, alone):
    assert ops.mid_head(rows, width, depth) == (rings < alone)


# us as measured: the rings, the fastest of the library and linear_wide.hip
@pytest.mark.parametrize("rows,width,depth,rings,other", [
    (128, 128256, 4096, 214, 239), (129, 131072, 4096, 217, 202),
    (160, 131072, 4096, 225, 205), (129, 65536, 8192, 191, 207),
    (160, 65536, 8192, 190, 204), (160, 128256, 8192, 412, 424),
    (161, 64000, 4096, 110, 131), (192, 64000, 4096, 112, 133),
    (192, 65536, 2048, 67, 77), (193, 64000, 2048, 69, 67),
    (161, 49152, 2048, 57.4, 56.1), (192, 49152, 2048, 60, 55),
    (256, 49152, 2048, 75, 56), (192, 57344, 2048, 64, 59),
    (192, 65536, 1536, 55, 48), (161, 32000, 1024, 21.5, 21.1),
    (256, 32000, 1024, 27, 24), (224, 32000, 2048, 37, 40),
    (256, 32000, 2048, 41.9, 40.3), (224, 32000, 3072, 51, 53),
    (225, 32000, 3072, 59, 54), (256, 32000, 4096, 71, 72),
    (224, 24576, 4096, 58, 60), (225, 24576, 4096, 64, 60)])
def test_output_heads_of_129_to_256_rows(rows, width, depth, rings, other):
    assert ops.mid_head(rows, width, depth) == (rings < other)


# us as measured: the rings, linear_wide.hip
@pytest.mark.parametrize("rows,width,depth,rings,wide", [
    (160, 5504, 2048, 20.4, 27.4), (256, 5504, 2048, 27.8, 31.1),
    (256, 8192, 1536, 25, 27), (256, 4096, 3072, 37, 47),
    (160, 9216, 1408, 22.1, 26.8), (161, 9216, 1408, 23.2, 21.7),
    (224, 9216, 1408, 25.8, 23.7), (160, 12288, 1024, 19.0, 20.4),
    (161, 12288, 1024, 20.5, 17.7), (224, 14336, 1024, 24.3, 19.8),
    (160, 16384, 768, 18.4, 17.6), (224, 16384, 768, 22.6, 17.6)])
def test_gated_projections_of_129_to_256_rows(rows, width, depth, rings, wide):
    assert ops.mid_gated(rows, width, depth) == (rings < wide)


@pytest.mark.parametrize("head_dim,own,ordered", [
    (64, False, True), (64, True, False), (32, False, False)])
@torch.no_grad()
def test_rows_are_ordered_for_attention_that_takes_it(head_dim, own, ordered,
                                                      monkeypatch):
    """Steps that are not told their slots: an attention of the caller's, and
    head sizes that attn_stream.hip does not have, get no order of the rows."""
    spec = dataclasses.replace(PRESETS["tiny"], head_dim=head_dim)
    kv = PagedKV(spec, CPU, torch.float32, n_blocks=16, block_size=16)
    r = Runner(spec, _weights(spec), kv, CPU, torch.float32)
    if own:
        r.decode_attn_fn = ops.attn_decode
    kv.new_seq(0)
    kv.extend_seq(0, 3)
    taken, op = [], ops.decode_plan
    monkeypatch.setattr(ops, "decode_plan", lambda *a: (
        taken.append(1), op(*a))[1])
    table, pos = kv.block_table([0]), torch.tensor([2], dtype=torch.int32)
    ids = torch.tensor([7])
    kv_before = [t.clone() for t in [*kv.k_cache, *kv.v_cache]]
    got = r.forward_decode(ids, pos, None, table, pos + 1)
    assert bool(taken) == ordered
    for t, old in zip([*kv.k_cache, *kv.v_cache], kv_before):
        t.copy_(old)
    want = r.forward_decode(ids, pos, decode_slot_mapping(table, pos, 16), table,
                            pos + 1)
    assert torch.equal(got, want)
