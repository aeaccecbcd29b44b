"""Pipeline parallelism on the HIP path: two processes share one MI355X
(gloo transport staging through host) and must produce greedy tokens of the
single-process GPU stack, but for ties: a stage's rows are rounded to bf16 on
their way to the next."""
import multiprocessing as mp
import pickle

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("requires MI355X", allow_module_level=True)

PROMPTS = [[11, 22, 33, 44], [7] * 9]
N_NEW = 6
SEED = 77


def _pp_worker(rank, world, port, out_path):
    import torch.distributed as dist

    from bee2bee_amd.parallel.pp import PipelineEngine

    dist.init_process_group(
        backend="gloo", init_method=f"tcp://127.0.0.1:{port}",
        rank=rank, world_size=world,
    )
    try:
        eng = PipelineEngine(
            "llama3.2-1b", device="cuda:0", max_batch=4, max_seq_len=128,
            seed=SEED,
        )
        outs = eng.generate(PROMPTS, N_NEW)
        if rank == world - 1:
            with open(out_path, "wb") as f:
                pickle.dump(outs, f)
    finally:
        dist.destroy_process_group()


@pytest.mark.timeout(600)
def test_pp2_gpu_matches_single(tmp_path):
    out_path = str(tmp_path / "pp_gpu.pkl")
    ctx = mp.get_context("spawn")
    procs = [
        ctx.Process(target=_pp_worker, args=(r, 2, 29721, out_path))
        for r in range(2)
    ]
    for p in procs:
        p.start()
    for p in procs:
        p.join(timeout=500)
        assert p.exitcode == 0, f"pp gpu worker exit {p.exitcode}"
    with open(out_path, "rb") as f:
        pp_outs = pickle.load(f)

    # the logits of a single process on the same GPU and weights decide
    from bee2bee_amd.engine.engine import InferenceEngine

    from tests.test_engine_gpu import NEAR_TIE, decoded_gaps

    eng = InferenceEngine("llama3.2-1b", device="cuda:0", max_batch=4,
                          max_seq_len=128, seed=SEED, use_graphs=False)
    try:
        gaps = [decoded_gaps(eng, p, out) for p, out in zip(PROMPTS, pp_outs)]
    finally:
        eng.shutdown()
    assert [len(g) for g in gaps] == [N_NEW] * len(PROMPTS)
    assert max(map(max, gaps)) <= NEAR_TIE, gaps
