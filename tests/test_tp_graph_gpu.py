"""hipGraph-captured decode step containing RCCL collectives (1 GPU).

Before an 8-GPU node runs TP decode graphs,
prove the capture mechanics on a single MI355X with a 1-rank NCCL(=RCCL)
group — the model's 2-per-layer all-reduces execute inside the captured
graph (numerically no-ops at world 1) and the replayed tokens match the
eager no-graph engine exactly.
"""
import os

import pytest
import torch

pytestmark = pytest.mark.gpu

PROMPT = [3, 1, 4, 1, 5, 9, 2, 6]
N = 12


def _run_engine(use_graphs: bool, group):
    from ollamamq_amd.models import LlamaModel, PRESETS
    from ollamamq_amd.engine import GenParams, LlamaEngine, PagedKVCache
    cfg = PRESETS["tiny"]
    model = LlamaModel(cfg, device="cuda:0", dtype=torch.bfloat16,
                       seed=1234, process_group=group)
    kv = PagedKVCache.for_model(cfg, n_pages=64, max_slots=4, max_ctx=256,
                                device="cuda:0", dtype=torch.bfloat16)
    eng = LlamaEngine(model, kv, max_batch=4)
    eng.use_graphs = use_graphs
    eng.use_pipeline = False   # compare plain step semantics
    sids = [eng.submit(PROMPT, GenParams(max_tokens=N)),
            eng.submit(PROMPT[::-1], GenParams(max_tokens=N))]
    seqs = [eng.seqs[s] for s in sids]
    for _ in range(80):
        eng.step()
        if not eng.has_work():
            break
    torch.cuda.synchronize()
    return [list(s.generated) for s in seqs]


@pytest.fixture(scope="module")
def nccl_world1():
    import torch.distributed as dist
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    os.environ.setdefault("MASTER_ADDR", "127.0.0.1")
    os.environ.setdefault("MASTER_PORT", "29531")
    torch.cuda.set_device(0)
    dist.init_process_group("nccl", rank=0, world_size=1)
    yield dist.group.WORLD
    dist.destroy_process_group()


def test_allreduce_inside_captured_graph(nccl_world1):
    """Bare mechanics: an RCCL all-reduce captured in a hipGraph replays."""
    import torch.distributed as dist
    x = torch.ones(4096, device="cuda:0")
    # communicator must exist before capture: one eager collective first
    dist.all_reduce(x)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        dist.all_reduce(x)
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        x.mul_(2.0)
        dist.all_reduce(x)
    for _ in range(3):
        g.replay()
    torch.cuda.synchronize()
    # initial ones -> *2 warmup leaves arbitrary start; assert finite and
    # consistent: value = start * 2^3 where start was x after warmups
    assert torch.isfinite(x).all()


def test_graphed_decode_with_collectives_matches_eager(nccl_world1):
    """Engine decode steps whose graphs CONTAIN the TP all-reduces produce
    the same tokens as the eager engine (greedy, bit-stable)."""
    eager = _run_engine(False, nccl_world1)
    graphed = _run_engine(True, nccl_world1)
    assert graphed == eager, f"{graphed} != {eager}"
    assert all(len(t) == N for t in graphed)
