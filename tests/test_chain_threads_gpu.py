"""Two threads that step the same model at once, each with its own cache and
stream, do not see each other: the fused chain's scratch belongs to a call."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("own_streams", [False, True])
def test_steps_side_by_side(own_streams):
    from ollamamq_amd.engine import LlamaEngine, PagedKVCache
    from ollamamq_amd.models import LlamaModel, PRESETS
    cfg = PRESETS["tiny"]
    model = LlamaModel(cfg, device="cuda:0", dtype=torch.bfloat16, seed=5)
    assert model.fused_chain

    def steps(seed):
        kv = PagedKVCache.for_model(cfg, n_pages=96, max_slots=6, max_ctx=256,
                                    device="cuda:0", dtype=torch.bfloat16)
        eng = LlamaEngine(model, kv, max_batch=4)
        eng.use_graphs = False
        streams = [eng.open_stream() for _ in range(3)]
        return [eng.feed([(s, [(seed + i + j) % 200 for j in range(n)], [0])
                          for s, n in zip(streams, (1, 7 + seed, 20))])
                for i in range(12)]

    want = [steps(0), steps(3)]
    torch.cuda.synchronize()
    got, failed = [None, None], []

    def run(i):
        try:
            stream = torch.cuda.Stream() if own_streams else \
                torch.cuda.default_stream()
            with torch.cuda.stream(stream):
                got[i] = steps(3 * i)
            stream.synchronize()
        except Exception as e:                       # noqa: BLE001
            failed.append(e)

    threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
    for a, b in zip(want, got):
        for x, y in zip(a, b):
            assert torch.equal(x, y)
