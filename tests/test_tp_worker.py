"""TP worker group lockstep on CPU/gloo: rank 0 serves, both ranks step the
same engine replica; generated tokens must match the single-rank engine."""
import os

import torch
import torch.multiprocessing as mp

from ollamamq_amd.engine import GenParams

PROMPT = [3, 1, 4, 1, 5, 9]
N = 5


def _single():
    from ollamamq_amd.models import LlamaModel, PRESETS
    from ollamamq_amd.engine import LlamaEngine, PagedKVCache
    cfg = PRESETS["tiny"]
    model = LlamaModel(cfg, device="cpu", dtype=torch.float32, seed=1234)
    kv = PagedKVCache.for_model(cfg, n_pages=32, max_slots=4, max_ctx=128)
    eng = LlamaEngine(model, kv, max_batch=4)
    sid = eng.submit(PROMPT, GenParams(max_tokens=N))
    seq = eng.seqs[sid]
    for _ in range(64):
        eng.step()
        if not eng.has_work():
            break
    return seq.generated


def _rank(rank, world, port, q):
    os.environ["MASTER_ADDR"] = "127.0.0.1"
    os.environ["MASTER_PORT"] = str(port)
    import torch.distributed as dist
    from ollamamq_amd.engine.tp_worker import TPWorker
    dist.init_process_group("gloo", rank=rank, world_size=world)
    w = TPWorker(rank, world, 0, max_batch=4, default_ctx=128)
    if rank == 0:
        err = w.load("tiny", 128)
        assert err is None, err
        toks = []
        import threading
        done = threading.Event()

        def on_token(t, fin):
            if fin:
                done.set()
            else:
                toks.append(t)

        w.generate("tiny", PROMPT,
                   GenParams(max_tokens=N), on_token)
        assert done.wait(timeout=120)
        q.put(toks)
    else:
        # follower: the engine loop thread does the work; idle here until
        # the parent kills the process
        import time
        time.sleep(120)


def test_tp_worker_lockstep_matches_single():
    expected = _single()
    ctx = mp.get_context("spawn")
    q = ctx.Queue()
    procs = [ctx.Process(target=_rank, args=(r, 2, 29587, q), daemon=True)
             for r in range(2)]
    for p in procs:
        p.start()
    toks = q.get(timeout=300)
    for p in procs:
        p.terminate()
        p.join(timeout=30)
    assert toks == expected, f"{toks} != {expected}"


def _rank_uds(rank, world, port, sock_path, q):
    """Rank 0 serves the REAL UDS wire (worker.serve + Conn), exercising
    Conn._request -> TPWorker.generate(..., num_ctx=...) and the
    keep_alive:0 -> unload(only_if_idle=True) path
    (TPWorker signatures must match worker.Worker's)."""
    os.environ["MASTER_ADDR"] = "127.0.0.1"
    os.environ["MASTER_PORT"] = str(port)
    import json
    import socket
    import threading
    import time
    import torch.distributed as dist
    from ollamamq_amd.engine.tp_worker import TPWorker
    from ollamamq_amd.engine import worker as worker_mod
    dist.init_process_group("gloo", rank=rank, world_size=world)
    w = TPWorker(rank, world, 0, max_batch=4, default_ctx=128)
    if rank != 0:
        time.sleep(120)
        return
    threading.Thread(target=worker_mod.serve, args=(sock_path, w),
                     daemon=True).start()
    for _ in range(100):
        if os.path.exists(sock_path):
            break
        time.sleep(0.05)

    def req(body):
        c = socket.socket(socket.AF_UNIX, socket.SOCK_STREAM)
        c.connect(sock_path)
        c.sendall((json.dumps({"cmd": "request", "method": "POST",
                               "path": "/api/generate",
                               "body": json.dumps(body)}) + "\n").encode())
        data = b""
        while True:
            chunk = c.recv(65536)
            if not chunk:
                break
            data += chunk
        c.close()
        return data.decode()

    # num_ctx flows through generate(..., num_ctx=96) into the on-demand
    # load; keep_alive:0 triggers unload(only_if_idle=True) after the
    # response — both raise TypeError if the TP signatures drift again
    out = req({"model": "tiny", "prompt": "hi",
               "options": {"num_ctx": 96, "num_predict": 3},
               "keep_alive": 0, "stream": False})
    lines = [json.loads(l) for l in out.splitlines() if l.strip()]
    assert lines[0]["status"] == 200, out
    assert lines[-1].get("done") is True, out
    # keep_alive:0 + idle engine => model was unloaded on all ranks
    deadline = time.time() + 10
    while time.time() < deadline and "tiny" in w.engines:
        time.sleep(0.05)
    q.put(("ok", "tiny" not in w.engines))


def test_tp_worker_uds_wire_and_keepalive_unload():
    ctx = mp.get_context("spawn")
    q = ctx.Queue()
    sock = f"/tmp/omq_tp_test_{os.getpid()}.sock"
    procs = [ctx.Process(target=_rank_uds, args=(r, 2, 29591, sock, q),
                         daemon=True) for r in range(2)]
    for p in procs:
        p.start()
    tag, unloaded = q.get(timeout=300)
    for p in procs:
        p.terminate()
        p.join(timeout=30)
    try:
        os.unlink(sock)
    except FileNotFoundError:
        pass
    assert tag == "ok"
    assert unloaded, "keep_alive:0 did not unload the idle model"


def _rank_storm(rank, world, port, q):
    """Lockstep under concurrent load: 4 parallel generates on one model
    interleaved with a load+unload of a SECOND model mid-flight.  The
    op-stream broadcast and SYNC_EVERY cadence must neither deadlock nor
    diverge; every generate completes with its full token budget."""
    os.environ["MASTER_ADDR"] = "127.0.0.1"
    os.environ["MASTER_PORT"] = str(port)
    import threading
    import time
    import torch.distributed as dist
    from ollamamq_amd.engine.tp_worker import TPWorker
    dist.init_process_group("gloo", rank=rank, world_size=world)
    w = TPWorker(rank, world, 0, max_batch=4, default_ctx=128)
    if rank != 0:
        time.sleep(180)
        return
    assert w.load("tiny", 128) is None
    counts = [0] * 4
    dones = [threading.Event() for _ in range(4)]

    def fire(i):
        def on_token(t, fin):
            if fin:
                dones[i].set()
            else:
                counts[i] += 1
        w.generate("tiny", [i + 1, 2, 3], GenParams(max_tokens=6 + i),
                   on_token)

    for i in range(2):
        fire(i)
    # mid-flight control ops on another model
    assert w.load("nano", 64) is None
    for i in range(2, 4):
        fire(i)
    assert w.unload("nano") is None
    for i, d in enumerate(dones):
        assert d.wait(timeout=120), f"generate {i} never finished"
    q.put(counts)


def test_tp_lockstep_concurrent_ops_storm():
    ctx = mp.get_context("spawn")
    q = ctx.Queue()
    procs = [ctx.Process(target=_rank_storm, args=(r, 2, 29593, q),
                         daemon=True) for r in range(2)]
    for p in procs:
        p.start()
    counts = q.get(timeout=300)
    for p in procs:
        p.terminate()
        p.join(timeout=30)
    assert counts == [6, 7, 8, 9], counts
