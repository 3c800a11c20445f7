"""Tensor-parallel correctness: a TP=2 model (gloo on CPU here; RCCL over
xGMI on the GPU box) must produce the same outputs as the TP=1 model built
from the same seed — the shard-from-full-tensor init guarantees identical
weights (gridllm_amd/models/llama.py _init_weights)."""

import os

import pytest
import torch
import torch.distributed as dist
import torch.multiprocessing as mp

from gridllm_amd.models.registry import get_spec

PORT = 29871


def _tp_worker(rank: int, world: int, port: int, q):
    try:
        dist.init_process_group(
            "gloo", init_method=f"tcp://127.0.0.1:{port}",
            rank=rank, world_size=world)
        from gridllm_amd.models.llama import LlamaModel
        from gridllm_amd.parallel.tp import TPContext
        tp = TPContext(rank=rank, size=world, group=None)
        spec = get_spec("tiny")
        model = LlamaModel(spec, device="cpu", dtype="fp32", tp=tp, seed=7,
                           kv_slots=4, max_seq=64)
        tokens = torch.arange(10, dtype=torch.int64) % spec.vocab
        slot = model.cache.alloc()
        logits = model.forward_prefill(tokens, slot)
        # a few decode steps
        decs = []
        for t in [3, 5, 7]:
            lg = model.forward_decode(
                torch.tensor([t], dtype=torch.int64),
                torch.tensor([slot], dtype=torch.int32))
            decs.append(lg[0])
        # context shift is per-rank-deterministic: each rank slides its own
        # KV shard; decode afterwards must still match TP=1
        model.shift_slot(slot)
        lg = model.forward_decode(torch.tensor([9], dtype=torch.int64),
                                  torch.tensor([slot], dtype=torch.int32))
        decs.append(lg[0])
        if rank == 0:
            q.put(("ok", logits.detach().tolist(), torch.stack(decs).detach().tolist()))
        dist.destroy_process_group()
    except Exception as e:  # noqa: BLE001
        import traceback
        if rank == 0:
            q.put(("err", traceback.format_exc(), None))


def _single():
    from gridllm_amd.models.llama import LlamaModel
    spec = get_spec("tiny")
    model = LlamaModel(spec, device="cpu", dtype="fp32", seed=7,
                       kv_slots=4, max_seq=64)
    tokens = torch.arange(10, dtype=torch.int64) % spec.vocab
    slot = model.cache.alloc()
    logits = model.forward_prefill(tokens, slot)
    decs = []
    for t in [3, 5, 7]:
        lg = model.forward_decode(torch.tensor([t], dtype=torch.int64),
                                  torch.tensor([slot], dtype=torch.int32))
        decs.append(lg[0])
    model.shift_slot(slot)
    lg = model.forward_decode(torch.tensor([9], dtype=torch.int64),
                              torch.tensor([slot], dtype=torch.int32))
    decs.append(lg[0])
    return logits, torch.stack(decs)


def test_tp2_matches_tp1():
    os.environ.setdefault("MASTER_ADDR", "127.0.0.1")
    ctx = mp.get_context("spawn")
    q = ctx.SimpleQueue()
    procs = [ctx.Process(target=_tp_worker, args=(r, 2, PORT, q))
             for r in range(2)]
    for p in procs:
        p.start()
    status, logits_tp, decs_tp = q.get()
    for p in procs:
        p.join(timeout=120)
    assert status == "ok", f"TP worker failed:\n{logits_tp}"
    logits_tp = torch.tensor(logits_tp)
    decs_tp = torch.tensor(decs_tp)
    logits_1, decs_1 = _single()
    assert torch.allclose(logits_tp, logits_1, atol=1e-3), \
        (logits_tp - logits_1).abs().max()
    assert torch.allclose(decs_tp, decs_1, atol=1e-3), \
        (decs_tp - decs_1).abs().max()


def _tp_serve_worker(rank: int, world: int, port: int, q):
    try:
        dist.init_process_group(
            "gloo", init_method=f"tcp://127.0.0.1:{port}",
            rank=rank, world_size=world)
        from gridllm_amd.config import EngineConfig
        from gridllm_amd.engine.engine import InferenceEngine
        from gridllm_amd.parallel.tp import TPContext
        from gridllm_amd.worker.tp_runner import TPBatcher, follower_loop
        tp = TPContext(rank=rank, size=world, group=None)
        eng = InferenceEngine(EngineConfig(
            model="tiny", device="cpu", dtype="fp32", max_seq_len=128,
            max_batch_size=4, use_hipgraph=False, seed=7), tp=tp)
        if rank == 0:
            batcher = TPBatcher(eng, tp)
            fut = batcher.submit_generate(
                "hello tp", {"temperature": 0.0, "num_predict": 5})
            res = fut.result(timeout=120)
            fut2 = batcher.submit_embedding(["vec me"])
            emb = fut2.result(timeout=120)
            batcher.shutdown()
            q.put(("ok", res.token_ids, emb[0][:4]))
        else:
            follower_loop(eng, tp)
        dist.destroy_process_group()
    except Exception:  # noqa: BLE001
        import traceback
        if rank == 0:
            q.put(("err", traceback.format_exc(), None))


def test_tp_serving_wave_matches_single():
    ctx = mp.get_context("spawn")
    q = ctx.SimpleQueue()
    procs = [ctx.Process(target=_tp_serve_worker, args=(r, 2, PORT + 1, q))
             for r in range(2)]
    for p in procs:
        p.start()
    status, tokens_tp, emb_tp = q.get()
    for p in procs:
        p.join(timeout=180)
    assert status == "ok", f"TP serving failed:\n{tokens_tp}"
    # single-rank reference with the same engine seed
    from gridllm_amd.config import EngineConfig
    from gridllm_amd.engine.engine import InferenceEngine
    eng = InferenceEngine(EngineConfig(
        model="tiny", device="cpu", dtype="fp32", max_seq_len=128,
        max_batch_size=4, use_hipgraph=False, seed=7))
    ref = eng.generate("hello tp", {"temperature": 0.0, "num_predict": 5})
    assert tokens_tp == ref.token_ids
    emb_ref = eng.embed(["vec me"])[0][:4]
    assert all(abs(a - b) < 1e-3 for a, b in zip(emb_tp, emb_ref))


def _tp_cancel_worker(rank: int, world: int, port: int, q):
    try:
        dist.init_process_group(
            "gloo", init_method=f"tcp://127.0.0.1:{port}",
            rank=rank, world_size=world)
        import threading
        from gridllm_amd.config import EngineConfig
        from gridllm_amd.engine.engine import InferenceEngine
        from gridllm_amd.parallel.tp import TPContext
        from gridllm_amd.worker.tp_runner import TPBatcher, follower_loop
        tp = TPContext(rank=rank, size=world, group=None)
        eng = InferenceEngine(EngineConfig(
            model="tiny", device="cpu", dtype="fp32", max_seq_len=128,
            max_batch_size=4, use_hipgraph=False, seed=7), tp=tp)
        if rank == 0:
            batcher = TPBatcher(eng, tp)
            cancel = threading.Event()
            # cancel as soon as the first token streams out — deterministic
            # mid-generation cancel regardless of host speed; the decision
            # must reach every rank through the engine's cancel broadcast
            fut = batcher.submit_generate(
                "long generation", {"temperature": 0.0, "num_predict": 100},
                on_token=lambda piece, done: cancel.set(),
                cancel=cancel)
            res = fut.result(timeout=120)
            batcher.shutdown()
            q.put(("ok", res.cancelled, len(res.token_ids)))
        else:
            follower_loop(eng, tp)
        dist.destroy_process_group()
    except Exception:  # noqa: BLE001
        import traceback
        if rank == 0:
            q.put(("err", traceback.format_exc(), None))


def test_tp_cancellation_is_synchronized():
    """Cancel mid-generation under TP: rank 0 observes the client cancel
    and BROADCASTS the decision so all ranks retire the row on the same
    step (engine._sync_cancel) — a rank-local check would desync the
    collectives."""
    ctx = mp.get_context("spawn")
    q = ctx.SimpleQueue()
    procs = [ctx.Process(target=_tp_cancel_worker, args=(r, 2, PORT + 2, q))
             for r in range(2)]
    for p in procs:
        p.start()
    status, cancelled, ntok = q.get()
    for p in procs:
        p.join(timeout=180)
    assert status == "ok", f"TP cancel failed:\n{cancelled}"
    assert cancelled is True
    assert ntok < 100, ntok        # stopped early


def _tp_interleave_worker(rank: int, world: int, port: int, q):
    try:
        dist.init_process_group(
            "gloo", init_method=f"tcp://127.0.0.1:{port}",
            rank=rank, world_size=world)
        import threading
        import time as _t
        from gridllm_amd.config import EngineConfig
        from gridllm_amd.engine.engine import InferenceEngine
        from gridllm_amd.parallel.tp import TPContext
        from gridllm_amd.worker.tp_runner import TPBatcher, follower_loop
        tp = TPContext(rank=rank, size=world, group=None)
        eng = InferenceEngine(EngineConfig(
            model="tiny", device="cpu", dtype="fp32", max_seq_len=128,
            max_batch_size=4, use_hipgraph=False, seed=7), tp=tp)
        if rank == 0:
            batcher = TPBatcher(eng, tp)
            order = []
            started = threading.Event()
            long_fut = batcher.submit_generate(
                "long one", {"temperature": 0.0, "num_predict": 60},
                on_token=lambda p, d: (started.set(),
                                       order.append("L") if d else None))
            assert started.wait(timeout=60)
            _t.sleep(0.05)       # long generation is mid-decode now
            short_fut = batcher.submit_generate(
                "quick", {"temperature": 0.0, "num_predict": 3},
                on_token=lambda p, d: order.append("S") if d else None)
            short_fut.result(timeout=120)
            long_fut.result(timeout=120)
            batcher.shutdown()
            q.put(("ok", order.index("S") < order.index("L"), order))
        else:
            follower_loop(eng, tp)
        dist.destroy_process_group()
    except Exception:  # noqa: BLE001
        import traceback
        if rank == 0:
            q.put(("err", traceback.format_exc(), None))


def test_tp_continuous_batching_interleaves():
    """A short request submitted while a long one is mid-decode under TP
    must JOIN the live batch and finish first,
    not wait for whole waves to complete."""
    ctx = mp.get_context("spawn")
    q = ctx.SimpleQueue()
    procs = [ctx.Process(target=_tp_interleave_worker,
                         args=(r, 2, PORT + 3, q))
             for r in range(2)]
    for p in procs:
        p.start()
    status, short_first, order = q.get()
    for p in procs:
        p.join(timeout=180)
    assert status == "ok", f"TP interleave failed:\n{short_first}"
    assert short_first, order


def _tp_forced_trace(eng, steps: int = 16):
    """Prefill a fixed prompt, then decode a FIXED token sequence;
    return per-step top-3 (ids, values). Deterministic on both the TP
    and the TP=1 engine — no argmax involved, so bf16 all-reduce
    rounding cannot flip the comparison (greedy-token identity was
    measured flaky across boxes: near-ties on random-init logits,
    profiles/r02_logs/r02ar discussion)."""
    import torch
    toks = eng.tokenizer.encode("tensor parallel on one device")
    m = eng.model
    slot = m.cache.alloc()
    dev = eng.device
    out = []
    logits = m.forward_prefill(
        torch.tensor(toks, dtype=torch.int64, device=dev), slot)
    forced = [(1009 * (i + 3)) % eng.spec.vocab for i in range(steps)]
    for t in forced:
        v, ix = logits.float().flatten().topk(3)
        out.append((ix.tolist(), [round(x, 4) for x in v.tolist()]))
        logits = m.forward_decode(
            torch.tensor([t], dtype=torch.int64, device=dev),
            torch.tensor([slot], dtype=torch.int32, device=dev))
    return out


def _tp_gpu_worker(rank: int, world: int, port: int, q):
    try:
        dist.init_process_group(
            "gloo", init_method=f"tcp://127.0.0.1:{port}",
            rank=rank, world_size=world)
        from gridllm_amd.config import EngineConfig
        from gridllm_amd.engine.engine import InferenceEngine
        from gridllm_amd.parallel.tp import TPContext
        tp = TPContext(rank=rank, size=world, group=None)
        # BOTH ranks share cuda:0 (single-lease validation): gloo carries
        # the collectives host-side, so the RCCL one-rank-per-device rule
        # does not apply; numerics and lockstep are what's tested
        eng = InferenceEngine(EngineConfig(
            model="llama3.2:1b", device="cuda:0", dtype="bf16",
            max_seq_len=256, max_batch_size=4, use_hipgraph=False,
            autotune=False, seed=11), tp=tp)
        # both ranks run the IDENTICAL forced sequence; the in-model
        # collectives keep them in lockstep — no broadcast needed
        trace = _tp_forced_trace(eng)
        if rank == 0:
            q.put(("ok", trace, None))
        dist.destroy_process_group()
    except Exception:  # noqa: BLE001
        import traceback
        if rank == 0:
            q.put(("err", traceback.format_exc(), None))


@pytest.mark.gpu
def test_tp2_gpu_logits_match_tp1():
    """TP=2 on ONE MI355X (2 procs, gloo collectives, shared cuda:0):
    per-step logits of a forced-token decode must match the TP=1 engine
    within bf16 all-reduce tolerance — the TP shard math runs the REAL
    HIP kernels on both ranks. Top-1 id must agree wherever the TP=1 margin is clear."""
    import torch as _t
    if not _t.cuda.is_available():
        pytest.skip("GPU required")
    ctx = mp.get_context("spawn")
    q = ctx.SimpleQueue()
    procs = [ctx.Process(target=_tp_gpu_worker, args=(r, 2, PORT + 4, q))
             for r in range(2)]
    for p in procs:
        p.start()
    status, trace_tp, _ = q.get()
    for p in procs:
        p.join(timeout=600)
    assert status == "ok", f"TP2-on-GPU failed:\n{trace_tp}"
    from gridllm_amd.config import EngineConfig
    from gridllm_amd.engine.engine import InferenceEngine
    eng = InferenceEngine(EngineConfig(
        model="llama3.2:1b", device="cuda:0", dtype="bf16",
        max_seq_len=256, max_batch_size=4, use_hipgraph=False,
        autotune=False, seed=11))
    trace_ref = _tp_forced_trace(eng)
    assert len(trace_tp) == len(trace_ref)
    for s, ((ids_tp, vs_tp), (ids_r, vs_r)) in enumerate(
            zip(trace_tp, trace_ref)):
        margin = vs_r[0] - vs_r[1]
        if margin > 0.10:              # clear winner: id must agree
            assert ids_tp[0] == ids_r[0], (s, ids_tp, ids_r, vs_tp, vs_r)
        assert abs(vs_tp[0] - vs_r[0]) <= 0.05 + 0.02 * abs(vs_r[0]), \
            (s, vs_tp, vs_r)
