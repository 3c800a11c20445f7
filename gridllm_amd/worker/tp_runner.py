"""Tensor-parallel worker: a TP group registers as ONE worker.

Launch with torch.distributed.run --nproc-per-node <TP> (one rank per GPU,
RCCL over xGMI). Rank 0 runs the normal WorkerAgent + control-plane
connection; ranks >0 run a follower loop that mirrors rank 0's CONTINUOUS
batching loop: one small control broadcast per decode iteration (gloo side
channel, parallel/tp.py) carries that iteration's admissions, then every
rank executes the identical start_rows/step_rows sequence so all RCCL
collectives line up. Rows join and leave the live batch in lockstep —
a long generation no longer blocks new arrivals (as
broadcasting whole run-to-completion waves would).

The decode step itself is hipGraph-captured per batch bucket INCLUDING
the per-layer all-reduces (engine._graph_ok allows tp>1 on nccl).

No reference analog (the reference had zero parallelism beyond request
sharding).

Determinism across ranks:
  * logits are bitwise-identical on every rank (all-reduced activations,
    replicated lm_head) so sampling matches — PROVIDED every request has a
    seed; rank 0 injects one into any request that lacks it before
    broadcasting the admission.
  * retirement (EOS/stop/length) is a pure function of the sampled tokens,
    so every rank prunes the same rows at the same step; cancellation is
    decided by rank 0 and broadcast per step (engine._sync_cancel).
"""

from __future__ import annotations

import asyncio
import queue as _q
import random
import time as _time

from gridllm_amd.bus.tcp import TcpBus
from gridllm_amd.config import EngineConfig, WorkerConfig
from gridllm_amd.engine.batcher import Batcher, _Pending
from gridllm_amd.engine.engine import InferenceEngine
from gridllm_amd.parallel.tp import TPContext, init_tp_from_env
from gridllm_amd.utils.logging import get_logger
from gridllm_amd.worker.agent import WorkerAgent

log = get_logger("tp-runner")


def _inject_seeds(items: list[tuple]) -> None:
    for _, opts, *_ in items:
        if opts.get("seed") is None:
            opts["seed"] = random.randint(0, 2**31 - 1)


class TPBatcher(Batcher):
    """Rank-0 continuous batcher: each loop iteration broadcasts a compact
    control message (admissions + embed inputs + stop flag) to followers,
    then all ranks run the identical admission/step."""

    def __init__(self, engine: InferenceEngine, tp: TPContext,
                 admit_per_step: int = 32):
        self.tp = tp
        super().__init__(engine, continuous=False,
                         admit_per_step=admit_per_step)

    # Batcher.__init__ starts _loop (wave mode) when continuous is False;
    # override the thread target selection by overriding _loop itself.
    def _loop(self) -> None:
        self._loop_tp()

    def _loop_tp(self) -> None:
        max_batch = max(1, self.engine.cfg.max_batch_size)
        live: list[tuple[_Pending, object]] = []   # (pending, engine row)
        while True:
            # progress stamp for the TP wedge watchdog (agent heartbeat
            # checks it): a hung collective blocks THIS thread while the
            # asyncio loop keeps heartbeating — without the stamp the
            # scheduler would keep routing jobs to a wedged group
            # (group failover must be atomic)
            self.last_progress = _time.monotonic()
            self.busy = bool(live)
            arrivals: list[_Pending] = []
            if not live:
                # idle: block (followers are parked in their broadcast)
                try:
                    arrivals.append(self.q.get(timeout=0.5))
                except _q.Empty:
                    if self._stop.is_set():
                        self._broadcast_iter([], [], stop=True)
                        return
                    continue
            while (len(live) + len(arrivals) < max_batch
                   and len(arrivals) < self.admit_per_step
                   and self.engine.model.cache.n_free > len(arrivals) + 1):
                try:
                    arrivals.append(self.q.get_nowait())
                except _q.Empty:
                    break
            stop_now = False
            gens: list[_Pending] = []
            embeds: list[_Pending] = []
            for p in arrivals:
                if p.kind == "__stop__":
                    stop_now = True
                elif p.kind == "embedding":
                    embeds.append(p)
                else:
                    gens.append(p)
            items = []
            ok_gens = []
            for p in gens:
                try:
                    prompt, opts = self._prep(p)
                except Exception as e:  # noqa: BLE001 — malformed
                    if not p.future.done():   # request: fail it alone
                        p.future.set_exception(e)
                    continue
                ok_gens.append(p)
                items.append((prompt, opts))
            gens = ok_gens
            _inject_seeds(items)
            embed_inputs = [p.inputs or [] for p in embeds]
            self._broadcast_iter(items, embed_inputs,
                                 stop=stop_now and not live and not gens)
            if stop_now and not live and not gens:
                for p in embeds:
                    p.future.set_exception(RuntimeError("batcher shut down"))
                return
            # ---- identical execution on every rank -----------------------
            if embeds:
                flat = [x for ins in embed_inputs for x in ins]
                try:
                    vecs = self.engine.embed(flat)
                    k = 0
                    for p in embeds:
                        n = len(p.inputs or [])
                        p.future.set_result(vecs[k:k + n])
                        k += n
                except Exception as e:  # noqa: BLE001
                    for p in embeds:
                        if not p.future.done():
                            p.future.set_exception(e)
            if items:
                try:
                    new_rows = self.engine.start_rows(
                        [(pr, op, p.on_token, p.cancel, None)
                         for (pr, op), p in zip(items, gens)])
                except Exception as e:  # noqa: BLE001
                    log.logger.exception("TP admission failed")
                    for p in gens:
                        p.future.set_exception(e)
                    new_rows = []
                for p, row in zip(gens, new_rows):
                    if row.done:
                        p.future.set_result(row.result)
                    else:
                        live.append((p, row))
            if live:
                try:
                    self.engine.step_rows([row for _, row in live])
                except Exception as e:  # noqa: BLE001
                    log.logger.exception("TP decode step failed")
                    self.engine.abort_rows([row for _, row in live])
                    for p, _ in live:
                        if not p.future.done():
                            p.future.set_exception(e)
                    live = []
                still = []
                for p, row in live:
                    if row.done:
                        p.future.set_result(row.result)
                    else:
                        still.append((p, row))
                live = still
            if self._stop.is_set() and not live:
                self._broadcast_iter([], [], stop=True)
                return

    def _broadcast_iter(self, items, embed_inputs, stop: bool) -> None:
        self.tp.bcast_obj(("it", items, embed_inputs, stop), src=0)

    def shutdown(self) -> None:
        self._stop.set()
        self.q.put(_Pending(kind="__stop__"))
        self._thread.join(timeout=10.0)


def follower_loop(engine: InferenceEngine, tp: TPContext) -> None:
    """Ranks >0: mirror rank 0's continuous loop. One control broadcast
    per iteration; rows retire by the same deterministic rules."""
    rows: list = []
    while True:
        kind, items, embed_inputs, stop = tp.bcast_obj(None, src=0)
        assert kind == "it"
        if embed_inputs:
            flat = [x for ins in embed_inputs for x in ins]
            try:
                engine.embed(flat)
            except Exception:  # noqa: BLE001
                log.logger.exception("follower embed failed")
        if items:
            try:
                new_rows = engine.start_rows(
                    [(pr, op, None, None, None) for pr, op in items])
                rows.extend(r for r in new_rows if not r.done)
            except Exception:  # noqa: BLE001
                log.logger.exception("follower admission failed")
        if rows:
            try:
                rows = engine.step_rows(rows)
            except Exception:  # noqa: BLE001
                log.logger.exception("follower step failed")
                engine.abort_rows(rows)
                rows = []
        if stop:
            return


async def _run_rank0(wcfg: WorkerConfig, engine: InferenceEngine,
                     tp: TPContext) -> None:
    bus = TcpBus(wcfg.bus_host, wcfg.bus_port)
    await bus.connect()
    batcher = TPBatcher(engine, tp)
    agent = WorkerAgent(bus, engine, wcfg, batcher=batcher)
    await agent.start()
    await asyncio.Event().wait()   # serve forever


def main() -> None:
    import os
    import torch
    tp = init_tp_from_env()
    wcfg = WorkerConfig.from_env()
    ecfg = EngineConfig.from_env()
    local_rank = int(os.environ.get("LOCAL_RANK", tp.rank))
    if torch.cuda.is_available():
        ecfg.device = f"cuda:{local_rank}"
    ecfg.tp_degree = tp.size
    engine = InferenceEngine(ecfg, tp=tp)
    if tp.rank == 0:
        wcfg.worker_id = wcfg.worker_id or f"tp-worker-{os.getpid()}"
        asyncio.run(_run_rank0(wcfg, engine, tp))
    else:
        follower_loop(engine, tp)


if __name__ == "__main__":
    main()
