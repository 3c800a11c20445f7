"""Worker agent: registers a GPU (or TP group) with the control plane and
executes assigned jobs on the in-process engine.

Reimplements the live worker path of the reference
(reference: client/src/services/WorkerClientService.ts):
  * register: hset workers + publish worker:registered (:175-206)
  * subscribe worker:<id>:job + worker:<id>:reregister (:208-227)
  * heartbeat every 5 s: publish + TTL key at 2x interval (:311-353)
  * resource/capability refresh with change-only status publish (:355-440)
  * job execution dispatched on request_type, streaming chunks published
    per chunk to job:stream:<id>, completion to job:completed AND
    job:result:<id> (:497-712)
Fixes over the reference:
  * job_cancellation is HONORED (the reference ignored it, :483-491) —
    the engine's cancel event aborts generation mid-decode.
  * concurrent jobs are coalesced into one batched decode (engine/batcher).
  * the engine is in-process — no Ollama HTTP hop, no per-token JSON chain.
"""

from __future__ import annotations

import asyncio
import json
import socket
import threading
import time
from typing import Optional

from gridllm_amd.bus.base import Bus
from gridllm_amd.config import WorkerConfig
from gridllm_amd.engine.batcher import Batcher
from gridllm_amd.engine.engine import GenerationResult, InferenceEngine
from gridllm_amd.types import (Channels, InferenceRequest, Keys,
                               WorkerInfo, WorkerStatus, now_ms)
from gridllm_amd.utils.logging import get_logger
from gridllm_amd.worker import telemetry

log = get_logger("worker")


class _Stream:
    """One streaming job's token buffer, drained by the agent's single
    shared flusher task."""
    __slots__ = ("job_id", "buf", "lk", "done_ev", "sent_any", "fin",
                 "splitter", "addr")

    def __init__(self, job_id: str, buf: list, lk: threading.Lock,
                 done_ev: threading.Event, splitter=None, addr=None):
        self.job_id = job_id
        self.buf = buf
        self.lk = lk
        self.done_ev = done_ev
        self.sent_any = False
        self.fin = asyncio.Event()     # set after the final chunk publishes
        self.splitter = splitter       # think mode: thinking/content split
        self.addr = addr               # direct gateway addr (bus/stream.py)


class WorkerAgent:
    def __init__(self, bus: Bus, engine: InferenceEngine,
                 cfg: Optional[WorkerConfig] = None,
                 batcher: Optional[Batcher] = None,
                 extra_engines: Optional[list[InferenceEngine]] = None):
        """One worker can serve SEVERAL models (the reference advertised
        Ollama's whole tag list, WorkerClientService.ts:129-154): pass
        extra_engines and jobs dispatch to the engine whose model matches.
        Each engine gets its own continuous batcher."""
        self.bus = bus
        self.engine = engine
        self.cfg = cfg or WorkerConfig()
        self.worker_id = self.cfg.worker_id or \
            f"worker-{socket.gethostname()}-{self.cfg.device}"
        self.batcher = batcher or Batcher(engine)
        # model name (incl. aliases) -> (engine, batcher)
        self._by_model: dict[str, tuple[InferenceEngine, Batcher]] = {}
        for name in engine.model_names():
            self._by_model[name] = (engine, self.batcher)
        self._extra_batchers: list[Batcher] = []
        for eng in (extra_engines or []):
            b = Batcher(eng)
            self._extra_batchers.append(b)
            for name in eng.model_names():
                self._by_model.setdefault(name, (eng, b))
        self.current_jobs = 0
        self._cancel_events: dict[str, threading.Event] = {}
        self._streams: dict[str, "_Stream"] = {}
        from gridllm_amd.bus.stream import StreamSink
        self._sink = StreamSink()      # direct worker->gateway chunk plane
        self._flush_task: Optional[asyncio.Task] = None
        self._flush_wake = asyncio.Event()
        self._tasks: list[asyncio.Task] = []
        self._job_tasks: set[asyncio.Task] = set()
        self._last_status: tuple = ()
        self.stream_drops = 0          # chunk publishes swallowed (at-most-
                                       # once streaming; result path owns
                                       # delivery) — surfaced in telemetry
        self._started = False
        self.paused = False
        self.draining = False

    # ------------------------------------------------------------- lifecycle

    async def start(self) -> None:
        await self.bus.identify(self.worker_id)
        # subscribe BEFORE announcing registration: the bus processes this
        # connection's frames in order and the scheduler only assigns
        # after it sees worker:registered, so the job channel is always
        # live by then. The reverse order LOST whole assignment bursts:
        # a respawned worker with a queued backlog was re-registered and
        # immediately assigned 16 jobs into the subscription gap — they
        # sat "active" on a live idle worker until the job timeout.
        await self.bus.subscribe(Channels.worker_job(self.worker_id),
                                 self._h_job_msg)
        await self.bus.subscribe(Channels.worker_reregister(self.worker_id),
                                 self._h_reregister)
        await self.bus.subscribe(Channels.worker_control(self.worker_id),
                                 self._h_control)
        await self.bus.subscribe(Channels.BROADCAST, self._h_control)
        await self._register()
        loop = asyncio.get_running_loop()
        self._tasks.append(loop.create_task(self._heartbeat_loop()))
        self._tasks.append(loop.create_task(self._resource_loop()))
        self._started = True
        log.worker("worker started", worker_id=self.worker_id,
                   models=self.engine.model_names())

    async def stop(self) -> None:
        for t in self._tasks:
            t.cancel()
        self._tasks.clear()
        for ev in self._cancel_events.values():
            ev.set()
        try:
            await self.bus.publish(Channels.WORKER_UNREGISTERED,
                                   {"workerId": self.worker_id})
        except Exception:  # noqa: BLE001
            pass
        self.batcher.shutdown()
        for b in self._extra_batchers:
            b.shutdown()
        await self._sink.close()

    def _info(self) -> WorkerInfo:
        stats = telemetry.gpu_stats(self.cfg.device)
        if self.paused:
            status = WorkerStatus.PAUSED.value
        elif self.current_jobs >= self.cfg.max_concurrent_tasks:
            status = WorkerStatus.BUSY.value
        else:
            status = WorkerStatus.ONLINE.value
        return WorkerInfo(
            id=self.worker_id,
            status=status,
            models=sorted(self._by_model),
            max_concurrent_jobs=self.cfg.max_concurrent_tasks,
            current_jobs=self.current_jobs,
            performance_tier=telemetry.performance_tier(stats),
            gpu={**stats.to_dict(), "stream_drops": self.stream_drops},
            tp_degree=self.engine.tp.size,
        )

    async def _register(self) -> None:
        info = self._info()
        await self.bus.hset(Keys.WORKERS, self.worker_id,
                            json.dumps(info.to_dict()))
        await self.bus.publish(Channels.WORKER_REGISTERED, info.to_dict())

    async def _h_reregister(self, _ch: str, _payload: dict) -> None:
        log.worker("re-registration requested", worker_id=self.worker_id)
        await self._register()

    # ------------------------------------------------------------ heartbeat

    async def _heartbeat_loop(self) -> None:
        interval = self.cfg.heartbeat_interval_ms / 1000.0
        while True:
            self._check_wedge()
            try:
                await self.bus.publish(Channels.WORKER_HEARTBEAT, {
                    "workerId": self.worker_id,
                    "status": self._info().status,
                    "currentJobs": self.current_jobs,
                    "timestamp": now_ms(),
                })
                await self.bus.kv_set(Keys.heartbeat(self.worker_id),
                                      str(now_ms()),
                                      ttl_ms=self.cfg.heartbeat_interval_ms * 2)
            except Exception:  # noqa: BLE001
                log.logger.warning("heartbeat publish failed")
            await asyncio.sleep(interval)

    def _check_wedge(self) -> None:
        """TP group failover must be atomic: a
        collective that hangs (peer rank dead/stuck) blocks the batcher
        thread while THIS loop keeps heartbeating, so the scheduler would
        keep routing jobs to a wedged group forever. When the batcher has
        had work in flight with no completed iteration for
        tp_wedge_timeout_ms, exit the process: the launcher (torchrun)
        tears down the remaining ranks, heartbeats stop, and orphan
        recovery requeues the jobs on live workers. TP-only — a
        single-process engine stall is a GPU hang with its own handling."""
        timeout_s = getattr(self.cfg, "tp_wedge_timeout_ms", 60_000) / 1000.0
        for eng, batcher in self._by_model.values():
            if not eng.tp.enabled:
                continue
            if batcher is not None and hasattr(batcher, "wedged") \
                    and batcher.wedged(timeout_s):
                log.logger.error(
                    "TP batcher wedged >%.0fs with work in flight — "
                    "exiting so the launcher fails the group over", timeout_s)
                self._wedge_exit(13)
                return

    @staticmethod
    def _wedge_exit(code: int) -> None:   # overridable in tests
        import os
        os._exit(code)

    async def _resource_loop(self) -> None:
        interval = self.cfg.resource_monitor_interval_ms / 1000.0
        while True:
            await asyncio.sleep(interval)
            try:
                info = self._info()
                key = (info.status, info.current_jobs, tuple(info.models))
                if key != self._last_status:
                    self._last_status = key
                    await self.bus.publish(Channels.WORKER_STATUS, {
                        "workerId": self.worker_id,
                        "status": info.status,
                        "currentJobs": info.current_jobs,
                        "models": info.models,
                        "gpu": info.gpu,
                    })
            except Exception:  # noqa: BLE001
                log.logger.warning("resource publish failed")

    async def _publish_status(self) -> None:
        info = self._info()
        await self.bus.publish(Channels.WORKER_STATUS, {
            "workerId": self.worker_id, "status": info.status,
            "currentJobs": info.current_jobs,
        })

    # --------------------------------------------------------------- control

    async def _h_control(self, _ch: str, payload: dict) -> None:
        """Maintenance verbs (pause/resume/drain) — adopted from the
        reference's dead broker path (BrokerClientService.ts:568-657)
        onto the live worker."""
        verb = payload.get("type")
        if verb == "pause":
            self.paused = True
            await self._publish_status()
            log.worker("paused", worker_id=self.worker_id)
        elif verb == "resume":
            self.paused = False
            self.draining = False
            await self._publish_status()
            log.worker("resumed", worker_id=self.worker_id)
        elif verb == "drain":
            self.paused = True
            self.draining = True
            await self._publish_status()
            log.worker("draining", worker_id=self.worker_id,
                       in_flight=len(self._job_tasks))
            if self._job_tasks:
                await asyncio.gather(*list(self._job_tasks),
                                     return_exceptions=True)
            await self.bus.publish(Channels.WORKER_UNREGISTERED,
                                   {"workerId": self.worker_id})
            log.worker("drained", worker_id=self.worker_id)

    # ------------------------------------------------------------------ jobs

    async def _h_job_msg(self, _ch: str, payload: dict) -> None:
        mtype = payload.get("type")
        if mtype == "job_assignment":
            req = InferenceRequest.from_dict(payload.get("job") or {})
            if self.paused:
                await self.bus.publish(Channels.JOB_FAILED, {
                    "jobId": req.id, "workerId": self.worker_id,
                    "error": "worker paused"})
                return
            if self.current_jobs >= self.cfg.max_concurrent_tasks:
                # busy rejection (reference :500-505)
                await self.bus.publish(Channels.JOB_FAILED, {
                    "jobId": req.id, "workerId": self.worker_id,
                    "error": "worker busy"})
                return
            self.current_jobs += 1
            await self._publish_status()
            t = asyncio.get_running_loop().create_task(self._run_job(req))
            self._job_tasks.add(t)
            t.add_done_callback(self._job_tasks.discard)
        elif mtype == "job_cancellation":
            jid = payload.get("jobId", "")
            ev = self._cancel_events.get(jid)
            if ev is not None:
                ev.set()
                log.job("job cancellation honored", job_id=jid)
        else:
            log.logger.warning(f"unknown job message type {mtype!r}")

    async def _run_job(self, req: InferenceRequest) -> None:
        loop = asyncio.get_running_loop()
        cancel = threading.Event()
        self._cancel_events[req.id] = cancel
        t_start = time.monotonic_ns()

        # Token hand-off: the engine's batcher THREAD appends to a plain
        # buffer under a lock; the asyncio pump POLLS it every
        # stream_flush_ms. A per-token call_soon_threadsafe wakeup (the
        # obvious design) costs a loop wakeup + GIL bounce per token —
        # at serving batch sizes that starves the decode thread.
        buf: list[str] = []
        lk = threading.Lock()
        done_ev = threading.Event()

        def on_token(piece: str, done: bool) -> None:
            if piece:
                with lk:
                    buf.append(piece)
            if done:
                done_ev.set()

        # thinking mode (Ollama `think: true`, reference forwards it at
        # server/src/routes/ollama.ts:216-239;
        # executed here, not silently ignored)
        think = bool((req.metadata or {}).get("think"))
        stream = None
        if req.stream:
            from gridllm_amd.engine import chat as chat_mod
            stream = self._register_stream(
                req.id, buf, lk, done_ev,
                splitter=chat_mod.ThinkSplitter() if think else None,
                addr=(req.metadata or {}).get("streamAddr"))
        try:
            pair = self._by_model.get(req.model)
            if pair is None:
                raise RuntimeError(
                    f"model {req.model!r} not served by this worker "
                    f"(has: {sorted(self._by_model)})")
            engine, batcher = pair
            # Ollama conversation continuation: `context` carries the prior
            # exchange's token ids; prepend their text to the prompt
            # (byte tokenizer -> exact roundtrip)
            ctx_ids = (req.metadata or {}).get("context")
            if ctx_ids and req.request_type != "embedding":
                try:
                    prefix = engine.tokenizer.decode(
                        [int(t) for t in ctx_ids])
                    req.prompt = prefix + req.prompt
                except Exception:  # noqa: BLE001
                    pass
            if req.request_type == "embedding":
                inputs = req.input if req.input is not None else [req.prompt]
                fut = batcher.submit_embedding(inputs)
                embeddings = await asyncio.wrap_future(fut)
                payload = {
                    "jobId": req.id, "workerId": self.worker_id, "done": True,
                    "model": req.model, "embeddings": embeddings,
                    "timings": {"total_duration": time.monotonic_ns() - t_start},
                }
            else:
                if req.request_type == "chat" and req.messages:
                    fut = batcher.submit_chat(
                        req.messages, req.options,
                        on_token=on_token if req.stream else None,
                        cancel=cancel, think=think)
                else:
                    if think:
                        from gridllm_amd.engine import chat as chat_mod
                        req.prompt = req.prompt + chat_mod.THINK_OPEN + "\n"
                    fut = batcher.submit_generate(
                        req.prompt, req.options,
                        on_token=on_token if req.stream else None,
                        cancel=cancel)
                result: GenerationResult = await asyncio.wrap_future(fut)
                thinking = None
                response_text = result.text
                if think:
                    from gridllm_amd.engine import chat as chat_mod
                    thinking, response_text = chat_mod.split_think(result.text)
                payload = {
                    "jobId": req.id, "workerId": self.worker_id, "done": True,
                    "model": req.model,
                    "response": response_text,
                    "done_reason": result.done_reason,
                    "cancelled": result.cancelled,
                    # Ollama context = ids encoding the WHOLE conversation
                    # (req.prompt already carries the decoded prior context)
                    "context": engine.tokenizer.encode(
                        req.prompt + result.text, bos=False)
                    if req.request_type != "chat" else [],
                    "timings": {
                        "total_duration": result.total_duration,
                        "load_duration": 0,
                        "prompt_eval_count": result.prompt_eval_count,
                        "prompt_eval_duration": result.prompt_eval_duration,
                        "eval_count": result.eval_count,
                        "eval_duration": result.eval_duration,
                    },
                }
                if thinking is not None:
                    payload["thinking"] = thinking
                if req.request_type == "chat":
                    payload["message"] = {"role": "assistant",
                                          "content": response_text}
                    if thinking is not None:
                        payload["message"]["thinking"] = thinking
            if stream is not None:
                done_ev.set()                  # flush remaining and stop
                try:                           # flusher sets fin after the
                    await asyncio.wait_for(    # done-chunk publish
                        stream.fin.wait(), timeout=10.0)
                except asyncio.TimeoutError:
                    self._streams.pop(req.id, None)
                stream = None
            await self.bus.publish(Channels.JOB_COMPLETED, {
                "jobId": req.id, "workerId": self.worker_id})
            await self.bus.publish(Channels.job_result(req.id), payload)
            log.job("job completed", job_id=req.id,
                    eval_count=payload.get("timings", {}).get("eval_count", 0))
        except Exception as e:  # noqa: BLE001
            log.logger.exception("job failed")
            err = {"jobId": req.id, "workerId": self.worker_id,
                   "error": str(e), "done": True}
            try:
                await self.bus.publish(Channels.JOB_FAILED, err)
                await self.bus.publish(Channels.job_result(req.id), err)
            except Exception:  # noqa: BLE001
                pass
        finally:
            if stream is not None:             # error path: drop the stream
                self._streams.pop(req.id, None)
            self._cancel_events.pop(req.id, None)
            self.current_jobs = max(0, self.current_jobs - 1)
            try:
                await self._publish_status()
            except Exception:  # noqa: BLE001
                pass

    def _register_stream(self, job_id: str, buf: list, lk: threading.Lock,
                         done_ev: threading.Event, splitter=None,
                         addr=None) -> _Stream:
        s = _Stream(job_id, buf, lk, done_ev, splitter=splitter, addr=addr)
        self._streams[job_id] = s
        self._flush_wake.set()         # break out of a long flush sleep
        if self._flush_task is None or self._flush_task.done():
            self._flush_task = asyncio.get_running_loop().create_task(
                self._flush_loop())
        return s

    async def _flush_loop(self) -> None:
        """Publish token chunks to job:stream:<id> (reference :613-626).
        ONE shared task drains EVERY active stream's token buffer each
        cycle and publishes whatever accumulated as one chunk per job
        (wire-compatible: "response" carries a few tokens). A per-job
        polling task — the previous design — cost ~10k timer wakeups/s
        at 192 concurrent streams (measured: 1.1M TimerHandle comparisons
        per 14 s in the worker loop thread); one shared timer removes
        that churn. Cycle shrinks to 4 ms while any stream still owes its
        first chunk, so TTFT pays a few ms at most."""
        flush_s = max(0.002, self.cfg.stream_flush_ms / 1000.0)
        while self._streams:
            fast = any(not s.sent_any for s in self._streams.values())
            self._flush_wake.clear()
            # Adaptive cycle: each cycle walks EVERY active stream and
            # publishes one chunk per job — at saturation (1000+ streams)
            # a fixed 25 ms cadence costs ~40k payloads/s of flusher +
            # gateway work on the same GIL as the decode thread (measured
            # ~11% serving throughput, r02ac vs r02ae). Stretch the cycle
            # with the stream count (0.1 ms per stream, capped 100 ms);
            # the 4 ms first-chunk fast path keeps TTFT unaffected.
            cyc = min(0.1, max(flush_s, len(self._streams) * 1e-4))
            try:
                await asyncio.wait_for(self._flush_wake.wait(),
                                       0.004 if fast else cyc)
            except asyncio.TimeoutError:
                pass
            ts = now_ms()
            # fast mini-cycles serve ONLY first chunks and finished jobs;
            # steady streams flush on the full cadence — otherwise the
            # admission ramp (new streams keep `fast` true) walks every
            # active stream every 4 ms
            now = time.monotonic()
            full = now - getattr(self, "_last_full_flush", 0.0) >= cyc
            if full:
                self._last_full_flush = now
            # direct-path chunks batch into ONE frame per gateway per
            # cycle (bus/stream.py); addr-less streams fall back to the
            # bus, one publish each (reference wire behavior)
            batches: dict[str, list] = {}
            finished: list[_Stream] = []
            for s in list(self._streams.values()):
                if not full and s.sent_any and not s.done_ev.is_set():
                    continue
                with s.lk:
                    pieces = s.buf[:]
                    s.buf.clear()
                # done only once the buffer is fully drained (done_ev is
                # set AFTER the engine's final piece lands in buf)
                done = s.done_ev.is_set() and len(s.buf) == 0
                if not pieces and not done:
                    continue
                s.sent_any = True
                chunk = {"id": s.job_id, "response": "".join(pieces),
                         "done": done}
                if s.splitter is not None:       # think mode: split fields
                    th, co = s.splitter.push(chunk["response"])
                    if done:
                        th2, co2 = s.splitter.flush()
                        th, co = th + th2, co + co2
                    chunk["response"] = co
                    if th:
                        chunk["thinking"] = th
                payload = {"jobId": s.job_id, "workerId": self.worker_id,
                           "chunk": chunk, "timestamp": ts}
                if s.addr:
                    batches.setdefault(s.addr, []).append(
                        (Channels.job_stream(s.job_id), payload))
                else:
                    try:
                        await self.bus.publish(
                            Channels.job_stream(s.job_id), payload)
                    except Exception:  # noqa: BLE001 — bus hiccup: chunks
                        self.stream_drops += 1   # are fire-and-forget; the
                                       # result path (and orphan recovery)
                                       # owns delivery; drops are COUNTED
                                       # (/metrics)
                if done:
                    finished.append(s)
            for addr, items in batches.items():
                try:
                    await self._sink.send(addr, items)
                except Exception:  # noqa: BLE001 — dead gateway: at-most-
                    self.stream_drops += len(items)   # once, counted
            for s in finished:
                self._streams.pop(s.job_id, None)
                s.fin.set()
        self._flush_task = None
