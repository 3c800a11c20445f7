"""Full multi-process end-to-end: real server process (TCP bus + uvicorn
HTTP) + 2 real worker processes (tiny CPU engines), driven over HTTP.

This is the reference's CI scenario (redis+server+client
full-stack) but self-contained, plus the chaos test the reference never had:
SIGKILL a busy worker and assert the orphaned request completes on the
survivor.
"""

import json
import os
import signal
import socket
import subprocess
import sys
import time

import httpx
import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _free_port() -> int:
    s = socket.socket()
    s.bind(("127.0.0.1", 0))
    p = s.getsockname()[1]
    s.close()
    return p


WORKER_SRC = r"""
import asyncio, os, sys
from gridllm_amd.bus.tcp import TcpBus
from gridllm_amd.config import EngineConfig, WorkerConfig
from gridllm_amd.engine import InferenceEngine
from gridllm_amd.worker.agent import WorkerAgent

async def main():
    wcfg = WorkerConfig(worker_id=os.environ["WORKER_ID"],
                        bus_port=int(os.environ["BUS_PORT"]),
                        max_concurrent_tasks=2, heartbeat_interval_ms=500)
    ecfg = EngineConfig(model="tiny", device="cpu", dtype="fp32",
                        max_seq_len=128, max_batch_size=4, use_hipgraph=False)
    slow = float(os.environ.get("WORKER_SLOW", "0"))
    engine = InferenceEngine(ecfg)
    if slow > 0:  # make decode slow so chaos test can kill mid-job
        orig = engine._decode_step
        import time as _t
        def slow_step(tokens, slots, **kw):
            _t.sleep(slow)
            return orig(tokens, slots)
        engine._decode_step = slow_step
    bus = TcpBus("127.0.0.1", wcfg.bus_port)
    await bus.connect()
    agent = WorkerAgent(bus, engine, wcfg)
    await agent.start()
    print("WORKER_READY", flush=True)
    await asyncio.Event().wait()

asyncio.run(main())
"""

SERVER_SRC = r"""
import asyncio, os
import uvicorn
from gridllm_amd.config import ServerConfig
from gridllm_amd.server.app import GridLLMServer

cfg = ServerConfig(port=int(os.environ["HTTP_PORT"]),
                   bus_port=int(os.environ["BUS_PORT"]),
                   worker_heartbeat_timeout_ms=2000,
                   worker_cleanup_interval_ms=300,
                   job_retry_attempts=1, job_retry_delay_ms=200)
server = GridLLMServer(cfg)
app = server.app

@app.on_event("startup")
async def _s():
    await server.start()
    print("SERVER_READY", flush=True)

uvicorn.run(app, host="127.0.0.1", port=cfg.port, log_level="error")
"""


def _spawn(src: str, env: dict, ready_tag: str, timeout=60) -> subprocess.Popen:
    proc = subprocess.Popen(
        [sys.executable, "-u", "-c", src],
        env={**os.environ, **env, "PYTHONPATH": REPO},
        stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
        cwd=REPO)
    t0 = time.time()
    while time.time() - t0 < timeout:
        line = proc.stdout.readline()
        if ready_tag in line:
            # keep draining stdout forever or the child blocks on a full pipe
            import threading

            def _drain(p=proc):
                try:
                    for _ in p.stdout:
                        pass
                except Exception:  # noqa: BLE001
                    pass

            threading.Thread(target=_drain, daemon=True).start()
            return proc
        if proc.poll() is not None:
            raise RuntimeError(f"process died:\n{proc.stdout.read()}")
    proc.kill()
    raise TimeoutError(f"no {ready_tag} within {timeout}s")


@pytest.fixture(scope="module")
def cluster():
    bus_port, http_port = _free_port(), _free_port()
    env = {"BUS_PORT": str(bus_port), "HTTP_PORT": str(http_port)}
    server = _spawn(SERVER_SRC, env, "SERVER_READY")
    workers = {}
    for wid, slow in (("w-a", "0.15"), ("w-b", "0")):
        workers[wid] = _spawn(WORKER_SRC,
                              {**env, "WORKER_ID": wid, "WORKER_SLOW": slow},
                              "WORKER_READY")
    base = f"http://127.0.0.1:{http_port}"
    # wait for registration
    with httpx.Client(base_url=base, timeout=30) as c:
        for _ in range(100):
            r = c.get("/health/workers")
            if r.status_code == 200 and r.json()["counts"]["total"] == 2:
                break
            time.sleep(0.1)
        else:
            raise TimeoutError("workers never registered")
    yield {"base": base, "server": server, "workers": workers,
           "bus_port": bus_port}
    for p in list(workers.values()) + [server]:
        if p.poll() is None:
            p.send_signal(signal.SIGKILL)
    for p in list(workers.values()) + [server]:
        p.wait(timeout=10)


def test_http_generate_across_processes(cluster):
    with httpx.Client(base_url=cluster["base"], timeout=60) as c:
        r = c.post("/api/generate", json={
            "model": "tiny", "prompt": "hello world", "stream": False,
            "options": {"temperature": 0.0, "num_predict": 4}})
        assert r.status_code == 200, r.text
        assert r.json()["done"] is True
        assert r.json()["eval_count"] >= 1


def test_http_streaming_across_processes(cluster):
    with httpx.Client(base_url=cluster["base"], timeout=60) as c:
        with c.stream("POST", "/api/generate", json={
                "model": "tiny", "prompt": "stream", "stream": True,
                "options": {"temperature": 0.0, "num_predict": 4}}) as r:
            assert r.status_code == 200
            lines = [json.loads(l) for l in r.iter_lines() if l]
        assert lines[-1]["done"] is True


def test_parallel_requests_use_both_workers(cluster):
    import concurrent.futures as cf

    def one(i):
        with httpx.Client(base_url=cluster["base"], timeout=120) as c:
            r = c.post("/api/generate", json={
                "model": "tiny", "prompt": f"req {i}", "stream": False,
                "options": {"temperature": 0.0, "num_predict": 3}})
            return r.status_code

    with cf.ThreadPoolExecutor(8) as ex:
        codes = list(ex.map(one, range(8)))
    assert codes == [200] * 8


def test_chaos_sigkill_busy_worker_orphan_requeue(cluster):
    """Kill the slow worker mid-job: the job must be orphaned, requeued at
    the front, and completed by the surviving worker — the ORIGINAL awaited
    HTTP request succeeds (reference guarantee: JobScheduler.ts:553-630)."""
    import concurrent.futures as cf
    slow = cluster["workers"]["w-a"]

    def long_req():
        with httpx.Client(base_url=cluster["base"], timeout=180) as c:
            return c.post("/api/generate", json={
                "model": "tiny", "prompt": "chaos", "stream": False,
                "priority": "high",
                "options": {"temperature": 0.0, "num_predict": 30}})

    with cf.ThreadPoolExecutor(4) as ex:
        # saturate both workers so the slow one is certainly busy
        futs = [ex.submit(long_req) for _ in range(4)]
        time.sleep(1.5)                    # jobs are mid-decode now
        slow.send_signal(signal.SIGKILL)   # hard kill
        slow.wait(timeout=10)
        results = [f.result() for f in futs]
    assert all(r.status_code == 200 for r in results), \
        [r.text[:200] for r in results]
    # the dead worker must be gone from the registry
    with httpx.Client(base_url=cluster["base"], timeout=30) as c:
        for _ in range(100):
            names = [w["id"] for w in
                     c.get("/health/workers").json()["workers"]]
            if "w-a" not in names:
                break
            time.sleep(0.2)
        assert "w-a" not in names


def test_chaos_sigkill_during_streaming(cluster):
    """SIGKILL a worker mid-STREAM: the orphaned job requeues and the
    ORIGINAL streaming HTTP response keeps going until a final done record
    arrives from the survivor (the job:result subscriber
    survives the worker)."""
    # w-a was killed by the previous test on some orderings; use whatever
    # workers remain and spawn a fresh disposable one to kill
    victim = _spawn(WORKER_SRC,
                    {"BUS_PORT": str(cluster["bus_port"]),
                     "WORKER_ID": "w-victim", "WORKER_SLOW": "0.2"},
                    "WORKER_READY")
    try:
        time.sleep(1.0)
        import concurrent.futures as cf

        def stream_req(i):
            lines = []
            with httpx.Client(base_url=cluster["base"], timeout=180) as c:
                with c.stream("POST", "/api/generate", json={
                        "model": "tiny", "prompt": f"s{i}", "stream": True,
                        "options": {"temperature": 0.0,
                                    "num_predict": 40}}) as r:
                    for ln in r.iter_lines():
                        if ln:
                            lines.append(json.loads(ln))
            return lines

        with cf.ThreadPoolExecutor(6) as ex:
            futs = [ex.submit(stream_req, i) for i in range(6)]
            time.sleep(2.0)                     # streams are mid-decode
            victim.send_signal(signal.SIGKILL)
            victim.wait(timeout=10)
            results = [f.result() for f in futs]
        for lines in results:
            assert lines, "stream produced nothing"
            assert lines[-1].get("done") is True
            assert not lines[-1].get("error"), lines[-1]
    finally:
        if victim.poll() is None:
            victim.send_signal(signal.SIGKILL)
            victim.wait(timeout=10)


def test_module_entrypoints_e2e():
    """The DOCUMENTED deployment commands (`python -m gridllm_amd.server`,
    `python -m gridllm_amd.worker`, README quickstart) boot, register,
    and serve a request."""
    import httpx

    def free():
        s = socket.socket()
        s.bind(("127.0.0.1", 0))
        p = s.getsockname()[1]
        s.close()
        return p

    hp, bp, wp = free(), free(), free()
    env = {**os.environ, "PORT": str(hp), "BUS_PORT": str(bp),
           "PYTHONPATH": REPO}
    srv = subprocess.Popen([sys.executable, "-m", "gridllm_amd.server"],
                           env=env, stdout=subprocess.PIPE,
                           stderr=subprocess.STDOUT, text=True)
    wenv = {**env, "ENGINE_MODEL": "tiny", "ENGINE_DEVICE": "cpu",
            "ENGINE_DTYPE": "fp32", "WORKER_PORT": str(wp),
            "BUS_HOST": "127.0.0.1", "WORKER_ID": "mod-entry-w"}
    wrk = None
    try:
        for _ in range(100):            # server HTTP up
            time.sleep(0.2)
            try:
                if httpx.get(f"http://127.0.0.1:{hp}/health",
                             timeout=2).status_code == 200:
                    break
            except Exception:  # noqa: BLE001
                pass
        else:
            raise AssertionError("server module entry did not come up")
        wrk = subprocess.Popen([sys.executable, "-m", "gridllm_amd.worker"],
                               env=wenv, stdout=subprocess.PIPE,
                               stderr=subprocess.STDOUT, text=True)
        for _ in range(150):            # worker registered
            time.sleep(0.2)
            try:
                r = httpx.get(f"http://127.0.0.1:{hp}/health/workers",
                              timeout=2)
                if r.status_code == 200 and \
                        r.json()["counts"].get("total", 0) >= 1:
                    break
            except Exception:  # noqa: BLE001
                pass
        else:
            raise AssertionError("worker module entry never registered")
        g = httpx.post(f"http://127.0.0.1:{hp}/api/generate",
                       json={"model": "tiny", "prompt": "hi",
                             "stream": False,
                             "options": {"num_predict": 4}}, timeout=60)
        assert g.status_code == 200 and g.json()["eval_count"] == 4, g.text
    finally:
        for p in (wrk, srv):
            if p is not None and p.poll() is None:
                p.send_signal(signal.SIGTERM)
        for p in (wrk, srv):
            if p is not None:
                try:
                    p.wait(timeout=10)
                except Exception:  # noqa: BLE001
                    p.kill()


def test_cancel_storm_drains_and_recovers():
    """Half of 64 concurrent streams are abandoned mid-flight (client
    walks away) for two rounds: no errors on the surviving half, the
    queue drains to zero (disconnect-cancel + deferred KV-slot frees
    under the pipelined decode don't leak), and the worker serves
    afterwards."""
    import asyncio
    import aiohttp
    import httpx
    bus_port, http_port = _free_port(), _free_port()
    env = {"BUS_PORT": str(bus_port), "HTTP_PORT": str(http_port)}
    server = _spawn(SERVER_SRC, env, "SERVER_READY")
    worker = _spawn(WORKER_SRC, {**env, "WORKER_ID": "w-cstorm"},
                    "WORKER_READY")
    try:
        base = f"http://127.0.0.1:{http_port}"
        with httpx.Client(base_url=base, timeout=30) as c:
            for _ in range(100):
                r = c.get("/health/workers")
                if r.status_code == 200 and \
                        r.json()["counts"]["total"] == 1:
                    break
                time.sleep(0.1)

        async def storm():
            stats = {"done": 0, "gone": 0, "err": 0}
            async with aiohttp.ClientSession(base) as s:
                async def gen(i):
                    try:
                        async with s.post("/api/generate", json={
                                "model": "tiny", "prompt": f"storm {i}",
                                "stream": True,
                                "options": {"temperature": 0.8, "seed": i,
                                            "num_predict": 48}},
                                timeout=aiohttp.ClientTimeout(
                                    total=60)) as r:
                            async for raw in r.content:
                                if raw.strip() and i % 2 == 1:
                                    stats["gone"] += 1
                                    return       # abandon mid-stream
                            stats["done"] += 1
                    except Exception:  # noqa: BLE001
                        stats["err"] += 1
                for rnd in range(2):
                    await asyncio.gather(
                        *(gen(rnd * 64 + i) for i in range(64)))
            return stats

        st = asyncio.run(storm())
        assert st["err"] == 0 and st["done"] == 64 and st["gone"] == 64, st
        with httpx.Client(base_url=base, timeout=30) as c:
            for _ in range(150):
                q = c.get("/inference/queue").json()["queue"]
                if q["active"] == 0 and q["queued"] == 0:
                    break
                time.sleep(0.2)
            else:
                raise AssertionError(f"not drained: {q}")
            r = c.post("/api/generate", json={
                "model": "tiny", "prompt": "after", "stream": False,
                "options": {"num_predict": 3}})
            assert r.status_code == 200 and r.json()["eval_count"] == 3
    finally:
        server.kill()
        worker.kill()
