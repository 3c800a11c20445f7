"""Control/data-plane split:

* standalone durable bus (`python -m gridllm_amd.bus`) — kill -9 the
  SERVER process mid-load, restart it against the surviving bus, and the
  queued jobs still complete (the reference's external-Redis guarantee,
  docker-compose.yml:12-30 + JobScheduler.ts:82-126);
* detached gateway replicas (`python -m gridllm_amd.gateway`) — a
  replica serves the full API against a remote scheduler over the bus,
  with token chunks arriving on its own direct stream plane;
* StreamServer/StreamSink unit round-trip and bus snapshot persistence.
"""

import asyncio
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


def _spawn(args, env, ready_tag, timeout=60):
    proc = subprocess.Popen(args, env={**os.environ, **env,
                                       "PYTHONPATH": REPO},
                            stdout=subprocess.PIPE,
                            stderr=subprocess.STDOUT, text=True, cwd=REPO)
    t0 = time.time()
    while time.time() - t0 < timeout:
        line = proc.stdout.readline()
        if ready_tag in line:
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


SERVER_SRC = r"""
import asyncio, os
import uvicorn
from gridllm_amd.config import ServerConfig
from gridllm_amd.server.app import GridLLMServer

cfg = ServerConfig(port=int(os.environ["HTTP_PORT"]),
                   bus_port=int(os.environ["BUS_PORT"]),
                   bus_external=True,
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

WORKER_SRC = r"""
import asyncio, os
from gridllm_amd.bus.tcp import TcpBus
from gridllm_amd.config import EngineConfig, WorkerConfig
from gridllm_amd.engine import InferenceEngine
from gridllm_amd.worker.agent import WorkerAgent

async def main():
    wcfg = WorkerConfig(worker_id=os.environ["WORKER_ID"],
                        bus_port=int(os.environ["BUS_PORT"]),
                        max_concurrent_tasks=4, heartbeat_interval_ms=500)
    ecfg = EngineConfig(model="tiny", device="cpu", dtype="fp32",
                        max_seq_len=128, max_batch_size=4,
                        use_hipgraph=False)
    engine = InferenceEngine(ecfg)
    slow = float(os.environ.get("WORKER_SLOW", "0"))
    if slow > 0:
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


def test_stream_server_sink_roundtrip():
    async def run():
        from gridllm_amd.bus.stream import StreamServer, StreamSink
        srv = StreamServer("127.0.0.1", 0)
        await srv.start()
        got = []

        async def h(ch, payload):
            got.append((ch, payload))

        srv.subscribe("job:stream:a", h)
        srv.subscribe("job:stream:b", h)
        sink = StreamSink()
        await sink.send(srv.addr, [
            ("job:stream:a", {"chunk": {"response": "x", "done": False}}),
            ("job:stream:b", {"chunk": {"response": "y", "done": True}}),
            ("job:stream:none", {"chunk": {}}),     # unsubscribed: dropped
        ])
        for _ in range(100):
            if len(got) >= 2:
                break
            await asyncio.sleep(0.01)
        assert sorted(c for c, _ in got) == ["job:stream:a", "job:stream:b"]
        # connection reuse: second batch on the same pooled conn
        await sink.send(srv.addr, [("job:stream:a", {"chunk": {"z": 1}})])
        for _ in range(100):
            if len(got) >= 3:
                break
            await asyncio.sleep(0.01)
        assert len(got) == 3
        await sink.close()
        await srv.stop()

    asyncio.run(run())


def test_bus_snapshot_roundtrip(tmp_path):
    from gridllm_amd.bus.tcp import BusServer
    a = BusServer("127.0.0.1", 0)
    a.kv["job_queue"] = ("[1,2,3]", 0.0)
    a.kv["ttl_key"] = ("v", __import__("time").monotonic() + 5.0)
    a.kv["expired"] = ("gone", __import__("time").monotonic() - 1.0)
    a.hashes["workers"]["w1"] = '{"id":"w1"}'
    p = str(tmp_path / "snap.bin")
    a.save_snapshot(p)
    b = BusServer("127.0.0.1", 0)
    assert b.load_snapshot(p)
    assert b.kv["job_queue"][0] == "[1,2,3]"
    assert "expired" not in b.kv          # expired keys not persisted
    assert not b.kv_expired("ttl_key")    # remaining TTL restored
    assert b.hashes["workers"]["w1"] == '{"id":"w1"}'


@pytest.fixture()
def durable_stack(tmp_path):
    bus_port, http_port = _free_port(), _free_port()
    snap = str(tmp_path / "bus.snap")
    env = {"BUS_PORT": str(bus_port), "HTTP_PORT": str(http_port)}
    bus = _spawn([sys.executable, "-m", "gridllm_amd.bus",
                  "--port", str(bus_port), "--snapshot", snap,
                  "--snapshot-interval-ms", "200"], env, "BUS_READY")
    procs = {"bus": bus}
    try:
        procs["server"] = _spawn([sys.executable, "-u", "-c", SERVER_SRC],
                                 env, "SERVER_READY")
        procs["worker"] = _spawn(
            [sys.executable, "-u", "-c", WORKER_SRC],
            {**env, "WORKER_ID": "w-dur", "WORKER_SLOW": "0.25"},
            "WORKER_READY")
        base = f"http://127.0.0.1:{http_port}"
        with httpx.Client(base_url=base, timeout=30) as c:
            for _ in range(100):
                r = c.get("/health/workers")
                if r.status_code == 200 and \
                        r.json()["counts"]["total"] == 1:
                    break
                time.sleep(0.1)
            else:
                raise TimeoutError("worker never registered")
        yield {"base": base, "env": env, "procs": procs,
               "http_port": http_port, "snap": snap}
    finally:
        for p in procs.values():
            if p.poll() is None:
                p.send_signal(signal.SIGKILL)
        for p in procs.values():
            p.wait(timeout=10)


def test_kill9_server_jobs_survive_on_external_bus(durable_stack):
    """kill -9 the SERVER while jobs are queued on the standalone bus:
    a restarted server reloads the queue and the jobs complete
    (reference guarantee via Redis AOF — JobScheduler.ts:82-126)."""
    import concurrent.futures as cf
    st = durable_stack
    server = st["procs"]["server"]

    def one(i):
        # generous timeout: these requests span the server restart
        with httpx.Client(base_url=st["base"], timeout=240) as c:
            return c.post("/api/generate", json={
                "model": "tiny", "prompt": f"durable {i}", "stream": False,
                "options": {"temperature": 0.0, "num_predict": 12}})

    with cf.ThreadPoolExecutor(8) as ex:
        # 8 jobs, worker capacity 4 and slowed: several stay QUEUED
        futs = [ex.submit(one, i) for i in range(8)]
        time.sleep(1.2)                    # some active, some queued
        server.send_signal(signal.SIGKILL)
        server.wait(timeout=10)
        # the original HTTP awaiters died with the server — the assertion
        # is about QUEUE SURVIVAL: restart and the queued work completes
        time.sleep(0.5)
        st["procs"]["server"] = _spawn(
            [sys.executable, "-u", "-c", SERVER_SRC], st["env"],
            "SERVER_READY")
        results = []
        for f in futs:
            try:
                results.append(f.result())
            except Exception as e:  # noqa: BLE001 — killed conn expected
                results.append(e)
    # the restarted server must be serving and must have RELOADED state:
    # wait for it to finish the recovered queue, then submit a fresh job
    with httpx.Client(base_url=st["base"], timeout=120) as c:
        for _ in range(200):
            r = c.get("/inference/queue")
            if r.status_code == 200:
                q = r.json()
                if q.get("queue", {}).get("queued", 0) == 0 and \
                        q.get("queue", {}).get("active", 0) == 0:
                    break
            time.sleep(0.2)
        r = c.post("/api/generate", json={
            "model": "tiny", "prompt": "after restart", "stream": False,
            "options": {"temperature": 0.0, "num_predict": 4}})
        assert r.status_code == 200, r.text
        # and the recovered queue actually ran: completed count covers
        # the pre-kill jobs that never got an HTTP response
        stats = c.get("/inference/queue").json()
        assert stats["queue"]["completed"] >= 1


def test_kill9_bus_snapshot_restores_state(durable_stack):
    """kill -9 the BUS process: a restart from its snapshot restores the
    worker hash and kv (Redis-AOF analog at the bus level)."""
    st = durable_stack
    with httpx.Client(base_url=st["base"], timeout=60) as c:
        r = c.post("/api/generate", json={
            "model": "tiny", "prompt": "warm", "stream": False,
            "options": {"temperature": 0.0, "num_predict": 3}})
        assert r.status_code == 200
    time.sleep(0.6)                        # snapshot interval 200 ms
    bus = st["procs"]["bus"]
    bus.send_signal(signal.SIGKILL)
    bus.wait(timeout=10)
    st["procs"]["bus"] = _spawn(
        [sys.executable, "-m", "gridllm_amd.bus",
         "--port", st["env"]["BUS_PORT"], "--snapshot", st["snap"],
         "--snapshot-interval-ms", "200"], st["env"], "BUS_READY")

    async def check():
        from gridllm_amd.bus.tcp import TcpBus
        b = TcpBus("127.0.0.1", int(st["env"]["BUS_PORT"]))
        await b.connect()
        try:
            workers = await b.hgetall("workers")
            assert "w-dur" in workers, workers.keys()
        finally:
            await b.close()

    asyncio.run(check())


@pytest.fixture()
def replica_stack():
    bus_port, http_port, gw_port = _free_port(), _free_port(), _free_port()
    env = {"BUS_PORT": str(bus_port), "HTTP_PORT": str(http_port)}
    procs = {}
    procs["server"] = _spawn([sys.executable, "-u", "-c",
                              SERVER_SRC.replace("bus_external=True",
                                                 "bus_external=False")],
                             env, "SERVER_READY")
    procs["worker"] = _spawn([sys.executable, "-u", "-c", WORKER_SRC],
                             {**env, "WORKER_ID": "w-rep"}, "WORKER_READY")
    procs["gateway"] = _spawn(
        [sys.executable, "-m", "gridllm_amd.gateway",
         "--port", str(gw_port), "--host", "127.0.0.1",
         "--bus", f"127.0.0.1:{bus_port}"], env, "GATEWAY_READY")
    base = f"http://127.0.0.1:{gw_port}"
    with httpx.Client(base_url=base, timeout=30) as c:
        for _ in range(100):
            try:
                r = c.get("/api/tags")
                if r.status_code == 200 and r.json()["models"]:
                    break
            except Exception:  # noqa: BLE001
                pass
            time.sleep(0.1)
        else:
            raise TimeoutError("gateway replica never saw the worker")
    yield {"base": base, "bus_port": bus_port}
    for p in procs.values():
        if p.poll() is None:
            p.send_signal(signal.SIGKILL)
    for p in procs.values():
        p.wait(timeout=10)


def test_gateway_replica_serves_full_api(replica_stack):
    base = replica_stack["base"]
    with httpx.Client(base_url=base, timeout=60) as c:
        # non-stream via bus submit -> scheduler process -> worker
        r = c.post("/api/generate", json={
            "model": "tiny", "prompt": "via replica", "stream": False,
            "options": {"temperature": 0.0, "num_predict": 4}})
        assert r.status_code == 200, r.text
        assert r.json()["eval_count"] == 4
        # streaming: chunks arrive on the replica's OWN stream server
        with c.stream("POST", "/api/generate", json={
                "model": "tiny", "prompt": "replica stream", "stream": True,
                "options": {"temperature": 0.0, "num_predict": 6}}) as r:
            assert r.status_code == 200
            lines = [json.loads(x) for x in r.iter_lines() if x]
        assert lines[-1]["done"] is True
        assert sum(len(c0.get("response", "")) for c0 in lines[:-1]) > 0
        # OpenAI surface + health/queue served from the stats snapshot
        r = c.post("/v1/completions", json={
            "model": "tiny", "prompt": "x", "max_tokens": 4})
        assert r.status_code == 200, r.text
        r = c.get("/inference/queue")
        assert r.status_code == 200
        assert "queue" in r.json()


def test_replica_stream_survives_worker_sigkill(replica_stack, request):
    """SIGKILL the worker mid-stream THROUGH A DETACHED REPLICA: the
    orphaned job requeues (metadata.streamAddr survives), the surviving
    worker streams to the replica's OWN stream server, and the original
    HTTP response completes."""
    # spawn a second worker so the requeue has somewhere to go
    bus_port = replica_stack.get("bus_port")
    if bus_port is None:
        pytest.skip("fixture lacks bus port")
    w2 = _spawn([sys.executable, "-u", "-c", WORKER_SRC],
                {"BUS_PORT": str(bus_port), "WORKER_ID": "w-rep2",
                 "WORKER_SLOW": "0"}, "WORKER_READY")
    victim = _spawn([sys.executable, "-u", "-c", WORKER_SRC],
                    {"BUS_PORT": str(bus_port), "WORKER_ID": "w-victim2",
                     "WORKER_SLOW": "0.15"}, "WORKER_READY")
    try:
        time.sleep(1.0)
        import concurrent.futures as cf

        def stream_req(i):
            lines = []
            with httpx.Client(base_url=replica_stack["base"],
                              timeout=180) as c:
                with c.stream("POST", "/api/generate", json={
                        "model": "tiny", "prompt": f"rs{i}",
                        "stream": True,
                        "options": {"temperature": 0.0,
                                    "num_predict": 40}}) as r:
                    for ln in r.iter_lines():
                        if ln:
                            lines.append(json.loads(ln))
            return lines

        with cf.ThreadPoolExecutor(6) as ex:
            futs = [ex.submit(stream_req, i) for i in range(6)]
            time.sleep(2.0)
            victim.send_signal(signal.SIGKILL)
            victim.wait(timeout=10)
            results = [f.result() for f in futs]
        for lines in results:
            assert lines, "stream produced nothing"
            assert lines[-1].get("done") is True
            assert not lines[-1].get("error"), lines[-1]
    finally:
        for p in (victim, w2):
            if p.poll() is None:
                p.send_signal(signal.SIGKILL)
                p.wait(timeout=10)


def test_worker_reconnects_after_bus_restart(tmp_path):
    """Kill -9 the standalone bus under a registered worker; restart the
    bus (same snapshot) and the server: the worker's reconnect loop
    (worker/main.py run_worker, exponential backoff — the reference's
    RedisConnectionManager policy, C4) re-registers WITHOUT duplicate
    subscriptions (bus/tcp.py subscribe dedupes bound methods) and the
    fleet serves again."""
    import httpx
    bus_port, http_port = _free_port(), _free_port()
    snap = str(tmp_path / "bus-rc.snap")
    env = {"BUS_PORT": str(bus_port), "HTTP_PORT": str(http_port)}
    bus_args = [sys.executable, "-m", "gridllm_amd.bus",
                "--port", str(bus_port), "--snapshot", snap,
                "--snapshot-interval-ms", "200"]
    procs = {}
    procs["bus"] = _spawn(bus_args, env, "BUS_READY")
    try:
        procs["server"] = _spawn([sys.executable, "-u", "-c", SERVER_SRC],
                                 env, "SERVER_READY")
        wenv = {**os.environ, **env, "PYTHONPATH": REPO,
                "ENGINE_MODEL": "tiny", "ENGINE_DEVICE": "cpu",
                "ENGINE_DTYPE": "fp32", "BUS_HOST": "127.0.0.1",
                "WORKER_ID": "w-reconnect", "WORKER_PORT": str(_free_port()),
                "RECONNECT_BASE_DELAY": "100"}
        procs["worker"] = subprocess.Popen(
            [sys.executable, "-m", "gridllm_amd.worker"], env=wenv,
            stdout=subprocess.DEVNULL, stderr=subprocess.STDOUT)
        base = f"http://127.0.0.1:{http_port}"
        with httpx.Client(base_url=base, timeout=30) as c:
            for _ in range(150):
                try:
                    r = c.get("/health/workers")
                    if r.status_code == 200 and \
                            r.json()["counts"]["total"] == 1:
                        break
                except Exception:  # noqa: BLE001
                    pass
                time.sleep(0.2)
            else:
                raise TimeoutError("worker never registered")
            r = c.post("/api/generate", json={
                "model": "tiny", "prompt": "before", "stream": False,
                "options": {"num_predict": 3}})
            assert r.status_code == 200 and r.json()["eval_count"] == 3

        # kill the BUS (and the server whose connection died with it)
        procs["bus"].send_signal(signal.SIGKILL)
        procs["bus"].wait(timeout=10)
        procs["server"].send_signal(signal.SIGKILL)
        procs["server"].wait(timeout=10)
        time.sleep(0.5)
        procs["bus"] = _spawn(bus_args, env, "BUS_READY")
        procs["server"] = _spawn([sys.executable, "-u", "-c", SERVER_SRC],
                                 env, "SERVER_READY")

        with httpx.Client(base_url=base, timeout=30) as c:
            for _ in range(200):       # worker backoff + re-register
                try:
                    r = c.get("/health/workers")
                    if r.status_code == 200 and \
                            r.json()["counts"]["total"] == 1:
                        break
                except Exception:  # noqa: BLE001
                    pass
                time.sleep(0.2)
            else:
                raise TimeoutError("worker did not re-register")
            r = c.post("/api/generate", json={
                "model": "tiny", "prompt": "after reconnect",
                "stream": False, "options": {"num_predict": 3}})
            assert r.status_code == 200 and r.json()["eval_count"] == 3, \
                r.text
    finally:
        for p in procs.values():
            if p.poll() is None:
                p.send_signal(signal.SIGKILL)
        for p in procs.values():
            p.wait(timeout=10)


def test_gateway_replica_survives_bus_restart(tmp_path):
    """Kill -9 the standalone bus under a detached gateway replica;
    restart bus + server: the replica's reconnect supervisor
    (gateway.py) re-attaches and serves — the full durable-fleet story
    (bus restart -> workers AND replicas reconnect, no process restarts
    except the bus-owning server)."""
    import httpx
    bus_port, http_port, gw_port = _free_port(), _free_port(), _free_port()
    snap = str(tmp_path / "bus-gw.snap")
    env = {"BUS_PORT": str(bus_port), "HTTP_PORT": str(http_port)}
    bus_args = [sys.executable, "-m", "gridllm_amd.bus",
                "--port", str(bus_port), "--snapshot", snap,
                "--snapshot-interval-ms", "200"]
    procs = {}
    procs["bus"] = _spawn(bus_args, env, "BUS_READY")
    try:
        procs["server"] = _spawn([sys.executable, "-u", "-c", SERVER_SRC],
                                 env, "SERVER_READY")
        wenv = {**os.environ, **env, "PYTHONPATH": REPO,
                "ENGINE_MODEL": "tiny", "ENGINE_DEVICE": "cpu",
                "ENGINE_DTYPE": "fp32", "BUS_HOST": "127.0.0.1",
                "WORKER_ID": "w-gwrc", "WORKER_PORT": str(_free_port()),
                "RECONNECT_BASE_DELAY": "100"}
        procs["worker"] = subprocess.Popen(
            [sys.executable, "-m", "gridllm_amd.worker"], env=wenv,
            stdout=subprocess.DEVNULL, stderr=subprocess.STDOUT)
        procs["gateway"] = _spawn(
            [sys.executable, "-m", "gridllm_amd.gateway",
             "--port", str(gw_port), "--host", "127.0.0.1",
             "--bus", f"127.0.0.1:{bus_port}"], env, "GATEWAY_READY")
        base = f"http://127.0.0.1:{gw_port}"

        def wait_serving(msg):
            with httpx.Client(base_url=base, timeout=30) as c:
                for _ in range(200):
                    try:
                        r = c.post("/api/generate", json={
                            "model": "tiny", "prompt": "p",
                            "stream": False,
                            "options": {"num_predict": 2}})
                        if r.status_code == 200 and \
                                r.json().get("eval_count") == 2:
                            return
                    except Exception:  # noqa: BLE001
                        pass
                    time.sleep(0.2)
            raise TimeoutError(msg)

        wait_serving("replica never served before restart")
        procs["bus"].send_signal(signal.SIGKILL)
        procs["bus"].wait(timeout=10)
        procs["server"].send_signal(signal.SIGKILL)
        procs["server"].wait(timeout=10)
        time.sleep(0.5)
        procs["bus"] = _spawn(bus_args, env, "BUS_READY")
        procs["server"] = _spawn([sys.executable, "-u", "-c", SERVER_SRC],
                                 env, "SERVER_READY")
        wait_serving("replica did not recover after bus restart")
    finally:
        for p in procs.values():
            if p.poll() is None:
                p.send_signal(signal.SIGKILL)
        for p in procs.values():
            p.wait(timeout=10)


def test_ndjson_client_disconnect_cancels_job(durable_stack):
    """Abruptly close the TCP connection mid-/api/generate NDJSON
    stream: the gateway must cancel the job on the worker, as on the
    SSE path. The
    fixture worker decodes at 0.25 s/step, so an uncancelled job holds
    active_jobs for minutes."""
    import socket as _socket
    base = durable_stack["base"]
    port = durable_stack["http_port"]
    body = json.dumps({"model": "tiny", "prompt": "disconnect probe",
                       "stream": True,
                       "options": {"temperature": 0.8, "seed": 9,
                                   "num_predict": 400}})
    req = ("POST /api/generate HTTP/1.1\r\nHost: x\r\n"
           "Content-Type: application/json\r\n"
           f"Content-Length: {len(body)}\r\n"
           "Connection: close\r\n\r\n" + body)
    s = _socket.create_connection(("127.0.0.1", port))
    s.sendall(req.encode())
    buf = b""
    while b'"response"' not in buf:          # first streamed chunk
        d = s.recv(65536)
        assert d, f"stream ended early: {buf[:200]!r}"
        buf += d
    s.close()                                # walk away mid-stream
    import httpx
    with httpx.Client(base_url=base, timeout=30) as c:
        for _ in range(100):                 # cancel beats the 100 s
            r = c.get("/inference/queue")    # generation by a wide margin
            if r.status_code == 200 and \
                    (r.json().get("queue") or {}).get("active") == 0:
                return
            time.sleep(0.2)
    raise AssertionError("job not cancelled after client disconnect: "
                         + r.text[:200])
