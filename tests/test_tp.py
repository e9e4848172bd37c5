"""Tensor parallelism: weight sharding (CPU), the leader/worker command channel over gloo with
world_size 2 (CPU, multi-process), and -- on a GPU box -- the xGMI one-shot all-reduce and a
TP=2/4/8 sharded model against TP=1 (several ranks sharing one GPU; tools/tp_check.py).  World 8 is
the strategic tier's target degree and AR_MAX_RANKS: its IPC mesh, one-shot pull over 7 peers and
vocab-parallel all-gather run here with 8 processes on one GPU (not a scaling measurement)."""
import json
import time
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_shard_tensor_column_and_row():
    from aios_amd.gguf.quants import BLOCK_INFO, GGMLType
    from aios_amd.runtime.loader import shard_tensor

    blk, bpb = BLOCK_INFO[GGMLType.Q4_K]
    rows, cols = 64, 1024  # 4 blocks per row
    raw = np.arange(rows * (cols // blk) * bpb, dtype=np.uint64).astype(np.uint8)
    parts = [shard_tensor("blk.0.attn_q.weight", raw, int(GGMLType.Q4_K), rows, cols, r, 4) for r in range(4)]
    assert all(p[1] == 16 and p[2] == cols for p in parts)
    assert np.array_equal(np.concatenate([p[0] for p in parts]), raw)  # column-parallel = row blocks
    rparts = [shard_tensor("blk.0.ffn_down.weight", raw, int(GGMLType.Q4_K), rows, cols, r, 2) for r in range(2)]
    assert all(p[1] == rows and p[2] == cols // 2 for p in rparts)
    full = raw.reshape(rows, cols // blk, bpb)
    back = np.concatenate([p[0].reshape(rows, -1, bpb) for p in rparts], axis=1)
    assert np.array_equal(back, full)  # row-parallel = K blocks
    same = shard_tensor("token_embd.weight", raw, int(GGMLType.Q4_K), rows, cols, 1, 4)
    assert same[0] is raw
    with pytest.raises(ValueError):
        shard_tensor("blk.0.ffn_down.weight", raw, int(GGMLType.Q4_K), rows, cols, 0, 8)  # 4 blocks / 8


WORKER = r"""
import os, sys, json
sys.path.insert(0, sys.argv[1])
import torch.distributed as dist
from aios_amd.parallel.tp import TPEngine, worker_loop

class FakeEngine:
    def __init__(self): self.calls = []
    def __getattr__(self, n):
        if n.startswith("_"): raise AttributeError(n)
        def f(*a, **k):
            self.calls.append([n, repr(a)])
            return len(self.calls)
        return f
class FakeComm:
    def error(self): return False

rank = int(sys.argv[2]); out = sys.argv[3]
dist.init_process_group("gloo", init_method="tcp://127.0.0.1:" + sys.argv[4], rank=rank, world_size=2)
eng = FakeEngine()
if rank == 0:
    tp = TPEngine(eng, FakeComm())
    tp.prefill(0, [1, 2, 3], 0, True)
    tp.decode([0], [5], [3], [0.0], [0], 0, b"")
    tp.decode_loop_run(1, 8, True)
    tp.close()
else:
    worker_loop(eng, FakeComm())
json.dump(eng.calls, open(out + str(rank), "w"))
dist.destroy_process_group()
"""


def test_tp_command_channel_gloo(tmp_path):
    import socket

    s = socket.socket()
    s.bind(("127.0.0.1", 0))
    port = str(s.getsockname()[1])
    s.close()
    script = tmp_path / "w.py"
    script.write_text(WORKER)
    out = str(tmp_path / "calls")
    env = dict(os.environ, CUDA_VISIBLE_DEVICES="", HIP_VISIBLE_DEVICES="")
    procs = [subprocess.Popen([sys.executable, str(script), ROOT, str(r), out, port], env=env) for r in range(2)]
    for p in procs:
        assert p.wait(timeout=120) == 0
    c0, c1 = (json.load(open(out + str(r))) for r in range(2))
    assert c0 == c1 and [c[0] for c in c0] == ["prefill", "decode", "decode_loop_run"]


FUSE_WORKER = r"""
import os, sys, json
sys.path.insert(0, sys.argv[1])
import torch.distributed as dist
import aios_amd.parallel.tp as tp

rank = int(sys.argv[2]); out = sys.argv[3]
dist.init_process_group("gloo", init_method="tcp://127.0.0.1:" + sys.argv[4], rank=rank, world_size=2)

class FakeComm:
    fused = True
    disabled = False
    def disable_fuse(self): self.disabled = True; self.fused = False

class FakeEngine:
    tp_fused = True
    disabled = False
    def tp_fuse_fits(self): return [1, 1, 1, 0] if rank == 1 else [1, 1, 1, 1]  # rank 1 misses one shape
    def disable_tp_fuse(self): self.disabled = True; self.tp_fused = False

ag = tp.gloo_allgather(None, 2)
res = {}
# 1. the fused self-test fails on rank 1 only: every rank disables the fused epilogue
tp.fused_self_test = lambda comm, r, w, d, g: r != 1
c = FakeComm()
res["fail_on"] = tp.check_fused_comm(c, rank, 2, 0, ag)
res["fail_disabled"] = c.disabled
# 2. it passes everywhere: fused stays on
tp.fused_self_test = lambda comm, r, w, d, g: True
c2 = FakeComm()
res["pass_on"] = tp.check_fused_comm(c2, rank, 2, 0, ag)
res["pass_disabled"] = c2.disabled
# 3. the self-test raises on rank 0: a failed check, not a hang
def boom(*a):
    if rank == 0:
        raise RuntimeError("peer mapping refused")
    return True
tp.fused_self_test = boom
c3 = FakeComm()
res["raise_on"] = tp.check_fused_comm(c3, rank, 2, 0, ag)
# 4. per-layer launch fits differ: every rank's engine turns fusion off
e = FakeEngine()
res["fits_on"] = tp.reconcile_tp_fuse(e, ag)
res["fits_disabled"] = e.disabled
json.dump(res, open(out + str(rank), "w"))
dist.destroy_process_group()
"""


def test_tp_fused_check_fails_safe_on_every_rank(tmp_path):
    """a fused-epilogue self-test failing on ONE rank (or raising there), and per-layer
    fused-launch fits that differ between ranks, turn the fused all-reduce epilogue off on EVERY rank
    (GEMV + separate all-reduce everywhere), over a real gloo world of 2 with mocked comms."""
    import socket

    s = socket.socket()
    s.bind(("127.0.0.1", 0))
    port = str(s.getsockname()[1])
    s.close()
    script = tmp_path / "f.py"
    script.write_text(FUSE_WORKER)
    out = str(tmp_path / "res")
    env = dict(os.environ, CUDA_VISIBLE_DEVICES="", HIP_VISIBLE_DEVICES="")
    procs = [subprocess.Popen([sys.executable, str(script), ROOT, str(r), out, port], env=env) for r in range(2)]
    for p in procs:
        assert p.wait(timeout=120) == 0
    for r in range(2):
        res = json.load(open(out + str(r)))
        assert res["fail_on"] is False and res["fail_disabled"] is True, res
        assert res["pass_on"] is True and res["pass_disabled"] is False, res
        assert res["raise_on"] is False, res
        assert res["fits_on"] is False and res["fits_disabled"] is True, res


def test_shard_tensor_vocab_parallel_output():
    from aios_amd.gguf.quants import BLOCK_INFO, GGMLType
    from aios_amd.runtime.loader import shard_tensor

    blk, bpb = BLOCK_INFO[GGMLType.Q6_K]
    rows, cols = 64, 512
    raw = np.arange(rows * (cols // blk) * bpb, dtype=np.uint64).astype(np.uint8)
    assert shard_tensor("output.weight", raw, int(GGMLType.Q6_K), rows, cols, 1, 2)[0] is raw  # replicated
    parts = [shard_tensor("output.weight", raw, int(GGMLType.Q6_K), rows, cols, r, 2, True) for r in range(2)]
    assert all(p[1] == rows // 2 and p[2] == cols for p in parts)
    assert np.array_equal(np.concatenate([p[0] for p in parts]), raw)


def test_engine_config_vocab_parallel_rules():
    from aios_amd.models.config import get_preset
    from aios_amd.runtime import native

    if native.load(build_if_missing=False) is None:
        pytest.skip("native engine not built")
    cfg = get_preset("test-tp8-shape")
    assert native.engine_config(cfg, tp_size=2).vocab_parallel == 1
    assert native.engine_config(cfg, tp_size=1).vocab_parallel == 0
    assert native.engine_config(cfg, tp_size=2, vocab_parallel=False).vocab_parallel == 0
    import dataclasses
    tied = dataclasses.replace(cfg, tie_embeddings=True)
    assert native.engine_config(tied, tp_size=2).vocab_parallel == 0


def test_collectives_of_ranks_that_share_a_gpu_leave_half_of_its_cus():
    """what waits for a peer must not stand on every CU: the peer's kernels may need one to themselves before its own collective"""
    from aios_amd.runtime import native

    E = native.load(build_if_missing=False)
    if E is None:
        pytest.skip("native engine not built")
    assert E.ar_waiting_wg(1, 256) == 512
    for ranks in range(2, 9):
        for cus in (304, 256, 120, 16):
            assert 1 <= E.ar_waiting_wg(ranks, cus) <= max(1, cus // 2 // ranks)


@pytest.mark.parametrize("ids,want", [(["n/0", "n/0"], 2), (["n/0", "n/1"], None), (["n/0", "n/1", "n/0", "n/1"], 2)])
def test_daemon_ranks_that_share_a_gpu_say_so_to_their_comm(monkeypatch, ids, want):
    """the daemon's setup bounds what waits for a peer as create_comm does (before any collective runs)"""
    import aios_amd.parallel.tp as tp

    calls = []

    class Comm:
        fuse_eligible = uncached = True

        def __getattr__(self, name):
            return lambda *a: calls.append((name, *a))

    monkeypatch.setattr(tp, "device_identity", lambda d: ids[d])
    monkeypatch.setattr(tp, "comm_self_test", lambda *a: calls.append(("self_test",)) or True)
    monkeypatch.setattr(tp, "check_fused_comm", lambda *a: None)
    tp.xgmi_handshake(Comm(), 0, len(ids), 0, lambda obj: list(ids) if isinstance(obj, str) else [obj] * len(ids))
    assert calls == ([("set_ranks_per_gpu", want)] if want else []) + [("self_test",)]


@pytest.mark.gpu
@pytest.mark.parametrize("world,gemm_prefill,prompt_len", [(2, 0, 21), (4, 0, 21), (8, 0, 21), (2, 1, 21),
                                                          (2, 1, 640), (2, 1, 9)])
def test_tp_xgmi_allreduce_and_sharded_model(tmp_path, world, gemm_prefill, prompt_len):
    """TP=N vs TP=1 on the same weights.  With the fp32-activation GEMV prefill (gemm_prefill=0)
    the only differences are fp32 summation order: 1e-3 of the logit scale.  The MFMA prefill
    path rounds activations to bf16 (and sums split-K partials atomically), so a rounding flip
    between the two shardings propagates: 1e-2 there -- a sharding bug is O(1).  The 640-token
    prompt runs the MFMA prefill in one chunk whose all-reduces (640 x d_model) take the two-shot
    path with bf16 staging, split over several calls; the 9-token one takes the skinny GEMM
    (prompts of 4-15 tokens)."""
    out = tmp_path / f"tp{world}.json"
    port = 29600 + world + 10 * gemm_prefill + (20 if prompt_len > 100 else 0)
    cmd = [sys.executable, "-m", "torch.distributed.run", "--nnodes", "1", "--nproc-per-node", str(world),
           "--master-addr", "127.0.0.1", "--master-port", str(port),
           os.path.join(ROOT, "tools", "tp_check.py"), "--out", str(out), "--model", "test-tp8-shape",
           "--prompt-len", str(prompt_len)]
    env = dict(os.environ, AIOS_PREFILL_GEMM=str(gemm_prefill))
    r = subprocess.run(cmd, cwd=ROOT, capture_output=True, text=True, timeout=600, env=env)
    assert r.returncode == 0, r.stderr[-3000:]
    res = json.loads(out.read_text())
    assert not res["comm_error_flag"] and not res["comm_error_flag_model"]
    assert res["vocab_parallel"]
    # the batch-1 O / down all-reduces run in the GEMV engine's epilogue (EPI_TP_RESID) by default,
    # with the engine grid capped so that every rank sharing this GPU is resident at once
    assert res["tp_fused"] == (os.environ.get("AIOS_TP_FUSE", "1") != "0")
    for e in res["allreduce"]:
        # fp32 staging: summation order only; bf16 two-shot staging: one bf16 rounding per partial
        tol = world * e["scale"] * 2.0 ** -8 if (e["bf16"] and e["two_shot"]) else 1e-4
        assert e["inplace_err"] < tol and e["fused_resid_err"] < tol + 1e-4, e
    assert any(e["two_shot"] for e in res["allreduce"])
    for e in res["allgather"]:
        assert e["err"] == 0.0, e
    m = res["model"]
    tol = (1e-2 if gemm_prefill else 1e-3) * max(1.0, m["logit_scale"])
    assert m["prefill_logit_max_abs_diff"] < tol
    assert max(m["decode_logit_max_abs_diff_per_step"]) < tol
    if not gemm_prefill:
        assert m["graph_tokens_match"]


@pytest.mark.gpu
@pytest.mark.parametrize("world", [2, 4, 8])
def test_tp_fused_epilogue_int8_activations(tmp_path, world):
    """the production TP decode path -- int8 GEMV activations, the batch-1 O / down
    all-reduces in the row-pair GEMV epilogue (EPI_TP_RESID: per-slot epochs, double-buffered stage
    halves, peer flags) -- against AIOS_TP_FUSE=0 (separate all-reduce launches) and against TP=1,
    over 24 decode steps (each stage half reused a dozen times per layer) plus the graph loop."""
    outs = {}
    for fuse in ("1", "0"):
        out = tmp_path / f"tpq{world}_{fuse}.json"
        cmd = [sys.executable, "-m", "torch.distributed.run", "--nnodes", "1", "--nproc-per-node", str(world),
               "--master-addr", "127.0.0.1", "--master-port", str(29700 + 2 * world + int(fuse)),
               os.path.join(ROOT, "tools", "tp_check.py"), "--out", str(out), "--model", "test-tp8-shape",
               "--prompt-len", "21", "--steps", "24", "--act-q8", "--dump-logits"]
        env = dict(os.environ, AIOS_TP_FUSE=fuse, AIOS_PREFILL_GEMM="0")
        r = subprocess.run(cmd, cwd=ROOT, capture_output=True, text=True, timeout=600, env=env)
        assert r.returncode == 0, r.stderr[-3000:]
        outs[fuse] = json.loads(out.read_text())
    on, off = outs["1"], outs["0"]
    assert on["tp_fused"] and not off["tp_fused"]
    for res in (on, off):
        assert not res["comm_error_flag"] and not res["comm_error_flag_model"]
        m = res["model"]
        assert m["act_q8"] and m["graph_tokens_match"]
        # the int8 path quantises the sharded activations per shard (norm-scaled x, the SwiGLU output of
        # each shard): ~1e-2 of the logit scale against TP=1 by design; a sharding bug is O(1)
        tol = 5e-2 * max(1.0, m["logit_scale"])
        assert max(m["decode_logit_max_abs_diff_per_step"]) < tol, m["decode_logit_max_abs_diff_per_step"]
    import numpy as np

    a, b = np.asarray(on["model"]["step_logits"]), np.asarray(off["model"]["step_logits"])
    assert on["model"]["tp_tokens"] == off["model"]["tp_tokens"]
    assert np.abs(a - b).max() < 1e-3 * max(1.0, np.abs(b).max())


@pytest.mark.gpu
def test_tp_shared_gpu_with_cotenant_decode(tmp_path):
    """TP=2 with both ranks sharing this GPU WHILE a third process runs a TinyLlama
    decode loop on the same GPU (the co-resident operational tier): the spinning all-reduce / fused
    epilogue workgroups must still meet (no comm.error(), numerics as without the co-tenant); the
    slowdown of both is recorded."""
    def tp_run(tag):
        out = tmp_path / f"tpc_{tag}.json"
        cmd = [sys.executable, "-m", "torch.distributed.run", "--nnodes", "1", "--nproc-per-node", "2",
               "--master-addr", "127.0.0.1", "--master-port", str(29760 + (tag == "cotenant")),
               os.path.join(ROOT, "tools", "tp_check.py"), "--out", str(out), "--model", "test-tp8-shape",
               "--prompt-len", "21", "--steps", "16", "--act-q8"]
        r = subprocess.run(cmd, cwd=ROOT, capture_output=True, text=True, timeout=600,
                           env=dict(os.environ, AIOS_PREFILL_GEMM="0"))
        assert r.returncode == 0, r.stderr[-3000:]
        return json.loads(out.read_text())

    alone = tp_run("alone")
    stop = tmp_path / "stop"
    co = subprocess.Popen([sys.executable, os.path.join(ROOT, "tools", "cotenant_decode.py"), "--seconds", "240",
                           "--stop-file", str(stop)], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
    try:
        line = ""
        t0 = time.time()
        while "ready" not in line and time.time() - t0 < 180:
            line = co.stdout.readline()
            if not line and co.poll() is not None:
                break
        assert "ready" in line, co.stderr.read()[-2000:]
        shared = tp_run("cotenant")
    finally:
        stop.write_text("1")
        try:
            outs, errs = co.communicate(timeout=60)
        except subprocess.TimeoutExpired:
            co.kill()
            outs, errs = co.communicate()
    assert co.returncode == 0, errs[-2000:]
    cot = json.loads([l for l in outs.splitlines() if l.startswith("{")][-1])
    for res in (alone, shared):
        assert not res["comm_error_flag"] and not res["comm_error_flag_model"]
        m = res["model"]
        assert m["graph_tokens_match"]
        assert max(m["decode_logit_max_abs_diff_per_step"]) < 5e-2 * max(1.0, m["logit_scale"])
    assert shared["model"]["tp_tokens"] == alone["model"]["tp_tokens"]
    print(json.dumps({"allreduce_us_8192_alone": alone["allreduce_us_8192"],
                      "allreduce_us_8192_with_cotenant": shared["allreduce_us_8192"],
                      "cotenant_tok_s": cot["tok_s"]}))


@pytest.mark.gpu
@pytest.mark.parametrize("norm_fuse", [1, 0])
def test_tp_batched_decode_fused_norm(tmp_path, norm_fuse):
    """Batched TP decode (B = 6: the skinny-GEMM path) with C1 / C2 fused with the next RMSNorm: the
    all-reduce writes bf16(x * g) and per-1024-column sums of squares (d_model 2048: two real parts,
    two zero pads) that the gate/up / next QKV / lm_head GEMMs consume -- every row's logits against
    the unsharded engine at the same batch; norm_fuse 0 is the separate-RMSNorm control.  Also the
    fused collective itself (one-shot and the two-shot + add-norm fallback) against torch."""
    out = tmp_path / "tpb.json"
    cmd = [sys.executable, "-m", "torch.distributed.run", "--nnodes", "1", "--nproc-per-node", "2",
           "--master-addr", "127.0.0.1", "--master-port", str(29680 + norm_fuse),
           os.path.join(ROOT, "tools", "tp_check.py"), "--out", str(out), "--model", "test-tp8-shape",
           "--prompt-len", "21", "--batch", "6", "--steps", "6"]
    env = dict(os.environ, AIOS_TP_NORM_FUSE=str(norm_fuse))
    r = subprocess.run(cmd, cwd=ROOT, capture_output=True, text=True, timeout=600, env=env)
    assert r.returncode == 0, r.stderr[-3000:]
    res = json.loads(out.read_text())
    assert not res["comm_error_flag"] and not res["comm_error_flag_model"]
    for e in res["allreduce_norm"]:
        tol = 2 * e["scale"] * 2.0 ** -8 if e["two_shot"] else 1e-4
        assert e["resid_err"] < tol, e
        assert e["out16_rel"] < 2.0 ** -7 and e["part_rel"] < (1e-2 if e["two_shot"] else 1e-5), e
    assert any(e["two_shot"] for e in res["allreduce_norm"])
    b = res["batched"]
    assert max(b["decode_logit_max_abs_diff_per_step"]) < 1e-2 * max(1.0, b["logit_scale"]), b


@pytest.mark.gpu
def test_runtime_serves_tp_model(tmp_path):
    """ModelManager hosts a TP=2 strategic model (worker process + xGMI all-reduce) and its
    greedy generations through the continuous-batching scheduler equal the TP=1 model's."""
    import asyncio
    import threading

    from aios_amd.models.config import get_preset
    from aios_amd.models.synthetic import write_synthetic_gguf
    from aios_amd.runtime.model_manager import ModelManager
    from aios_amd.runtime.scheduler import GenRequest

    path = str(tmp_path / "m.gguf")
    write_synthetic_gguf(path, get_preset("test-tp8-shape"), "Q4_K_M", seed=3)
    mgr = ModelManager(max_batch=4, max_slots=4)

    def gen(m, prompts):
        outs, evs = [None] * len(prompts), [threading.Event() for _ in prompts]
        for i, p in enumerate(prompts):
            def done(r, i=i):
                outs[i] = r
                evs[i].set()
            m.scheduler.submit(GenRequest(prompt_ids=m.tokenizer.encode(p), on_done=done, max_tokens=10))
        for e in evs:
            assert e.wait(120)
        return [o.token_ids for o in outs]

    async def load(name, spec):
        m = await mgr.load_model(name, spec, context_length=256)
        assert m.status == "ready", m.error
        return m

    prompts = ["alpha beta gamma", "the strategic tier", "json { }"]
    m1 = asyncio.run(load("ref", path + "#q8=0"))
    ref = gen(m1, prompts)
    asyncio.run(mgr.unload_model("ref"))
    m2 = asyncio.run(load("llama3-70b", path + "#tp=2&q8=0"))
    try:
        assert type(m2.engine).__name__ == "TPEngine"
        assert mgr.select_model_for_level("strategic") == "llama3-70b"
        assert gen(m2, prompts) == ref
    finally:
        asyncio.run(mgr.unload_model("llama3-70b"))


def test_comm_kind_selection(monkeypatch):
    from aios_amd.parallel.tp import comm_kind

    monkeypatch.delenv("AIOS_TP_COMM", raising=False)
    assert comm_kind() == "xgmi"
    monkeypatch.setenv("AIOS_TP_COMM", "RCCL")
    assert comm_kind() == "rccl"
    monkeypatch.setenv("AIOS_TP_COMM", "mpi")
    with pytest.raises(ValueError):
        comm_kind()


@pytest.mark.gpu
def test_rccl_comm_single_rank():
    """RcclComm (librccl dlopen'd): a world-1 communicator on the box's GPU -- all-reduce is the
    identity plus the fused residual add, the column all-gather a no-op; captured into a hipGraph
    as the engine captures it.  (World > 1 needs one GPU per rank: RCCL refuses shared devices.)"""
    import torch

    from aios_amd.runtime import native

    m = native.require()
    assert m.RcclComm.available()
    uid = m.RcclComm.unique_id()
    assert isinstance(uid, bytes) and len(uid) == 128
    comm = m.RcclComm(0, 1, 0, uid)
    assert comm.rank == 0 and comm.world == 1 and not comm.error()
    st = torch.cuda.current_stream()
    data = torch.randn(4096, device="cuda")
    res = torch.randn(4096, device="cuda")
    want = res + data
    comm.allreduce(data.data_ptr(), data.numel(), res.data_ptr(), st.cuda_stream)
    torch.cuda.synchronize()
    assert torch.allclose(res, want)
    # fused residual add + split-RMSNorm producer (the batched TP decode's C1 / C2 epilogue)
    rows, d = 3, 3072
    parts = m.resid_norm_parts(d)
    assert parts == 4
    x, r0, gw = torch.randn(rows, d, device="cuda"), torch.randn(rows, d, device="cuda"), torch.rand(d, device="cuda")
    r = r0.clone()
    o16 = torch.empty(rows, d, dtype=torch.bfloat16, device="cuda")
    pt = torch.full((rows, parts), 5.0, device="cuda")
    comm.allreduce_norm(x.data_ptr(), rows, d, r.data_ptr(), gw.data_ptr(), o16.data_ptr(), d, pt.data_ptr(), parts,
                        st.cuda_stream)
    torch.cuda.synchronize()
    assert torch.allclose(r, r0 + x)
    assert torch.allclose(o16.float(), (r * gw).bfloat16().float())
    wp = torch.cat([(r.reshape(rows, 3, 1024) ** 2).sum(-1), torch.zeros(rows, 1, device="cuda")], 1)
    assert torch.allclose(pt, wp, rtol=1e-5)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        comm.allreduce(data.data_ptr(), data.numel(), res.data_ptr(), torch.cuda.current_stream().cuda_stream)
    g.replay()
    torch.cuda.synchronize()
    assert torch.allclose(res, want + data)
    logits = torch.randn(2, 64, device="cuda")
    before = logits.clone()
    comm.allgather_cols(logits.data_ptr(), 2, 64, 64, st.cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(logits, before)
    assert not comm.error()
