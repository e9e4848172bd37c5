"""Decode steps of few rows as one resident launch (kernels/decode_stream.hip) against the chain of launches it stands in for."""
import dataclasses
import threading
import time

import numpy as np
import pytest
import torch

from aios_amd.models.config import get_preset
from aios_amd.models.reference import ReferenceModel
from aios_amd.models.synthetic import write_synthetic_gguf
from aios_amd.runtime.loader import load_engine

pytestmark = pytest.mark.gpu

BASE = get_preset("test-mistral-shape")  # 1024 wide, 8 / 2 heads of 128, 2048 hidden, 1024 tokens
SHAPES = {
    "gqa4-128": {},
    "gqa2-128": dict(n_kv_heads=4, vocab_size=1002),              # a head of a vocabulary that no workgroup count divides
    "gqa8-64": dict(d_model=1536, n_heads=16, n_kv_heads=2, head_dim=64, d_ff=1536),  # rows of 48 chunks: eight lanes share one
    "gqa4-64": dict(n_heads=16, n_kv_heads=4, head_dim=64, d_ff=2560),
    "mha-64": dict(d_model=512, n_heads=8, n_kv_heads=8, head_dim=64, d_ff=1024, vocab_size=4098),
    "qwen": dict(n_kv_heads=4, qk_norm=True, rope_mode=2, d_ff=3072),
}
# both int8-activation paths are 0.013 from 64 bits (perf/cases.py); they differ in the order of fp32 sums and in codes that this rounds
# the other way, so by no more than the two distances together
TOL = 0.026
# bf16 weights and operands: 0.0036 from 64 bits each (perf/cases.py), and further apart in the largest of a few hundred rows
TOL16 = 0.015


@pytest.fixture(scope="module")
def models(tmp_path_factory):
    d, held = tmp_path_factory.mktemp("resident"), {}

    def get(name, recipe="Q4_K_M"):
        if (name, recipe) not in held:
            cfg = dataclasses.replace(BASE, max_ctx=2048, **SHAPES[name])
            held[name, recipe] = write_synthetic_gguf(str(d / f"{name}-{recipe}.gguf"), cfg, recipe, seed=11)
        return held[name, recipe]

    return get


def _engine(path, **kw):
    eng, cfg, _ = load_engine(path, max_ctx=kw.pop("max_ctx", 2048), max_batch=kw.pop("max_batch", 2), **kw)
    assert eng.decode_resident
    return eng, cfg


def _steps(eng, slot, tokens, pos, on=None):
    out = []
    for i, t in enumerate(tokens):
        eng.decode([slot], [t], [pos + i])
        assert on is None or eng.decode_resident_last == on
        out.append(np.asarray(eng.last_logits(1), np.float64).reshape(-1))
    return np.array(out)


def _rel(a, b):
    return np.linalg.norm(a - b, axis=-1) / np.linalg.norm(b, axis=-1)


# the first token, one cached key, a block's border, the borders of one workgroup a head (512 keys of 128, 1280 of 64), passes of 128 and 256
# keys, a last pass that holds the row's own key alone
POSITIONS = [0, 1, 127, 128, 510, 511, 512, 767, 1023, 1024, 1278, 1279, 1280, 1500]


@pytest.mark.parametrize("kv", ["bf16", "fp8_e4m3"])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_resident_step_is_the_chains(models, shape, kv):
    eng, cfg = _engine(models(shape), kv_dtype=kv)
    if kv != "bf16":
        eng.set_kv_scales([1 / 64] * (2 * cfg.n_layers))
    rng = np.random.default_rng(3)
    for pos in POSITIONS:
        prompt = [int(t) for t in rng.integers(3, cfg.vocab_size, pos)]
        tokens = [int(t) for t in rng.integers(3, cfg.vocab_size, 3)]
        got = []
        for slot, on in ((0, False), (1, True)):
            eng.set_decode_resident(on)
            eng.release_slot(slot)
            if pos:
                eng.prefill(slot, prompt, 0, False)
            got.append(_steps(eng, slot, tokens, pos, on))
        assert np.isfinite(got[1]).all()
        assert _rel(got[1], got[0]).max() < TOL, (pos, _rel(got[1], got[0]))
    assert eng.decode_resident_failed == 0


def _rows(eng, cfg, contexts, slots, seed, on=None):
    """Logits of two steps of a batch behind contexts of these lengths"""
    rng = np.random.default_rng(seed)
    for s, n in zip(slots, contexts):
        eng.release_slot(s)
        if n:
            eng.prefill(s, [int(t) for t in rng.integers(3, cfg.vocab_size, n)], 0, False)
    out = []
    for i in range(2):
        eng.decode(slots, [int(t) for t in rng.integers(3, cfg.vocab_size, len(slots))], [n + i for n in contexts])
        assert on is None or eng.decode_resident_last == on
        out.append(np.asarray(eng.last_logits(len(slots)), np.float64).reshape(len(slots), -1))
    return np.concatenate(out)


# one to four rows; short ones beside one that has its keys split, and beside one in its last pass
BATCHES = [[0], [300], [700], [0, 1], [128, 511], [40, 512], [1, 0, 500], [1500, 3, 700], [7, 130, 256, 33], [1023, 1, 512, 1300]]


@pytest.mark.parametrize("kv", ["bf16", "fp8_e4m3"])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_resident_step_of_bf16_rows_is_the_chains(models, shape, kv):
    eng, cfg = _engine(models(shape, "BF16"), kv_dtype=kv, max_batch=4, max_slots=8)
    assert eng.decode_resident == 4
    if kv != "bf16":
        eng.set_kv_scales([1 / 64] * (2 * cfg.n_layers))
    for n, contexts in enumerate(BATCHES):
        got = []
        for at, on in ((0, False), (4, True)):
            eng.set_decode_resident(on)
            got.append(_rows(eng, cfg, contexts, list(range(at, at + len(contexts))), n, on))
        assert np.isfinite(got[1]).all()
        assert _rel(got[1], got[0]).max() < TOL16, (contexts, _rel(got[1], got[0]))
    assert eng.decode_resident_failed == 0


@pytest.mark.parametrize("shape", ["gqa4-128", "gqa8-64", "qwen"])
def test_resident_step_matches_the_reference(models, shape):
    path = models(shape)
    eng, cfg = _engine(path)
    ref = ReferenceModel.from_gguf(path, kv_bf16=True, act_q8=True)
    toks = [1] + [int(t) for t in np.random.default_rng(5).integers(3, cfg.vocab_size, 43)]
    eng.prefill(0, toks[:40], 0, False)
    got = torch.from_numpy(_steps(eng, 0, toks[40:], 40, True))
    want = ref.forward(toks)[40:].double()
    assert (got - want).abs().max().item() < 2e-2 * max(want.abs().max().item(), 1.0)


@pytest.mark.parametrize("shape,recipe,batch", [("gqa8-64", "Q4_K_M", 1), ("qwen", "BF16", 1), ("gqa4-64", "BF16", 3), ("mha-64", "BF16", 4)])
def test_a_step_done_again_gives_the_same_logits(models, shape, recipe, batch):
    """Rows whose sums have more terms than two, added in the order in which the waves come"""
    eng, cfg = _engine(models(shape, recipe), max_batch=4, max_slots=4)
    slots = list(range(batch))
    for s in slots:
        eng.prefill(s, [int(t) for t in np.random.default_rng(s).integers(3, cfg.vocab_size, 40 + s)], 0, False)
    first = None
    for _ in range(30):
        eng.decode(slots, [11 + s for s in slots], [40 + s for s in slots])
        assert eng.decode_resident_last
        got = np.asarray(eng.last_logits(batch)).copy()
        first = got if first is None else first
        assert np.array_equal(got, first)


def test_pipelined_and_looped_steps_are_resident_too(models):
    eng, cfg = _engine(models("gqa4-128"))
    prompt = [int(t) for t in np.random.default_rng(7).integers(3, cfg.vocab_size, 120)]
    made = []
    for on in (False, True, True):
        eng.set_decode_resident(on)
        eng.release_slot(0)
        eng.prefill(0, prompt, 0, False)
        eng.decode_submit([0], [17], [120])
        assert eng.decode_resident_last == on
        eng.decode_sample()
        toks = []
        for i in range(1, 12):
            eng.decode_submit([0], [], [120 + i])
            assert eng.decode_resident_last == on
            toks += eng.decode_collect()
            eng.decode_sample()
        toks += eng.decode_collect()
        eng.release_slot(0)
        eng.prefill(0, prompt, 0, False)
        eng.decode_loop_prepare([0], [17], [120])
        eng.decode_loop_run(1, 12, True)
        assert eng.decode_resident_last == on
        eng.synchronize()
        assert eng.decode_loop_history(1, 121, 12) == toks
        made.append(toks)
    assert made[0] == made[1] == made[2]


@pytest.mark.parametrize("shape,pos", [("gqa8-64", 0), ("gqa8-64", 600), ("qwen", 5), ("gqa4-128", 1023)])
def test_a_launch_that_cannot_be_resident_is_done_by_the_one_behind(models, shape, pos):
    """No time to wait for the other workgroups: the resident launch gives up, and the launch behind it does the step; the next steps
    take the chain"""
    eng, cfg = _engine(models(shape))
    prompt = [int(t) for t in np.random.default_rng(9).integers(3, cfg.vocab_size, pos)]
    got = []
    for on in (False, True):
        eng.set_decode_resident(on)
        eng.set_decode_resident_wait(0)
        eng.release_slot(0)
        if pos:
            eng.prefill(0, prompt, 0, False)
        got.append(_steps(eng, 0, [21, 22, 23], pos))
    assert eng.decode_resident_failed == 1
    assert _rel(got[1], got[0]).max() < TOL


@pytest.mark.parametrize("shape,recipe,batch", [("gqa8-64", "Q4_K_M", 1), ("qwen", "BF16", 3)])
def test_a_launch_that_loses_a_wait_is_done_by_the_one_behind(models, shape, recipe, batch):
    """No time to wait behind the open gate: waits end with words of no number, the last workgroup to sign out sees the flag of the
    first that gave up, and the launch behind does the step over"""
    eng, cfg = _engine(models(shape, recipe), max_batch=4, max_slots=4)
    contexts = [600, 30, 5][:batch]
    want = _rows(eng, cfg, contexts, list(range(batch)), 3)
    assert eng.decode_resident_last and eng.decode_resident_failed == 0
    eng.set_decode_resident_wait(2000000, 0)
    got = _rows(eng, cfg, contexts, list(range(batch)), 3)
    assert eng.decode_resident_failed == 1
    assert _rel(got, want).max() < (TOL if recipe == "Q4_K_M" else TOL16)


@pytest.mark.parametrize("contexts", [[5], [3, 600, 40], [0, 10, 20, 30]])
def test_bf16_rows_are_done_by_the_launch_behind(models, contexts):
    eng, cfg = _engine(models("gqa8-64", "BF16"), max_batch=4, max_slots=4)
    got = []
    for on in (False, True):
        eng.set_decode_resident(on)
        eng.set_decode_resident_wait(0)
        got.append(_rows(eng, cfg, contexts, list(range(len(contexts))), 3))
    assert eng.decode_resident_failed == 1
    assert _rel(got[1], got[0]).max() < TOL16


def test_engines_beside_each_other(models):
    """Two engines of a process stepping in two threads: neither holds CUs that the other waits for"""
    engs = [_engine(models(n))[0] for n in ("gqa4-128", "gqa8-64")]
    tokens = [int(t) for t in np.random.default_rng(13).integers(3, 1000, 100)]
    want, got = [None, None], [None, None]

    def run(i, out):
        engs[i].release_slot(0)
        engs[i].prefill(0, [5, 6, 7, 8], 0, False)
        out[i] = _steps(engs[i], 0, tokens, 4)

    for i in range(2):
        run(i, want)
    threads = [threading.Thread(target=run, args=(i, got)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert [e.decode_resident_failed for e in engs] == [0, 0]
    for g, w in zip(got, want):
        assert _rel(g, w).max() < TOL


def test_a_step_beside_another_engines_takes_the_chain(models):
    """A resident launch leaves no room for another engine's launches: both take the chain until one of them rests"""
    a, b = (_engine(models(n))[0] for n in ("gqa4-128", "gqa8-64"))
    for e in (a, b):
        e.prefill(0, [5, 6, 7, 8], 0, False)

    def alone(e):
        time.sleep(0.05)
        e.decode([0], [9], [4])
        return e.decode_resident_last

    assert alone(a) and alone(b)
    time.sleep(0.05)
    b.decode_loop_prepare([0], [9], [5])
    b.decode_loop_run(1, 1500, True)  # some hundred milliseconds
    a.decode([0], [9], [5])
    assert not a.decode_resident_last
    b.synchronize()
    assert alone(a)
    del b
    a.decode([0], [9], [6])
    assert a.decode_resident_last


def test_a_warmed_engine_has_the_graphs_of_both_routes(models):
    """What capture_graphs is for: no step captures, whichever route it takes"""
    eng, cfg = _engine(models("gqa4-128"))
    eng.prefill(0, [5, 6, 7, 8], 0, False)
    eng.decode([0], [9], [4])
    assert eng.decode_resident_last and eng.decode_resident == 1
    assert eng.capture_graphs(2) == 6  # two batch sizes: the step, masked and not, and the forward alone
    assert eng.decode_resident_last    # (of the last step still)
    held = eng.decode_graphs
    assert held == 9
    mask = b"\xff" * ((cfg.vocab_size + 7) // 8)
    for on in (True, False):
        eng.set_decode_resident(on)
        eng.decode([0], [9], [4])
        assert eng.decode_resident_last == on
        eng.decode([0], [9], [4], mask=mask)
        eng.decode_submit([0], [9], [4])
        eng.decode_sample()
        eng.decode_collect()
        eng.decode([0, 1], [9, 9], [4, 0])
    assert eng.decode_graphs == held


def test_a_loop_queues_few_resident_steps_ahead(models):
    """A route is chosen when a step is queued: what is queued must not be hundreds of steps old when it runs, in one call or in many"""
    eng, cfg = _engine(models("gqa4-128"))
    for n, calls in ((1000, 1), (10, 100)):
        eng.release_slot(0)
        eng.prefill(0, [5, 6, 7, 8], 0, False)
        eng.decode_loop_prepare([0], [9], [4])
        eng.decode_loop_run(1, 8, True)
        eng.synchronize()
        t0 = time.perf_counter()
        for _ in range(calls):
            eng.decode_loop_run(1, n, True)
        t1 = time.perf_counter()
        assert eng.decode_resident_last
        eng.synchronize()
        t2 = time.perf_counter()
        assert t2 - t1 < 0.1 * (t2 - t0), (t1 - t0, t2 - t1)  # (four steps of a thousand, and what waiting takes)


def test_an_engine_that_captures_is_seen(models):
    """An engine that has only run alone has no graph of the chain.  Its first step beside another captures one, and the other engine's steps,
    resident until then, leave it the GPU meanwhile"""
    a, b = (_engine(models(n))[0] for n in ("gqa4-128", "gqa8-64"))
    for e in (a, b):
        e.prefill(0, [5, 6, 7, 8], 0, False)
        time.sleep(0.05)
        e.decode([0], [9], [4])
        assert e.decode_resident_last
    b.decode_loop_prepare([0], [9], [5])
    b.decode_loop_run(1, 1, True)
    time.sleep(0.05)
    routes, done = [], threading.Event()

    def loop():
        for _ in range(1500):
            b.decode_loop_run(1, 1, True)
            routes.append(b.decode_resident_last)
            if done.is_set():
                return

    t = threading.Thread(target=loop)
    t.start()
    time.sleep(0.02)
    for i in range(20):
        a.decode([0], [9], [5 + i])
        assert not a.decode_resident_last
    done.set()
    t.join()
    b.synchronize()
    assert routes[0] and not routes[-1]  # alone at first; not beside the other
    assert a.decode_resident_failed == b.decode_resident_failed == 0


@pytest.mark.parametrize("kind", ["short", "long", "layered"])
def test_a_step_beside_a_prompt_takes_the_chain(models, kind, tmp_models):
    """A prompt's launches need CUs too: those of another engine's prompt are seen as its decode steps are"""
    a, cfg = _engine(models("gqa4-128"))
    if kind == "layered":
        import test_seledra_gpu

        p = test_seledra_gpu.engine(test_seledra_gpu.model("aligned", tmp_models)[0])
        prompt = [3 + i % 80 for i in range(400)]
    else:
        p = _engine(models("gqa8-64"))[0]
        prompt = [int(t) for t in np.random.default_rng(17).integers(3, 1000, 6 if kind == "short" else 2000)]
    a.prefill(0, [5, 6, 7, 8], 0, False)
    p.prefill(0, prompt, 0, False)
    time.sleep(0.05)
    tokens = [int(t) for t in np.random.default_rng(19).integers(3, 1000, 60)]
    want = _steps(a, 0, tokens, 4, True)
    done = threading.Event()

    def prompts():
        while not done.is_set():
            p.prefill(0, prompt, 0, False)

    t = threading.Thread(target=prompts)
    t.start()
    time.sleep(0.02)
    got, chain = [], 0
    for i, tok in enumerate(tokens):
        a.decode([0], [tok], [4 + i])
        chain += not a.decode_resident_last
        got.append(np.asarray(a.last_logits(1), np.float64).reshape(-1))
    done.set()
    t.join()
    assert chain > len(tokens) // 2  # (between two prompts a step may run resident)
    assert a.decode_resident_failed == 0
    assert _rel(np.array(got), want).max() < TOL
    time.sleep(0.05)
    a.decode([0], [9], [4])
    assert a.decode_resident_last


def test_what_the_resident_step_leaves_to_the_chain(tmp_path):
    """Formats, widths and engines that it is not built for take the chain"""
    small = write_synthetic_gguf(str(tmp_path / "small.gguf"), dataclasses.replace(BASE, d_model=768), "Q4_K_M", seed=7)
    plain = write_synthetic_gguf(str(tmp_path / "plain.gguf"), dataclasses.replace(BASE, d_ff=1280), "BF16", seed=7)
    quant = write_synthetic_gguf(str(tmp_path / "quant.gguf"), BASE, "Q4_K_M", seed=7)
    for path, kw in ((small, {}), (plain, {}), (quant, dict(act_q8=False)), (quant, dict(cu_mask=[0xFFFFFFFF] * 4))):
        eng, cfg, _ = load_engine(path, max_ctx=128, max_batch=1, **kw)
        assert not eng.decode_resident
        assert 0 <= eng.decode([0], [1], [0])[0] < cfg.vocab_size


@pytest.mark.parametrize("recipe,name,value", [
    ("Q4_K_M", "AIOS_DECODE_RESIDENT", "0"), ("Q4_K_M", "AIOS_FF16", "0"), ("BF16", "AIOS_FF16", "0"), ("BF16", "AIOS_GEMV_BF16_LDS", "0"),
    ("Q4_K_M", "AIOS_GEMV_LDS", "0"), ("Q4_K_M", "AIOS_GEMV_GRID_O", "128"), ("Q4_K_M", "AIOS_DECODE_GEMM_MIN_B", "1"),
    ("BF16", "AIOS_DECODE_GEMM_MIN_B", "5"), ("Q4_K_M", "AIOS_FF16", "1"), ("BF16", "AIOS_DECODE_RESIDENT", "1")])
def test_what_the_environment_asks_of_the_chain_is_done_by_it(models, monkeypatch, recipe, name, value):
    monkeypatch.setenv(name, value)
    eng, _, _ = load_engine(models("gqa4-64", recipe), max_ctx=256, max_batch=2)
    default = value == "1" and name != "AIOS_DECODE_GEMM_MIN_B"
    assert bool(eng.decode_resident) == default
    eng.decode([0], [5], [0])
    assert eng.decode_resident_last == default
