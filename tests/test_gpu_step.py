"""A session's decode step as one launch for all layers (wr_hip_attn_step_dev) against the
chain of launches it stands for: same logits, bit for bit, and the same cache behind them."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from wayruntime_amd import engine as E, gguf_writer as gw, hipattn

pytestmark = pytest.mark.gpu

VOCAB = 512


def test_refusals():
    """What the launch is not built for is refused before anything is launched."""
    hipattn.init()
    lib = hipattn.lib()
    w = {n: hipattn.Weight([np.zeros(n, np.uint16)]) for n in [(1024, 512), (512, 512), (640, 512), (1024, 640)]}
    vec = lib.wr_hip_attn_dev_alloc(4096)

    def create(qkv, o, gu, down, nq=4, nkv=2, hd=128):
        y = hipattn.StepLayer(w[qkv].h, w[o].h, w[gu].h, w[down].h, vec, vec, None, None)
        h = C.c_void_p()
        rc = lib.wr_hip_attn_step_create(1, C.byref(y), nq, nkv, hd, 1e-6, C.byref(h))
        return rc, h

    rc, h = create((1024, 512), (512, 512), (1024, 512), (512, 512))
    assert rc == hipattn.OK
    assert create((1024, 512), (512, 512), (1024, 512), (512, 512), hd=64)[0] == hipattn.ERR_UNSUPPORTED
    assert create((640, 512), (512, 512), (1024, 512), (512, 512))[0] == hipattn.ERR_UNSUPPORTED
    assert create((1024, 640), (512, 512), (1024, 512), (512, 512))[0] == hipattn.ERR_UNSUPPORTED
    assert create((1024, 512), (512, 512), (1024, 512), (512, 512), nq=3)[0] == hipattn.ERR_INVAL
    kv = hipattn.KVCache(1, 128, 2, 64)
    other = hipattn.KVCache(1, 64, 2, 64)
    assert lib.wr_hip_attn_step_dev(h, kv.h, 64, vec, None, 0, 0.0) == hipattn.ERR_CTX_FULL
    assert lib.wr_hip_attn_step_dev(h, other.h, 0, vec, None, 0, 0.0) == hipattn.ERR_INVAL
    assert lib.wr_hip_attn_step_dev(h, kv.h, 0, vec, None, 8, 0.0) == hipattn.ERR_INVAL
    assert lib.wr_hip_attn_step_dev(h, kv.h, 0, vec + 4, None, 0, 0.0) == hipattn.ERR_UNSUPPORTED
    lib.wr_hip_attn_set_tuning(0, 1)
    try:
        assert lib.wr_hip_attn_step_dev(h, kv.h, 0, vec, None, 0, 0.0) == hipattn.ERR_UNSUPPORTED
    finally:
        lib.wr_hip_attn_set_tuning(0, 0)
    lib.wr_hip_attn_step_destroy(h)
    for x in (kv, other):
        x.close()
    for x in w.values():
        x.close()
    lib.wr_hip_attn_dev_free(vec)


def test_tags_begin_again():
    """Rows travel with a 32-bit number of their layer: a plan whose numbers run out clears its rows and begins again,
    and the steps on either side are those of any other numbers.  One split of the keys, and several."""
    hipattn.init()
    lib, rng = hipattn.lib(), np.random.default_rng(8)
    n, hidden = 2, 512
    w = [[hipattn.Weight([(rng.standard_normal((o, 512)) / 16).astype(np.float16).view(np.uint16)]) for o in (1024, 512, 1024, 512)]
         for _ in range(n)]
    vec = hipattn.DeviceBuffer.from_host(rng.standard_normal(hidden).astype(np.float32))
    layers = (hipattn.StepLayer * n)(*[hipattn.StepLayer(*[x.h for x in ws], vec.p, vec.p, None, None) for ws in w])
    plan, kv = C.c_void_p(), hipattn.KVCache(n, 128, 2, 400)
    assert lib.wr_hip_attn_step_create(n, layers, 4, 2, 128, 1e-6, C.byref(plan)) == hipattn.OK
    x = rng.standard_normal(hidden).astype(np.float32)
    row = hipattn.DeviceBuffer(hidden * 4)

    def step(pos):
        assert lib.wr_hip_attn_h2d(row.p, x.ctypes.data, x.nbytes) == hipattn.OK
        assert lib.wr_hip_attn_step_dev(plan, kv.h, pos, row.p, None, 0, 0.0) == hipattn.OK
        assert lib.wr_hip_attn_step_done() == hipattn.OK
        return row.to_host((hidden,)).tobytes()

    last = 2 ** 32 - 1 - 2 * n                               # the last number that a step's may begin at
    for pos in (10, 390):
        want = step(pos)
        assert np.isfinite(np.frombuffer(want, np.float32)).all()
        for tag in (last + 1, last, last - 1, last - 3, 2):
            lib.wr_hip_attn_step_set_tag(plan, tag)
            assert all(step(pos) == want for _ in range(4)), (pos, tag)
    lib.wr_hip_attn_step_destroy(plan)
    kv.close()
    for ws in w:
        for x in ws:
            x.close()
    for b in (vec, row):
        b.free()


def test_memory_that_steps_wrote_comes_back_cleared():
    """A step writes its K and V by itself, in every layer: the next cache of that size finds zeros there too."""
    hipattn.init()
    lib, rng = hipattn.lib(), np.random.default_rng(9)
    n, hidden, ctx = 2, 512, 1000
    w = [[hipattn.Weight([(rng.standard_normal((o, 512)) / 16).astype(np.float16).view(np.uint16)]) for o in (1024, 512, 1024, 512)]
         for _ in range(n)]
    vec = hipattn.DeviceBuffer.from_host(rng.standard_normal(hidden).astype(np.float32))
    layers = (hipattn.StepLayer * n)(*[hipattn.StepLayer(*[x.h for x in ws], vec.p, vec.p, None, None) for ws in w])
    plan = C.c_void_p()
    assert lib.wr_hip_attn_step_create(n, layers, 4, 2, 128, 1e-6, C.byref(plan)) == hipattn.OK
    row = hipattn.DeviceBuffer.from_host(rng.standard_normal(hidden).astype(np.float32))
    for pos in (0, 31, 32, 300, 7):
        kv = hipattn.KVCache(n, 128, 2, ctx)
        for layer in range(n):
            assert not any(x.any() for x in kv.read_f16(layer, 0, ctx)), pos
        assert lib.wr_hip_attn_step_dev(plan, kv.h, pos, row.p, None, 0, 0.0) == hipattn.OK
        assert lib.wr_hip_attn_step_done() == hipattn.OK
        for layer in range(n):
            assert all(x.any() for x in kv.read_f16(layer, pos, 1))
        kv.close()
    lib.wr_hip_attn_step_destroy(plan)
    for ws in w:
        for x in ws:
            x.close()
    for b in (vec, row):
        b.free()


@pytest.fixture(scope="module")
def eng():
    hipattn.shutdown()
    e = E.Engine(E.HOST_SO)
    yield e
    e.close()


def _models(eng, tmp_path, monkeypatch, **shape):
    """The model with its steps in one launch, and as a chain."""
    p = str(tmp_path / "m.gguf")
    gw.write_model(p, gw.ModelShape(head_dim=128, vocab=VOCAB, context=8192, **shape), std=0.08)
    out = []
    for chain in ("0", "1"):
        monkeypatch.setenv("WAYRT_STEP_LAUNCHES", chain)
        out.append(eng.load(p, max_context=8192))
    return out


def _steps(model, prompt, tokens):
    s = model.session()
    if len(prompt):
        assert s.prefill(prompt) == len(prompt)
    rows = [np.array(s.step(int(t))) for t in tokens]
    # the cache that the steps left: a prompt pass over it
    assert s.prefill(tokens) == len(tokens)
    rows.append(np.array(s.step(int(tokens[0]))))
    s.close()
    return rows


def _batches(model, prompts, tokens):
    ss = [model.session() for _ in prompts]
    for s, p in zip(ss, prompts):
        assert s.prefill(p) == len(p)
    rows = []
    for t in tokens:
        rc, got = E.batch_step(ss, [int(t)] * len(ss))
        assert rc == len(ss)
        rows += [np.array(r) for r in got]
    for s in ss:
        s.close()
    return rows


def _launches(model, session=None):
    lib, ms, n = hipattn.lib(), C.c_double(), C.c_uint32()
    s = session or model.session()
    assert lib.wr_hip_attn_profile_begin(1000) == hipattn.OK
    s.step(1)
    assert lib.wr_hip_attn_profile_end(C.byref(ms), C.byref(n)) == hipattn.OK
    if not session:
        s.close()
    return n.value


# the fewest inputs and the most that a wave holds; KV groups of 1 to 8; with head norms and without
@pytest.mark.parametrize("shape", [
    dict(n_layers=2, hidden=512, ffn=512, n_q=4, n_kv=4),
    dict(n_layers=1, hidden=512, ffn=2560, n_q=8, n_kv=1),
    dict(n_layers=3, hidden=1536, ffn=3072, n_q=12, n_kv=3),
    dict(n_layers=2, hidden=1024, ffn=1536, n_q=24, n_kv=3),
    dict(n_layers=2, hidden=1024, ffn=3072, n_q=16, n_kv=8, arch="llama"),
])
def test_one_launch_equals_the_chain(eng, tmp_path, monkeypatch, shape):
    one, chain = _models(eng, tmp_path, monkeypatch, **shape)
    rng = np.random.default_rng(5)
    # nothing cached; ends of a tile; the last split on its own; splits of a short, a medium and a long session
    for n in (0, 1, 30, 31, 32, 33, 159, 160, 161, 300, 1000, 2047, 2100, 4096, 8100):
        prompt, tokens = rng.integers(0, VOCAB, n).astype(np.uint32), rng.integers(0, VOCAB, 4).astype(np.uint32)
        for a, b in zip(_steps(one, prompt, tokens), _steps(chain, prompt, tokens)):
            assert np.isfinite(b).all() and np.array_equal(a, b), n
    # (the layers and the LM head; five launches a layer and the head)
    assert _launches(one) == 2 and _launches(chain) == 5 * shape["n_layers"] + 1
    for m in (one, chain):
        m.close()


def test_a_step_that_gives_up_is_made_again(eng, tmp_path, monkeypatch):
    one, chain = _models(eng, tmp_path, monkeypatch, n_layers=2, hidden=1024, ffn=3072, n_q=16, n_kv=8)
    rng = np.random.default_rng(6)
    prompt, tokens = rng.integers(0, VOCAB, 200).astype(np.uint32), rng.integers(0, VOCAB, 5).astype(np.uint32)
    lib = hipattn.lib()
    calls = eng.counters()[E.WR_CTR_ATTENTION_CALLS]
    want = _steps(chain, prompt, tokens)
    a_run = eng.counters()[E.WR_CTR_ATTENTION_CALLS] - calls
    lib.wr_hip_attn_set_step_limit(1)            # every wait ends at once, the launch runs through without its rows
    try:
        got = _steps(one, prompt, tokens)
    finally:
        lib.wr_hip_attn_set_step_limit(0)
    assert all(np.array_equal(a, b) for a, b in zip(got, want))
    assert all(np.array_equal(a, b) for a, b in zip(_steps(one, prompt, tokens), want))
    assert eng.counters()[E.WR_CTR_ATTENTION_CALLS] - calls == 3 * a_run
    for m in (one, chain):
        m.close()


def test_threads_step_beside_each_other(eng, tmp_path, monkeypatch):
    """One launch at a time is on the device; whoever comes second takes the chain, and nobody sees a difference."""
    one, chain = _models(eng, tmp_path, monkeypatch, n_layers=4, hidden=1024, ffn=3072, n_q=16, n_kv=8)
    rng = np.random.default_rng(7)
    work = [(rng.integers(0, VOCAB, 40 + 90 * i).astype(np.uint32), rng.integers(0, VOCAB, 24).astype(np.uint32)) for i in range(4)]
    want = [_steps(chain, *w) for w in work]
    got = [None] * 4

    def run(i):
        got[i] = _steps(one, *work[i])

    threads = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g, w in zip(got, want):
        assert g is not None and all(np.array_equal(a, b) for a, b in zip(g, w))
    for m in (one, chain):
        m.close()


@pytest.mark.parametrize("rows", [1, 8, 64])
def test_a_step_beside_another_threads_work(eng, tmp_path, monkeypatch, rows):
    """One launch would keep another thread's chain of launches or its prompt waiting for as long as it runs: the step
    goes layer by layer then.  Beside a batched step's products, which fill the device too, it does not."""
    one, chain = _models(eng, tmp_path, monkeypatch, n_layers=2, hidden=1024, ffn=3072, n_q=16, n_kv=8)
    lib = hipattn.lib()
    monkeypatch.setattr(hipattn, "_inited", True)            # by the engine
    T, nq, hd = 8192, 32, 128
    kv, w = hipattn.KVCache(1, hd, 8, T), hipattn.Weight([np.zeros((64, 64), np.uint16)])
    q, out, x, y = (hipattn.DeviceBuffer(n * 4) for n in (T * nq * hd, T * nq * hd, 64 * 64, 64 * 64))
    waiting, done = threading.Event(), threading.Event()

    def other():
        for _ in range(150):                                 # some 150 ms of it
            assert lib.wr_hip_attn_prefill_dev(kv.h, 0, 0, T, q.p, out.p, nq, 0.0, 0) == hipattn.OK
        assert lib.wr_hip_proj_rows_dev(w.h, rows, x.p, 64, None, y.p, 64) == hipattn.OK
        waiting.set()
        hipattn.sync()
        done.set()

    s = one.session()                                        # (making one and ending it waits for the whole device)
    _launches(one, s)                                        # (a first call on every path)
    t = threading.Thread(target=other)
    t.start()
    assert waiting.wait(60)
    time.sleep(0.002)
    beside = _launches(one, s)
    assert not done.is_set()                                 # it was under way all the time
    t.join()
    assert beside == (2 if rows == 8 else 11)
    assert _launches(one, s) == 2
    s.close()
    for o in (kv, w):
        o.close()
    for b in (q, out, x, y):
        b.free()
    for m in (one, chain):
        m.close()


@pytest.mark.parametrize("limit", [0, 1])                    # 1: whichever step takes the launch gives up
def test_steps_beside_prompts_and_batches(eng, tmp_path, monkeypatch, limit):
    one, chain = _models(eng, tmp_path, monkeypatch, n_layers=3, hidden=1024, ffn=3072, n_q=16, n_kv=8)
    rng = np.random.default_rng(9)
    ids = lambda n: rng.integers(0, VOCAB, n).astype(np.uint32)
    jobs = [(_steps, ids(50), ids(40)), (_steps, ids(700), ids(40)), (_steps, ids(1500), ids(2)),
            (_batches, [ids(20 + 30 * i) for i in range(5)], ids(25))]
    want = [f(chain, *args) for f, *args in jobs]
    got = [None] * len(jobs)

    def run(i):
        f, *args = jobs[i]
        got[i] = [f(one, *args) for _ in range(3)]

    hipattn.lib().wr_hip_attn_set_step_limit(limit)
    try:
        threads = [threading.Thread(target=run, args=(i,)) for i in range(len(jobs))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        hipattn.lib().wr_hip_attn_set_step_limit(0)
    for g, w in zip(got, want):
        assert g is not None and all(np.array_equal(a, b) for again in g for a, b in zip(again, w))
    assert _launches(one) == 2                               # and alone again
    for m in (one, chain):
        m.close()


def test_more_sessions_than_rows_of_logits_are_kept(eng, tmp_path, monkeypatch):
    one, chain = _models(eng, tmp_path, monkeypatch, n_layers=2, hidden=512, ffn=512, n_q=4, n_kv=4)
    want = []
    for i in range(20):
        s = chain.session(64)
        want.append(np.array(s.step(i)))
        s.close()
    for _ in range(3):                                       # sixteen of a round's rows are the next round's
        ss = [one.session(64) for _ in range(20)]
        rows = [s.step(i) for i, s in enumerate(ss)]
        assert all(np.array_equal(a, b) for a, b in zip(rows, want))
        for s in ss:
            s.close()
    for m in (one, chain):
        m.close()
