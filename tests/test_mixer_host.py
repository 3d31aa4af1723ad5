"""Mixer-stack models through the host engine on the CPU test double (plain loops
in place of the device steps, 32-bit): reading and rearranging weights, the cache
pool, the mixed step, rollback and the error contract, against the plain
implementation of tests/mixer_oracle.py."""
import ctypes as C
import json
import os

import numpy as np
import pytest

import oracle
from tests import mixer_oracle as O
from tests.golden.make_e2e_golden import TINY
from wayruntime_amd import engine as E, gguf_writer as gw, mix_writer as mw

LIGHT = mw.lightning(2, 12, 20, decay=[0.6, 0.99])
LATENT = mw.latent_attention(3, 10, 14, q_rank=18, kv_rank=22, rot_dim=6, window=20, base=777.0, scale=0.3)
CFG = mw.config(40, 61, [(LIGHT, mw.dense(26)), (LATENT, mw.moe(5, 2, 18)), (LIGHT, None),
                         (mw.latent_attention(2, 8, 8, 16, 16, 4, window=70), mw.moe(3, 3, 10))],
                loop=(0, 2, 2), eps=1e-5, logit_scale=0.3)


@pytest.fixture(scope="module")
def eng():
    oracle.build(ref=False)
    e = E.Engine(oracle.HOSTCPU_SO, threads=4)
    e.lib.wrh_debug_poison_scratch(1)
    yield e
    e.lib.wrh_debug_poison_scratch(0)
    e.close()


@pytest.fixture(scope="module")
def made(tmp_path_factory):
    bits = dict(mw.random_tensors(CFG, 4))
    return mw.write_model(str(tmp_path_factory.mktemp("mix") / "m"), CFG, bits), {k: O.bf16_to_f32(v) for k, v in bits.items()}


@pytest.fixture()
def model(eng, made):
    m = eng.load(made[0], max_context=256, quant=E.WR_QUANT_F32)
    yield m
    m.close()


def toks(n, seed=0):
    return np.random.default_rng(seed).integers(0, CFG["vocab"], n)


def near(got, want):
    assert np.sqrt(((got - want) ** 2).mean(-1)).max() < 2e-5 * np.sqrt((want ** 2).mean(-1)).max()


def test_info(model):
    i = model.info
    assert (i.arch, i.quant, i.vocab_size, i.hidden_dim, i.max_context) == (b"Bipotar", b"BF16", 61, 40, 256)
    assert i.n_layers == 6                                  # layer runs: the looped ones count each time


def test_prompt_portions_and_single_tokens(model, made):
    t = toks(150)
    want = O.forward(CFG, made[1], t, np.float64)
    for cuts in ([150], [1], [2, 63, 1, 64, 17, 3]):
        s, at, i = model.session(), 0, 0
        while at < len(t):
            n = min(cuts[i % len(cuts)], len(t) - at)
            rc, lg = E.mixed_step([(s, t[at:at + n], range(n))])
            assert rc == n
            near(lg[0], want[at:at + n])
            at, i = at + n, i + 1
        assert s.pos == 150
        s.close()


def test_want_order_and_repeats(model, made):
    t = toks(20)
    want = O.forward(CFG, made[1], t, np.float64)
    a, b = model.session(), model.session()
    rc, lg = E.mixed_step([(a, t, [19, 0, 7, 7]), (b, t[:5], [])])
    assert rc == 4 and lg[1].shape == (0, 61)
    near(lg[0], want[[19, 0, 7, 7]])
    a.close()
    b.close()


def test_batch_equals_alone_and_pages_come_back(eng, made):
    m = eng.load(made[0], max_context=256, quant=E.WR_QUANT_F32)
    m.set_cache_pool(320, 2)                                # five pages, two slots
    want = {n: O.forward(CFG, made[1], toks(n, n), np.float64) for n in (130, 70, 200, 3)}
    for pair in ((130, 70), (200, 3), (70, 130), (3, 200)):
        ss = [m.session() for _ in pair]
        with pytest.raises(E.EngineError) as e:
            m.session()                                     # no third state slot
        assert e.value.rc == E.WR_ERR_BUSY
        half = [n // 2 + 1 for n in pair]
        rc, _ = E.mixed_step([(s, toks(n, n)[:h], []) for s, n, h in zip(ss, pair, half)])
        assert rc == 0
        rc, lg = E.mixed_step([(s, toks(n, n)[h:], range(n - h)) for s, n, h in zip(ss, pair, half)])
        for n, h, x in zip(pair, half, lg):
            near(x, want[n][h:])
        for s in ss:
            s.close()
    m.close()


def test_pool_exhaustion_changes_nothing(eng, made):
    m = eng.load(made[0], max_context=256, quant=E.WR_QUANT_F32)
    m.set_cache_pool(128, 2)
    a, b = m.session(), m.session()
    assert a.prefill(toks(64)) == 64
    rc, _ = E.mixed_step([(b, toks(64, 1), []), (a, [1], [0])])      # three pages wanted, two there
    assert rc == E.WR_ERR_BUSY and (a.pos, b.pos) == (64, 0) and a.status == E.WR_ERR_BUSY
    assert b.prefill(toks(64, 1)) == 64                     # b alone fits
    assert a.step(1) is None and a.status == E.WR_ERR_BUSY
    b.close()
    t = list(toks(64)) + [1]
    near(a.step(1)[None], O.forward(CFG, made[1], t, np.float64)[-1:])
    a.close()
    with pytest.raises(E.EngineError) as e:
        m.set_cache_pool(64, 1)                             # fixed by the first session
    assert e.value.rc == E.WR_ERR_STATE
    m.close()


def test_failure_anywhere_changes_nothing(model, made):
    t = toks(90)
    want = O.forward(CFG, made[1], t, np.float64)
    s, other = model.session(), model.session()
    assert s.prefill(t[:33]) == 33 and other.prefill(t[:3]) == 3
    for k in (1, 2, 9, 30):
        s.lib.wr_hip_mix_debug_fail_product_in(k)
        rc, _ = E.mixed_step([(s, t[33:70], [0]), (other, t[3:5], [])])
        assert rc == E.WR_ERR_INTERNAL and (s.pos, other.pos) == (33, 3)
    s.lib.wr_hip_mix_debug_fail_product_in(0)
    for run in range(6):
        s.lib.wrh_debug_fail_attention_at(run)
        assert s.step(int(t[33])) is None and s.status == E.WR_ERR_INTERNAL and s.pos == 33
    rc, lg = E.mixed_step([(s, t[33:], range(57)), (other, t[3:5], [0, 1])])
    near(lg[0], want[33:])
    near(lg[1], want[3:5])
    s.close()
    other.close()


def test_wait_that_fails_leaves_positions_and_logits(model, made):
    # the wait behind a step's logits reports an error: sessions keep the logits of the step before, whose rows the
    # caller still holds, and their positions
    t = toks(12)
    ss, fn = [model.session() for _ in range(3)], model.eng.lib.wr_hip_attn_debug_fail_wait_in
    assert all(s.prefill(t[:5]) == 5 for s in ss)
    hs, at = (C.c_void_p * 3)(*[s.h for s in ss]), (C.c_uint32 * 3)(1, 2, 3)
    rows = (C.POINTER(C.c_float) * 3)()
    assert model.lib.wr_batch_step(hs, at, 3, rows) == 3
    kept = [np.ctypeslib.as_array(r, shape=(model.vocab,)) for r in rows]
    before = [k.copy() for k in kept]
    for single in (False, True):
        fn(1)
        if single:
            assert ss[0].step(9) is None
        else:
            assert model.lib.wr_batch_step(hs, (C.c_uint32 * 3)(7, 8, 9), 3, None) == E.WR_ERR_INTERNAL
        fn(0)
        assert [s.pos for s in ss] == [6, 6, 6] and ss[0].status == E.WR_ERR_INTERNAL
        assert all(np.array_equal(a, b) for a, b in zip(kept, before))
    near(ss[1].step(9)[None], O.forward(CFG, made[1], list(t[:5]) + [2, 9], np.float64)[-1:])
    for s in ss:
        s.close()


def test_refusals(model):
    s = model.session(40)
    assert s.prefill(toks(30)) == 30
    for entries, rc in (([(s, [61], [0])], E.WR_ERR_INVAL),               # outside the vocabulary
                        ([(s, [1, 2], [2])], E.WR_ERR_INVAL),             # a place that is not there
                        ([(s, toks(11), [])], E.WR_ERR_CTX_FULL),
                        ([(s, [1], []), (s, [2], [])], E.WR_ERR_INVAL),   # the same session twice
                        ([(s, [], [])], E.WR_ERR_INVAL)):
        assert E.mixed_step(entries)[0] == rc
        assert s.pos == 30
    assert s.prefill(toks(11)) == E.WR_ERR_CTX_FULL and s.prefill(toks(10)) == 10
    assert s.step(0) is None and s.status == E.WR_ERR_CTX_FULL
    s.close()


def test_long_prompt_takes_several_passes(eng, tmp_path):
    cfg = mw.config(16, 20, [(mw.lightning(1, 4, 4, decay=[0.999]), None), (mw.latent_attention(1, 4, 4, 8, 8, 4, window=30), None)])
    bits = dict(mw.random_tensors(cfg, 2))
    m = eng.load(mw.write_model(str(tmp_path / "m"), cfg, bits), max_context=8192, quant=E.WR_QUANT_F32)
    t = np.random.default_rng(1).integers(0, 20, 4200)
    want = O.forward(cfg, {k: O.bf16_to_f32(v) for k, v in bits.items()}, t, np.float64)
    a, b = m.session(), m.session()
    rc, lg = E.mixed_step([(b, t[:9], [8]), (a, t, [0, 4085, 4086, 4087, 4095, 4096, 4199])])
    near(lg[0], want[[8]])
    near(lg[1], want[[0, 4085, 4086, 4087, 4095, 4096, 4199]])
    s = a
    s.lib.wr_hip_mix_debug_fail_product_in(10)              # in the second pass of a second call
    rc, _ = E.mixed_step([(b, np.resize(t, 4150), [])])
    s.lib.wr_hip_mix_debug_fail_product_in(0)
    assert rc == E.WR_ERR_INTERNAL and b.pos == 9
    near(E.mixed_step([(b, t[9:40], [30])])[1][0], want[[39]])
    a.close()
    b.close()
    m.close()


def test_greedy_through_step_and_batch(model, made):
    p = toks(9)
    t = list(p)
    for _ in range(6):
        t.append(int(O.forward(CFG, made[1], t, np.float64)[-1].argmax()))
    s, u = model.session(), model.session()
    s.prefill(p[:-1])
    u.prefill(p[:-1])
    tok, got = int(p[-1]), []
    for _ in range(3):
        tok = int(s.step(tok).argmax())
        got.append(tok)
    u.prefill([int(p[-1])] + got[:-1])
    for _ in range(3):
        rc, lg = E.batch_step([s, u], [tok, tok])
        assert rc == 2 and np.allclose(lg[0], lg[1], atol=1e-5)
        tok = int(lg[0].argmax())
        got.append(tok)
    assert got == t[9:]
    s.close()
    u.close()


def test_mixed_step_of_a_model_that_owns_its_caches(eng, tmp_path):
    p = str(tmp_path / "tiny.gguf")
    gw.write_model(p, TINY)
    m = eng.load(p)
    t = np.random.default_rng(2).integers(0, TINY.vocab, 30)
    ref, want = m.session(), []
    for x in t:
        want.append(ref.step(int(x)))
    want = np.stack(want)
    a, b, c = m.session(), m.session(), m.session()
    a.prefill(t[:5])
    rc, lg = E.mixed_step([(a, t[5:6], [0]), (b, t[:20], [3, 19, 3]), (c, t[:4], [])])
    assert rc == 4 and (a.pos, b.pos, c.pos) == (6, 20, 4)
    assert np.allclose(lg[0], want[[5]], atol=1e-5) and np.allclose(lg[1], want[[3, 19, 3]], atol=1e-5)
    rc, _ = E.mixed_step([(a, t[6:7], [0]), (b, [TINY.vocab], [0])])
    assert rc == E.WR_ERR_INVAL and (a.pos, b.pos) == (6, 20)
    assert np.allclose(a.step(int(t[6])), want[6], atol=1e-5)
    with pytest.raises(E.EngineError) as e:
        m.set_cache_pool(64, 1)
    assert e.value.rc == E.WR_ERR_UNSUPPORTED
    for s in (ref, a, b, c):
        s.close()
    m.close()


# ---- reading ---------------------------------------------------------------

def _load_rc(eng, folder):
    try:
        eng.load(str(folder), max_context=64, quant=E.WR_QUANT_F32).close()
    except E.EngineError as e:
        return e.rc
    return E.WR_OK


def _broken(tmp_path, change=None, tensors=None, text=None):
    cfg = json.loads(json.dumps(CFG))
    d = mw.write_model(str(tmp_path / "b"), cfg, tensors)
    if change:
        change(cfg)
        text = json.dumps(cfg)
    if text is not None:
        with open(os.path.join(d, "config.json"), "w") as f:
            f.write(text)
    return d


def _set(path, value):
    def change(cfg):
        for k in path[:-1]:
            cfg = cfg[k]
        if value is None:
            del cfg[path[-1]]
        else:
            cfg[path[-1]] = value
    return change


@pytest.mark.parametrize("path,value,rc", [
    (("architecture",), "Another", E.WR_ERR_UNSUPPORTED),
    (("architecture",), None, E.WR_ERR_FORMAT),
    (("layers", 0, "type"), "other", E.WR_ERR_UNSUPPORTED),
    (("layers", 1, "mlp", "kind"), "other", E.WR_ERR_UNSUPPORTED),
    (("width",), 41, E.WR_ERR_FORMAT),                      # no tensor has that shape
    (("width",), 40.5, E.WR_ERR_FORMAT),
    (("vocab",), None, E.WR_ERR_FORMAT),
    (("norm", "eps"), None, E.WR_ERR_FORMAT),
    (("layers", 0, "mixer", "decay"), [0.5], E.WR_ERR_FORMAT),
    (("layers", 1, "mixer", "mask"), None, E.WR_ERR_FORMAT),
    (("layers", 1, "mixer", "rot", "dims"), 5, E.WR_ERR_FORMAT),
    (("layers", 1, "mlp", "router", "top"), 6, E.WR_ERR_FORMAT),
    (("loop", "stop"), 9, E.WR_ERR_LIMIT),
    (("layers",), [], E.WR_ERR_FORMAT),
])
def test_bad_configurations_are_refused(eng, tmp_path, path, value, rc):
    assert _load_rc(eng, _broken(tmp_path, _set(path, value))) == rc


@pytest.mark.parametrize("text", ["", "{", "[1, 2", '{"architecture": "Bipotar",}', '{"a": 1} x', '{"a": tru}', '{"a": "\\q"}',
                                  "[" * 100 + "]" * 100])
def test_malformed_text_is_refused(eng, tmp_path, text):
    assert _load_rc(eng, _broken(tmp_path, text=text)) == E.WR_ERR_FORMAT


def test_optional_parts(eng, tmp_path):
    for change in (_set(("loop",), None), _set(("logit_scale",), None)):
        assert _load_rc(eng, _broken(tmp_path, change)) == E.WR_OK


def test_bad_files_are_refused(eng, tmp_path):
    d = _broken(tmp_path)
    st = os.path.join(d, "model.safetensors")
    whole = open(st, "rb").read()
    for cut in (0, 4, 8, 100, len(whole) - 10):
        with open(st, "wb") as f:
            f.write(whole[:cut])
        assert _load_rc(eng, d) == E.WR_ERR_FORMAT
    with open(st, "wb") as f:
        f.write(whole.replace(b'"l1.mix.uk"', b'"l1.mix.kk"'))
    assert _load_rc(eng, d) == E.WR_ERR_FORMAT              # a required tensor is missing
    with open(st, "wb") as f:
        f.write(whole.replace(b'"dtype": "BF16", "shape": [61, 40]', b'"dtype": "F16", "shape": [61, 40] '))
    assert _load_rc(eng, d) == E.WR_ERR_UNSUPPORTED
    os.remove(st)
    assert _load_rc(eng, d) == E.WR_ERR_IO
    os.remove(os.path.join(d, "config.json"))
    assert _load_rc(eng, d) == E.WR_ERR_IO
