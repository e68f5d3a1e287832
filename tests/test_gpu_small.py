"""The layers of a small model's token as one launch, on one die (kernels_decode_small.hip) or over the device (kernels_decode_mid.hip): shapes at the edges of what it covers (two
rows per wave, heads of 8 to 64, grouped queries, biases and NeoX pairs), both formats and cache types, positions past one and two passes of
its attention (120 positions each), against the oracle; a launch that gives up; several models taking turns on one context."""
import threading
import time

import numpy as np
import pytest

from gpu_common import backend, rel_err  # noqa: F401
from slai_amd import _ffi
from slai_amd import gguf_writer as gw
from helpers import OracleGguf
from slai_amd.runtime import Backend, Gguf, Gpt2, Llama2
from test_gpu_models import check_llama

pytestmark = pytest.mark.gpu
LAUNCHES, ONE_LAUNCH = 0, 2                # decode_form_at

SHAPES = {                                 # dim, hidden, heads, kv heads
    "15 M parameters": (288, 768, 6, 6),
    "widest": (480, 960, 15, 3),           # 15 rows a workgroup, 30 gated pairs
    "heads of 64": (256, 1024 - 64, 4, 4),
    "heads of 8, fewer rows than waves": (64, 96, 8, 2),
    "one head": (32, 32, 1, 1),
}


def model(shape, wtype, seq, seed=31, **kw):
    dim, hidden, heads, kv = SHAPES[shape]
    return gw.llama_gguf(dim=dim, hidden_dim=hidden, n_layers=3, n_heads=heads, n_kv_heads=kv, vocab=500, seq_len=seq, wtype=wtype, seed=seed, std=0.08,
                         norm_random=True, **kw)


def llama_form(backend, data, pos=0, model_type=_ffi.MODEL_LLAMA):
    g = Gguf(data)
    m = Llama2(backend, g, model_type, _ffi.KV_F16)
    form = m.decode_form_at(pos)
    m.destroy(); g.close()
    return form


@pytest.mark.parametrize("kv_f16", [False, True])
@pytest.mark.parametrize("wtype", [8, 2], ids=["q8_0", "q4_0"])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_small_shapes(backend, shape, wtype, kv_f16):
    prompt = np.random.Generator(np.random.PCG64(3)).integers(0, 500, 9)
    data = model(shape, wtype, 64)
    assert llama_form(backend, data, 63) == ONE_LAUNCH
    check_llama(backend, data, prompt, 40, kv_f16=kv_f16)


@pytest.mark.parametrize("wtype", [8, 2], ids=["q8_0", "q4_0"])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_small_shapes_in_launches(monkeypatch, shape, wtype):
    """The form that a launch which gives up falls back to."""
    monkeypatch.setenv("SLAI_PERSISTENT", "0")
    b = Backend(0)
    data = model(shape, wtype, 64)
    assert llama_form(b, data) == LAUNCHES
    check_llama(b, data, np.random.Generator(np.random.PCG64(3)).integers(0, 500, 9), 40, kv_f16=wtype == 2)
    b.close()


def test_small_bias_neox(backend):
    data = model("widest", 8, 64, arch="qwen2", bias=True, rope_base=1000000.0, rms_eps=1e-6)
    assert llama_form(backend, data, model_type=_ffi.MODEL_QWEN2) == ONE_LAUNCH
    check_llama(backend, data, [5, 400, 17], 30, model_type=_ffi.MODEL_QWEN2, neox=1, name=b"qwen2")


@pytest.mark.parametrize("kv_f16", [False, True])
def test_small_positions_beyond_one_pass(backend, kv_f16):
    prompt = np.random.Generator(np.random.PCG64(4)).integers(0, 500, 230)
    data = model("15 M parameters", 8, 256)
    assert llama_form(backend, data, 255) == ONE_LAUNCH
    check_llama(backend, data, prompt, 252, kv_f16=kv_f16, check_logit_steps=125)


def test_small_gives_up_and_the_call_is_repeated(monkeypatch):
    """One look at a counter is never enough: every wait gives up at once, and the calls come back from launches per step."""
    data = model("15 M parameters", 8, 64)
    prompt = np.array([3, 77, 410, 8], np.int32)
    results = []
    for spins in ("4096", "1"):
        monkeypatch.setenv("SLAI_SMALL_SPINS", spins)
        b = Backend(0)
        g = Gguf(data)
        m = Llama2(b, g, _ffi.MODEL_LLAMA, _ffi.KV_F32)
        assert m.decode_form_at(0) == ONE_LAUNCH
        ids, _ = m.generate(prompt, 20)
        assert m.decode_form_at(0) == (LAUNCHES if spins == "1" else ONE_LAUNCH)
        first = Llama2(b, g, _ffi.MODEL_LLAMA, _ffi.KV_F32)
        results.append((ids, m.forward_logits(20, int(ids[-1])), first.forward_logits(0, 3)))
        first.destroy(); m.destroy(); g.close(); b.close()
    assert np.array_equal(results[0][0], results[1][0])
    assert rel_err(results[1][1], results[0][1]) < 1e-5 and rel_err(results[1][2], results[0][2]) < 1e-5


def test_small_models_in_turn(backend):
    data = [model(s, 8, 64, seed=40 + i) for i, s in enumerate(("15 M parameters", "heads of 64"))]
    gs = [Gguf(d) for d in data]
    ms = [Llama2(backend, g, _ffi.MODEL_LLAMA, _ffi.KV_F16) for g in gs]
    assert [m.decode_form_at(0) for m in ms] == [ONE_LAUNCH] * 2
    alone = [m.generate(np.array([9, 2], np.int32), 24)[0] for m in ms]
    mixed = [[], []]
    for i in range(24):
        for k, m in enumerate(ms):
            seq = np.concatenate([[9, 2], alone[k][1:i + 1]]).astype(np.int32)[:max(i + 1, 2)]
            mixed[k].append(int(m.generate(seq, 1, start_pos=i)[0][0]))
    for k in range(2):
        assert mixed[k] == alone[k].tolist()
    for m in ms:
        m.destroy()
    for g in gs:
        g.close()


# GPT-2 shapes: embedding, FFN, heads, context
GPT2 = {
    "small": (768, 3072, 12, 256),         # nine rows a workgroup, three waves a row of the FFN's width
    "widest": (1024, 2560, 16, 64),        # twelve rows a workgroup
    "heads of 8, most workgroups without a row": (96, 160, 12, 64),
    "heads of 40": (320, 1056, 8, 64),     # rows end inside a chunk of 64
}


def check_gpt2(backend, data, kv_f16, n_prompt, steps, vocab, form=ONE_LAUNCH):
    g = OracleGguf(data); L = g.L
    om = L.slo_gpt2_from_gguf(g.h, int(kv_f16))
    prompt = np.random.Generator(np.random.PCG64(8)).integers(0, vocab, n_prompt).astype(np.int32)
    ref, ref_logits = np.zeros(steps, np.int32), np.zeros((steps, vocab), np.float32)
    assert L.slo_gpt2_generate(om, prompt.ctypes.data, n_prompt, 0, steps, -1, ref.ctypes.data, ref_logits.ctypes.data) == steps
    gg = Gguf(data)
    m = Gpt2(backend, gg, _ffi.KV_F16 if kv_f16 else _ffi.KV_F32)
    if form is not None:
        assert m.decode_form_at(0) == m.decode_form_at(steps - 1) == form
    tok = int(prompt[0])
    for pos in range(steps):
        assert rel_err(m.forward_logits(pos, tok), ref_logits[pos]) < 1e-2
        tok = int(ref[pos])
    m.destroy()
    m = Gpt2(backend, gg, _ffi.KV_F16 if kv_f16 else _ffi.KV_F32)
    got, _ = m.generate(prompt, steps)
    assert np.array_equal(got, ref)
    m.destroy(); gg.close(); L.slo_gpt2_free(om); g.close()


@pytest.mark.parametrize("kv_f16", [False, True])
@pytest.mark.parametrize("wtype", [8, 2], ids=["q8_0", "q4_0"])
@pytest.mark.parametrize("shape", sorted(GPT2))
def test_gpt2_in_one_launch(monkeypatch, shape, wtype, kv_f16):
    monkeypatch.setenv("SLAI_SMALL_MAX_POS", "1024")           # (also where launches are the faster form)
    b = Backend(0)
    dim, hidden, heads, seq = GPT2[shape]
    data = gw.gpt2_gguf(n_embd=dim, n_layer=2, n_head=heads, ff_len=hidden, vocab=700, n_seq=seq, wtype=wtype, seed=61, std=0.05)
    # ("small": positions past two passes of the attention)
    check_gpt2(b, data, kv_f16, seq - 30 if shape == "small" else 7, seq - 4 if shape == "small" else 30, 700)
    b.close()


@pytest.mark.parametrize("wtype", [8, 2], ids=["q8_0", "q4_0"])
def test_gpt2_in_launches(monkeypatch, wtype):
    monkeypatch.setenv("SLAI_PERSISTENT", "0")
    b = Backend(0)
    check_gpt2(b, gw.gpt2_gguf(n_embd=768, n_layer=2, n_head=12, ff_len=3072, vocab=700, n_seq=64, wtype=wtype, seed=61, std=0.05), wtype == 2, 7, 30, 700, LAUNCHES)
    b.close()


def test_gpt2_in_one_launch_single_layer(monkeypatch):
    monkeypatch.setenv("SLAI_SMALL_MAX_POS", "1024")
    b = Backend(0)
    data = gw.gpt2_gguf(n_embd=64, n_layer=1, n_head=2, ff_len=128, vocab=700, n_seq=32, wtype=8, seed=62, std=0.08)
    check_gpt2(b, data, False, 4, 20, 700)
    b.close()


def test_gpt2_gives_up_and_the_call_is_repeated(monkeypatch):
    data = gw.gpt2_gguf(n_embd=768, n_layer=2, n_head=12, ff_len=3072, vocab=700, n_seq=64, wtype=8, seed=63, std=0.05)
    results = []
    for spins in ("4096", "1"):
        monkeypatch.setenv("SLAI_SMALL_SPINS", spins)
        b = Backend(0)
        g = Gguf(data)
        m = Gpt2(b, g, _ffi.KV_F32)
        assert m.decode_form_at(0) == ONE_LAUNCH
        ids, _ = m.generate(np.array([3, 77], np.int32), 20)
        assert m.decode_form_at(0) == (LAUNCHES if spins == "1" else ONE_LAUNCH)
        first = Gpt2(b, g, _ffi.KV_F32)
        results.append((ids, m.forward_logits(20, int(ids[-1])), first.forward_logits(0, 3)))
        first.destroy(); m.destroy(); g.close(); b.close()
    assert np.array_equal(results[0][0], results[1][0])
    assert rel_err(results[1][1], results[0][1]) < 1e-5 and rel_err(results[1][2], results[0][2]) < 1e-5


def small_and_gpt2():
    return [(lambda b, g: Llama2(b, g, _ffi.MODEL_LLAMA, _ffi.KV_F32), model("15 M parameters", 8, 256)),
            (lambda b, g: Gpt2(b, g, _ffi.KV_F32), gw.gpt2_gguf(n_embd=768, n_layer=2, n_head=12, ff_len=3072, vocab=700, n_seq=256, wtype=8, seed=63, std=0.05))]


@pytest.mark.parametrize("which", [0, 1], ids=["llama", "gpt2"])
def test_one_time_limit_for_all_queued_tokens(monkeypatch, which):
    """A launch without one of its workgroups waits out its limit (32768 looks, at least 10 ms); the tokens queued behind it do not."""
    monkeypatch.setenv("SLAI_SMALL_ABSENT", "1")
    monkeypatch.setenv("SLAI_SMALL_SPINS", "32768")
    make, data = small_and_gpt2()[which]
    b = Backend(0)
    g = Gguf(data)
    m = make(b, g)
    assert m.decode_form_at(0) == ONE_LAUNCH
    t0 = time.perf_counter()
    ids, _ = m.generate(np.array([3, 77], np.int32), 1)
    one = time.perf_counter() - t0                             # a time limit, twice a capture and a token in launches
    m.destroy()
    m = make(b, g)
    t0 = time.perf_counter()
    m.generate(np.array([3, 77], np.int32), 200)
    many = time.perf_counter() - t0
    assert many < 5 * one + 0.2, (one, many)
    m.destroy(); g.close(); b.close()


def test_form_by_position(backend):
    """Small models take one launch a token only as far as that is the faster one, and launches beyond."""
    for dim, hidden, heads, kv, line in ((64, 96, 8, 2, 448), (288, 768, 6, 6, 672)):
        g = Gguf(gw.llama_gguf(dim=dim, hidden_dim=hidden, n_layers=2, n_heads=heads, n_kv_heads=kv, vocab=500, seq_len=4096, wtype=8, seed=64, std=0.08))
        m = Llama2(backend, g, _ffi.MODEL_LLAMA, _ffi.KV_F16)
        assert [m.decode_form_at(p) for p in (0, line - 1, line, 4095)] == [ONE_LAUNCH, ONE_LAUNCH, LAUNCHES, LAUNCHES]
        m.destroy(); g.close()
    for dim, line in ((96, 153), (768, 1024)):
        g = Gguf(gw.gpt2_gguf(n_embd=dim, n_layer=2, n_head=12, ff_len=4 * dim, vocab=700, n_seq=2048, wtype=8, seed=65, std=0.05))
        m = Gpt2(backend, g, _ffi.KV_F32)
        assert [m.decode_form_at(p) for p in (0, line - 1, line, 2047)] == [ONE_LAUNCH, ONE_LAUNCH, LAUNCHES, LAUNCHES]
        m.destroy(); g.close()


# columns, layers, context, line (0: launches at every position)
@pytest.mark.parametrize("dim,layers,seq,line", [(96, 2, 1024, 0), (96, 6, 64, 0), (64, 1, 512, 0), (64, 2, 1024, 102), (128, 1, 1024, 204), (96, 1, 2048, 153)])
def test_form_of_narrow_gpt2(backend, dim, layers, seq, line):
    g = Gguf(gw.gpt2_gguf(n_embd=dim, n_layer=layers, n_head=4, ff_len=2 * dim, vocab=700, n_seq=seq, wtype=8, seed=65, std=0.05))
    m = Gpt2(backend, g, _ffi.KV_F32)
    assert [m.decode_form_at(p) for p in (0, max(line, 1) - 1, line)] == [ONE_LAUNCH if line else LAUNCHES] * 2 + [LAUNCHES]
    m.destroy(); g.close()


@pytest.mark.parametrize("dim,layers,seq,line", [(64, 1, 1024, 0), (128, 1, 512, 0), (192, 1, 512, 448), (64, 1, 2048, 256), (64, 2, 1024, 448), (256, 1, 1024, 672)])
def test_form_of_narrow_llama(backend, dim, layers, seq, line):
    g = Gguf(gw.llama_gguf(dim=dim, hidden_dim=2 * dim, n_layers=layers, n_heads=4, n_kv_heads=4, vocab=500, seq_len=seq, wtype=8, seed=64, std=0.08))
    m = Llama2(backend, g, _ffi.MODEL_LLAMA, _ffi.KV_F16)
    assert [m.decode_form_at(p) for p in (0, max(line, 1) - 1, line)] == [ONE_LAUNCH if line else LAUNCHES] * 2 + [LAUNCHES]
    m.destroy(); g.close()


def test_tokens_across_the_line(backend):
    """The caches are the same in both forms: a call that passes from one to the other, and one that begins beyond."""
    prompt = np.random.Generator(np.random.PCG64(5)).integers(0, 500, 440)
    check_llama(backend, gw.llama_gguf(dim=64, hidden_dim=96, n_layers=2, n_heads=8, n_kv_heads=2, vocab=500, seq_len=512, wtype=8, seed=66, std=0.08, norm_random=True),
                prompt, 470, check_logit_steps=460)
    check_gpt2(backend, gw.gpt2_gguf(n_embd=64, n_layer=2, n_head=8, ff_len=160, vocab=700, n_seq=192, wtype=8, seed=67, std=0.05), True, 90, 130, 700, None)


@pytest.mark.parametrize("which", [0, 1], ids=["llama", "gpt2"])
def test_elapsed_time_of_a_repeated_call(monkeypatch, which):
    """The time that a call reports has the launch that gave up in it: at least 65536 looks of 0.3 us, where eight tokens in launches take 1.2 ms."""
    monkeypatch.setenv("SLAI_SMALL_ABSENT", "1")
    monkeypatch.setenv("SLAI_SMALL_SPINS", "65536")
    make, data = small_and_gpt2()[which]
    b = Backend(0)
    g = Gguf(data)
    m = make(b, g)
    assert m.decode_form_at(0) == ONE_LAUNCH
    t0 = time.perf_counter()
    ids, ms = m.generate(np.array([3, 77], np.int32), 8)
    host = (time.perf_counter() - t0) * 1e3
    again, ms_launches = m.generate(np.array([3, 77], np.int32), 8)
    assert m.decode_form_at(0) == LAUNCHES and np.array_equal(ids, again)
    assert ms_launches + 15.0 < ms < host, (ms, ms_launches, host)
    m.destroy(); g.close(); b.close()


@pytest.mark.parametrize("which", [0, 1], ids=["llama", "gpt2"])
def test_the_form_comes_back(monkeypatch, which):
    """A model whose launch gave up takes launches for 64 calls and then tries again; it rests twice as long after the second failure."""
    monkeypatch.setenv("SLAI_SMALL_SPINS", "1")
    make, data = small_and_gpt2()[which]
    b = Backend(0)
    g = Gguf(data)
    m = make(b, g)
    prompt = np.array([3, 77], np.int32)
    ref, _ = m.generate(prompt, 8)
    for rest in (64, 128):
        for i in range(rest):
            assert m.decode_form_at(0) == LAUNCHES
            if i % 2:
                m.forward_logits(0, 3)
            else:
                assert np.array_equal(m.generate(prompt, 8)[0], ref)
        assert m.decode_form_at(0) == ONE_LAUNCH
        assert np.array_equal(m.generate(prompt, 8)[0], ref)   # (gives up again)
    m.destroy(); g.close(); b.close()


def test_without_memory_for_row_copies(monkeypatch):
    """A GPT-2 model in tiles whose row copies are not allowed the memory loads all the same and takes launches."""
    monkeypatch.setenv("SLAI_PROMPT_COPY_MB", "0")
    b = Backend(0)
    check_gpt2(b, gw.gpt2_gguf(n_embd=768, n_layer=2, n_head=12, ff_len=3072, vocab=700, n_seq=64, wtype=8, seed=61, std=0.05), False, 7, 20, 700, LAUNCHES)
    b.close()


def test_time_steps_of_the_form_that_runs(monkeypatch):
    """slai_llama2_time_steps names the launches that generate makes at that position, and those of a model that rests after it gave up."""
    for env, names in ((None, ["embedding row", "llama2 layers", "llama2 output"]), ("SLAI_SMALL_SPINS", None)):
        if env:
            monkeypatch.setenv(env, "1")
        b = Backend(0)
        g = Gguf(model("15 M parameters", 8, 1024))
        m = Llama2(b, g, _ffi.MODEL_LLAMA, _ffi.KV_F32)
        steps = m.time_steps(8, 5, reps=3)
        if names:
            assert [s[0] for s in steps] == names and all(s[2] == 1 and s[1] > 0.0 and s[3] == s[1] for s in steps)
            steps = m.time_steps(900, 5, reps=3)
        assert {"llama2 qkv", "llama2 ffn_down"} <= {s[0] for s in steps}, steps
        m.destroy(); g.close(); b.close()


@pytest.mark.parametrize("which", [0, 1], ids=["llama", "gpt2"])
def test_gives_up_before_the_resident_launch(monkeypatch, which):
    """The time limit, with what two tokens take besides, is below the 20 ms after which the resident launch of the 7B shape reports an error."""
    monkeypatch.setenv("SLAI_SMALL_ABSENT", "1")
    make, data = small_and_gpt2()[which]
    b = Backend(0)
    g = Gguf(data)
    m = make(b, g)
    _, ms = m.generate(np.array([3, 77], np.int32), 2)
    assert m.decode_form_at(0) == LAUNCHES and ms < 15.0, ms
    m.destroy(); g.close(); b.close()


def test_beside_a_resident_launch():
    """A program that decodes with the resident launch, whose workgroups take every compute unit, beside one with a small model: neither sees an error."""
    g = [Gguf(gw.llama_gguf(dim=4096, hidden_dim=11008, n_layers=2, n_heads=32, n_kv_heads=32, vocab=1024, seq_len=128, wtype=12, v_type=14, out_type=14, embd_type=12, seed=71,
                            std=0.02, distinct_layers=1)), Gguf(model("15 M parameters", 8, 128))]
    prompt = np.array([3, 77, 5], np.int32)
    got = [[], []]

    def work(i):
        b = Backend(0)
        for _ in range(1 if i == 0 else 4):                    # (a new small model now and then: one that gave up rests)
            m = Llama2(b, g[i], _ffi.MODEL_LLAMA, _ffi.KV_F16)
            assert m.decode_form_at(0) == (1 if i == 0 else ONE_LAUNCH)
            for _ in range(30 if i == 0 else 12):
                got[i].append(m.generate(prompt, 48)[0].tolist())
            m.destroy()
        b.close()
    for i in (0, 1):
        work(i)
    alone = [x[0] for x in got]
    threads = [threading.Thread(target=work, args=(i,)) for i in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(got[0]) == 60 and len(got[1]) == 96
    assert all(x == alone[i] for i in (0, 1) for x in got[i])
    for x in g:
        x.close()
