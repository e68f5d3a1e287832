"""Wide prompt passes whose tiles are no multiple of the compute units (wide_share_kernel): against the kernels for up to 32 tokens."""
import numpy as np
import pytest

from gpu_common import backend, rel_err  # noqa: F401
from slai_amd import _ffi
from slai_amd import gguf_writer as gw
from test_gpu_prefill import SELF_TOL

pytestmark = pytest.mark.gpu
NAMES = {2: "q4_0", 8: "q8_0", 12: "q4_k", 13: "q5_k", 14: "q6_k"}


QKV, OUTPUT, FFN, DOWN = range(4)                              # prompt_form's steps
PLAIN, SHARED = 0, 3                                           # its forms: large workgroups alone, with shared tiles
# format, hidden columns of a model 2048 wide, tokens (one fewer is read); how gate + up are dealt out: whole rounds, most rests a workgroup has to finish (None: in plain
# rounds, q/k/v share).  Row units of 256 rows of both matrices, token blocks of 64: a last unit with 32 rows (5664), last blocks with 1, 32, 33 and 64 tokens, one to
# four rests, workgroups with fewer than the others (22, 23 and 25 tiles), a whole round in front, two and then a single tile.
DEALS = [(12, 5632, 450, 0, 3), (12, 5888, 482, 0, 3), (8, 5632, 513, 0, 3), (13, 5632, 513, 0, 3), (2, 5632, 450, 0, 3), (14, 5632, 513, 0, 3), (8, 5664, 481, 0, 3), (12, 8192, 257, 0, 1),
         (12, 4608, 642, 0, 4), (8, 11008, 641, 1, 3), (12, 9216, 705, 1, 2), (8, 11008, 706, 2, 1), (8, 11008, 898, None, None)]


def logits_of(m, prompt, chunk):
    m.prefill(prompt[:-1], 0, chunk)
    out = m.forward_logits(prompt.size - 1, int(prompt[-1]))
    m.destroy()
    return out


@pytest.mark.parametrize("t,hidden,n,rounds,rests", DEALS, ids=["%s-%d-%d" % (NAMES[d[0]], d[1], d[2]) for d in DEALS])
def test_shared_tiles_llama(backend, t, hidden, n, rounds, rests):
    from slai_amd.runtime import Gguf, Llama2
    print("case", NAMES[t], hidden, n, flush=True)
    g = Gguf(gw.llama_gguf(2048, hidden, 2, 16, 16, 512, 1024, t, v_type=t, out_type=t, embd_type=t, std=0.03, norm_random=True))
    prompt = np.random.Generator(np.random.PCG64(n)).integers(0, 512, n).astype(np.int32)
    m = Llama2(backend, g, _ffi.MODEL_LLAMA, _ffi.KV_F32)
    assert m.prompt_form(n - 1, FFN) == (PLAIN if rounds is None else SHARED) and SHARED in [m.prompt_form(n - 1, step) for step in range(4)]
    m.destroy()
    got, again, ref = (logits_of(Llama2(backend, g, _ffi.MODEL_LLAMA, _ffi.KV_F32), prompt, chunk) for chunk in (0, 0, 32))
    assert np.array_equal(got, again)                          # whoever of a tile's two workgroups comes last
    assert rel_err(got, ref) < SELF_TOL
    g.close()


# 24 row units at 7 token blocks are 21 tiles a die, whose rests are dealt out to eleven workgroups, the last of them with fewer; 43 at 5 are 27, which would leave six rests to
# each of five workgroups: gate + up in plain rounds, q/k/v (24 units, 15 tiles a die) in two ranges of columns
@pytest.mark.parametrize("hidden,n,forms", [(11008, 301, (PLAIN, PLAIN)), (6144, 449, (SHARED, SHARED))])
def test_last_rests(backend, hidden, n, forms):
    from slai_amd.runtime import Gguf, Llama2
    t = 12
    print("case", hidden, n, flush=True)
    g = Gguf(gw.llama_gguf(4096, hidden, 2, 32, 32, 512, 512, t, v_type=t, out_type=t, embd_type=t, std=0.02, norm_random=True, distinct_layers=1))
    prompt = np.random.Generator(np.random.PCG64(n)).integers(0, 512, n).astype(np.int32)
    m = Llama2(backend, g, _ffi.MODEL_LLAMA, _ffi.KV_F32)
    assert (m.prompt_form(n - 1, QKV), m.prompt_form(n - 1, FFN)) == forms
    m.destroy()
    got, again, ref = (logits_of(Llama2(backend, g, _ffi.MODEL_LLAMA, _ffi.KV_F32), prompt, chunk) for chunk in (0, 0, 32))
    assert np.array_equal(got, again)
    assert rel_err(got, ref) < SELF_TOL
    g.close()


# the MLP's first matrix (its GELU as pairs); that and q/k/v with their bias
@pytest.mark.parametrize("n,steps", [(490, [FFN]), (706, [QKV, FFN])])
def test_shared_tiles_gpt2(n, steps):
    from slai_amd.runtime import Backend, Gguf, Gpt2
    b = Backend(0)                                             # (a context that has held no other model)
    g = Gguf(gw.gpt2_gguf(2048, 2, 32, 8192, 512, 1024, 8, std=0.02))
    prompt = np.random.Generator(np.random.PCG64(3)).integers(0, 512, n).astype(np.int32)
    m = Gpt2(b, g, _ffi.KV_F32)
    assert [step for step in range(4) if m.prompt_form(n - 1, step) == SHARED] == steps
    m.destroy()
    got, ref = (logits_of(Gpt2(b, g, _ffi.KV_F32), prompt, chunk) for chunk in (0, 32))
    assert rel_err(got, ref) < SELF_TOL
    g.close(); b.close()


def test_without_memory_for_shared_tiles(monkeypatch):
    """A prompt whose launches would share tiles is read all the same, in the plain forms, where the sums of shared tiles are not allowed their 64 MB."""
    from slai_amd.runtime import Backend, Gguf, Llama2
    t, n = 8, 513
    g = Gguf(gw.llama_gguf(2048, 5632, 2, 16, 16, 512, 1024, t, v_type=t, out_type=t, embd_type=t, std=0.03, norm_random=True))
    prompt = np.random.Generator(np.random.PCG64(n)).integers(0, 512, n).astype(np.int32)
    logits = []
    for mb, form in ((64, SHARED), (63, PLAIN)):
        monkeypatch.setenv("SLAI_PROMPT_SHARE_MB", str(mb))
        b = Backend(0)
        m = Llama2(b, g, _ffi.MODEL_LLAMA, _ffi.KV_F32)
        assert m.prompt_form(n - 1, FFN) == form
        logits.append(logits_of(m, prompt, 0))
        b.close()
    assert rel_err(logits[1], logits[0]) < SELF_TOL
    g.close()
