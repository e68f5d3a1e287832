"""Wide prompt passes whose tiles are no multiple of the compute units (wide_share_kernel): against the kernels for up to 32 tokens."""
import numpy as np
import pytest

from gpu_common import backend, rel_err  # noqa: F401
from slai_amd import _ffi
from slai_amd import gguf_writer as gw
from test_gpu_prefill import SELF_TOL

pytestmark = pytest.mark.gpu
NAMES = {2: "q4_0", 8: "q8_0", 12: "q4_k", 13: "q5_k", 14: "q6_k"}


def logits_of(m, prompt, chunk):
    m.prefill(prompt[:-1], 0, chunk)
    out = m.forward_logits(prompt.size - 1, int(prompt[-1]))
    m.destroy()
    return out


# gate + up of 22 or 23 row units (the last a quarter full) at 7 and 8 token blocks (the last with 1, 33 and 64 tokens): one main per group and three; and an incomplete second round
@pytest.mark.parametrize("t,hidden,n", [(12, 5632, 450), (12, 5888, 482), (8, 5632, 513), (13, 5632, 513), (2, 5632, 450), (14, 5632, 513), (8, 11008, 705)],
                         ids=lambda v: NAMES.get(v, str(v)))
def test_shared_tiles_llama(backend, t, hidden, n):
    from slai_amd.runtime import Gguf, Llama2
    print("case", NAMES[t], hidden, n, flush=True)
    g = Gguf(gw.llama_gguf(2048, hidden, 2, 16, 16, 512, 1024, t, v_type=t, out_type=t, embd_type=t, std=0.03, norm_random=True))
    prompt = np.random.Generator(np.random.PCG64(n)).integers(0, 512, n).astype(np.int32)
    got, again, ref = (logits_of(Llama2(backend, g, _ffi.MODEL_LLAMA, _ffi.KV_F32), prompt, chunk) for chunk in (0, 0, 32))
    assert np.array_equal(got, again)                          # whoever of a tile's two workgroups comes last
    assert rel_err(got, ref) < SELF_TOL
    g.close()


# 43 row units at 5 token blocks are 27 tiles a die, whose rests are dealt out to five workgroups, the last of them with fewer; 24 units at 7: 21 and eleven
@pytest.mark.parametrize("hidden,n", [(11008, 301), (6144, 449)])
def test_last_rests(backend, hidden, n):
    from slai_amd.runtime import Gguf, Llama2
    t = 12
    print("case", hidden, n, flush=True)
    g = Gguf(gw.llama_gguf(4096, hidden, 2, 32, 32, 512, 512, t, v_type=t, out_type=t, embd_type=t, std=0.02, norm_random=True, distinct_layers=1))
    prompt = np.random.Generator(np.random.PCG64(n)).integers(0, 512, n).astype(np.int32)
    got, again, ref = (logits_of(Llama2(backend, g, _ffi.MODEL_LLAMA, _ffi.KV_F32), prompt, chunk) for chunk in (0, 0, 32))
    assert np.array_equal(got, again)
    assert rel_err(got, ref) < SELF_TOL
    g.close()


def test_shared_tiles_gpt2(backend):
    from slai_amd.runtime import Gguf, Gpt2
    g = Gguf(gw.gpt2_gguf(2048, 2, 32, 8192, 512, 1024, 8, std=0.02))
    prompt = np.random.Generator(np.random.PCG64(3)).integers(0, 512, 490).astype(np.int32)
    got, ref = (logits_of(Gpt2(backend, g, _ffi.KV_F32), prompt, chunk) for chunk in (0, 32))
    assert rel_err(got, ref) < SELF_TOL
    g.close()


def test_without_memory_for_shared_tiles(monkeypatch):
    """A prompt whose launches would share tiles is read all the same, in the plain forms, where the sums of shared tiles are not allowed their 64 MB."""
    from slai_amd.runtime import Backend, Gguf, Llama2
    t, n = 8, 513
    g = Gguf(gw.llama_gguf(2048, 5632, 2, 16, 16, 512, 1024, t, v_type=t, out_type=t, embd_type=t, std=0.03, norm_random=True))
    prompt = np.random.Generator(np.random.PCG64(n)).integers(0, 512, n).astype(np.int32)
    logits = []
    for mb, form in ((64, 3), (63, 0)):
        monkeypatch.setenv("SLAI_PROMPT_SHARE_MB", str(mb))
        b = Backend(0)
        m = Llama2(b, g, _ffi.MODEL_LLAMA, _ffi.KV_F32)
        assert m.prompt_form(n - 1, 2) == form
        logits.append(logits_of(m, prompt, 0))
        b.close()
    assert rel_err(logits[1], logits[0]) < SELF_TOL
    g.close()
