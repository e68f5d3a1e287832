"""Slim launches of a prompt pass that fill the device a little more than once: their columns in two and in four ranges, at the edges of the rule
(256 to 384 workgroups of 64 rows x 32 tokens, four ranges up to 320 of more than 32 super-blocks): against the kernels for up to 32 tokens."""
import numpy as np
import pytest

from gpu_common import backend, rel_err  # noqa: F401
from slai_amd import _ffi
from slai_amd import gguf_writer as gw
from test_gpu_prefill import SELF_TOL

pytestmark = pytest.mark.gpu


# 32 row blocks: 8 tiles of 32 tokens are 256 workgroups, 9: 288, 10: 320, 11: 352, 12: 384; hidden rows of 32 and 34 super-blocks (the last range the longest), output of 8
@pytest.mark.parametrize("tokens", [256, 257, 320, 321, 384, 385])
@pytest.mark.parametrize("t,hidden", [(12, 8704), (8, 8192), (14, 8704)], ids=["q4_k", "q8_0", "q6_k"])
def test_ranges(backend, t, hidden, tokens):
    from slai_amd.runtime import Gguf, Llama2
    print("case", t, hidden, tokens, flush=True)
    g = Gguf(gw.llama_gguf(2048, hidden, 2, 16, 16, 512, 512, t, v_type=t, out_type=t, embd_type=t, std=0.03, norm_random=True))
    prompt = np.random.Generator(np.random.PCG64(tokens)).integers(0, 512, tokens + 1).astype(np.int32)
    out = []
    for chunk in (0, 0, 32):
        m = Llama2(backend, g, _ffi.MODEL_LLAMA, _ffi.KV_F32)
        m.prefill(prompt[:-1], 0, chunk)
        out.append(m.forward_logits(tokens, int(prompt[-1])))
        m.destroy()
    assert np.array_equal(out[0], out[1])
    assert rel_err(out[0], out[2]) < SELF_TOL
    g.close()
