"""The norm in front of a prompt pass's projections at the widths where its workgroups change (2048, 4096 and 8192 columns) and with token counts around
its runs of eight tokens a die (64 to a round): against the kernels for up to 32 tokens."""
import numpy as np
import pytest

from gpu_common import backend, rel_err  # noqa: F401
from slai_amd import _ffi
from slai_amd import gguf_writer as gw
from test_gpu_prefill import SELF_TOL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,tokens", [(2048, 63), (2048, 65), (2304, 9), (4096, 57), (4352, 71), (8192, 12), (8448, 129)])
def test_norm_widths(backend, dim, tokens):
    from slai_amd.runtime import Gguf, Llama2
    print("case", dim, tokens, flush=True)
    t = 12
    g = Gguf(gw.llama_gguf(dim, 512, 2, dim // 128, 1, 512, 256, t, v_type=t, out_type=t, embd_type=t, std=0.02, norm_random=True, distinct_layers=1))
    prompt = np.random.Generator(np.random.PCG64(dim)).integers(0, 512, tokens + 1).astype(np.int32)
    out = []
    for chunk in (0, 32):
        m = Llama2(backend, g, _ffi.MODEL_LLAMA, _ffi.KV_F32)
        m.prefill(prompt[:-1], 0, chunk)
        assert m.prefill_fp32_repeats() == 0
        out.append(m.forward_logits(tokens, int(prompt[-1])))
        m.destroy()
    assert rel_err(out[0], out[1]) < SELF_TOL
    g.close()
