"""Attention of a prompt pass at the edges of its blocks of 32 queries and 32 positions, with four waves a workgroup and with eight
(from 513 positions on, where a launch has at most one workgroup per compute unit): against the kernels for up to 32 tokens."""
import numpy as np
import pytest

from gpu_common import backend, rel_err  # noqa: F401
from slai_amd import _ffi
from slai_amd import gguf_writer as gw
from test_gpu_prefill import SELF_TOL

pytestmark = pytest.mark.gpu


# tokens on top of cached ones: 512 and 513 positions, one wave's block more than eight waves have, the last block with 1, 31 and 32 positions
@pytest.mark.parametrize("start,n", [(479, 33), (480, 33), (511, 65), (800, 31), (575, 97)])
@pytest.mark.parametrize("kv_f16", [False, True])
@pytest.mark.parametrize("dim,heads,kv_heads", [(896, 7, 1), (512, 8, 8), (288, 6, 6)], ids=["128, grouped", "64", "48"])
def test_blocks(backend, dim, heads, kv_heads, kv_f16, start, n):
    from slai_amd.runtime import Gguf, Llama2
    print("case", dim, kv_f16, start, n, flush=True)
    q8_0 = 8
    g = Gguf(gw.llama_gguf(dim, 768, 2, heads, kv_heads, 512, 1024, q8_0, v_type=q8_0, out_type=q8_0, embd_type=q8_0, std=0.05, norm_random=True))
    prompt = np.random.Generator(np.random.PCG64(start + n)).integers(0, 512, start + n + 1).astype(np.int32)
    out = []
    for chunk in (0, 32):
        m = Llama2(backend, g, _ffi.MODEL_LLAMA, _ffi.KV_F16 if kv_f16 else _ffi.KV_F32)
        m.prefill(prompt[:start], 0, 32)
        m.prefill(prompt[start:-1], start, chunk)
        assert m.prefill_fp32_repeats() == 0
        out.append(m.forward_logits(start + n, int(prompt[-1])))
        m.destroy()
    assert rel_err(out[0], out[1]) < SELF_TOL
    g.close()
