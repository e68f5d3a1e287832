"""Row tiles spread evenly over the device (gemv_spread_kernel): where its tiles and runs meet."""
import numpy as np
import pytest

from gpu_common import backend  # noqa: F401
from slai_amd import synth

pytestmark = pytest.mark.gpu
NAMES = {2: "q4_0", 8: "q8_0", 12: "q4_k", 13: "q5_k", 14: "q6_k"}


# rows: the last tile whole, one row of it, tiles of a die beyond the others'; columns: the fewest groups, runs that end inside
# tiles and at their ends, two units per wave.  Beside the rule's edges: too few units for every run (32 tiles of 10 groups), tiles too small for a second round (352 of 92 KB)
@pytest.mark.parametrize("t,rows,cols,gated,spread", [(12, 2048, 2560, True, False), (12, 2560, 2560, True, True), (8, 1985, 3584, True, True), (13, 4609, 3584, True, True),
                                                      (12, 6144, 2560, True, True), (2, 6100, 4096, True, True), (14, 3072, 2560, False, True), (12, 8192, 5120, False, True),
                                                      (8, 16385, 2048, True, True), (12, 22528, 4096, True, True), (14, 18944, 3584, False, True), (12, 22465, 2560, False, False),
                                                      (12, 22465, 2560, True, True)],
                         ids=lambda v: NAMES.get(v, str(v)))
def test_spread_against_float64(backend, t, rows, cols, gated, spread):
    from slai_amd import _ffi
    from slai_amd.runtime import GpuQuantMatrix, GpuTensor, LlmContext
    print("case", NAMES[t], rows, cols, gated, flush=True)
    mats = [GpuQuantMatrix(backend, t, rows, cols, synth.normal_quantized(5 + i, t, rows, cols, 0.02), layout=_ffi.LAYOUT_TILE64) for i in range(2 if gated else 1)]
    x, w = synth.normal(7, cols, 1.0), 1 + synth.normal(8, cols, 0.1)
    xd, wd, prep, out = GpuTensor.vector(backend, x), GpuTensor.vector(backend, w if gated else np.ones(cols, np.float32)), GpuTensor(backend, cols + cols // 16), GpuTensor(backend, rows)
    c = LlmContext(backend)
    c.rms_norm_prepare(prep, xd, wd)
    results, before = [], backend.spread_launches()
    for _ in range(3):                                         # the counts are back at zero after each launch
        if gated:
            c.ffn_gate_up_silu_prepared(out, mats[0], mats[1], xd, prep, 1e-5)
        else:
            c.matmul_quant_assign_prepared(out, mats[0], prep)
        results.append(out.read())
    assert backend.spread_launches() - before == (3 if spread else 0)
    assert all(np.array_equal(results[0], r) for r in results[1:])
    x64 = x.astype(np.float64)
    if gated:
        n = x64 * w / np.sqrt(np.mean(x64 * x64) + 1e-5)
        g, u = (np.array([np.dot(row, n) for row in m.dequantize().astype(np.float64)]) for m in mats)
        ref = u * g / (1 + np.exp(-g))
    else:
        ref = mats[0].dequantize().astype(np.float64) @ x64
    # sums of at most 5120 products in 32 bits, taken in lanes and blocks: a few 2^-24 of their norm, twice in a gated product
    assert np.linalg.norm(results[0] - ref) / np.linalg.norm(ref) < 1.5e-6
    for o in mats + [xd, wd, prep, out]:
        o.destroy()


# q/k/v of grouped queries in one launch, v in another format: 72 tiles with biases (behind the projection), and heads of 96 whose keys and values are tiles with 32 rows missing
@pytest.mark.parametrize("dim,heads,kv_heads,t,bias,kv_f16", [(3584, 28, 4, 12, True, True), (3584, 28, 4, 12, False, False), (3072, 32, 1, 13, False, False)],
                         ids=["Qwen2-7B shape", "without biases, f32 cache", "one head of 96"])
def test_decode_of_mixed_formats_vs_oracle(backend, dim, heads, kv_heads, t, bias, kv_f16):
    from slai_amd import _ffi
    from slai_amd import gguf_writer as gw
    from test_gpu_models import check_llama
    q6_k, layers, steps = 14, 3, 10
    print("case", dim, heads, kv_heads, NAMES[t], flush=True)
    data = gw.llama_gguf(dim, 1024, layers, heads, kv_heads, 512, 64, t, v_type=q6_k, out_type=q6_k, embd_type=t, arch="qwen2" if bias else "llama", bias=bias, std=0.03, norm_random=True)
    before = backend.spread_launches()
    check_llama(backend, data, [5, 77, 300, 9], steps, kv_f16=kv_f16, model_type=_ffi.MODEL_QWEN2 if bias else _ffi.MODEL_LLAMA, neox=int(bias), name=b"qwen2" if bias else b"llama")
    # q/k/v of every layer but the first, whose input no projection has prepared, at each of eight positions in fused kernels, and when the loop's graphs are captured
    assert backend.spread_launches() - before >= 8 * (layers - 1)


def test_whatever_was_loaded_before():
    """A call's last bits are those of a context of its own also where a model was loaded in between: a prepared operator call and a GPT-2 that has no one-launch form."""
    from slai_amd import _ffi
    from slai_amd import gguf_writer as gw
    from slai_amd.runtime import Backend, Gguf, GpuQuantMatrix, GpuTensor, Gpt2, Llama2, LlmContext
    b = Backend(0)
    rows, cols, t = 2048, 4096, 8
    mat = GpuQuantMatrix(b, t, rows, cols, synth.normal_quantized(5, t, rows, cols, 0.02), layout=_ffi.LAYOUT_TILE64)
    xd, wd, prep, out = GpuTensor.vector(b, synth.normal(7, cols, 1.0)), GpuTensor.vector(b, np.ones(cols, np.float32)), GpuTensor(b, cols + cols // 16), GpuTensor(b, rows)
    c = LlmContext(b)
    c.rms_norm_prepare(prep, xd, wd)
    wide = Gguf(gw.gpt2_gguf(2048, 2, 32, 8192, 512, 1024, t, std=0.02))
    prompt = np.random.Generator(np.random.PCG64(3)).integers(0, 512, 490).astype(np.int32)

    def both():
        c.matmul_quant_assign_prepared(out, mat, prep)
        m = Gpt2(b, wide, _ffi.KV_F32)
        m.prefill(prompt[:-1], 0, 0)
        logits = m.forward_logits(prompt.size - 1, int(prompt[-1]))
        m.destroy()
        return out.read(), logits

    before = both()
    g = Gguf(gw.llama_gguf(256, 512, 1, 2, 2, 512, 64, 12, v_type=14, out_type=14, embd_type=12))
    Llama2(b, g, _ffi.MODEL_LLAMA, _ffi.KV_F16).destroy()
    after = both()
    assert all(np.array_equal(x, y) for x, y in zip(before, after))
    for o in (mat, xd, wd, prep, out, g, wide, b):
        o.close() if hasattr(o, "close") else o.destroy()


def test_the_attention_switch_leaves_them_alone(monkeypatch):
    """SLAI_FUSE_QKV_ATTN=0 is about q/k/v and attention: what a comparison by it measures is not also the sharing of tiles."""
    from slai_amd import _ffi
    from slai_amd import gguf_writer as gw
    from slai_amd.runtime import Backend, Gguf, GpuQuantMatrix, GpuTensor, Gpt2, LlmContext
    rows, cols, t = 2048, 4096, 8
    wide = Gguf(gw.gpt2_gguf(2048, 2, 32, 8192, 512, 1024, t, std=0.02))
    prompt = np.random.Generator(np.random.PCG64(3)).integers(0, 512, 490).astype(np.int32)
    results = []
    for switch in ("1", "0"):
        monkeypatch.setenv("SLAI_FUSE_QKV_ATTN", switch)
        b = Backend(0)
        mat = GpuQuantMatrix(b, t, rows, cols, synth.normal_quantized(5, t, rows, cols, 0.02), layout=_ffi.LAYOUT_TILE64)
        xd, wd, prep, out = GpuTensor.vector(b, synth.normal(7, cols, 1.0)), GpuTensor.vector(b, np.ones(cols, np.float32)), GpuTensor(b, cols + cols // 16), GpuTensor(b, rows)
        c = LlmContext(b)
        c.rms_norm_prepare(prep, xd, wd)
        c.matmul_quant_assign_prepared(out, mat, prep)
        m = Gpt2(b, wide, _ffi.KV_F32)
        m.prefill(prompt[:-1], 0, 0)
        results.append((out.read(), m.forward_logits(prompt.size - 1, int(prompt[-1]))))
        for o in (mat, xd, wd, prep, out, m):
            o.destroy()
        b.close()
    wide.close()
    assert np.array_equal(results[0][0], results[1][0])
    assert np.array_equal(results[0][1], results[1][1])
