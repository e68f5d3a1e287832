"""The wide prompt pass (kernels_prompt_wide.hip, kernels_prompt_attention.hip) at the edges of its tiles: 64-token blocks of
two 32-token tiles, 256-row blocks (the 2816-row matrices end inside one), every block format and tile height, both head
sizes and cache types, passes of more than 1024 tokens and passes on top of cached positions.  The bars are those of
test_gpu_prefill.py: greedy ids identical to the oracle's, caches and logits within f16 rounding / summation order of the
token-by-token pass."""
import numpy as np
import pytest

from gpu_common import backend, rel_err  # noqa: F401
from slai_amd import _ffi
from slai_amd import gguf_writer as gw
from test_gpu_prefill import check_prefill

pytestmark = pytest.mark.gpu


def prompt_of(n, vocab, seed=9):
    return np.random.Generator(np.random.PCG64(seed)).integers(0, vocab, n)


@pytest.mark.parametrize("n", [34, 65, 66, 97, 129, 290])      # n - 1 tokens are read in one pass
@pytest.mark.parametrize("kv_f16", [False, True])
def test_wide_token_tile_edges(backend, n, kv_f16):
    data = gw.llama_gguf(dim=1024, hidden_dim=2816, n_layers=2, n_heads=8, n_kv_heads=4, vocab=512, seq_len=320, wtype=12, v_type=14, seed=21, std=0.05,
                         norm_random=True)
    check_prefill(backend, data, prompt_of(n, 512), 6, [0], kv_f16)


@pytest.mark.parametrize("wtype", [12, 13, 14, 8, 2], ids=["q4_k", "q5_k", "q6_k", "q8_0", "q4_0"])
@pytest.mark.parametrize("dims", [(768, 1536, 12), (512, 2816, 8), (1024, 16640, 8)], ids=["64-row tiles", "32-row tiles", "more than 64 super-blocks"])
def test_wide_formats_and_tile_heights(backend, wtype, dims):
    dim, hidden, heads = dims
    data = gw.llama_gguf(dim=dim, hidden_dim=hidden, n_layers=2, n_heads=heads, n_kv_heads=heads, vocab=512, seq_len=128, wtype=wtype, seed=22, std=0.05,
                         norm_random=True)
    check_prefill(backend, data, prompt_of(71, 512), 6, [0], True)


@pytest.mark.parametrize("n", [9, 10, 32, 33, 34])             # n - 1 tokens: the fewest of a pass, and around one token tile
@pytest.mark.parametrize("wtype", [12, 13, 14, 8, 2], ids=["q4_k", "q5_k", "q6_k", "q8_0", "q4_0"])
@pytest.mark.parametrize("dims", [(256, 768, 4), (1024, 3072, 8)], ids=["fewer super-blocks than waves", "several super-blocks a wave"])
def test_wide_few_tokens(backend, wtype, dims, n):
    """The form for few tokens, in which the waves of a workgroup share the super-blocks out: some without one, some with several."""
    dim, hidden, heads = dims
    data = gw.llama_gguf(dim=dim, hidden_dim=hidden, n_layers=2, n_heads=heads, n_kv_heads=heads // 2, vocab=512, seq_len=64, wtype=wtype, seed=26, std=0.05,
                         norm_random=True)
    check_prefill(backend, data, prompt_of(n, 512), 6, [0], n % 2 == 0)


def test_wide_bias_neox_grouped_queries_continued(backend):
    """Qwen2 form: biases, NeoX pairs, seven query heads per cache head; a second pass on top of 45 cached positions."""
    data = gw.llama_gguf(dim=1792, hidden_dim=2048, n_layers=2, n_heads=14, n_kv_heads=2, vocab=512, seq_len=192, wtype=12, v_type=14, seed=23, std=0.05,
                         arch="qwen2", bias=True, norm_random=True, rope_base=1000000.0, rms_eps=1e-6)
    check_prefill(backend, data, prompt_of(160, 512), 6, [0], True, model_type=_ffi.MODEL_QWEN2, neox=1, name=b"qwen2", split_at=45)


def test_wide_more_than_one_pass(backend):
    data = gw.llama_gguf(dim=512, hidden_dim=512, n_layers=2, n_heads=4, n_kv_heads=4, vocab=512, seq_len=1216, wtype=8, seed=24, std=0.05, norm_random=True)
    check_prefill(backend, data, prompt_of(1172, 512), 6, [0], False)


@pytest.mark.parametrize("scale,repeats", [(1.0, 0), (5.0e4, 1)])
def test_wide_values_beyond_f16_repeat_in_fp32(backend, scale, repeats):
    data = gw.llama_gguf(dim=1024, hidden_dim=2816, n_layers=2, n_heads=8, n_kv_heads=8, vocab=500, seq_len=96, wtype=12, v_type=14, seed=77, std=0.05,
                         ffn_norm_scale=scale)
    check_prefill(backend, data, prompt_of(70, 500, 78), 6, [0], True, expect_repeats=repeats)


@pytest.mark.parametrize("kv_f16", [False, True])
@pytest.mark.parametrize("wtype", [8, 14], ids=["q8_0", "q6_k"])
def test_wide_gpt2(backend, kv_f16, wtype):
    from helpers import OracleGguf
    from slai_amd.runtime import Gguf, Gpt2
    data = gw.gpt2_gguf(n_layer=2, seed=51, std=0.05, wtype=wtype, vocab=2000, n_seq=256)
    g = OracleGguf(data); L = g.L
    om = L.slo_gpt2_from_gguf(g.h, int(kv_f16))
    n, n_gen = 150, 6
    prompt = prompt_of(n, 2000, 52).astype(np.int32)
    steps = n - 1 + n_gen
    ref, ref_logits = np.zeros(steps, np.int32), np.zeros((steps, 2000), np.float32)
    assert L.slo_gpt2_generate(om, prompt.ctypes.data, n, 0, steps, -1, ref.ctypes.data, ref_logits.ctypes.data) == steps
    gg = Gguf(data)
    m = Gpt2(backend, gg, _ffi.KV_F16 if kv_f16 else _ffi.KV_F32)
    m.generate(prompt, n - 1)
    base = m.forward_logits(n - 1, int(prompt[-1]))
    m.destroy()
    for split in (None, 40):
        m = Gpt2(backend, gg, _ffi.KV_F16 if kv_f16 else _ffi.KV_F32)
        if split:
            m.prefill(prompt[:split], 0)
        m.prefill(prompt[split or 0:-1], split or 0)
        logits = m.forward_logits(n - 1, int(prompt[-1]))
        assert rel_err(logits, ref_logits[n - 1]) < 1e-2
        assert rel_err(logits, base) < 1e-3
        got, _ = m.generate(prompt, n_gen, start_pos=n - 1)
        assert np.array_equal(got, ref[n - 1:])
        m.destroy()
    gg.close(); L.slo_gpt2_free(om); g.close()


@pytest.mark.parametrize("n", [5, 34, 70])
@pytest.mark.parametrize("kv_f16", [False, True])
@pytest.mark.parametrize("wtype,hidden", [(8, 768), (2, 800)], ids=["q8_0", "q4_0, 800 hidden columns"])
def test_wide_rows_that_are_no_multiple_of_256(backend, n, kv_f16, wtype, hidden):
    """Rows of 288 and heads of 48: the pass reads padded copies in tiles (the model's own matrices keep the row layout)."""
    data = gw.tiny_llama_gguf(seed=99, std=0.1, norm_random=True, vocab=4096, wtype=wtype, hidden_dim=hidden)
    check_prefill(backend, data, prompt_of(n, 4096), 8, [0], kv_f16, expect_path=0)


@pytest.mark.parametrize("setting,copies", [(None, True), (("SLAI_TILED", "0"), False), (("SLAI_PROMPT_COPY_MB", "1"), False)], ids=["default", "rows asked for", "too little memory allowed"])
def test_padded_copies_are_bounded(monkeypatch, setting, copies):
    """Padded copies (6 MB here) are made only where tiles are allowed and within the bound; without them the prompt goes
    through the token loop, to the bit."""
    from slai_amd.runtime import Backend, Gguf, Llama2
    from test_gpu_prefill import read_cache
    if setting:
        monkeypatch.setenv(*setting)
    b = Backend(0)
    gg = Gguf(gw.tiny_llama_gguf(seed=99, std=0.1, norm_random=True, vocab=4096))
    prompt = prompt_of(41, 4096).astype(np.int32)
    caches = []
    for loop in (True, False):
        m = Llama2(b, gg, _ffi.MODEL_LLAMA, _ffi.KV_F32)
        m.generate(prompt, 40) if loop else m.prefill(prompt[:40])
        caches.append(np.concatenate([a for l in range(6) for a in read_cache(b, m, l, 40 * 288 * 4)]))
        m.destroy()
    gg.close(); b.close()
    assert np.array_equal(*caches) == (not copies)


@pytest.mark.parametrize("scale,repeats", [(1.0, 0), (5.0e4, 1)])
def test_wide_padded_copies_repeat_in_the_token_loop(backend, scale, repeats):
    """Values beyond f16 in a model whose pass reads padded copies: the repeat is the token loop, whose caches it leaves."""
    data = gw.tiny_llama_gguf(seed=98, std=0.1, norm_random=True, vocab=4096, ffn_norm_scale=scale)
    check_prefill(backend, data, prompt_of(50, 4096), 8, [0], False, expect_path=0, expect_repeats=repeats)


@pytest.mark.parametrize("scale,repeats", [(1.0, 0), (5.0e4, 1)])
def test_wide_gpt2_values_beyond_f16_repeat_in_fp32(backend, scale, repeats):
    from helpers import OracleGguf
    from slai_amd.runtime import Gguf, Gpt2
    data = gw.gpt2_gguf(n_layer=2, seed=53, std=0.05, vocab=2000, n_seq=256, ffn_norm_scale=scale)
    g = OracleGguf(data); L = g.L
    om = L.slo_gpt2_from_gguf(g.h, 0)
    n, n_gen = 70, 6
    prompt = prompt_of(n, 2000, 54).astype(np.int32)
    steps = n - 1 + n_gen
    ref, ref_logits = np.zeros(steps, np.int32), np.zeros((steps, 2000), np.float32)
    assert L.slo_gpt2_generate(om, prompt.ctypes.data, n, 0, steps, -1, ref.ctypes.data, ref_logits.ctypes.data) == steps
    gg = Gguf(data)
    m = Gpt2(backend, gg, _ffi.KV_F32)
    assert m.prefill(prompt[:-1], 0) > 0
    assert m.prefill_fp32_repeats() == repeats
    assert rel_err(m.forward_logits(n - 1, int(prompt[-1])), ref_logits[n - 1]) < 1e-2
    got, _ = m.generate(prompt, n_gen, start_pos=n - 1)
    assert np.array_equal(got, ref[n - 1:])
    m.destroy(); gg.close(); L.slo_gpt2_free(om); g.close()


@pytest.mark.parametrize("wtype", [12, 13, 14, 8, 2], ids=["q4_k", "q5_k", "q6_k", "q8_0", "q4_0"])
@pytest.mark.parametrize("hidden,n,form", [(16640, 1000, 3), (2816, 640, 2), (4096, 1000, 0), (3072, 640, 1)],
                         ids=["whole rounds, then shared tiles", "slim workgroups", "large workgroups", "small workgroups"])
def test_wide_many_tokens_against_passes_of_32(backend, wtype, hidden, n, form):
    """Gate + up in each form that many tokens take (down in large workgroups for 1000 tokens, in slim ones for 640), against the kernels for up to 32
    tokens.  Either is within 1.3e-6 of exact sums (2-norm, values of a second layer); the largest element of a million is five times that of each."""
    from slai_amd.runtime import Gguf, Llama2
    import ctypes as C
    g = Gguf(gw.llama_gguf(dim=1024, hidden_dim=hidden, n_layers=2, n_heads=8, n_kv_heads=8, vocab=512, seq_len=1024, wtype=wtype, seed=26, std=0.05, norm_random=True))
    rows = []
    for chunk in (0, 32):
        m = Llama2(backend, g, _ffi.MODEL_LLAMA, _ffi.KV_F32)
        assert m.prompt_form(n, 2) == form
        m.prefill(prompt_of(n, 512), 0, chunk)
        out = []
        for b in m.kv_buffers(1):
            a = np.empty((n, 1024), np.float32)
            backend.check(backend.L.slai_read_buffer(backend.h, b, 0, a.ctypes.data, C.c_size_t(a.nbytes)))
            out.append(a)
        rows.append(out)
        m.destroy()
    for a, b in zip(*rows):
        assert rel_err(a, b) < 1.5e-5
    g.close()


def test_wide_pass_of_fewer_tokens_is_no_slower(backend):
    """Two layers of the 7B shape, Q8_0: with q/k/v in the form for few tokens 831 of them took 1.13 times as long as 896, now 0.96 to 1.02 times (either has the same
    rounds of large workgroups, and runs differ by 2 %)."""
    from slai_amd.runtime import Gguf, Llama2
    g = Gguf(gw.llama_gguf(dim=4096, hidden_dim=11008, n_layers=2, n_heads=32, n_kv_heads=32, vocab=512, seq_len=1024, wtype=8, seed=27, std=0.02, distinct_layers=1))
    m = Llama2(backend, g, _ffi.MODEL_LLAMA, _ffi.KV_F16)
    best = {n: min(m.prefill(prompt_of(n, 512), 0) for _ in range(20)) for n in (831, 896)}
    assert best[831] < 1.07 * best[896], best
    m.destroy(); g.close()
