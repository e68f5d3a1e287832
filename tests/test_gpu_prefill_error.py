"""The error of the wide prompt pass against float64, operator by operator: a model of two layers whose other parts are
switched off (zero matrices) and whose embeddings are tiny, so that the values the second layer caches are the normalised,
projected result of exactly one operator of the first.  Activations of ordinary and of small size (a trained norm's gains and
hidden values of 0.05, 0.001): the pairs the matrix cores multiply have to hold either."""
import numpy as np
import pytest

from gpu_common import backend  # noqa: F401
from slai_amd import _ffi
from slai_amd import gguf_writer as gw
from test_gpu_prefill import read_cache

pytestmark = pytest.mark.gpu

N = 70                                                         # tokens of the prompt: two 32-token tiles and a part of one


class Model:
    """A two-layer model file and its float64 pass.  part: "attention" or "ffn", what the first layer adds to the residual."""

    def __init__(self, lib, part, wtype, dim, hidden, heads, kv_heads, gain, seed=3, also=None):
        self.lib, self.dim, self.hidden, self.heads, self.kv_heads, self.w = lib, dim, hidden, heads, kv_heads, {}
        off = {"attention": "ffn_down", "ffn": "attn_output"}[part]

        def hook(name, dims, t, data):
            if name == "blk.0.%s.weight" % off:
                data = np.zeros_like(data)
            if name.startswith("token_embd"):         # the residual is the operator's result and next to nothing else
                data = (data.view(np.float32) * np.float32(1e-6)).view(np.uint8)
            if name.endswith("_norm.weight") and name.startswith("blk.0"):
                data = (data.view(np.float32) * np.float32(gain)).view(np.uint8)
            if also:
                dims, t, data = also(name, dims, t, data)
            self.w[name] = (dims, t, data)
            return dims, t, data

        # (rope_base 1: every angle is the position itself, exactly, so the rotation adds no error of its own)
        self.data = gw.llama_gguf(dim=dim, hidden_dim=hidden, n_layers=2, n_heads=heads, n_kv_heads=kv_heads, vocab=128, seq_len=96, wtype=wtype, embd_type=0,
                                  out_type=0, seed=seed, std=0.05, norm_random=True, rope_base=1.0, rms_eps=1e-20, tensor_hook=hook)

    def matrix(self, name):
        dims, t, raw = self.w[name]
        n = int(np.prod(dims))
        if t == 0:
            out = raw.view(np.float32)
        else:
            out = np.empty(n, np.float32)
            raw = np.ascontiguousarray(raw)
            assert self.lib.slo_dequantize(t, raw.ctypes.data, n, out.ctypes.data) == 0
        return out.reshape(dims[::-1] if len(dims) > 1 else (n,)).astype(np.float64)

    def exact(self, tokens):
        """[(keys, values)] of both layers, rows of positions."""
        n, hs, mul = len(tokens), self.dim // self.heads, self.heads // self.kv_heads
        x = self.matrix("token_embd.weight")[tokens]
        c, s = np.cos(np.arange(n, dtype=np.float64))[:, None, None], np.sin(np.arange(n, dtype=np.float64))[:, None, None]

        def rotate(v):
            v = v.reshape(n, -1, hs // 2, 2)
            return np.stack([c * v[..., 0] - s * v[..., 1], s * v[..., 0] + c * v[..., 1]], -1).reshape(n, -1, hs)

        out = []
        for l in range(2):
            m = lambda nm: self.matrix("blk.%d.%s.weight" % (l, nm))  # noqa: E731
            norm = lambda v, nm: v / np.sqrt((v * v).mean(1, keepdims=True) + 1e-20) * m(nm)  # noqa: E731
            a = norm(x, "attn_norm")
            q, k, v = rotate(a @ m("attn_q").T), rotate(a @ m("attn_k").T), a @ m("attn_v").T
            out.append((k.reshape(n, -1), v))
            vh, o = v.reshape(n, -1, hs), np.empty((n, self.heads, hs))
            for h in range(self.heads):
                sc = q[:, h] @ k[:, h // mul].T / np.sqrt(hs)
                sc[np.triu_indices(n, 1)] = -np.inf
                p = np.exp(sc - sc.max(1, keepdims=True))
                o[:, h] = p / p.sum(1, keepdims=True) @ vh[:, h // mul]
            x = x + o.reshape(n, -1) @ m("attn_output").T
            f = norm(x, "ffn_norm")
            g = f @ m("ffn_gate").T
            x = x + (g / (1 + np.exp(-g)) * (f @ m("ffn_up").T)) @ m("ffn_down").T
        return out


def errors(backend, m, kv_f16=False, chunk=0, exact=None, tokens=None):
    """(keys, values of layer 0, values of layer 1) against float64, 2-norms."""
    from slai_amd.runtime import Gguf, Llama2
    if tokens is None:
        tokens = np.random.Generator(np.random.PCG64(5)).integers(0, 128, N).astype(np.int32)
    exact = exact or m.exact(tokens)
    gg = Gguf(m.data)
    dev = Llama2(backend, gg, _ffi.MODEL_LLAMA, _ffi.KV_F16 if kv_f16 else _ffi.KV_F32)
    dev.prefill(tokens, 0, chunk)
    assert dev.prefill_fp32_repeats() == 0
    kvd, dt = m.dim // m.heads * m.kv_heads, np.float16 if kv_f16 else np.float32
    got = [[a.view(dt).astype(np.float64).reshape(-1, kvd) for a in read_cache(backend, dev, l, N * kvd * np.dtype(dt).itemsize)] for l in range(2)]
    dev.destroy(); gg.close()
    rel = lambda a, b: float(np.linalg.norm(a - b) / np.linalg.norm(b))  # noqa: E731
    return rel(got[0][0], exact[0][0]), rel(got[0][1], exact[0][1]), rel(got[1][1], exact[1][1])


SHAPES = {"heads of 128": (512, 1024, 4, 2), "heads of 64": (768, 1536, 12, 12), "heads of 48, rows of 288": (288, 768, 6, 6)}
Q4_0, Q8_0, Q4_K, Q5_K, Q6_K = 2, 8, 12, 13, 14
# 2-norms of errors, relative.  An operator's result: pairs of f16 keep 23 bits of an activation (4.5e-8), a normalised row's
# factor 24 (6e-8), and 32-bit sums over n products err by about 2^-25 sqrt(n / 16 roundings) (n = 1536: 2.9e-7 at most, the
# partial sums being smaller than the last): 3e-7.  The second layer's values lie behind four to five of them: sqrt(5) as much.
BAR = (3e-7, 7e-7)


@pytest.mark.parametrize("part", ["attention", "ffn"])
@pytest.mark.parametrize("wtype", [Q4_K, Q5_K], ids=["q4_k", "q5_k"])
def test_error_of_formats_with_offsets(backend, oracle_lib, part, wtype):
    m = Model(oracle_lib, part, wtype, *SHAPES["heads of 128"], 1.0)
    _, first, second = errors(backend, m)
    assert first < BAR[0] and second < BAR[1], (first, second)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("wtype", [Q8_0, Q4_0, Q4_K, Q6_K], ids=["q8_0", "q4_0", "q4_k", "q6_k"])
@pytest.mark.parametrize("gain", [1.0, 0.05, 0.001])
def test_error_with_small_activations(backend, oracle_lib, shape, wtype, gain):
    """Normalised rows of every size (the first layer's values), and hidden values (the second's) down to about 5e-7."""
    if SHAPES[shape][0] % 256 and wtype not in (Q8_0, Q4_0):
        pytest.skip("blocks of 256 do not divide the rows")
    m = Model(oracle_lib, "ffn", wtype, *SHAPES[shape], gain)
    _, first, second = errors(backend, m)
    assert first < BAR[0] and second < BAR[1], (first, second)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kv_f16", [False, True])
@pytest.mark.parametrize("gain", [1.0, 0.05, 0.01])
def test_error_of_attention(backend, oracle_lib, shape, kv_f16, gain):
    """Queries, keys and values of every size.  An f16 cache rounds what it holds to 2^-11 (2.1e-4 of the values' 2-norm)."""
    m = Model(oracle_lib, "attention", Q8_0, *SHAPES[shape], gain)
    _, first, second = errors(backend, m, kv_f16)
    assert first < (2.5e-4 if kv_f16 else BAR[0]) and second < (6e-4 if kv_f16 else BAR[1]), (first, second)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kv_f16", [False, True])
def test_error_of_sharp_attention(backend, oracle_lib, shape, kv_f16):
    """Queries of 2e-3 against keys of 6e2 and the other way round: the scores are ordinary ones, the pairs are not."""
    for up in ("attn_q", "attn_k"):
        def hook(name, dims, t, data, up=up):
            if name.startswith("blk.0.attn_q.") or name.startswith("blk.0.attn_k."):
                data = data.copy()
                d = data.reshape(-1, 34)[:, :2].copy().view(np.float16) * np.float16(2.0 ** 9 if up in name else 2.0 ** -9)
                data.reshape(-1, 34)[:, :2] = d.view(np.uint8)
            return dims, t, data

        m = Model(oracle_lib, "attention", Q8_0, *SHAPES[shape], 1.0, also=hook)
        keys, _, second = errors(backend, m, kv_f16)
        assert second < (6e-4 if kv_f16 else 2 * BAR[1]), (up, keys, second)


@pytest.mark.parametrize("wtype,block", [(Q8_0, 34), (Q4_K, 144)], ids=["q8_0", "q4_k"])
def test_aligned_activations_are_read_once(backend, oracle_lib, wtype, block):
    """Normalised rows of about 3000 of one sign: each fits f16, the sum of 32 does not.  Such a prompt needs no fp32 repeat
    (`errors` looks), whether the format reads the sums or not."""
    def hook(name, dims, t, data):
        if name.startswith("token_embd"):
            data = (1 + 0.1 * np.random.Generator(np.random.PCG64(1)).standard_normal(data.size // 4)).astype(np.float32).view(np.uint8)
        if name in ("blk.0.ffn_gate.weight", "blk.0.ffn_up.weight"):        # hidden values of about 5
            data = data.copy().reshape(-1, block)
            scales = 2 if t == Q8_0 else 4
            data[:, :scales] = (data[:, :scales].copy().view(np.float16) * np.float16(2.0 ** -10)).view(np.uint8)
            data = data.reshape(-1)
        return dims, t, data

    m = Model(oracle_lib, "ffn", wtype, *SHAPES["heads of 128"], 3000.0, also=hook)
    _, first, second = errors(backend, m)
    # Q4_K multiplies q - 8, on average half a step below zero: over 256 activations of one sign its partial sums reach 0.5 * 256
    # steps against a result of sqrt(256) * 4.6, 1.7 times as much, and round accordingly
    assert first < 2 * BAR[0] and second < 2 * BAR[1], (first, second)
