"""The prompt GEMMs in the modes that only a session launches: added to the hidden rows (O, down), the
gate/up pair and the pair as two launches, and Q, K and V in one.

Each format runs a two-layer SiLU model whose prompt lengths take every kernel and token tile: few
workgroups share a row's chunks between waves, more take 8, 16 and then 32 tokens a workgroup.  "ff" has
a wide feed-forward (the pair's tiles), "embd" wide hidden rows (the added ones).  The oracle evaluates the
longest prompt once; the second layer's cached keys and values come from everything the first computes, so
each prompt's must equal the oracle's rows to the bit.
"""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from brisk_hip import HipSession, gguf as G, model, synth  # noqa: E402
import pyoracle  # noqa: E402

FORMATS = {"q4_0": G.T_Q4_0, "q4_1": G.T_Q4_1, "q5_0": G.T_Q5_0, "q8_0": G.T_Q8_0, "q4_k": G.T_Q4_K, "q5_k": G.T_Q5_K,
           "q6_k": G.T_Q6_K, "tq2_0": G.T_TQ2_0}
SHAPES = {"ff": (512, 8, 2048), "embd": (2304, 4, 256)}  # hidden width, query heads, feed-forward width
LENGTHS = (2, 5, 8, 16, 33, 64, 130, 200, 250, 517)
VARIANTS = [(f, {}) for f in FORMATS] + [("q4_k", {"BRISK_HIP_PAIR_SPLIT": "1"}), ("q4_k", {"BRISK_HIP_PREFILL_Q4X": "1"}),
                                         ("q5_k", {"BRISK_HIP_PREFILL_MX": "0"}), ("q6_k", {"BRISK_HIP_PREFILL_MX": "0"})]


def tiny(tmp_path, fmt, shape):
    embd, heads, ff = SHAPES[shape]
    spec = synth.ModelSpec(f"modes-{fmt}-{shape}", "llama", embd, 2, heads, 2, 64, ff, 512, 5e5, eps=1e-5, context=1024,
                           fmt={r: FORMATS[fmt] for r in ("q", "k", "v", "o", "gate", "up", "down")})
    return model.load(synth.write_model(spec, str(tmp_path / "m.gguf")))


def cached(s, cfg, layer, value, n):
    hip = C.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    ptr, nbytes = s.kv_cache(layer, value)
    host = np.empty(nbytes // 2, np.uint16)
    assert hip.hipMemcpy(C.c_void_p(host.ctypes.data), C.c_void_p(ptr), nbytes, 2) == 0  # hipMemcpyDeviceToHost
    return host.reshape(cfg.kv_heads, -1, cfg.head_dim)[:, :n]


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("fmt,env", VARIANTS, ids=[f + "".join("-" + k.rsplit("_", 1)[1].lower() for k in e) for f, e in VARIANTS])
def test_modes_at_each_tile(tmp_path, monkeypatch, fmt, env, shape):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    f, cfg, table = tiny(tmp_path, fmt, shape)
    longest = max(LENGTHS)
    prompt = synth.prompt_ids(longest, cfg.vocab, seed=21)
    o = pyoracle.Oracle(cfg, table, longest + 8)
    o.eval(prompt)
    want = [o.kv(1, v)[:, :longest].copy() for v in (False, True)]
    o.rollback(0)
    scored = o.eval(prompt[:6], all_logits=True)
    o.close()
    with HipSession((f, cfg, table), max_context=longest + 8) as s:
        for n in LENGTHS:
            print(f"[gemm modes] {fmt} {env} {shape}: {n} prompt ids", flush=True)
            s.rollback(0)
            s.eval(prompt[:n])
            for value in (False, True):
                np.testing.assert_array_equal(cached(s, cfg, 1, value, n), want[value][:, :n], err_msg=f"{n} ids, value {value}")
        s.rollback(0)  # drafted tokens, every row's logits
        np.testing.assert_array_equal(s.eval_all(prompt[:6]).view(np.uint32), scored.view(np.uint32))
