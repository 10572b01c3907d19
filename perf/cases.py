"""Performance cases of the token path: what a program that uses the library has it do.

Kernel-level cases call the C ABI's quantise / matmul / gemv on device memory, as code written
against KernelSet does.  Session cases call ``HipSession`` (Engine's eval / eval_all): a decode
step that returns logits for a host sampler, a prompt, a verification of drafted tokens, a chunk
of a perplexity run.  Shapes and formats are ``brisk_hip.synth.SPECS``'; most session cases run a
slice of a model's layers with a small vocabulary, so that the blocks themselves are what is timed,
and two run a whole model.  Weights, caches and inputs are random, made from the seed on the GPU.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "brisk-llm_amd"))
from brisk_hip import HipSession, gguf as G, lib as L, model as M, synth  # noqa: E402

CONTEXT = 4096        # positions of every session (a chat program's usual context)
SLICE_VOCAB = 4096    # vocabulary of the sessions that run a slice of a model's layers

FORMATS = {"q4_0": G.T_Q4_0, "q4_1": G.T_Q4_1, "q5_0": G.T_Q5_0, "q8_0": G.T_Q8_0, "q4_k": G.T_Q4_K, "q5_k": G.T_Q5_K,
           "q6_k": G.T_Q6_K, "tq2_0": G.T_TQ2_0}
K_FORMATS = (G.T_Q4_K, G.T_Q5_K, G.T_Q6_K, G.T_TQ2_0)  # multiplied with Q8_K activations, the others with Q8_0
# layers of a slice: enough to hold each kind of layer the family has
SLICE_LAYERS = {"qwen3-0.6b": 4, "qwen3-1.7b": 4, "llama-3.2-1b": 4, "bitnet-2b": 4, "gemma3-1b": 6, "qwen35-0.8b": 4}


def listed():
    return [
        # one small projection with its norm fused, the smallest call: launch and latency
        {"name": "gemv_2048", "kind": "gemv", "format": "q4_0", "rows": 2048, "cols": 2048},
        # an up projection for five drafted tokens
        {"name": "matmul_q4_k_5", "kind": "matmul", "format": "q4_k", "rows": 8192, "cols": 2048, "n": 5},
        # a feed-forward projection for a full batch of 512 rows
        {"name": "matmul_q8_0_512", "kind": "matmul", "format": "q8_0", "rows": 6144, "cols": 2048, "n": 512},
        # a whole model's decode step, its logits back on the host
        {"name": "decode_qwen3_whole", "kind": "eval", "shape": "qwen3-0.6b", "whole": True, "position": 100, "n": 1},
        # decode late in a long conversation
        {"name": "decode_long", "kind": "eval", "shape": "qwen3-1.7b", "whole": False, "position": 4000, "n": 1},
        # decode of a family with sliding windows, post-norms and 256-wide heads, past its window
        {"name": "decode_gemma3", "kind": "eval", "shape": "gemma3-1b", "whole": False, "position": 700, "n": 1},
        # speculative decoding: six drafted tokens verified in one call
        {"name": "verify_llama_6", "kind": "eval_all", "shape": "llama-3.2-1b", "whole": False, "position": 300, "n": 6},
        # perplexity: a 64-token chunk scored, every row's logits
        {"name": "score_bitnet_64", "kind": "eval_all", "shape": "bitnet-2b", "whole": False, "position": 128, "n": 64},
        # a whole model's 512-token prompt
        {"name": "prompt_llama_whole_512", "kind": "eval", "shape": "llama-3.2-1b", "whole": True, "position": 0, "n": 512},
        # a short chat turn on top of an earlier conversation
        {"name": "prompt_qwen3_33", "kind": "eval", "shape": "qwen3-0.6b", "whole": False, "position": 200, "n": 33},
        # an ordinary prompt of the recurrent family
        {"name": "prompt_qwen35_517", "kind": "eval", "shape": "qwen35-0.8b", "whole": False, "position": 0, "n": 517},
        # a long document as the prompt
        {"name": "prompt_long_3001", "kind": "eval", "shape": "qwen3-1.7b", "whole": False, "position": 0, "n": 3001},
    ]


def draw(rng):
    def between(lo, hi):  # over the logarithm
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["gemv", "matmul", "matmul", "decode", "decode", "eval_all", "prompt", "prompt"])
    if kind in ("gemv", "matmul"):
        case = {"kind": kind, "format": rng.choice(sorted(FORMATS)), "rows": between(300, 12000), "cols": 256 * between(1, 32)}
        if kind == "matmul":
            case["n"] = between(2, 512)
        return case
    shapes = ["qwen3-0.6b", "qwen3-1.7b", "llama-3.2-1b", "bitnet-2b", "gemma3-1b"]
    if kind == "decode":
        return {"kind": "eval", "shape": rng.choice(shapes), "whole": False, "position": between(8, 3600), "n": 1}
    if kind == "eval_all":
        return {"kind": "eval_all", "shape": rng.choice(shapes), "whole": False, "position": between(8, 1500), "n": between(2, 64)}
    # a recurrent model's prompt starts the sequence: its state cannot be set from outside
    return {"kind": "eval", "shape": rng.choice(shapes + ["qwen35-0.8b"]), "whole": False, "position": 0, "n": between(2, 2048)}


# ---------------------------------------------------------------- inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(1000003 * (int(seed) + 1))


def _half_bytes(gen, n, lo, hi):
    return torch.empty(n, device="cuda").uniform_(lo, hi, generator=gen).half().view(torch.uint8).view(n, 2)


def _blocks(gen, ttype, rows, cols):
    """[rows, blocks, bytes] random blocks with synth's distributions."""
    elems, size = G.BLOCK[ttype]
    n = rows * cols // elems
    b = torch.randint(0, 256, (n, size), dtype=torch.uint8, device="cuda", generator=gen)
    if ttype in (G.T_Q4_0, G.T_Q4_1, G.T_Q5_0):
        b[:, 0:2] = _half_bytes(gen, n, 0.001, 0.02)
        if ttype == G.T_Q4_1:
            b[:, 2:4] = _half_bytes(gen, n, -0.15, 0.0)
    elif ttype == G.T_Q8_0:
        b[:, 2:][b[:, 2:] == 128] = 129  # quantisers do not write -128
        b[:, 0:2] = _half_bytes(gen, n, 0.0002, 0.004)
    elif ttype in (G.T_Q4_K, G.T_Q5_K):
        b[:, 0:2] = _half_bytes(gen, n, 0.0001, 0.001)
        b[:, 2:4] = _half_bytes(gen, n, 0.0001, 0.001)
    elif ttype == G.T_Q6_K:
        b[:, 192:208] = (b[:, 192:208] % 64) - 32
        b[:, 208:210] = _half_bytes(gen, n, 0.00002, 0.0002)
    else:  # TQ2_0: codes 0..2, one scale a tensor
        code = b[:, :64] % 81
        b[:, :64] = (code % 3) | ((code // 3 % 3) << 2) | ((code // 9 % 3) << 4) | ((code // 27) << 6)
        b[:, 64:66] = _half_bytes(gen, 1, 0.01, 0.03)
    return b.view(rows, cols // elems, size)


class _Weights:
    """A model's tensors by GGUF name, on the GPU (blocks, or floats for vectors), made in a fixed order."""

    def __init__(self, case, gen):
        spec = synth.SPECS[case["shape"]]
        self.spec, ex = spec, {k: v[1] for k, v in spec.extra.items()}
        whole = case["whole"]
        self.layers = spec.layers if whole else SLICE_LAYERS[case["shape"]]
        self.vocab = spec.vocab if whole else SLICE_VOCAB
        self.arch = "bitnet" if spec.arch.startswith("bitnet") else spec.arch
        self.recurrent = tuple(l for l in spec.recurrent_layers if l < self.layers)
        c = self.config = M.ModelConfig(M._ARCH[spec.arch], spec.arch, self.vocab, spec.embd, self.layers, spec.heads, spec.kv_heads,
                                        spec.head_dim, spec.ff, spec.context, spec.rope_base, spec.eps)
        if self.arch == "gemma3":
            c.sliding_window, c.rope_base_local, c.rope_scale = ex["attention.sliding_window"], ex["rope.freq_base_swa"], 1.0
        if self.arch == "qwen35":
            c.rope_dim, c.ssm_state, c.ssm_k_heads = ex["rope.dimension_count"], ex["ssm.state_size"], ex["ssm.group_count"]
            c.ssm_v_heads, c.ssm_inner, c.ssm_conv = ex["ssm.time_step_rank"], ex["ssm.inner_size"], ex["ssm.conv_kernel"]
            c.recurrent_layers = self.recurrent
        self.tensors = {}

        def mat(name, rows, cols, ttype):
            self.tensors[name] = (ttype, rows, cols, _blocks(gen, ttype, rows, cols))

        def vec(name, n, lo=0.8, hi=1.2):
            self.tensors[name] = (G.T_F32, 1, n, torch.empty(n, device="cuda").uniform_(lo, hi, generator=gen))

        e, qd, kvd, f = spec.embd, spec.query_dim, spec.kv_dim, spec.fmt
        mat("token_embd.weight", self.vocab, e, spec.embd_fmt)
        vec("output_norm.weight", e)
        if spec.out_fmt is not None:
            mat("output.weight", self.vocab, e, spec.out_fmt)
        for l in range(self.layers):
            b = f"blk.{l}."
            vec(b + "attn_norm.weight", e)
            if l in self.recurrent:
                inner, heads = c.ssm_inner, c.ssm_v_heads
                mat(b + "attn_qkv.weight", 3 * inner, e, f["q"])
                mat(b + "attn_gate.weight", inner, e, f["q"])
                mat(b + "ssm_alpha.weight", heads, e, f["k"])
                mat(b + "ssm_beta.weight", heads, e, f["k"])
                vec(b + "ssm_a", heads, -4.0, -0.5)
                vec(b + "ssm_dt.bias", heads, -1.0, 1.0)
                vec(b + "ssm_conv1d.weight", c.ssm_conv * 3 * inner, -1.0, 1.0)
                vec(b + "ssm_norm.weight", c.ssm_state)
                mat(b + "ssm_out.weight", e, inner, f["o"])
            else:
                mat(b + "attn_q.weight", 2 * qd if self.arch == "qwen35" else qd, e, f["q"])
                mat(b + "attn_k.weight", kvd, e, f["k"])
                mat(b + "attn_v.weight", kvd, e, f["v"])
                mat(b + "attn_output.weight", e, qd, f["o"])
                if self.arch in ("qwen3", "gemma3", "qwen35"):
                    vec(b + "attn_q_norm.weight", spec.head_dim)
                    vec(b + "attn_k_norm.weight", spec.head_dim)
                if self.arch == "gemma3":
                    vec(b + "post_attention_norm.weight", e)
                    vec(b + "post_ffw_norm.weight", e)
                if self.arch == "bitnet":
                    vec(b + "attn_sub_norm.weight", e)
                    vec(b + "ffn_sub_norm.weight", spec.ff)
            vec(b + ("post_attention_norm.weight" if self.arch == "qwen35" else "ffn_norm.weight"), e)
            mat(b + "ffn_gate.weight", spec.ff, e, f["gate"])
            mat(b + "ffn_up.weight", spec.ff, e, f["up"])
            mat(b + "ffn_down.weight", e, spec.ff, f["down"])

    def attends(self, l):
        return l not in self.recurrent


def _session_inputs(case, seed):
    """(weights, tokens, {(layer, value): cached rows [kv heads][position][head size]})."""
    gen = _generator(seed)
    w = _Weights(case, gen)
    tokens = torch.randint(0, w.vocab, (case["n"],), device="cuda", generator=gen).cpu().numpy().astype(np.int32)
    rows = {}
    if case["position"]:
        for l in range(w.layers):
            for value in (False, True):
                rows[l, value] = torch.randn((w.spec.kv_heads, case["position"], w.spec.head_dim), device="cuda", generator=gen).half()
    return w, tokens, rows


def _kernel_inputs(case, seed):
    gen = _generator(seed)
    t = FORMATS[case["format"]]
    blocks = _blocks(gen, t, case["rows"], case["cols"])
    x = torch.randn((case.get("n", 1), case["cols"]), device="cuda", generator=gen)
    norm = torch.empty(case["cols"], device="cuda").uniform_(0.8, 1.2, generator=gen)
    return t, blocks, x, norm


def _lut(case, t):  # a session's ternary matrices of whole 16-row groups take the 7-bit arithmetic; kernel-level callers say so
    return 1 if t == G.T_TQ2_0 and case["rows"] % 16 == 0 else 0


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def prepare(case, seed):
    lib = L.load()
    if case["kind"] in ("gemv", "matmul"):
        t, blocks, x, norm = _kernel_inputs(case, seed)
        packed = torch.empty(lib.brisk_hip_packed_bytes(t, case["rows"], case["cols"]), dtype=torch.uint8, device="cuda")
        L.check(lib.brisk_hip_pack(t, _ptr(blocks), case["rows"], case["cols"], _ptr(packed), None))
        torch.cuda.synchronize()
        n = x.shape[0]
        row = case["cols"] // 256 * 292 if t in K_FORMATS else case["cols"] // 32 * 34
        return {"case": case, "type": t, "packed": packed, "x": x, "norm": norm, "flags": _lut(case, t),
                "rows8": torch.empty(n * row, dtype=torch.uint8, device="cuda"),
                "out": torch.empty((n, case["rows"]), dtype=torch.float32, device="cuda")}
    w, tokens, rows = _session_inputs(case, seed)
    table = [M.TensorRef(name, t, r, c, data.cpu().numpy().reshape(-1).view(np.uint8)) for name, (t, r, c, data) in w.tensors.items()]
    s = HipSession((None, w.config, table), max_context=CONTEXT)
    if rows:
        hip = C.CDLL("libamdhip64.so")
        hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
        for (layer, value), r in rows.items():
            dst, nbytes = s.kv_cache(layer, value)
            full = torch.zeros((r.shape[0], nbytes // (2 * r.shape[0] * r.shape[2]), r.shape[2]), dtype=torch.float16, device="cuda")
            full[:, :r.shape[1]] = r
            torch.cuda.synchronize()
            assert hip.hipMemcpy(C.c_void_p(dst), _ptr(full), nbytes, 3) == 0
        s.set_position(case["position"])
    return {"case": case, "session": s, "tokens": tokens}


def run(state):
    case = state["case"]
    if case["kind"] in ("gemv", "matmul"):
        lib, st = L.load(), C.c_void_p(torch.cuda.current_stream().cuda_stream)
        t, rows, cols, n = state["type"], case["rows"], case["cols"], case.get("n", 1)
        if case["kind"] == "gemv":
            L.check(lib.brisk_hip_gemv(t, state["flags"], _ptr(state["packed"]), rows, cols, _ptr(state["x"]), _ptr(state["norm"]), 1e-6,
                                       _ptr(state["out"]), 0, st))
            return state["out"]
        if t in K_FORMATS:
            L.check(lib.brisk_hip_quantize_q8_k(_ptr(state["x"]), _ptr(state["rows8"]), n * cols, 7 if state["flags"] else 8, st))
        else:
            L.check(lib.brisk_hip_quantize_q8_0(_ptr(state["x"]), _ptr(state["rows8"]), n * cols, st))
        L.check(lib.brisk_hip_matmul(t, state["flags"], _ptr(state["packed"]), rows, cols, _ptr(state["rows8"]), n, _ptr(state["out"]),
                                     rows, st))
        return state["out"]
    s = state["session"]
    s.rollback(case["position"])
    return s.eval(state["tokens"]) if case["kind"] == "eval" else s.eval_all(state["tokens"])


# ---------------------------------------------------------------- what a pass cannot do without

def _layer_matrices(case):
    """(rows, cols, type) of every matrix of the case's layers."""
    spec = synth.SPECS[case["shape"]]
    layers = spec.layers if case["whole"] else SLICE_LAYERS[case["shape"]]
    e, qd, kvd, f, out = spec.embd, spec.query_dim, spec.kv_dim, spec.fmt, []
    for l in range(layers):
        if l in spec.recurrent_layers:
            inner, heads = spec.extra["ssm.inner_size"][1], spec.extra["ssm.time_step_rank"][1]
            out += [(4 * inner, e, f["q"]), (2 * heads, e, f["k"]), (e, inner, f["o"])]
        else:
            out += [((2 if spec.arch == "qwen35" else 1) * qd, e, f["q"]), (kvd, e, f["k"]), (kvd, e, f["v"]), (e, qd, f["o"])]
        out += [(spec.ff, e, f["gate"]), (spec.ff, e, f["up"]), (e, spec.ff, f["down"])]
    return out, layers


def work(case):
    def size(rows, cols, t):
        return rows * cols // G.BLOCK[t][0] * G.BLOCK[t][1]

    if case["kind"] in ("gemv", "matmul"):
        n, rows, cols = case.get("n", 1), case["rows"], case["cols"]
        return {"bytes": size(rows, cols, FORMATS[case["format"]]) + 4 * n * (rows + cols), "flops": 2 * n * rows * cols}
    spec, n, p = synth.SPECS[case["shape"]], case["n"], case["position"]
    mats, layers = _layer_matrices(case)
    vocab = spec.vocab if case["whole"] else SLICE_VOCAB
    scored = n if case["kind"] == "eval_all" else 1
    bytes_ = sum(size(*m) for m in mats) + size(vocab, spec.embd, spec.out_fmt if spec.out_fmt is not None else spec.embd_fmt)
    flops = sum(2 * n * r * c for r, c, _ in mats) + 2 * scored * vocab * spec.embd
    window = spec.extra.get("attention.sliding_window", (None, 0))[1]
    for l in range(layers):
        if l in spec.recurrent_layers:
            flops += 8 * n * spec.extra["ssm.inner_size"][1] * spec.extra["ssm.state_size"][1]
            bytes_ += 8 * spec.extra["ssm.inner_size"][1] * spec.extra["ssm.state_size"][1]
            continue
        seen = sum(min(p + i + 1, window) if window and l % 6 != 5 else p + i + 1 for i in range(n))
        flops += 4 * seen * spec.query_dim
        first = max(0, p + 1 - window) if window and l % 6 != 5 else 0
        bytes_ += 4 * spec.kv_dim * (p + n - first) + 4 * spec.kv_dim * n
    return {"bytes": bytes_ + 4 * scored * vocab, "flops": flops}


def tolerance(case):
    # Kernel-level: 32-bit sums over rows already quantised, where an activation that lies on a
    # rounding boundary may go the other way.  Sessions: such a step moves what follows, layer by layer.
    if case["kind"] in ("gemv", "matmul"):
        return {"rel": 1e-3}
    return {"rel": 0.03 if case["whole"] else 0.02}


# ---------------------------------------------------------------- the same in 64 bits

def _half(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(ttype, b):
    """[rows, blocks, bytes] -> [rows, cols] float64 (the GGUF block formats)."""
    i8 = lambda v: v.contiguous().view(torch.int8).double()  # noqa: E731
    if ttype == G.T_Q8_0:
        v = i8(b[..., 2:]) * _half(b[..., 0:2])
    elif ttype in (G.T_Q4_0, G.T_Q4_1):
        q = b[..., 2:] if ttype == G.T_Q4_0 else b[..., 4:]
        v = torch.cat([q & 15, q >> 4], -1).double()
        v = (v - 8) * _half(b[..., 0:2]) if ttype == G.T_Q4_0 else v * _half(b[..., 0:2]) + _half(b[..., 2:4])
    elif ttype == G.T_Q5_0:
        bit = ((b[..., 2:6, None] >> torch.arange(8, device=b.device, dtype=torch.uint8)) & 1).flatten(-2)
        v = (torch.cat([b[..., 6:] & 15, b[..., 6:] >> 4], -1).double() + 16 * bit.double() - 16) * _half(b[..., 0:2])
    elif ttype in (G.T_Q4_K, G.T_Q5_K):
        s = b[..., 4:16].int()
        sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1).double()
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1).double()
        q = b[..., -128:].unflatten(-1, (4, 1, 32))
        v = torch.cat([q & 15, q >> 4], -2).flatten(-3, -2).double()  # [.., 8, 32]
        if ttype == G.T_Q5_K:
            v = v + 16 * ((b[..., None, 16:48] >> torch.arange(8, device=b.device, dtype=torch.uint8)[:, None]) & 1).double()
        v = (v * sc[..., None] * _half(b[..., 0:2])[..., None] - mn[..., None] * _half(b[..., 2:4])[..., None]).flatten(-2)
    elif ttype == G.T_Q6_K:
        ql, qh = b[..., 0:128].unflatten(-1, (2, 2, 32)), b[..., 128:192].unflatten(-1, (2, 1, 32))
        lo = torch.cat([ql & 15, ql >> 4], -2)  # [.., 2, 4, 32]
        hi = torch.cat([(qh >> k) & 3 for k in (0, 2, 4, 6)], -2)
        v = (lo | (hi << 4)).double().flatten(-3) - 32
        v = (v.unflatten(-1, (16, 16)) * i8(b[..., 192:208])[..., None]).flatten(-2) * _half(b[..., 208:210])
    else:  # TQ2_0
        q = b[..., 0:64].unflatten(-1, (2, 1, 32))
        v = torch.cat([(q >> k) & 3 for k in (0, 2, 4, 6)], -2).double().flatten(-3) - 1
        v = v * _half(b[..., 64:66])
    return v.flatten(-2)


def _quantised(x, ttype, bits=8):
    """Rows as their Q8_0 or Q8_K blocks hold them."""
    if ttype not in K_FORMATS:
        v = x.unflatten(-1, (-1, 32))
        d = v.abs().amax(-1, keepdim=True) / 127
        q = torch.round(v / torch.where(d > 0, d, torch.ones_like(d)))
        return (q * d.half().double()).flatten(-2)
    v = x.unflatten(-1, (-1, 256))
    at = v.abs().argmax(-1, keepdim=True)
    top = v.gather(-1, at)
    inv = -(63.0 if bits == 7 else 127.0) / torch.where(top != 0, top, torch.ones_like(top))
    return torch.where(top != 0, torch.round(inv * v).clamp(max=127) / inv, torch.zeros_like(v)).flatten(-2)


def _rms(x, w, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _angles(positions, base, dim):
    """The position angles the models are defined with: a float32 recurrence over the pairs."""
    theta, step, out = positions.astype(np.float32), np.float32(base) ** np.float32(-2.0 / dim), []
    for _ in range(dim // 2):
        out.append(theta.astype(np.float64))
        theta = (theta * step).astype(np.float32)
    return torch.from_numpy(np.stack(out, -1)).cuda()


def _rope(x, ang, adjacent):
    """x [n, heads, dim], the first 2 * pairs dimensions rotated."""
    r = 2 * ang.shape[-1]
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = (x[..., 0:r:2], x[..., 1:r:2]) if adjacent else (x[..., :r // 2], x[..., r // 2:r])
    ra, rb = a * c - b * s, a * s + b * c
    rot = torch.stack([ra, rb], -1).flatten(-2) if adjacent else torch.cat([ra, rb], -1)
    return torch.cat([rot, x[..., r:]], -1)


def _silu(x):
    return x * torch.sigmoid(x)


def _recurrence(w, b, x, mul):
    """A Gated DeltaNet layer over the tokens of x, from the zero state."""
    c, t = w.config, lambda name: w.tensors[b + name][3].double()  # noqa: E731
    heads, dim, taps, n = c.ssm_v_heads, c.ssm_state, c.ssm_conv, x.shape[0]
    qkv, z = mul(b + "attn_qkv.weight", x), mul(b + "attn_gate.weight", x)
    alpha, beta = mul(b + "ssm_alpha.weight", x), mul(b + "ssm_beta.weight", x)
    padded = torch.cat([torch.zeros(taps - 1, qkv.shape[1], dtype=torch.float64, device="cuda"), qkv])
    cw = t("ssm_conv1d.weight").view(-1, taps)
    conv = _silu(sum(padded[i:i + n] * cw[:, i] for i in range(taps))).view(n, 3, heads, dim)
    q, k, v = conv[:, 0], conv[:, 1], conv[:, 2]
    q = q / torch.sqrt(q.square().sum(-1, keepdim=True) + c.eps) / math.sqrt(dim)
    k = k / torch.sqrt(k.square().sum(-1, keepdim=True) + c.eps)
    decay = torch.exp(torch.nn.functional.softplus(alpha + t("ssm_dt.bias"), threshold=40) * t("ssm_a"))
    beta = torch.sigmoid(beta)
    S = torch.zeros(heads, dim, dim, dtype=torch.float64, device="cuda")  # [value][key]
    rows = []
    for i in range(n):
        S = S * decay[i, :, None, None]
        d = (v[i] - torch.matmul(S, k[i, :, :, None])[..., 0]) * beta[i, :, None]
        S = S + d[:, :, None] * k[i, :, None, :]
        rows.append(torch.matmul(S, q[i, :, :, None])[..., 0])
    o = _rms(torch.stack(rows), t("ssm_norm.weight"), c.eps) * _silu(z).view(n, heads, dim)
    return mul(b + "ssm_out.weight", o.flatten(1))


def exact(case, seed):
    if case["kind"] in ("gemv", "matmul"):
        t, blocks, x, norm = _kernel_inputs(case, seed)
        x = x.double()
        if case["kind"] == "gemv":
            x = _rms(x, norm.double(), 1e-6)
        return _quantised(x, t, 7 if _lut(case, t) else 8) @ _dequant(t, blocks).T
    w, tokens, cached = _session_inputs(case, seed)
    spec, n, p0 = w.spec, case["n"], case["position"]
    heads, kvh, hd, eps = spec.heads, spec.kv_heads, spec.head_dim, spec.eps

    def vec(name):
        return w.tensors[name][3].double()

    def mul(name, x):
        t, rows, cols, blocks = w.tensors[name]
        return _quantised(x, t, 7 if t == G.T_TQ2_0 and rows % 16 == 0 else 8) @ _dequant(t, blocks).T

    ids = torch.from_numpy(tokens.astype(np.int64)).cuda()
    et, _, _, eb = w.tensors["token_embd.weight"]
    h = _dequant(et, eb[ids])
    if w.arch == "gemma3":
        h = h * float(np.sqrt(np.float32(spec.embd)))
    positions = np.arange(p0, p0 + n)
    ang = _angles(positions, spec.rope_base, w.config.rope_dim or hd)
    local = _angles(positions, w.config.rope_base_local, hd) if w.arch == "gemma3" else None
    at, seen = torch.arange(p0, p0 + n, device="cuda")[:, None], torch.arange(p0 + n, device="cuda")[None]
    for l in range(w.layers):
        b = f"blk.{l}."
        x = _rms(h, vec(b + "attn_norm.weight"), eps)
        if not w.attends(l):
            h = h + _recurrence(w, b, x, mul)
        else:
            slides = w.arch == "gemma3" and l % 6 != 5
            q, k, v = mul(b + "attn_q.weight", x), mul(b + "attn_k.weight", x).view(n, kvh, hd), mul(b + "attn_v.weight", x).view(n, kvh, hd)
            gate = None
            if w.arch == "qwen35":
                q, gate = q.view(n, heads, 2, hd).unbind(2)
            q = q.reshape(n, heads, hd)
            if b + "attn_q_norm.weight" in w.tensors:
                q, k = _rms(q, vec(b + "attn_q_norm.weight"), eps), _rms(k, vec(b + "attn_k_norm.weight"), eps)
            q, k = (_rope(y, local if slides else ang, w.arch == "llama") for y in (q, k))
            k, v = k.half().double().transpose(0, 1), v.half().double().transpose(0, 1)
            if cached:
                k, v = torch.cat([cached[l, False].double(), k], 1), torch.cat([cached[l, True].double(), v], 1)
            masked = (seen > at) | ((seen <= at - w.config.sliding_window) if slides else torch.zeros_like(seen > at))
            rows = []
            for i in range(heads):
                s = (q[:, i] @ k[i * kvh // heads].T / math.sqrt(hd)).masked_fill(masked, -math.inf)
                rows.append(torch.softmax(s, -1) @ v[i * kvh // heads])
            a = torch.stack(rows, 1)
            if gate is not None:
                a = a * torch.sigmoid(gate)
            a = a.flatten(1)
            if w.arch == "bitnet":
                a = _rms(a, vec(b + "attn_sub_norm.weight"), eps)
            o = mul(b + "attn_output.weight", a)
            h = h + (_rms(o, vec(b + "post_attention_norm.weight"), eps) if w.arch == "gemma3" else o)
        x = _rms(h, vec(b + ("post_attention_norm.weight" if w.arch == "qwen35" else "ffn_norm.weight")), eps)
        g, u = mul(b + "ffn_gate.weight", x), mul(b + "ffn_up.weight", x)
        if w.arch == "bitnet":
            a = _rms(torch.relu(g).square() * u, vec(b + "ffn_sub_norm.weight"), eps)
        elif w.arch == "gemma3":
            a = torch.nn.functional.gelu(g, approximate="tanh") * u
        else:
            a = _silu(g) * u
        o = mul(b + "ffn_down.weight", a)
        h = h + (_rms(o, vec(b + "post_ffw_norm.weight"), eps) if w.arch == "gemma3" else o)
    if case["kind"] == "eval":
        h = h[-1:]
    out = "output.weight" if "output.weight" in w.tensors else "token_embd.weight"
    logits = mul(out, _rms(h, vec("output_norm.weight"), eps))
    return logits[0] if case["kind"] == "eval" else logits
