"""The work a user of this framework has it do, as cases to measure.

A case is one call (or, for a model, one step) through the C ABI binding:
attention over a KV cache (decode steps, prompts, prompt chunks), ragged
batched decode, image-encoder attention, F32 and quantized matrix products, a
quantized feed-forward block and a whole F32 Llama-family step. `listed()` has the sizes that matter
most, `draw(rng)` others of the same ranges.

All single calls share one arena, as the layers of a session do, so the
passes of several states run in order on one stream.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from synapse_amd import capi
from synapse_amd.capi import (NO_OFFSET, SYN_ADD, SYN_F16, SYN_F32, SYN_SILU_MUL, Arena, AttnDesc, AttnRopeDesc,
                              ElementwiseDesc, KvDesc, MatmulDesc, MatmulQDesc, NormDesc, SelfDesc, SeqDesc, check,
                              lib)
from synapse_amd.gguf import BLOCK, F32, Q4_0, Q4_K, Q5_0, Q6_K, Q8_0, GGUFError, TensorInfo
from synapse_amd.llama import DeviceLlama, rope_theta_scale

ARENA_BYTES = 10 << 30
ROPE_BASE = 500000.0
RMS_EPS = 1e-5
QTYPES = {"q4_0": Q4_0, "q5_0": Q5_0, "q8_0": Q8_0, "q4_k": Q4_K, "q6_k": Q6_K}

# ---- the cases ---------------------------------------------------------------


def listed() -> list[dict]:
    return [
        # One decode step of one layer of a Llama-3-8B-shaped model, RoPE and
        # cache append included: what a chat does per layer and token.
        dict(name="decode-4k", kind="attention", rope=True, dtype="f32", heads=32, kv_heads=8, head_dim=128,
             pos=4096, n=1, max_ctx=8192),
        # The same call where nothing but launches and latency is left: a small
        # model's early token.
        dict(name="decode-small", kind="attention", rope=True, dtype="f32", heads=14, kv_heads=2, head_dim=64, pos=300,
             n=1, max_ctx=2048),
        # A whole prompt in one run, binary16 rows.
        dict(name="prefill-2048", kind="attention", rope=False, dtype="f16", heads=32, kv_heads=8, head_dim=128,
             pos=0, n=2048, max_ctx=2048),
        # A further chunk of a long prompt (or a later turn of a chat) against
        # what is cached already; neither end on a tile edge.
        dict(name="chunk-509-at-7683", kind="attention", rope=True, dtype="f32", heads=32, kv_heads=8, head_dim=128,
             pos=7683, n=509, max_ctx=8192),
        # Continuous batching: 16 sequences of very different lengths.
        dict(name="ragged-16", kind="ragged", heads=32, kv_heads=8, head_dim=128, seqs=16, shortest=512,
             longest=32768),
        # A batch of ViT-L/14 images on binary16 rows.
        dict(name="vit-f16-32x257", kind="image", dtype="f16", heads=16, head_dim=64, n=257, batch=32),
        # One image of the f32 encoder (a 32 x 32 grid of patches).
        dict(name="image-f32-1024", kind="image", dtype="f32", heads=12, head_dim=64, n=1024, batch=1),
        # That encoder's largest product (its MLP's first half).
        dict(name="matmul-f32-1024", kind="matmul", n=1024, rows=3072, cols=768, bias=True),
        # One token through a quantized layer's feed-forward half (norm, gate,
        # up, SiLU, down, residual): the bulk of a decode step.
        dict(name="ffn-q4_k_m-1", kind="ffn", n=1, embd=4096, ff=14336),
        # A prompt chunk through that block's first matrix.
        dict(name="gemm-q4_k-512", kind="matmul_q", type="q4_k", n=512, rows=14336, cols=4096, bias=False),
        # A short prompt through the FFN's last matrix.
        dict(name="gemm-q6_k-24", kind="matmul_q", type="q6_k", n=24, rows=4096, cols=14336, bias=False),
        # A whole decode step of a small F32 model: every op of the graph, by
        # the model runner. (F32: in a quantized model one activation rounded
        # the other way changes the logits by percents.)
        dict(name="llama-f32-step", kind="llama", layers=2, embd=2048, ff=5632, heads=16, kv_heads=8, head_dim=128,
             vocab=16000, pos=1000, max_ctx=2048),
    ]


# Head layouts (query heads, KV heads, head size): grouped and ungrouped, the
# odd group of 7, sizes that are not powers of two.
LAYOUTS = [(32, 8, 128), (8, 8, 32), (14, 2, 64), (28, 4, 128), (16, 16, 80), (24, 8, 96), (32, 32, 64)]
# Weight shapes (rows, columns) of language models' layers; the last ones,
# too small to be timed alone with one token, only with several.
SHAPES_Q = [(14336, 4096), (4096, 14336), (4096, 4096), (8192, 2048), (2048, 8192), (1024, 4096), (3072, 1024),
            (2050, 2048), (1000, 768)]
# Weight shapes of image encoders.
SHAPES_F32 = [(3072, 768), (768, 3072), (768, 768), (1152, 588), (577, 768), (1024, 1024)]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def draw(rng) -> dict:
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "ragged", "image", "image", "matmul", "matmul_q",
                       "matmul_q", "matmul_q", "ffn", "llama"])
    if kind in ("decode", "prompt"):
        heads, kv_heads, head_dim = rng.choice(LAYOUTS)
        if kind == "decode":
            n, pos = 1, _log_int(rng, 200, 32767)
        else:
            n = _log_int(rng, 2, 2048)
            pos = rng.choice([0, _log_int(rng, 1, 7680)])
        return dict(kind="attention", rope=rng.random() < 0.7, dtype="f32", heads=heads, kv_heads=kv_heads,
                    head_dim=head_dim, pos=pos, n=n, max_ctx=pos + n + rng.randrange(512)) | (
                        {"rope": False, "dtype": "f16"} if rng.random() < 0.3 else {})
    if kind == "ragged":
        heads, kv_heads, head_dim = rng.choice(LAYOUTS[:4])
        return dict(kind="ragged", heads=heads, kv_heads=kv_heads, head_dim=head_dim, seqs=rng.randint(2, 40),
                    shortest=_log_int(rng, 1, 512), longest=_log_int(rng, 1024, 12000))
    if kind == "image":
        dtype = rng.choice(["f16", "f32"])
        n = _log_int(rng, 49, 1024)
        return dict(kind="image", dtype=dtype, heads=rng.choice([12, 16]), head_dim=rng.choice([32, 64, 72, 80]), n=n,
                    batch=rng.randint(1, max(1, (8192 if dtype == "f16" else 700) // n)))
    if kind == "matmul":
        rows, cols = rng.choice(SHAPES_F32)
        return dict(kind="matmul", n=_log_int(rng, 16, 1024), rows=rows, cols=cols, bias=rng.random() < 0.7)
    if kind == "matmul_q":
        n = rng.choice([1, _log_int(rng, 2, 31), _log_int(rng, 32, 512)])
        rows, cols = rng.choice(SHAPES_Q[:5] if n == 1 else SHAPES_Q)
        return dict(kind="matmul_q", type=rng.choice(sorted(QTYPES)), n=n, rows=rows, cols=cols,
                    bias=rng.random() < 0.3)
    if kind == "ffn":
        embd, ff = rng.choice([(4096, 14336), (4096, 11008), (2048, 8192), (2048, 5632), (1024, 2816)])
        return dict(kind="ffn", n=rng.choice([1, _log_int(rng, 2, 31), _log_int(rng, 32, 256)]), embd=embd, ff=ff)
    heads, kv_heads, head_dim = rng.choice([(16, 16, 64), (16, 8, 128), (14, 2, 64)])
    return dict(kind="llama", layers=rng.randint(1, 3), embd=rng.choice([512, 896, 2048]),
                ff=rng.choice([1536, 2816, 4864]), heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                vocab=rng.choice([2000, 8000, 16000]), pos=_log_int(rng, 1, 2000), max_ctx=2048)


# ---- one session's arena -------------------------------------------------------

_TYPESTR = {torch.float32: "<f4", torch.float16: "<f2", torch.uint8: "|u1"}


class _Session:
    """One arena, its device address, and a first-fit list of free ranges."""

    def __init__(self):
        self.arena = Arena(ARENA_BYTES)
        # The arena object starts with its device address. Outputs are looked
        # at in place through it; a round trip shows that it is the address.
        self.base = ctypes.c_void_p.from_address(self.arena.handle.value).value
        self.free = [(0, ARENA_BYTES)]
        tag = np.random.default_rng().integers(0, 255, 64, dtype=np.uint8)
        self.arena.upload(0, tag)
        self.arena.sync()
        if not np.array_equal(self.view(None, 0, (64,), torch.uint8).cpu().numpy(), tag):
            raise RuntimeError("the arena's device address was not found")

    def view(self, owner, offset: int, shape, dtype) -> torch.Tensor:
        return torch.as_tensor(_View(owner, self.base + offset, tuple(shape), _TYPESTR[dtype]), device="cuda")

    def take(self, nbytes: int) -> int:
        nbytes = capi.align(nbytes)
        for i, (at, size) in enumerate(self.free):
            if size >= nbytes:
                self.free[i] = (at + nbytes, size - nbytes)
                return at
        raise MemoryError(f"out of memory: {nbytes} bytes of the arena")

    def give(self, at: int, nbytes: int) -> None:
        merged = []
        for lo, size in sorted(self.free + [(at, capi.align(nbytes))]):
            if merged and merged[-1][0] + merged[-1][1] == lo:
                merged[-1] = (merged[-1][0], merged[-1][1] + size)
            elif size:
                merged.append((lo, size))
        self.free = merged


class _View:
    def __init__(self, owner, address, shape, typestr):
        self.owner = owner  # keeps the range while a tensor looks at it
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (address, False), "version": 3,
                                         "strides": None}


_session: _Session | None = None


def _open() -> _Session:
    global _session
    if _session is None:
        _session = _Session()
    return _session


class _Range:
    def __init__(self, session: _Session, nbytes: int):
        self.session, self.nbytes = session, nbytes
        self.at = session.take(nbytes)

    def __del__(self):
        self.session.give(self.at, self.nbytes)


class State:
    """A case's tensors in the arena (named views) and its call."""

    def __init__(self):
        self.session = _open()
        self.t: dict[str, torch.Tensor] = {}
        self.at: dict[str, int] = {}
        self.call = None     # () -> None: queues the pass
        self.outputs = None

    def room(self, name: str, shape, dtype) -> torch.Tensor:
        size = math.prod(shape) * torch.empty((), dtype=dtype).element_size()
        r = _Range(self.session, max(size, 256))
        self.at[name] = r.at
        self.t[name] = self.session.view(r, r.at, shape, dtype)
        return self.t[name]

    def put(self, name: str, x: torch.Tensor) -> int:
        self.room(name, x.shape, x.dtype).copy_(x)
        return self.at[name]


# ---- inputs, from the seed alone --------------------------------------------------


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed * 7919 + 12345)


def _normal(g, shape, sigma: float = 1.0, dtype=torch.float32) -> torch.Tensor:
    return torch.empty(shape, device="cuda", dtype=dtype).normal_(0.0, sigma, generator=g)


def _cache_rows(g, length: int, max_ctx: int, row: int):
    """K rows [max_ctx][row] and V^T [row][stride], zero past `length` as a
    reset session leaves them."""
    stride = lib().syn_hip_kv_ctx_stride(max_ctx)
    k = torch.zeros((max_ctx, row), device="cuda", dtype=torch.float16)
    vt = torch.zeros((row, stride), device="cuda", dtype=torch.float16)
    k[:length] = _normal(g, (length, row), dtype=torch.float16)
    vt[:, :length] = _normal(g, (row, length), dtype=torch.float16)
    return k, vt


def _attention_inputs(c, seed):
    g = _generator(seed)
    row, dt = c["kv_heads"] * c["head_dim"], torch.float16 if c["dtype"] == "f16" else torch.float32
    q = _normal(g, (c["n"], c["heads"] * c["head_dim"])).to(dt)
    k, v = _normal(g, (c["n"], row)).to(dt), _normal(g, (c["n"], row)).to(dt)
    return q, k, v, *_cache_rows(g, c["pos"], c["max_ctx"], row)


def _ragged_lengths(c) -> list[int]:
    # The same for every seed: the case's size does not hang on its values.
    r = np.random.default_rng(c["seqs"] * 1000003 + c["longest"])
    return [int(x) for x in r.integers(c["shortest"], c["longest"] + 1, c["seqs"])]


def _ragged_inputs(c, seed):
    g = _generator(seed)
    for length in _ragged_lengths(c):
        yield (length, _normal(g, (c["heads"] * c["head_dim"],)),
               *_cache_rows(g, length, length, c["kv_heads"] * c["head_dim"]))


def _image_inputs(c, seed):
    g = _generator(seed)
    dt = torch.float16 if c["dtype"] == "f16" else torch.float32
    shape = (c["batch"] * c["n"], c["heads"] * c["head_dim"])
    return [_normal(g, shape).to(dt) for _ in range(3)]


def _matmul_inputs(c, seed):
    g = _generator(seed)
    w = _normal(g, (c["rows"], c["cols"]), c["cols"] ** -0.5)
    return w, _normal(g, (c["n"], c["cols"])), _normal(g, (c["rows"],)) if c["bias"] else None


def _blocks(g, t: int, rows: int, cols: int) -> torch.Tensor:
    """Rows of quantized blocks: random quants, block scales that give weights
    a standard deviation near 0.03 and a mean near zero."""
    per, size = BLOCK[t]
    raw = torch.randint(0, 256, (rows, cols // per, size), device="cuda", dtype=torch.uint8, generator=g)

    def scale(at, sigma):
        d = torch.empty(raw.shape[:2], device="cuda").uniform_(0.7, 1.3, generator=g) * sigma
        raw[..., at:at + 2] = d.half().view(torch.uint8).view(*d.shape, 2)

    if t == Q4_K:
        scale(0, 9e-5)
        scale(2, 6.8e-4)
    elif t == Q6_K:
        raw[..., 192:208] = torch.randint(-32, 33, (*raw.shape[:2], 16), device="cuda", dtype=torch.int8,
                                          generator=g).view(torch.uint8)
        scale(208, 9e-5)
    else:
        scale(0, {Q8_0: 4e-4, Q4_0: 6.5e-3, Q5_0: 3.2e-3}[t])
    return raw.view(rows, -1)


def _matmul_q_inputs(c, seed):
    g = _generator(seed)
    w = _blocks(g, QTYPES[c["type"]], c["rows"], c["cols"])
    return w, _normal(g, (c["n"], c["cols"])), _normal(g, (c["rows"],)) if c["bias"] else None


# The feed-forward matrices' formats in a Q4_K_M file.
FFN = (("gate", Q4_K), ("up", Q4_K), ("down", Q6_K))


def _ffn_inputs(c, seed):
    g, e, f = _generator(seed), c["embd"], c["ff"]
    w = {name: _blocks(g, t, *((e, f) if name == "down" else (f, e))) for name, t in FFN}
    return w, 1.0 + _normal(g, (e,), 0.1), _normal(g, (c["n"], e))


class _ModelFile:
    """A GGUF file's metadata and tensors, held in memory."""

    def __init__(self, c, seed):
        g = _generator(seed)
        e, f, hd, v = c["embd"], c["ff"], c["head_dim"], c["vocab"]
        q_rows, kv_rows = c["heads"] * hd, c["kv_heads"] * hd
        self.metadata = {"general.architecture": "llama", "llama.attention.head_count": c["heads"],
                         "llama.attention.head_count_kv": c["kv_heads"], "llama.embedding_length": e,
                         "llama.attention.key_length": hd, "llama.context_length": c["max_ctx"],
                         "llama.block_count": c["layers"], "llama.feed_forward_length": f,
                         "llama.attention.layer_norm_rms_epsilon": RMS_EPS, "llama.rope.freq_base": ROPE_BASE}
        self.tensors, self.data = {}, {}

        def matrix(name, rows, cols):
            self.tensors[name] = TensorInfo(name, (cols, rows), F32, 0)
            self.data[name] = _normal(g, (rows, cols), cols ** -0.5)

        def norm(name):
            self.tensors[name] = TensorInfo(name, (e,), F32, 0)
            self.data[name] = 1.0 + _normal(g, (e,), 0.1)

        matrix("token_embd.weight", v, e)
        matrix("output.weight", v, e)
        norm("output_norm.weight")
        for l in range(c["layers"]):
            b = f"blk.{l}."
            norm(b + "attn_norm.weight")
            norm(b + "ffn_norm.weight")
            for name, rows, cols in (("attn_q", q_rows, e), ("attn_k", kv_rows, e), ("attn_v", kv_rows, e),
                                     ("attn_output", e, q_rows), ("ffn_gate", f, e), ("ffn_up", f, e),
                                     ("ffn_down", e, f)):
                matrix(f"{b}{name}.weight", rows, cols)
        row = c["kv_heads"] * hd
        self.cached = [_cache_rows(g, c["pos"], c["max_ctx"], row) for _ in range(c["layers"])]
        self.token = int(torch.randint(0, v, (1,), device="cuda", generator=g).item())

    def get(self, key, default=None):
        return self.metadata.get(key, default)

    def require(self, key):
        if key not in self.metadata:
            raise GGUFError(f"missing metadata {key}")
        return self.metadata[key]

    def tensor(self, name):
        return self.data[name].cpu().numpy()


# ---- prepare and run ----------------------------------------------------------------


def _rope_desc(s: State, c) -> AttnRopeDesc:
    s.room("q_out", (c["n"], c["heads"] * c["head_dim"]), torch.float32)
    return AttnRopeDesc(q_out_offset=s.at["q_out"], freq_factors_offset=NO_OFFSET,
                        theta_scale=rope_theta_scale(ROPE_BASE, c["head_dim"]), mode=0, freq_scale=1.0,
                        ext_factor=0.0, attn_factor=1.0)


def _prepare_attention(c, seed) -> State:
    s = State()
    q, k, v, kc, vt = _attention_inputs(c, seed)
    row = c["kv_heads"] * c["head_dim"]
    for name, x in (("q", q), ("k", k), ("v", v), ("kc", kc), ("vt", vt)):
        s.put(name, x)
    s.room("out", q.shape, torch.float32)
    scratch = int(lib().syn_hip_attention_scratch_bytes(c["heads"], c["kv_heads"], c["head_dim"], c["max_ctx"], c["n"]))
    s.room("scratch", (max(scratch, 256),), torch.uint8)
    dt = SYN_F16 if c["dtype"] == "f16" else SYN_F32
    d = AttnDesc(cache=KvDesc(k_offset=s.at["kc"], v_offset=s.at["vt"], max_ctx=c["max_ctx"],
                              n_kv_heads=c["kv_heads"], head_dim=c["head_dim"], ctx_stride=vt.shape[1]),
                 q_offset=s.at["q"], k_offset=s.at["k"], v_offset=s.at["v"], out_offset=s.at["out"],
                 scratch_offset=s.at["scratch"], scratch_bytes=scratch, n_heads=c["heads"], pos=c["pos"], n=c["n"],
                 scale=c["head_dim"] ** -0.5, q_dtype=dt, kv_dtype=dt)
    at = slice(c["pos"], c["pos"] + c["n"])
    s.outputs = {"out": s.t["out"], "k": s.t["kc"][at], "vt": s.t["vt"][:, at]}
    handle, L = s.session.arena.handle, lib()
    if c["rope"]:
        r = _rope_desc(s, c)
        s.call = lambda: check(L.syn_hip_attention_rope(handle, ctypes.byref(d), ctypes.byref(r)))
    else:
        s.call = lambda: check(L.syn_hip_attention(handle, ctypes.byref(d)))
    return s


def _prepare_ragged(c, seed) -> State:
    s = State()
    seqs = (SeqDesc * c["seqs"])()
    size = c["heads"] * c["head_dim"]
    out = s.room("out", (c["seqs"], size), torch.float32)
    for i, (length, q, kc, vt) in enumerate(_ragged_inputs(c, seed)):
        cache = KvDesc(k_offset=s.put(f"k{i}", kc), v_offset=s.put(f"v{i}", vt), max_ctx=length,
                       n_kv_heads=c["kv_heads"], head_dim=c["head_dim"], ctx_stride=vt.shape[1])
        seqs[i] = SeqDesc(cache=cache, q_offset=s.put(f"q{i}", q), out_offset=s.at["out"] + 4 * size * i,
                          pos=length - 1)
    need = int(lib().syn_hip_attend_batch_scratch_bytes(seqs, c["seqs"], c["heads"]))
    s.room("scratch", (max(need, 256),), torch.uint8)
    s.outputs = {"out": out}
    handle, L, scratch = s.session.arena.handle, lib(), s.at["scratch"]
    n, heads, scale = c["seqs"], c["heads"], c["head_dim"] ** -0.5
    s.call = lambda: check(L.syn_hip_attend_batch(handle, seqs, n, heads, scale, SYN_F32, scratch, need))
    return s


def _prepare_image(c, seed) -> State:
    s = State()
    q, k, v = (s.put(name, x) for name, x in zip("qkv", _image_inputs(c, seed)))
    out = s.room("out", s.t["q"].shape, torch.float32)
    d = SelfDesc(q_offset=q, k_offset=k, v_offset=v, out_offset=s.at["out"], n=c["n"], batch=c["batch"],
                 n_heads=c["heads"], head_dim=c["head_dim"], scale=c["head_dim"] ** -0.5,
                 in_dtype=SYN_F16 if c["dtype"] == "f16" else SYN_F32)
    s.outputs = {"out": out}
    handle, L = s.session.arena.handle, lib()
    s.call = lambda: check(L.syn_hip_self_attention(handle, ctypes.byref(d)))
    return s


def _prepare_product(c, seed) -> State:
    s = State()
    quantized = c["kind"] == "matmul_q"
    w, x, bias = (_matmul_q_inputs if quantized else _matmul_inputs)(c, seed)
    s.put("w", w)
    s.put("x", x)
    b = s.put("bias", bias) if bias is not None else NO_OFFSET
    s.outputs = {"out": s.room("out", (c["n"], c["rows"]), torch.float32)}
    handle, L = s.session.arena.handle, lib()
    if quantized:
        t = QTYPES[c["type"]]
        s.room("act", (int(L.syn_hip_matmul_q_act_bytes(t, c["n"], c["cols"])),), torch.uint8)
        d = MatmulQDesc(w_offset=s.at["w"], x_offset=s.at["x"], act_offset=s.at["act"], bias_offset=b,
                        out_offset=s.at["out"], w_type=t, n=c["n"], rows=c["rows"], cols=c["cols"])
        s.call = lambda: check(L.syn_hip_matmul_q(handle, ctypes.byref(d)))
    else:
        d = MatmulDesc(w_offset=s.at["w"], x_offset=s.at["x"], bias_offset=b, out_offset=s.at["out"], n=c["n"],
                       rows=c["rows"], cols=c["cols"])
        s.call = lambda: check(L.syn_hip_matmul(handle, ctypes.byref(d)))
    return s


def _prepare_ffn(c, seed) -> State:
    s = State()
    n, e, f = c["n"], c["embd"], c["ff"]
    w, gamma, x = _ffn_inputs(c, seed)
    for name, blocks in w.items():
        s.put(name, blocks)
    s.put("gamma", gamma)
    s.put("x", x)
    handle, L = s.session.arena.handle, lib()
    out = s.room("out", (n, e), torch.float32)
    for name, cols in (("h", e), ("g", f), ("u", f), ("d", e)):
        s.room(name, (n, cols), torch.float32)
    s.room("act", (max(int(L.syn_hip_matmul_q_act_bytes(t, n, cols)) for t, cols in ((Q4_K, e), (Q6_K, f))),),
           torch.uint8)
    at = s.at

    def product(name, x, y):
        rows, cols = (e, f) if name == "down" else (f, e)
        return MatmulQDesc(w_offset=at[name], x_offset=at[x], act_offset=at["act"], bias_offset=NO_OFFSET,
                           out_offset=at[y], w_type=dict(FFN)[name], n=n, rows=rows, cols=cols)

    def elementwise(op, a, b, y, count):
        return ElementwiseDesc(a_offset=at[a], b_offset=at[b], out_offset=at[y], count=count, op=op)

    norm = NormDesc(in_offset=at["x"], weight_offset=at["gamma"], out_offset=at["h"], n=n, size=e, eps=RMS_EPS)
    calls = [(L.syn_hip_rms_norm, norm), (L.syn_hip_matmul_q, product("gate", "h", "g")),
             (L.syn_hip_matmul_q, product("up", "h", "u")),
             (L.syn_hip_elementwise, elementwise(SYN_SILU_MUL, "g", "u", "g", n * f)),
             (L.syn_hip_matmul_q, product("down", "g", "d")),
             (L.syn_hip_elementwise, elementwise(SYN_ADD, "d", "x", "out", n * e))]
    calls = [(fn, d, ctypes.byref(d)) for fn, d in calls]

    def call():
        for fn, _, d in calls:
            check(fn(handle, d))

    s.call, s.outputs = call, {"out": out}
    return s


class ModelState:
    def __init__(self, c, seed):
        f = _ModelFile(c, seed)
        self.token, self.pos = f.token, c["pos"]
        self.model = DeviceLlama(f, c["max_ctx"])
        for cache, (k, vt) in zip(self.model.caches, f.cached):
            v = vt[:, :c["pos"]].T.contiguous()
            capi.upload_cache(self.model.arena, cache, k[:c["pos"]].cpu().numpy().view(np.uint16),
                              v.cpu().numpy().view(np.uint16))
        self.model.arena.sync()

    def __del__(self):
        if hasattr(self, "model") and lib is not None:  # (None when the interpreter ends)
            self.model.close()


_PREPARE = {"attention": _prepare_attention, "ragged": _prepare_ragged, "image": _prepare_image,
            "matmul": _prepare_product, "matmul_q": _prepare_product, "ffn": _prepare_ffn, "llama": ModelState}


def prepare(case, seed):
    torch.cuda.synchronize()  # ranges given back may still be read by queued passes
    s = _PREPARE[case["kind"]](case, seed)
    torch.cuda.synchronize()
    return s


def run(state):
    if isinstance(state, ModelState):
        return {"logits": state.model.step(state.token, state.pos)}
    state.call()
    return state.outputs


# ---- what a pass cannot do without -----------------------------------------------------


def work(case) -> dict:
    c, kind = case, case["kind"]
    if kind == "attention":
        row, size = c["kv_heads"] * c["head_dim"], c["heads"] * c["head_dim"]
        el = 2 if c["dtype"] == "f16" else 4
        return {"bytes": 4 * row * (c["pos"] + c["n"]) + 2 * c["n"] * row * el + c["n"] * size * (el + 4),
                "flops": 4 * size * (c["n"] * c["pos"] + c["n"] * (c["n"] + 1) // 2)}
    if kind == "ragged":
        row, size, total = c["kv_heads"] * c["head_dim"], c["heads"] * c["head_dim"], sum(_ragged_lengths(c))
        return {"bytes": 4 * row * total + 8 * size * c["seqs"], "flops": 4 * size * total}
    if kind == "image":
        size = c["heads"] * c["head_dim"]
        return {"bytes": c["batch"] * c["n"] * size * (10 if c["dtype"] == "f16" else 16),
                "flops": 4 * size * c["n"] * c["n"] * c["batch"]}
    if kind in ("matmul", "matmul_q"):
        per, size = BLOCK[QTYPES[c["type"]]] if kind == "matmul_q" else (1, 4)
        return {"bytes": c["rows"] * c["cols"] // per * size + 4 * c["n"] * (c["rows"] + c["cols"])
                + (4 * c["rows"] if c["bias"] else 0), "flops": 2 * c["n"] * c["rows"] * c["cols"]}
    if kind == "ffn":
        e, f = c["embd"], c["ff"]
        return {"bytes": 2 * e * f * 144 // 256 + e * f * 210 // 256 + 4 * e * (2 * c["n"] + 1),
                "flops": 6 * c["n"] * e * f}
    e, size, row = c["embd"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    weights = c["layers"] * e * (2 * size + 2 * row + 3 * c["ff"]) + c["vocab"] * e
    return {"bytes": 4 * (weights + c["layers"] * row * (c["pos"] + 1) + c["vocab"] + e * (2 * c["layers"] + 2)),
            "flops": 2 * weights + 4 * c["layers"] * size * (c["pos"] + 1)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("attention", "ragged") or (kind == "image" and case["dtype"] == "f16"):
        return {"rel": 8e-4}  # binary16 operands and probabilities: 1.3e-4 to 2.2e-4 off the 64-bit result
    if kind in ("image", "matmul", "matmul_q"):
        return {"rel": 4e-6}  # f32 sums in another order: 1e-7 to 6e-7, and up to 1e-6 for one chain over 4096
    if kind == "ffn":
        return {"rel": 4e-3}  # the down product's activations are rounded to int8: one of a row rounded the other way is 7e-4
    return {"rel": 1e-3}  # q and the cache in binary16 in each layer: 2.4e-4 off the 64-bit result


# ---- the same in 64 bits ------------------------------------------------------------------


def _attend64(q, k, vt, heads, kv_heads, scale, first):
    """q [n][heads*hd], k [L][kv_heads*hd], vt [kv_heads*hd][L], all double;
    query i sees keys 0..first+i (all of them if first is None)."""
    n, hd, group = q.shape[0], q.shape[1] // heads, heads // kv_heads
    out = torch.empty_like(q)
    if first is not None:
        hidden = torch.arange(k.shape[0], device=q.device)[None, :] > first + torch.arange(n, device=q.device)[:, None]
    for h in range(heads):
        a = slice(h * hd, (h + 1) * hd)
        b = slice(h // group * hd, (h // group + 1) * hd)
        s = (q[:, a] @ k[:, b].T.contiguous()) * scale
        if first is not None:
            s.masked_fill_(hidden, -math.inf)
        out[:, a] = torch.softmax(s, 1) @ vt[b].T.contiguous()
    return out


def _rope64(x, head_dim, pos):
    """Rows rotated at pos, pos+1, ... in interleaved pairs; the angle of pair
    i is pos times theta_scale, i times over, in f32."""
    n, size = x.shape
    angle = np.empty((n, head_dim // 2), np.float32)
    angle[:, 0] = np.arange(pos, pos + n, dtype=np.float32)
    for i in range(1, head_dim // 2):
        angle[:, i] = angle[:, i - 1] * np.float32(rope_theta_scale(ROPE_BASE, head_dim))
    angle = torch.from_numpy(angle).to(x.device).double()[:, None, :]
    pairs = x.double().view(n, size // head_dim, head_dim // 2, 2)
    a, b = pairs[..., 0], pairs[..., 1]
    cos, sin = angle.cos(), angle.sin()
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).reshape(n, size)


def _dequant64(t: int, raw: torch.Tensor, cols: int) -> torch.Tensor:
    """Rows of blocks to doubles, from the published block layouts."""
    per, size = BLOCK[t]
    b = raw.view(raw.shape[0], cols // per, size)
    half = lambda at: b[..., at:at + 2].contiguous().view(torch.float16).double()  # noqa: E731  [..., 1]
    if t == Q4_K:
        s = b[..., 4:16].int()
        sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | (s[..., :4] >> 6 << 4)], -1)
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | (s[..., 4:8] >> 6 << 4)], -1)
        q = b[..., 16:].view(*b.shape[:2], 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], -2).view(*b.shape[:2], 8, 32)
        w = (half(0) * sc).unsqueeze(-1) * q - (half(2) * mn).unsqueeze(-1)
    elif t == Q6_K:
        lo, hi = b[..., :128].view(*b.shape[:2], 2, 2, 32), b[..., 128:192].view(*b.shape[:2], 2, 1, 32)
        lo = torch.cat([lo & 15, lo >> 4], -2)
        hi = torch.cat([hi & 3, hi >> 2 & 3, hi >> 4 & 3, hi >> 6], -2)
        q = (lo | hi << 4).view(*b.shape[:2], 16, 16).to(torch.int8) - 32
        w = (half(208) * b[..., 192:208].contiguous().view(torch.int8)).unsqueeze(-1) * q
    elif t == Q8_0:
        w = half(0) * b[..., 2:].contiguous().view(torch.int8)
    else:
        q = b[..., size - 16:]
        q = torch.cat([q & 15, q >> 4], -1).to(torch.int8)
        if t == Q5_0:
            bits = b[..., 2:6].unsqueeze(-1) >> torch.arange(8, device=b.device, dtype=torch.uint8) & 1
            q |= (bits.view(*b.shape[:2], 32) << 4).to(torch.int8)
        w = half(0) * (q - (16 if t == Q5_0 else 8))
    return w.reshape(raw.shape[0], cols)


def _product64(t: int, raw: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """x (f32) quantized as ggml pairs it with the weights (Q8_K or Q8_0, in
    f32 as ggml does), then the product in doubles."""
    x = x.float().cpu()
    n, cols = x.shape
    if t in (Q4_K, Q6_K):
        b = x.view(n, cols // 256, 256)
        top = b.gather(-1, b.abs().argmax(-1, keepdim=True))
        inv = torch.where(top == 0, top, torch.full_like(top, -127.0) / top)
        q = torch.round(inv * b).clamp(max=127)
        d = torch.where(top == 0, top, 1.0 / inv)
    else:
        b = x.view(n, cols // 32, 32)
        d = b.abs().amax(-1, keepdim=True)
        d = d / torch.full_like(d, 127.0)
        y = b * torch.where(d == 0, d, 1.0 / d)
        q = torch.sign(y) * torch.floor(y.abs() + 0.5)
        d = d.half()
    a = (q.double() * d.double()).view(n, cols).cuda()
    out = torch.empty((n, raw.shape[0]), device="cuda", dtype=torch.float64)
    for r in range(0, raw.shape[0], 4096):
        out[:, r:r + 4096] = a @ _dequant64(t, raw[r:r + 4096], cols).T.contiguous()
    return out


def _rms_norm64(x, gamma):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + RMS_EPS) * gamma.double()


def _exact_step(c, seed):
    f = _ModelFile(c, seed)

    def norm(x, name):
        return _rms_norm64(x, f.data[name])

    def product(name, x):
        return x @ f.data[name].double().T.contiguous()

    x = f.data["token_embd.weight"][f.token:f.token + 1].double()
    for l in range(c["layers"]):
        b = f"blk.{l}."
        h = norm(x, b + "attn_norm.weight")
        q, k = (_rope64(product(f"{b}attn_{i}.weight", h), c["head_dim"], c["pos"]) for i in "qk")
        v = product(b + "attn_v.weight", h)
        kc, vt = f.cached[l]
        kc = torch.cat([kc[:c["pos"]].double(), k.half().double()])
        vt = torch.cat([vt[:, :c["pos"]].double(), v.half().double().T], 1)
        a = _attend64(q.half().double(), kc, vt, c["heads"], c["kv_heads"], c["head_dim"] ** -0.5, None)
        x = x + product(b + "attn_output.weight", a)
        h = norm(x, b + "ffn_norm.weight")
        g = product(b + "ffn_gate.weight", h)
        x = x + product(b + "ffn_down.weight", g * torch.sigmoid(g) * product(b + "ffn_up.weight", h))
    return {"logits": product("output.weight", norm(x, "output_norm.weight")).view(-1)}


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "attention":
        q, k, v, kc, vt = _attention_inputs(c, seed)
        if c["rope"]:
            q, k = (_rope64(x, c["head_dim"], c["pos"]) for x in (q, k))
        end = c["pos"] + c["n"]
        kc[c["pos"]:end] = k.half()
        vt[:, c["pos"]:end] = v.half().T
        out = _attend64(q.half().double(), kc[:end].double(), vt[:, :end].double(), c["heads"], c["kv_heads"],
                        c["head_dim"] ** -0.5, c["pos"])
        return {"out": out, "k": kc[c["pos"]:end].double(), "vt": vt[:, c["pos"]:end].double()}
    if kind == "ragged":
        return {"out": torch.cat([
            _attend64(q[None].half().double(), kc.double(), vt[:, :length].double(), c["heads"], c["kv_heads"],
                      c["head_dim"] ** -0.5, None) for length, q, kc, vt in _ragged_inputs(c, seed)])}
    if kind == "image":
        q, k, v = (x.double() for x in _image_inputs(c, seed))
        images = [slice(i * c["n"], (i + 1) * c["n"]) for i in range(c["batch"])]
        return {"out": torch.cat([_attend64(q[i], k[i], v[i].T.contiguous(), c["heads"], c["heads"],
                                            c["head_dim"] ** -0.5, None) for i in images])}
    if kind == "llama":
        return _exact_step(c, seed)
    if kind == "ffn":
        w, gamma, x = _ffn_inputs(c, seed)
        x = x.double()
        h = _rms_norm64(x, gamma)
        g, u = _product64(Q4_K, w["gate"], h), _product64(Q4_K, w["up"], h)
        return {"out": x + _product64(Q6_K, w["down"], g * torch.sigmoid(g) * u)}
    if kind == "matmul_q":
        w, x, bias = _matmul_q_inputs(c, seed)
        out = _product64(QTYPES[c["type"]], w, x)
    else:
        w, x, bias = _matmul_inputs(c, seed)
        out = x.double() @ w.double().T.contiguous()
    return {"out": out if bias is None else out + bias.double()}
