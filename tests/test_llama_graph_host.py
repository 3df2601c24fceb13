"""DeviceLlama's laid-out graph on the CPU: the calls a step makes, against a C
ABI that records them and launches nothing."""
from __future__ import annotations

import pathlib
import types

import numpy as np
import pytest

import synapse_amd.llama as llama
from synapse_amd import capi
from synapse_amd.gguf import F32, GGUFFile

DATA = pathlib.Path(__file__).resolve().parent / "golden" / "reference"


class _Recorder:
    """Entry points by name; each call's (name, descriptors) is kept."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def entry(handle, *args):
            self.calls.append((name, [getattr(a, "_obj", a) for a in args]))
            return 0
        return entry


def _model(monkeypatch, n_layer=2):
    abi = _Recorder()
    monkeypatch.setattr(llama, "lib", lambda: abi)
    m = llama.DeviceLlama.__new__(llama.DeviceLlama)
    c = m.config = llama.read_config(GGUFFile(DATA / "llama_tiny_f32.gguf"))
    assert c.n_layer >= n_layer
    m.max_ctx, m.tied, m.freq_factors = 8, False, None
    names = ["token_embd.weight", "output.weight", "output_norm.weight"]
    names += [f"blk.{l}.{s}.weight" for l in range(c.n_layer)
              for s in ("attn_norm", "attn_q", "attn_k", "attn_v", "attn_output", "ffn_norm", "ffn_gate", "ffn_up",
                        "ffn_down")]
    m.off = {name: 4096 * i for i, name in enumerate(names)}
    m.wtype = {name: (F32, c.n_embd) for name in names}
    m.act = {name: 1 << 20 for name in ("x", "h", "q", "qr", "k", "kr", "v", "attn", "o", "gate", "up", "down",
                                        "logits")}
    m.qact, m.scratch, m.theta_scale, m.scale = 0, (0, 0), 1.0, 1.0
    m.arena = types.SimpleNamespace(handle=None, download=lambda off, shape, dtype: np.zeros(shape, dtype))
    m.caches = _states(c, 0)
    m._lay_out_graph()
    return m, abi


def _states(c, base):
    return [capi.KvDesc(k_offset=base + 1024 * l, v_offset=base + 1024 * l + 512, max_ctx=8, n_kv_heads=c.n_head_kv,
                        head_dim=c.head_dim, ctx_stride=64) for l in range(c.n_layer)]


def _attended(abi):
    """(position, K offset) of each attention call, in order."""
    return [(d[0].pos, d[0].cache.k_offset) for name, d in abi.calls if name == "syn_hip_attention_rope"]


def test_steps_use_the_states_the_model_has(monkeypatch):
    """A program that decodes two sequences gives the model one's KV states,
    then the other's: each step appends to and attends those."""
    m, abi = _model(monkeypatch)
    first, second = m.caches, _states(m.config, 1 << 16)
    seen = []
    for pos, states in ((0, first), (0, second), (1, first), (1, second)):
        m.caches = states
        abi.calls.clear()
        # (the recorded descriptors are the graph's own: looked at before the next step)
        m.step(3, pos)
        seen.append(_attended(abi))
    want = lambda pos, states: [(pos, s.k_offset) for s in states]  # noqa: E731
    assert seen == [want(0, first), want(0, second), want(1, first), want(1, second)]
    m.caches = [first[0], *second[1:]]
    m.caches[0] = second[0]  # (one layer's alone)
    abi.calls.clear()
    m.step(3, 2)
    assert _attended(abi) == want(2, m.caches)


def test_a_step_needs_a_state_per_layer(monkeypatch):
    m, _ = _model(monkeypatch)
    m.caches = m.caches[:-1]
    with pytest.raises((ValueError, IndexError)):
        m.step(3, 0)
