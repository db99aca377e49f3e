"""Chunk buffers of multi-token calls are lent for the call: sessions that take
prompts one after another hold no more memory than one, and sessions prompted
from several threads at once get buffers of their own (the bits of a session
alone). Chunks of other sizes (CQ35_PREFILL_ROWS, as where memory is short)
change no bit."""
import gc
import threading

import numpy as np
import pytest
import torch

import cq35
import cq35.config as cc

pytestmark = pytest.mark.gpu


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def shape(name):
    base, _, layers = name.partition("@")
    cfg = dict(cc.preset(base))
    if layers:
        cfg.update(layers=int(layers), vocab=4096)
    return cfg


ALL = cq35.Session.MATRIX_PROJECTIONS | cq35.Session.MATRIX_EXPERTS | cq35.Session.MATRIX_ATTENTION


@pytest.mark.parametrize("name, components", [("qwen35-2b@4", 0), ("qwen36-35b-a3b@4", ALL)])
def test_sessions_share_the_buffers(name, components):
    cfg = shape(name)
    gc.collect()
    m = cq35.Model.synthetic(cfg, seed=3)
    prompt = np.random.default_rng(1).integers(0, cfg["vocab"], 40).tolist()
    sessions = [m.session(2100) for _ in range(5)]
    for s in sessions:
        s.set_matrix_prefill(components)
    print("prompt memory", name, flush=True)
    sessions[0].step_raw(prompt)
    one = free_bytes()
    for s in sessions[1:]:
        s.step_raw(prompt)
    assert one - free_bytes() < 4 << 20, "every session holds buffers of its own"
    del sessions, s
    gc.collect()
    m.close()


def test_threads_have_their_own():
    cfg = shape("qwen35-2b@4")
    m = cq35.Model.synthetic(cfg, seed=4)
    prompts = [np.random.default_rng(t).integers(0, cfg["vocab"], 150 + 97 * t).tolist() for t in range(4)]
    alone = []
    for p in prompts:
        s = m.session(600)
        alone.append((s.step_raw(p), s.export_state(0)))
    wrong = []

    def work(t):
        for _ in range(6):
            s = m.session(600)
            (logits, token), state = s.step_raw(prompts[t]), s.export_state(0)
            if token != alone[t][0][1] or not np.array_equal(logits, alone[t][0][0]) or not np.array_equal(state, alone[t][1]):
                wrong.append(t)

    print("prompts from four threads", flush=True)
    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("name, components, n", [("mini", 0, 300), ("mini-moe", 0, 300), ("mini-moe", ALL, 1061)])
def test_chunk_rows_change_no_bit(monkeypatch, name, components, n):
    cfg = shape(name)
    m = cq35.Model.synthetic(cfg, seed=5)
    prompt = np.random.default_rng(n).integers(0, cfg["vocab"], n).tolist()
    out = []
    for rows in (0, 16, 256, 336):
        monkeypatch.setenv("CQ35_PREFILL_ROWS", str(rows))
        s = m.session(n)
        s.set_matrix_prefill(components)
        print("chunk rows", name, rows, flush=True)
        out.append((s.step_raw(prompt)[0], s.export_state(0)))
    for logits, state in out[1:]:
        assert np.array_equal(logits, out[0][0]) and np.array_equal(state, out[0][1])
