"""A step's inputs and logits across the bus: logits to ordinary memory through the ring of page-locked pieces against one
copy to page-locked memory, bit for bit, for sizes around a piece and past the ring; inputs after a longer
prompt (the token rows' stride grows with it) against a fresh engine."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def engine(ti, streams, vocab=50000):
    e = ti.Engine(vocab, 256, 1, 4, 2, 64, 512, bits=8, max_seq=64, max_batch=streams)
    e.synth(3)
    return e


@pytest.mark.parametrize("streams,vocab", [(1, 50000), (8, 50000), (8, 32768), (24, 16384), (64, 50000), (61, 49984)])
def test_logits_by_pieces(ti, streams, vocab):
    e = engine(ti, streams, vocab)
    tok, pos = np.arange(1, streams + 1, dtype=np.int32), np.zeros(streams, np.int32)
    got = [e.step(tok, pos) for _ in range(2)]
    pin = torch.empty(streams, vocab, dtype=torch.float32, pin_memory=True)
    ti.check(ti.lib().ti_engine_step(e.h, streams, tok.ctypes.data_as(C.c_void_p), pos.ctypes.data_as(C.c_void_p),
                                     C.c_void_p(pin.data_ptr())))
    ref = pin.numpy()
    e.close()
    assert np.isfinite(ref).all() and np.abs(ref).max() > 0
    assert all((g == ref).all() for g in got)


def test_inputs_behind_a_longer_prompt(ti):
    out = []
    for first in (3, 40):
        e = engine(ti, 3, 4096)
        e.prefill(2, np.arange(first, dtype=np.int32))
        for s in range(3):
            e.prefill(s, np.arange(5 + s, dtype=np.int32) + 7)
        a = e.step(np.array([9, 8, 7], np.int32), np.array([5, 6, 7], np.int32))
        b = e.step(np.array([4, 5, 6], np.int32), np.array([6, 7, 8], np.int32))
        e.close()
        out.append((a, b))
    assert all((x == y).all() for x, y in zip(*out))
