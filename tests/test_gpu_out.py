"""Logits on their way to the host: through the engine's page-locked ring to ordinary memory, against the direct
copy that page-locked memory takes."""
import ctypes as C

import numpy as np
import pytest

import turboinfer_amd as T

pytestmark = pytest.mark.gpu


def host_memory(shape, dtype, fill):
    """Page-locked host memory (held until the process ends)."""
    p, n = C.c_void_p(), int(np.prod(shape))
    malloc = T.lib().hipHostMalloc   # (of the runtime that the library is linked with)
    malloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    assert malloc(C.byref(p), n * 4, 0) == 0
    a = np.frombuffer((C.c_char * (n * 4)).from_address(p.value), dtype).reshape(shape)
    a[...] = fill
    return a


def ptr(a):
    return a.ctypes.data_as(C.c_void_p)


# rows x vocab: less than a chunk, a chunk and a bit, several pieces, the ring of 8 MiB nearly filled and wrapped (8.4 and
# 17 MB, ends inside a piece and inside a chunk)
@pytest.mark.parametrize("n,vocab", [(1, 528), (1, 4112), (9, 32000), (64, 32000), (66, 32016), (128, 33328)])
def test_logits_ring(n, vocab):
    e = T.Engine(vocab, 128, 1, 2, 2, 64, 256, bits=16, max_seq=16, max_batch=n)
    e.synth(3, 0.1)
    tok = np.arange(n, dtype=np.int32) % vocab
    pinned = host_memory((n, vocab), np.float32, -1.0)
    for pos in range(2):   # (each slot of the ring, and its flags, a second time)
        p = np.full(n, pos, np.int32)
        got = e.step(tok, p)
        T.check(T.lib().ti_engine_step(e.h, n, ptr(tok), ptr(p), ptr(pinned)))
        assert np.array_equal(got, pinned)
        odd = np.zeros(n * vocab + 1, np.float32)[1:].reshape(n, vocab)   # (not on 16 bytes)
        T.check(T.lib().ti_engine_step(e.h, n, ptr(tok), ptr(p), ptr(odd)))
        assert np.array_equal(odd, got)
    e.close()


@pytest.mark.parametrize("n", [1, 3, 4, 5, 4095, 4096, 4099, 70001])
def test_rows_out_tails(n):
    T.init(0)
    src = np.random.default_rng(n).standard_normal(n + 8).astype(np.float32)
    dev, words = T.DeviceBuffer.from_array(src), T.DeviceBuffer.from_array(np.array([7, 9, 11], np.int32))
    dst, out = host_memory((n + 8,), np.float32, -1.0), host_memory((3,), np.int32, 0)
    flags = host_memory((n // 4096 + 2,), np.int32, 0)
    T.check(T.lib().ti_rows_out(C.c_void_p(dev.ptr), ptr(dst), C.c_int64(n), ptr(flags), C.c_uint32(5), C.c_void_p(words.ptr),
                                ptr(out), None))
    T.sync()
    chunks = (n + 4095) // 4096
    assert np.array_equal(dst[:n], src[:n]) and (dst[n:] == -1).all()
    assert flags.tolist() == [5] * chunks + [0] * (flags.size - chunks) and out.tolist() == [7, 9, 0]


@pytest.mark.parametrize("want", [[0], [4, 5, 6], [2, 9], [0, 1, 2, 3, 4, 5, 30, 31, 39], [15, 16, 17]])
def test_prefill_wanted_rows(want):
    """Rows in place (consecutive) and gathered, over chunks of 16 and more of them than the logits buffer holds."""
    e = T.Engine(528, 128, 2, 2, 2, 64, 256, bits=16, max_seq=64, max_batch=4)
    e.synth(5, 0.1)
    t = (np.arange(40) * 7 % 528).astype(np.int32)
    T.check(T.lib().ti_engine_set_prefill(e.h, 16))
    all_rows = np.concatenate([e.prefill(0, t, want=[i]) for i in range(40)])
    got = e.prefill(1, t, want=want)
    assert np.abs(got - all_rows[want]).max() <= 1e-3 * np.abs(all_rows).max()   # (head products of 1 .. 4 rows: fp32 sums)
    e.prefill(2, t, want=[])
    e.close()
