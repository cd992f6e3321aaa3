"""The wave decoder's arithmetic decoder (t1_wave_mq.h) compiled for the host, where its byte
handling can be checked by the tens of thousands of codewords and under sanitizers: against the
sequential decoder (t1_decode_block.h) decision by decision, and whole code-blocks against the
oracle. The column side of the wave decoder (t1_decode_wave.h) runs on the GPU only."""
import ctypes as C
import json
import os
import subprocess

import numpy as np
import pytest

from oracle_bind import _p, random_block, reference

HERE = os.path.dirname(os.path.abspath(__file__))
NATIVE = os.path.join(HERE, "native")


@pytest.fixture(scope="module")
def lib():
    path = os.path.join(NATIVE, "libwavemq_host.so")
    if not os.path.exists(path):
        pytest.skip("tests/native/libwavemq_host.so not built (make -C tests/native)")
    L = C.CDLL(path)
    L.host_wave_t1_words.restype = C.c_int
    L.host_wave_t1_words.argtypes = [C.c_void_p, C.c_uint32] + [C.c_int] * 5 + [C.c_void_p]
    L.host_wave_mq_fuzz.restype = C.c_int
    L.host_wave_mq_fuzz.argtypes = [C.c_uint32, C.c_int]
    return L


def _words(lib, data, w, h, orient, nbps, passes):
    buf = np.frombuffer(bytes(data) or b"\0", np.uint8).copy()
    out = np.zeros(w * h, np.uint32)
    assert lib.host_wave_t1_words(_p(buf), len(data), w, h, orient, nbps, passes, _p(out)) == 0
    return out.reshape(h, w)


def overlap_blocks():
    """Codewords (random bytes) with a byte of 0x80-0x8F after 0xFF that falls due in a refinement
    pass exactly when the upper half of the code register is Qe - 1, with no bit left below it:
    adding the byte before the shift that needs it turns an MPS into an LPS."""
    with open(os.path.join(HERE, "golden", "t1_overlap_blocks.json")) as f:
        return [dict(b, data=bytes.fromhex(b["data"])) for b in json.load(f)]


@pytest.mark.parametrize("i", range(9))
def test_overlapping_byte_waits_for_its_shift(oracle, lib, i):
    b = overlap_blocks()[i]
    args = (b["data"], b["w"], b["h"], b["orient"], b["nbps"], b["passes"])
    want = oracle.t1_decode_words(*args)
    ref = reference()
    if ref is not None:
        assert np.array_equal(ref.t1_decode_words(*args), want)
    assert np.array_equal(_words(lib, *args), want)


def test_decisions_match_the_sequential_decoder(lib):
    assert lib.host_wave_mq_fuzz(5, 60000) == 0


def test_blocks_match_the_oracle(oracle, lib):
    """Coded blocks at every truncation point, and damaged codewords."""
    rng = np.random.default_rng(17)
    for trial in range(60):
        c, w, h, orient = random_block(rng, trial)
        r = oracle.t1_encode(c, w, h, orient)
        for k in range(1, r["num_passes"] + 1):
            data = r["data"][:r["pass_len"][k - 1]]
            assert np.array_equal(_words(lib, data, w, h, orient, r["nbps"], k),
                                  oracle.t1_decode_words(data, w, h, orient, r["nbps"], k)), (w, h, orient, k)
    for trial in range(200):
        w, h, nbps = 1 + int(rng.integers(32)), 1 + int(rng.integers(32)), 1 + int(rng.integers(30))
        data = rng.integers(0, 256, int(rng.integers(0, 400)), dtype=np.uint8)
        data[rng.random(len(data)) < 0.3] = 0xFF
        passes = 1 + int(rng.integers(3 * nbps - 2))
        assert np.array_equal(_words(lib, bytes(data), w, h, trial % 4, nbps, passes),
                              oracle.t1_decode_words(bytes(data), w, h, trial % 4, nbps, passes)), trial


def test_under_sanitizers():
    exe = os.path.join(NATIVE, "stub", "asan", "wavemq_check")
    if not os.path.exists(exe):
        pytest.skip("tests/native/stub/asan/wavemq_check not built (make -C tests/native)")
    r = subprocess.run([exe, "10000"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
