"""The wave decoder of a code-block on codewords made to reach its edges, against the oracle: bytes
that are mostly 0xFF, 0x80-0x8F after it (added to the bits before them only when those are
used), markers in mid-codeword, runs of zeros; codewords of 0 to 700 bytes, so that some end in
the first decisions and some take several windows; 1 to 30 bit-planes; any number of passes;
blocks of every width and height at the frame's edges. Every word is exact."""
import json
import os

import numpy as np
import pytest

import libgail_amd as g

pytestmark = pytest.mark.gpu


def _bytes(rng, kind, n):
    if kind == "random":
        return rng.integers(0, 256, n, dtype=np.uint8)
    if kind == "stuffed":  # 0xFF followed by what may follow it, and by what overlaps it
        a = rng.integers(0, 256, n, dtype=np.uint8)
        at = np.flatnonzero(rng.random(n - 1) < 0.2)
        a[at] = 0xFF
        a[at + 1] = rng.choice(np.array([0x00, 0x7F, 0x80, 0x85, 0x8F], np.uint8), len(at))
        return a
    return rng.choice(np.array([0xFF, 0xFF, 0x80, 0x8F, 0x90, 0x00], np.uint8), n)


@pytest.mark.parametrize("kind", ["random", "stuffed", "markers"])
@pytest.mark.parametrize("w,h,fourk", [(64, 64, 0), (203, 131, 1), (479, 333, 0)])
def test_wave_decoder_edges(device, oracle, w, h, fourk, kind):
    layout = g.FrameLayout(w, h, fourk)
    rng = np.random.default_rng(w + len(kind))
    data = _bytes(rng, kind, 20000)
    n = layout.num_cblks
    codes = np.zeros(n, g.CBLK_CODE)
    codes["offset"] = rng.integers(0, len(data) - 700, n)
    codes["len"] = np.where(rng.random(n) < 0.3, rng.integers(0, 8, n), rng.integers(0, 700, n))
    codes["nbps"] = rng.integers(1, 31, n)
    codes["passes"] = np.minimum(rng.integers(1, 92, n), 255)
    dec = g.Decoder(device, layout, 0, True)
    try:
        print(f"[wave] {w}x{h} {kind}: {n} blocks", flush=True)
        got, _, wav = dec.decode(data, codes, wavelet=True)
    finally:
        dec.close()
    want, want_wav = oracle.decode_frame(w, h, fourk, data, codes, 0, True, want_wavelet=True)
    bad = int(np.count_nonzero(wav.view(np.uint32) != want_wav.view(np.uint32)))
    assert bad == 0, f"{bad} coefficients differ"
    assert np.array_equal(got, want)


def test_overlapping_byte_waits_for_its_shift(device, oracle):
    """Codewords with a byte of 0x80-0x8F after 0xFF that falls due in a refinement pass when its
    carry into the upper half of the code register would turn a decision, if it were added before
    the shift that needs it."""
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "t1_overlap_blocks.json")
    with open(path) as f:
        blocks = json.load(f)
    layout = g.FrameLayout(64, 64, 0)
    orient = np.array([layout.bands[b].orient for b in layout.cblks[:, 0]])
    dec = g.Decoder(device, layout, 0, True)
    try:
        for b in blocks:
            data = np.frombuffer(bytes.fromhex(b["data"]), np.uint8)
            at = np.flatnonzero((orient == b["orient"]) & (layout.cblks[:, 3] == b["w"]) & (layout.cblks[:, 4] == b["h"]))
            codes = np.zeros(layout.num_cblks, g.CBLK_CODE)
            codes[at[0]] = (0, len(data), b["passes"], b["nbps"], 0)
            got, _, wav = dec.decode(data, codes, wavelet=True)
            want, want_wav = oracle.decode_frame(64, 64, 0, data, codes, 0, True, want_wavelet=True)
            assert np.array_equal(wav.view(np.uint32), want_wav.view(np.uint32)), b["data"]
            assert np.array_equal(got, want), b["data"]
    finally:
        dec.close()
