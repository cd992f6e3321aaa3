"""A lane per code-block, which frames take when decoders keep the device busy with long codewords:
every word exact against the oracle, as with a wave per block. The rule counts a frame's bytes in
units of its longest block: blocks of nearly one length make it many of few bytes."""
import threading

import numpy as np
import pytest

import libgail_amd as g

pytestmark = pytest.mark.gpu


def _codes(rng, layout, longest, shortest, damaged):
    """Codewords of random bytes (0xFF and what may follow it among them) and a table of them."""
    data = rng.integers(0, 256, 30000, dtype=np.uint8)
    if damaged:
        at = np.flatnonzero(rng.random(len(data) - 1) < 0.15)
        data[at] = 0xFF
        data[at + 1] = rng.choice(np.array([0x00, 0x7F, 0x80, 0x8F, 0x90, 0xFF], np.uint8), len(at))
    n = layout.num_cblks
    codes = np.zeros(n, g.CBLK_CODE)
    codes["len"] = rng.integers(shortest, longest + 1, n)
    codes["offset"] = rng.integers(0, len(data) - longest, n)
    codes["nbps"] = rng.integers(1, 17, n)  # so that picture values stay within an int
    codes["passes"] = rng.integers(1, 50, n)
    return data, codes


def _units(codes, cus=256):
    return codes["len"].astype(np.int64).sum() / (int(codes["len"].max()) * cus)


@pytest.mark.parametrize("longest,shortest,lanes", [(24, 22, True), (1, 1, True), (24, 8, False)])
@pytest.mark.parametrize("damaged", [False, True])
def test_one_decoder_by_units(device, oracle, longest, shortest, lanes, damaged):
    """Alone, a frame of 78 units a compute unit has lanes and one of fewer has waves."""
    w, h, k = g.CONTAINERS["4k_full"]
    layout = g.FrameLayout(w, h, k)
    data, codes = _codes(np.random.default_rng(longest + damaged), layout, longest, shortest, damaged)
    assert (_units(codes) >= 78) == lanes
    want, want_wav = oracle.decode_frame(w, h, k, data, codes, 0, True, threads=16, want_wavelet=True)
    dec = g.Decoder(device, layout, 0, True)
    try:
        print(f"[lanes] {len(codes)} blocks of {shortest}-{longest} bytes, {_units(codes):.1f} units", flush=True)
        for _ in range(2):
            got, _, wav = dec.decode(data, codes, wavelet=True)
            assert np.array_equal(wav.view(np.uint32), want_wav.view(np.uint32))
            assert np.array_equal(got, want)
    finally:
        dec.close()


def test_decoders_at_once(device, oracle):
    """Six decoders on threads, ragged 2K frames and a table that grows from call to call: whether a
    call finds enough bytes under way for lanes or not, the pictures are the oracle's."""
    layout = g.FrameLayout(1999, 1077, 0)
    rng = np.random.default_rng(5)
    frames = []
    for longest, shortest in ((40, 30), (300, 1), (90, 90)):
        data, codes = _codes(rng, layout, longest, shortest, True)
        codes["passes"][rng.random(len(codes)) < 0.1] = 0
        frames.append((data, codes, oracle.decode_frame(1999, 1077, 0, data, codes, 0, False, threads=16)[0]))
    decs = [g.Decoder(device, layout, 0, False) for _ in range(6)]
    bad = []

    def work(j):
        try:
            for i in range(6):
                data, codes, want = frames[(i + j) % 3]
                got, _, _ = decs[j].decode(data, codes)
                if not np.array_equal(got, want):
                    bad.append((j, i))
        except Exception as e:  # noqa: BLE001
            bad.append((j, repr(e)))

    try:
        ts = [threading.Thread(target=work, args=(j,)) for j in range(6)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    finally:
        for d in decs:
            d.close()
    assert not bad, bad
