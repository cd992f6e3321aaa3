"""MQ coding with deferred byte-outs against the oracle, where it can go wrong: launches of one
block per wave up to dozens (several lanes then code the same block), ragged lane groups, both
read widths, and contents that drive the code register to its edges: full-range noise (many
0xFF bytes, carries and stuffed bits), constants (blocks without a symbol), isolated extremes
(long runs of the most probable symbol, then shifts of many bits at once), checkerboards.
Every byte, length and distortion is exact."""
import numpy as np
import pytest

import libgail_amd as g
from t1_compare import compare_tier1

pytestmark = pytest.mark.gpu


def _content(kind, w, h, seed):
    rng = np.random.default_rng(seed)
    if kind == "noise":
        return rng.integers(0, 4096, size=(3, h, w), dtype=np.uint16)
    if kind == "constant":
        return np.full((3, h, w), 1000 + seed, np.uint16)
    if kind == "checker":
        y, x = np.mgrid[0:h, 0:w]
        return np.broadcast_to((((x + y) & 1) * 4095).astype(np.uint16), (3, h, w)).copy()
    a = np.full((3, h, w), 2048, np.uint16)  # isolated extremes
    n = max(1, w * h // 300)
    a[rng.integers(0, 3, n), rng.integers(0, h, n), rng.integers(0, w, n)] = rng.choice([0, 4095], n).astype(np.uint16)
    return a


@pytest.mark.parametrize("w,h,fourk,count", [(64, 64, 0, 1), (65, 67, 0, 2), (200, 131, 1, 5), (640, 500, 0, 5),
                                             (1000, 700, 1, 9)])
@pytest.mark.parametrize("mq_read", [16, 64])
def test_mq_edges(device, oracle, w, h, fourk, count, mq_read):
    layout = g.FrameLayout(w, h, fourk)
    kinds = ["noise", "extremes", "constant", "checker", "synth"]
    frames = []
    for i in range(count):
        kind = kinds[i % len(kinds)]
        frames.append(g.synth_frame(i, w, h) if kind == "synth" else _content(kind, w, h, i))
    slopes = [0.0 if i % 2 == 0 else 300.0 for i in range(count)]
    b = g.Batch(device, [layout] * count, [g.xyz_settings(layout)] * count, mq_read=mq_read)
    try:
        for i, f in enumerate(frames):
            b.upload(i, f)
            b.set_slope(i, slopes[i])
        print(f"[mq] {count} frames {w}x{h}, {count * layout.num_cblks} blocks", flush=True)
        outs, _ = b.encode()
    finally:
        b.close()
    for i, f in enumerate(frames):
        bad, lines = compare_tier1(outs[i], oracle.encode_frame_xyz(f, fourk, thr=slopes[i], threads=16))
        for ln in lines:
            print("[mq]", ln, flush=True)
        assert bad == 0, f"frame {i} ({kinds[i % len(kinds)]}): {bad} code-blocks differ"
