"""Device rate control at sizes, contents and budgets that reach its edges, against the host rate
control on the oracle's Tier-1 result: frames of one packet per resolution and of ragged precincts,
headers with long runs of 0xFF, quads and bands without an included block, budgets that leave
almost nothing or everything, and component caps, which take more measurements than the first
launches make. Passes, thresholds, sizes and the number of measurements are equal; the distortion
left is the same sum in another order."""
import numpy as np
import pytest

import libgail_amd as g

pytestmark = pytest.mark.gpu


def _frame(kind, w, h):
    rng = np.random.default_rng(w * 7 + h)
    if kind == "noise":
        return rng.integers(0, 4096, (3, h, w), dtype=np.uint16)
    if kind == "sparse":  # flat, with a few textured squares in one component
        x = np.full((3, h, w), 1800, np.uint16)
        for _ in range(6):
            i, j = int(rng.integers(0, h - 20)), int(rng.integers(0, w - 20))
            x[1, i:i + 20, j:j + 20] = rng.integers(1200, 2600, (20, 20))
        return x
    return g.synth_frame(77, w, h)


@pytest.mark.parametrize("kind", ["synth", "noise", "sparse"])
@pytest.mark.parametrize("w,h,fourk", [(64, 64, 0), (97, 65, 1), (333, 479, 0), (1031, 260, 1)])
def test_search_matches_host(device, oracle, w, h, fourk, kind):
    layout = g.FrameLayout(w, h, fourk)
    x = _frame(kind, w, h)
    ref = oracle.encode_frame_xyz(x, fourk, threads=8)
    empty = g.empty_codestream_bytes(layout)
    full = empty + int(np.asarray(ref["data"]).size)
    budgets = [(int(empty + r * (full - empty)), int(c * full)) for r, c in
               ((2.0, 2.0), (0.7, 2.0), (0.2, 2.0), (0.01, 2.0), (0.8, 0.12), (2.0, 0.05), (0.3, 0.02))]
    settings = []
    for total, comp in budgets:
        s = g.with_rate_control(g.xyz_settings(layout))
        s.rcMaxTotal, s.rcMaxComp = total, max(comp, 1)
        settings.append(s)
    b = g.Batch(device, [layout] * len(budgets), settings)
    try:
        for i in range(len(budgets)):
            b.upload(i, x)
            b.set_slope(i, 0.0)
        outs, _ = b.encode()
        rates = [b.rate(i) for i in range(len(budgets))]
    finally:
        b.close()
    counts = []
    for (total, comp), out, rate in zip(budgets, outs, rates):
        want = g.rate_allocate(layout, ref, total, max(comp, 1))
        label = f"{w}x{h} {kind} {total}/{comp}"
        assert rate["iterations"] == want["iterations"], label
        assert list(rate["lambda"]) == list(want["lambdas"]), label
        assert rate["total"] == want["total"] and list(rate["comp"]) == want["comp"], label
        assert np.array_equal(np.asarray(out.info)[:, 1], want["passes"]), label
        # the same terms, all positive, in two orders of at most n additions
        assert rate["distortion"] == pytest.approx(want["distortion"], rel=64 * layout.num_cblks * 2.0 ** -52), label
        counts.append(want["iterations"])
    print(f"[search] {w}x{h} {kind}: {counts} measurements", flush=True)
