"""Both directions of a calibration pass in one call (rxmet_gru_forward_calibrate_dirs): bit for
bit the single-direction entry point on the time-reversed input and on the other weight layout,
and the oracle's values, at the edges of the unit tiles, K chunks and cluster counts."""
import numpy as np
import pytest
import torch

import gru_ops
import gru_oracle as GO
from test_quant_gru_gpu import _close, _gpu_calibrate, _haste, _weights

pytestmark = pytest.mark.gpu
f32 = np.float32


# (T, B, I, H): one unit; a tile edge either side; one, two (an item per wave) and three chunks
# (chunks per wave); ragged sizes above 512 and at the end; more tiles than clusters (16-unit
# members of 1024 units fill the GPU four times over); beyond the clustered form
SHAPES = [(3, 2, 1, 1), (3, 17, 5, 15), (3, 16, 5, 17), (4, 33, 23, 100), (3, 18, 7, 129),
          (3, 5, 9, 250), (2, 20, 6, 520), (2, 40, 8, 1000), (2, 200, 8, 1024), (2, 530, 4, 256),
          (2, 3, 4, 1040)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("torch_layout", [False, True])
def test_directions_equal_single_calls_and_oracle(cuda, shape, torch_layout):
    T, B, I, H = shape
    print(f"[gru calib dirs] {shape} torch={torch_layout}", flush=True)
    g = np.random.default_rng(H)
    x = g.standard_normal((T, B, I)).astype(f32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    dirs, single = [], []
    for d in range(2):
        pt = _weights(I, H, 31 + d)
        h0 = (g.standard_normal((B, H)) * 0.5).astype(f32) if d else None
        ranges = gru_ops.GRUQuantizationRanges(H, device=cuda)
        w = pt if torch_layout else _haste(*pt)
        dirs.append((*map(t, w), t(x), t(h0) if d else None, ranges, bool(d)))
        xd = x[::-1] if d else x
        h, v, r = _gpu_calibrate(cuda, *_haste(*pt), xd, h0)
        single.append((h, v, r.stats.cpu().numpy()))
        he, ve, se = GO.forward_calibrate(*_haste(*pt), np.ascontiguousarray(xd), h0)
        _close(h, he, "h")
        _close(v, ve, "v")
        _close(single[-1][2], se, "stats")
    outs = gru_ops.forward_calibrate_dirs(True, T, B, I, H, dirs, torch_layout=torch_layout)
    for d, (h, v) in enumerate(outs):
        for n, a, e in zip(("h", "v", "stats"), (h, v, dirs[d][6].stats), single[d]):
            np.testing.assert_array_equal(a.cpu().numpy(), e, err_msg=f"direction {d}: {n}")


def test_torch_layout_ranges_skip_non_finite_weights(cuda):
    """The row-wise parameter ranges: non-finite entries skipped, a channel without a finite
    entry contributing 0, merged into the running ranges."""
    T, B, I, H = 2, 3, 70, 40
    pt = [a.copy() for a in _weights(I, H, 15)]
    pt[0][3, 5], pt[0][50, 69], pt[1][2, H - 1] = np.nan, np.inf, -np.inf
    pt[1][9] = np.inf
    pt[2][4], pt[3][11] = np.nan, -np.inf
    x = np.random.default_rng(16).standard_normal((T, B, I)).astype(f32)
    first = _weights(I, H, 17, amp=3.0)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    a, b = (gru_ops.GRUQuantizationRanges(H, device=cuda) for _ in range(2))
    for w in (first, pt):
        gru_ops.forward_calibrate_dirs(False, T, B, I, H, [(*map(t, w), t(x), None, a, False)],
                                       torch_layout=True)
        gru_ops.forward_calibrate_dirs(False, T, B, I, H,
                                       [(*map(t, _haste(*w)), t(x), None, b, False)])
    np.testing.assert_array_equal(a.stats.cpu().numpy(), b.stats.cpu().numpy())
    assert np.isfinite(a.stats.cpu().numpy()).all()
