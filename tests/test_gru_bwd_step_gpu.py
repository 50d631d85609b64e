"""The stepped GRU backward (one launch per step): gradients against the oracle, and bit for bit the
same from the saved codes as from the float format, for both tile shapes, one and two planes of R,
and sizes at the edges of the tiles, the 32-channel chunks and the batch."""
import numpy as np
import pytest
import torch

import gru_ops
import gru_oracle as GO
from test_gru_gpu import _case, _gpu_backward, _gpu_forward

pytestmark = pytest.mark.gpu
f32 = np.float32

# (T, B, I, H, config): 32 x 32 tiles, one row and one unit tile up to a remainder on either side;
# a gate's channels padded to 32 (H = 16, 48, 272); 12-bit R (two planes); 64 x 64 tiles (from 128
# of them) with B and H remainders, one and two planes
CASES = [(3, 1, 5, 16, "8b-sym"), (1, 32, 3, 32, "c3"), (3, 33, 5, 48, "c3"), (4, 64, 7, 64, "r12-pot2"),
         (3, 65, 8, 272, "8b-asym"), (2, 530, 4, 1024, "c3"), (2, 1030, 4, 480, "c3"),
         (2, 1030, 4, 480, "r12-pot2")]


@pytest.mark.parametrize("case", CASES)
def test_stepped_backward(cuda, case, monkeypatch):
    T, B, I, H, cfg = case
    print(f"[gru bwd step] {case}", flush=True)
    monkeypatch.setenv("RXMET_BWD_STEPPED", "1")
    W, R, bw, br, x, h0, qp = _case(T, B, I, H, cfg, 41, True)
    fwd = _gpu_forward(cuda, W, R, bw, br, x, h0, qp, True)
    g = np.random.default_rng(42)
    dh_new = (g.standard_normal((T + 1, B, H)) * 1e-2).astype(f32)
    dh_new[0] = 0
    got = _gpu_backward(cuda, fwd, dh_new, qp, T, B, I, H)
    names = ("dx", "dW", "dR", "dbw", "dbr", "dh0")
    # the oracle's cost; the last case is the only one of 64 x 64 tiles with two planes
    if B <= 600 or cfg == "r12-pot2":
        exp = GO.backward_quant(GO.forward_quant(W, R, bw, br, x, qp, h0=h0, training=True), dh_new, qp)
        for name, a in zip(names, got):
            e = exp[name]
            np.testing.assert_allclose(a, e, rtol=1e-4, atol=1e-5 * max(float(np.abs(e).max()), 1e-30),
                                       err_msg=name)
    # saved codes, dh read from the output gradient; two directions in one call
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    args = (t(W), t(R), t(bw), t(br), t(x), t(h0), gru_ops.GRUQuantParams.from_struct(qp))
    for ndir in (1, 2):
        cod = gru_ops.forward_quant_codes_dirs(True, T, B, I, H, [args] * ndir)
        gout = t(np.concatenate([dh_new[1:], dh_new[1:][::-1]][:ndir], axis=2))
        views, keep = gru_ops.grad_views(gout, None, T, B, H, False, ndir)
        res = gru_ops.backward_quant_codes_dirs(
            T, B, I, H, [(c[2], c[3], c[4], c[5], c[6], None, c[0], c[1], args[6], c[7:]) for c in cod],
            torch_layout=False, views=views)
        torch.cuda.synchronize()
        big = lambda n: n * -(-B // 64) * -(-H // 64) >= 128
        for d in range(ndir):
            for name, a, e in zip(names, res[d], got):
                a = a.cpu().numpy()
                if big(ndir) == big(1):  # the same tiles: the same sums in the same order
                    np.testing.assert_array_equal(a, e, err_msg=f"{ndir} {d} {name}")
                else:
                    np.testing.assert_allclose(a, e, rtol=1e-4, atol=1e-5 * np.abs(e).max(),
                                               err_msg=f"{ndir} {d} {name}")
