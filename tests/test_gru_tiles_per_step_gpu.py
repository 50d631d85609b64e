"""The clustered GRU forward whose clusters run several batch tiles in every step: every output
bit for bit the oracle's, staged (H >= 512) and not, one and two byte planes of h, one and two
directions, with a remainder in the last tile and an uneven share of tiles per cluster."""
import numpy as np
import pytest
import torch

import gru_ops
import gru_oracle as GO
from test_gru_gpu import NAMES, _case

pytestmark = pytest.mark.gpu


# 256 CUs hold 12 clusters of 20 (H = 320, two unit tiles each: 25 of 10), 16 of 16 (H = 512), 8 of
# 32 (H = 1024): more 16-row tiles than that
@pytest.mark.parametrize("T,B,I,H,cfg,ndir", [
    (3, 500, 3, 320, "8b-asym", 1), (3, 450, 3, 320, "16b-act-pot2", 2), (3, 530, 3, 512, "8b-sym", 1),
    (2, 300, 3, 512, "16b-act-pot2", 2), (2, 330, 2, 1024, "16b-act-pot2", 1)])
def test_forward_bit_exact(cuda, T, B, I, H, cfg, ndir):
    print(f"[gru tiles per step] {T} {B} {I} {H} {cfg} {ndir}", flush=True)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    args, exp = [], []
    for d in range(ndir):
        W, R, bw, br, x, h0, qp = _case(T, B, I, H, cfg, 51 + d, True)
        args.append((t(W), t(R), t(bw), t(br), t(x), t(h0), gru_ops.GRUQuantParams.from_struct(qp)))
        exp.append(GO.forward_quant(W, R, bw, br, x, qp, h0=h0, training=True))
    got = gru_ops.forward_quant_float_storage_dirs(True, T, B, I, H, args)
    torch.cuda.synchronize()
    for d in range(ndir):
        for name, a in zip(NAMES, got[d]):
            np.testing.assert_array_equal(a.cpu().numpy(), exp[d][name], err_msg=f"{d} {name}")
