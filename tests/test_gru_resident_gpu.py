"""The resident GRU recurrences (one workgroup per two or four sequences, R_q in registers; H up
to 256) at the edges of their ranges: one step and one sequence, a batch that leaves a workgroup
partly empty, unit counts around each K-step width, the four-sequence form, and every output
format.  Forward outputs equal the oracle bit for bit, and the clustered form (which a poll limit
other than the default selects) bit for bit."""
import numpy as np
import pytest
import torch

import gru_ops
import gru_oracle as GO
from test_gru_gpu import NAMES, _case, _gpu_forward

pytestmark = pytest.mark.gpu

# (T, B, I, H, config).  Two sequences per workgroup; from 515 sequences on, four
CASES = [(1, 1, 3, 16, "8b-sym"), (2, 3, 5, 64, "c3"), (5, 2, 4, 80, "c3"),
         (4, 5, 7, 128, "8b-asym"), (3, 7, 4, 144, "16b-act-pot2"), (5, 3, 9, 256, "c3"),
         (2, 515, 4, 32, "h-unsigned"), (3, 517, 3, 240, "c3"), (2, 514, 3, 176, "8b-sym")]
OTHER_LIMIT = str((1 << 20) - 1)


def _dirs(cuda, case):
    T, B, I, H, cfg = case
    args = []
    for d in range(2):
        W, R, bw, br, x, h0, qp = _case(T, B, I, H, cfg, 31 + d, d == 1)
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
        args.append((t(W), t(R), t(bw), t(br), t(x),
                     t(h0) if h0 is not None else torch.empty(0, device=cuda),
                     gru_ops.GRUQuantParams.from_struct(qp)))
    return args


@pytest.mark.parametrize("case", CASES)
def test_resident_forward_matches_oracle_and_clustered(cuda, case, monkeypatch):
    T, B, I, H, cfg = case
    print(f"[gru resident fwd] {case}", flush=True)
    W, R, bw, br, x, h0, qp = _case(T, B, I, H, cfg, 7, True)
    exp = GO.forward_quant(W, R, bw, br, x, qp, h0=h0, training=True)
    got = _gpu_forward(cuda, W, R, bw, br, x, h0, qp, True)
    for name, tensor in zip(NAMES, got):
        np.testing.assert_array_equal(tensor.cpu().numpy(), exp[name], err_msg=name)
    infer = _gpu_forward(cuda, W, R, bw, br, x, h0, qp, False)
    assert torch.equal(infer[0], got[0])
    # saved codes of both directions, against the clustered form
    args = _dirs(cuda, case)
    res = gru_ops.forward_quant_codes_dirs(True, T, B, I, H, args)
    monkeypatch.setenv("RXMET_TEST_SPIN_LIMIT", OTHER_LIMIT)
    clu = gru_ops.forward_quant_codes_dirs(True, T, B, I, H, args)
    torch.cuda.synchronize()
    for a, b in zip(res, clu):
        assert torch.equal(a[0], b[0])
        for k, f in ((1, 4), (len(a) - 1, 1)):
            u, v = (np.ascontiguousarray(gru_ops.unblock_codes(o[k].cpu().numpy(), B, H, f))
                    for o in (a, b))
            np.testing.assert_array_equal(u, v)
