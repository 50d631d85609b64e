"""The resident LSTM recurrences (W_hh in registers: one workgroup up to H = 256, clusters of
workgroups of 128 units up to H = 512) at the edges of their ranges: one step and one sequence,
batches that leave a workgroup or a cluster partly empty, unit counts around each K-step width
and member boundary, the four-sequence form, 8- and 16-bit h, every table kind (gates and tanh in
LDS, the 16-bit tanh table, global tables) and every output format.  Forward outputs and every
saved tensor equal the oracle bit for bit."""
import numpy as np
import pytest
import torch

import lstm_ops
import lstm_oracle as LO
from test_lstm_gpu import _case, _dev, _gpu_forward, _wrap

pytestmark = pytest.mark.gpu


# (T, B, I, H, config, initial state)
CASES = [(1, 1, 3, 16, "default", False), (3, 3, 5, 64, "c4", True), (4, 2, 4, 80, "16b-act", True),
         (3, 5, 7, 128, "c4", False), (3, 7, 4, 144, "pot2-gate", True), (4, 3, 9, 256, "c4", True),
         (2, 517, 3, 48, "default", False), (2, 515, 3, 208, "c4", True),
         (2, 514, 3, 192, "16b-act", False), (3, 1, 4, 272, "default", True),
         (4, 13, 6, 384, "c4", True), (3, 19, 5, 400, "16b-act", False), (3, 37, 4, 512, "c4", True),
         (2, 600, 3, 512, "default", False)]


@pytest.mark.parametrize("case", CASES)
def test_resident_forward_matches_oracle(cuda, case):
    T, B, I, H, cfg, state = case
    print(f"[lstm resident fwd] {case}", flush=True)
    args, _, p = _case(T, B, I, H, cfg, 11, True, state)
    exp = LO.forward_quant(*args[:5], p, args[5], args[6], mode=LO.ACT_LIBM_EXACT)
    out, hn, cn, saved = _gpu_forward(cuda, args, p, True)
    for n, t in (("output", out), ("h_n", hn), ("c_n", cn)):
        np.testing.assert_array_equal(t.cpu().numpy(), exp[n], err_msg=n)
    for n, t in saved.items():
        if t is not None and exp.get(n) is not None:
            np.testing.assert_array_equal(t.cpu().numpy(), exp[n], err_msg=n)
    out2, hn2, cn2, _ = _gpu_forward(cuda, args, p, False)
    assert torch.equal(out, out2) and torch.equal(hn, hn2) and torch.equal(cn, cn2)
    # saved codes decode to the reference format
    Wi, Wh, bi, bh, x, h0, c0 = (_dev(a, cuda) for a in args)
    prm = _wrap(p)
    cod = lstm_ops.forward_quant(x, Wi, Wh, bi, bh, h0, c0, prm, True, codes=True)
    torch.cuda.synchronize()
    assert torch.equal(cod[0], out)
    dec = lstm_ops.decode_saved_codes(cod[3], prm, B)
    for n in lstm_ops.CODED_FIELDS:
        np.testing.assert_array_equal(saved[n].cpu().numpy(), dec[n].cpu().numpy(), err_msg=n)


def test_cluster_timeout_poisons_the_outputs(cuda, monkeypatch):
    """A poll limit of zero makes the members' waits give up: the outputs become NaN, and the
    next call with the normal limit is as before."""
    args, _, p = _case(6, 24, 5, 512, "default", 12, True, False)
    ref = _gpu_forward(cuda, args, p, False)
    monkeypatch.setenv("RXMET_TEST_SPIN_LIMIT", "0")
    bad = _gpu_forward(cuda, args, p, False)
    monkeypatch.delenv("RXMET_TEST_SPIN_LIMIT")
    again = _gpu_forward(cuda, args, p, False)
    for r, b, a in zip(ref[:3], bad[:3], again[:3]):
        assert torch.isnan(b).all() and torch.equal(r, a)
