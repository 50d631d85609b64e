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
import rxmet_lstm_abi as L
from test_lstm_gpu import _case, _config, _dev, _gpu_forward, _weights, _wrap

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


@pytest.mark.parametrize("case", [(3, 9, 4, 272), (3, 11, 4, 512)])
@pytest.mark.parametrize("gate_bits", [9, 10])
def test_tables_that_do_not_fit_beside_two_h_planes(cuda, case, gate_bits):
    """Two planes of h above H = 256, a 16-bit cell grid and 4096 gate-input codes together (four
    10-bit grids) ask for 164352 bytes of LDS with the 16-bit tanh table, more than a workgroup
    has (163840): the table stays in global memory.  Four 9-bit grids leave room for it."""
    T, B, I, H = case
    print(f"[lstm resident tables] {case} {gate_bits}", flush=True)
    c = _config("c4")
    for n in ("input", "forget", "cell", "output"):
        c.op[L.OP[f"{n}_gate_input"]].bits = gate_bits
    c.op[L.OP["output"]].bits = 10
    Wi, Wh, bi, bh = _weights(I, H, 21)
    g = np.random.default_rng(22)
    x = (g.random((T, B, I)) * 2 - 1).astype(np.float32)
    p = LO.finalize(LO.calibrate(Wi, Wh, bi, bh, x, None, None, mode=LO.ACT_CR), c, H, True)
    args = (Wi, Wh, bi, bh, x, None, None)
    exp = LO.forward_quant(*args[:5], p, None, None, mode=LO.ACT_LIBM_EXACT)
    for training in (True, False):
        out, hn, cn, _ = _gpu_forward(cuda, args, p, training)
        for n, t in (("output", out), ("h_n", hn), ("c_n", cn)):
            np.testing.assert_array_equal(t.cpu().numpy(), exp[n], err_msg=n)


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


@pytest.mark.parametrize("case", CASES)
def test_resident_backward_matches_oracle(cuda, case):
    """Gradients within 1e-5 of the oracle's 64-bit sums relative to each tensor's norm (32-bit
    sums over at most 4 H and T B terms: a few 1e-7 expected); the saved formats agree bit for
    bit."""
    T, B, I, H, cfg, state = case
    print(f"[lstm resident bwd] {case}", flush=True)
    args, _, p = _case(T, B, I, H, cfg, 11, True, state)
    exp_f = LO.forward_quant(*args[:5], p, args[5], args[6], mode=LO.ACT_LIBM_EXACT)
    g = np.random.default_rng(9)
    go, gh, gc = ((g.standard_normal(s) * 0.1).astype(np.float32)
                  for s in ((T, B, H), (B, H), (B, H)))
    exp = LO.backward_quant(exp_f, p, go, gh, gc)
    Wi, Wh, bi, bh, x, h0, c0 = (_dev(a, cuda) for a in args)
    prm, res = _wrap(p), []
    for codes in (False, True):
        saved = lstm_ops.forward_quant(x, Wi, Wh, bi, bh, h0, c0, prm, True, codes=codes)[3]
        res.append(lstm_ops.backward_quant(saved, prm, *(_dev(a, cuda) for a in (go, gh, gc))))
    torch.cuda.synchronize()
    for n, a, b in zip(("dx", "dW_ih", "dW_hh", "db_ih", "db_hh", "dh0", "dc0"), *res):
        assert torch.equal(a, b), n
        e = np.asarray(exp[n], np.float64)
        assert np.linalg.norm(a.cpu().numpy() - e) <= 1e-5 * (np.linalg.norm(e) + 1e-30), n


@pytest.mark.parametrize("case", [(3, 5, 7, 128, "c4", True), (4, 19, 9, 256, "default", True)])
def test_clustered_backward_matches_oracle(cuda, case, monkeypatch):
    """The clustered backward, which takes what the resident one declines and which a poll limit
    other than the default selects up to H = 256: both saved formats, to the bound above."""
    T, B, I, H, cfg, state = case
    print(f"[lstm clustered bwd] {case}", flush=True)
    args, _, p = _case(T, B, I, H, cfg, 18, True, state)
    exp_f = LO.forward_quant(*args[:5], p, args[5], args[6], mode=LO.ACT_LIBM_EXACT)
    go = (np.random.default_rng(19).standard_normal((T, B, H)) * 0.1).astype(np.float32)
    exp = LO.backward_quant(exp_f, p, go, None, None)
    Wi, Wh, bi, bh, x, h0, c0 = (_dev(a, cuda) for a in args)
    prm, res = _wrap(p), []
    monkeypatch.setenv("RXMET_TEST_SPIN_LIMIT", str((1 << 20) - 1))
    for codes in (False, True):
        saved = lstm_ops.forward_quant(x, Wi, Wh, bi, bh, h0, c0, prm, True, codes=codes)[3]
        res.append(lstm_ops.backward_quant(saved, prm, _dev(go, cuda), None, None))
    torch.cuda.synchronize()
    for n, a, b in zip(("dx", "dW_ih", "dW_hh", "db_ih", "db_hh", "dh0", "dc0"), *res):
        assert torch.equal(a, b), n
        e = np.asarray(exp[n], np.float64)
        assert np.linalg.norm(a.cpu().numpy() - e) <= 1e-5 * (np.linalg.norm(e) + 1e-30), n


@pytest.mark.parametrize("case", [(5, 3, 4, 128), (5, 5, 4, 208), (3, 515, 3, 256), (5, 9, 4, 384),
                                  (4, 19, 3, 512)])
@pytest.mark.parametrize("small", [1e-5, 1e-9, 1e-20])
def test_resident_backward_keeps_small_groups(cuda, case, small):
    """Groups of 64 units of two kinds that W_hh does not couple, the output gradients of the second
    kind `small` times the first's (a member of a cluster holds one group of each): its dh0, dc0 and
    its channels of dW_hh and db_hh are as close to the oracle's 64-bit sums as the first's, relative
    to their own norm (each term within 2^-30 of its group's largest, sums of at most 4 H and T B
    terms: a few 1e-7)."""
    T, B, I, H = case
    print(f"[lstm resident bwd small] {case} {small}", flush=True)
    args, _, p = _case(T, B, I, H, "default", 16, True, True)
    second = np.arange(H) // 64 % 2 == 1
    rows = np.tile(second, 4)
    args = list(args)
    args[1] = np.where(rows[:, None] == second[None, :], args[1], np.float32(0))
    exp_f = LO.forward_quant(*args[:5], p, args[5], args[6], mode=LO.ACT_LIBM_EXACT)
    g = np.random.default_rng(10)
    scale = np.where(second, np.float32(small), np.float32(1))
    go, gh, gc = ((g.standard_normal(s) * 0.1).astype(np.float32) * scale
                  for s in ((T, B, H), (B, H), (B, H)))
    exp = LO.backward_quant(exp_f, p, go, gh, gc)
    Wi, Wh, bi, bh, x, h0, c0 = (_dev(a, cuda) for a in args)
    prm = _wrap(p)
    saved = lstm_ops.forward_quant(x, Wi, Wh, bi, bh, h0, c0, prm, True, codes=True)[3]
    got = lstm_ops.backward_quant(saved, prm, *(_dev(a, cuda) for a in (go, gh, gc)))
    torch.cuda.synchronize()
    got = dict(zip(("dx", "dW_ih", "dW_hh", "db_ih", "db_hh", "dh0", "dc0"), got))
    for kind in (second, ~second):
        r = np.tile(kind, 4)
        for n, pick in (("dh0", np.s_[:, kind]), ("dc0", np.s_[:, kind]), ("dW_hh", r), ("db_hh", r)):
            e, a = (np.asarray(v, np.float64)[pick] for v in (exp[n], got[n].cpu().numpy()))
            err = np.linalg.norm(a - e) / (np.linalg.norm(e) + 1e-300)
            assert err <= 1e-5, (n, int(kind.sum()), err)


@pytest.mark.parametrize("H", [64, 512])
def test_resident_backward_keeps_nan_in_its_sequence(cuda, H):
    """A NaN and an infinity in two sequences' output gradients reach every unit's dh0 of those
    sequences, and leave the others' dx and dh0 as they are without them."""
    args, _, p = _case(4, 12, 3, H, "default", 14, True, True)
    Wi, Wh, bi, bh, x, h0, c0 = (_dev(a, cuda) for a in args)
    prm = _wrap(p)
    saved = lstm_ops.forward_quant(x, Wi, Wh, bi, bh, h0, c0, prm, True, codes=True)[3]
    res = []
    for bad in (False, True):
        go = torch.full((4, 12, H), 1e-2, device=cuda)
        if bad:
            go[1, 1, 7], go[2, 9, 9] = float("nan"), float("inf")
        res.append(lstm_ops.backward_quant(saved, prm, go, None, None))
    torch.cuda.synchronize()
    keep = [b for b in range(12) if b not in (1, 9)]
    for k in (0, 5):
        a, b = res[0][k], res[1][k]
        assert torch.equal(*((t[:, keep] if k == 0 else t[keep]) for t in (a, b)))
    assert torch.isnan(res[1][5][1]).all() and torch.isnan(res[1][5][9]).all()


def test_cluster_timeout_poisons_the_gradients(cuda, monkeypatch):
    args, _, p = _case(6, 24, 5, 384, "default", 15, True, False)
    Wi, Wh, bi, bh, x, h0, c0 = (_dev(a, cuda) for a in args)
    prm = _wrap(p)
    saved = lstm_ops.forward_quant(x, Wi, Wh, bi, bh, h0, c0, prm, True, codes=True)[3]
    go = torch.full((6, 24, 384), 1e-2, device=cuda)
    run = lambda: lstm_ops.backward_quant(saved, prm, go, None, None)
    ref = run()
    monkeypatch.setenv("RXMET_TEST_SPIN_LIMIT", "0")
    bad = run()
    monkeypatch.delenv("RXMET_TEST_SPIN_LIMIT")
    again = run()
    for r, b, a in zip(ref, bad, again):
        assert torch.isnan(b).all() and torch.equal(r, a)
