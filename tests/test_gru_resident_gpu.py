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


@pytest.mark.parametrize("case", CASES)
def test_resident_backward_matches_oracle_and_clustered(cuda, case, monkeypatch):
    """Gradients within 1e-5 of the oracle's 64-bit sums, relative to each tensor's norm (32-bit
    sums over at most 3 H and T B terms: a few 1e-7 expected), in both saved formats; the two
    formats agree bit for bit, and the clustered form to the same bound."""
    T, B, I, H, cfg = case
    print(f"[gru resident bwd] {case}", flush=True)
    args = _dirs(cuda, case)
    ref = gru_ops.forward_quant_float_storage_dirs(True, T, B, I, H, args)
    cod = gru_ops.forward_quant_codes_dirs(True, T, B, I, H, args)
    g = np.random.default_rng(5)
    dh = [torch.from_numpy((g.standard_normal((T + 1, B, H)) * 1e-2).astype(np.float32)).to(cuda)
          for _ in range(2)]
    pack = lambda outs: [(o[2], o[3], o[4], o[5], o[6], dh[d], o[0], o[1], args[d][6], o[7:])
                         for d, o in enumerate(outs)]
    f = gru_ops.backward_quant_float_storage_dirs(T, B, I, H, pack(ref))
    c = gru_ops.backward_quant_codes_dirs(T, B, I, H, pack(cod), torch_layout=False)
    monkeypatch.setenv("RXMET_TEST_SPIN_LIMIT", OTHER_LIMIT)
    k = gru_ops.backward_quant_codes_dirs(T, B, I, H, pack(cod), torch_layout=False)
    torch.cuda.synchronize()
    for d in range(2):
        W, R, bw, br, x, h0, qp = _case(T, B, I, H, cfg, 31 + d, d == 1)
        fwd = GO.forward_quant(W, R, bw, br, x, qp, h0=h0, training=True)
        exp = GO.backward_quant(fwd, dh[d].cpu().numpy(), qp)
        for n, a, b, q in zip(("dx", "dW", "dR", "dbw", "dbr", "dh0"), f[d], c[d], k[d]):
            assert torch.equal(a, b), (d, n)
            e = np.asarray(exp[n], np.float64)
            scale = np.linalg.norm(e) + 1e-30
            assert np.linalg.norm(b.cpu().numpy() - e) <= 1e-5 * scale, (d, n)
            assert np.linalg.norm(q.cpu().numpy() - e) <= 1e-5 * scale, (d, n)


@pytest.mark.parametrize("case", [(6, 3, 5, 64, "8b-sym"), (6, 5, 4, 128, "c3"), (6, 4, 5, 256, "c3"),
                                  (3, 515, 4, 256, "8b-sym")])
@pytest.mark.parametrize("small", [1e-5, 1e-9, 1e-20])
def test_resident_backward_keeps_small_gradients(cuda, case, small):
    """Two blocks of units that R does not couple, the output gradients of the second `small` times
    the first's: its dh0, its channels of dR and its bias gradients are as close to the 64-bit sums as
    the first's, relative to their own norm (32-bit sums over 3 H and T B terms: a few 1e-7)."""
    T, B, I, H, cfg = case
    print(f"[gru resident bwd small] {case} {small}", flush=True)
    W, R, bw, br, x, h0, qp = _case(T, B, I, H, cfg, 51, True)
    half = np.arange(H) >= H // 2
    mixed = np.arange(H) % 3 == 0  # every K chunk holds units of both blocks
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    for second in (half, mixed):
        cols = np.tile(second, 3)
        R2 = np.where(second[:, None] == cols[None, :], R, np.float32(0))
        dh = (np.random.default_rng(6).standard_normal((T + 1, B, H)) * 1e-2).astype(np.float32)
        dh[..., second] *= np.float32(small)
        fwd = GO.forward_quant(W, R2, bw, br, x, qp, h0=h0, training=True)
        exp = GO.backward_quant(fwd, dh, qp)
        args = [(t(W), t(R2), t(bw), t(br), t(x), t(h0), gru_ops.GRUQuantParams.from_struct(qp))]
        o = gru_ops.forward_quant_codes_dirs(True, T, B, I, H, args)[0]
        got = gru_ops.backward_quant_codes_dirs(
            T, B, I, H, [(o[2], o[3], o[4], o[5], o[6], t(dh), o[0], o[1], args[0][6], o[7:])],
            torch_layout=False)[0]
        torch.cuda.synchronize()
        got = dict(zip(("dx", "dW", "dR", "dbw", "dbr", "dh0"), (a.cpu().numpy() for a in got)))
        for block, c in ((second, cols), (~second, ~cols)):
            for n, sel in (("dh0", block), ("dR", c), ("dW", c), ("dbr", c)):
                e, a = (np.asarray(v[n], np.float64)[..., sel] for v in (exp, got))
                err = np.linalg.norm(a - e) / (np.linalg.norm(e) + 1e-300)
                assert err <= 1e-5, (n, int(block.sum()), err)


def test_resident_backward_keeps_nan_in_its_sequence(cuda):
    """A NaN and an infinity in two sequences' output gradients reach every unit's dh0 and the
    weight gradients, and leave the other sequences' dx and dh0 as they are without them."""
    case = (4, 5, 3, 64, "c3")
    T, B, I, H, _ = case
    args = _dirs(cuda, case)[:1]
    o = gru_ops.forward_quant_codes_dirs(True, T, B, I, H, args)[0]
    res = []
    for bad in (False, True):
        dh = torch.full((T + 1, B, H), 1e-2, device=cuda)
        if bad:
            dh[2, 1, 7], dh[3, 2, 9] = float("nan"), float("inf")
        res.append(gru_ops.backward_quant_codes_dirs(
            T, B, I, H, [(o[2], o[3], o[4], o[5], o[6], dh, o[0], o[1], args[0][6], o[7:])],
            torch_layout=False)[0])
    torch.cuda.synchronize()
    (dx0, _, _, _, _, h00), (dx1, dW1, _, _, _, h01) = res
    keep = [0, 3, 4]
    assert torch.equal(dx0[:, keep], dx1[:, keep]) and torch.equal(h00[keep], h01[keep])
    assert torch.isnan(h01[1]).all() and torch.isnan(h01[2]).all() and torch.isnan(dW1).any()
