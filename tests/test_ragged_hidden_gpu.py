"""Hidden sizes that are no whole number of unit tiles: the modules widen and narrow their tensors
with one block copy per direction of a pass and keep the saved state for whole tiles; outputs,
gradients and the decoded saved state equal the reference-format route (saved state off, every
tensor padded around each call) bit for bit."""
import numpy as np
import pytest
import torch

import quant_gru as QG
import quant_lstm as QL
import rxmet_lib

pytestmark = pytest.mark.gpu


# (outer, rows src / dst, groups, cols src / dst): nothing to do, one element, tile edges, more
# elements than one grid covers (4096 workgroups of 256), rows and columns at once
@pytest.mark.parametrize("geo", [
    (3, (5, 16), 1, (7, 7)), (3, (16, 5), 1, (16, 5)), (1, (1, 1), 1, (1, 1)),
    (7, (1, 1), 2, (1, 16)), (7, (1, 1), 2, (17, 32)), (3000, (1, 1), 2, (250, 256)),
    (2, (33, 48), 3, (15, 16)), (0, (4, 4), 1, (4, 4))])
def test_block_copy(cuda, geo):
    outer, rows, groups, cols = geo
    src = torch.randn(outer, rows[0], groups, cols[0], device=cuda)
    dst = torch.full((outer, rows[1], groups, cols[1]), float("nan"), device=cuda)
    more = [torch.arange(k + 1, dtype=torch.float32, device=cuda) for k in range(20)]
    out = [torch.empty(18, device=cuda) for _ in more]  # more jobs than one launch holds
    rxmet_lib.block_copy([(src, dst, outer, rows, groups, cols)] + [
        (m, o, 1, (1, 1), 1, (m.numel(), 18)) for m, o in zip(more, out)], cuda)
    exp = np.zeros(dst.shape, np.float32)
    r, c = min(rows), min(cols)
    exp[:, :r, :, :c] = src.cpu().numpy()[:, :r, :, :c]
    np.testing.assert_array_equal(dst.cpu().numpy(), exp)
    for m, o in zip(more, out):
        e = np.zeros(18, np.float32)
        e[:m.numel()] = m.cpu().numpy()[:18]
        np.testing.assert_array_equal(o.cpu().numpy(), e)
    with pytest.raises(RuntimeError):  # a source of another size
        rxmet_lib.block_copy([(more[0], out[0], 1, (1, 1), 1, (2, 18))], cuda)


def _equal(a, b, name):
    assert (a is None) == (b is None), name
    if a is not None:
        assert a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b), name


@pytest.mark.parametrize("form", ["dense", "sum", "output_only", "no_state"])
@pytest.mark.parametrize("H,B,I,bidir,first", [
    (20, 7, 5, False, False), (100, 50, 23, True, True), (1, 1, 1, True, False),
    (250, 18, 9, False, True), (300, 20, 8, True, True)])
def test_gru_ragged_equals_reference_format(cuda, monkeypatch, H, B, I, bidir, first, form):
    torch.manual_seed(H)
    T, D = 5, 2 if bidir else 1
    m = QG.QuantGRU(I, H, batch_first=first, bidirectional=bidir)
    m.set_all_bitwidth(8, is_symmetric=False)
    m._bitwidth_config.h_ = 16
    m = m.to(cuda)
    x = torch.randn((B, T, I) if first else (T, B, I), device=cuda)
    h0 = None if form == "no_state" else torch.randn(D, B, H, device=cuda) * 0.3
    with m.calibration_context():
        m(x)
    m.use_quantization = True
    g = torch.randn(*x.shape[:2], D * H, device=cuda)
    res = []
    for codes in (True, False):
        monkeypatch.setattr(QG, "SAVE_STATE_AS_CODES", codes)
        m.train()
        m.zero_grad(set_to_none=True)
        xx = x.clone().requires_grad_()
        hh = None if h0 is None else h0.clone().requires_grad_()
        out, hn = m(xx, hh)
        if form == "sum":
            (out.sum() + hn.sum()).backward()
        elif form == "output_only":
            out.backward(g)
        else:
            torch.autograd.backward([out, hn], [g, hn.detach()])
        m.eval()
        with torch.no_grad():
            ev = m(x, h0)
        res.append([out.detach(), hn.detach(), *ev, xx.grad, None if hh is None else hh.grad,
                    *(p.grad for p in m.parameters())])
    names = ["output", "h_n", "eval output", "eval h_n", "dx", "dh0",
             *(n for n, _ in m.named_parameters())]
    for n, a, b in zip(names, *res):
        _equal(a, b, n)
    _equal(res[0][0], res[0][2], "training and inference output")


@pytest.mark.parametrize("form", ["dense", "output_only", "no_state", "no_bias"])
@pytest.mark.parametrize("H,B,I,bidir", [
    (20, 7, 5, False), (100, 50, 23, True), (1, 1, 1, False), (250, 18, 9, False),
    (300, 20, 8, False)])
def test_lstm_ragged_equals_reference_format(cuda, monkeypatch, H, B, I, bidir, form):
    torch.manual_seed(H)
    T, D = 5, 2 if bidir else 1
    m = QL.QuantLSTM(I, H, bidirectional=bidir, bias=form != "no_bias").to(cuda)
    x = torch.randn(T, B, I, device=cuda)
    hx = None if form == "no_state" else tuple(torch.randn(D, B, H, device=cuda) * 0.3
                                               for _ in range(2))
    m.calibrating = True
    m(x)
    m.calibrating = False
    m.finalize_calibration()
    m.use_quantization = True
    g = torch.randn(T, B, D * H, device=cuda)
    res, states = [], []
    for codes in (True, False):
        monkeypatch.setattr(QL, "SAVE_STATE_AS_CODES", codes)
        m.train()
        m.zero_grad(set_to_none=True)
        xx = x.clone().requires_grad_()
        hh = None if hx is None else tuple(h.clone().requires_grad_() for h in hx)
        out, (hn, cn) = m(xx, hh)
        if form == "output_only":
            out.backward(g)
        else:
            torch.autograd.backward([out, hn, cn], [g, hn.detach(), cn.detach()])
        st = m.qat_saved_state()
        states.append(st)
        m.eval()
        with torch.no_grad():
            eo, (eh, ec) = m(x, hx)
        res.append([out.detach(), hn.detach(), cn.detach(), eo, eh, ec, xx.grad,
                    *(() if hh is None else (h.grad for h in hh)),
                    *(p.grad for p in m.parameters())])
    for k, (a, b) in enumerate(zip(*res)):
        _equal(a, b, k)
    _equal(res[0][0], res[0][3], "training and inference output")

    def flat(d, pre=""):
        out = {}
        for k, v in d.items():
            out.update(flat(v, pre + k + ".") if isinstance(v, dict) else {pre + k: v})
        return out

    a, b = flat(states[0]), flat(states[1])
    assert a.keys() == b.keys()
    for k in a:
        if a[k] is None or b[k] is None:
            assert a[k] is b[k], k
        else:
            assert a[k].shape == b[k].shape and a[k].dtype == b[k].dtype, k
            assert torch.equal(a[k], b[k]), k
