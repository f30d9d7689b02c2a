"""The persistent LSTM recurrence for batches and hidden sizes that are no
multiple of 16 against float64, at the edges of its tiles and each padded
width, with gradients of every step and of the last one only."""
import ctypes

import pytest
import torch

from cppnet_amd import _capi, ops

pytestmark = pytest.mark.gpu

CASES = [(1, 2, 3, 1), (3, 5, 4, 8), (17, 6, 64, 64), (16, 4, 5, 65), (40, 6, 12, 71), (33, 5, 7, 129), (130, 3, 9, 300),
         (5, 9, 16, 511), (100, 4, 128, 256), (120, 3, 8, 512),
         # multiples of 16 and tuned hidden sizes: two and more blocks a CU
         (1600, 3, 5, 64), (4000, 3, 5, 64), (2000, 3, 5, 128), (1600, 3, 64, 64)]


@pytest.mark.parametrize("B,S,I,H", CASES)
@pytest.mark.parametrize("last", [False, True])
@pytest.mark.parametrize("path", ["persistent", "per-step"])
def test_lstm_any_matches_float64(gpu, monkeypatch, B, S, I, H, last, path):
    print(f"[lstm] B={B} S={S} I={I} H={H} last={last} {path}", flush=True)
    monkeypatch.setenv("CNHIP_RECURRENCE_PERSISTENT", "1" if path == "persistent" else "0")
    gen = torch.Generator("cuda").manual_seed(B + S + I + H)
    r = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    X, Wi, Wh = r(I, S, B), r(4 * H, I) / (I + H) ** 0.5, r(4 * H, H) / (2 * H) ** 0.5
    b, dY = 0.1 * r(4 * H), (r(H, B) / B if last else r(H, S, B) / (B * S))
    e = lambda *s: torch.full(s, float("nan"), device="cuda")  # noqa: E731
    Y, gates, c, tc = e(H, S, B), e(4 * H, S, B), e(H, S, B), e(H, S, B)
    gWi, gWh, gb, dX = e(4 * H, I), e(4 * H, H), e(4 * H), e(I, S, B)

    def run():
        odd = torch.ones(3 * 256, device="cuda")  # the next grid starts from another XCD
        ops.relu_forward(odd, torch.empty_like(odd))
        ops.lstm_forward(X, Wi, Wh, b, Y, gates, c, tc, B, S, I, H)
        back = ops.lstm_backward_last if last else ops.lstm_backward
        back(X, Wi, Wh, Y, gates, c, tc, dY, gWi, gWh, gb, dX, B, S, I, H)
        torch.cuda.synchronize()
        return [t.clone() for t in (Y, gates, c, tc, gWi, gWh, gb, dX)]

    got = run()
    x = X.double().permute(1, 2, 0).contiguous().requires_grad_()
    wi, wh, bb = (t.double().T.contiguous().requires_grad_() if t.dim() == 2 else t.double().requires_grad_()
                  for t in (Wi, Wh, b))
    h = cc = torch.zeros(B, H, dtype=torch.float64, device="cuda")
    ys, gs, cs = [], [], []
    for s in range(S):
        i, f, g, o = (x[s] @ wi + bb + h @ wh).split(H, 1)
        i, f, g, o = torch.sigmoid(i), torch.sigmoid(f), torch.tanh(g), torch.sigmoid(o)
        cc = f * cc + i * g
        h = o * torch.tanh(cc)
        ys.append(h)
        gs.append(torch.cat([i, f, g, o], 1))
        cs.append(cc)
    y = torch.stack(ys)
    loss = (y[-1] * dY.double().T).sum() if last else (y * dY.double().permute(1, 2, 0)).sum()
    gx, gwi, gwh, gbb = torch.autograd.grad(loss, [x, wi, wh, bb])
    st = lambda v: v.detach().permute(2, 0, 1)  # noqa: E731
    cst = st(torch.stack(cs))
    want = [st(y), st(torch.stack(gs)), cst, cst.tanh(), gwi.T, gwh.T, gbb, st(gx)]
    # fp32 sums of at most max(B S, 4 H, H + I) terms (2^-24 sqrt(K) of the
    # result's size), carried through S steps: S terms of it, times 8
    lim = 8 * 2.0 ** -24 * max(B * S, 4 * H, H + I) ** 0.5 * S ** 0.5 + 1e-6
    for name, a, w in zip(("Y", "gates", "c", "tanh_c", "gWi", "gWh", "gb", "dX"), got, want):
        rel = float((a.double() - w).norm() / w.norm().clamp_min(1e-30))
        assert rel <= lim, f"{name}: {rel:.3g} > {lim:.3g}"
    for a, w in zip(got, run()):
        assert torch.equal(a, w), "two runs differ"


def recurrence_launches(fn):
    """MFMA launches of fn (its GEMMs and the recurrence's)."""
    lib = _capi.load()
    n, ms, fl = ctypes.c_int64(), ctypes.c_double(), ctypes.c_double()
    _capi.check(lib.cnhip_gemm_timing_enable(1))
    try:
        fn()
        _capi.check(lib.cnhip_gemm_timing_read(ctypes.byref(n), ctypes.byref(ms), ctypes.byref(fl)))
    finally:
        _capi.check(lib.cnhip_gemm_timing_enable(0))
    return n.value


# (B, S, H, whether forward / backward run in one launch).  Few steps are faster
# step by step; two sample tiles an XCD (B > 128) fit beside each other at H <=
# 256, where the backward needs less than half of a CU's LDS, and not at 300
@pytest.mark.parametrize("B,S,H,fwd,bwd", [(17, 2, 65, False, False), (17, 3, 65, True, False), (17, 6, 65, True, True),
                                           (100, 3, 256, False, False), (100, 16, 256, True, True), (5, 8, 511, True, True),
                                           (200, 6, 100, True, True), (250, 16, 200, True, True), (130, 16, 300, False, False),
                                           (4001, 6, 64, False, True), (4001, 10, 64, True, True)])
def test_lstm_any_path(gpu, monkeypatch, B, S, H, fwd, bwd):
    I = 8
    gen = torch.Generator("cuda").manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    X, Wi, Wh, b, dY = r(I, S, B), r(4 * H, I) / 4, r(4 * H, H) / (2 * H) ** 0.5, r(4 * H) / 10, r(H, S, B) / B
    e = lambda *s: torch.empty(*s, device="cuda")  # noqa: E731
    out = {}
    for path in ("1", "0"):
        monkeypatch.setenv("CNHIP_RECURRENCE_PERSISTENT", path)
        Y, gates, c, tc, gWi, gWh, gb, dX = (e(H, S, B), e(4 * H, S, B), e(H, S, B), e(H, S, B), e(4 * H, I), e(4 * H, H),
                                             e(4 * H), e(I, S, B))
        nf = recurrence_launches(lambda: ops.lstm_forward(X, Wi, Wh, b, Y, gates, c, tc, B, S, I, H))
        nb = recurrence_launches(
            lambda: ops.lstm_backward(X, Wi, Wh, Y, gates, c, tc, dY, gWi, gWh, gb, dX, B, S, I, H))
        out[path] = (nf, nb, Y, gates, c, gWi, gWh, gb, dX)
    (nf, nb, *got), (sf, sb, *want) = out["1"], out["0"]
    # one launch in place of S - 1; the rest of both passes is the same
    assert sf - nf == (S - 2 if fwd else 0), (sf, nf)
    assert sb - nb == (S - 2 if bwd else 0), (sb, nb)
    for g, w in zip(got, want):
        # two fp32 forms of sums of at most max(B S, 4 H) terms through S steps
        lim = 16 * 2.0 ** -24 * max(B * S, 4 * H) ** 0.5 * S ** 0.5 + 1e-6
        assert float((g - w).norm()) <= lim * float(w.norm()) + 1e-30
