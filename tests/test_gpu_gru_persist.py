"""The persistent GRU recurrence (one launch per pass) against float64, at
the edges of its tiles: batches and hidden sizes that are no multiple of 16,
each padded width, one and several sample tiles per XCD; and its fault path."""
import numpy as np
import pytest
import torch

from cppnet_amd import _capi, ops

pytestmark = pytest.mark.gpu


def tensors(B, S, I, H, seed):
    gen = torch.Generator("cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    t = dict(X=r(I, S, B), Wi=r(3 * H, I) * (1 / (I + H)) ** 0.5, Wh=r(3 * H, H) * (1 / (2 * H)) ** 0.5, b=0.1 * r(3 * H),
             dY=r(H, S, B) / (B * S))
    e = lambda *s: torch.full(s, float("nan"), device="cuda")  # noqa: E731
    t.update(Y=e(H, S, B), gates=e(3 * H, S, B), rh=e(H, S, B), gWi=e(3 * H, I), gWh=e(3 * H, H), gb=e(3 * H),
             dX=e(I, S, B))
    return t


def run(t, B, S, I, H):
    ops.gru_forward(t["X"], t["Wi"], t["Wh"], t["b"], t["Y"], t["gates"], t["rh"], B, S, I, H)
    ops.gru_backward(t["X"], t["Wi"], t["Wh"], t["Y"], t["gates"], t["rh"], t["dY"], t["gWi"], t["gWh"], t["gb"],
                     t["dX"], B, S, I, H)
    torch.cuda.synchronize()
    return {k: t[k].clone() for k in ("Y", "gates", "rh", "gWi", "gWh", "gb", "dX")}


def exact(t, B, S, I, H):
    X = t["X"].double().permute(1, 2, 0).contiguous().requires_grad_()
    Wi, Wh, b = (t[k].double().T.contiguous().requires_grad_() if k != "b" else t[k].double().requires_grad_()
                 for k in ("Wi", "Wh", "b"))
    h, out, gates, rhs = torch.zeros(B, H, dtype=torch.float64, device="cuda"), [], [], []
    for s in range(S):
        x = X[s] @ Wi + b
        z, r = torch.sigmoid(x[:, :2 * H] + h @ Wh[:, :2 * H]).split(H, 1)
        n = torch.tanh(x[:, 2 * H:] + (r * h) @ Wh[:, 2 * H:])
        rhs.append(r * h)
        h = (1 - z) * n + z * h
        out.append(h)
        gates.append(torch.cat([z, r, n], 1))
    Y = torch.stack(out)
    g = torch.autograd.grad((Y * t["dY"].double().permute(1, 2, 0)).sum(), [X, Wi, Wh, b])
    st = lambda v: v.detach().permute(2, 0, 1)  # noqa: E731
    return dict(Y=st(Y), gates=st(torch.stack(gates)), rh=st(torch.stack(rhs)), gWi=g[1].T, gWh=g[2].T, gb=g[3],
                dX=st(g[0]))


CASES = [(1, 2, 3, 1), (3, 5, 4, 8), (16, 4, 8, 64), (17, 6, 5, 65), (40, 6, 12, 71), (33, 5, 7, 129), (130, 3, 9, 300),
         (5, 9, 16, 511), (200, 4, 8, 250), (128, 64, 128, 512)]


@pytest.mark.parametrize("B,S,I,H", CASES)
@pytest.mark.parametrize("path", ["persistent", "per-step"])
def test_gru_matches_float64(gpu, monkeypatch, B, S, I, H, path):
    print(f"[gru] B={B} S={S} I={I} H={H} {path}", flush=True)
    monkeypatch.setenv("CNHIP_RECURRENCE_PERSISTENT", "1" if path == "persistent" else "0")
    t = tensors(B, S, I, H, B + S + I + H)
    odd = torch.ones(3 * 256, device="cuda")  # the next grid starts from another XCD
    ops.relu_forward(odd, torch.empty_like(odd))
    got, want = run(t, B, S, I, H), exact(t, B, S, I, H)
    for k, w in want.items():
        # fp32 sums of at most max(B S, 2 H + I) terms (error 2^-24 sqrt(K)
        # of the result's size), carried through S steps whose Jacobian has
        # norm about 1: S terms of it, times 8.
        lim = 8 * 2.0 ** -24 * max(B * S, 2 * H + I) ** 0.5 * S ** 0.5 + 1e-6
        rel = float((got[k].double() - w).norm() / w.norm().clamp_min(1e-30))
        assert rel <= lim, f"{k}: {rel:.3g} > {lim:.3g}"
    again = run(t, B, S, I, H)
    for k in got:
        assert torch.equal(got[k], again[k]), f"{k} differs between two runs"


def test_gru_fault_is_reported_and_taken(gpu, monkeypatch):
    """A wait that gives up at once (a host-set limit; every block exits) is
    reported by the next recurrent call, after which calls work again."""
    B, S, I, H = 32, 6, 8, 64
    t = tensors(B, S, I, H, 9)
    want = run(t, B, S, I, H)
    monkeypatch.setenv("CNHIP_RECURRENCE_SPIN_LIMIT", "-1")
    ops.gru_forward(t["X"], t["Wi"], t["Wh"], t["b"], t["Y"], t["gates"], t["rh"], B, S, I, H)
    torch.cuda.synchronize()
    monkeypatch.delenv("CNHIP_RECURRENCE_SPIN_LIMIT")
    with pytest.raises(_capi.CnhipError, match="gave up waiting"):
        ops.gru_forward(t["X"], t["Wi"], t["Wh"], t["b"], t["Y"], t["gates"], t["rh"], B, S, I, H)
    got = run(t, B, S, I, H)
    for k in want:
        assert torch.equal(got[k], want[k]), k


def test_exchange_area_is_zeroed_whole(gpu):
    """The first recurrent launch in a stream's exchange buffer zeroes all of
    it, so that the larger exchange of a later launch in the same allocation
    (the backward's) never reads words that were not zeroed."""
    B, S, I, H = 32, 4, 8, 64
    t = tensors(B, S, I, H, 5)
    lib = _capi.load()

    def filled(fn):
        _capi.check(lib.cnhip_hbm_timing_enable(1))
        try:
            fn()
            return sum(r["total_bytes"] for r in _capi.hbm_timing_rows() if r["kernel"] == "fill_bytes_kernel")
        finally:
            _capi.check(lib.cnhip_hbm_timing_enable(0))

    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()):
        first = filled(lambda: ops.gru_forward(t["X"], t["Wi"], t["Wh"], t["b"], t["Y"], t["gates"], t["rh"], B, S, I, H))
        later = filled(lambda: ops.gru_backward(t["X"], t["Wi"], t["Wh"], t["Y"], t["gates"], t["rh"], t["dY"], t["gWi"],
                                                t["gWh"], t["gb"], t["dX"], B, S, I, H))
        torch.cuda.synchronize()
    need = 256 + 6 * B * H * 8  # the backward's six areas of 8-byte words
    assert later == 0, "the exchange buffer was grown or zeroed again: not the case that is tested"
    assert first >= need, f"zeroed {first} bytes, the backward polls up to {need}"
