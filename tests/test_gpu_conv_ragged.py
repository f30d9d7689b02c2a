"""Conv2D at batches that are no multiple of the weight gradient's k-tile or
of 4, and input gradients of strided convolutions (which list the taps that
reach each pixel), against float64."""
import pytest
import torch
import torch.nn.functional as F

from cppnet_amd import ops

pytestmark = pytest.mark.gpu

# (N, C, H, W, OC, KS, S, P): padded k-tiles of 16, 32 and 64 samples, whole
# and with 1 .. 3 samples left over; few samples (packed); strides 2 and 3
# with pixels that no tap reaches; OC not a multiple of 4 (a float4 of W' that
# spans two taps); more taps than a wave (9 x 9); tables beyond their limit
CASES = [(100, 17, 29, 27, 40, 5, 2, 2), (101, 3, 9, 8, 70, 3, 1, 1), (33, 5, 8, 7, 33, 3, 2, 1), (17, 40, 6, 6, 20, 3, 1, 1),
         (5, 6, 9, 9, 12, 3, 2, 0), (49, 2, 12, 11, 5, 1, 3, 0), (18, 3, 13, 13, 6, 9, 2, 4), (35, 4, 10, 10, 130, 2, 3, 1),
         (50, 33, 7, 7, 66, 3, 2, 1), (9, 8, 6, 6, 520, 3, 2, 1)]


@pytest.mark.parametrize("N,C,H,W,OC,KS,S,P", CASES)
@pytest.mark.parametrize("off", [0, 1])
def test_conv_ragged_matches_float64(gpu, N, C, H, W, OC, KS, S, P, off):
    print(f"[conv] N={N} C={C} {H}x{W} OC={OC} KS={KS} S={S} P={P} off={off}", flush=True)
    gen = torch.Generator("cuda").manual_seed(N + C + OC + KS)
    HO, WO = (H + 2 * P - KS) // S + 1, (W + 2 * P - KS) // S + 1

    def rnd(*shape):  # contiguous, `off` floats past a 16-byte boundary
        n = 1
        for v in shape:
            n *= v
        return torch.randn(n + off, generator=gen, device="cuda")[off:].view(shape)

    X, Wt, b, dY = rnd(W, H, C, N), rnd(KS, KS, C, OC), rnd(OC), rnd(WO, HO, OC, N)
    Y, gW, gb = torch.empty_like(dY), torch.empty_like(Wt), torch.empty_like(b)
    dX = torch.full_like(X, float("nan"))
    ops.conv2d_forward(X, Wt, b, Y, N, C, H, W, OC, KS, S, P)
    ops.conv2d_backward(X, Wt, dY, gW, gb, dX, N, C, H, W, OC, KS, S, P)
    lg = lambda t: t.double().permute(3, 2, 1, 0).contiguous()  # noqa: E731
    x, w, g = lg(X), lg(Wt), lg(dY)
    cols, flat = F.unfold(x, KS, padding=P, stride=S), g.reshape(N, OC, -1)
    wm = w.reshape(OC, -1)
    want = [(torch.matmul(wm, cols) + b.double()[None, :, None]).reshape(N, OC, HO, WO),
            torch.einsum("nop,nkp->ok", flat.cpu(), cols.cpu()).cuda().reshape(w.shape), flat.sum((0, 2)),
            F.fold(torch.matmul(wm.T.contiguous(), flat), (H, W), KS, padding=P, stride=S)]
    K = [C * KS * KS, N * HO * WO, N * HO * WO, OC * KS * KS]
    for name, got, v, k in zip(("Y", "gW", "gb", "dX"), (Y, gW, gb, dX), want, K):
        got = got.double() if name == "gb" else lg(got)
        # fp32 sum of k zero-mean products, as a share of the result: 2^-24
        # sqrt(k / 2) rms; times 8
        rel = float((got - v).norm() / v.norm())
        assert rel <= 8 * 2.0 ** -24 * max(k / 2, 1) ** 0.5, f"{name}: {rel:.3g}"
