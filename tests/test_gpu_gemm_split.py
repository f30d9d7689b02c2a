"""The GEMM shapes that run on the bf16 matrix cores with operands split in
three, and the fp32 tile beside them: tile edges, remainders of K, odd leading
dimensions and unaligned operands, every orientation and tile shape, against
float64; and what bf16 terms cannot hold (infinities, NaN, values near the ends of the fp32 range),
against IEEE fp32 semantics."""
import numpy as np
import pytest
import torch

from cppnet_amd import ops

pytestmark = pytest.mark.gpu


def operand(gen, trans, rows, k, pad, off):
    """X(r, k), k-contiguous when trans, as a flat tensor at an element offset."""
    ld = (k if trans else rows) + pad
    flat = torch.randn(ld * (rows if trans else k) + off, generator=gen, device="cuda")
    x = flat[off:]
    m = x.view(rows, ld)[:, :k] if trans else x.view(k, ld)[:, :rows].T
    return x, m, ld


# (M, N, K, batch): the fp32 64 x 64 tile with and without split-K, 128 x 128
# tiles whole and ragged, and 256 x 256 tiles whole, with edges, and with edges and a ragged K
# in 2, 8 and 16 splits (tests/test_gemm_plan.py asserts which runs where)
SHAPES = [(65, 63, 700, 1), (100, 515, 2000, 1), (257, 129, 33, 40), (1001, 515, 785, 1), (2000, 130, 70, 1),
          (8192, 512, 512, 1), (515, 517, 8191, 1), (256, 250, 500, 32), (4096, 4096, 2048, 1), (4090, 4087, 2051, 1),
          (1024, 4096, 4096, 1), (2050, 1561, 425, 1), (196, 2287, 3134, 1), (6731, 586, 2027, 1), (4057, 257, 5017, 1),
          (1361, 385, 8687, 1)]


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("M,N,K,batch", SHAPES)
def test_gemm_split_matches_float64(gpu, ta, tb, M, N, K, batch):
    gen = torch.Generator("cuda").manual_seed(M + 3 * N + 7 * K + ta + 2 * tb)
    if batch > 1:
        A = torch.randn(batch, *((M, K) if ta else (K, M)), generator=gen, device="cuda")
        B = torch.randn(batch, *((K, N) if tb else (N, K)), generator=gen, device="cuda")
        C = torch.empty(batch, N, M, device="cuda")
        ops.gemm_batched(bool(ta), bool(tb), M, N, K, A, K if ta else M, M * K, B, N if tb else K, N * K, C, M, M * N,
                         batch)
        a = (A if ta else A.transpose(1, 2)).double().contiguous()
        b = (B if tb else B.transpose(1, 2)).double().contiguous()
        got, want = C.transpose(1, 2).double(), torch.bmm(a, b)
        size = torch.bmm(a.square(), b.square())
    else:
        x, a, lda = operand(gen, ta, M, K, 1 if K < 2000 else 0, 1)
        y, b, ldb = operand(gen, not tb, N, K, 3 if K < 2000 else 0, 3)
        pad = torch.full(((M + 5) * N,), 7.0, device="cuda")
        ops.gemm(bool(ta), bool(tb), M, N, K, x, lda, y, ldb, pad, M + 5)
        C = pad.view(N, M + 5)
        assert bool((C[:, M:] == 7.0).all()), "wrote past the rows of C"
        a, b = a.double().contiguous(), b.T.double().contiguous()
        got, want, size = C[:, :M].T.double(), a @ b, a.square() @ b.square()
    # An fp32 sum of K zero-mean products: partial sums grow to sqrt(sum
    # (ab)^2), each rounding adds 2^-24 of one, so the error is ~ 2^-24
    # sqrt(K/2) sqrt(sum (ab)^2) rms; 8 of these covers 16 M outputs.
    lim = 8 * 2.0 ** -24 * (K / 2) ** 0.5 * size.sqrt()
    err = (got - want).abs()
    assert bool((err <= lim).all()), f"worst error / bound {float((err / lim).max()):.3g}"
    # and its mean keeps no drift: 6 standard errors of a mean of M N batch
    # such errors
    rms = float(want.square().mean().sqrt())
    assert abs(float((got - want).mean())) <= (6 / (M * N * batch) ** 0.5 + 0.02) * 2.0 ** -24 * (K / 2) ** 0.5 * rms


@pytest.mark.parametrize("M,N,K", [(64, 80, 700), (1001, 515, 785), (196, 2287, 3134), (2048, 2048, 512), (4096, 4096, 2048)])
def test_gemm_split_nonfinite_and_range_ends(gpu, M, N, K):
    gen = torch.Generator("cuda").manual_seed(K)
    A = torch.randn(K, M, generator=gen, device="cuda")  # A(m, k) at [k, m]
    B = torch.randn(N, K, generator=gen, device="cuda")
    A[3, 5] = float("inf")
    A[4, 7] = float("nan")
    A[9, 11] = 3.4e38       # its bf16 term is infinite
    B[:, 9] = B[:, 9].clamp(-0.5, 0.5)
    B[13, K - 1] = float("-inf")
    A[:, 17] = A[:, 17] * 1e-36
    A[:, 19] = A[:, 19] * 2.0 ** -128  # subnormal
    C = torch.empty(N, M, device="cuda")
    ops.gemm(False, False, M, N, K, A, M, B, K, C, M)
    want = (B.double() @ A.double())
    got = C.double()
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isinf(), want.isinf())
    assert bool((got[want.isinf()] == want[want.isinf()]).all())
    ok = want.isfinite()
    size = (B.double().square() @ A.double().square()).sqrt()
    # 2^-149: half of the smallest subnormal for each of K products
    lim = 8 * 2.0 ** -24 * (K / 2) ** 0.5 * size + K * 2.0 ** -149
    assert bool(((got - want).abs()[ok] <= lim[ok]).all()), float(((got - want).abs()[ok] / lim[ok]).max())


@pytest.mark.parametrize("scale", [(-116, 122), (-58, -58)])
@pytest.mark.parametrize("M,N,K", [(65, 80, 700), (300, 515, 785), (4096, 4096, 2048)])
def test_gemm_split_terms_that_flush(gpu, M, N, K, scale):
    """Ordinary outputs of values whose low bf16 terms fall below their grid, and
    outputs so small that products of low terms are subnormal."""
    gen = torch.Generator("cuda").manual_seed(M)
    A = torch.randn(K, M, generator=gen, device="cuda")
    B = torch.randn(N, K, generator=gen, device="cuda")
    sa, sb = 2.0 ** scale[0], 2.0 ** scale[1]
    if scale[1] > 0:
        A[K // 2] *= sa
        B[:, K // 2] *= sb
    else:
        A *= sa
        B *= sb
    C = torch.empty(N, M, device="cuda")
    ops.gemm(False, False, M, N, K, A, M, B, K, C, M)
    want = B.double() @ A.double()
    size = (B.double().square() @ A.double().square()).sqrt()
    assert bool(((C.double() - want).abs() <= 8 * 2.0 ** -24 * (K / 2) ** 0.5 * size + K * 2.0 ** -149).all())


def low_end(A, B, case):
    """A [K, M] (A(m, k) at [k, m]) and B [N, K] moved to the low end of the
    range: one k, every element, one row of A, or one row of A and one column
    of B, which alone are small enough for products to be subnormal."""
    kind, ea, eb = case
    sa, sb = 2.0 ** ea, 2.0 ** eb
    k = A.shape[0] // 2
    if kind == "k":
        A[k] *= sa
        B[:, k] *= sb
    elif kind == "all":
        A *= sa
        B *= sb
    elif kind == "row":
        A[:, 5] *= sa
        B *= sb
    else:
        A[:, 5] *= sa
        B[7] *= sb


@pytest.mark.parametrize("case", [("k", -116, 122), ("k", -136, 126), ("k", -147, 127), ("all", -58, -58), ("all", -66, -66),
                                  ("all", -100, -36), ("row", -140, 100), ("row", -120, 20), ("cross", -66, -66),
                                  ("cross", -70, -72)], ids=str)
@pytest.mark.parametrize("sign", ["mixed", "one"])
@pytest.mark.parametrize("M,N,K", [(65, 80, 700), (300, 515, 785), (196, 2287, 3134), (2048, 2048, 512),
                                   (4096, 4096, 2048)])
def test_gemm_split_low_end_of_the_range(gpu, M, N, K, case, sign):
    """Operands whose low bits, or all of them, lie below the bf16 terms' grid,
    and products that are subnormal."""
    gen = torch.Generator("cuda").manual_seed(M)
    A = torch.randn(K, M, generator=gen, device="cuda")
    B = torch.randn(N, K, generator=gen, device="cuda")
    if sign == "one":
        A.abs_()
        B.abs_()
    # no product of one k overflows: |a b| < 2^126
    A.clamp_(-4, 4)
    low_end(A, B.clamp_(-1, 1) if case[0] == "k" else B, case)
    C = torch.empty(N, M, device="cuda")
    ops.gemm(False, False, M, N, K, A, M, B, K, C, M)
    want = B.double() @ A.double()
    size = (B.double().square() @ A.double().square()).sqrt()
    # sums of one sign grow to sqrt(K) of that size; 2^-149: half of the
    # smallest subnormal for each of K products
    grow = 1 if sign == "mixed" else 0.5 * K ** 0.5
    lim = 8 * 2.0 ** -24 * (K / 2) ** 0.5 * size * grow + K * 2.0 ** -149
    err = (C.double() - want).abs()
    assert bool((err <= lim).all()), f"worst error / bound {float((err / lim).max()):.3g}"


# relative error measured with the fp32 MFMA tiles on these inputs:
# what the split form must not exceed (with 3% for the plan's split counts)
@pytest.mark.parametrize("B,I,O,fp32", [(1001, 785, 515, 1.435e-7), (292, 490, 2842, 1.142e-7), (3726, 224, 47, 1.444e-7)])
def test_gemm_split_weight_gradient_error(gpu, B, I, O, fp32):
    """X^T dY of a hidden layer (half of both operands zero), where an fp32
    product of zero adds no rounding: the 2-norm error against float64 stays
    within that of the fp32 MFMA."""
    gen = torch.Generator("cuda").manual_seed(B)
    r = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    X, dY = torch.relu(r(I, B)), torch.relu(r(O, B)) * r(O, B)
    gW = torch.empty(O, I, device="cuda")
    ops.gemm(True, False, I, O, B, X, B, dY, B, gW, I)
    want = dY.double() @ X.double().T.contiguous()
    err = float((gW.double() - want).norm() / want.norm())
    assert err <= 1.03 * fp32, f"{err:.3e} against {fp32:.3e} of the fp32 MFMA"


def timed(fn):
    """Milliseconds of one call, the best of 5 groups of 5."""
    fn()
    best = float("inf")
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(5):
            fn()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) / 5)
    return best


@pytest.mark.parametrize("kind,limit", [("tails", 1.4), ("dead", 4.0), ("nan", 4.0)])
@pytest.mark.parametrize("B,I,O", [(8192, 2048, 512), (4096, 4096, 4096)])
def test_gemm_split_values_at_the_low_end_are_not_slow(gpu, B, I, O, kind, limit):
    """Activations of which some lie below 2^-110 (GELU tails, the
    probabilities of a peaked softmax) cost next to nothing beside ordinary
    outputs; where every wave has to be formed again (an output that is zero
    beside such a value, or a NaN in every column) the product costs the fp32
    matrix rate on top, not memory's latency."""
    gen = torch.Generator("cuda").manual_seed(B)
    X = torch.randn(I, B, generator=gen, device="cuda")
    W = torch.randn(O, I, generator=gen, device="cuda") / I ** 0.5
    b = torch.zeros(O, device="cuda")
    Y = torch.empty(O, B, device="cuda")
    run = lambda: ops.linear_forward(X, W, b, Y, B, I, O)  # noqa: E731
    plain = timed(run)
    X[:, ::7] *= 2.0 ** -118 if kind != "nan" else 1.0
    X[::3, 1::7] *= 2.0 ** -118 if kind != "nan" else 1.0
    if kind == "tails":
        X[:, ::7] *= 2.0 ** 118
    if kind == "dead":
        W[::16] = 0
    if kind == "nan":
        X[0, ::16] = float("nan")
    slow = timed(run)
    want = W.double() @ X.double()
    ok = want.isfinite()
    assert torch.equal(Y.isfinite(), ok)
    size = (W.double().square() @ X.double().square()).sqrt()
    lim = 8 * 2.0 ** -24 * (I / 2) ** 0.5 * size + I * 2.0 ** -149
    assert bool(((Y.double() - want).abs()[ok] <= lim[ok]).all())
    print(f"[split] {B}x{I}x{O} {kind}: {plain:.4f} -> {slow:.4f} ms", flush=True)
    assert slow <= limit * plain, f"{plain:.4f} ms ordinary, {slow:.4f} ms with {kind}"


def test_linear_residual_in_place(gpu):
    """The skip branch added into its own buffer (Z is Y): a tile whose half
    sums would wait in C must not clobber it."""
    B, I, O = 4096, 2048, 4096
    gen = torch.Generator("cuda").manual_seed(5)
    X = torch.randn(I, B, generator=gen, device="cuda")
    W = torch.randn(O, I, generator=gen, device="cuda") / I ** 0.5
    b = torch.randn(O, generator=gen, device="cuda")
    Z = torch.randn(O, B, generator=gen, device="cuda")
    Y = torch.empty_like(Z)
    ops.linear_forward_act(X, W, b, Y, Z, B, I, O, "residual")
    want = W.double() @ X.double() + b.double()[:, None] + Z.double()
    assert float((Y.double() - want).abs().max()) < 1e-4
    ops.linear_forward_act(X, W, b, Z, Z, B, I, O, "residual")
    assert float((Z.double() - want).abs().max()) < 1e-4
