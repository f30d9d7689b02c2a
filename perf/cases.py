"""The framework's performance cases: single layers, forward and backward, and
one small training session, at the sizes its configurations, tests and
benchmark use.

Everything is fp32 (the framework's only floating type).  Tensors follow the
framework's ColMajor layout: a [rows, cols] matrix is a torch tensor of shape
(cols, rows), so `t.T` is the logical matrix; [B, S, D] is (D, S, B) and
[N, C, H, W] is (W, H, C, N).

Backward passes read saved activations (ReLU outputs, max-pool argmax) from the
prepared inputs and not from the same pass's forward, so that a pre-activation
within rounding of zero cannot flip a whole gradient entry between two correct
implementations.
"""
import math

import numpy as np
import torch

from cppnet_amd import ops, trainer

F64 = torch.float64


# ------------------------------------------------------------------ helpers
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _xavier(g, fan_in, fan_out):
    """xavier-uniform [fan_in, fan_out], ColMajor."""
    lim = math.sqrt(6.0 / (fan_in + fan_out))
    return (torch.rand((fan_out, fan_in), generator=g, device="cuda") * 2 - 1) * lim


def _bias(g, n):
    return 0.1 * _randn(g, n)


def _empty(*shape):
    return torch.empty(shape, device="cuda")


def _onehot(g, batch, classes):
    """[batch, classes] ColMajor, uniform labels."""
    labels = torch.randint(0, classes, (batch,), generator=g, device="cuda")
    return (labels[None, :] == torch.arange(classes, device="cuda")[:, None]).float()


def _d(t):
    return t.to(F64)


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi], odd ones among them."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# ------------------------------------------------------------------- Linear
# Linear -> ReLU forward, and the backward whose input gradient carries the
# mask of the ReLU below: a hidden layer of an MLP.
def _linear_prepare(c, g):
    B, I, O = c["batch"], c["inputs"], c["outputs"]
    s = {"X": torch.relu(_randn(g, I, B)), "W": _xavier(g, I, O), "b": _bias(g, O),
         "dY": torch.relu(_randn(g, O, B)).mul_(_randn(g, O, B)).div_(B)}
    s.update(Y=_empty(O, B), gW=_empty(O, I), gb=_empty(O), dX=_empty(I, B) if c["input_grad"] else None)
    return s


def _linear_run(c, s):
    B, I, O = c["batch"], c["inputs"], c["outputs"]
    ops.linear_forward_act(s["X"], s["W"], s["b"], s["Y"], None, B, I, O, "relu")
    ops.linear_backward_act(s["X"], s["W"], s["dY"], s["gW"], s["gb"], s["dX"], s["X"], B, I, O, "relu")
    return [s["Y"], s["gW"], s["gb"], s["dX"]]


def _linear_exact(c, s):
    X, W, dY = _d(s["X"]), _d(s["W"]), _d(s["dY"])
    dX = (W.T @ dY) * (X > 0) if c["input_grad"] else None
    return [torch.relu(W @ X + _d(s["b"])[:, None]), dY @ X.T, dY.sum(1), dX]


def _linear_work(c):
    B, I, O, dx = c["batch"], c["inputs"], c["outputs"], c["input_grad"]
    return {"flops": 2 * B * I * O * (3 if dx else 2),
            "bytes": 4 * (B * I * (2 if dx else 1) + 2 * I * O + 2 * B * O + 2 * O)}


# ------------------------------------------------------------------ the head
# Classifier head: Linear, softmax cross-entropy forward and backward, Linear
# backward with the mask of the ReLU below.
def _head_prepare(c, g):
    B, I, O = c["batch"], c["inputs"], c["outputs"]
    return {"X": torch.relu(_randn(g, I, B)), "W": _xavier(g, I, O), "b": _bias(g, O), "T": _onehot(g, B, O),
            "Z": _empty(O, B), "P": _empty(O, B), "loss": _empty(1), "dZ": _empty(O, B), "gW": _empty(O, I),
            "gb": _empty(O), "dX": _empty(I, B)}


def _head_run(c, s):
    B, I, O = c["batch"], c["inputs"], c["outputs"]
    ops.linear_forward(s["X"], s["W"], s["b"], s["Z"], B, I, O)
    ops.softmax_ce_forward(s["Z"], s["T"], s["P"], s["loss"], B, O)
    ops.softmax_ce_backward(s["P"], s["T"], s["dZ"], B, O)
    ops.linear_backward_act(s["X"], s["W"], s["dZ"], s["gW"], s["gb"], s["dX"], s["X"], B, I, O, "relu")
    return [s[k] for k in ("Z", "P", "loss", "dZ", "gW", "gb", "dX")]


def _head_exact(c, s):
    X, W, T = _d(s["X"]), _d(s["W"]), _d(s["T"])
    Z = W @ X + _d(s["b"])[:, None]
    P = torch.softmax(Z, 0)
    loss = -(T * torch.log_softmax(Z, 0)).sum() / c["batch"]
    dZ = (P - T) / c["batch"]
    return [Z, P, loss.reshape(1), dZ, dZ @ X.T, dZ.sum(1), (W.T @ dZ) * (X > 0)]


def _head_work(c):
    B, I, O = c["batch"], c["inputs"], c["outputs"]
    return {"flops": 6 * B * I * O, "bytes": 4 * (2 * B * I + 2 * I * O + 4 * B * O + 2 * O)}


# ------------------------------------------------------------------- Conv2D
# Conv2D -> ReLU (-> MaxPool2D) and its backward; "first" is a model's first
# layer, whose input is data and takes no gradient.
def _conv_dims(c):
    N, C, H, W, OC, KS, S, P = (c[k] for k in ("batch", "channels", "height", "width", "filters", "kernel",
                                               "stride", "padding"))
    return N, C, H, W, OC, KS, S, P, (H + 2 * P - KS) // S + 1, (W + 2 * P - KS) // S + 1


def _logical(t):
    """(W, H, C, N) storage -> a float64 [N, C, H, W] tensor."""
    return _d(t).permute(3, 2, 1, 0).contiguous()


def _stored(t):
    return t.permute(3, 2, 1, 0).contiguous()


def _unfold(c, X):
    return torch.nn.functional.unfold(X, c["kernel"], padding=c["padding"], stride=c["stride"])


def _conv64(c, s):
    """float64 relu(conv) [N, OC, HO, WO]."""
    N, C, H, W, OC, KS, S, P, HO, WO = _conv_dims(c)
    cols = _unfold(c, _logical(s["X"]))
    K = _logical(s["W"]).reshape(OC, C * KS * KS)
    y = torch.matmul(K, cols).reshape(N, OC, HO, WO)
    return torch.relu(y + _d(s["b"])[None, :, None, None])


def _pool64(y, p):
    """Max and its first window index ph*p + pw over p x p windows."""
    HP, WP = y.shape[2] // p, y.shape[3] // p
    win = y[:, :, :HP * p, :WP * p].reshape(y.shape[0], y.shape[1], HP, p, WP, p)
    best = win[:, :, :, 0, :, 0].clone()
    at = torch.zeros_like(best, dtype=torch.int32)
    for k in range(1, p * p):
        v = win[:, :, :, k // p, :, k % p]
        m = v > best
        best = torch.where(m, v, best)
        at = torch.where(m, torch.full_like(at, k), at)
    return best, at


def _conv_prepare(c, g):
    N, C, H, W, OC, KS, S, P, HO, WO = _conv_dims(c)
    p = c["pool"]
    lim = math.sqrt(6.0 / (KS * KS * (C + OC)))
    s = {"X": torch.rand((W, H, C, N), generator=g, device="cuda"),
         "W": (torch.rand((KS, KS, C, OC), generator=g, device="cuda") * 2 - 1) * lim, "b": 0.05 * _randn(g, OC)}
    if p:
        HP, WP = HO // p, WO // p
        best, at = _pool64(_conv64(c, s), p)
        s.update(Pout=_stored(best.float()), at=_stored(at), dP=_randn(g, WP, HP, OC, N).div_(N),
                 Y=_empty(WP, HP, OC, N), idx=torch.empty((WP, HP, OC, N), dtype=torch.int32, device="cuda"))
        s["dC"] = _empty(WO, HO, OC, N)
    else:
        s.update(Y=_empty(WO, HO, OC, N), dC=torch.relu(_randn(g, WO, HO, OC, N)).div_(N))
    s.update(gW=_empty(KS, KS, C, OC), gb=_empty(OC), dX=None if c["first"] else _empty(W, H, C, N))
    return s


def _conv_run(c, s):
    N, C, H, W, OC, KS, S, P, HO, WO = _conv_dims(c)
    p = c["pool"]
    dims = (N, C, H, W, OC, KS, S, P)
    if not p:
        ops.conv2d_forward_relu(s["X"], s["W"], s["b"], s["Y"], *dims)
        ops.conv2d_backward(s["X"], s["W"], s["dC"], s["gW"], s["gb"], s["dX"], *dims)
        return [s["Y"], s["gW"], s["gb"], s["dX"]]
    ops.conv2d_forward_relu_maxpool(s["X"], s["W"], s["b"], s["Y"], s["idx"], *dims, p)
    if c["first"] and ops.conv2d_backward_maxpool_relu_fits(*dims, p):
        ops.conv2d_backward_maxpool_relu(s["X"], s["dP"], s["at"], s["Pout"], s["gW"], s["gb"], *dims, p)
    else:
        ops.maxpool2d_backward_relu_pooled(s["dP"], s["at"], s["Pout"], s["dC"], N, OC, HO, WO, p)
        ops.conv2d_backward(s["X"], s["W"], s["dC"], s["gW"], s["gb"], s["dX"], *dims)
    return [s["Y"], s["idx"], s["gW"], s["gb"], s["dX"]]


def _conv_exact(c, s):
    N, C, H, W, OC, KS, S, P, HO, WO = _conv_dims(c)
    p = c["pool"]
    y = _conv64(c, s)
    if p:
        best, at = _pool64(y, p)
        dP, sat = _logical(s["dP"]) * (_logical(s["Pout"]) > 0), s["at"].permute(3, 2, 1, 0)
        dC = torch.zeros((N, OC, HO, WO), dtype=F64, device="cuda")
        for k in range(p * p):
            dC[:, :, k // p:(HO // p) * p:p, k % p:(WO // p) * p:p] = dP * (sat == k)
        head = [_stored(best), _stored(at)]
    else:
        dC = _logical(s["dC"])
        head = [_stored(y)]
    cols = _unfold(c, _logical(s["X"]))                     # [N, C KS KS, HO WO]
    flat = dC.reshape(N, OC, HO * WO)
    gW = torch.zeros((OC, C * KS * KS), dtype=F64, device="cuda")
    for n in range(0, N, 16):
        gW += torch.bmm(flat[n:n + 16], cols[n:n + 16].transpose(1, 2).contiguous()).sum(0)
    dX = None
    if not c["first"]:
        K = _logical(s["W"]).reshape(OC, C * KS * KS)
        dX = _stored(torch.nn.functional.fold(torch.matmul(K.T.contiguous(), flat), (H, W), KS, padding=P, stride=S))
    return head + [_stored(gW.reshape(OC, C, KS, KS)), flat.sum((0, 2)), dX]


def _conv_work(c):
    N, C, H, W, OC, KS, S, P, HO, WO = _conv_dims(c)
    p = c["pool"]
    x, w = N * C * H * W, OC * C * KS * KS
    y = N * OC * (HO // p) * (WO // p) if p else N * OC * HO * WO
    saved = 3 * y if p else y  # pooled gradient, argmax, pooled output / the output's gradient
    return {"flops": 2 * N * HO * WO * w * (2 if c["first"] else 3),
            "bytes": 4 * (x * (1 if c["first"] else 2) + 2 * w + 2 * OC + y * (2 if p else 1) + saved)}


# ---------------------------------------------------------------- LSTM, GRU
# A recurrent layer over whole sequences, forward and backward through time.
# "last": the gradient reaches the last step's output only (sequence to one).
def _rnn_prepare(c, g):
    B, S, I, H = c["batch"], c["steps"], c["inputs"], c["hidden"]
    G = trainer.GATES[c["layer"]] * H
    li, lh = math.sqrt(6.0 / (I + H)), math.sqrt(6.0 / (2 * H))
    b = torch.zeros(G, device="cuda")
    if c["layer"] == "lstm":
        b[H:2 * H] = 1.0
    s = {"X": _randn(g, I, S, B), "Wi": (torch.rand((G, I), generator=g, device="cuda") * 2 - 1) * li,
         "Wh": (torch.rand((G, H), generator=g, device="cuda") * 2 - 1) * lh, "b": b + 0.01 * _randn(g, G),
         "dY": _randn(g, H, B).div_(B) if c["last"] else _randn(g, H, S, B).div_(B * S)}
    s.update(Y=_empty(H, S, B), gates=_empty(G, S, B), gWi=_empty(G, I), gWh=_empty(G, H), gb=_empty(G),
             dX=_empty(I, S, B) if c["input_grad"] else None)
    if c["layer"] == "lstm":
        s.update(c=_empty(H, S, B), tc=_empty(H, S, B))
    else:
        s.update(rh=_empty(H, S, B))
    return s


def _rnn_run(c, s):
    d = (c["batch"], c["steps"], c["inputs"], c["hidden"])
    if c["layer"] == "lstm":
        ops.lstm_forward(s["X"], s["Wi"], s["Wh"], s["b"], s["Y"], s["gates"], s["c"], s["tc"], *d)
        back = ops.lstm_backward_last if c["last"] else ops.lstm_backward
        back(s["X"], s["Wi"], s["Wh"], s["Y"], s["gates"], s["c"], s["tc"], s["dY"], s["gWi"], s["gWh"], s["gb"],
             s["dX"], *d)
    else:
        ops.gru_forward(s["X"], s["Wi"], s["Wh"], s["b"], s["Y"], s["gates"], s["rh"], *d)
        ops.gru_backward(s["X"], s["Wi"], s["Wh"], s["Y"], s["gates"], s["rh"], s["dY"], s["gWi"], s["gWh"], s["gb"],
                         s["dX"], *d)
    return [s["Y"], s["gWi"], s["gWh"], s["gb"], s["dX"]]


def _rnn_exact(c, s):
    H, S = c["hidden"], c["steps"]
    X = _d(s["X"]).permute(1, 2, 0).contiguous().requires_grad_()          # [S, B, I]
    Wi, Wh, b = (_d(s[k]).T.contiguous().requires_grad_() if k != "b" else _d(s[k]).requires_grad_()
                 for k in ("Wi", "Wh", "b"))
    h = torch.zeros((c["batch"], H), dtype=F64, device="cuda")
    cell, out = h, []
    for t in range(S):
        xi = X[t] @ Wi + b
        if c["layer"] == "lstm":
            i, f, z, o = (xi + h @ Wh).split(H, 1)
            cell = torch.sigmoid(f) * cell + torch.sigmoid(i) * torch.tanh(z)
            h = torch.sigmoid(o) * torch.tanh(cell)
        else:
            z, r = torch.sigmoid(xi[:, :2 * H] + h @ Wh[:, :2 * H]).split(H, 1)
            n = torch.tanh(xi[:, 2 * H:] + (r * h) @ Wh[:, 2 * H:])
            h = (1 - z) * n + z * h
        out.append(h)
    Y = torch.stack(out)                                                   # [S, B, H]
    dY = _d(s["dY"])
    if c["last"]:
        loss = (Y[-1] * dY.T).sum()
    else:
        loss = (Y * dY.permute(1, 2, 0)).sum()
    gX, gWi, gWh, gb = torch.autograd.grad(loss, [X, Wi, Wh, b])
    st = lambda t: t.detach().permute(2, 0, 1).contiguous()  # noqa: E731
    return [st(Y), gWi.T.contiguous(), gWh.T.contiguous(), gb, st(gX) if c["input_grad"] else None]


def _rnn_work(c):
    B, S, I, H = c["batch"], c["steps"], c["inputs"], c["hidden"]
    G = trainer.GATES[c["layer"]] * H
    x, y = B * S * I, B * S * H
    return {"flops": 2 * B * S * G * ((3 if c["input_grad"] else 2) * I + 3 * H),
            "bytes": 4 * (x * (2 if c["input_grad"] else 1) + 2 * y + 2 * G * (I + H + 1))}


# ---------------------------------------------------------------- attention
# Self-attention with its skip connection, forward and backward, on sequences
# whose rows are grouped by sample (as the encoder keeps them).
def _mha_prepare(c, g):
    B, S, D = c["batch"], c["steps"], c["dim"]
    s = {"x": _randn(g, D, B * S), "W": torch.stack([_xavier(g, D, D) for _ in range(4)]),
         "dY": _randn(g, D, B * S).div_(B * S), "out": _empty(D, B * S), "gW": _empty(4, D, D), "dX": _empty(D, B * S)}
    s["cache"] = _empty(ops.mha_cache_floats(B, S, D))
    return s


def _mha_run(c, s):
    B, S, D, heads = c["batch"], c["steps"], c["dim"], c["heads"]
    x, W, gW = s["x"], s["W"], s["gW"]
    ops.mha_forward_residual(x, x, x, W[0], W[1], W[2], W[3], x, s["out"], s["cache"], B, S, D, heads,
                             ops.ROWS_BY_SAMPLE)
    ops.mha_backward_residual(x, x, x, W[0], W[1], W[2], W[3], s["cache"], s["dY"], s["dY"], gW[0], gW[1], gW[2],
                              gW[3], s["dX"], B, S, D, heads, ops.ROWS_BY_SAMPLE)
    return [s["out"], gW, s["dX"]]


def _mha_exact(c, s):
    B, S, D = c["batch"], c["steps"], c["dim"]
    x = _d(s["x"]).T.contiguous().requires_grad_()                         # [B S, D]
    Wq, Wk, Wv, Wo = W = [_d(s["W"][k]).T.contiguous().requires_grad_() for k in range(4)]
    q, k, v = ((x @ w).reshape(B, S, D) for w in (Wq, Wk, Wv))
    A = torch.softmax(torch.bmm(q, k.transpose(1, 2).contiguous()) / math.sqrt(D / c["heads"]), 2)
    out = torch.bmm(A, v).reshape(B * S, D) @ Wo + x
    grads = torch.autograd.grad((out * _d(s["dY"]).T).sum(), [x] + W)
    return [out.detach().T.contiguous(), torch.stack([w.T for w in grads[1:]]), grads[0].T.contiguous()]


def _mha_work(c):
    B, S, D = c["batch"], c["steps"], c["dim"]
    return {"flops": 3 * (8 * B * S * D * D + 4 * B * S * S * D), "bytes": 4 * (4 * B * S * D + 8 * D * D)}


# ------------------------------------------------------- encoder feed-forward
# BatchNorm -> Linear -> GELU -> Linear with the skip sum, forward and
# backward: the second half of an encoder block over `rows` tokens.
def _ffn_prepare(c, g):
    N, D, F = c["rows"], c["dim"], c["hidden"]
    s = {"x": _randn(g, D, N), "gamma": 1 + 0.1 * _randn(g, D), "beta": 0.1 * _randn(g, D), "rm": torch.zeros(D, device="cuda"),
         "rv": torch.ones(D, device="cuda"), "W1": _xavier(g, D, F), "b1": _bias(g, F), "W2": _xavier(g, F, D),
         "b2": _bias(g, D), "dY": _randn(g, D, N).div_(N)}
    for k, n in (("bm", D), ("bv", D), ("gg", D), ("gbe", D), ("gb1", F), ("gb2", D)):
        s[k] = _empty(n)
    for k, r in (("h", D), ("y", D), ("dh", D), ("dx", D), ("z", F), ("a", F), ("dz", F)):
        s[k] = _empty(r, N)
    s.update(gW1=_empty(F, D), gW2=_empty(D, F))
    return s


def _ffn_run(c, s):
    N, D, F = c["rows"], c["dim"], c["hidden"]
    ops.batchnorm_forward(s["x"], s["h"], None, s["gamma"], s["beta"], s["rm"], s["rv"], s["bm"], s["bv"], N, D)
    ops.linear_forward(s["h"], s["W1"], s["b1"], s["z"], N, D, F)
    ops.gelu_forward(s["z"], s["a"])
    ops.linear_forward_act(s["a"], s["W2"], s["b2"], s["y"], s["h"], N, F, D, "residual")
    ops.linear_backward_act(s["a"], s["W2"], s["dY"], s["gW2"], s["gb2"], s["dz"], s["z"], N, F, D, "gelu")
    ops.linear_backward_act(s["h"], s["W1"], s["dz"], s["gW1"], s["gb1"], s["dh"], s["dY"], N, D, F, "residual")
    ops.batchnorm_backward(s["dh"], s["x"], None, s["gamma"], s["bm"], s["bv"], s["gg"], s["gbe"], s["dx"], N, D)
    return [s[k] for k in ("y", "rm", "rv", "gW1", "gb1", "gW2", "gb2", "gg", "gbe", "dx")]


def _ffn_exact(c, s):
    p = [_d(s[k]).T.contiguous().requires_grad_() for k in ("x", "W1", "b1", "W2", "b2", "gamma", "beta")]
    x, W1, b1, W2, b2, gamma, beta = p
    mean, var = x.mean(0), x.var(0, unbiased=False)
    h = (x - mean) / torch.sqrt(var + 1e-5) * gamma + beta
    z = h @ W1 + b1
    y = (0.5 * z * (1 + torch.erf(z / math.sqrt(2.0)))) @ W2 + b2 + h
    gx, g1, gb1, g2, gb2, gg, gbe = torch.autograd.grad((y * _d(s["dY"]).T).sum(), p)
    return [y.detach().T.contiguous(), 0.1 * mean.detach(), 0.9 + 0.1 * var.detach(), g1.T.contiguous(), gb1,
            g2.T.contiguous(), gb2, gg, gbe, gx.T.contiguous()]


def _ffn_work(c):
    N, D, F = c["rows"], c["dim"], c["hidden"]
    return {"flops": 12 * N * D * F, "bytes": 4 * (4 * N * D + 4 * D * F + 2 * F + 8 * D)}


# --------------------------------------------------------------------- Adam
# The optimizer's update of every tensor of an MLP of `widths`.
def _adam_shapes(c):
    w = [int(v) for v in c["widths"].split("-")]
    return [n for i, o in zip(w[:-1], w[1:]) for n in (i * o, o)]


def _adam_prepare(c, g):
    t = [(0.05 * _randn(g, n), 1e-3 * _randn(g, n), 1e-3 * _randn(g, n), (1e-3 * _randn(g, n)).square_())
         for n in _adam_shapes(c)]
    return {"t": t, "params": [p + (1 - 0.9 ** 10, 1 - 0.999 ** 10) for p in t]}


def _adam_run(c, s):
    ops.adam_step_multi(s["params"], 1e-3, 0.9, 0.999, 1e-8)
    return [[p[0], p[2], p[3]] for p in s["t"]]


def _adam_exact(c, s):
    out = []
    for W, grad, m, v in s["t"]:
        W, grad, m, v = _d(W), _d(grad), _d(m), _d(v)
        m, v = 0.9 * m + 0.1 * grad, 0.999 * v + 0.001 * grad * grad
        out.append([W - 1e-3 * (m / (1 - 0.9 ** 10)) / (torch.sqrt(v / (1 - 0.999 ** 10)) + 1e-8), m, v])
    return out


def _adam_work(c):
    n = sum(_adam_shapes(c))
    return {"flops": 12 * n, "bytes": 28 * n}


# ------------------------------------------------------------ training session
# A binary classifier (Linear -> ReLU -> Linear -> Sigmoid, BCE, Adam) trained
# for one epoch of a resident DataLoader; the program reads the last loss and
# the weights at the end.
def _epoch_cfg(c):
    return trainer.MLPConfig("classifier", [c["inputs"], c["hidden"], 1], "relu", "sigmoid", "bce", c["batch"])


def _epoch_data(c, seed):
    rng = np.random.default_rng(int(seed))
    cfg = _epoch_cfg(c)
    n = c["batch"] * c["batches"]
    params, _, _ = trainer.synthetic_mlp(cfg, rng)
    X = rng.standard_normal((c["inputs"], n)).astype(np.float32)
    Y = (X[:3].sum(0, keepdims=True) + rng.standard_normal((1, n)) > 0).astype(np.float32)
    return cfg, params, X, Y


def _epoch_prepare(c, seed):
    cfg, params, X, Y = _epoch_data(c, seed)
    sess = trainer.Session(cfg)
    sess.set_params(params)
    loader = trainer.Loader(X, Y, X.shape[1], c["inputs"], 1, c["batch"], shuffle=False)
    loader.to_device("resident")
    return {"sess": sess, "loader": loader}


def _epoch_run(c, s):
    sess, loader = s["sess"], s["loader"]
    loader.reset()
    for _ in range(c["batches"] - 1):
        loader.next_batch(sess)
        sess.step(read_loss=False)
    loader.next_batch(sess)
    loss = sess.step()
    return [loss, sess.get_params()]


def _epoch_exact(c, seed):
    cfg, params, X, Y = _epoch_data(c, seed)
    I, H, B = c["inputs"], c["hidden"], c["batch"]
    W1, b1, W2, b2 = p = [v.astype(np.float64) for v in params]
    m, v = [np.zeros_like(a) for a in p], [np.zeros_like(a) for a in p]
    for t in range(1, c["batches"] + 1):
        x, y = (a[:, (t - 1) * B:t * B].astype(np.float64) for a in (X, Y))
        z = W1.reshape(H, I) @ x + b1[:, None]
        a = np.maximum(z, 0)
        q = 1 / (1 + np.exp(-(W2[None] @ a + b2[:, None])))
        loss = -np.mean(y * np.log(q) + (1 - y) * np.log(1 - q))
        d = (q - y) / B
        da = (W2[:, None] @ d) * (z > 0)
        for k, grad in enumerate(((da @ x.T).ravel(), da.sum(1), (a @ d.T).ravel(), d.sum(1))):
            m[k] = 0.9 * m[k] + 0.1 * grad
            v[k] = 0.999 * v[k] + 0.001 * grad * grad
            p[k] -= 1e-3 * (m[k] / (1 - 0.9 ** t)) / (np.sqrt(v[k] / (1 - 0.999 ** t)) + 1e-8)
    return [float(loss), p]


def _epoch_work(c):
    n, I, H = c["batch"] * c["batches"], c["inputs"], c["hidden"]
    return {"flops": n * (4 * I * H + 6 * H), "bytes": 4 * (n * (I + 1) + 2 * (I * H + 2 * H + 1))}


# ------------------------------------------------------------------- the list
# kind -> (prepare, run, exact, work, tolerance).  Tolerances are about four
# times the largest distance from the float64 result seen over the declared
# ranges: fp32 sums over the longest contraction of each kind.
KINDS = {
    "linear": (_linear_prepare, _linear_run, _linear_exact, _linear_work, {"rel": 4e-6}),
    "head": (_head_prepare, _head_run, _head_exact, _head_work, {"rel": 1e-6}),
    "conv": (_conv_prepare, _conv_run, _conv_exact, _conv_work, {"rel": 1.5e-6, "differ": 1e-5}),
    "rnn": (_rnn_prepare, _rnn_run, _rnn_exact, _rnn_work, {"rel": 4e-6}),
    "mha": (_mha_prepare, _mha_run, _mha_exact, _mha_work, {"rel": 1e-5}),
    "ffn": (_ffn_prepare, _ffn_run, _ffn_exact, _ffn_work, {"rel": 4e-6}),
    "adam": (_adam_prepare, _adam_run, _adam_exact, _adam_work, {"rel": 6e-7}),
    "epoch": (_epoch_prepare, _epoch_run, _epoch_exact, _epoch_work, {"rel": 1e-5}),
}


def _conv(name, n, c, h, w, oc, ks, s, p, pool, first):
    return {"name": name, "kind": "conv", "batch": n, "channels": c, "height": h, "width": w, "filters": oc,
            "kernel": ks, "stride": s, "padding": p, "pool": pool, "first": first}


def listed():
    return [
        # the quick-start binary classifier (30-64-1, batch 512): launch latency
        {"name": "classifier_epoch", "kind": "epoch", "batch": 512, "inputs": 30, "hidden": 64, "batches": 16},
        # the wide MLP benchmark's hidden layer: large square products
        {"name": "mlp_hidden", "kind": "linear", "batch": 4096, "inputs": 4096, "outputs": 4096, "input_grad": True},
        # a user's own layer sizes: odd batch, odd widths (a last batch, 28 x 28 images with a bias column)
        {"name": "mlp_ragged", "kind": "linear", "batch": 1001, "inputs": 785, "outputs": 515, "input_grad": True},
        # the wide MLP's classifier head with its loss: bandwidth
        {"name": "mlp_head", "kind": "head", "batch": 4096, "inputs": 4096, "outputs": 10},
        # the CNN benchmark's two blocks (RGB 32 x 32, batch 256)
        _conv("cnn_rgb_block", 256, 3, 32, 32, 32, 3, 1, 1, 2, True),
        _conv("cnn_mid_block", 256, 32, 16, 16, 64, 3, 1, 1, 2, False),
        # a strided 5 x 5 layer at an odd batch and odd sizes, without pooling
        _conv("cnn_odd_layer", 100, 17, 29, 27, 40, 5, 2, 2, 0, False),
        # the sequence benchmark (LSTM 128 -> 512, 64 steps, batch 128) and its GRU form
        {"name": "lstm_sequence", "kind": "rnn", "layer": "lstm", "batch": 128, "steps": 64, "inputs": 128,
         "hidden": 512, "last": True, "input_grad": False},
        {"name": "gru_sequence", "kind": "rnn", "layer": "gru", "batch": 128, "steps": 64, "inputs": 128,
         "hidden": 512, "last": False, "input_grad": True},
        # the encoder benchmark's two halves (batch 32, 256 tokens, width 512, FFN 2048)
        {"name": "encoder_attention", "kind": "mha", "batch": 32, "steps": 256, "dim": 512, "heads": 8},
        {"name": "encoder_ffn", "kind": "ffn", "rows": 8192, "dim": 512, "hidden": 2048},
        # the wide MLP's optimizer step: a pure stream
        {"name": "adam_step", "kind": "adam", "widths": "1024-4096-4096-10"},
    ]


def draw(rng):
    kind = rng.choice(["linear", "linear", "head", "conv", "conv", "lstm", "gru", "mha", "ffn", "adam", "epoch"])
    if kind == "linear":
        return {"kind": kind, "batch": _log(rng, 16, 4096), "inputs": _log(rng, 16, 4096),
                "outputs": _log(rng, 17, 4096), "input_grad": rng.random() < 0.75}
    if kind == "head":
        return {"kind": kind, "batch": _log(rng, 64, 4096), "inputs": _log(rng, 64, 4096), "outputs": rng.randint(2, 32)}
    if kind == "conv":
        first = rng.random() < 0.4
        ks, pool = rng.choice([(3, 2), (3, 0), (5, 2), (5, 0)])
        stride = 1 if pool else rng.choice([1, 2])
        h = rng.randint(5, 16) * 2
        c = _conv("", _log(rng, 16, 256), rng.choice([1, 3]) if first else rng.randint(4, 32), h,
                  h if pool else rng.randint(10, 32), rng.randint(8, 64), ks, stride, ks // 2, pool, first)
        del c["name"]
        return c
    if kind in ("lstm", "gru"):
        return {"kind": "rnn", "layer": kind, "batch": _log(rng, 8, 128), "steps": rng.randint(8, 64),
                "inputs": rng.choice([32, 64, 128, _log(rng, 8, 128)]),
                "hidden": rng.choice([64, 128, 256, _log(rng, 32, 512)]),
                "last": kind == "lstm" and rng.random() < 0.5, "input_grad": rng.random() < 0.5}
    if kind == "mha":
        return {"kind": kind, "batch": _log(rng, 2, 32), "steps": rng.randint(16, 256), "dim": 8 * rng.randint(8, 64),
                "heads": 8}
    if kind == "ffn":
        return {"kind": kind, "rows": _log(rng, 128, 8192), "dim": rng.randint(64, 512), "hidden": rng.randint(128, 2048)}
    if kind == "adam":
        return {"kind": kind, "widths": "-".join(str(_log(rng, 16, 4096)) for _ in range(3)) + "-10"}
    return {"kind": kind, "batch": 16 * rng.randint(2, 64), "inputs": rng.randint(4, 64), "hidden": rng.randint(8, 64),
            "batches": rng.randint(4, 16)}


def prepare(case, seed):
    p = KINDS[case["kind"]][0]
    state = p(case, seed) if case["kind"] == "epoch" else p(case, _gen(seed))
    state["case"] = case
    return state


def run(state):
    c = state["case"]
    return KINDS[c["kind"]][1](c, state)


def exact(case, seed):
    e = KINDS[case["kind"]][2]
    if case["kind"] == "epoch":
        return e(case, seed)
    return e(case, KINDS[case["kind"]][0](case, _gen(seed)))


def work(case):
    return KINDS[case["kind"]][3](case)


def tolerance(case):
    return dict(KINDS[case["kind"]][4])
