"""The recurrences on the bf16 matrix cores (h, the gate gradients and R as sums of three bfloat16):
the edges of their tiles against the fp64 oracle, and values whose parts would overflow or are not finite."""
import numpy as np
import pytest

from oracle import haste_oracle as O
from util import dev, host, problem, relerr

pytestmark = pytest.mark.gpu

# Largest error over the largest value.  A step's sums are rounded a few times at 2^-24 and the gates lose some 2^-23
# each; over the steps here, whose states forget, the errors add up to no more than 2^-20.
BOUND = 2.0 ** -20


def forward(cell, p, training, zoneout):
    from haste_amd import ops
    if cell == "lstm":
        h, c, v = ops.lstm_forward(training, zoneout, dev(p["x"]), dev(p["h0"]), dev(p["c0"]), dev(p["W"]), dev(p["R"]),
                                   dev(p["b"]), dev(p["mask"]))
        return (h, c, v) if training else (h, c)
    h, v = ops.gru_forward(training, zoneout, dev(p["x"]), dev(p["h0"]), dev(p["W"]), dev(p["R"]), dev(p["b"]), dev(p["b2"]),
                           dev(p["mask"]))
    return (h, v) if training else (h,)


def reference(cell, p, training, zoneout):
    if cell == "lstm":
        out = O.lstm_forward(p["W"], p["R"], p["b"], p["x"], p["h0"], p["c0"], training, zoneout, p["mask"])
    else:
        out = O.gru_forward(p["W"], p["R"], p["b"], p["b2"], p["x"], p["h0"], training, zoneout, p["mask"])
    return out if training else out[:-1]


# rows around the tiles' edges (4-, 8- and 16-row tiles); groups of 32 hidden units per wavefront one more and one fewer;
# rows of H floats that do not start on 16 bytes; the fewest steps the rule takes (input sizes that are no multiple of 4:
# nothing is computed beside the waits)
FORWARD = [(24, 2, 257), (25, 29, 384), (24, 32, 385), (26, 7, 512), (24, 33, 257), (25, 40, 320), (24, 64, 384), (27, 41, 511),
           (24, 64, 512), (2, 65, 225), (5, 127, 256), (4, 128, 257), (6, 128, 384), (3, 127, 385), (7, 66, 510),
           (9, 100, 512), (3, 121, 511)]


@pytest.mark.parametrize("T,N,H", FORWARD)
@pytest.mark.parametrize("training,zoneout", [(True, 0.2), (False, 0.2), (True, 0.0)])
@pytest.mark.parametrize("cell", ["lstm", "gru"])
def test_tiles(cell, training, zoneout, T, N, H):
    print("split recurrence", cell, training, zoneout, T, N, H, flush=True)
    p = problem(T + N + H, T, N, 18, H, 4 if cell == "lstm" else 3, zoneout)
    for ours, theirs in zip(forward(cell, p, training, zoneout), reference(cell, p, training, zoneout)):
        assert relerr(host(ours), theirs) < BOUND


EXTREME_FORWARD = [(24, 20, 270), (24, 40, 270), (24, 100, 270)]


@pytest.mark.parametrize("what", ["state", "state_inf", "weight", "weight_inf", "nan"])
@pytest.mark.parametrize("N", [N for _, N, _ in EXTREME_FORWARD])
@pytest.mark.parametrize("cell", ["lstm", "gru"])
def test_values_that_do_not_split(cell, N, what):
    """Where fp32 arithmetic gives a finite value it is that value; elsewhere neither is finite."""
    print("split recurrence, extreme values", cell, N, what, flush=True)
    T, H = 24, 270
    p = problem(5 + N, T, N, 13, H, 4 if cell == "lstm" else 3)
    p["h0"][3, 7], p["R"][9, 11] = {"state": (2.0 ** 90, 0.01), "state_inf": (np.inf, 0.01), "weight": (0.5, 2.0 ** 100),
                                    "weight_inf": (0.5, -np.inf), "nan": (np.nan, 0.01)}[what]
    p["h0"][:, 9] = 0.5  # no 0 * inf
    with np.errstate(all="ignore"):
        expected = reference(cell, p, False, 0.0)
    for ours, theirs in zip(forward(cell, p, False, 0.0), expected):
        ours = host(ours)
        same = np.isfinite(theirs)
        assert np.array_equal(np.isfinite(ours), same)
        assert np.array_equal(np.isnan(ours), np.isnan(theirs))
        large = np.abs(theirs) > 2.0 ** 40  # the state itself, where a cell keeps some of it
        ordinary = same & ~large
        assert np.max(np.abs(ours[ordinary] - theirs[ordinary])) < BOUND * max(1.0, np.max(np.abs(theirs[ordinary])))
        if np.any(same & large):
            assert np.max(np.abs(ours[same & large] / theirs[same & large] - 1.0)) < 1e-5


@pytest.mark.parametrize("N", [10, 50, 90])
def test_dropconnect(N):
    """The mask applied while R is read gives what R masked beforehand gives, bit for bit."""
    import torch
    from haste_amd import ops
    T, C, H = 24, 15, 300
    p = problem(77 + N, T, N, C, H, 4, 0.0)
    keep = (np.random.default_rng(N).uniform(size=p["R"].shape) >= 0.3).astype(np.float64)
    scale = 2.0
    none = torch.empty(0, device="cuda")
    first = (dev(p["x"]), dev(p["h0"]), dev(p["c0"]), dev(p["W"]))
    a = ops.lstm_forward(False, 0.0, *first, dev(p["R"]), dev(p["b"]), none, dev(keep), scale)
    b = ops.lstm_forward(False, 0.0, *first, dev(p["R"] * keep * scale), dev(p["b"]), none)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def backward(cell, p, states):
    """Gradients for the states and activations of the reference's forward pass, by name."""
    from haste_amd import ops
    x_t = dev(p["x"]).permute(2, 0, 1).contiguous()
    W_t, R_t = dev(p["W"]).t().contiguous(), dev(p["R"]).t().contiguous()
    if cell == "lstm":
        h, c, v = (dev(a) for a in states)
        out = ops.lstm_backward(x_t, W_t, R_t, dev(p["b"]), dev(p["mask"]), h, c, v, dev(p["dh_new"]), dev(p["dc_new"]))
        return dict(zip(("dx", "dh0", "dc0", "dW", "dR", "db", "dv"), map(host, out + (v,))))
    h, v = (dev(a) for a in states)
    out = ops.gru_backward(x_t, W_t, R_t, dev(p["b"]), dev(p["b2"]), dev(p["mask"]), h, v, dev(p["dh_new"]))
    return dict(zip(("dx", "dh0", "dW", "dR", "dbx", "dbr"), map(host, out)))


def backward_reference(cell, p, states):
    states = tuple(np.float64(np.float32(a)) for a in states)
    if cell == "lstm":
        out = O.lstm_backward(p["W"], p["R"], p["b"], p["x"], *states, p["dh_new"], p["dc_new"], p["mask"])
        return dict(zip(("dx", "dW", "dR", "db", "dh0", "dc0", "dv"), out))
    out = O.gru_backward(p["W"], p["R"], p["b"], p["b2"], p["x"], *states, p["dh_new"], p["mask"])
    return dict(zip(("dx", "dW", "dR", "dbx", "dbr", "dh0"), out))


# The same for the backward pass, whose rule has more units and rows instead of more steps, and sizes beside the rule: one
# unit or row fewer runs on the fp32 instruction.
BACKWARD = [(1, 33, 129), (3, 64, 144), (4, 39, 257), (5, 64, 384), (2, 41, 385), (7, 50, 511), (9, 64, 512), (1, 65, 65),
            (5, 65, 80), (4, 128, 256), (3, 127, 258), (6, 96, 384), (2, 113, 400), (7, 66, 510), (9, 128, 512)]
BESIDE_BACKWARD = [(1, 33, 33), (3, 64, 16), (6, 40, 128), (1, 65, 32), (5, 65, 31), (2, 70, 64), (3, 32, 512)]


@pytest.mark.parametrize("T,N,H", BACKWARD + BESIDE_BACKWARD)
@pytest.mark.parametrize("zoneout", [0.0, 0.2])
@pytest.mark.parametrize("cell", ["lstm", "gru"])
def test_backward_tiles(cell, zoneout, T, N, H):
    print("split backward recurrence", cell, zoneout, T, N, H, flush=True)
    p = problem(T + N + H, T, N, 12, H, 4 if cell == "lstm" else 3, zoneout)
    states = reference(cell, p, True, zoneout)
    # The partial sums give their last bit (2^-24) to the exchange at every step, the gradients of the weights add up
    # T * N terms: 2^-18 of the largest value holds both.
    ours, theirs = backward(cell, p, states), backward_reference(cell, p, states)
    for name in ours:
        assert relerr(ours[name], theirs[name]) < 2.0 ** -18, name


EXTREME_BACKWARD = [(4, 40, 140), (4, 40, 270), (4, 64, 400), (4, 100, 70), (4, 100, 270)]
EXTREME_BESIDE_BACKWARD = [(4, 40, 70)]


@pytest.mark.parametrize("what", ["gradient", "gradient_inf", "weight", "weight_inf", "nan"])
@pytest.mark.parametrize("T,N,H", EXTREME_BACKWARD + EXTREME_BESIDE_BACKWARD)
@pytest.mark.parametrize("cell", ["lstm", "gru"])
def test_backward_values_that_do_not_split(cell, T, N, H, what):
    """Every gradient is finite, infinite and not a number where the reference is; those that are no sums over the rows are equal
    where finite, batch row 5, which has the extreme gradient, by itself; the LSTM's sums are those of its own dv."""
    print("split backward recurrence, extreme values", cell, N, H, what, flush=True)
    p = problem(9 + N, T, N, 8, H, 4 if cell == "lstm" else 3)
    states = reference(cell, p, True, 0.0)
    p["dh_new"][3, 5, 6], p["R"][9, 11] = {"gradient": (2.0 ** 60, 0.01), "gradient_inf": (np.inf, 0.01),
                                           "weight": (1.0, 2.0 ** 40), "weight_inf": (1.0, np.inf),
                                           "nan": (np.nan, 0.01)}[what]
    with np.errstate(all="ignore"):
        ours, theirs = backward(cell, p, states), backward_reference(cell, p, states)
    for name in theirs:
        a, b = ours[name], theirs[name]
        assert np.array_equal(np.isnan(a), np.isnan(b)), name
        assert np.array_equal(np.isfinite(a), np.isfinite(b)), name
        if name in ("dh0", "dc0", "dx", "dv"):
            row = np.broadcast_to((np.arange(N) == 5)[:, None], b.shape)
            for part in (np.isfinite(b) & row, np.isfinite(b) & ~row):
                if np.any(part):
                    assert np.max(np.abs(a[part] - b[part])) <= 1e-5 * np.max(np.abs(b[part])), name
    if cell == "lstm":
        dv = ours["dv"].reshape(T * N, 4 * H)
        for name, left in (("db", np.ones((T * N, 1))), ("dW", p["x"].reshape(T * N, -1)),
                           ("dR", np.float64(np.float32(states[0]))[:T].reshape(T * N, H))):
            with np.errstate(all="ignore"):
                total, terms = left.T @ dv, np.abs(left).T @ np.abs(dv)
            finite = np.isfinite(terms)
            error = np.abs(ours[name].reshape(total.shape)[finite] - total[finite])
            # T * N float sums in any order: T * N roundings of 2^-24 at most
            assert (error <= T * N * 2.0 ** -24 * terms[finite] + 1e-30).all(), name


# 2-norm of the error over the 2-norm of the result, T = 100, C = H = 512, against the same passes in double: what the
# recurrences on the fp32 instruction gave (the mean over 3 - 20 seeds; 1e-7), for y, dx, the gradients of kernel, recurrent kernel
# and biases.  A seed's biases differ by up to 11 % from the mean (this one's, LSTM, 64 rows, fp32 instruction: 2.85).
FP32_ERRORS = {("lstm", 64): (3.22, 2.69, 3.40, 4.36, 2.58), ("lstm", 128): (2.06, 3.53, 3.98, 4.22, 2.50),
               ("gru", 64): (1.55, 1.86, 2.56, 2.97, 2.12, 2.21), ("gru", 128): (1.56, 2.02, 3.46, 3.76, 2.20, 2.34)}


@pytest.mark.parametrize("cell,N", list(FP32_ERRORS))
def test_errors_are_no_larger_than_with_the_fp32_instruction(cell, N):
    import copy
    import torch
    from haste_amd import layers
    torch.manual_seed(N)
    T, H = 100, 512
    layer = {"lstm": layers.LSTM, "gru": layers.GRU}[cell](H, H).cuda()
    with torch.no_grad():
        for p in layer.parameters():
            p.uniform_(-H ** -0.5, H ** -0.5)
        if cell == "lstm":
            layer.bias[2 * H:3 * H] += 1.0
    x, dy = torch.randn(T, N, H, device="cuda"), torch.randn(T, N, H, device="cuda")

    def run(layer, x, dy):
        x = x.clone().requires_grad_(True)
        y, _ = layer(x)
        y.backward(dy)
        grads = dict(layer.named_parameters())
        names = ("kernel", "recurrent_kernel", "bias") + (("recurrent_bias",) if cell == "gru" else ())
        return [y.detach(), x.grad] + [grads[name].grad for name in names]
    exact = run(copy.deepcopy(layer).double(), x.double(), dy.double())
    for ours, theirs, bound in zip(run(layer, x, dy), exact, FP32_ERRORS[cell, N]):
        error = float((ours.double() - theirs).norm() / theirs.norm())
        print("split recurrence, error", cell, N, "%.3g of %.3g" % (error, bound * 1e-7), flush=True)
        assert error < 1.15 * bound * 1e-7
