"""The forward recurrences on the bf16 matrix cores (h and R as sums of three bfloat16):
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
@pytest.mark.parametrize("T,N,H", [(24, 2, 257), (25, 29, 384), (24, 32, 385), (26, 7, 512), (24, 33, 257), (25, 40, 320),
                                   (24, 64, 384), (27, 41, 511), (24, 64, 512), (2, 65, 225), (5, 127, 256), (4, 128, 257),
                                   (6, 128, 384), (3, 127, 385), (7, 66, 510), (9, 100, 512), (3, 121, 511)])
@pytest.mark.parametrize("training,zoneout", [(True, 0.2), (False, 0.2), (True, 0.0)])
@pytest.mark.parametrize("cell", ["lstm", "gru"])
def test_tiles(cell, training, zoneout, T, N, H):
    print("split recurrence", cell, training, zoneout, T, N, H, flush=True)
    p = problem(T + N + H, T, N, 18, H, 4 if cell == "lstm" else 3, zoneout)
    for ours, theirs in zip(forward(cell, p, training, zoneout), reference(cell, p, training, zoneout)):
        assert relerr(host(ours), theirs) < BOUND


@pytest.mark.parametrize("what", ["state", "state_inf", "weight", "weight_inf", "nan"])
@pytest.mark.parametrize("N", [20, 40, 100])
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
