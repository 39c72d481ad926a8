"""LSTM and GRU forward recurrences: x*W computed inside the recurrence (4-row tiles) gives, to rounding,
what the recurrence gives on x*W from a GEMM launched before it.

The variant with the separate GEMM is selected by an environment variable that the library reads
once, so it runs in a child process.  The shapes have 8-row tiles run as two 4-row sets per
workgroup: a ragged last set, a set without rows, full sets."""
import os
import subprocess
import sys
import tempfile

import numpy as np
import pytest

from util import dev, host, problem, relerr

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# (T, N, C, H)
SHAPES = [(6, 41, 24, 512), (5, 64, 32, 256), (4, 36, 8, 72), (5, 40, 300, 320), (4, 13, 512, 400)]


def run_cells(T, N, C, H):
    """LSTM and GRU forward + backward with zoneout; every output as float64 arrays."""
    import torch
    from haste_amd import ops
    out = {}
    p = problem(900 + T + N + C + H, T, N, C, H, 4, 0.2)
    mask = dev(p["mask"])
    h, c, cache = ops.lstm_forward(True, 0.2, dev(p["x"]), dev(p["h0"]), dev(p["c0"]),
                                   dev(p["W"]), dev(p["R"]), dev(p["b"]), mask)
    x_t = dev(p["x"]).permute(2, 0, 1).contiguous()
    grads = ops.lstm_backward(x_t, dev(p["W"]).t().contiguous(), dev(p["R"]).t().contiguous(),
                              dev(p["b"]), mask, h, c, cache, dev(p["dh_new"]), dev(p["dc_new"]))
    for name, t in zip(("h", "c", "dx", "dh", "dc", "dW", "dR", "db", "dv"), (h, c) + tuple(grads) + (cache,)):
        out["lstm_" + name] = host(t)

    p = problem(901 + T + N + C + H, T, N, C, H, 3, 0.2)
    mask = dev(p["mask"])
    W, R, bx, br = dev(p["W"]), dev(p["R"]), dev(p["b"]), dev(p["b2"])
    h, cache = ops.gru_forward(True, 0.2, dev(p["x"]), dev(p["h0"]), W, R, bx, br, mask)
    x_t = dev(p["x"]).permute(2, 0, 1).contiguous()
    grads = ops.gru_backward(x_t, W.t().contiguous(), R.t().contiguous(), bx, br, mask, h, cache,
                             dev(p["dh_new"]))
    for i, t in enumerate((h,) + tuple(grads)):
        out["gru_%d" % i] = host(t)
    torch.cuda.synchronize()
    return out


def child(path):
    arrays = {}
    for shape in SHAPES:
        for k, v in run_cells(*shape).items():
            arrays["%d_%d_%d_%d_%s" % (shape + (k,))] = v
    np.savez(path, **arrays)


def _child_outputs(d, name, **env_vars):
    path = os.path.join(d, name + ".npz")
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([ROOT, os.path.join(ROOT, "tests")]), **env_vars)
    res = subprocess.run([sys.executable, os.path.abspath(__file__), path], env=env,
                         capture_output=True, text=True, timeout=110)
    assert res.returncode == 0, res.stdout + res.stderr
    return np.load(path)


def test_input_projection_inside_the_recurrence_matches_the_separate_gemm():
    """x*W computed by the forward recurrence beside its waits (this process) against x*W from
    the GEMM launched before it (child process): the same sums in another order, so equal to
    rounding, forward and -- through the saved activations -- backward."""
    with tempfile.TemporaryDirectory() as d:
        separate = _child_outputs(d, "separate", HASTE_HIP_FUSED_INPUT="0")
        for shape in SHAPES:
            print("fused input projection vs separate GEMM", shape, flush=True)
            for k, v in run_cells(*shape).items():
                ref = separate["%d_%d_%d_%d_%s" % (shape + (k,))]
                assert relerr(v, ref) < 5e-6, (shape, k)


@pytest.mark.parametrize("T,N,C,H", [(63, 9, 512, 512), (64, 9, 512, 512), (257, 29, 512, 256), (513, 3, 128, 256),
                                     (70, 33, 512, 512)])
@pytest.mark.parametrize("lent", [False, True])
def test_either_side_of_the_rule_for_the_input_projection(T, N, C, H, lent):
    """T * C * H, C * H and N just below and above what sends x*W to the GEMM, in the library's own workspace and in
    memory that holds the recurrence's exchange tiles but not the GEMM's partial tiles, against
    the oracle in fp64.  The bound is the forward parity tests'."""
    import torch
    from haste_amd import ops
    from oracle import haste_oracle as O
    print("projection rule", T, N, C, H, lent, flush=True)
    p = problem(17 + T + N + C + H, T, N, C, H, 4, 0.0)
    q = problem(18 + T + N + C + H, T, N, C, H, 3, 0.0)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        memory = torch.empty(1 << 20, dtype=torch.uint8, device="cuda:0") if lent else None
        if lent:
            ops.set_workspace(memory)
        try:
            h, c, _ = ops.lstm_forward(True, 0.0, dev(p["x"]), dev(p["h0"]), dev(p["c0"]), dev(p["W"]), dev(p["R"]),
                                       dev(p["b"]), torch.empty(0, device="cuda:0"))
            with_gru = not lent or H >= 512  # below, the GRU takes the GEMM at any T
            hg = None if not with_gru else ops.gru_forward(True, 0.0, dev(q["x"]), dev(q["h0"]), dev(q["W"]), dev(q["R"]), dev(q["b"]),
                                    dev(q["b2"]), torch.empty(0, device="cuda:0"))[0]
            s.synchronize()
        finally:
            s.synchronize()
            if lent:
                ops.set_workspace(None)
    ho, co, _ = O.lstm_forward(p["W"], p["R"], p["b"], p["x"], p["h0"], p["c0"])
    go, _ = O.gru_forward(q["W"], q["R"], q["b"], q["b2"], q["x"], q["h0"])
    assert relerr(host(h), ho) < 1e-4 and relerr(host(c), co) < 1e-4
    assert not with_gru or relerr(host(hg), go) < 1e-4


if __name__ == "__main__":
    child(sys.argv[1])
