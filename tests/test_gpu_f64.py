"""The double-precision entry points (haste_hip_*_f64, what ForwardPass<double> /
BackwardPass<double> bind to) against the fp64 oracle: the float parity tests of every cell
are run again with float64 tensors and a tolerance of 1e-10."""
import numpy as np
import pytest

import test_gpu_cpp_api
import test_gpu_gru
import test_gpu_indrnn
import test_gpu_iterate
import test_gpu_layer_norm
import test_gpu_layer_norm_cells
import test_gpu_lstm
from util import host, relerr

pytestmark = pytest.mark.gpu

TOL64 = 1e-10
MODULES = (test_gpu_lstm, test_gpu_gru, test_gpu_layer_norm_cells, test_gpu_indrnn,
           test_gpu_layer_norm, test_gpu_iterate)
# (T, N, C, H): tiny, ragged, a few tiles, and one with more rows than a column-sum chunk
SHAPES = [(1, 1, 3, 4), (3, 2, 3, 4), (5, 3, 7, 5), (6, 17, 20, 36), (4, 16, 32, 64),
          (7, 33, 48, 128), (3, 70, 24, 300)]


def dev64(a):
    import torch
    if a is None:
        return torch.empty(0, 0, 0, dtype=torch.float64, device="cuda")
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()


@pytest.fixture
def double_precision(monkeypatch):
    for mod in MODULES:
        monkeypatch.setattr(mod, "dev", dev64)
        if hasattr(mod, "TOL"):
            monkeypatch.setattr(mod, "TOL", TOL64)


@pytest.mark.parametrize("zoneout", [0.0, 0.3])
@pytest.mark.parametrize("T,N,C,H", SHAPES)
def test_f64_lstm_gru(double_precision, T, N, C, H, zoneout):
    test_gpu_lstm.test_lstm_training_forward_backward(T, N, C, H, zoneout)
    test_gpu_gru.test_gru_training_forward_backward(T, N, C, H, zoneout)


@pytest.mark.parametrize("zoneout", [0.0, 0.3])
@pytest.mark.parametrize("T,N,C,H", SHAPES)
def test_f64_layer_norm_cells(double_precision, T, N, C, H, zoneout):
    test_gpu_layer_norm_cells.test_layer_norm_lstm_training_forward_backward(T, N, C, H, zoneout)
    test_gpu_layer_norm_cells.test_layer_norm_gru_training_forward_backward(T, N, C, H, zoneout)


# A workgroup a row: one wavefront and a unit more, 1, 2 and 4 units a thread at their ends, and a row that is not held;
# the product in chunks and, with more than 32 and 16 rows of many units, whole.
@pytest.mark.parametrize("T,N,C,H", [(2, 3, 4, 64), (2, 3, 4, 65), (3, 2, 4, 1024), (2, 2, 4, 1025), (2, 2, 4, 2050),
                                     (2, 2, 4, 4096), (2, 2, 4, 4100), (2, 33, 4, 639), (2, 33, 4, 640), (2, 17, 4, 3073)])
def test_f64_layer_norm_cells_row_by_row(double_precision, T, N, C, H):
    test_f64_layer_norm_cells(None, T, N, C, H, 0.3)


@pytest.mark.parametrize("layer_norm", [False, True])
@pytest.mark.parametrize("zoneout", [0.0, 0.3])
@pytest.mark.parametrize("T,N,C,H", SHAPES[1:])
def test_f64_indrnn(double_precision, T, N, C, H, zoneout, layer_norm):
    test_gpu_indrnn.test_indrnn_training_forward_backward(T, N, C, H, zoneout, layer_norm)


def test_f64_inference_dropconnect_determinism(double_precision):
    for zoneout in (0.0, 0.25):
        test_gpu_lstm.test_lstm_inference_forward(zoneout, 20, 16, 128, 256)
        test_gpu_gru.test_gru_inference_forward(zoneout, 20, 16, 128, 256)
    test_gpu_layer_norm_cells.test_layer_norm_lstm_inference_forward()
    test_gpu_lstm.test_lstm_dropconnect_fused_equals_premasked_weights(6, 8, 16, 64)
    test_gpu_gru.test_gru_dropconnect_fused_equals_premasked_weights(6, 8, 16, 64)
    test_gpu_lstm.test_lstm_accumulates_into_weight_gradients_and_is_deterministic()


@pytest.mark.parametrize("with_beta", [False, True])
@pytest.mark.parametrize("rows,D", [(1, 1), (3, 5), (7, 33), (100, 256), (37, 1000), (300, 2048), (5, 5000)])
def test_f64_layer_norm(double_precision, rows, D, with_beta):
    test_gpu_layer_norm.test_layer_norm_forward_backward(rows, D, with_beta)


# 0.25: the inference-mode blend takes the probability as float, as the reference's signatures
# do, so only a probability float represents exactly matches the oracle to 1e-10
@pytest.mark.parametrize("zoneout", [0.0, 0.25])
@pytest.mark.parametrize("T,N,C,H", [(3, 2, 3, 4), (4, 5, 7, 20), (3, 64, 48, 128)])
def test_f64_iterate(double_precision, T, N, C, H, zoneout):
    test_gpu_iterate.test_lstm_iterate(T, N, C, H, zoneout)
    test_gpu_iterate.test_gru_iterate(T, N, C, H, zoneout)


# One kernel for a step: a row, partly filled tiles of 16 rows and units, several runs, sides of any length.
@pytest.mark.parametrize("training", [True, False])
@pytest.mark.parametrize("N,C,H", [(1, 512, 512), (3, 100, 333), (16, 16, 512), (17, 5, 47), (40, 60, 1500), (128, 3, 1)])
def test_f64_single_step_kernel(double_precision, N, C, H, training):
    test_gpu_iterate.test_single_step_kernel(N, C, H, training, 0.25)


@pytest.mark.parametrize("N,C,H", [(4, 48, 200), (33, 48, 200)])
def test_f64_single_step_dropconnect(double_precision, N, C, H):
    test_gpu_lstm.test_lstm_dropconnect_fused_equals_premasked_weights(1, N, C, H)


@pytest.mark.parametrize("trans_a,M,N,K", [(False, 1, 1, 1), (False, 37, 53, 29), (False, 128, 192, 64),
                                           (True, 70, 130, 45), (True, 5, 20, 33), (False, 300, 100, 1000),
                                           # few tiles, long contractions: cut along K into pieces
                                           (False, 64, 512, 2048), (True, 33, 70, 3001),
                                           # whole panels and columns inside the problem: the loads without
                                           # bounds checks (rows beyond M beyond the buffer's range)
                                           (True, 128, 256, 640), (False, 100, 128, 96), (True, 192, 128, 2080)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_f64_gemm_and_transpose(trans_a, M, N, K, accumulate):
    from haste_amd import ops
    import torch
    r = np.random.default_rng(M * 7 + N * 3 + K)
    a = r.standard_normal((K, M) if trans_a else (M, K))
    b = r.standard_normal((K, N))
    c0 = r.standard_normal((M, N))
    out = dev64(c0)
    ops.gemm(dev64(a), dev64(b), out=out, trans_a=trans_a, accumulate=accumulate)
    ref = (a.T if trans_a else a) @ b + (c0 if accumulate else 0.0)
    assert relerr(host(out), ref) < 1e-13
    t = ops.transpose(dev64(a))
    assert torch.equal(t, dev64(a).t().contiguous())


@pytest.mark.parametrize("trans_a,M,N,K", [
    # the last tiles cut behind whole ones, loads in pairs of whole and ragged panels and single
    (False, 1100, 1024, 512), (True, 1030, 1022, 770), (False, 1041, 1021, 515), (True, 1088, 1021, 516),
    # all tiles cut; a last round that fills the chip and is not; pairs in a panel of less than 32
    (True, 512, 2048, 512), (False, 1920, 1024, 512), (False, 70, 66, 2), (True, 66, 70, 30),
    # pieces of fewer rows and columns than a tile
    (False, 4, 130, 1030), (True, 67, 5, 1031), (False, 1, 1, 4096),
    # two pieces of whole panels are longer than the product: not cut
    (True, 520, 1560, 333),
    # whole tiles taken as they are numbered: 28 columns of tiles, 24 with the last tiles cut
    (False, 520, 1792, 40), (True, 1100, 1536, 512)])
@pytest.mark.parametrize("room", [True, False])
def test_f64_gemm_in_pieces(trans_a, M, N, K, room):
    """Error of a sum of K products in double, in any order: below K * 2^-53 of the sum of their magnitudes.  Without
    room for the pieces (a lent buffer of 128 KiB) a product is not cut, and is right."""
    from haste_amd import ops
    import torch
    r = np.random.default_rng(M + N + K)
    a = r.standard_normal((K, M) if trans_a else (M, K))
    b = r.standard_normal((K, N))
    c0 = r.standard_normal((M, N))
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        lent = None if room else torch.empty(128 * 1024, dtype=torch.uint8, device="cuda")
        ops.set_workspace(lent)
        try:
            wide = torch.full((M, N + 3), 7.0, dtype=torch.float64, device="cuda")   # what lies beside C stays
            wide[:, :N] = dev64(c0)
            ops.gemm(dev64(a), dev64(b), out=wide[:, :N], trans_a=trans_a, accumulate=True)
        finally:
            s.synchronize()
            ops.set_workspace(None)
    at = a.T if trans_a else a
    out = host(wide)
    bound = K * 2.0 ** -53 * (np.abs(at) @ np.abs(b) + np.abs(c0))
    assert (np.abs(out[:, :N] - (at @ b + c0)) <= 2 * bound).all()   # twice: the reference's own sum
    assert (out[:, N:] == 7.0).all()


# One to five panels of 32 k, whole, a pair and an element longer, the last ones written out: loads in whole panels, in pairs
# (even sizes) and element by element (odd ones).
@pytest.mark.parametrize("K", [1, 2, 31, 32, 33, 34, 64, 65, 66, 96, 97, 98, 128, 129, 130, 160, 161, 162])
@pytest.mark.parametrize("trans_a,M,N", [(False, 70, 66), (True, 70, 66), (True, 67, 65)])
def test_f64_gemm_short_contractions(trans_a, M, N, K):
    test_f64_gemm_in_pieces(trans_a, M, N, K, True)


def test_f64_layers_match_torch_nn():
    """haste_amd.LSTM / GRU in double against torch.nn.LSTM / GRU in double on the CPU."""
    import torch
    import haste_amd
    torch.manual_seed(3)
    T, N, C, H = 9, 5, 12, 20
    x = torch.randn(T, N, C, dtype=torch.float64)
    for ours_cls, theirs_cls in ((haste_amd.LSTM, torch.nn.LSTM), (haste_amd.GRU, torch.nn.GRU)):
        ours = ours_cls(C, H).double().cuda()
        theirs = theirs_cls(C, H).double()
        with torch.no_grad():
            for name, value in zip(("weight_ih_l0", "weight_hh_l0", "bias_ih_l0", "bias_hh_l0"),
                                   ours.to_native_weights()):
                getattr(theirs, name).copy_(value.cpu())
        xg = x.cuda().requires_grad_(True)
        xc = x.clone().requires_grad_(True)
        yo, _ = ours(xg)
        yt, _ = theirs(xc)
        assert relerr(host(yo), yt.detach().numpy()) < TOL64
        dy = torch.randn(T, N, H, dtype=torch.float64)
        yo.backward(dy.cuda())
        yt.backward(dy)
        assert relerr(host(xg.grad), xc.grad.numpy()) < TOL64


@pytest.mark.parametrize("cell", ["lstm", "layer_norm_lstm", "lstm_iterate", "gru", "layer_norm_gru",
                                  "gru_iterate", "indrnn", "layer_norm_indrnn"])
def test_f64_cpp_classes(monkeypatch, cell):
    """ForwardPass<double> / BackwardPass<double> of every namespace of include/haste.h."""
    monkeypatch.setattr(test_gpu_cpp_api, "DTYPE", np.float64)
    monkeypatch.setattr(test_gpu_cpp_api, "TOL", TOL64)
    T, N, C, H, zoneout = 9, 20, 24, 64, 0.3
    ln = "iterate" if cell.endswith("_iterate") else cell.startswith("layer_norm")
    if "lstm" in cell:
        test_gpu_cpp_api.test_cpp_lstm(T, N, C, H, zoneout, ln)
    elif "gru" in cell:
        test_gpu_cpp_api.test_cpp_gru(T, N, C, H, zoneout, ln)
    else:
        test_gpu_cpp_api.test_cpp_indrnn(T, N, C, H, zoneout, ln)


# The recurrences in one launch: weights in registers alone and shared with LDS, 8 and 16 units per
# workgroup, groups within and across XCDs, ragged last units, rows and quarters of the contraction;
# (4, 70, 8, 768): forward too large for it, backward not.
ONE_LAUNCH_SHAPES = [(4, 1, 4, 1), (5, 64, 8, 512), (4, 128, 8, 512), (4, 16, 8, 513), (6, 33, 12, 300), (4, 20, 8, 700),
                     (4, 70, 8, 768), (4, 113, 4, 72), (4, 129, 4, 250)]


@pytest.mark.parametrize("zoneout", [0.0, 0.3])
@pytest.mark.parametrize("T,N,C,H", ONE_LAUNCH_SHAPES)
def test_f64_recurrence_in_one_launch(double_precision, T, N, C, H, zoneout):
    test_gpu_lstm.test_lstm_training_forward_backward(T, N, C, H, zoneout)
    test_gpu_gru.test_gru_training_forward_backward(T, N, C, H, zoneout)


# Enough steps for every exchange tile to be written twice.  Groups of 8 rows: one workgroup; 8 units per workgroup up to
# 32 of them, 16 from there; polled up to 64 backward steps' worth of k, behind the barrier above; 8 rows across XCDs.
# Groups of 16 rows from 65 rows or 513 units on; none, where the GRU's forward pass finds no kernel (37 rows, 800 units).
@pytest.mark.parametrize("T,N,C,H", [(9, 8, 4, 16), (9, 9, 4, 256), (9, 64, 4, 257), (10, 61, 4, 340), (9, 65, 4, 128),
                                     (9, 37, 4, 520), (9, 3, 4, 513), (5, 37, 4, 800)])
def test_f64_recurrence_tiles(double_precision, T, N, C, H):
    test_gpu_lstm.test_lstm_training_forward_backward(T, N, C, H, 0.3)
    test_gpu_gru.test_gru_training_forward_backward(T, N, C, H, 0.3)


@pytest.mark.parametrize("N,H", [(8, 64), (64, 512), (70, 64)])
def test_f64_recurrence_carries_every_nan(N, H):
    """A state whose bits mark unwritten elements: its row turns to NaN, the others do not, nobody waits for it."""
    import torch
    from haste_amd import layers, ops
    torch.manual_seed(1)
    layer = layers.GRU(16, H).cuda().double()
    x = torch.randn(9, N, 16, device="cuda", dtype=torch.float64)
    h0 = torch.zeros(1, N, H, device="cuda", dtype=torch.float64)
    with torch.no_grad():
        expected, _ = layer(x, h0)
        h0[0, 2].view(torch.int64).fill_(-1)
        y, _ = layer(x, h0)
    ops.stream_status()
    assert torch.isnan(y[:, 2]).all()
    others = [n for n in range(N) if n != 2]
    assert torch.equal(y[:, others], expected[:, others])


@pytest.mark.parametrize("T,N,C,H", ONE_LAUNCH_SHAPES[1:5])
def test_f64_inference_in_one_launch(double_precision, T, N, C, H):
    test_gpu_lstm.test_lstm_inference_forward(0.25, T, N, C, H)
    test_gpu_gru.test_gru_inference_forward(0.25, T, N, C, H)


def test_f64_recurrence_under_capture():
    """A captured call runs step by step; every replay gives what the eager call gives to rounding."""
    import torch
    from haste_amd import ops
    T, N, C, H = 6, 20, 16, 64
    r = np.random.default_rng(5)
    arrays = [dev64(r.uniform(-0.3, 0.3, s)) for s in ((T, N, C), (N, H), (N, H), (C, 4 * H), (H, 4 * H), (4 * H,))]
    x, h0, c0, W, R, b = arrays
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        ops.lstm_forward(False, 0.0, x, h0, c0, W, R, b, dev64(None))
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            h, c, _ = ops.lstm_forward(False, 0.0, x, h0, c0, W, R, b, dev64(None))
    for k in range(3):
        x.copy_(dev64(r.uniform(-1, 1, (T, N, C))))
        graph.replay()
        eager, _, _ = ops.lstm_forward(False, 0.0, x, h0, c0, W, R, b, dev64(None))
        torch.cuda.synchronize()
        assert relerr(host(h), host(eager)) < 1e-13, k
