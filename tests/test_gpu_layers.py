"""The torch.nn layers on the GPU: outputs and parameter gradients against torch.nn.LSTM /
torch.nn.GRU on the CPU (through the native-weight maps, as the reference's
validation/pytorch.py:60-89 does) and against the fp64 oracle for the options torch.nn
lacks (zoneout, DropConnect, layer norm, IndRNN); batch_first, lengths and
return_state_sequence handling."""
import numpy as np
import pytest
import torch

import haste_amd
from oracle import haste_oracle as O
from util import TOL, relerr

pytestmark = pytest.mark.gpu


def npy(t):
    return t.detach().cpu().double().numpy()


def test_lstm_layer_matches_torch_nn():
    T, N, C, H = 12, 9, 20, 32
    torch.manual_seed(0)
    layer = haste_amd.LSTM(C, H, batch_first=True).cuda()
    ref = torch.nn.LSTM(C, H, batch_first=True).double()
    for name, w in zip(("weight_ih_l0", "weight_hh_l0", "bias_ih_l0", "bias_hh_l0"), layer.to_native_weights()):
        setattr(ref, name, torch.nn.Parameter(w.detach().cpu().double()))
    x = torch.randn(N, T, C)
    h0, c0 = torch.randn(1, N, H) * 0.5, torch.randn(1, N, H) * 0.5
    xg = x.cuda().requires_grad_()
    y, (hn, cn) = layer(xg, (h0.cuda(), c0.cuda()))
    xr = x.double().requires_grad_()
    yr, (hr, cr) = ref(xr, (h0.double(), c0.double()))
    assert tuple(y.shape) == (N, T, H) and tuple(hn.shape) == (1, N, H)
    assert relerr(npy(y), npy(yr)) < TOL and relerr(npy(hn), npy(hr)) < TOL and relerr(npy(cn), npy(cr)) < TOL
    dy = torch.randn(N, T, H)
    dcn = torch.randn(1, N, H)
    ((y * dy.cuda()).sum() + (cn * dcn.cuda()).sum()).backward()
    ((yr * dy.double()).sum() + (cr * dcn.double()).sum()).backward()
    assert relerr(npy(xg.grad), npy(xr.grad)) < TOL
    # gradients of the native-layout weights, mapped back to the haste layout
    back = haste_amd.LSTM(C, H).double()
    back.from_native_weights(ref.weight_ih_l0.grad, ref.weight_hh_l0.grad, ref.bias_ih_l0.grad,
                             torch.zeros_like(ref.bias_hh_l0.grad))
    assert relerr(npy(layer.kernel.grad), npy(back.kernel)) < TOL
    assert relerr(npy(layer.recurrent_kernel.grad), npy(back.recurrent_kernel)) < TOL
    assert relerr(npy(layer.bias.grad), npy(back.bias)) < TOL
    with pytest.raises(RuntimeError, match="twice"):
        layer.zero_grad()
        y2, _ = layer(xg)
        y2.sum().backward(retain_graph=True)
        y2.sum().backward()


def test_gru_layer_matches_torch_nn():
    T, N, C, H = 10, 7, 16, 24
    torch.manual_seed(1)
    layer = haste_amd.GRU(C, H).cuda()
    with torch.no_grad():
        layer.bias.normal_(0, 0.1)
        layer.recurrent_bias.normal_(0, 0.1)
    ref = torch.nn.GRU(C, H).double()
    for name, w in zip(("weight_ih_l0", "weight_hh_l0", "bias_ih_l0", "bias_hh_l0"), layer.to_native_weights()):
        setattr(ref, name, torch.nn.Parameter(w.detach().cpu().double()))
    x = torch.randn(T, N, C)
    xg = x.cuda().requires_grad_()
    y, hn = layer(xg)
    xr = x.double().requires_grad_()
    yr, hr = ref(xr)
    assert relerr(npy(y), npy(yr)) < TOL and relerr(npy(hn), npy(hr)) < TOL
    dy = torch.randn(T, N, H)
    (y * dy.cuda()).sum().backward()
    (yr * dy.double()).sum().backward()
    assert relerr(npy(xg.grad), npy(xr.grad)) < TOL
    back = haste_amd.GRU(C, H).double()
    back.from_native_weights(ref.weight_ih_l0.grad, ref.weight_hh_l0.grad, ref.bias_ih_l0.grad,
                             ref.bias_hh_l0.grad)
    for name in ("kernel", "recurrent_kernel", "bias", "recurrent_bias"):
        assert relerr(npy(getattr(layer, name).grad), npy(getattr(back, name))) < TOL, name


def _drawn_masks(layer, T, N, seed):
    """The DropConnect and zoneout masks the layer will draw after torch.manual_seed(seed):
    it draws the DropConnect mask first, then the zoneout mask."""
    torch.manual_seed(seed)
    dmask, dscale = None, 1.0
    if getattr(layer, "dropout", 0.0) and layer.training:
        dmask = torch.empty_like(layer.recurrent_kernel).bernoulli_(1.0 - layer.dropout)
        dscale = 1.0 / (1.0 - layer.dropout)
    zmask = None
    if layer.zoneout:
        zmask = torch.empty(T, N, layer.hidden_size, device="cuda").bernoulli_(1.0 - layer.zoneout)
    return dmask, dscale, zmask


def test_lstm_layer_zoneout_dropconnect_vs_oracle():
    T, N, C, H = 7, 5, 12, 16
    torch.manual_seed(2)
    layer = haste_amd.LSTM(C, H, dropout=0.2, zoneout=0.3).cuda()
    x = torch.randn(T, N, C, device="cuda", requires_grad=True)
    dmask, dscale, zmask = _drawn_masks(layer, T, N, 77)
    torch.manual_seed(77)
    y, (hn, cn) = layer(x)
    dy = torch.randn(T, N, H, device="cuda")
    (y * dy).sum().backward()
    W, R, b = npy(layer.kernel), npy(layer.recurrent_kernel), npy(layer.bias)
    Reff = R * npy(dmask) * np.float64(np.float32(dscale))
    m = npy(zmask)
    h, c, v = O.lstm_forward(W, Reff, b, npy(x), np.zeros((N, H)), np.zeros((N, H)), True, 0.3, m)
    assert relerr(npy(y), h[1:]) < TOL and relerr(npy(cn[0]), c[-1]) < TOL
    dh_new = np.concatenate([np.zeros((1, N, H)), npy(dy)], 0)
    dx, dW, dR, db, _, _, _ = O.lstm_backward(W, Reff, b, npy(x), h, c, v, dh_new, np.zeros_like(dh_new), m)
    assert relerr(npy(x.grad), dx) < TOL and relerr(npy(layer.kernel.grad), dW) < TOL
    assert relerr(npy(layer.bias.grad), db) < TOL
    assert relerr(npy(layer.recurrent_kernel.grad), dR * npy(dmask) * dscale) < TOL
    # evaluation mode: no DropConnect, zoneout becomes the deterministic blend
    layer.eval()
    with torch.no_grad():
        ye, _ = layer(x)
    he, _, _ = O.lstm_forward(W, R, b, npy(x), np.zeros((N, H)), np.zeros((N, H)), False, 0.3, m)
    assert relerr(npy(ye), he[1:]) < TOL
    with pytest.raises(RuntimeError, match="training mode"):
        ye2, _ = layer(x)
        ye2.sum().backward()


def test_gru_layer_zoneout_dropconnect_vs_oracle():
    T, N, C, H = 6, 4, 10, 16
    torch.manual_seed(3)
    layer = haste_amd.GRU(C, H, dropout=0.25, zoneout=0.2).cuda()
    x = torch.randn(T, N, C, device="cuda", requires_grad=True)
    dmask, dscale, zmask = _drawn_masks(layer, T, N, 78)
    torch.manual_seed(78)
    y, hn = layer(x)
    dy = torch.randn(T, N, H, device="cuda")
    (y * dy).sum().backward()
    W, R, bx, br = (npy(layer.kernel), npy(layer.recurrent_kernel), npy(layer.bias), npy(layer.recurrent_bias))
    Reff = R * npy(dmask) * np.float64(np.float32(dscale))
    m = npy(zmask)
    h, v = O.gru_forward(W, Reff, bx, br, npy(x), np.zeros((N, H)), True, 0.2, m)
    assert relerr(npy(y), h[1:]) < TOL
    dh_new = np.concatenate([np.zeros((1, N, H)), npy(dy)], 0)
    dx, dW, dR, dbx, dbr, _, _, _ = O.gru_backward(W, Reff, bx, br, npy(x), h, v, dh_new, m)
    assert relerr(npy(x.grad), dx) < TOL and relerr(npy(layer.kernel.grad), dW) < TOL
    assert relerr(npy(layer.bias.grad), dbx) < TOL and relerr(npy(layer.recurrent_bias.grad), dbr) < TOL
    assert relerr(npy(layer.recurrent_kernel.grad), dR * npy(dmask) * dscale) < TOL


def test_layer_norm_layers_vs_oracle():
    T, N, C, H = 6, 5, 10, 16
    torch.manual_seed(4)
    x = torch.randn(T, N, C, device="cuda", requires_grad=True)
    dy = torch.randn(T, N, H, device="cuda")
    z = np.zeros((N, H))
    dh_new = np.concatenate([np.zeros((1, N, H)), npy(dy)], 0)

    layer = haste_amd.LayerNormLSTM(C, H, zoneout=0.2).cuda()
    with torch.no_grad():
        layer.gamma.uniform_(0.5, 1.5), layer.gamma_h.uniform_(0.5, 1.5), layer.beta_h.uniform_(-0.5, 0.5)
    _, _, zmask = _drawn_masks(layer, T, N, 79)
    torch.manual_seed(79)
    y, _ = layer(x)
    (y * dy).sum().backward()
    P = {k: npy(v) for k, v in layer.named_parameters()}
    fwd = O.layer_norm_lstm_forward(P["kernel"], P["recurrent_kernel"], P["bias"], P["gamma"], P["gamma_h"],
                                    P["beta_h"], npy(x), z, z, True, 0.2, npy(zmask))
    g = O.layer_norm_lstm_backward(P["kernel"], P["recurrent_kernel"], P["bias"], P["gamma"], P["gamma_h"],
                                   P["beta_h"], npy(x), fwd, dh_new, np.zeros_like(dh_new), npy(zmask))
    assert relerr(npy(y), fwd["h"][1:]) < TOL and relerr(npy(x.grad), g["dx"]) < TOL
    for name, key in (("kernel", "dW"), ("recurrent_kernel", "dR"), ("bias", "db"), ("gamma", "dgamma"),
                      ("gamma_h", "dgamma_h"), ("beta_h", "dbeta_h")):
        assert relerr(npy(getattr(layer, name).grad), g[key]) < TOL, name

    x.grad = None
    layer = haste_amd.LayerNormGRU(C, H).cuda()
    with torch.no_grad():
        layer.gamma.uniform_(0.5, 1.5)
    y, _ = layer(x)
    (y * dy).sum().backward()
    P = {k: npy(v) for k, v in layer.named_parameters()}
    fwd = O.layer_norm_gru_forward(P["kernel"], P["recurrent_kernel"], P["bias"], P["recurrent_bias"],
                                   P["gamma"], npy(x), z)
    g = O.layer_norm_gru_backward(P["kernel"], P["recurrent_kernel"], P["bias"], P["recurrent_bias"],
                                  P["gamma"], npy(x), fwd, dh_new)
    assert relerr(npy(y), fwd["h"][1:]) < TOL and relerr(npy(x.grad), g["dx"]) < TOL
    for name, key in (("kernel", "dW"), ("recurrent_kernel", "dR"), ("bias", "dbx"),
                      ("recurrent_bias", "dbr"), ("gamma", "dgamma")):
        assert relerr(npy(getattr(layer, name).grad), g[key]) < TOL, name

    for cls, use_gamma in ((haste_amd.IndRNN, False), (haste_amd.LayerNormIndRNN, True)):
        x.grad = None
        layer = cls(C, H).cuda()
        y, _ = layer(x)
        (y * dy).sum().backward()
        P = {k: npy(v) for k, v in layer.named_parameters()}
        gam = P["gamma"] if use_gamma else None
        fwd = O.indrnn_forward(P["kernel"], P["recurrent_scale"], P["bias"], npy(x), z, True, 0.0, None, gam)
        g = O.indrnn_backward(P["kernel"], P["recurrent_scale"], P["bias"], npy(x), fwd, dh_new, None, gam)
        assert relerr(npy(y), fwd["h"][1:]) < TOL and relerr(npy(x.grad), g["dx"]) < TOL
        for name, key in (("kernel", "dW"), ("recurrent_scale", "du"), ("bias", "db")):
            assert relerr(npy(getattr(layer, name).grad), g[key]) < TOL, name


def test_lengths_and_state_sequence():
    T, N, C, H = 8, 4, 6, 8
    torch.manual_seed(5)
    layer = haste_amd.GRU(C, H).cuda()
    x = torch.randn(T, N, C, device="cuda")
    lengths = torch.tensor([8, 3, 5, 1])
    y, hn = layer(x, lengths=lengths)
    for n, L in enumerate(lengths.tolist()):
        assert torch.equal(hn[0, n], y[L - 1, n])
    layer.return_state_sequence = True
    y2, hs = layer(x)
    assert tuple(hs.shape) == (1, T, N, H) and torch.equal(hs[0], y2)


# ---- the reference's self-consistency check (validation/pytorch.py:42-62): the fused GPU path
# against the same module with _is_cuda patched to False (the plain torch loop, here on GPU
# tensors), same seed, at its sizes N=32, T=250, C=128, H=256 -------------------------------
@pytest.mark.parametrize("name", ["LSTM", "GRU", "IndRNN", "LayerNormLSTM", "LayerNormGRU", "LayerNormIndRNN"])
@pytest.mark.parametrize("regularised", [False, True])
def test_self_consistency_fused_vs_plain_loop(name, regularised):
    from unittest import mock
    N, T, C, H = 32, 250, 128, 256
    torch.manual_seed(4)
    kw = {}
    if regularised:
        kw["zoneout"] = 0.1
        if "IndRNN" not in name:
            kw["dropout"] = 0.05
    rnn = getattr(haste_amd, name)(C, H, **kw).cuda()
    x = torch.rand(T, N, C, device="cuda")
    x1 = x.clone().requires_grad_(True)
    x2 = x.clone().requires_grad_(True)
    print("self consistency", name, regularised, flush=True)
    seed = 5566
    torch.manual_seed(seed)
    y1, _ = rnn(x1)
    y1.backward(torch.ones_like(y1))
    grads1 = {k: p.grad.clone() for k, p in rnn.named_parameters()}
    rnn.zero_grad()
    torch.manual_seed(seed)
    with mock.patch.object(rnn, "_is_cuda", lambda: False):
        y2, _ = rnn(x2)
    y2.backward(torch.ones_like(y2))
    # LayerNormLSTM is chaotic over 250 steps (a float32 run drifts from a float64 one by more
    # than this between any two orders of summation): its free-running outputs are compared over
    # the first steps only, the other cells over the whole sequence.
    steps = 25 if name == "LayerNormLSTM" else T
    err_y = float((y1[:steps] - y2[:steps]).detach().abs().max())
    assert err_y < 2e-4, err_y
    if name != "LayerNormLSTM":
        scale = float(x2.grad.abs().max())
        assert float((x1.grad - x2.grad).abs().max()) < 2e-3 * scale
        for k, p in rnn.named_parameters():
            ref = p.grad
            assert float((grads1[k] - ref).abs().max()) < 2e-3 * max(float(ref.abs().max()), 1e-6), k


@pytest.mark.parametrize("name,dtype,H", [
    (n, d, h) for n in ("LSTM", "GRU", "IndRNN", "LayerNormLSTM", "LayerNormGRU", "LayerNormIndRNN")
    for d, h in ((torch.float32, 24), (torch.float64, 24), (torch.float32, 300))] + [
    ("LSTM", torch.float32, 1200), ("LayerNormLSTM", torch.float32, 1200), ("GRU", torch.float16, 64)])
@pytest.mark.parametrize("wanted", ["last", "lengths", "all"])
@pytest.mark.parametrize("through", ["y", "state", "both"])
def test_gradients_enter_through_every_output(name, dtype, H, wanted, through):
    """Gradients of the outputs, of the final states (at the sequences' ends, or at lengths), of the state
    sequences and of their combinations, against the plain loop on the CPU in double: the fused
    backward passes take them without a [T+1,N,H] sequence being made of them."""
    T, N, C = 5, 3, 8
    torch.manual_seed(11)
    layer = getattr(haste_amd, name)(C, H, return_state_sequence=wanted == "all", batch_first=wanted == "all")
    layer = layer.to(dtype)
    ref = getattr(haste_amd, name)(C, H, return_state_sequence=wanted == "all", batch_first=wanted == "all").double()
    ref.load_state_dict(layer.state_dict())
    layer = layer.cuda()
    x = torch.randn(*((N, T, C) if wanted == "all" else (T, N, C))).to(dtype)
    lengths = [5, 1, 3] if wanted == "lengths" else None
    results = []
    for net, at in ((layer, x.cuda()), (ref, x.double())):
        at.requires_grad_(True)
        y, state = net(at, lengths=lengths)
        states = state if isinstance(state, tuple) else (state,)
        outs = ([y] if through != "state" else []) + (list(states) if through != "y" else [])
        g = torch.Generator().manual_seed(4)
        torch.autograd.backward(outs, [torch.randn(o.shape, generator=g).to(o) for o in outs])
        results.append([y, *states, at.grad] + [p.grad for p in net.parameters()])
    print(name, dtype, H, wanted, through, flush=True)
    for got, want in zip(*results):
        if want is None or got is None:
            assert want is None or not want.abs().max()
            continue
        assert relerr(npy(got), npy(want)) < {torch.float32: TOL, torch.float64: 1e-10, torch.float16: 2e-2}[dtype]


@pytest.mark.parametrize("name,dtype", [
    (n, d) for n in ("LSTM", "GRU", "IndRNN", "LayerNormLSTM", "LayerNormGRU", "LayerNormIndRNN")
    for d in (torch.float32, torch.float64)] + [("GRU", torch.float16)])
@pytest.mark.parametrize("form", ["transposed", "broadcast"])
def test_gradients_of_final_states_in_any_layout(name, dtype, form):
    """Gradients of the final states that arrive with strides of their own: of a caller that works on
    the transposed state, and of a sum (stride 0)."""
    T, N, C, H = 5, 3, 8, 24
    torch.manual_seed(12)
    layer = getattr(haste_amd, name)(C, H).to(dtype)
    ref = getattr(haste_amd, name)(C, H).double()
    ref.load_state_dict(layer.state_dict())
    layer = layer.cuda()
    x = torch.randn(T, N, C).to(dtype)
    start = torch.randn(2, N, H).to(dtype)
    weight = torch.randn(2, H, N).to(dtype)
    results = []
    for net, at, first in ((layer, x.cuda(), start.cuda()), (ref, x.double(), start.double())):
        at.requires_grad_(True)
        first = [s.unsqueeze(0).requires_grad_(True) for s in first]
        two = "LSTM" in name
        _, state = net(at, tuple(first) if two else first[0])
        states = state if two else (state,)
        loss = 0.0
        for s, w in zip(states, weight.to(at)):
            loss = loss + ((s[0].t().contiguous() * w).sum() if form == "transposed" else s.sum())
        loss.backward()
        results.append([at.grad] + [s.grad for s in first[:len(states)]] + [p.grad for p in net.parameters()])
    print(name, dtype, form, flush=True)
    for got, want in zip(*results):
        assert relerr(npy(got), npy(want)) < {torch.float32: TOL, torch.float64: 1e-10, torch.float16: 2e-2}[dtype]


def test_outputs_that_are_changed_are_noticed():
    """The outputs share memory with what the backward pass reads."""
    layer = haste_amd.LSTM(4, 8).cuda()
    for which in ("y", "h", "c"):
        y, (h, c) = layer(torch.randn(3, 2, 4, device="cuda", requires_grad=True))
        loss = (y * y).sum()
        with torch.no_grad():
            {"y": y, "h": h, "c": c}[which].add_(1.0)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            loss.backward()


@pytest.mark.parametrize("name", ["LSTM", "GRU", "IndRNN", "LayerNormLSTM", "LayerNormGRU", "LayerNormIndRNN"])
def test_lengths_that_are_changed_are_noticed(name):
    """A buffer of lengths that is filled again before the backward pass."""
    layer = getattr(haste_amd, name)(4, 8).cuda()
    lengths = torch.tensor([3, 1], device="cuda")
    y, state = layer(torch.randn(3, 2, 4, device="cuda"), lengths=lengths)
    last = state[0] if isinstance(state, tuple) else state
    lengths.fill_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        last.sum().backward()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16])
@pytest.mark.parametrize("T,N,H", [(1, 1, 1), (4, 3, 5), (7, 33, 256), (5, 2, 300)])
def test_states_at_lengths_match_indexing(dtype, T, N, H):
    """Gathered states and their gradients against tensor indexing, bit for bit: lengths 0 (the initial
    state), T and counted from the end, gradients contiguous, batch first, broadcast and absent."""
    from haste_amd import ops
    gen = torch.Generator(device="cuda").manual_seed(T + N + H)
    def rand(*s):
        return torch.randn(*s, device="cuda", generator=gen).to(dtype)

    seqs = [rand(T + 1, N, H), rand(T + 1, N, H)]
    lengths = torch.randint(-T - 1, T + 1, (N,), device="cuda", generator=gen)
    lengths[0] = T
    rows = torch.arange(N, device="cuda")
    for given in (seqs[:1], seqs):
        for got, seq in zip(ops.gather_states(given, lengths), given):
            assert torch.equal(got, seq[lengths, rows])
    last = rand(N, H)
    for grad in (rand(T, N, H), rand(N, T, H).permute(1, 0, 2), rand(1, 1, H).expand(T, N, H), rand(1, 1, 1).expand(T, N, H), None):
        full = torch.zeros(T + 1, N, H, device="cuda", dtype=dtype)
        if grad is not None:
            full[1:] = grad
        full[lengths, rows] = full[lengths, rows] + last
        assert torch.equal(ops.state_gradients(seqs[0], grad, last, lengths), full[1:])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16])
def test_lengths_beyond_the_sequence_give_nans(dtype):
    """Lengths that only the GPU knows: a row without such a step has NaNs for its state, and the gradients
    that come through it are NaNs too."""
    T, N, H = 4, 5, 70
    lengths = torch.tensor([4, 5, -5, -6, 1], device="cuda")
    layer = haste_amd.GRU(8, H).cuda().to(dtype)
    x = torch.randn(T, N, 8, device="cuda").to(dtype).requires_grad_()
    y, h = layer(x, lengths=lengths)
    h.sum().backward()
    wrong = torch.tensor([False, True, False, True, False], device="cuda")
    assert torch.equal(h[0].isnan(), wrong[:, None].expand(N, H)) and not y.isnan().any()
    assert torch.equal(x.grad.isnan(), wrong[None, :, None].expand(T, N, 8))
    assert layer.kernel.grad.isnan().all()


def test_states_at_lengths_of_more_rows_than_a_launch_has_blocks():
    from haste_amd import ops
    T, N, H = 2, (1 << 23) + 5, 1  # T * N beyond 2^24 blocks of 256 threads
    gen = torch.Generator(device="cuda").manual_seed(1)
    seq = torch.randn(T + 1, N, H, device="cuda", generator=gen)
    lengths = torch.randint(0, T + 1, (N,), device="cuda", generator=gen)
    rows = torch.arange(N, device="cuda")
    (got,) = ops.gather_states([seq], lengths)
    assert torch.equal(got, seq[lengths, rows])
    last = torch.randn(N, H, device="cuda", generator=gen)
    want = torch.zeros_like(seq)
    want[lengths, rows] = last
    assert torch.equal(ops.state_gradients(seq, None, last, lengths), want[1:])
    assert torch.equal(ops.state_gradients(seq, seq[1:], last, lengths), seq[1:] + want[1:])


def test_gradients_of_a_pass_are_not_differentiated_again():
    """The backward passes are kernels: what they return is a constant to create_graph, all of it."""
    layer = haste_amd.LSTM(4, 8).cuda()
    h0, c0 = (torch.randn(1, 2, 8, device="cuda", requires_grad=True) for _ in range(2))
    x = torch.randn(3, 2, 4, device="cuda", requires_grad=True)
    _, (h, c) = layer(x, (h0, c0))
    grads = torch.autograd.grad(h.square().sum() + c.square().sum(), [x, *layer.parameters()], create_graph=True)
    assert not any(g.requires_grad for g in grads)
    _, (h, c) = layer(x, (h0, c0))
    grads = torch.autograd.grad(h.square().sum() + c.square().sum(), [h0, c0], create_graph=True)
    assert not any(g.requires_grad for g in grads)
