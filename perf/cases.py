"""The workloads whose speed is tracked: the recurrent layers as a program that uses them calls
them, over the sizes, directions, data types and options they are used with.

Sizes come from bench.py (its headline and the other configurations), haste_amd/benchmark_grid.py
(batch 1 .. 128, hidden 128 .. 4096, input 64 .. 512), the IndRNN speed script's shape and the
ragged shapes of the tests.  A case is a dict:

  cell     the layer: lstm, gru, indrnn, layer_norm_lstm, layer_norm_gru, layer_norm_indrnn
  mode     "train": forward and backward pass; "infer": forward pass without gradients;
           "step": one single step (lstm and gru), the state handed over by the caller
  dtype    float32, float64, or for the gru float16
  T, N, C, H   time steps, batch rows, input size, hidden size
  zoneout, dropout   the layers' probabilities (dropout acts on the recurrent matrix)
  lengths  the batch's sequences have lengths of their own and the final state is used
  batch_first   the input is [N, T, C] instead of [T, N, C]
"""
import math

import torch

from haste_amd import layers, ops

_LAYERS = {"lstm": layers.LSTM, "gru": layers.GRU, "indrnn": layers.IndRNN,
           "layer_norm_lstm": layers.LayerNormLSTM, "layer_norm_gru": layers.LayerNormGRU,
           "layer_norm_indrnn": layers.LayerNormIndRNN}
_DTYPES = {"float32": torch.float32, "float64": torch.float64, "float16": torch.float16}


def _case(cell, mode, T, N, C, H, dtype="float32", zoneout=0.0, dropout=0.0, lengths=False,
          batch_first=False, **name):
    return dict(name, cell=cell, mode=mode, dtype=dtype, T=T, N=N, C=C, H=H, zoneout=zoneout,
                dropout=dropout, lengths=lengths, batch_first=batch_first)


def listed():
    return [
        # A streaming recogniser or a sampler's inner loop: one step per call, nothing to batch.
        _case("lstm", "step", 1, 1, 512, 512, name="lstm_step_n1"),
        # One long utterance at a time through a layer that is already trained.
        _case("lstm", "infer", 2000, 1, 512, 512, name="lstm_infer_n1_long"),
        # A small serving batch of sequences of different lengths, padded.
        _case("lstm", "infer", 100, 16, 128, 256, lengths=True, name="lstm_infer_small_batch"),
        # The ordinary training step: the size the benchmark's headline is quoted at.
        _case("lstm", "train", 100, 64, 512, 512, name="lstm_train"),
        # The same layer at twice the batch, the largest of the benchmark's grid.
        _case("lstm", "train", 100, 128, 512, 512, name="lstm_train_n128"),
        # A regularised training step: zoneout on the state, DropConnect on the recurrent matrix.
        _case("gru", "train", 100, 64, 512, 512, zoneout=0.1, dropout=0.05, name="gru_train_regularised"),
        # Features and vocabulary sizes are seldom powers of two; nor is the last batch full.
        _case("gru", "train", 83, 37, 75, 300, lengths=True, batch_first=True, name="gru_train_ragged"),
        # Training with tensors kept in half precision.
        _case("gru", "train", 100, 64, 512, 512, dtype="float16", zoneout=0.1, name="gru_train_half"),
        # Training in double precision, where float's rounding is too coarse.
        _case("lstm", "train", 100, 64, 512, 512, dtype="float64", name="lstm_train_double"),
        # A layer-normalised cell over long sequences at a moderate width.
        _case("layer_norm_lstm", "train", 500, 32, 256, 256, zoneout=0.1, name="layer_norm_lstm_train"),
        # A wide layer: the recurrent matrix (64 MiB) no longer stays on the chip.
        _case("lstm", "train", 50, 64, 512, 2048, name="lstm_train_wide"),
        # Very long sequences through a wide elementwise recurrence, the speed script's shape.
        _case("indrnn", "train", 2500, 64, 256, 4096, name="indrnn_train_long"),
    ]


def _spread(rng, low, high):
    """A whole number between low and high, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    cell = rng.choice(["lstm", "lstm", "lstm", "gru", "gru", "gru", "layer_norm_lstm", "layer_norm_gru",
                       "indrnn", "layer_norm_indrnn"])
    mode = rng.choice(["train", "train", "infer"] + (["step"] if cell in ("lstm", "gru") else []))
    dtype = rng.choice(["float32"] * 4 + ["float64"] + (["float16"] if cell == "gru" else []))
    while True:
        N, C = _spread(rng, 1, 128), _spread(rng, 32, 512)
        wide = cell.endswith("indrnn") or mode != "train"
        H = _spread(rng, 64, 4096 if wide and cell in ("lstm", "gru", "indrnn") else 2048)
        T = 1 if mode == "step" else _spread(rng, 20, 500)
        if rng.random() < 0.5:  # widths that a configuration file would have
            C, H = max(32, C // 32 * 32), max(64, H // 64 * 64)
        if dtype == "float64" and mode != "step":
            H, T = min(H, 768), min(T, 100)
        case = _case(cell, mode, T, N, C, H, dtype=dtype)
        if work(case)["flops"] <= 3e11 and (H <= 1024 or T <= 100 or cell.endswith("indrnn")):
            break
    if mode == "train":
        case["zoneout"] = rng.choice([0.0, 0.1])
        case["dropout"] = rng.choice([0.0, 0.05]) if not cell.endswith("indrnn") else 0.0
    if mode != "step":
        case["lengths"] = rng.random() < 0.25
        case["batch_first"] = rng.random() < 0.25
    return case


def prepare(case, seed):
    dtype, dev = _DTYPES[case["dtype"]], torch.device("cuda")
    T, N, C, H = case["T"], case["N"], case["C"], case["H"]
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device=dev, dtype=torch.float32).to(dtype)

    options = {"dropout": case["dropout"]} if case["dropout"] else {}
    with torch.device("meta"):  # the values come from `gen` below
        layer = _LAYERS[case["cell"]](C, H, batch_first=case["batch_first"], zoneout=case["zoneout"], **options)
    layer = layer.to(dtype).to_empty(device=dev)
    with torch.no_grad():
        for name, p in layer.named_parameters():
            # The scale of torch.nn's recurrent layers; gains around the value they start at.
            p.uniform_(-H ** -0.5, H ** -0.5, generator=gen)
            if name == "gamma" and case["cell"] == "layer_norm_lstm":
                # The gain recurrent normalisation is usually started from. At 1 this cell's state is
                # chaotic: after 500 steps two roundings of the same sums have nothing in common.
                p.add_(0.1)
            elif name.startswith("gamma"):
                p.add_(1.0)
            elif name == "recurrent_scale":
                p.mul_(0.5 * H ** 0.5)
            elif name == "bias" and "lstm" in case["cell"]:
                p[2 * H:3 * H].add_(1.0)  # the layers' forget bias
    state = {"case": case, "seed": seed, "layer": layer}
    if case["mode"] == "step":
        state["x"] = normal(N, C)
        state["h"], state["c"] = (0.5 * normal(N, H)).tanh(), normal(N, H)
        return state
    layer.train(case["mode"] == "train")
    first, second = (N, T) if case["batch_first"] else (T, N)
    state["x"] = normal(first, second, C)
    state["lengths"] = torch.randint(max(1, T // 2), T + 1, (N,), generator=gen, device=dev) if case["lengths"] else None
    if case["mode"] == "train":
        state["x"].requires_grad_(True)  # the output of the layer before it
        state["dy"] = normal(first, second, H)
        state["dh"] = normal(1, N, H) if case["lengths"] else None
    return state


def run(state):
    case, layer, x = state["case"], state["layer"], state["x"]
    if case["mode"] == "step":
        with torch.no_grad():
            if case["cell"] == "lstm":
                return ops.lstm_forward_iterate(False, 0.0, x, state["h"], state["c"], layer.kernel,
                                                layer.recurrent_kernel, layer.bias)[:2]
            return ops.gru_forward_iterate(False, 0.0, x, state["h"], layer.kernel, layer.recurrent_kernel,
                                           layer.bias, layer.recurrent_bias)[0]
    if case["mode"] == "infer":
        with torch.no_grad():
            return layer(x, lengths=state["lengths"])
    if case["zoneout"] or case["dropout"]:
        torch.manual_seed(state["seed"])  # the layers draw their masks from torch's generator
    layer.zero_grad(set_to_none=True)
    x.grad = None
    y, last = layer(x, lengths=state["lengths"])
    h_n = last[0] if isinstance(last, tuple) else last
    if state["dh"] is None:
        y.backward(state["dy"])
    else:
        torch.autograd.backward([y, h_n], [state["dy"], state["dh"]])
    grads = {name: p.grad for name, p in layer.named_parameters()}
    return {"y": y.detach(), "h_n": h_n.detach(), "dx": x.grad, "grads": grads}


def work(case):
    T, N, C, H = case["T"], case["N"], case["C"], case["H"]
    size = {"float32": 4, "float64": 8, "float16": 2}[case["dtype"]]
    gates = 4 if case["cell"].endswith("lstm") else 3 if case["cell"].endswith("gru") else 1
    recurrent = 0 if case["cell"].endswith("indrnn") else H * gates * H
    weights = C * gates * H + recurrent + 2 * gates * H
    flops = 2 * T * N * (C * gates * H + recurrent)
    values = T * N * C + weights + T * N * H + N * H
    if case["mode"] == "train":  # each product has two in the backward pass; dy in, dx and the weights' gradients out
        flops *= 3
        values += T * N * H + T * N * C + weights
    return {"bytes": values * size, "flops": flops}


def tolerance(case):
    # About four times what the float passes differ by from the same passes in float64 (half: in
    # float32) and from passes with the hidden units in another order, over these cases and draws:
    # double 1.4e-15 (one value: 1.1e-14), float 1.4e-6 (1.7e-5), half 4.3e-4 (2.9e-3), the chained
    # norms of the layer_norm_lstm over 500 steps 1.1e-5 (1.7e-4).
    if case["dtype"] == "float64":
        scale = 10 if case["cell"] == "layer_norm_lstm" else 1
        return {"rel": 6e-15 * scale, "max": 5e-14 * scale}
    if case["dtype"] == "float16":
        return {"rel": 2e-3, "max": 1.2e-2}
    return {"rel": 4e-5, "max": 7e-4} if case["cell"] == "layer_norm_lstm" else {"rel": 5e-6, "max": 7e-5}
