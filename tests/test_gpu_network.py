"""GPU tests of the C++ network sequencer (cnt_network_*): a network file in the reference's JSON structure is
turned into the layer list, and forward pass, error, backward pass and optimizer step of a fraction are compared
with the CPU oracle doing the same steps.  Tolerance 1e-4 on L2-normalised differences (fp32, different summation
orders), the tolerance of the layer kernels themselves."""
import itertools
import json

import numpy as np
import pytest

import oracle_lib as O
import oracle_models as OM
import parity_cases as PC
import synth as WD
from torch_models import make_pat_types

pytestmark = pytest.mark.gpu
TOL = 1e-4


def _sections(doc_weights, name, w, n_in, n_bias):
    doc_weights[name] = {"input": w[:n_in].tolist(), "bias": w[n_in:n_in + n_bias].tolist(),
                         "internal": w[n_in + n_bias:].tolist()}


@pytest.mark.parametrize("option,momentum,overlap", [(0, 0.9, True), (5, 0.0, True), (0, 0.0, False)])
def test_stacked_network_trains_like_the_oracle(option, momentum, overlap):
    import torch

    print("network case", option, momentum, overlap, flush=True)
    pkg = PC.pkg()
    capi, networks = pkg.capi, PC.networks()
    P, Q, S = 20, 6, 4
    specs = [{"name": "ff1", "type": "feedforward_tanh", "size": 32, "bias": 1.0},
             {"name": "bl1", "type": "blstm", "size": 128, "bias": 1.0},
             {"name": "l2", "type": "lstm", "size": 64, "bias": 1.0},
             {"name": "out", "type": "feedforward_identity", "size": Q, "bias": 1.0},
             {"name": "postoutput", "type": "sse", "size": Q}]
    weights = OM.init_weights(P, specs, 4, 0.1)
    doc = {"layers": [{"size": P, "name": "input", "type": "input"}] + specs, "weights": {}}
    wi, prev = iter(weights), P
    for sp in specs:
        n_in, n_bias, _ = networks.weight_sections(sp, prev)
        if n_in:
            _sections(doc["weights"], sp["name"], next(wi), n_in, n_bias)
        prev = sp["size"]
    maxT = 30
    net = capi.Network(json.dumps(doc, indent=1), S, maxT, overlap=overlap)
    assert net.input_size == P and net.output_size == Q and net.n_weights == sum(w.size for w in weights)
    assert [L["type"] for L in net.layers] == ["input"] + [s["type"] for s in specs]
    for L, w in zip([L for L in net.layers if L["weight_count"]], weights):
        assert np.array_equal(L["weights"].cpu().numpy(), w)

    rng = np.random.default_rng(6)
    ow = [w.copy() for w in weights]
    deltas = [np.zeros_like(w) for w in ow]
    stats = [np.zeros(2 * w.size, np.float32) for w in ow]
    b1 = b2 = 1.0
    for step, lengths in enumerate(([30, 22, 13, 9], [17, 26, 28, 11], [19, 24, 8, 15])):
        T, Tmin = max(lengths), min(lengths)
        pat = make_pat_types(lengths, T)
        x = rng.standard_normal((T, S, P)).astype(np.float32)
        tgt = (0.3 * rng.standard_normal((T, S, Q))).astype(np.float32)
        valid = (pat != 0).reshape(T, S)
        x[~valid] = 0
        tgt[~valid] = 0
        net.load_sequences(PC.dev(pat), T, Tmin, PC.dev(x.reshape(-1)), PC.dev(tgt.reshape(-1)))
        net.forward()
        loss = float(net.calculate_error().item())
        net.backward()
        ref = OM.OracleNetwork(P, specs, S, T, Tmin, pat, ow)
        ref.forward(x.reshape(-1), tgt.reshape(-1))
        assert abs(loss - ref.error()) <= TOL * max(1.0, abs(ref.error()))
        ref.backward()
        grads = [L["updates"] for L in ref.layers if "updates" in L]
        torch.cuda.synchronize()
        for L, g in zip([L for L in net.layers if L["weight_count"]], grads):
            assert PC.relerr(L["updates"].cpu().numpy(), g) < TOL, (step, L["name"])
        frac = float(sum(lengths))
        net.update(option, 1e-3, momentum, frac)
        if option == 5:
            b1 = O.opt_next_beta_accum(b1, 1)
            b2 = O.opt_next_beta_accum(b2, 2)
        for w, g, d, st in zip(ow, grads, deltas, stats):
            cur = np.empty_like(g)
            O.opt_accumulate(g, cur, False)
            O.opt_adjust_gradient(option, cur, st, None, frac, b1, b2)
            O.opt_update_weights(w, cur, d, None, 1e-3, momentum)
    net.check()
    got = [L["weights"].cpu().numpy() for L in net.layers if L["weight_count"]]
    for g, w, w0 in zip(got, ow, weights):
        assert PC.relerr(g, w) < TOL
        assert PC.relerr(g, w0) > 1e-5  # the weights did move
    # export and re-import: same layers, bit-identical weights
    text = net.export_json()
    back = json.loads(text)
    assert [l["name"] for l in back["layers"]] == ["input"] + [s["name"] for s in specs]
    assert back["layers"][2] == specs[1]
    again = capi.Network(text, S, maxT)
    assert np.array_equal(again.weights.cpu().numpy(), net.weights.cpu().numpy())
    again.close()
    net.close()


def test_weight_gradients_of_a_fraction_that_is_mostly_padding():
    """One long sequence beside seven of a single frame: the weight gradients sum over the valid slots only (a list of them,
    made when the fraction is loaded), a recurrent layer's recurrent weights over the list without the first or the last
    time step, and most splits of the narrow layers' split-K products are left without a single slot."""
    import torch

    print("network case: mostly padding", flush=True)
    capi, networks = PC.pkg().capi, PC.networks()
    P, Q, S, T = 16, 8, 8, 600
    lengths = [T, 1, 1, 1, 1, 1, 1, 1]
    specs = [{"name": "ff1", "type": "feedforward_tanh", "size": 64, "bias": 1.0},
             {"name": "bl1", "type": "blstm", "size": 128, "bias": 1.0},
             {"name": "out", "type": "feedforward_identity", "size": Q, "bias": 1.0},
             {"name": "postoutput", "type": "sse", "size": Q}]
    weights = OM.init_weights(P, specs, 9, 0.1)
    doc = {"layers": [{"size": P, "name": "input", "type": "input"}] + specs, "weights": {}}
    wi, prev = iter(weights), P
    for sp in specs:
        n_in, n_bias, _ = networks.weight_sections(sp, prev)
        if n_in:
            _sections(doc["weights"], sp["name"], next(wi), n_in, n_bias)
        prev = sp["size"]
    net = capi.Network(json.dumps(doc), S, T)
    rng = np.random.default_rng(10)
    # a fraction without padding first: every split of the split-K products leaves its partial sums in the scratch buffer,
    # where a split of the next pass that wrote nothing would let them be counted again
    full = make_pat_types([T] * S, T)
    net.load_sequences(PC.dev(full), T, T, PC.dev(rng.standard_normal(T * S * P).astype(np.float32)),
                       PC.dev(rng.standard_normal(T * S * Q).astype(np.float32)))
    net.forward()
    net.backward()
    pat = make_pat_types(lengths, T)
    x = rng.standard_normal((T, S, P)).astype(np.float32)
    tgt = (0.3 * rng.standard_normal((T, S, Q))).astype(np.float32)
    valid = (pat != 0).reshape(T, S)
    x[~valid] = 0
    tgt[~valid] = 0
    net.load_sequences(PC.dev(pat), T, 1, PC.dev(x.reshape(-1)), PC.dev(tgt.reshape(-1)))
    net.forward()
    net.backward()
    net.check()
    ref = OM.OracleNetwork(P, specs, S, T, 1, pat, [w.copy() for w in weights])
    ref.forward(x.reshape(-1), tgt.reshape(-1))
    ref.backward()
    grads = [L["updates"] for L in ref.layers if "updates" in L]
    torch.cuda.synchronize()
    for L, g in zip([L for L in net.layers if L["weight_count"]], grads):
        assert PC.relerr(L["updates"].cpu().numpy(), g) < TOL, L["name"]
    net.close()


@pytest.mark.parametrize("lengths", [(400, 250, 3), (353, 352, 352)])
def test_weight_gradients_of_wide_dense_layers(lengths):
    """1024 x 1028 weights in three splits of 64 x 64 tiles, with the fraction's valid slots or all of them as the inner dimension."""
    import torch

    print("network case: wide dense layers", lengths, flush=True)
    capi, networks = PC.pkg().capi, PC.networks()
    P, Q, S, T = 20, 8, 3, lengths[0]
    specs = [{"name": "ff1", "type": "feedforward_tanh", "size": 1024, "bias": 1.0},
             {"name": "ff2", "type": "feedforward_logistic", "size": 1028, "bias": 0.5},
             {"name": "out", "type": "feedforward_identity", "size": Q, "bias": 1.0},
             {"name": "postoutput", "type": "sse", "size": Q}]
    weights = OM.init_weights(P, specs, 19, 0.1)
    doc = {"layers": [{"size": P, "name": "input", "type": "input"}] + specs, "weights": {}}
    wi, prev = iter(weights), P
    for sp in specs:
        n_in, n_bias, _ = networks.weight_sections(sp, prev)
        if n_in:
            _sections(doc["weights"], sp["name"], next(wi), n_in, n_bias)
        prev = sp["size"]
    net = capi.Network(json.dumps(doc), S, T)
    rng = np.random.default_rng(20)
    pat = make_pat_types(list(lengths), T)
    x = rng.standard_normal((T, S, P)).astype(np.float32)
    tgt = (0.3 * rng.standard_normal((T, S, Q))).astype(np.float32)
    valid = (pat != 0).reshape(T, S)
    x[~valid] = 0
    tgt[~valid] = 0
    net.load_sequences(PC.dev(pat), T, min(lengths), PC.dev(x.reshape(-1)), PC.dev(tgt.reshape(-1)))
    net.forward()
    net.backward()
    net.check()
    ref = OM.OracleNetwork(P, specs, S, T, min(lengths), pat, [w.copy() for w in weights])
    ref.forward(x.reshape(-1), tgt.reshape(-1))
    ref.backward()
    grads = [L["updates"] for L in ref.layers if "updates" in L]
    torch.cuda.synchronize()
    for L, g in zip([L for L in net.layers if L["weight_count"]], grads):
        assert PC.relerr(L["updates"].cpu().numpy(), g) < TOL, L["name"]
    net.close()


@pytest.mark.parametrize("lengths", [(2000, 1900, 1801), (2000, 30, 1), (2000, 2000, 2000)])
def test_weight_gradients_of_large_tiles_over_listed_slots(lengths):
    """1024 x 1028 weights over 6000 slots on eight waves, bias gradient included, through the list of valid slots: a last tile and a
    last split that are not full, splits that the list leaves empty, no padding at all.  Against 64-bit sums of the network's own
    inputs and deltas, within the bound of fp32 sums in any order; the same bits in a second pass."""
    import torch

    print("network case: large tiles over listed slots", lengths, flush=True)
    capi = PC.pkg().capi
    P, Q, S, T, bias = 20, 8, 3, lengths[0], 0.5
    N = S * T
    assert capi.probe_gemm_plan(1024, 1028, N, weight_gradient=True)[:2] == (128, 8)
    layers = [{"size": P, "name": "input", "type": "input"}, {"name": "ff1", "type": "feedforward_tanh", "size": 1024, "bias": 1.0},
              {"name": "ff2", "type": "feedforward_logistic", "size": 1028, "bias": bias},
              {"name": "out", "type": "feedforward_identity", "size": Q, "bias": 1.0}, {"name": "postoutput", "type": "sse", "size": Q}]
    net = capi.Network(json.dumps({"layers": layers}), S, T)
    net.randomize(3, 0.1)
    gen = torch.Generator(device="cuda").manual_seed(4)
    pat = PC.dev(make_pat_types(list(lengths), T))
    live = (pat != 0).view(N, 1)
    x, tgt = torch.randn(N, P, device="cuda", generator=gen) * live, torch.randn(N, Q, device="cuda", generator=gen) * live
    got = []
    for _ in range(2):
        net.load_sequences(pat, T, min(lengths), x.reshape(-1), tgt.reshape(-1))
        net.updates.fill_(float("nan"))
        net.forward()
        net.backward()
        torch.cuda.synchronize()
        got.append(net.layer("ff2")["updates"].clone())
    assert torch.equal(got[0], got[1])
    below, delta = net.layer("ff1")["outputs"].view(N, 1024).double() * live, net.layer("ff2")["errors"].view(N, 1028).double()
    assert not bool((delta * ~live).any())
    want = torch.cat([(delta.t() @ below).reshape(-1), bias * delta.sum(0)])
    size = torch.cat([(delta.abs().t() @ below.abs()).reshape(-1), bias * delta.abs().sum(0)])
    assert bool(((got[0] - want).abs() <= (N + 2) * 2.0 ** -24 * size).all())
    net.close()


@pytest.mark.parametrize("layers,S,T", [
    ([("feedforward_tanh", 32), ("blstm", 128)], 4, 30),                                  # in line
    ([("feedforward_tanh", 16), ("lstm", 16)], 1, 2048), ([("feedforward_tanh", 16), ("lstm", 16)], 1, 2049),  # either side of the slots
    ([("blstm", 512), ("blstm", 512)], 8, 170), ([("blstm", 512), ("blstm", 512)], 8, 176),  # 2.9e9 and 3.1e9 multiply-adds
    ([("feedforward_logistic", 1300), ("feedforward_tanh", 1300)], 8, 206), ([("feedforward_logistic", 1300), ("feedforward_tanh", 1300)], 8, 222)])
def test_weight_halves_on_other_streams_and_in_line(layers, S, T):
    """Where the weight halves of a pass run is the sequencer's choice: the gradients, and those of a second pass over other
    lengths, are the ones of a network told to use the caller's stream alone.  (The products sum over the same slots in the same
    tiles but for batches of one shape, 2^-24 per addition over at most a tile's chain: 1e-6.)"""
    import torch

    print("weight halves", layers, S, T, flush=True)
    capi = PC.pkg().capi
    P, Q = 30, 7
    doc = {"layers": [{"size": P, "name": "input", "type": "input"}] +
           [{"size": n, "name": "l%d" % i, "type": t, "bias": 1.0} for i, (t, n) in enumerate(layers)] +
           [{"size": Q, "name": "out", "type": "feedforward_identity", "bias": 1.0}, {"size": Q, "name": "post", "type": "sse"}]}
    nets = [capi.Network(json.dumps(doc), S, T, overlap=overlap) for overlap in (True, False)]
    gen = torch.Generator(device="cuda").manual_seed(3)
    nets[0].weights.uniform_(-0.1, 0.1, generator=gen)
    nets[1].weights.copy_(nets[0].weights)
    for shortest in (T, max(1, T // 3)):
        lengths = [T - (T - shortest) * i // max(1, S - 1) for i in range(S)]
        pat = PC.dev(make_pat_types(lengths, T))
        valid = (pat != 0).reshape(-1, 1)
        x = (torch.randn(S * T, P, device="cuda", generator=gen) * valid).reshape(-1)
        target = (torch.randn(S * T, Q, device="cuda", generator=gen) * valid).reshape(-1)
        updates = []
        for net in nets:
            net.load_sequences(pat, T, min(lengths), x, target)
            net.forward()
            net.calculate_error()
            net.backward()
            updates.append(net.updates.clone())
        torch.cuda.synchronize()
        assert float(updates[1].norm()) > 0
        assert float((updates[0] - updates[1]).norm()) <= 1e-6 * float(updates[1].norm())
    for net in nets:
        net.close()


@pytest.mark.parametrize("lengths,count", [([30, 22, 13, 9], 3), ([30, 30], 3), ([17, 5, 1], 36), ([700, 650, 600], 5), ([1], 34)])
def test_weight_gradients_of_a_small_pass_in_one_launch(lengths, count):
    """Layers of other sizes, more of them than a launch holds, over listed slots and over all: every gradient against the 64-bit
    product of the layer's inputs and deltas, bound of a sum in any order as for the products alone."""
    import torch

    print("one launch of gradients", lengths, count, flush=True)
    capi = PC.pkg().capi
    S, T, P, Q = len(lengths), max(lengths), 33, 6
    sizes = [(5, 64, 31, 96, 4, 130)[i % 6] for i in range(count)]
    doc = {"layers": [{"size": P, "name": "input", "type": "input"}] +
           [{"size": n, "name": "l%d" % i, "type": "feedforward_tanh", "bias": 0.8} for i, n in enumerate(sizes)] +
           [{"size": Q, "name": "out", "type": "feedforward_identity", "bias": 1.0}, {"size": Q, "name": "post", "type": "sse"}]}
    net = capi.Network(json.dumps(doc), S, T)
    gen = torch.Generator(device="cuda").manual_seed(count)
    net.weights.uniform_(-0.3, 0.3, generator=gen)
    pat = PC.dev(make_pat_types(lengths, T))
    valid = (pat != 0).reshape(-1, 1)
    x = (torch.randn(S * T, P, device="cuda", generator=gen) * valid).reshape(-1)
    target = (torch.randn(S * T, Q, device="cuda", generator=gen) * valid).reshape(-1)
    net.load_sequences(pat, T, min(lengths), x, target)
    net.forward()
    net.calculate_error()
    net.updates.fill_(7.0)
    net.backward()
    torch.cuda.synchronize()
    below, at = x.double().reshape(S * T, P), 0
    for i, n in enumerate(sizes + [Q]):
        name = "l%d" % i if i < count else "out"
        layer = net.layer(name)
        delta = layer["errors"].double().reshape(S * T, n)
        bias = 0.8 if i < count else 1.0
        w = below.shape[1] * n
        got, got_bias = net.updates[at:at + w].double().reshape(n, -1), net.updates[at + w:at + w + n].double()
        k = 2.0 ** -24 * (S * T + 2)
        assert float(delta.abs().sum()) > 0
        assert bool(((got - delta.T.contiguous() @ below).abs() <= k * (delta.abs().T.contiguous() @ below.abs())).all()), name
        assert bool(((got_bias - bias * delta.sum(0)).abs() <= k * bias * delta.abs().sum(0)).all()), name
        below, at = layer["outputs"].double().reshape(S * T, n), at + w + n
    assert at == net.n_weights
    net.close()


@pytest.mark.parametrize("sizes,lengths", [
    ([300, 700], [900, 700, 600, 500, 11]), ([299, 701], [900, 700, 600, 500, 11]), ([1024, 1028], [1700] + [900] * 6),  # three tiles
    ([512, 512], [64] * 64 + [1] * 8), ([130, 640], [3000, 1, 1]), ([1024, 1024], [2100, 1000, 1000, 1000, 1000])])
def test_errors_of_a_fraction_with_padding(sizes, lengths):
    """Products over the listed columns: the deltas that reach a layer against the 64-bit product of those above, zeros on every padding
    slot whatever stood there; column counts within, at and around tiles.  (k + 4) * 2^-24 of the terms: a sum in any order and the
    factor of the activation."""
    import torch

    print("errors with padding", sizes, lengths, flush=True)
    capi = PC.pkg().capi
    S, T, P, Q = len(lengths), max(lengths), 21, 9
    sizes = sizes + [450]
    doc = {"layers": [{"size": P, "name": "input", "type": "input"}] +
           [{"size": n, "name": "l%d" % i, "type": "feedforward_" + ("tanh", "logistic", "identity")[i % 3], "bias": 0.8} for i, n in enumerate(sizes)] +
           [{"size": Q, "name": "out", "type": "feedforward_identity", "bias": 1.0}, {"size": Q, "name": "post", "type": "sse"}]}
    net = capi.Network(json.dumps(doc), S, T)
    gen = torch.Generator(device="cuda").manual_seed(T)
    net.weights.uniform_(-0.1, 0.1, generator=gen)
    pat = PC.dev(make_pat_types(lengths, T))
    valid = (pat != 0).reshape(-1, 1)
    x = torch.randn(S * T * P, device="cuda", generator=gen)  # (anything on padding slots)
    target = (torch.randn(S * T, Q, device="cuda", generator=gen) * valid).reshape(-1)
    net.load_sequences(pat, T, min(lengths), x, target)
    net.forward()
    net.calculate_error()
    for i in range(len(sizes)):
        net.layer("l%d" % i)["errors"].fill_(7.0)
    net.backward()
    torch.cuda.synchronize()
    above = net.layer("out")
    for i in range(len(sizes) - 1, -1, -1):
        layer = net.layer("l%d" % i)
        n, m = sizes[i], above["size"]
        W = above["weights"][:n * m].double().reshape(m, n)
        delta, y = above["errors"].double().reshape(S * T, m), layer["outputs"].double().reshape(S * T, n)
        slope = (1 - y * y, y * (1 - y), torch.ones_like(y))[i % 3]
        got = layer["errors"].double().reshape(S * T, n)
        assert not bool(got[~valid[:, 0]].any()), i
        bound = (m + 4) * 2.0 ** -24 * (delta.abs() @ W.abs()) * slope.abs() + 2.0 ** -22 * (delta @ W).abs()  # (1 - y y in 32 bits)
        assert bool(((got - delta @ W * slope).abs() <= bound).all()), i
        assert float(got.abs().sum()) > 0
        above = layer
    net.close()


@pytest.mark.parametrize("sizes,lengths", [
    ((40, 64, 36), [30, 21, 8]), ((96, 130, 64), [50, 50, 3, 1]),  # products of few blocks
    ((512, 512, 512), [130, 125] + [20] * 18)])                     # in tiles
@pytest.mark.parametrize("where,value", [
    ("padding", 3e38), ("padding", float("nan")), ("padding", float("-inf")), ("valid", 2.0 ** 113), ("valid", float("nan")),
    ("target", float("nan")), ("target", 3e38)])
def test_values_without_a_split_stay_in_their_slot(sizes, lengths, where, value):
    """A fraction with padding whose products have an operand that the bf16 split has no finite parts for: on a padding slot
    nothing but that slot changes, on a valid one nothing but its own sequence and the gradients.  Blocks of sums that were infinite are summed again in
    fp32, (k + 2) * 2^-24 of the terms beside the split's; through the recursion's steps 1e-5 in the 2-norm."""
    import torch

    print("values without a split", sizes, lengths, where, value, flush=True)
    capi = PC.pkg().capi
    S, T, P, Q = len(lengths), max(lengths), 32, 8
    a, b, c = sizes
    doc = {"layers": [{"size": P, "name": "input", "type": "input"}, {"size": a, "name": "a", "type": "blstm", "bias": 0.8},
                      {"size": b, "name": "b", "type": "blstm", "bias": 1.0}, {"size": c, "name": "c", "type": "feedforward_logistic", "bias": 1.0},
                      {"size": Q, "name": "out", "type": "feedforward_identity", "bias": 1.0}, {"size": Q, "name": "post", "type": "sse"}]}
    net = capi.Network(json.dumps(doc), S, T)
    gen = torch.Generator(device="cuda").manual_seed(b)
    net.weights.uniform_(-0.1, 0.1, generator=gen)
    types = make_pat_types(lengths, T)
    pat = PC.dev(types)
    valid = (pat != 0).reshape(-1, 1)
    x = (torch.randn(S * T, P, device="cuda", generator=gen) * valid).reshape(-1)
    target = (torch.randn(S * T, Q, device="cuda", generator=gen) * valid).reshape(-1)
    # the first slot of padding of the shortest sequence, or a slot of the first sequence beside it
    step = min(lengths) if where == "padding" else min(lengths) - 1
    slot = step * S + (lengths.index(min(lengths)) if where == "padding" else 0)
    assert (types.reshape(-1)[slot] == 0) == (where == "padding")
    others = valid[:, 0].clone()
    if where != "padding":
        others[0::S] = False

    def passed():
        net.load_sequences(pat, T, min(lengths), x, target)
        net.forward()
        net.calculate_error()
        net.backward()
        torch.cuda.synchronize()
        return {"%s.%s" % (n, kind): net.layer(n)[kind].reshape(S * T, -1)[others].clone() for n in ("a", "b", "c", "out") for kind in ("outputs", "errors")}, net.updates.clone()

    want, gradients = passed()
    (target if where == "target" else x).reshape(S * T, -1)[slot, 5] = value
    got, changed = passed()
    for name in want:
        assert float(want[name].norm()) > 0
        assert float((got[name] - want[name]).norm()) <= 1e-5 * float(want[name].norm()), name
    if where == "padding" and np.isfinite(value):  # (a forget gate that is NaN on a slot of padding is multiplied with the zero error there)
        assert float((changed - gradients).norm()) <= 1e-5 * float(gradients.norm())
    net.close()


@pytest.mark.parametrize("layers,P,S,T", [
    ([("feedforward_tanh", 512), ("feedforward_tanh", 512)], 382, 12, 500), ([("blstm", 200), ("lstm", 96)], 61, 10, 300),
    ([("feedforward_tanh", 1024)], 1300, 1, 2048)])  # (in line, its product cut along k)
@pytest.mark.parametrize("overlap", [True, False])
@pytest.mark.parametrize("own_stream", [True, False])
def test_a_pass_takes_no_scratch_of_the_callers_stream(layers, P, S, T, overlap, own_stream):
    """Products that are cut along k and run on the caller's stream find their scratch with the network: a pass on a stream that has none
    leaves it so, and the gradients are those of a stream that has.  The same under capture, whose replays give the same bits."""
    import torch

    print("scratch of the caller's stream", layers, P, S, T, overlap, own_stream, flush=True)
    capi = PC.pkg().capi
    Q = 7
    doc = {"layers": [{"size": P, "name": "input", "type": "input"}] +
           [{"size": n, "name": "l%d" % i, "type": t, "bias": 1.0} for i, (t, n) in enumerate(layers)] +
           [{"size": Q, "name": "out", "type": "feedforward_identity", "bias": 1.0}, {"size": Q, "name": "post", "type": "sse"}]}
    net = capi.Network(json.dumps(doc), S, T, overlap=overlap)
    gen = torch.Generator(device="cuda").manual_seed(P)
    net.weights.uniform_(-0.1, 0.1, generator=gen)
    pat = PC.dev(make_pat_types([T] * S, T))
    x, target = (torch.randn(S * T * n, device="cuda", generator=gen) for n in (P, Q))
    stream = torch.cuda.Stream() if own_stream else None

    def passed(stream):
        net.load_sequences(pat, T, T, x, target, stream=stream)
        net.forward(stream=stream)
        net.calculate_error(stream=stream)
        net.backward(stream=stream)

    torch.cuda.synchronize()
    capi.gemm_release(stream)
    held, got = capi.lib().cnt_gemm_scratch_buffers(), []
    for reserved in (False, True):
        if reserved:
            capi.gemm_reserve(stream)
        net.updates.fill_(3.0)
        torch.cuda.synchronize()
        passed(stream)
        torch.cuda.synchronize()
        got.append(net.updates.clone())
        assert capi.lib().cnt_gemm_scratch_buffers() == held + reserved
    capi.gemm_release(stream)
    assert float(got[0].norm()) > 0 and torch.equal(got[0], got[1])
    if own_stream:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
            passed(stream)
        assert capi.lib().cnt_gemm_scratch_buffers() == held
        for _ in range(3):
            net.updates.fill_(3.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            # (captured passes keep other batches of products: 1e-6, as above)
            assert float((net.updates - got[0]).norm()) <= 1e-6 * float(got[0].norm())
        again = net.updates.clone()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(again, net.updates)
        del graph
    net.close()


def test_networks_share_the_stream_of_their_weight_gradients():
    """Networks on one stream, on streams and threads of their own, one of them destroyed while the others go on, a new one made, and one more
    pass under capture beside them: every pass's gradients are those of the same network, weights, inputs and targets on the caller's
    stream alone (1e-6, as above).  No two networks have the same, so that one's sums in another's are seen."""
    import threading

    import torch

    capi = PC.pkg().capi
    S, T, P, Q = 6, 500, 40, 30
    doc = json.dumps({"layers": [{"size": P, "name": "input", "type": "input"}, {"size": 256, "name": "a", "type": "feedforward_tanh", "bias": 1.0},
                                 {"size": 128, "name": "b", "type": "blstm", "bias": 1.0},
                                 {"size": Q, "name": "out", "type": "feedforward_identity", "bias": 1.0}, {"size": Q, "name": "post", "type": "sse"}]})
    pat = PC.dev(make_pat_types([T] * S, T))

    class Run:
        def __init__(self, seed):
            gen = torch.Generator(device="cuda").manual_seed(seed)
            self.x, self.target = (torch.randn(S * T * n, device="cuda", generator=gen) for n in (P, Q))
            self.net = capi.Network(doc, S, T, overlap=False)
            weights = self.net.weights.uniform_(-0.1, 0.1, generator=gen).clone()
            self.go()
            torch.cuda.synchronize()
            self.want = self.net.updates.clone()
            self.net.close()
            self.net = capi.Network(doc, S, T)
            self.net.weights.copy_(weights)
            torch.cuda.synchronize()

        def go(self, stream=None):
            self.net.load_sequences(pat, T, T, self.x, self.target, stream=stream)
            self.net.forward(stream=stream)
            self.net.calculate_error(stream=stream)
            self.net.backward(stream=stream)

        def right(self):
            return float((self.net.updates - self.want).norm()) <= 1e-6 * float(self.want.norm())

    runs = [Run(seed) for seed in range(5, 8)]
    for a in runs:
        for b in runs:
            assert a is b or float((a.want - b.want).norm()) > 0.1 * float(a.want.norm())
    wrong = []

    def work(run):
        stream = torch.cuda.Stream()
        for _ in range(4):
            run.net.updates.fill_(3.0)
            torch.cuda.synchronize()
            run.go(stream)
            stream.synchronize()
            if not run.right():
                wrong.append(run)

    threads = [threading.Thread(target=work, args=(r,)) for r in runs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    runs.pop(0).net.close()
    runs.append(Run(8))
    for _ in range(2):
        for run in runs:
            run.net.updates.fill_(3.0)
            run.go()
    torch.cuda.synchronize()
    assert all(run.right() for run in runs)
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        runs[0].go(torch.cuda.current_stream())
    for _ in range(3):
        for run in runs[:2]:
            run.net.updates.fill_(3.0)
        graph.replay()
        runs[1].go()
        torch.cuda.synchronize()
        assert all(run.right() for run in runs)
    for run in runs:
        run.net.close()


def dense_network(capi, seed, S=8, T=512, P=64, n=256, Q=32, overlap=True):
    """A feed-forward network, by itself one whose pass is too large for weight gradients in line, and what a pass of it takes."""
    import torch

    doc = {"layers": [{"size": P, "name": "input", "type": "input"}] +
           [{"size": n, "name": "l%d" % i, "type": "feedforward_tanh", "bias": 1.0} for i in range(3)] +
           [{"size": Q, "name": "out", "type": "feedforward_identity", "bias": 1.0}, {"size": Q, "name": "post", "type": "sse"}]}
    net = capi.Network(json.dumps(doc), S, T, overlap=overlap)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    net.weights.uniform_(-0.1, 0.1, generator=gen)
    pat = PC.dev(make_pat_types([T] * S, T))
    x, target = (torch.randn(S * T * k, device="cuda", generator=gen) for k in (P, Q))

    def go(stream):
        net.load_sequences(pat, T, T, x, target, stream=stream)
        net.forward(stream=stream)
        net.calculate_error(stream=stream)
        net.backward(stream=stream)

    return net, go


def test_a_network_does_not_wait_for_another_callers_stream():
    """Two networks on two streams, one of which is busy with something else first: the other one's pass ends meanwhile.  (Streams that the
    runtime puts on one hardware queue do wait for each other, so several pairs of streams and networks are tried; one is enough.)"""
    import torch

    capi = PC.pkg().capi
    first, first_go = dense_network(capi, 1)
    others = [dense_network(capi, seed) for seed in (2, 3)]
    begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    for go in [first_go] + [o[1] for o in others]:
        go(None)
    for _ in range(2):  # (the first sleep loads its code)
        torch.cuda.synchronize()
        begin.record()
        torch.cuda._sleep(1 << 20)
        end.record()
    torch.cuda.synchronize()
    cycles = int((1 << 20) * 20.0 / begin.elapsed_time(end))  # 20 ms
    streams = [torch.cuda.Stream() for _ in range(5)]
    free = []
    for (_, other_go), busy, mine in itertools.product(others, streams, streams):
        if busy is mine or any(free):
            continue
        with torch.cuda.stream(busy):
            torch.cuda._sleep(cycles)
            slept = torch.cuda.Event()
            slept.record()
        other_go(busy)
        first_go(mine)
        mine.synchronize()
        free.append(not slept.query())
        torch.cuda.synchronize()
    assert any(free)
    for net in [first] + [o[0] for o in others]:
        net.close()


@pytest.mark.parametrize("T", [781, 782, 2048, 2049])  # 1.7e9 multiply-adds above the lowest layer, and the slots' line
def test_gradients_in_line_and_beside_the_callers_stream(T):
    """Feed-forward gradients at the lines between weight halves on the caller's stream and on the one beside it, against all on the
    caller's (1e-6, as above)."""
    import torch

    capi = PC.pkg().capi
    got = []
    for overlap in (True, False):
        net, go = dense_network(capi, 4, 1, T, 16, 1024 if T < 2000 else 256, 76 if T < 2000 else 32, overlap)
        net.updates.fill_(3.0)
        go(None)
        torch.cuda.synchronize()
        got.append(net.updates.clone())
        net.close()
    assert float(got[1].norm()) > 0 and float((got[0] - got[1]).norm()) <= 1e-6 * float(got[1].norm())


def test_the_stream_beside_the_callers_is_one_for_a_callers_stream():
    """The gradients of passes that alternate between networks and streams, of a pass between a capture's pass and its end, and of
    networks whose predecessor on the shared stream is gone: bit for bit those of the network's first pass."""
    import torch

    capi = PC.pkg().capi
    nets = [dense_network(capi, seed) for seed in (1, 2, 3)]
    want = []
    for net, go in nets:
        go(None)
        torch.cuda.synchronize()
        want.append(net.updates.clone())
    streams = [None, torch.cuda.Stream(), torch.cuda.Stream()]

    def check(order):
        torch.cuda.synchronize()
        for i, stream in order:
            nets[i][0].updates.fill_(3.0)
            torch.cuda.synchronize()
        for i, stream in order:
            nets[i][1](stream)
        torch.cuda.synchronize()
        for i, _ in order:
            assert torch.equal(nets[i][0].updates, want[i]), (i, order)

    for order in ([0, 1, 2], [1, 2, 0], [2, 2, 1], [0, 0, 0], [1, 1, 2]):
        check([(i, streams[s]) for i, s in enumerate(order)])
    # a network's own stream that takes part in a capture may take nothing else before the capture's end
    check([(0, streams[1]), (1, streams[2])])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream(), capture_error_mode="relaxed"):
        nets[1][1](torch.cuda.current_stream())
        nets[1][1](streams[2])
    torch.cuda.synchronize()
    assert float((nets[1][0].updates - want[1]).norm()) <= 1e-6 * float(want[1].norm())  # (in line: other batches of products)
    for _ in range(3):
        nets[1][0].updates.fill_(3.0)
        graph.replay()
        torch.cuda.synchronize()
        assert float((nets[1][0].updates - want[1]).norm()) <= 1e-6 * float(want[1].norm())
    del graph
    check([(0, streams[1])])
    nets[0][0].close()
    nets.pop(0)
    want.pop(0)
    check([(0, streams[2]), (1, streams[1])])
    for net, _ in nets:
        net.close()


@pytest.mark.parametrize("T", [40, 700])
def test_weight_gradients_of_a_fraction_without_a_valid_slot(T):
    """Every weight gradient over an empty list of slots is zero, whatever the updates held: one split, several, narrow and wide."""
    import torch

    print("network case: no valid slot", T, flush=True)
    capi = PC.pkg().capi
    P, Q, S = 20, 8, 3
    layers = [{"size": P, "name": "input", "type": "input"}, {"name": "ff1", "type": "feedforward_tanh", "size": 64, "bias": 1.0},
              {"name": "ff2", "type": "feedforward_logistic", "size": 512, "bias": 0.5},
              {"name": "ff3", "type": "feedforward_tanh", "size": 512, "bias": 0.5},
              {"name": "out", "type": "feedforward_identity", "size": Q, "bias": 1.0}, {"name": "postoutput", "type": "sse", "size": Q}]
    net = capi.Network(json.dumps({"layers": layers}), S, T)
    net.randomize(3, 0.1)
    x, tgt = torch.randn(T * S * P, device="cuda"), torch.randn(T * S * Q, device="cuda")
    for pat, zero in ((make_pat_types([T] * S, T), False), (np.zeros(T * S, dtype=np.int8), True)):
        net.load_sequences(PC.dev(pat), T, 1 if zero else T, x, tgt)
        net.updates.fill_(5.0)
        net.forward()
        net.backward()
        torch.cuda.synchronize()
        assert bool((net.updates == 0).all()) == zero
    net.close()


def test_network_reports_a_later_lstm_layer_that_gave_up_and_keeps_the_weights():
    """Failure handling at network level, forced from the host: the SECOND recurrent layer's recursions get a spin
    limit of zero, the first layer's stay as they are.  Every kernel still ends normally; the failure is reported by
    cnt_network_check (which looks at every recurrent layer) or by the call into the network that follows the failed
    launch, the optimizer step of that pass does not touch the weights, and with the bounds restored the same network
    handle trains on."""
    import torch

    print("network give-up case", flush=True)
    capi = PC.pkg().capi
    P, Q, S, T = 16, 5, 6, 40
    specs = [{"name": "bl1", "type": "blstm", "size": 128, "bias": 1.0},
             {"name": "bl2", "type": "blstm", "size": 512, "bias": 1.0},
             {"name": "out", "type": "feedforward_identity", "size": Q, "bias": 1.0},
             {"name": "postoutput", "type": "sse", "size": Q}]
    doc = {"layers": [{"size": P, "name": "input", "type": "input"}] + specs}
    net = capi.Network(json.dumps(doc), S, T)
    rng = np.random.default_rng(8)
    net.weights.copy_(torch.from_numpy(rng.uniform(-0.1, 0.1, net.n_weights).astype(np.float32)))
    pat = torch.full((T * S,), 2, dtype=torch.int8, device="cuda")
    x = PC.dev(rng.standard_normal(T * S * P).astype(np.float32))
    tgt = PC.dev(rng.standard_normal(T * S * Q).astype(np.float32))

    def one_pass():
        net.load_sequences(pat, T, T, x, tgt)
        net.forward()
        net.backward()
        net.update(0, 1e-3, 0.0, float(T * S))
        net.check()

    one_pass()
    torch.cuda.synchronize()
    before = net.weights.clone()
    second = [i for i, L in enumerate(net.layers) if L["type"] == "blstm"][1]
    with pytest.raises(RuntimeError):
        net.set_wait_bounds(0, 0, 0, 0)  # the input layer is not a recurrent layer
    net.set_wait_bounds(second, 0, 0, 0)
    failures = 0
    for _ in range(3):  # an attempt only fails if some poll really comes back incomplete
        try:
            one_pass()
        except RuntimeError as e:
            assert "gave up" in str(e)
            failures += 1
            torch.cuda.synchronize()
            try:
                net.check()  # a second failed launch of the same attempt may have ended meanwhile
            except RuntimeError:
                pass
            # the pass that failed did not reach the weights
            assert torch.equal(net.weights, before)
            break
        before = net.weights.clone()  # a pass in which every poll happened to succeed is an ordinary pass
    assert failures >= 1
    net.set_wait_bounds(second, 1 << 22, 28, 34)
    one_pass()
    torch.cuda.synchronize()
    assert not torch.equal(net.weights, before)
    assert bool(torch.isfinite(net.weights).all())
    net.close()


def test_network_give_up_on_a_nonblocking_stream_keeps_weights_and_adam_state():
    """The same failure, on a stream of the caller's own (non-blocking: nothing orders it against the legacy default
    stream) and without a check between the calls of a pass, with Adam: the failed pass's optimizer step is skipped on the
    device -- weights, moments and the bias-correction products stay where they were -- so that after two good passes
    around the failed one the weights equal those of a twin network that ran only the two good passes."""
    import torch

    print("network give-up on a non-blocking stream, Adam", flush=True)
    capi = PC.pkg().capi
    P, Q, S, T = 16, 5, 6, 40
    specs = [{"name": "bl1", "type": "blstm", "size": 512, "bias": 1.0},
             {"name": "out", "type": "feedforward_identity", "size": Q, "bias": 1.0},
             {"name": "postoutput", "type": "sse", "size": Q}]
    doc = json.dumps({"layers": [{"size": P, "name": "input", "type": "input"}] + specs})
    rng = np.random.default_rng(9)
    w0 = torch.from_numpy(rng.uniform(-0.1, 0.1, 10 ** 7).astype(np.float32))
    pat = torch.full((T * S,), 2, dtype=torch.int8, device="cuda")
    x = PC.dev(rng.standard_normal(T * S * P).astype(np.float32))
    tgt = PC.dev(rng.standard_normal(T * S * Q).astype(np.float32))
    stream = torch.cuda.Stream()

    def make():
        net = capi.Network(doc, S, T)
        net.weights.copy_(w0[:net.n_weights])
        torch.cuda.synchronize()
        return net

    def enqueue_pass(net):
        net.load_sequences(pat, T, T, x, tgt, stream=stream)
        net.forward(stream=stream)
        net.backward(stream=stream)
        net.update(5, 1e-3, 0.0, float(T * S), stream=stream)

    twin = make()
    enqueue_pass(twin); enqueue_pass(twin)
    twin.check(stream=stream)
    net = make()
    enqueue_pass(net)
    net.check(stream=stream)
    before = net.weights.clone()
    layer = [i for i, L in enumerate(net.layers) if L["type"] == "blstm"][0]
    net.set_wait_bounds(layer, 0, 0, 0)
    failed = False
    for _ in range(4):  # an attempt only fails if some poll really comes back incomplete
        try:
            enqueue_pass(net)       # no check in between: whichever call comes after the failed launch reports it
            net.check(stream=stream)
        except RuntimeError as e:
            assert "gave up" in str(e)
            failed = True
            stream.synchronize()
            try:
                net.check(stream=stream)  # the forward recursion of the same attempt may have given up as well
            except RuntimeError:
                pass
            break
        pytest.skip("every poll happened to succeed: nothing to check")
    assert failed
    torch.cuda.synchronize()
    assert torch.equal(net.weights, before)
    net.set_wait_bounds(layer, 1 << 22, 28, 34)
    enqueue_pass(net)
    net.check(stream=stream)
    torch.cuda.synchronize()
    a, b = (net.weights - w0[:net.n_weights].cuda()).cpu().numpy(), (twin.weights - w0[:twin.n_weights].cuda()).cpu().numpy()
    # Adam normalises every step to about the learning rate: a bias correction one step off would change the second
    # step by some 30 %; the sums inside the weight gradients are added in a different order from run to run
    assert PC.relerr(a, b) < 2e-2
    net.close(); twin.close()


# the last case has channel counts that are not multiples of four: no 16-byte accesses anywhere, and the skip layers'
# backward steps run as launches of their own instead of in the epilogue of the following layer's product
# The fifth case is a stack with benchmark config 4's layer sizes (64 residual / 128 skip channels, 80 conditioning
# dimensions up-sampled 80 times) and one full cycle of its dilations, 1 ... 512, over waveforms long enough that
# every dilation reaches valid history and the sequences' ragged ends, against the oracle's graph.
@pytest.mark.parametrize("nb,cnn_tanh,R,K,Q,C,lengths,cycle,upsample", [
    (4, 1, 32, 64, 64, 20, [120, 90], 3, 20), (11, 0, 32, 64, 64, 20, [120, 90], 3, 20),
    (3, 1, 30, 50, 64, 20, [120, 90], 3, 20),
    # the other widths the fused block launch is built for
    (3, 1, 64, 256, 64, 20, [70, 52], 3, 20), (3, 0, 64, 64, 64, 20, [70, 52], 3, 20),
    (3, 1, 32, 128, 64, 20, [70, 52], 3, 20), (3, 0, 32, 32, 64, 20, [70, 52], 3, 20),
    (3, 0, 64, 96, 64, 21, [70, 52], 3, 20), (3, 1, 32, 96, 64, 20, [70, 52], 3, 20),
    (3, 1, 32, 256, 64, 22, [70, 52], 3, 20), (3, 0, 48, 32, 64, 20, [70, 52], 3, 20), (3, 1, 48, 64, 64, 45, [70, 52], 3, 20),
    (3, 1, 48, 96, 64, 20, [70, 52], 3, 20), (3, 0, 48, 128, 64, 80, [70, 52], 3, 20), (3, 1, 48, 256, 64, 20, [70, 52], 3, 20),
    # skip channels that it is not built for
    (3, 1, 48, 80, 64, 20, [70, 52], 3, 20), (3, 1, 64, 32, 64, 20, [70, 52], 3, 20),
    (10, 1, 64, 128, 256, 80, [4000, 3300], 10, 80),
])
def test_wavenet_network_file_against_oracle_graph(nb, cnn_tanh, R, K, Q, C, lengths, cycle, upsample):
    import torch

    print("wavenet network file", nb, cnn_tanh, R, K, Q, C, lengths, cycle, flush=True)
    pkg = PC.pkg()
    capi, networks = pkg.capi, PC.networks()
    O.use_all_cores()
    S, T = len(lengths), max(lengths)
    pat, onehot, ctx, target, N = WD.make(lengths, Q, C, upsample=upsample, seed=2)
    ref = networks.WaveNet(OM.OracleBackend(), nb, S, T, Q=Q, R=R, K=K, C=C, cnn_tanh=cnn_tanh, dilation_cycle=cycle)
    shapes = {k: len(ref.buf[k]["W"]) for k in ref.weight_names()}
    W = WD.init_weights(shapes, seed=3)
    for k, w in W.items():
        ref.buf[k]["W"][:] = w
    ref.set_inputs(pat, onehot, ctx, target)
    ref.forward()
    ref.calculate_error()
    ref.backward()

    doc = PC.pkg().specs.wavenet_network_doc(nb, Q, R, K, C, cnn_tanh, cycle)
    net = capi.Network(json.dumps(doc), S, T + 7, mdn_config=[1, 0, Q, 0, 1, -1])   # buffers longer than the fraction
    names = [L["name"] for L in net.layers if L["weight_count"]]
    assert sorted(names) == sorted(W)
    for L in net.layers:
        if L["weight_count"]:
            assert L["weight_count"] == W[L["name"]].size
            L["weights"].copy_(torch.from_numpy(W[L["name"]]))
    ctx_d = torch.zeros(C * S * (T + 7), dtype=torch.float32, device="cuda")
    ctx_d[: ctx.size].copy_(torch.from_numpy(ctx))
    net.set_context(ctx_d)
    dummy_in = torch.zeros(S * T, dtype=torch.float32, device="cuda")
    for _ in range(2):  # a second pass over the same fraction gives the same result (buffers cleared properly)
        net.load_sequences(PC.dev(pat), T, min(lengths), dummy_in, PC.dev(target))
        net.forward()
        loss = float(net.calculate_error().item())
        net.backward()
        torch.cuda.synchronize()
        ref_loss = float(ref.loss[0])
        assert abs(loss - ref_loss) <= TOL * abs(ref_loss)
        # teacher-forced one-hot input: equal on every valid slot (a padding slot right after a sequence's end holds
        # the one-hot of the last sample, as in the reference, where the oracle's input has zeros)
        fb = net.layer("feedbackBottom")["outputs"][: N * Q].cpu().numpy().reshape(N, Q)
        valid = pat != 0
        assert np.array_equal(fb[valid], onehot.reshape(N, Q)[valid])
        worst = 0.0
        for L in net.layers:
            if L["weight_count"]:
                e = PC.relerr(L["updates"].cpu().numpy(), ref.buf[L["name"]]["dW"])
                worst = max(worst, e)
                if e > TOL:
                    print("   ", L["name"], e, flush=True)
        assert worst < TOL
    # the comparison above was made on the path it is meant for: one launch per residual block where the library has
    # a block kernel for the widths (and layer by layer for the others), the block above folded in from the second on
    net.forward()
    capi.profile_enable(True)
    net.backward()
    torch.cuda.synchronize()
    launches = {k: n for k, (n, _) in capi.profile_read().items()}
    capi.profile_enable(False)
    if R in (32, 48, 64) and K in (32, 64, 96, 128, 256) and (R, K) != (64, 32):
        assert launches.get("wavenet_block_errors") == 1 and launches.get("wavenet_block_errors+cnn") == nb - 1, launches
    else:
        assert "wavenet_block_errors" not in launches and "wavenet_block_errors+cnn" not in launches, launches
    net.update(0, 1e-4, 0.0, float(sum(lengths)))
    torch.cuda.synchronize()
    moved = net.layer("cnn0")["weights"].cpu().numpy()
    assert PC.relerr(moved, W["cnn0"] - 1e-4 * ref.buf["cnn0"]["dW"]) < TOL
    net.close()


# block launches of 16, 64 and 128 samples per workgroup: a part of one workgroup, one and a sample more, and both sides of the lines
# between them (8192 samples, at 64 and 48 channels also 16 384); 32 channels behind the second line
@pytest.mark.parametrize("R,K,lengths", [(64, 64, [1]), (64, 128, [64]), (32, 64, [65]), (64, 64, [8192, 8101]), (64, 64, [8193, 8050]), (32, 32, [8193, 8192]),
                                         (64, 128, [15]), (64, 128, [4096, 4001]), (64, 96, [4097, 4003]), (32, 256, [17]), (48, 64, [4096, 4093]),
                                         (48, 96, [1]), (48, 32, [65]), (48, 128, [8192, 8101]), (48, 96, [8193, 8050])])
def test_wavenet_block_errors_of_both_workgroup_sizes(R, K, lengths):
    test_wavenet_network_file_against_oracle_graph(2, 1, R, K, 16, 4, lengths, 2, 5)


# inputs and targets that start on and off a 16-byte boundary, counts that are no multiple of four, with and without a slot order
# and recurrent layers' clears beside the copies
@pytest.mark.parametrize("shift", [0, 1, 2])
@pytest.mark.parametrize("P,D,lengths,recurrent", [(1, 3, [1], False), (3, 5, [7, 4], True), (37, 2, [300, 299, 151], True), (382, 187, [600] * 10, False)])
def test_inputs_and_targets_of_any_alignment(shift, P, D, lengths, recurrent):
    import torch

    S, T = len(lengths), max(lengths)
    N = S * T
    mid = [{"size": 32, "name": "l", "type": "lstm", "bias": 1.0}] if recurrent else []
    net = PC.pkg().capi.Network(json.dumps({"layers": [{"size": P, "name": "input", "type": "input"}] + mid + [
        {"size": D, "name": "o", "type": "feedforward_identity", "bias": 1.0}, {"size": D, "name": "post", "type": "sse"}]}), S, T + 3)
    x, y = torch.randn(P * N + shift, device="cuda")[shift:], torch.randn(D * N + shift, device="cuda")[shift:]
    net.layers[0]["outputs"].fill_(9.0)
    net.layers[-1]["outputs"].fill_(9.0)
    net.load_sequences(PC.dev(make_pat_types(lengths, T)), T, min(lengths), x, y)
    torch.cuda.synchronize()
    for layer, given in ((net.layers[0], x), (net.layers[-1], y)):
        assert torch.equal(layer["outputs"][: given.numel()], given)
        assert bool((layer["outputs"][given.numel():] == 9.0).all())
    net.close()


# slots of one lane, of a part of a wave, of a wave and more; one workgroup, several, and more slots than they take at a time
@pytest.mark.parametrize("D,lengths", [(1, [1]), (3, [700, 650]), (16, [40, 3]), (64, [5]), (65, [300, 299]), (187, [600] * 9 + [20])])
def test_squared_error_with_its_gradient(D, lengths):
    import torch

    S, T = len(lengths), max(lengths)
    N = S * T
    net = PC.pkg().capi.Network(json.dumps({"layers": [{"size": 2, "name": "input", "type": "input"},
                                                       {"size": D, "name": "o", "type": "feedforward_identity", "bias": 1.0},
                                                       {"size": D, "name": "post", "type": "sse"}]}), S, T)
    net.randomize(3, 0.3)
    pat = make_pat_types(lengths, T)
    x, t = torch.randn(2 * N, device="cuda"), torch.randn(D * N, device="cuda")
    net.load_sequences(PC.dev(pat), T, min(lengths), x, t)
    valid = PC.dev(pat).view(N, 1) != 0
    for repeat in range(3):
        net.forward()
        for _ in range(2):
            loss = float(net.calculate_error().item())
        if repeat == 1:
            net.backward()  # a layer turns the errors into its deltas in place; the second pass forms them again
        net.backward()
        torch.cuda.synchronize()
        want = torch.where(valid, net.layer("o")["outputs"][: N * D].view(N, D) - t.view(N, D), 0.0)
        assert torch.equal(net.layer("o")["errors"][: N * D].view(N, D), want)
        exact = 0.5 * float((want.double() ** 2).sum())
        assert abs(loss - exact) <= (N * D / 256 + 300) * 2.0 ** -24 * exact  # a thread's chain, waves, workgroups
    net.close()


@pytest.mark.parametrize("act,D,lengths", [("identity", 3, [70, 65]), ("tanh", 187, [300, 299])])
def test_squared_error_leaves_the_errors_alone(act, D, lengths):
    """The error of a fraction can be asked for at any time: the gradient comes from the outputs and targets that are there when
    the backward pass runs, and the deltas a backward pass has left stay."""
    import torch

    S, T = len(lengths), max(lengths)
    N = S * T
    net = PC.pkg().capi.Network(json.dumps({"layers": [{"size": 5, "name": "input", "type": "input"},
                                                       {"size": D, "name": "o", "type": "feedforward_" + act, "bias": 1.0},
                                                       {"size": D, "name": "post", "type": "sse"}]}), S, T)
    net.randomize(3, 0.3)
    pat = make_pat_types(lengths, T)
    valid = PC.dev(pat).view(N, 1) != 0
    net.load_sequences(PC.dev(pat), T, min(lengths), torch.randn(5 * N, device="cuda"), torch.randn(D * N, device="cuda"))
    net.forward()
    net.calculate_error()
    o, tgt = net.layer("o"), net.layers[-1]["outputs"]
    tgt.mul_(0.5).add_(1.0)
    o["outputs"].mul_(0.75)
    net.backward()
    y = o["outputs"].view(N, D)
    want = torch.where(valid, y - tgt.view(N, D), 0.0)
    if act == "tanh":
        want = (1.0 - y * y) * want
    deltas = o["errors"].clone()
    assert float((deltas.view(N, D) - want).abs().max()) <= 4e-7 * float(want.abs().max())
    loss = float(net.calculate_error().item())
    assert torch.equal(o["errors"], deltas)
    exact = 0.5 * float((torch.where(valid, y - tgt.view(N, D), 0.0).double() ** 2).sum())
    assert abs(loss - exact) <= 1.001 * 2.0 ** -24 * exact  # summed in 64 bits, rounded once
    net.close()


# slots of one lane, of a few, of a wave and of more than one store per lane; the columns taken from the layer before end
# inside a group of four; sizes that are no multiple of four
@pytest.mark.parametrize("P,lo,hi,Q,lengths", [(3, 0, 3, 1, [4, 2]), (3, 1, 3, 6, [1]), (5, 0, 5, 30, [9, 4, 7]), (6, 2, 5, 253, [31, 30]),
                                               (4, 0, 0, 1024, [700, 650]), (7, 0, 7, 26, [40])])
def test_feedback_of_the_true_class(P, lo, hi, Q, lengths):
    import torch

    S, T = len(lengths), max(lengths)
    N, D = S * T, hi - lo + Q
    doc = {"layers": [{"size": P, "name": "input", "type": "input"},
                      {"size": P, "name": "below", "type": "feedforward_tanh", "bias": 1.0},
                      {"size": D, "name": "fb", "type": "feedback", "bias": 1.0, "previousDimStart": lo, "previousDimEnd": hi},
                      {"size": Q, "name": "out", "type": "feedforward_identity", "bias": 1.0},
                      {"size": 1, "name": "post", "type": "mdn"}]}
    net = PC.pkg().capi.Network(json.dumps(doc), S, T, mdn_config=[1, 0, Q, 0, 1, -1])
    net.randomize(3, 0.3)
    rng = np.random.default_rng(P + Q)
    pat = make_pat_types(lengths, T)
    cls = rng.integers(0, Q, N)
    net.load_sequences(PC.dev(pat), T, min(lengths), PC.dev(rng.standard_normal(P * N).astype(np.float32)), PC.dev(cls.astype(np.float32)))
    net.forward()
    torch.cuda.synchronize()
    want = np.zeros((N, D), np.float32)
    want[:, : hi - lo] = net.layer("below")["outputs"].cpu().numpy()[: N * P].reshape(N, P)[:, lo:hi]
    for n in range(S, N):
        if pat[n - S]:
            want[n, hi - lo + cls[n - S]] = 1.0
    assert np.array_equal(net.layer("fb")["outputs"].cpu().numpy()[: N * D].reshape(N, D), want)
    net.close()


def test_network_file_rejections():
    capi = PC.pkg().capi

    def make(layers, weights=None):
        doc = {"layers": layers}
        if weights is not None:
            doc["weights"] = weights
        return json.dumps(doc)

    inp = {"size": 3, "name": "input", "type": "input"}
    post = {"size": 4, "name": "post", "type": "sse"}
    with pytest.raises(RuntimeError, match="does not cover"):
        capi.Network(make([inp, {"size": 4, "name": "c", "type": "maxpooling", "bias": 1.0}, post]), 2, 10)
    with pytest.raises(RuntimeError, match="expected 12"):
        capi.Network(make([inp, {"size": 4, "name": "o", "type": "feedforward_identity", "bias": 1.0}, post],
                          {"o": {"input": [0.0] * 11, "bias": [0.0] * 4, "internal": []}}), 2, 10)
    with pytest.raises(RuntimeError, match="Missing value 'bias'|missing value 'bias'"):
        capi.Network(make([inp, {"size": 4, "name": "o", "type": "feedforward_identity"}, post]), 2, 10)
    with pytest.raises(RuntimeError, match="post-output"):
        capi.Network(make([inp, {"size": 4, "name": "o", "type": "feedforward_identity", "bias": 1.0},
                           {"size": 4, "name": "o2", "type": "feedforward_identity", "bias": 1.0}]), 2, 10)
    with pytest.raises(RuntimeError, match="linked to"):
        capi.Network(make([inp, {"size": 4, "name": "o", "type": "feedforward_identity", "bias": 1.0},
                           {"size": 5, "name": "s", "type": "skipini", "bias": 1.0}, post]), 2, 10)
    with pytest.raises(RuntimeError, match="resolution"):
        capi.Network(make([inp, {"size": 4, "name": "o", "type": "feedforward_identity", "bias": 1.0, "resolution": 80},
                           post]), 2, 10)
    net = capi.Network(make([inp, {"size": 4, "name": "o", "type": "feedforward_identity", "bias": 1.0}, post]), 2, 10)
    with pytest.raises(RuntimeError, match="no fraction"):
        net.forward()
    net.close()


def test_layer_specific_learning_rate():
    """A layer's own "learningRate" replaces the optimizer's for that layer (0 freezes it)."""
    import torch

    capi = PC.pkg().capi
    doc = {"layers": [{"size": 3, "name": "input", "type": "input"},
                      {"size": 5, "name": "frozen", "type": "feedforward_tanh", "bias": 1.0, "learningRate": 0.0},
                      {"size": 4, "name": "fast", "type": "feedforward_identity", "bias": 1.0, "learningRate": 0.5},
                      {"size": 4, "name": "plain", "type": "feedforward_identity", "bias": 1.0},
                      {"size": 4, "name": "post", "type": "sse"}]}
    S, T = 2, 6
    net = capi.Network(json.dumps(doc), S, T)
    net.randomize(3, 0.3)
    w0 = net.weights.clone()
    rng = np.random.default_rng(2)
    pat = make_pat_types([T, T], T)
    net.load_sequences(PC.dev(pat), T, T, PC.dev(rng.standard_normal(3 * S * T).astype(np.float32)),
                       PC.dev(rng.standard_normal(4 * S * T).astype(np.float32)))
    net.forward()
    net.backward()
    net.update(0, 0.01, 0.0, float(S * T))
    torch.cuda.synchronize()
    g = net.updates
    for name, lr in (("frozen", 0.0), ("fast", 0.5), ("plain", 0.01)):
        L = net.layer(name)
        a, b = L["weight_offset"], L["weight_offset"] + L["weight_count"]
        assert torch.allclose(net.weights[a:b], w0[a:b] - lr * g[a:b], rtol=1e-6, atol=1e-7), name
    net.close()


class _CondOracleBackend(OM.OracleBackend):
    """Oracle back end whose gated layers also accumulate the gradient with respect to the conditioning features."""
    ctx_grad = None

    def wavnetc_backward(self, D, C, N, pat, W, ctx, core, cth, err, prev_err, dW):
        O.wavnetc_backward(D, C, N, pat, W, ctx, core, cth, err, prev_err, dW, self.ctx_grad)


# one launch per residual block: tiles of 16, 32 and 64 samples with a ragged last one, conditioning rows that end inside
# a 16-byte piece or start off a 16-byte boundary, fewer skip than residual channels, the widest conditioning, none
@pytest.mark.parametrize("cnn_tanh,R,K,C,lengths", [
    (1, 32, 32, 4, [1]), (1, 64, 32, 7, [40, 33, 1]), (0, 48, 96, 45, [70, 51]), (1, 48, 256, 112, [17]), (1, 64, 80, 81, [2050, 1999]),
    (1, 32, 64, 20, [12300, 12295]), (1, 64, 128, 100, [8200, 7000, 8199]),
    (1, 32, 32, 0, [40, 33]), (0, 48, 16, 0, [16]), (1, 64, 128, 0, [2200, 2001]),
])
def test_wavenet_block_forward_edges(cnn_tanh, R, K, C, lengths):
    import torch

    print("wavenet block forward", cnn_tanh, R, K, C, lengths, flush=True)
    capi, networks = PC.pkg().capi, PC.networks()
    O.use_all_cores()
    nb, Q, S, T = 2, 32, len(lengths), max(lengths)
    pat, _, ctx, target, N = WD.make(lengths, Q, C or 4, upsample=5, seed=7)
    onehot = np.zeros((N, Q), np.float32)  # the feedback layer's: also in the first padding slot behind a sequence
    follows = np.flatnonzero(pat[: N - S] != 0)
    onehot[follows + S, np.asarray(target).reshape(-1)[follows].astype(int)] = 1
    ref = networks.WaveNet(OM.OracleBackend(), nb, S, T, Q=Q, R=R, K=K, C=C or 4, cnn_tanh=cnn_tanh, dilation_cycle=10)
    W = WD.init_weights({k: len(ref.buf[k]["W"]) for k in ref.weight_names()}, seed=3)
    for k, w in W.items():
        if not C and k.startswith("wav"):
            w[:] = 0  # a layer without conditioning features is one whose features count nothing
        ref.buf[k]["W"][:] = w
    ref.set_inputs(pat, onehot.reshape(-1), ctx, target)
    ref.forward()
    net = capi.Network(json.dumps(PC.pkg().specs.wavenet_network_doc(nb, Q, R, K, C, cnn_tanh, 10)), S, T, mdn_config=[1, 0, Q, 0, 1, -1])
    for L in net.layers:
        if L["weight_count"]:
            L["weights"].copy_(torch.from_numpy(W[L["name"]]))
    ctx_d = PC.dev(ctx)
    if C:
        net.set_context(ctx_d)
    net.load_sequences(PC.dev(pat), T, min(lengths), torch.zeros(N, dtype=torch.float32, device="cuda"), PC.dev(target))
    for layer in net.layers:
        if layer["type"] == "cnn":
            layer["outputs"].fill_(3.0)  # padding slots of a convolution layer keep what they hold
    net.forward()
    torch.cuda.synchronize()
    valid = (pat != 0).repeat(2 * R)
    for layer in net.layers:
        name = layer["name"]
        if name not in ref.buf or name == "postoutput":
            continue
        got, want = layer["outputs"].cpu().numpy()[: ref.buf[name]["out"].size], ref.buf[name]["out"]
        if layer["type"] == "cnn":
            assert np.all(got[~valid] == 3.0)
            got, want = got[valid], want[valid]
        assert np.abs(got - want).max() <= 2e-5 * max(1.0, np.abs(want).max()), name
    net.close()


@pytest.mark.parametrize("option,rate,sgd_before", [(1, 1e-2, True), (1, 1e-2, False), (5, 1e-3, True), (5, 1e-3, False)])
def test_first_optimizer_step_under_capture(option, rate, sgd_before):
    """AdaGrad's and Adam's state is set up by the first update.  Where that one is captured, the replays go on from the state
    as eager updates do, instead of starting over with each.  The step rounds every operation on its own: equal bits.
    (Plain steps may come before, they keep no statistics.)"""
    import torch

    print("first update captured", option, sgd_before, flush=True)
    capi = PC.pkg().capi
    S, T, lengths = 2, 9, [9, 7]
    doc = json.dumps({"layers": [{"size": 5, "name": "input", "type": "input"},
                                 {"size": 3, "name": "o", "type": "feedforward_tanh", "bias": 1.0},
                                 {"size": 3, "name": "post", "type": "sse"}]})
    pat, x, t = PC.dev(make_pat_types(lengths, T)), torch.randn(5 * S * T, device="cuda"), torch.randn(3 * S * T, device="cuda")
    nets = [capi.Network(doc, S, T) for _ in range(2)]
    for net in nets:
        net.randomize(3, 0.3)
        net.load_sequences(pat, T, min(lengths), x, t)
        net.forward()
        net.backward()
    graphed, eager = nets
    graphed.updates.copy_(eager.updates)
    if sgd_before:
        for net in nets:
            net.update(0, 1e-2, 0.0, 1.0)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, capture_error_mode="relaxed"):
        graphed.update(option, rate, 0.0, float(sum(lengths)))
    torch.cuda.synchronize()
    assert torch.equal(graphed.weights, eager.weights)  # nothing has run yet
    for step in range(4):
        gradient = torch.randn_like(eager.updates) * (step + 1)
        for net in nets:
            net.updates.copy_(gradient)
        graph.replay()
        eager.update(option, rate, 0.0, float(sum(lengths)))
        torch.cuda.synchronize()
        assert torch.equal(graphed.weights, eager.weights), step
    for net in nets:
        net.close()


# block launches that form the gate's pre-activations again (tanh convolution), ones that read them, ones without conditioning
# features.  Not compared: the layer below the blocks, whose errors go through a sum that only a forward pass clears, and the
# conditioning part of layers whose pre-activations are kept: its gradient takes the place of its values.
@pytest.mark.parametrize("cnn_tanh,R,K,C,lengths,conditioning_again", [
    (1, 32, 64, 20, [120, 90], True), (1, 64, 128, 81, [700, 333], True), (1, 64, 256, 7, [16500], True), (0, 32, 64, 20, [120, 90], False),
    (1, 64, 64, 0, [70, 52], True), (1, 48, 96, 20, [120, 90], True),
])
def test_second_backward_pass_of_a_wavenet_stack(cnn_tanh, R, K, C, lengths, conditioning_again):
    import torch

    print("wavenet second backward pass", cnn_tanh, R, K, C, lengths, flush=True)
    capi = PC.pkg().capi
    nb, Q, S, T = 3, 32, len(lengths), max(lengths)
    pat, _, ctx, target, N = WD.make(lengths, Q, C or 4, upsample=5, seed=7)
    net = capi.Network(json.dumps(PC.pkg().specs.wavenet_network_doc(nb, Q, R, K, C, cnn_tanh, 3)), S, T, mdn_config=[1, 0, Q, 0, 1, -1])
    net.randomize(11, 0.2)
    ctx_d = PC.dev(ctx)
    if C:
        net.set_context(ctx_d)
    net.load_sequences(PC.dev(pat), T, min(lengths), torch.zeros(N, dtype=torch.float32, device="cuda"), PC.dev(target))
    net.forward()
    net.calculate_error()
    net.backward()
    first = {L["name"]: L["updates"].cpu().numpy() for L in net.layers if L["weight_count"]}
    assert all(np.abs(v).max() > 0 for v in first.values())
    net.backward()
    for L in net.layers:
        if L["weight_count"] and L["name"] != "emb" and (conditioning_again or L["type"] != "wavnetc"):
            # the same products; only the order of their atomic sums may differ
            assert PC.relerr(L["updates"].cpu().numpy(), first[L["name"]]) < 1e-5, L["name"]
    net.close()


@pytest.mark.parametrize("context_mv", [False, True])
def test_wavenet_with_frame_rate_conditioning_network(context_mv, tmp_path):
    """The reference example's layout in full: externalloader -> skipini -> blstm -> cnn -> skipcat at one slot per
    R time steps, flagged as the wavnetc layers' input; the oracle side walks the same graph with the oracle's
    primitives (conditioning part spelled out here, sample-rate part by the shared graph walk).  With context_mv the
    wavnetc layers name a "contextMV" file (means and standard deviations of the conditioning features, one of them
    vanishing), which the first of them applies while it up-samples (layers/wavNetCore.cu:143-190, :322-351)."""
    import torch

    print("wavenet network file with conditioning sub-network, contextMV", context_mv, flush=True)
    pkg = PC.pkg()
    capi, networks = pkg.capi, PC.networks()
    nb, Q, R, K = 3, 64, 32, 64
    E, HB, DC, C, RES = 12, 128, 10, 11, 4
    lengths = [120, 90]
    S, T = len(lengths), max(lengths)
    Tr = -(-T // RES)
    lengths_r = [-(-n // RES) for n in lengths]
    pat, onehot, _, target, N = WD.make(lengths, Q, C, upsample=RES, seed=2)
    pat_r = make_pat_types(lengths_r, Tr)
    Nr = S * Tr
    rng = np.random.default_rng(11)
    frame_index = np.zeros((T, S), dtype=np.float32)
    for s, n in enumerate(lengths):
        frame_index[:n, s] = np.arange(n) // RES
    data = rng.standard_normal((Tr, S, E)).astype(np.float32)
    mean_std = np.concatenate([0.1 * rng.standard_normal(E), rng.uniform(0.5, 2.0, E)]).astype(np.float32)
    mean_std[E + 3] = 1e-7   # a vanishing deviation counts as 1

    # ---- oracle: conditioning part -----------------------------------------------------------------------------
    valid_r = (pat_r != 0)
    sd = np.where(mean_std[E:] < 1e-5, 1.0, mean_std[E:])
    ext = ((data - mean_std[:E]) / sd).astype(np.float32).reshape(Nr, E)
    ext[~valid_r] = 0
    ext = np.ascontiguousarray(ext.reshape(-1))
    w_lstm = rng.uniform(-0.1, 0.1, OM.weight_count({"type": "blstm", "size": HB}, E)).astype(np.float32)
    hw, it = np.ones(DC, dtype=np.int32), np.ones(DC, dtype=np.int32)
    w_cnn = rng.uniform(-0.1, 0.1, HB * 3 * DC + DC).astype(np.float32)
    desc = O.LstmDesc(E, HB, 1, S, Tr, min(lengths_r), 1.0)
    fw, bw = O.LstmState(HB // 2, Nr), O.LstmState(HB // 2, Nr)
    l2 = np.zeros(HB * Nr, dtype=np.float32)
    O.lstm_forward(desc, w_lstm, pat_r, ext, fw, bw, l2)
    l3 = np.zeros(DC * Nr, dtype=np.float32)
    con = np.zeros(3 * DC * Nr, dtype=np.float32)
    O.cnn_forward(HB, DC, S, Tr, 0, 0, 1.0, hw, it, pat_r, w_cnn, l2, con, l3)
    cat = np.concatenate([l3.reshape(Nr, DC), ext.reshape(Nr, E)[:, 11:12]], axis=1).astype(np.float32)
    ctx = np.zeros(C * N, dtype=np.float32)
    ctx_mv = None
    if context_mv:
        ctx_mv = np.concatenate([0.2 * rng.standard_normal(C), rng.uniform(0.4, 1.5, C)]).astype(np.float32)
        ctx_mv[C + 2] = 1e-6   # a vanishing deviation counts as 1
        ctx_mv.tofile(tmp_path / "context.mv")
    O.wavnetc_load_context(C, S, N, Tr, False, np.ascontiguousarray(cat.reshape(-1)), frame_index.reshape(-1), ctx_mv, pat, ctx)

    # ---- oracle: sample-rate part --------------------------------------------------------------------------------
    backend = _CondOracleBackend()
    backend.ctx_grad = np.zeros(C * N, dtype=np.float32)
    ref = networks.WaveNet(backend, nb, S, T, Q=Q, R=R, K=K, C=C, cnn_tanh=1, dilation_cycle=3)
    W = WD.init_weights({k: len(ref.buf[k]["W"]) for k in ref.weight_names()}, seed=3)
    for k, w in W.items():
        ref.buf[k]["W"][:] = w
    ref.set_inputs(pat, onehot, ctx, target)
    ref.forward()
    ref.calculate_error()
    ref.backward()
    cat_err = np.zeros(C * Nr, dtype=np.float32)
    O.wavnetc_sum_context_grad(C, S, RES, Nr, N, pat_r, pat, backend.ctx_grad, cat_err)
    cat_err = cat_err.reshape(Nr, C)
    l3_err = np.zeros((Nr, DC), dtype=np.float32)
    l3_err[valid_r] = cat_err[valid_r, :DC]
    l3_err = np.ascontiguousarray(l3_err.reshape(-1))
    l2_err = np.zeros(HB * Nr, dtype=np.float32)
    dw_cnn = np.zeros_like(w_cnn)
    O.cnn_backward(HB, DC, S, Tr, 0, 0, 1.0, hw, it, pat_r, w_cnn, l2, l3, l3_err, con, l2_err, dw_cnn)
    skip_err = np.zeros(E * Nr, dtype=np.float32)
    dw_lstm = np.zeros_like(w_lstm)
    O.lstm_backward(desc, w_lstm, pat_r, ext, l2_err, fw, bw, skip_err, dw_lstm)
    W["exL2"], W["exL3"] = w_lstm, w_cnn
    dW_ref = {k: ref.buf[k]["dW"] for k in ref.weight_names()}
    dW_ref["exL2"], dW_ref["exL3"] = dw_lstm, dw_cnn

    # ---- the library, from the network file ---------------------------------------------------------------------
    doc = PC.pkg().specs.wavenet_network_doc(nb, Q, R, K, C, 1, 3)
    cond = [{"size": E, "name": "exL1", "type": "externalloader", "bias": 1.0, "resolution": RES},
            {"size": E, "name": "exSkip", "bias": 1.0, "type": "skipini", "resolution": RES},
            {"size": HB, "name": "exL2", "bias": 1.0, "type": "blstm", "resolution": RES},
            {"size": DC, "name": "exL3", "bias": 1.0, "type": "cnn", "window_width": "%d*1" % DC,
             "window_tap_interval": "%d*1" % DC, "tanhoutput": 0, "resolution": RES},
            {"size": C, "name": "exAdd", "bias": 1.0, "type": "skipcat", "resolution": RES,
             "preSkipLayer": "exL3,exSkip", "preSkipLayerDim": "0_%d_11_12" % DC,
             "layerFlag": "wavenetConditionInputLayer"}]
    doc["layers"] = doc["layers"][:1] + cond + doc["layers"][1:]
    if context_mv:
        for layer in doc["layers"]:
            if layer["type"] == "wavnetc":
                layer["contextMV"] = str(tmp_path / "context.mv")
        bad = json.loads(json.dumps(doc))
        (tmp_path / "short.mv").write_bytes(ctx_mv[:-1].tobytes())
        [l for l in bad["layers"] if l["type"] == "wavnetc"][1]["contextMV"] = str(tmp_path / "short.mv")
        with pytest.raises(RuntimeError, match="mean variance dim unequal"):
            capi.Network(json.dumps(bad), S, T + 6, mdn_config=[1, 0, Q, 0, 1, -1])
    net = capi.Network(json.dumps(doc), S, T + 6, mdn_config=[1, 0, Q, 0, 1, -1])
    assert net.layer("exL2")["resolution"] == RES and net.layer("emb")["resolution"] == 1
    for L in net.layers:
        if L["weight_count"]:
            assert L["weight_count"] == W[L["name"]].size, L["name"]
            L["weights"].copy_(torch.from_numpy(W[L["name"]]))
    net.set_external_input("exL1", PC.dev(data.reshape(-1)), Tr, PC.dev(mean_std))
    with pytest.raises(RuntimeError, match="computes the conditioning features itself"):
        net.set_context(PC.dev(ctx))
    for _ in range(2):
        net.load_sequences(PC.dev(pat), T, min(lengths), PC.dev(frame_index.reshape(-1)), PC.dev(target))
        net.forward()
        loss = float(net.calculate_error().item())
        net.backward()
        net.check()
        torch.cuda.synchronize()
        assert PC.relerr(net.layer("exL1")["outputs"][: ext.size].cpu().numpy(), ext) < 1e-6
        assert PC.relerr(net.layer("exAdd")["outputs"][: cat.size].cpu().numpy(), cat.reshape(-1)) < TOL
        ref_loss = float(ref.loss[0])
        assert abs(loss - ref_loss) <= TOL * abs(ref_loss)
        assert PC.relerr(net.layer("exAdd")["errors"][: cat_err.size].cpu().numpy(), cat_err.reshape(-1)) < TOL
        worst = 0.0
        for L in net.layers:
            if L["weight_count"]:
                e = PC.relerr(L["updates"].cpu().numpy(), dW_ref[L["name"]])
                worst = max(worst, e)
                if e > TOL:
                    print("   ", L["name"], e, flush=True)
        assert worst < TOL
    net.close()


def test_full_size_acoustic_backward_is_affine_in_the_targets():
    """benchmark configs[1] at its real size (T = 600, S = 10, 382-512-512-blstm512-blstm512-187), where the oracle
    would take minutes: with the forward state fixed, the SSE error is y - target and every later step of the
    backward pass is linear in it as long as no LSTM delta reaches the clipping bound, so
    dW(t1) + dW(t2) = dW(t1 + t2) + dW(0) for every weight tensor.  A wrong accumulation, a stale buffer (the stored
    output-gate deltas are read-modify-write) or a race between the streams breaks it."""
    import torch

    print("full-size acoustic linearity", flush=True)
    pkg = PC.pkg()
    capi, networks = pkg.capi, PC.networks()
    S, Tmax = 10, 600
    input_size, specs = PC.pkg().specs.acoustic_model_spec()
    rng = np.random.default_rng(77)
    lengths = [int(v) for v in rng.integers(300, Tmax + 1, size=S)]
    T = max(lengths)
    pat = make_pat_types(lengths, T)
    valid = (pat != 0).reshape(T, S)
    x = rng.standard_normal((T, S, input_size)).astype(np.float32)
    x[~valid] = 0
    layers = [{"size": input_size, "name": "input", "type": "input"}]
    layers += [dict(sp, name="l%d" % i) for i, sp in enumerate(specs)]
    net = capi.Network(json.dumps({"layers": layers}), S, Tmax)
    net.randomize(5, 0.08)
    pat_d, x_d = PC.dev(pat), PC.dev(x.reshape(-1))

    def grads(target):
        tgt = target.copy()
        tgt[~valid] = 0
        net.load_sequences(pat_d, T, min(lengths), x_d, PC.dev(tgt.reshape(-1)))
        net.forward()
        net.backward()
        net.check()
        torch.cuda.synchronize()
        return net.updates.clone()

    t1 = (0.05 * rng.standard_normal((T, S, 187))).astype(np.float32)
    t2 = (0.05 * rng.standard_normal((T, S, 187))).astype(np.float32)
    g1, g2, g12, g0 = grads(t1), grads(t2), grads(t1 + t2), grads(np.zeros_like(t1))
    assert float(g1.abs().max()) > 0
    for L in net.layers:
        if not L["weight_count"]:
            continue
        a, b = L["weight_offset"], L["weight_offset"] + L["weight_count"]
        lhs = (g1[a:b] + g2[a:b]).cpu().numpy()
        rhs = (g12[a:b] + g0[a:b]).cpu().numpy()
        assert PC.relerr(lhs, rhs) < TOL, L["name"]
    net.close()


def test_full_size_wavenet_sequencer_matches_layer_by_layer_walk():
    """benchmark configs[3] at its real size (30 blocks, 2 x 16000 samples, 1024 classes): the sequencer (shared sums,
    aliased buffers, fan-in / fan-out tables, side streams, fused delta) against the plain layer-by-layer walk over
    the same kernels, which the shortened-stack tests tie to the oracle.  Loss equal to 1e-6, every weight gradient
    to the tolerance of the split-K atomics' summation order.  What each frame contributes is compared by itself (the last
    product adds 128 terms below one: 128 * 2^-24 per logit, twice that in the log-probability), and each pass's loss with the
    64-bit sum of its own frames (2^-20 per frame for exponential, sum and quotient of a probability at exponents of a few
    units, 2^-22 of the value for its logarithm), so that a frame computed wrongly is not taken for rounding."""
    import torch

    print("full-size wavenet sequencer vs walk", flush=True)
    pkg = PC.pkg()
    capi, networks = pkg.capi, PC.networks()
    nb, Q, R, K, C = 30, 1024, 64, 128, 80
    lengths = [16000, 15000]
    S, T = 2, 16000
    pat, onehot, ctx, target, N = WD.make(lengths, Q, C, upsample=80, seed=4)
    walk = networks.WaveNet(networks.HipBackend(), nb, S, T, Q=Q, R=R, K=K, C=C, cnn_tanh=1)
    W = WD.init_weights({k: len(walk.buf[k]["W"]) for k in walk.weight_names()}, seed=5)
    for k, w in W.items():
        walk.buf[k]["W"].copy_(torch.from_numpy(w))
    pat_d, ctx_d, tgt_d = PC.dev(pat), PC.dev(ctx), PC.dev(target)
    walk.set_inputs(pat_d, PC.dev(onehot), ctx_d, tgt_d)
    walk.forward()
    walk.calculate_error()
    walk.backward()
    net = capi.Network(json.dumps(PC.pkg().specs.wavenet_network_doc(nb, Q, R, K, C, 1, 10)), S, T, mdn_config=[1, 0, Q, 0, 1, -1])
    for L in net.layers:
        if L["weight_count"]:
            L["weights"].copy_(torch.from_numpy(W[L["name"]]))
    net.set_context(ctx_d)
    net.load_sequences(pat_d, T, min(lengths), torch.zeros(N, dtype=torch.float32, device="cuda"), tgt_d)
    net.forward()
    loss = float(net.calculate_error().item())
    net.backward()
    torch.cuda.synchronize()
    ref_loss = float(walk.loss.item())

    def by_frame(logits):
        v = torch.log_softmax(logits[: N * Q].view(N, Q).double(), 1)
        return -v[torch.arange(N, device="cuda"), tgt_d.long()][pat_d != 0]

    frames, ref_frames = by_frame(net.layer("output")["outputs"]), by_frame(walk.buf["output"]["out"])
    assert float((frames - ref_frames).abs().max()) <= 2 * 128 * 2.0 ** -24
    for total, each in ((loss, frames), (ref_loss, ref_frames)):
        exact = float(each.sum())
        assert abs(total - exact) <= len(each) * 2.0 ** -20 + exact * 2.0 ** -22
    assert abs(loss - ref_loss) <= 1e-6 * abs(ref_loss)
    for L in net.layers:
        if L["weight_count"]:
            assert PC.relerr(L["updates"].cpu().numpy(), walk.buf[L["name"]]["dW"].cpu().numpy()) < TOL, L["name"]
    walk.close()
    net.close()


def test_gatedact_layer_and_dft_post_output_in_a_network_file():
    """Two more layer types of the reference's registry through the sequencer: `gatedact` inside a small stack with
    an sse output, and a `dft` post-output layer (two resolutions, spectral distance type 1, phase term) after a
    stack that produces a waveform -- each against the oracle's primitives."""
    import torch

    print("gatedact and dft layers in network files", flush=True)
    capi = PC.pkg().capi
    rng = np.random.default_rng(21)

    # ---- gatedact ------------------------------------------------------------------------------------------------
    P, D, Q, lengths = 6, 8, 5, [20, 13, 17]
    S, T = len(lengths), max(lengths)
    N = S * T
    pat = make_pat_types(lengths, T)
    valid = pat != 0
    x = rng.standard_normal((N, P)).astype(np.float32); x[~valid] = 0
    tgt = rng.standard_normal((N, Q)).astype(np.float32); tgt[~valid] = 0
    w1 = rng.uniform(-0.5, 0.5, P * 2 * D + 2 * D).astype(np.float32)
    w2 = rng.uniform(-0.5, 0.5, D * Q + Q).astype(np.float32)
    h1, g, y = np.zeros(2 * D * N, np.float32), np.zeros(D * N, np.float32), np.zeros(Q * N, np.float32)
    O.dense_forward(P, 2 * D, N, 0, 1.0, w1, x.reshape(-1), h1)
    O.gated_forward(D, N, pat, h1, g)
    O.dense_forward(D, Q, N, 1, 1.0, w2, g, y)
    ref_loss = O.sse_error(Q, N, pat, y, tgt.reshape(-1))
    ey, eg, eh1 = np.zeros(Q * N, np.float32), np.zeros(D * N, np.float32), np.zeros(2 * D * N, np.float32)
    dw1, dw2 = np.zeros_like(w1), np.zeros_like(w2)
    O.sse_backward(Q, N, pat, y, tgt.reshape(-1), ey)
    O.dense_backward(D, Q, N, 1, 1.0, w2, g, y, ey, eg, dw2)
    O.gated_backward(D, N, pat, h1, eg, eh1)
    O.dense_backward(P, 2 * D, N, 0, 1.0, w1, x.reshape(-1), h1, eh1, None, dw1)
    doc = {"layers": [{"size": P, "name": "input", "type": "input"},
                      {"size": 2 * D, "name": "pre", "type": "feedforward_identity", "bias": 1.0},
                      {"size": D, "name": "gate", "type": "gatedact", "bias": 1.0},
                      {"size": Q, "name": "out", "type": "feedforward_tanh", "bias": 1.0},
                      {"size": Q, "name": "post", "type": "sse"}]}
    net = capi.Network(json.dumps(doc), S, T)
    net.layer("pre")["weights"].copy_(torch.from_numpy(w1))
    net.layer("out")["weights"].copy_(torch.from_numpy(w2))
    net.load_sequences(PC.dev(pat), T, min(lengths), PC.dev(x.reshape(-1)), PC.dev(tgt.reshape(-1)))
    net.forward()
    loss = float(net.calculate_error().item())
    net.backward()
    torch.cuda.synchronize()
    assert abs(loss - ref_loss) <= TOL * abs(ref_loss)
    assert PC.relerr(net.layer("gate")["outputs"][: g.size].cpu().numpy(), g) < TOL
    assert PC.relerr(net.layer("pre")["updates"].cpu().numpy(), dw1) < TOL
    assert PC.relerr(net.layer("out")["updates"].cpu().numpy(), dw2) < TOL
    net.close()

    # ---- dft -------------------------------------------------------------------------------------------------------
    P, Hd, T, maxT = 4, 16, 900, 1000
    pat = make_pat_types([T], T)
    x = rng.standard_normal((T, P)).astype(np.float32)
    tgt = (0.3 * rng.standard_normal(T)).astype(np.float32)
    w1 = rng.uniform(-0.5, 0.5, P * Hd + Hd).astype(np.float32)
    w2 = rng.uniform(-0.5, 0.5, Hd + 1).astype(np.float32)
    h1, y = np.zeros(Hd * T, np.float32), np.zeros(T, np.float32)
    O.dense_forward(P, Hd, T, 1, 1.0, w1, x.reshape(-1), h1)
    O.dense_forward(Hd, 1, T, 0, 1.0, w2, h1, y)
    res = [(128, 100, 25), (64, 64, 16)]
    gamma, zeta, dis, beta = 0.7, 0.4, 1, 0.3
    src = np.zeros(maxT, np.float32); src[:T] = y
    tg = np.zeros(maxT, np.float32); tg[:T] = tgt
    ey, ref_loss = np.zeros(maxT, np.float64), 0.0
    for (Nf, Nw, Hs) in res:
        gbuf = np.zeros(maxT, np.float32)
        ref_loss += O.dft_spectral_loss(dis, Nf, Nw, Hs, 0, maxT, T, gamma, 1e-5, src.copy(), tg.copy(), gbuf)
        gbuf[T:] = 0
        ey += gbuf
        ref_loss += O.dft_phase_loss(Nf, Nw, Hs, 0, maxT, T, zeta, src.copy(), tg.copy(), gbuf)
        gbuf[T:] = 0
        ey += gbuf
    ey = (ey[:T] + beta * (y.astype(np.float64) - tgt)).astype(np.float32)   # waveform MSE term: gradient only
    eh1, dw1, dw2 = np.zeros(Hd * T, np.float32), np.zeros_like(w1), np.zeros_like(w2)
    O.dense_backward(Hd, 1, T, 0, 1.0, w2, h1, y, ey, eh1, dw2)
    O.dense_backward(P, Hd, T, 1, 1.0, w1, x.reshape(-1), h1, eh1, None, dw1)
    doc = {"layers": [{"size": P, "name": "input", "type": "input"},
                      {"size": Hd, "name": "h", "type": "feedforward_tanh", "bias": 1.0},
                      {"size": 1, "name": "wave", "type": "feedforward_identity", "bias": 1.0},
                      {"size": 1, "name": "post", "type": "dft", "gamma": gamma, "zeta": zeta, "specDisType": dis, "beta": beta,
                       "fftLength": 128, "frameLength": 100, "frameShift": 25,
                       "fftLength2": 64, "frameLength2": 64, "frameShift2": 16}]}
    net = capi.Network(json.dumps(doc), 1, maxT)
    net.layer("h")["weights"].copy_(torch.from_numpy(w1))
    net.layer("wave")["weights"].copy_(torch.from_numpy(w2))
    for _ in range(2):
        net.load_sequences(PC.dev(pat), T, T, PC.dev(x.reshape(-1)), PC.dev(tgt))
        net.forward()
        loss = float(net.calculate_error().item())
        net.backward()
        torch.cuda.synchronize()
        assert abs(loss - ref_loss) <= TOL * abs(ref_loss)
        assert PC.relerr(net.layer("wave")["errors"][:T].cpu().numpy(), ey) < TOL
        assert PC.relerr(net.layer("h")["updates"].cpu().numpy(), dw1) < TOL
        assert PC.relerr(net.layer("wave")["updates"].cpu().numpy(), dw2) < TOL
    net.close()
    with pytest.raises(RuntimeError, match="parallel_sequences = 1"):
        capi.Network(json.dumps(doc), 2, maxT)
    doc["layers"][-1]["kappa"] = 1.0
    with pytest.raises(RuntimeError, match="'kappa' term"):
        capi.Network(json.dumps(doc), 1, maxT)


def test_mixture_density_network_file():
    """benchmark config 3's layout in small: ... -> feedforward_identity -> mdn with one untied-variance mixture unit
    (mdn config [1, 0, Lp, 0, D, M]); loss, the error handed to the output layer and the weight gradients against
    the oracle."""
    import torch

    print("mixture density network file", flush=True)
    capi = PC.pkg().capi
    rng = np.random.default_rng(31)
    P, Hd, M, D = 5, 8, 4, 3
    Lp = M + 2 * M * D
    lengths = [14, 9, 14, 11]
    S, T = len(lengths), max(lengths)
    N = S * T
    pat = make_pat_types(lengths, T)
    valid = pat != 0
    x = rng.standard_normal((N, P)).astype(np.float32); x[~valid] = 0
    tgt = rng.standard_normal((N, D)).astype(np.float32); tgt[~valid] = 0
    w1 = rng.uniform(-0.5, 0.5, P * Hd + Hd).astype(np.float32)
    w2 = rng.uniform(-0.5, 0.5, Hd * Lp + Lp).astype(np.float32)
    h1, y = np.zeros(Hd * N, np.float32), np.zeros(Lp * N, np.float32)
    O.dense_forward(P, Hd, N, 1, 1.0, w1, x.reshape(-1), h1)
    O.dense_forward(Hd, Lp, N, 0, 1.0, w2, h1, y)
    para, tmp = np.zeros(N * M * (1 + 2 * D), np.float32), np.zeros(N * M + N, np.float32)
    O.mdn_mixture_forward(N, Lp, 0, M, D, 0.0, pat, y, para)
    ref_loss = O.mdn_mixture_error(N, D, 0, M, D, pat, tgt.reshape(-1), para, tmp)
    ey = np.zeros(Lp * N, np.float32)
    O.mdn_mixture_backward(N, Lp, D, 0, 0, M, D, 0.0, pat, tgt.reshape(-1), para, tmp, ey)
    eh1, dw1, dw2 = np.zeros(Hd * N, np.float32), np.zeros_like(w1), np.zeros_like(w2)
    O.dense_backward(Hd, Lp, N, 0, 1.0, w2, h1, y, ey.copy(), eh1, dw2)
    O.dense_backward(P, Hd, N, 1, 1.0, w1, x.reshape(-1), h1, eh1, None, dw1)
    doc = {"layers": [{"size": P, "name": "input", "type": "input"},
                      {"size": Hd, "name": "h", "type": "feedforward_tanh", "bias": 1.0},
                      {"size": Lp, "name": "out", "type": "feedforward_identity", "bias": 1.0},
                      {"size": D, "name": "post", "type": "mdn"}]}
    net = capi.Network(json.dumps(doc), S, T + 3, mdn_config=[1, 0, Lp, 0, D, M])
    net.layer("h")["weights"].copy_(torch.from_numpy(w1))
    net.layer("out")["weights"].copy_(torch.from_numpy(w2))
    net.load_sequences(PC.dev(pat), T, min(lengths), PC.dev(x.reshape(-1)), PC.dev(tgt.reshape(-1)))
    net.forward()
    loss = float(net.calculate_error().item())
    net.backward()
    torch.cuda.synchronize()
    assert abs(loss - ref_loss) <= TOL * abs(ref_loss)
    assert PC.relerr(net.layer("out")["errors"][: ey.size].cpu().numpy(), ey) < TOL
    assert PC.relerr(net.layer("h")["updates"].cpu().numpy(), dw1) < TOL
    assert PC.relerr(net.layer("out")["updates"].cpu().numpy(), dw2) < TOL
    net.close()
    with pytest.raises(RuntimeError, match="mdn config"):
        capi.Network(json.dumps(doc), S, T)


# either side of the line from which a stack of blocks runs as two halves of the samples, a middle that is no workgroup's edge, dilations that
# reach from the later half to the earlier one's beginning and past it, one and several blocks, several sequences
@pytest.mark.parametrize("R,K,nb,cycle,lengths", [(64, 64, 2, 2, [8192, 8100]), (64, 64, 2, 2, [8193, 8100]), (64, 32, 1, 1, [17000]),
                                                  (48, 64, 3, 14, [7301, 7282, 7000]), (32, 64, 15, 15, [33001]), (64, 128, 4, 4, [21111])])
def test_blocks_in_two_halves_of_the_samples(R, K, nb, cycle, lengths):
    """Both ways give the same values bit for bit, in every layer: on the caller's stream alone, with the later half beside it, on another
    stream of the caller's, and replayed from a graph between eager passes."""
    import torch

    print("block halves", R, K, nb, cycle, lengths, flush=True)
    capi = PC.pkg().capi
    Q, C, S, T = 64, 20, len(lengths), max(lengths)
    N = S * T
    pat, onehot, ctx, target, _ = WD.make(lengths, Q, C, upsample=20, seed=2)
    doc = json.dumps(PC.pkg().specs.wavenet_network_doc(nb, Q, R, K, C, 1, cycle))
    fraction = (PC.dev(pat), T, min(lengths), torch.zeros(N, device="cuda"), PC.dev(target))
    ctx = PC.dev(ctx)
    want = None
    for overlap in (False, True):
        net = capi.Network(doc, S, T, mdn_config=[1, 0, Q, 0, 1, -1], overlap=overlap)
        net.randomize(7, 0.1)
        net.set_context(ctx)
        net.load_sequences(*fraction)
        layers = [L for L in net.layers if L["outputs"] is not None]
        values = lambda: [L["outputs"][: N * L["size"]].clone() for L in layers]
        if not overlap:
            net.forward()
            want = values()
            net.close()
            continue

        def same():
            torch.cuda.synchronize()
            for L, a, b in zip(layers, values(), want):
                assert torch.equal(a.view(torch.int32), b.view(torch.int32)), L["name"]

        def spoil():
            for L in layers[1:]:
                if L["type"] != layers[-1]["type"] and L["outputs"].data_ptr() != layers[-1]["outputs"].data_ptr():
                    L["outputs"].zero_()  # (padding slots of some layers stay as they are: zeros, as in a new network)
        net.forward()
        same()
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            net.forward()
        same()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            net.forward()
        for _ in range(3):
            spoil()
            graph.replay()
            same()
            net.forward()
            same()
        net.close()
