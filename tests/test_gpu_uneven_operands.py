"""Products whose operands hold values of very different size: every term keeps the bits of its own two values, whatever stands beside
them in a row.  A value that meets a zero takes nothing from the others."""
import json

import pytest

import parity_cases as PC
from torch_models import make_pat_types

pytestmark = pytest.mark.gpu


def _bound(a, b):
    """Of sums of k exact products in fp32 in any order; what is left out of a product is below 2^-25 of it; a product below the normal
    range is off by 2^-149."""
    k = a.shape[1]
    return (k + 2) * 2.0 ** -24 * (a.double().abs() @ b.double().abs().t().contiguous()) + k * 2.0 ** -149


def _close(c, a, b):
    return bool(((c.double() - a.double() @ b.double().t().contiguous()).abs() <= _bound(a, b)).all())


# 64 x 64 tiles and 128 x 128 on four and on eight waves, lines of no multiple of four, k that ends one to three values into a tile, rows fewer
# than a vector
@pytest.mark.parametrize("tA,tB", [(True, False), (False, False), (False, True)])
@pytest.mark.parametrize("m,n,k", [(701, 999, 129), (2, 30001, 163), (29000, 3, 130), (2050, 1795, 300), (1936, 6000, 256), (515, 7200, 1025)])
@pytest.mark.parametrize("what", ["exponents", "late", "large beside zeros", "tiny"])
def test_product_of_uneven_rows(m, n, k, tA, tB, what):
    import torch
    print("uneven product", m, n, k, tA, tB, what, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(m + 7 * n + 31 * k)
    A, B = torch.randn(m * k, device="cuda", generator=gen), torch.randn(n * k, device="cuda", generator=gen)
    a, b = A.view(m, k) if tA else A.view(k, m).t(), B.view(k, n).t() if tB else B.view(n, k)
    if what == "exponents":  # of rows, and of columns of A against those of B
        a *= torch.exp2(torch.randint(-30, 31, (m, 1), device="cuda", generator=gen).float())
        at_k = torch.randint(-13, 14, (1, k), device="cuda", generator=gen).float()
        a *= torch.exp2(at_k)
        b *= torch.exp2(-at_k)
    elif what == "late":
        a[::3], b[::5] = 0.0, 0.0
        a[m - 1], b[n - 1] = 0.0, 0.0
        a[m - 1, k // 3], b[n - 1, k - 1] = 1e-25, 3e20
    elif what == "large beside zeros":
        for at in (3, (k + 31) // 64 * 32 + 5, k - 1):
            a[:, at] *= 2.0 ** 40
            b[:, at] = 0.0
    else:
        a *= 2.0 ** -126
        b *= 2.0 ** 60
    C = torch.full((m * n + 4,), 7.0, device="cuda")
    PC.pkg().capi.matrix_product(C, m, n, k, A, tA, B, tB, False)
    assert bool((C[m * n:] == 7.0).all())
    assert _close(C[:m * n].view(n, m).t(), a, b)


@pytest.mark.parametrize("P,D,N", [(128, 700, 1000), (382, 512, 3000), (425, 1024, 9000)])
def test_dense_forward_of_inputs_in_different_units(P, D, N):
    """Inputs over 10^-4 to 10^4 with weights to match, and two inputs of 2^40 that no unit uses."""
    import torch
    capi = PC.pkg().capi
    gen = torch.Generator(device="cuda").manual_seed(P)
    unit = 10.0 ** torch.randint(-4, 5, (P,), device="cuda", generator=gen).float()
    unused = [3, (P + 31) // 64 * 32 + 5]
    x, w = torch.randn(N, P, device="cuda", generator=gen) * unit, torch.randn(D, P, device="cuda", generator=gen) / unit
    x[:, unused] = 2.0 ** 40
    w[:, unused] = 0.0
    W = torch.cat([w.reshape(-1), torch.zeros(D, device="cuda")])
    y = torch.empty(N * D, device="cuda")
    capi.dense_forward(P, D, N, 0, 1.0, W, x.reshape(-1), y)
    assert _close(y.view(N, D), x, w)


def _passes(layers, P, S, T, dress):
    """Everything that a pass leaves behind, for two sizes of values that all other values meet as zeros."""
    import torch
    capi = PC.pkg().capi
    Q = layers[-1][1]
    doc = {"layers": [{"size": P, "name": "input", "type": "input"}] +
           [{"size": n, "name": "l%d" % i, "type": t, "bias": 1.0} for i, (t, n) in enumerate(layers)] + [{"size": Q, "name": "post", "type": "sse"}]}
    lengths = [T - T // 3 * i // S for i in range(S)]
    pat = PC.dev(make_pat_types(lengths, T))
    valid = (pat != 0).reshape(T, S, 1)
    results = []
    for large in (2.0 ** 7, 2.0 ** 40):
        gen = torch.Generator(device="cuda").manual_seed(len(layers) + P)
        net = capi.Network(json.dumps(doc), S, T)
        net.weights.uniform_(-0.1, 0.1, generator=gen)
        x = torch.randn(T, S, P, device="cuda", generator=gen)
        target = torch.randn(T, S, Q, device="cuda", generator=gen)
        shapes = [P] + [n for _, n in layers]
        w = [net.layer("l%d" % i)["weights"][:net.layer("l%d" % i)["sections"][0]].view(-1, shapes[i]) for i in range(len(layers))]
        dress(large, net, x, target, w)
        x, target = x * valid, target * valid
        net.load_sequences(pat, T, min(lengths), x.reshape(-1).contiguous(), target.reshape(-1).contiguous())
        net.forward()
        net.calculate_error()
        net.backward()
        torch.cuda.synchronize()
        results.append(({L["name"]: (L["outputs"].clone(), L["errors"].clone()) for L in net.layers[1:] if L["name"] != "post" and L["errors"] is not None},
                        {"l%d" % i: net.layer("l%d" % i)["updates"].clone() for i in range(len(layers))}))
        net.close()
    return results, valid


def _same(a, b, what):
    import torch
    assert bool(a.isfinite().all()) and float(a.abs().sum()) > 0, what
    assert torch.equal(a, b), what


def _compare(results, without=None):
    (one, updates_one), (other, updates_other) = results
    for name in one:
        _same(one[name][0], other[name][0], name + " outputs")
        _same(one[name][1], other[name][1], name + " errors")
    for name in updates_one:
        u, v = updates_one[name], updates_other[name]
        if without and without[0] == name:
            keep = without[1](u)
            u, v = u[keep], v[keep]
        _same(u, v, name + " updates")


RECURRENT = [[("feedforward_tanh", 256)], [("blstm", 256)], [("lstm", 192)]]


@pytest.mark.parametrize("seen", ["in both", "in one"])
@pytest.mark.parametrize("layer", RECURRENT, ids=lambda l: l[0][0])
def test_large_inputs_that_no_unit_uses(layer, seen):
    """Inputs of 2^7 or of 2^40 beside zero weights: every value of the pass but those weights' own gradients is the same bit for bit.  The
    others are ordinary numbers, or zeros and a few ones as in coded linguistic inputs."""
    import torch
    P, (kind, n) = 382, layer[0]
    unused = [3, 200] if seen == "in both" else [3]

    def dress(large, net, x, target, w):
        if seen == "in one":
            x.copy_((x > 1.5).float())
            x[:, :, 192:224] = 0.0
        x[:, :, unused] = large
        w[0][:, unused] = 0.0

    def others(u):
        keep = torch.ones(u.numel(), dtype=torch.bool, device="cuda")
        rows = n if kind.startswith("feedforward") else 4 * n
        keep[:rows * P].view(rows, P)[:, unused] = False
        return keep
    results, _ = _passes(layer + [("feedforward_identity", 33)], P, 16, 300, dress)
    _compare(results, ("l0", others))


@pytest.mark.parametrize("kind", ["feedforward_tanh", "blstm", "lstm"])
def test_large_weights_whose_errors_are_zero(kind):
    """Units, or input gates, that one constant unit below holds at exactly 1, by a weight of 2^7 or of 2^40: their errors are zeros, and the errors
    handed down beside theirs are the same bit for bit."""
    n, below = 256, 5

    def dress(large, net, x, target, w):
        l0 = net.layer("l0")
        w[0][below] = 0.0
        l0["weights"][l0["sections"][0]:][below] = 1.0
        rows = w[1] if kind.startswith("feedforward") else w[1].view(4, n, -1)[1]  # input gates
        for unit in (2, 7, n // 2 + 3, n // 2 + 9, n - 1):
            rows[unit] = 0.0
            rows[unit, below] = large
    results, valid = _passes([("feedforward_identity", 256), (kind, n), ("feedforward_identity", 33)], 40, 16, 300, dress)
    assert bool((results[0][0]["l0"][0].view(300, 16, -1)[:, :, below][valid[:, :, 0]] == 1.0).all())
    _compare(results)


@pytest.mark.parametrize("n,Q,T", [(256, 128, 300), (382, 187, 300), (1024, 700, 600)])
def test_large_errors_where_the_inputs_are_zero(n, Q, T):
    """Slots with errors of 2^7 or of 2^40 where the layer's inputs are zeros: the weights' gradients are the same bit for bit."""
    import torch
    slots = [0, 1, T // 2 - 40, T // 2 - 39, T // 2, T // 2 + 1]

    def dress(large, net, x, target, w):
        x[slots] = 0.0
        target[slots] = large
    (one, two), _ = _passes([("feedforward_identity", Q)], n, 16, T, dress)
    _same(one[1]["l0"][:n * Q], two[1]["l0"][:n * Q], "updates")
    assert not torch.equal(one[1]["l0"][n * Q:], two[1]["l0"][n * Q:])
