"""Weight gradients of a WaveNet stack's residual blocks, all blocks of a launch together (csrc/wavenet_weights.hip), against 64-bit
products of the network's own inputs and errors.

Tolerance: a gradient is a sum over the slots, in runs of 128 slots (8 tiles of six instructions: 48 roundings of at most
2^-24 of the sum so far) that are added up in at most some forty additions more; sqrt(48 + 40) * 2^-24 = 5.6e-7 of the result's
2-norm if they are independent.  Measured: 0.6 to 1.7e-7."""
import json

import numpy as np
import pytest

import parity_cases as PC

pytestmark = pytest.mark.gpu
TOL = 5.6e-7


def passed_network(capi, specs, blocks, R, K, C, lengths, seed=1, spike=None, overlap=True):
    """A stack after one forward and one backward pass, its conditioning features and the mask of its valid slots"""
    import torch

    S, T = len(lengths), max(lengths)
    N, Q = S * T, 16
    gen = torch.Generator(device="cuda").manual_seed(seed)
    net = capi.Network(json.dumps(specs.wavenet_network_doc(blocks, Q, R, K, C, 0, 4)), S, T, mdn_config=[1, 0, Q, 0, 1, -1], overlap=overlap)
    net.weights.copy_(torch.empty(net.n_weights, device="cuda").uniform_(-0.1, 0.1, generator=gen))
    t = torch.arange(T, device="cuda")[:, None]
    valid = t < torch.tensor(lengths, device="cuda")
    pat = valid.to(torch.int8) * 2
    pat[0] = 1
    ctx = torch.randn(N, C, device="cuda", generator=gen) * valid.reshape(-1, 1)
    if spike is not None:
        ctx[spike[0], spike[1]] = spike[2]
    target = torch.randint(0, Q, (N,), device="cuda", generator=gen).float() * valid.reshape(-1)
    net.set_context(ctx.reshape(-1))
    net.load_sequences(pat.reshape(-1).contiguous(), T, min(lengths), torch.zeros(N, device="cuda"), target)
    net.forward()
    net.backward()
    torch.cuda.synchronize()
    return net, ctx, valid


def gradient_errors(capi, specs, blocks, R, K, C, lengths, seed=1, spike=None, overlap=True):
    """2-norm errors of every gradient of every block, and the gradients themselves"""
    import torch

    net, ctx, valid = passed_network(capi, specs, blocks, R, K, C, lengths, seed, spike, overlap)
    S, T = len(lengths), max(lengths)
    N = S * T
    live = valid.reshape(-1, 1)
    of = lambda name, what: net.layer(name)[what].reshape(N, -1).double()  # noqa: E731
    errors, got = {}, {}

    def compare(name, want):
        have = net.layer(name)["updates"]
        got[name] = have.clone()
        errors[name] = ((have.double() - want).norm() / want.norm().clamp_min(1e-300)).item()

    below = "causalSkip"
    for b in range(blocks):
        shift = S * 2 ** (b % 4)
        x, delta = of(below, "outputs"), of("cnn%d" % b, "errors")
        masked = torch.where(live, x, torch.zeros_like(x))
        earlier = torch.zeros_like(x)
        if shift < N:
            earlier[shift:] = masked[:-shift]
        earlier = torch.where(live, earlier, torch.zeros_like(x))
        # [filter][tap: earlier, now, the dead one ahead][channel], then the biases
        conv = torch.stack([delta.T @ earlier, delta.T @ masked, torch.zeros(2 * R, R, device="cuda").double()], 1)
        compare("cnn%d" % b, torch.cat([conv.reshape(-1), delta.sum(0)]))
        part = torch.tanh(ctx.double() @ net.layer("wav%d" % b)["weights"].double().reshape(2 * R, C).T)
        compare("wav%d" % b, (((1 - part * part) * delta).T @ ctx.double()).reshape(-1))
        for name, source in (("out%d" % b, "wav%d" % b), ("sot%d" % b, "temp%d" % b)):
            e = of(name, "errors")
            compare(name, torch.cat([(e.T @ of(source, "outputs")).reshape(-1), e.sum(0)]))
        below = "temp2_%d" % b
    net.close()
    return errors, got


# tails of a tile and of a run, one slot, padding, a look back beyond the first slot, features that are no multiple of four and more
# than one segment of them, 256 skip channels (two jobs), more blocks than fit one launch
@pytest.mark.parametrize("blocks,R,K,C,lengths", [
    (2, 64, 128, 80, [333, 250]), (1, 32, 64, 5, [17]), (2, 64, 256, 65, [1200, 1]), (3, 32, 32, 67, [40, 40, 33]),
    (2, 64, 64, 111, [145]), (2, 32, 128, 4, [1]), (9, 64, 128, 20, [700]), (11, 32, 64, 61, [263, 90]), (1, 64, 128, 112, [5003]),
])
def test_block_weight_gradients(blocks, R, K, C, lengths):
    pkg = PC.pkg()
    print("wavenet block weights", blocks, R, K, C, lengths, flush=True)
    pkg.capi.profile_enable(True)
    try:
        errors, first = gradient_errors(pkg.capi, pkg.specs, blocks, R, K, C, lengths)
        launches = pkg.capi.profile_read()["wavenet_block_weights"][0]
    finally:
        pkg.capi.profile_enable(False)
    assert launches == -(-blocks // 8)
    assert max(errors.values()) < TOL, errors
    _, again = gradient_errors(pkg.capi, pkg.specs, blocks, R, K, C, lengths)
    assert all(bool((first[n] == again[n]).all()) for n in first)  # the order of all additions is fixed


@pytest.mark.parametrize("overlap", [True, False])
def test_block_weight_gradients_of_the_largest_values(overlap):
    """A conditioning feature of 3e38: its split has an infinite part, its gate is flat, so that the gradients stay what they are."""
    pkg = PC.pkg()
    errors, got = gradient_errors(pkg.capi, pkg.specs, 2, 64, 128, 80, [200, 170], spike=(77, 41, 3e38), overlap=overlap)
    assert all(np.isfinite(v.cpu().numpy()).all() for v in got.values())
    assert max(errors.values()) < TOL, errors


def test_block_weight_gradients_under_capture():
    """A forward and a backward pass recorded once: every replay gives the eager passes' gradients, bit for bit."""
    import torch

    pkg = PC.pkg()
    net, ctx, _ = passed_network(pkg.capi, pkg.specs, 9, 64, 128, 20, [300, 211])
    want = net.updates.clone()
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
        net.forward(stream=stream)
        net.backward(stream=stream)
    for _ in range(3):
        net.updates.fill_(5.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert bool((net.updates == want).all())
    net.close()


@pytest.mark.parametrize("R,K,sums", [(64, 128, 16), (48, 96, 12), (32, 256, 4), (64, 32, 0), (48, 80, 0)])
def test_scratch_of_the_common_launches_only_where_they_are_made(R, K, sums):
    """The blocks' scratch of a stack whose widths have the launch for the errors holds 32 x 32 blocks of sums, as many as the job with the most
    has, and 256 more for each of 512 workgroups: 34, 26 and 9 MB.  A stack of other widths sums its weight gradients without."""
    import torch

    pkg = PC.pkg()

    def taken(C):
        doc = json.dumps(pkg.specs.wavenet_network_doc(1, 16, R, K, C, 0, 4))
        pkg.capi.Network(doc, 1, 64, mdn_config=[1, 0, 16, 0, 1, -1]).close()
        before = torch.cuda.mem_get_info()[0]
        net = pkg.capi.Network(doc, 1, 64, mdn_config=[1, 0, 16, 0, 1, -1])
        after = torch.cuda.mem_get_info()[0]
        net.close()
        return before - after

    # (beside the same stack without conditioning features, which never has it; the layers' own buffers and what an allocation is rounded up
    # to differ by less than 4 MB)
    need = 512 * (sums * 1024 + 256) * 4 if sums else 0
    assert abs(taken(20) - taken(0) - need) < 4 << 20
