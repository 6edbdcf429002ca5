"""GPU parity tests (through the C ABI) for the matrix product seam, dense / SSE layers and the LSTM.
Tolerance: 1e-4 on the L2-normalised difference per tensor (fp32, different summation order);
masking and indexing are asserted bit-exactly inside parity_cases."""
import os
import re

import pytest

import parity_cases as PC

pytestmark = pytest.mark.gpu
TOL = 1e-4


@pytest.mark.parametrize("m,n,k,tA,tB,acc", [
    (128, 128, 64, 0, 0, 0), (128, 128, 64, 1, 0, 0), (128, 128, 64, 0, 1, 0),
    (382, 800, 256, 0, 0, 1), (256, 800, 382, 1, 0, 0), (382, 256, 800, 0, 1, 0),
    (187, 333, 77, 0, 0, 0), (5, 3, 2, 1, 0, 1), (1, 1, 1, 0, 0, 0), (130, 129, 17, 0, 1, 1),
])
def test_matrix_product(m, n, k, tA, tB, acc):
    print("gemm case", m, n, k, tA, tB, acc, flush=True)
    assert PC.run_gemm_case(m, n, k, tA, tB, acc, seed=m + n + k) < TOL


# Launches whose last level of large tiles is full enough for eight waves per tile: 212 to 256 tiles, two levels, four levels; edges
# and ends of k that are no multiple of the tile, of four, of a vector.  Tolerance: k products of six parts each in steps of sixteen,
# 6 k / 16 roundings of 2^-24 of the sum so far: sqrt(6 * 2050 / 16) * 2^-24 = 1.7e-6.
@pytest.mark.parametrize("m,n,k,tA,tB,acc", [
    (1000, 3460, 385, 0, 0, 0), (1000, 3460, 388, 1, 0, 1), (2040, 1793, 384, 1, 0, 0), (128, 27300, 420, 0, 0, 0), (1020, 6100, 900, 1, 0, 0),
    (1018, 6101, 769, 0, 0, 1), (1024, 15900, 387, 1, 0, 0), (1021, 3300, 2050, 0, 0, 0),
])
def test_matrix_product_on_eight_waves(m, n, k, tA, tB, acc):
    import torch

    print("gemm case on eight waves", m, n, k, tA, tB, acc, flush=True)
    assert PC.pkg().capi.probe_gemm_plan(m, n, k, 1, tA, not tB)[:2] == (128, 8)
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    A, B, C = (torch.randn(c, device="cuda", generator=gen) for c in (m * k, k * n, m * n))
    want = B.double().reshape(n, k) @ (A.double().reshape(m, k).T if tA else A.double().reshape(k, m)).contiguous()
    if acc:
        want += C.double().reshape(n, m)
    PC.pkg().capi.matrix_product(C, m, n, k, A, tA, B, tB, acc)
    assert ((C.double().reshape(n, m) - want).norm() / want.norm()).item() < 2e-6


# The weight gradients that take eight waves: one wide dense layer (with its bias gradient), tiles at the output's edges, slots that
# are no multiple of the tile.  Tolerance as above: at most 1600 slots per split, 1.5e-6.
@pytest.mark.parametrize("P,D,N", [(1024, 1024, 6200), (1000, 1022, 6401), (1300, 900, 6163)])
def test_wide_dense_gradient_on_eight_waves(P, D, N):
    import torch

    print("wide dense gradient", P, D, N, flush=True)
    assert PC.pkg().capi.probe_gemm_plan(P, D, N, weight_gradient=True)[:2] == (128, 8)
    gen = torch.Generator(device="cuda").manual_seed(P + D + N)
    x, e = torch.randn(N * P, device="cuda", generator=gen), torch.randn(N * D, device="cuda", generator=gen)
    W, y = torch.zeros(P * D + D, device="cuda"), torch.zeros(N * D, device="cuda")
    updates, below = torch.full((P * D + D,), 3.0, device="cuda"), torch.zeros(N * P, device="cuda")
    want = torch.cat([(e.double().reshape(N, D).T.contiguous() @ x.double().reshape(N, P)).reshape(-1), 0.5 * e.double().reshape(N, D).sum(0)])
    PC.pkg().capi.dense_backward(P, D, N, 0, 0.5, W, x, y, e, below, updates)
    assert ((updates.double() - want).norm() / want.norm()).item() < 3e-6


def test_matrix_product_rejects_double_transpose():
    import torch

    capi = PC.pkg().capi
    a = torch.zeros(4, device="cuda")
    with pytest.raises(RuntimeError):
        capi.matrix_product(a, 2, 2, 2, a, 1, a, 1, 0)


@pytest.mark.parametrize("P,D,N,act", [
    (382, 512, 600, 1), (512, 187, 600, 0), (33, 65, 130, 2), (64, 64, 256, 3),
    # small layers, long contraction (the shapes of a WaveNet-style stack's 1x1 layers): split-K weight gradients
    # with one, several and ragged tiles, sizes that are not multiples of the tile
    (64, 128, 3000, 0), (128, 1024, 777, 1), (80, 20, 1501, 2), (12, 8, 200, 0), (128, 132, 999, 3),
])
def test_dense(P, D, N, act):
    print("dense case", P, D, N, act, flush=True)
    assert PC.run_dense_case(P, D, N, act, 1.0, seed=P + D) < TOL


@pytest.mark.parametrize("P,D,N,bias", [
    # narrow layers over long inputs take the split-K path that sums partial products and carries the bias
    # gradient (row sums of the errors, times the layer's bias value) along; 300 x 300 is too large an output for it and
    # takes the atomic path with its separate column sum
    (64, 128, 3000, 0.5), (64, 64, 5000, 2.0), (100, 96, 2500, 0.25), (300, 300, 2500, 0.5),
])
def test_dense_bias_value_scales_the_bias_gradient(P, D, N, bias):
    print("dense bias case", P, D, N, bias, flush=True)
    assert PC.run_dense_case(P, D, N, 0, bias, seed=P + D + N) < TOL


def test_sse():
    print("sse case", flush=True)
    assert PC.run_sse_case(187, [40, 33, 40, 12], seed=2) < 1e-5


@pytest.mark.parametrize("P,L,bidir,lengths", [
    (24, 64, False, [9, 9, 9]),
    (24, 64, False, [12, 7, 12, 5]),
    (40, 128, True, [10, 10]),
    (40, 128, True, [14, 6, 11, 14, 3]),
    (50, 256, False, [20, 20, 20, 15]),
    (48, 512, True, [16, 9, 13, 16, 16, 5, 16, 12, 10, 16]),
    (33, 256, True, [1]),
    (33, 128, False, [6] * 20),
    (32, 512, False, [8, 8, 5, 8]),        # 512 cells per direction: the largest recursion kernel
    (32, 1024, True, [7, 5, 7]),
    (20, 256, False, [5] * 24),            # more than 16 parallel sequences with 256 cells
    (16, 128, True, [1, 1]),               # a single time step, two sequences
    (24, 256, True, [7, 4, 7] * 6),        # 18 parallel sequences, bidirectional: the recursion that spans the XCDs
    (24, 128, False, [3, 9, 1, 9, 2]),     # very ragged, one sequence of a single step among longer ones
    # 2400 slots of which a third is valid: the layer lists the valid slots itself and its weight gradients sum over those
    (24, 128, True, [300, 50, 300, 20, 100, 300, 7, 1]),
    (20, 64, False, [1, 600, 1, 1]),       # the same for a forward-only layer: one long sequence beside three single frames
    # geometries without a persistent recursion kernel: step-by-step recursion
    (12, 64, True, [30, 23]),              # 32 cells per direction (the reference example's conditioning BLSTM)
    (7, 20, False, [9, 4, 9]),             # 20 cells, sizes that are no multiple of anything
    (25, 200, True, [11, 11, 6, 2]),       # 100 cells per direction
    (10, 64, False, [6] * 40),             # more than 32 parallel sequences
    (9, 6, True, [1, 1, 1]),               # a single time step
])
def test_lstm(P, L, bidir, lengths):
    print("lstm case", P, L, bidir, lengths, flush=True)
    assert PC.run_lstm_case(P, L, bidir, lengths, seed=len(lengths) + L) < TOL


# the sums over the patterns with two cells and one cell per thread: a workgroup's cells and one more, chunks that end inside
# a row of workgroups' patterns
@pytest.mark.parametrize("P,L,bidir,lengths", [(3, 2, True, [5, 2]), (4, 500, True, [9, 8]), (5, 258, False, [17, 3]), (5, 257, False, [16]),
                                               (6, 30, True, [2100, 1999]), (3, 7, False, [700] * 6)])
def test_lstm_bias_and_peephole_gradients(P, L, bidir, lengths):
    print("lstm bias and peepholes", P, L, bidir, lengths, flush=True)
    assert PC.run_lstm_case(P, L, bidir, lengths, seed=L) < TOL


def test_lstm_clip_and_repeat_backward():
    """Large errors activate the [-1,1] clip; a second backward without load_sequences adds the stored
    output-gate deltas, as in the reference."""
    print("lstm clip case", flush=True)
    assert PC.run_lstm_case(24, 64, False, [10, 6, 10], seed=4, wscale=0.5, escale=20.0) < TOL
    assert PC.run_lstm_case(24, 128, True, [10, 6, 10], seed=5, wscale=0.5, escale=20.0, repeat_backward=True) < TOL


def test_weight_gradients_spread_between_runs():
    """The weight gradients are summed with fp32 atomics or per-split partial sums, so their bits may depend on the
    order in which workgroups finish.  Three passes over the same inputs: the layer's errors must be bit-identical
    (the recursion and the error products have a fixed summation order), the weight gradients within 1e-5
    L2-normalised of each other (the parity tolerance against the oracle is 1e-4)."""
    import numpy as np
    import torch

    print("lstm run-to-run spread", flush=True)
    capi = PC.pkg().capi
    P, L, S, T = 96, 512, 10, 160
    rng = np.random.default_rng(11)
    lengths = [int(v) for v in rng.integers(80, T + 1, size=S)]
    lengths[0] = T
    W, x, outerr = PC.lstm_inputs(P, L, True, S, T, lengths, 1)
    pat = PC.make_pat_types(lengths, T)
    Wd, xd, pd, ed = PC.dev(W), PC.dev(x), PC.dev(pat), PC.dev(outerr)
    out = torch.zeros(L * T * S, device="cuda")
    layer = capi.Lstm(P, L, True, S, T)
    runs = []
    for _ in range(3):
        ex = torch.zeros(P * T * S, device="cuda"); dW = torch.zeros_like(Wd)
        layer.load_sequences(pd, T, min(lengths))
        layer.forward(Wd, xd, out)
        layer.backward(Wd, xd, out, ed.clone(), ex, dW)
        layer.check()
        torch.cuda.synchronize()
        runs.append((ex.cpu().numpy().copy(), dW.cpu().numpy().copy()))
    layer.close()
    for ex, dW in runs[1:]:
        assert np.array_equal(ex, runs[0][0])
        assert PC.relerr(dW, runs[0][1]) < 1e-5


@pytest.mark.parametrize("L,bidir,S,T,cuts", [
    (512, True, 10, 60, [45]), (512, True, 10, 60, [1, 30, 59]), (256, False, 7, 50, [37]), (128, True, 3, 9, [2, 3]),
])
def test_lstm_recursion_in_several_launches_is_the_same_recursion(L, bidir, S, T, cuts):
    """The backward recursion run as ranges of its steps, and the error product for the preceding layer computed for
    the time steps that are final early and for the rest afterwards: every state array and every error is
    bit-identical to the single launch and the single product."""
    import numpy as np
    import torch

    print("lstm split recursion", L, bidir, S, T, cuts, flush=True)
    capi = PC.pkg().capi
    P = 40
    rng = np.random.default_rng(L + S)
    lengths = [int(v) for v in rng.integers(max(1, T // 2), T + 1, size=S)]
    lengths[0] = T
    W, x, outerr = PC.lstm_inputs(P, L, bidir, S, T, lengths, 3)
    pat = PC.make_pat_types(lengths, T)
    Wd, xd, pd, ed = PC.dev(W), PC.dev(x), PC.dev(pat), PC.dev(outerr)
    out = torch.zeros(L * T * S, device="cuda")
    layer = capi.Lstm(P, L, bidir, S, T)
    assert layer.backward_can_split()
    names = ["herr", "dni", "dig", "dfg", "dog", "cerr"]

    def snapshot(err, ex):
        torch.cuda.synchronize()
        got = {"outerr": err.cpu().numpy().copy(), "ex": ex.cpu().numpy().copy()}
        for d in range(2 if bidir else 1):
            for k in names:
                got["%s%d" % (k, d)] = layer.state(d, k).cpu().numpy().copy()
        return got

    layer.load_sequences(pd, T, min(lengths))
    layer.forward(Wd, xd, out)
    err, ex = ed.clone(), torch.full((P * T * S,), 7.0, device="cuda")
    layer.backward_errors(Wd, err, ex)
    layer.check()
    whole = snapshot(err, ex)

    layer.load_sequences(pd, T, min(lengths))
    layer.forward(Wd, xd, out)
    err, ex = ed.clone(), torch.full((P * T * S,), 7.0, device="cuda")
    edges = [0] + cuts + [T]
    done_lo, done_hi = T, T  # time steps whose columns of ex are written
    for a, b in zip(edges, edges[1:]):
        layer.backward_errors_range(Wd, err, a, b)
        lo, hi = layer.backward_steps_done(b)
        if hi > lo and done_lo == done_hi:
            layer.backward_prev_errors_range(Wd, ex, lo, hi)  # once, as soon as some time steps are final
            done_lo, done_hi = lo, hi
    if done_lo == done_hi:
        done_lo = done_hi = 0
    layer.backward_prev_errors_range(Wd, ex, 0, done_lo)
    layer.backward_prev_errors_range(Wd, ex, done_hi, T)
    layer.check()
    parts = snapshot(err, ex)
    layer.close()
    for k in whole:
        assert np.array_equal(whole[k], parts[k]), k


def test_lstm_abandoned_partial_recursion_does_not_leak_into_the_next_pass():
    """A range of the backward recursion that ends before T leaves its last partial errors in the mailbox for the range
    that continues it.  When the pass is abandoned instead -- the caller starts over at step 0, with or without a new
    fraction in between -- the next recursion must not consume them: every result equals that of a clean pass, a range
    that does not start where the last one ended is refused."""
    import numpy as np
    import torch

    print("lstm abandoned partial recursion", flush=True)
    capi = PC.pkg().capi
    P, L, S, T = 40, 512, 6, 30
    lengths = [T, 21, T, 17, 25, T]
    W, x, outerr = PC.lstm_inputs(P, L, True, S, T, lengths, 4)
    pat = PC.make_pat_types(lengths, T)
    Wd, xd, pd, ed = PC.dev(W), PC.dev(x), PC.dev(pat), PC.dev(outerr)
    out = torch.zeros(L * T * S, device="cuda")
    layer = capi.Lstm(P, L, True, S, T)

    def clean_pass():
        layer.load_sequences(pd, T, min(lengths))
        layer.forward(Wd, xd, out)
        err, ex = ed.clone(), torch.zeros(P * T * S, device="cuda")
        layer.backward_errors(Wd, err, ex)
        layer.check()
        torch.cuda.synchronize()
        return ex.cpu().numpy().copy(), [layer.state(d, k).cpu().numpy().copy() for d in range(2) for k in ("dni", "dog", "cerr")]

    ex0, st0 = clean_pass()
    # abandoned after 11 steps, new fraction loaded
    layer.load_sequences(pd, T, min(lengths))
    layer.forward(Wd, xd, out)
    layer.backward_errors_range(Wd, ed.clone(), 0, 11)
    with pytest.raises(RuntimeError, match="stands at step"):
        layer.backward_errors_range(Wd, ed.clone(), 14, T)   # not where the last range ended
    ex1, st1 = clean_pass()
    assert np.array_equal(ex0, ex1)
    for a, b in zip(st0, st1):
        assert np.array_equal(a, b)
    # abandoned, then a full recursion on the same fraction (no load_sequences: the stored output-gate deltas of the
    # eleven steps already done are added once more, as in the reference; every other array is that of a clean pass)
    layer.load_sequences(pd, T, min(lengths))
    layer.forward(Wd, xd, out)
    layer.backward_errors_range(Wd, ed.clone(), 0, 11)
    layer.load_sequences(pd, T, min(lengths))   # clears the stored output-gate deltas
    err, ex = ed.clone(), torch.zeros(P * T * S, device="cuda")
    layer.backward_errors(Wd, err, ex)
    layer.check()
    torch.cuda.synchronize()
    assert np.array_equal(ex0, ex.cpu().numpy())
    # a range after a forward pass has nothing to continue
    layer.load_sequences(pd, T, min(lengths))
    layer.forward(Wd, xd, out)
    layer.backward_errors_range(Wd, ed.clone(), 0, 7)
    layer.forward(Wd, xd, out)
    with pytest.raises(RuntimeError, match="stands at step"):
        layer.backward_errors_range(Wd, ed.clone(), 7, T)
    ex2, _ = clean_pass()
    assert np.array_equal(ex0, ex2)
    layer.close()


def test_hop_probes_measure_a_plausible_exchange():
    """The measurement hooks behind the benchmark's latency floor: a word between two workgroups of one XCD takes a
    fraction of a microsecond, across XCDs longer, and a 16 KB message longer than a 4 KB one (the reason the forward
    recursion exchanges outputs, 4 KB per workgroup and step, and not partial pre-activations, 16 KB)."""
    capi = PC.pkg().capi
    print("hop probes: word same XCD / across XCDs, message 4 KB / 16 KB", flush=True)
    near = capi.probe_hop_latency(True, False, 500)
    far = capi.probe_hop_latency(False, False, 500)
    m4 = capi.probe_hop_message(4, 500)
    m16 = capi.probe_hop_message(16, 500)
    assert 0.05 < near < 5.0 and near < far < 20.0
    assert near < m4 < m16 < 10.0
    with pytest.raises(RuntimeError, match="4, 8, 12 or 16 KB"):
        capi.probe_hop_message(5, 10)


def test_activation_functions_against_the_cpu_functions():
    """The scalar semantics of the path (Logistic.cuh / Tanh.cuh with the clamps at +-88.72) and the quick forms the
    forward recursion uses instead (hardware exp2 and reciprocal): swept over the whole unclamped range and across
    the clamps, against the CPU oracle's scalar functions.  Tolerances: the exact forms 2e-7 absolute (one rounding of
    exp and of the quotient) and 2e-5 relative, the quick forms 4e-6 (logistic) and 8e-6 (tanh) absolute and 1e-4 relative."""
    import numpy as np
    import torch

    import oracle_lib as O

    capi = PC.pkg().capi
    xs = np.concatenate([np.linspace(-89.5, 89.5, 40001), np.linspace(-12, 12, 40001), np.linspace(-1, 1, 4001),
                         np.array([-88.73, -88.72, -88.71, 88.71, 88.72, 88.73, 0.0, -0.0, 1e-30, -1e-30])]).astype(np.float32)
    L = O.lib()
    want_l = np.array([L.orc_logistic(float(v)) for v in xs], dtype=np.float32)
    want_t = np.array([L.orc_tanh(float(v)) for v in xs], dtype=np.float32)
    xd = PC.dev(xs)
    out = torch.empty_like(xd)
    got = []
    for which in range(4):
        capi.probe_activation(which, xd, out)
        torch.cuda.synchronize()
        got.append(out.cpu().numpy().copy())
    for g, w, quick, tol in ((got[0], want_l, False, 2e-7), (got[1], want_t, False, 4e-7), (got[2], want_l, True, 4e-6),
                             (got[3], want_t, True, 8e-6)):
        assert np.abs(g - w).max() <= tol
        big = np.abs(w) > 1e-30
        rel = np.abs(g[big] - w[big]) / np.abs(w[big])
        # tanh near 0 is a difference of nearly equal numbers in both forms: relative error only where |tanh| >= 0.01
        if w is want_t:
            rel = rel[np.abs(w[big]) >= 0.01]
        assert rel.max() <= (1e-4 if quick else 2e-5)   # the device's and the host's expf differ by an ulp or two
        # the clamps are exact in both forms
        assert np.all(g[xs <= -88.73] == (0.0 if w is want_l else -1.0))
        assert np.all(g[xs >= 88.73] == 1.0)


def test_activation_functions_against_double_precision():
    """Both forms, everywhere as exact as an fp32 exponential and quotient: 2.62 ulp and 1.79e-7 absolute at most over every
    float between 3e-8 and 87 (the largest of these errors are properties of the hardware's exp2), every 61st of them here."""
    import torch
    capi = PC.pkg().capi
    bits = torch.arange(0x33000000, 0x42AE0000, 61, device="cuda", dtype=torch.int32)
    x = bits.view(torch.float32)
    x = torch.cat([x, -x])
    out = torch.empty_like(x)
    for which in range(4):
        capi.probe_activation(which, x, out)
        if which % 2 == 0:
            want = 1 / (1 + torch.exp(-x.double()))
            error, limit = (out.double() - want).abs() / torch.exp2(torch.floor(torch.log2(want)) - 23), 2.7
        else:
            error, limit = (out.double() - torch.tanh(x.double())).abs(), 1.85e-7
        assert error.max().item() <= limit, (which, error.max().item(), x[error.argmax()].item())


def test_lstm_config1_unidirectional():
    """benchmark config 1: P=382, H=256, T=200, S=4 with one sequence of 150 frames."""
    print("lstm config 1", flush=True)
    assert PC.run_lstm_case(382, 256, False, [200, 200, 200, 150], seed=1) < TOL


def test_lstm_gives_up_cleanly_and_recovers():
    """Failure handling, forced from the host: with a spin limit of zero and no pause before the first poll a
    workgroup gives up the moment a neighbour's data is not there yet; every workgroup then drains, the kernels
    end normally, cnt_lstm_check reports the failure, and the same handle works again afterwards."""
    import numpy as np
    import torch

    print("lstm give-up case", flush=True)
    capi = PC.pkg().capi
    P, L, S, T = 24, 512, 6, 40
    rng = np.random.default_rng(3)
    W = torch.from_numpy(rng.uniform(-0.1, 0.1, capi.lib().cnt_lstm_weight_count(P, L, 1)).astype(np.float32)).cuda()
    x = torch.from_numpy(rng.standard_normal(P * T * S).astype(np.float32)).cuda()
    pat = torch.full((T * S,), 2, dtype=torch.int8, device="cuda")
    out = torch.zeros(L * T * S, device="cuda"); err = torch.ones(L * T * S, device="cuda") * 0.01
    ex = torch.zeros(P * T * S, device="cuda"); dW = torch.zeros_like(W)
    layer = capi.Lstm(P, L, True, S, T)
    layer.load_sequences(pat, T, T)
    layer.forward(W, x, out)
    layer.backward(W, x, out, err.clone(), ex, dW)
    layer.check()
    good_out, good_ex, good_dW = out.clone(), ex.clone(), dW.clone()
    layer.set_wait_bounds(0, 0, 0)
    failures = 0
    for _ in range(3):  # an attempt only fails if some poll really comes back incomplete
        # a recursion that gave up is reported by cnt_lstm_check, or by whichever call into the handle comes
        # after the failed launch has ended -- a caller that never checks still gets the error
        try:
            layer.load_sequences(pat, T, T)
            layer.forward(W, x, out)
            layer.backward(W, x, out, err.clone(), ex, dW)
            layer.check()
        except RuntimeError as e:
            assert "gave up" in str(e)
            failures += 1
            torch.cuda.synchronize()
            try:
                layer.check()   # a second failed launch of the same attempt may have ended meanwhile
            except RuntimeError:
                pass
    assert failures >= 1
    layer.set_wait_bounds(1 << 22, 28, 34)
    layer.load_sequences(pat, T, T)
    layer.forward(W, x, out)
    layer.backward(W, x, out, err.clone(), ex, dW)
    layer.check()
    torch.cuda.synchronize()
    assert PC.relerr(out.cpu().numpy(), good_out.cpu().numpy()) < 1e-6
    assert PC.relerr(ex.cpu().numpy(), good_ex.cpu().numpy()) < 1e-6
    assert PC.relerr(dW.cpu().numpy(), good_dW.cpu().numpy()) < 1e-5   # atomic accumulation order differs
    layer.close()


def test_lstm_layers_on_two_streams_at_once():
    """Two layers of the benchmark's size driven from two non-blocking streams at the same time.  Each XCD-local
    recursion wants a compute unit per workgroup and all of them at once; the library orders recursion launches of
    different streams one behind the other, so both passes run to their end with the results each gives alone."""
    import numpy as np
    import torch

    print("two lstm layers on two streams", flush=True)
    capi = PC.pkg().capi
    P, L, S, T = 64, 512, 10, 200
    N = T * S
    rng = np.random.default_rng(9)
    pat = torch.full((N,), 2, dtype=torch.int8, device="cuda")
    layers, data, alone = [], [], []
    for k in range(2):
        W = torch.from_numpy(rng.uniform(-0.08, 0.08, capi.lib().cnt_lstm_weight_count(P, L, 1)).astype(np.float32)).cuda()
        x = torch.from_numpy(rng.standard_normal(P * N).astype(np.float32)).cuda()
        err = torch.from_numpy((0.1 * rng.standard_normal(L * N)).astype(np.float32)).cuda()
        layer = capi.Lstm(P, L, True, S, T)
        out = torch.zeros(L * N, device="cuda"); ex = torch.zeros(P * N, device="cuda"); dW = torch.zeros_like(W)
        layer.load_sequences(pat, T, T)
        layer.forward(W, x, out)
        layer.backward(W, x, out, err.clone(), ex, dW)
        layer.check()
        layers.append(layer); data.append((W, x, err)); alone.append((out.clone(), ex.clone(), dW.clone()))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = []
    for k in range(2):
        W, x, err = data[k]
        out = torch.zeros(L * N, device="cuda"); ex = torch.zeros(P * N, device="cuda"); dW = torch.zeros_like(W)
        got.append((out, ex, dW))
    torch.cuda.synchronize()
    for _ in range(3):   # forward and backward recursions of the two layers interleaved on the two streams
        for k in range(2):
            W, x, _ = data[k]
            layers[k].load_sequences(pat, T, T, stream=streams[k])
            layers[k].forward(W, x, got[k][0], stream=streams[k])
        for k in range(2):
            W, x, err = data[k]
            # a bidirectional layer leaves its output errors as they are: the same buffer serves every pass
            layers[k].backward(W, x, got[k][0], err, got[k][1], got[k][2], stream=streams[k])
    torch.cuda.synchronize()
    for k in range(2):
        layers[k].check()
        assert PC.relerr(got[k][0].cpu().numpy(), alone[k][0].cpu().numpy()) < 1e-6
        assert PC.relerr(got[k][1].cpu().numpy(), alone[k][1].cpu().numpy()) < 1e-6
        assert PC.relerr(got[k][2].cpu().numpy(), alone[k][2].cpu().numpy()) < 1e-5
        layers[k].close()


def test_lstm_step_by_step_recursion_equals_the_persistent_kernels(monkeypatch):
    """The two implementations of the recursion on a geometry both cover (clip active, ragged lengths): the handle
    created with CNT_LSTM_STEPWISE set runs step by step."""
    print("lstm stepwise vs persistent", flush=True)
    monkeypatch.setenv("CNT_LSTM_STEPWISE", "1")
    assert PC.run_lstm_case(24, 128, True, [10, 6, 10], seed=5, wscale=0.5, escale=20.0, repeat_backward=True) < TOL
    assert PC.run_lstm_case(30, 256, False, [12, 12, 7], seed=6) < TOL


@pytest.mark.parametrize("L,bidir,lengths", [
    (512, True, [30, 17, 40, 38, 25, 40, 9, 33, 28, 36]),        # a job for the longest, others share
    (256, True, [5, 40, 2, 40, 0, 31, 1, 22, 17, 12]),           # an empty sequence, two teams of an XCD
    (300, True, [40 - 2 * (i % 15) for i in range(20)]),         # sixteen cells per workgroup
    (200, False, [7] * 30 + [40, 39]),                           # two long sequences among many short ones
    (130, False, [3 + (7 * i) % 38 for i in range(64)]),         # as many as are planned, several launches
    (130, False, [3 + (7 * i) % 38 for i in range(65)]),         # one more: dealt evenly
    (512, False, [12, 40, 33]), (512, True, [21, 20, 20, 20, 20, 20, 20, 20] * 2), (600, True, [20, 5, 20, 11, 3] * 4),
])
def test_lstm_sequences_dealt_by_length(L, bidir, lengths):
    """Jobs hold sequences by length and leave out the steps on which all of theirs are padding: every state array, also on the
    padding slots that a longer fraction has used before, is what the step-by-step schedule leaves."""
    import torch

    print("lstm dealt by length", L, bidir, lengths, flush=True)
    capi = PC.pkg().capi
    P, S, T = 16, len(lengths), 40
    fractions = []
    for k, ends in enumerate(([T] * S, lengths)):
        W, x, outerr = PC.lstm_inputs(P, L, bidir, S, T, ends, 5 + k)
        pat = PC.make_pat_types(ends, T).reshape(T, S)
        pat[:, [s for s in range(S) if ends[s] == 0]] = 0
        fractions.append((PC.dev(W), PC.dev(x), PC.dev(outerr), PC.dev(pat.reshape(-1)), min(ends)))
    got = []
    for stepwise in (False, True):
        if stepwise:
            os.environ["CNT_LSTM_STEPWISE"] = "1"
        try:
            layer = capi.Lstm(P, L, bidir, S, T)
        finally:
            os.environ.pop("CNT_LSTM_STEPWISE", None)
        out, ex = torch.zeros(L * T * S, device="cuda"), torch.zeros(P * T * S, device="cuda")
        dW = torch.zeros_like(fractions[0][0])
        for W, x, outerr, pat, shortest in fractions:
            err = outerr.clone()
            layer.load_sequences(pat, T, shortest)
            layer.forward(W, x, out)
            layer.backward(W, x, out, err, ex, dW)
            layer.check()
        r = {"out": out, "err": err, "ex": ex, "dW": dW}
        for d in range(2 if bidir else 1):
            for k in ("ni", "ig", "fg", "og", "c", "h", "dni", "dig", "dfg", "dog", "cerr") + (("herr",) if bidir else ()):
                r["%s%d" % (k, d)] = layer.state(d, k)
        got.append({k: v.cpu().numpy() for k, v in r.items()})
        layer.close()
    for k in got[0]:
        assert PC.relerr(got[0][k], got[1][k]) < TOL, k


@pytest.mark.parametrize("cells", [8, 16])
@pytest.mark.parametrize("L,bidir,lengths", [
    (512, True, [21]), (512, True, [21, 9]), (200, False, [17]), (258, True, [13, 12, 5]),  # a job per sequence
    (512, True, [20, 20, 11, 7, 3] * 4), (150, False, [15] * 9), (300, False, [12, 8]), (100, False, [9, 4]),
])
def test_lstm_cells_per_workgroup_by_the_environment(L, bidir, lengths, cells, monkeypatch):
    """CNT_LSTM_LOCAL_JB: mailboxes, launch and kernel go by the same number of sequences per job, also where a layer would not take
    that many cells per workgroup by itself; sizes without such a kernel go step by step."""
    print("lstm cells per workgroup", cells, L, bidir, lengths, flush=True)
    monkeypatch.setenv("CNT_LSTM_LOCAL_JB", str(cells))
    assert PC.run_lstm_two_recursions(21, L, bidir, lengths, seed=cells + L) < TOL


@pytest.mark.parametrize("L,bidir,lengths", [(256, True, [110, 104, 90]), (256, False, [107]), (600, True, [104] * 34), (1024, True, [106, 105])])
def test_lstm_recursion_clocks(L, bidir, lengths, monkeypatch, capfd):
    """CNT_LSTM_TIMING / CNT_LSTM_TRACE: the recursion kernels with clocks compute the same, and cnt_lstm_check prints what the
    parts of a step took and when every workgroup of a team passed the points of the traced steps."""
    print("lstm recursion clocks", L, bidir, lengths, flush=True)
    monkeypatch.setenv("CNT_LSTM_TIMING", "1")
    monkeypatch.setenv("CNT_LSTM_TRACE", "1")
    assert PC.run_lstm_two_recursions(16, L, bidir, lengths, seed=4) < TOL
    lines = capfd.readouterr().err.splitlines()
    for kind in ("forward", "backward"):
        mean, = [line for line in lines if line.startswith("lstm %s per step" % kind)]
        part = {k: float(re.search(k + r" ([0-9.]+)", mean).group(1)) for k in (r"pause\+poll", "barrier", "loop")}
        assert 0 < part[r"pause\+poll"] < part["loop"] and 0 < part["barrier"] < part["loop"], mean
        traces = [line for line in lines if line.startswith("trace %s block" % kind)]
        assert len(traces) == int(re.search(r"(\d+) workgroups", mean).group(1)) > 0
        for line in traces:
            points = [int(v) for v in line.split(":")[1].split()]
            assert len(points) == 20
            for i in range(0, 20, 5):
                assert 0 < points[i] <= points[i + 1] <= points[i + 2] and 0 < points[i + 3] <= points[i + 4], line


@pytest.mark.parametrize("bidir", [False, True])
def test_lstm_recursion_clocks_count_a_jobs_own_steps(bidir, monkeypatch, capfd):
    """Per-step times are sums over the steps that the jobs took: as many as their sequences are long (where time runs forward one
    more, the slot behind the sequence), not as the fraction is."""
    print("lstm recursion clocks, own steps", bidir, flush=True)
    monkeypatch.setenv("CNT_LSTM_TIMING", "1")
    lengths, L = [107, 30, 64], 512 if bidir else 256
    assert PC.run_lstm_two_recursions(16, L, bidir, lengths, seed=6) < TOL
    lines = capfd.readouterr().err.splitlines()
    mean = {kind: [line for line in lines if line.startswith("lstm %s per step" % kind)][0] for kind in ("forward", "backward")}
    taken = {kind: float(re.search(r"([0-9.]+) steps of a job", line).group(1)) for kind, line in mean.items()}
    alone, behind = sum(lengths) / 3, sum(min(n + 1, 107) for n in lengths) / 3
    want = {"forward": (alone + behind) / 2 if bidir else behind, "backward": (alone + behind) / 2 if bidir else alone}
    assert all(abs(taken[k] - want[k]) < 0.051 for k in want), (taken, want)


def test_lstm_config2_layer_full_length_two_recursions():
    """A BLSTM layer of benchmark config 2 at its full size (512 inputs, 256 cells per direction, T=600, S=10,
    lengths drawn from 300..600): the persistent recursion kernels against the step-by-step schedule.  The CPU
    oracle needs two minutes for this fraction, so the full-length check is the agreement of two independent
    implementations, each of which the shorter cases above compare with the oracle."""
    print("lstm config 2 layer, full length, persistent vs stepwise", flush=True)
    import numpy as np

    rng = np.random.default_rng(2)
    lengths = [int(v) for v in rng.integers(300, 601, size=10)]
    lengths[3] = 600
    assert PC.run_lstm_two_recursions(512, 512, True, lengths, seed=12, wscale=0.08) < TOL


def test_lstm_config2_layer_full_length_against_oracle():
    """The same full-size BLSTM layer (512 inputs, 256 cells per direction, T=600, S=10, lengths drawn from
    300..600) against the CPU oracle: outputs, error to the preceding layer, every weight-gradient class and
    every state array, 1e-4 L2-normalised; exact zeros on padding slots.  The oracle shares its outputs out
    over the host's cores for this one (the sums themselves stay sequential)."""
    print("lstm config 2 layer, full length, against the oracle", flush=True)
    import numpy as np

    import oracle_lib as O

    O.use_all_cores()
    rng = np.random.default_rng(2)
    lengths = [int(v) for v in rng.integers(300, 601, size=10)]
    lengths[3] = 600
    assert PC.run_lstm_case(512, 512, True, lengths, seed=12, wscale=0.08) < TOL


def test_lstm_invalid_geometry_is_an_error():
    capi = PC.pkg().capi
    with pytest.raises(RuntimeError):
        capi.Lstm(10, 129, True, 4, 10)      # odd size of a bidirectional layer
    with pytest.raises(RuntimeError):
        capi.Lstm(10, 0, False, 4, 10)


def test_lstm_partial_recursion_rejects_what_it_cannot_do():
    import torch

    capi = PC.pkg().capi
    T, S = 12, 3
    pat = PC.dev(PC.make_pat_types([T] * S, T))
    # 20 cells: step-by-step recursion, which has no partial form
    small = capi.Lstm(8, 20, False, S, T)
    small.load_sequences(pat, T, T)
    assert not small.backward_can_split()
    W = torch.zeros(int(capi.lib().cnt_lstm_weight_count(8, 20, 0)), device="cuda")
    err = torch.zeros(20 * T * S, device="cuda")
    with pytest.raises(RuntimeError, match="cannot run a range"):
        small.backward_errors_range(W, err, 0, 6)
    small.close()
    layer = capi.Lstm(8, 128, True, S, T)
    layer.load_sequences(pat, T, T)
    assert layer.backward_can_split()
    W = torch.zeros(int(capi.lib().cnt_lstm_weight_count(8, 128, 1)), device="cuda")
    err = torch.zeros(128 * T * S, device="cuda")
    ex = torch.zeros(8 * T * S, device="cuda")
    for a, b in ((0, 0), (5, 4), (-1, 3), (0, T + 1)):
        with pytest.raises(RuntimeError, match="steps"):
            layer.backward_errors_range(W, err, a, b)
    with pytest.raises(RuntimeError, match="time steps"):
        layer.backward_prev_errors_range(W, ex, 3, T + 1)
    assert layer.backward_steps_done(0) == (T, T)
    assert layer.backward_steps_done(T) == (0, T)
    assert layer.backward_steps_done(9) == (3, 9)
    assert layer.backward_steps_done(4) == (8, 8)   # nothing final yet in a bidirectional layer
    layer.close()


@pytest.mark.parametrize("L,bidir,lengths", [
    # one workgroup per job: one cell, the edges of its sixteen-cell waves, sequence groups that do not come out even
    (1, False, [3]), (30, True, [9, 4]), (32, True, [1, 6, 6, 2, 5]), (34, True, [13, 8, 13]), (63, False, [7] * 9),
    (128, True, [21, 3, 17] * 7),
    # teams: the first size above, last workgroups and waves that own few cells, as many jobs as XCDs and one more
    (65, False, [8, 8, 5]), (254, True, [6, 9]), (129, False, [5, 7] * 4), (300, True, [6, 4, 6] * 6), (385, True, [5, 5, 2]),
    # 16 cells per workgroup, two teams per XCD, more jobs than one launch holds
    (512, True, [12, 9] * 10), (257, False, [4, 6]), (450, False, [3] * 7), (512, False, [6, 5] * 20), (512, True, [4] * 70),
    # the first size the step-by-step schedule takes
    (513, False, [3, 2]),
])
def test_lstm_recursion_geometries(L, bidir, lengths):
    """Persistent recursions against the step-by-step schedule at the sizes where their dispatch and their remainders
    change (cells per direction, number of (direction, four sequences) jobs)."""
    print("lstm geometry", L, bidir, lengths, flush=True)
    if bidir and L % 2:
        L += 1
    assert PC.run_lstm_two_recursions(19, L, bidir, lengths, seed=L + len(lengths)) < TOL


@pytest.mark.parametrize("T", [1, 2, 3, 5, 8, 9, 17])
@pytest.mark.parametrize("L,bidir,S", [
    (256, True, 3), (300, True, 4), (70, False, 1),       # jobs of one sequence, 8 cells per workgroup
    (400, True, 7), (130, False, 9),                      # of one and two
    (512, True, 9), (200, False, 21),                     # of two and three
    (300, False, 5), (258, False, 11), (480, False, 30),  # 16 cells per workgroup: one, one and two, three and four
])
def test_lstm_job_sizes_and_batches_of_steps(L, bidir, S, T):
    """Kernels for jobs of one, two and up to four sequences, at step counts around the batches in which their inputs are
    requested (four or eight steps) and their results stored (one to eight): ragged lengths, both directions."""
    print("lstm jobs", L, bidir, S, T, flush=True)
    lengths = [max(1, T - 3 * i % 4) for i in range(S)]
    assert PC.run_lstm_two_recursions(19, L, bidir, lengths, seed=L + S + T) < TOL


@pytest.mark.parametrize("H", [1, 3, 4, 5, 18, 31, 47, 50, 61])
@pytest.mark.parametrize("bidir,lengths", [(True, [9, 4, 6]), (False, [1]), (True, [5, 5, 2, 5, 3]), (False, [13, 2])])
def test_lstm_small_layers_move_their_cells_in_vectors(H, bidir, lengths):
    """One-workgroup recursions whose cells are no multiple of four: the last vector overlaps the one before it, below four
    cells there are no vectors."""
    print("lstm small", H, bidir, lengths, flush=True)
    assert PC.run_lstm_two_recursions(11, H * (2 if bidir else 1), bidir, lengths, seed=H + len(lengths)) < TOL


@pytest.mark.parametrize("L,bidir,S,T,cuts", [(512, True, 3, 26, [3, 8, 17]), (256, True, 8, 14, [1, 2, 7]), (400, False, 20, 11, [2, 6])])
def test_lstm_recursion_resumes_between_batches_of_steps(L, bidir, S, T, cuts):
    """Cuts inside the batches of steps whose inputs are requested and results stored together."""
    test_lstm_recursion_in_several_launches_is_the_same_recursion(L, bidir, S, T, cuts)


@pytest.mark.parametrize("L,bidir,lengths", [
    (1, False, [1]), (3, False, [5, 2]), (8, True, [9, 9, 1]), (10, True, [6, 5, 4, 3, 2]), (50, False, [13] * 4), (128, True, [30, 8, 21, 3, 17]),
    (65, False, [40]), (200, True, [7, 30, 2, 19]), (256, True, [11] * 33), (512, True, [29, 3, 3, 3, 3, 2, 2, 1, 1, 1]), (300, False, [12, 4, 8]),
    (512, False, [21, 5]), (1024, True, [9, 9, 2]), (130, True, [3 + i % 9 for i in range(70)]), (520, False, [6, 4])])
def test_lstm_small_gradients_of_a_whole_backward_call(L, bidir, lengths):
    """In a whole backward call the recursion sums them up on the way (groups of sequences apart, some with no sequence; a job's last
    steps where a batch of them is not full); after the error half alone a launch of their own reads the states.  Both against 64-bit
    sums over the states, the call twice in a row over two fractions.  A sum is rounded once per lane, up to seven times between lanes and
    once per group of sequences, the launch of its own up to 64 / 4 times per chunk of patterns: 24 + groups times 2^-24 of the terms."""
    import torch

    print("lstm small gradients", L, bidir, lengths, flush=True)
    capi = PC.pkg().capi
    S, T, P, bias, dirs = len(lengths), max(lengths), 5, 0.7, 2 if bidir else 1
    H = L // dirs
    gen = torch.Generator(device="cuda").manual_seed(L + S)
    W = torch.empty(int(capi.lib().cnt_lstm_weight_count(P, L, int(bidir))), device="cuda").uniform_(-0.2, 0.2, generator=gen)
    layer = capi.Lstm(P, L, bidir, S, T, bias)
    for shift in (0, 1):
        lens = [max(1, n - shift * (n // 2)) if shift else n for n in lengths]
        pat = torch.tensor([[(1 if t == 0 else 3 if t == n - 1 else 2) if t < n else 0 for n in lens] for t in range(T)], dtype=torch.int8, device="cuda").reshape(-1)
        valid = (pat != 0).reshape(-1, 1)
        x = (torch.randn(T * S, P, device="cuda", generator=gen) * valid).reshape(-1)
        errors = (torch.randn(T * S, L, device="cuda", generator=gen) * valid).reshape(-1)
        out, prev = torch.zeros(T * S * L, device="cuda"), torch.zeros(T * S * P, device="cuda")
        layer.load_sequences(pat, T, min(lens))
        layer.forward(W, x, out)
        dW = [torch.full_like(W, 7.0) for _ in range(2)]
        layer.backward(W, x, out, errors.clone(), prev, dW[0])
        states = [{n: layer.state(d, n).double().reshape(T, S, H) for n in ("dni", "dig", "dfg", "dog", "c")} for d in range(dirs)]
        layer.backward_weights(x, dW[1])
        layer.check()
        at_bias, at_peep = 4 * P * L, 4 * P * L + 4 * L + 4 * L * H
        for d, st in enumerate(states):
            c, before = st["c"], torch.zeros(T, S, H, dtype=torch.float64, device="cuda")
            if d == 0: before[1:] = c[:-1]
            else: before[:-1] = c[1:]
            terms = [bias * st[n] for n in ("dni", "dig", "dfg", "dog")] + [st["dig"] * before, st["dfg"] * before, st["dog"] * c]
            for k, term in enumerate(terms):
                at = (at_bias + k * L if k < 4 else at_peep + (k - 4) * L) + d * H
                bound = (24 + S) * 2.0 ** -24 * term.abs().sum((0, 1))
                for g in dW:
                    assert bool(((g[at:at + H].double() - term.sum((0, 1))).abs() <= bound).all()), (d, k)
    layer.close()


@pytest.mark.parametrize("L,bidir,lengths", [
    (3, False, [5, 2]), (6, True, [7, 7]), (50, False, [13] * 4), (128, True, [30, 8, 21, 30, 17]), (130, False, [9]), (200, True, [7, 7, 2, 5]),
    (512, True, [29, 29, 3, 3, 3, 2, 2, 1, 1, 1]), (300, False, [12, 4, 12]), (130, True, [9 - i % 3 for i in range(70)])])
def test_lstm_peephole_gradients_where_the_last_delta_is_not_finite(L, bidir, lengths):
    """The step a recursion ends with has no earlier cell state, so its delta is in no gradient of an input or forget gate's peephole, whatever
    it is; those gradients are what they are with a finite delta there, bit for bit."""
    import torch

    print("lstm last delta", L, bidir, lengths, flush=True)
    capi = PC.pkg().capi
    S, T, P, dirs = len(lengths), max(lengths), 5, 2 if bidir else 1
    H = L // dirs
    gen = torch.Generator(device="cuda").manual_seed(L + S)
    W = torch.empty(int(capi.lib().cnt_lstm_weight_count(P, L, int(bidir))), device="cuda").uniform_(-0.2, 0.2, generator=gen)
    pat = PC.dev(PC.make_pat_types(lengths, T))
    valid = (pat != 0).reshape(-1, 1)
    layer = capi.Lstm(P, L, bidir, S, T, 0.7)
    x = (torch.randn(T * S, P, device="cuda", generator=gen) * valid).reshape(-1)
    errors = torch.randn(T * S, L, device="cuda", generator=gen) * valid
    out, prev = torch.zeros(T * S * L, device="cuda"), torch.zeros(T * S * P, device="cuda")
    got = []
    for value in (1.0, float("nan")):
        layer.load_sequences(pat, T, min(lengths))
        layer.forward(W, x, out)
        e, dW = errors.clone(), torch.full_like(W, 7.0)
        e[:S, :H] = value
        if bidir:
            e[(T - 1) * S:, H:][valid[(T - 1) * S:, 0]] = value
        layer.backward(W, x, out, e.reshape(-1), prev, dW)
        layer.check()
        got.append(dW[4 * P * L + 4 * L + 4 * L * H:].clone())
        bias = dW[4 * P * L:4 * P * L + 4 * L]
        assert bool(bias.isfinite().all()) == (value == 1.0)
    assert bool(got[0].isfinite().all()) and torch.equal(got[0][:2 * L], got[1][:2 * L])
    layer.close()


@pytest.mark.parametrize("P,L,bidir,lengths", [
    (61, 512, True, [130, 125] + [20] * 18), (382, 300, True, [513] + [70] * 9), (40, 256, False, [700, 1, 1, 1]), (128, 400, True, [65] * 30 + [17] * 8)])
def test_lstm_products_of_a_fraction_with_padding(P, L, bidir, lengths):
    """Input projections and errors of the layer below over the listed slots, against the oracle; slots of padding are zeros."""
    print("lstm products with padding", P, L, bidir, lengths, flush=True)
    assert PC.run_lstm_case(P, L, bidir, lengths, seed=P + L) < TOL


def _product(m, n, k, tA, tB, A, B):
    import torch
    C = torch.empty(m * n, device="cuda")
    PC.pkg().capi.matrix_product(C, m, n, k, A, tA, B, tB, False)
    A64 = (A.view(m, k) if tA else A.view(k, m).t()).double()
    B64 = (B.view(k, n) if tB else B.view(n, k).t()).double()
    return C.view(n, m).t().double(), A64, B64


# sizes around the two tiles' edges, k around the staged depth, every vector width and both orientations; with 3000 rows and more
# 128 x 128 tiles, on eight waves where one operand is k-contiguous and k below 768, on four waves otherwise
# (test_gemm_plans.py)
@pytest.mark.parametrize("m,n,k,tA,tB", [
    (63, 65, 31, False, False), (64, 64, 32, True, False), (66, 130, 33, False, True), (132, 68, 36, True, False),
    (257, 129, 97, False, False), (130, 66, 34, False, True), (1, 1, 1, False, False), (4, 1000, 100, False, True),
    (3100, 3076, 516, True, False), (3076, 3100, 540, False, True),
    # lines of no multiple of four: vectors that cross the end of a line, last lines and last tiles float by float
    (3, 2, 200, False, True), (1, 1, 70, False, True), (2, 1, 35, False, False), (61, 187, 425, True, False), (425, 64, 131, False, True),
    (131, 66, 34, False, True), (129, 255, 99, False, False), (3101, 3077, 517, True, False), (3077, 3101, 541, False, True),
    (3102, 3079, 515, False, False), (3101, 3077, 801, True, False), (3102, 3079, 770, False, False), (3100, 3076, 800, False, False),
])
def test_matrix_product_is_as_exact_as_fp32_sums(m, n, k, tA, tB):
    """The operands are multiplied as three bf16 parts each: what the six part products leave out is below 2^-25 of
    |a||b| per term, and every sum is fp32, so the bound of a plain fp32 product holds: (k + 2) * 2^-24 * |A||B|."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + 7 * n + 31 * k)
    A = torch.randn(m * k + 1, device="cuda", generator=g) * torch.exp2(
        torch.randint(-20, 20, (m * k + 1,), device="cuda", generator=g).float())
    A = A[1:] if k % 2 else A[:-1]  # odd cases: an operand aligned to 4 bytes only
    B = torch.randn(n * k, device="cuda", generator=g)
    C, A64, B64 = _product(m, n, k, tA, tB, A, B)
    bound = (k + 2) * 2.0 ** -24 * (A64.abs() @ B64.abs())
    assert bool(((C - A64 @ B64).abs() <= bound).all())


# products of few blocks: eight waves share k in steps of sixteen; blocks and k around 32, 16 and 128, fewer rows than a vector,
# the last sizes before the tiled kernel takes over (640 blocks) and the first behind them
@pytest.mark.parametrize("tA,tB", [(True, False), (False, False), (False, True)])
@pytest.mark.parametrize("m,n,k", [
    (32, 32, 16), (33, 31, 15), (31, 35, 17), (34, 66, 127), (65, 32, 128), (5, 97, 129), (4, 4, 257), (36, 29, 143), (3, 70, 300), (70, 2, 33),
    (640, 1024, 40), (641, 1023, 41), (640, 1025, 24), (96, 100, 2100),
])
def test_matrix_product_of_few_blocks(m, n, k, tA, tB):
    """Bound of an fp32 product in any order of its sums, as above; infinite and missing values in two rows give what a sum of
    single terms gives."""
    import torch
    test_matrix_product_is_as_exact_as_fp32_sums(m, n, k, tA, tB)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    A, B = torch.randn(m * k, device="cuda", generator=g), torch.randn(n * k, device="cuda", generator=g)
    row = (lambda i, q: i * k + q) if tA else (lambda i, q: q * m + i)
    A[row(0, k - 1)], A[row(m - 1, k // 2)] = float("inf"), float("nan")
    C, A64, B64 = _product(m, n, k, tA, tB, A, B)
    assert bool(C[m - 1].isnan().all())
    assert torch.equal(C[0].isposinf(), B64[k - 1] > 0) and torch.equal(C[0].isneginf(), B64[k - 1] < 0)
    bound = (k + 2) * 2.0 ** -24 * (A64.abs() @ B64.abs())
    assert bool(((C - A64 @ B64).abs() <= bound)[1:m - 1].all())


@pytest.mark.parametrize("m,n,k,tA,tB", [(1024, 11900, 256, True, False), (1024, 11900, 256, False, False), (1012, 12001, 300, True, False),
                                         (1936, 5999, 508, False, False), (1024, 11000, 252, True, False),
                                         (1024, 5370, 768, True, False), (1020, 5110, 768, False, False), (1024, 12700, 516, False, False),
                                         (1020, 9000, 800, False, False), (1024, 5370, 900, False, False),
                                         # an eighth and a sixth of the large tiles' rows empty
                                         (430, 21700, 640, True, False), (432, 31350, 512, False, False), (300, 28900, 640, True, False)])
def test_matrix_product_of_short_runs_and_full_generations(m, n, k, tA, tB):
    """Both sides of the lines between the tile sizes, and between four and eight waves, by length of run and number of tiles; rows
    and columns that end inside a tile (test_gemm_plans.py has what each case takes)."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    A, B = torch.randn(m * k, device="cuda", generator=g), torch.randn(n * k, device="cuda", generator=g)
    C, A64, B64 = _product(m, n, k, tA, tB, A, B)
    assert bool(((C - A64 @ B64).abs() <= (k + 2) * 2.0 ** -24 * (A64.abs() @ B64.abs())).all())


@pytest.mark.parametrize("static", [False, True])
@pytest.mark.parametrize("P,D,N", [(32, 32, 16), (20, 33, 120), (37, 35, 130), (5, 4, 7), (3, 60, 200), (60, 2, 200), (256, 2048, 100), (288, 2048, 100),
                                   (100, 90, 2048), (100, 90, 2049)])
def test_weight_gradient_of_few_blocks(P, D, N, static):
    """Both sides of the line between the kernel that sums over all slots in one workgroup, bias gradient included, and
    the one that cuts them (512 blocks, 2048 slots); rows at the edge of a block whose vectors overlap."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(P + D + N)
    x, err = torch.randn(N, P, device="cuda", generator=g), torch.randn(N, D, device="cuda", generator=g)
    dW = torch.full((P * D + D,), 3.0, device="cuda")
    capi = PC.pkg().capi
    (capi.dense_backward_weights_static if static else capi.dense_backward_weights)(P, D, N, 0.5, x, err, dW)
    want, size = err.double().t() @ x.double(), err.double().abs().t() @ x.double().abs()
    assert bool(((dW[:P * D].view(D, P) - want).abs() <= (N + 2) * 2.0 ** -24 * size).all())
    assert bool(((dW[P * D:] - 0.5 * err.double().sum(0)).abs() <= (N + 2) * 2.0 ** -24 * 0.5 * err.double().abs().sum(0)).all())


@pytest.mark.parametrize("P,D,N", [(1024, 1024, 6200), (512, 514, 2501), (401, 600, 3001), (260, 4100, 2600), (4100, 64, 2066)])
def test_bias_gradient_beside_atomic_sums(P, D, N):
    """Weight gradients of several splits bring the bias gradient along: large and small tiles, rows that end
    inside a tile, operands whose rows are no multiple of four long, a last split of another length, one infinite delta."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(P + D + N)
    x, err = torch.randn(N, P, device="cuda", generator=g), torch.randn(N, D, device="cuda", generator=g)
    err[N - 1, D - 1] = float("inf")
    dW = torch.full((P * D + D,), 3.0, device="cuda")
    PC.pkg().capi.dense_backward_weights(P, D, N, 0.5, x, err, dW)
    size = err.double().abs().sum(0)
    assert torch.isposinf(dW[-1])
    assert bool(((dW[P * D:] - 0.5 * err.double().sum(0)).abs()[:-1] <= (N + 2) * 2.0 ** -24 * 0.5 * size[:-1]).all())
    want = err.double().t() @ x.double()
    assert bool(((dW[:P * D].view(D, P) - want).abs() <= (N + 2) * 2.0 ** -24 * (err.double().abs().t() @ x.double().abs()))[:-1].all())


# two to eleven splits of 64 x 64 and 128 x 128 tiles; sums and bias gradients that end inside a quad; few outputs; one split, which
# stores, and one workgroup per block of the output; a row of large tiles
@pytest.mark.parametrize("P,D,N", [(1024, 1028, 653), (1024, 1028, 1200), (1024, 1024, 6200), (512, 514, 2501), (401, 603, 3001), (1026, 7, 1200), (37, 1, 2300),
                                   (2048, 3072, 70), (2049, 3071, 300), (128, 8192, 9000)])
def test_weight_gradient_is_the_same_in_every_call(P, D, N):
    """The splits of a weight gradient meet in a fixed order: the same bits whatever the updates held before, within the bound
    of fp32 sums in any order."""
    import torch
    print("weight gradient repeated", P, D, N, flush=True)
    g = torch.Generator(device="cuda").manual_seed(P + D + N)
    x, err = torch.randn(N, P, device="cuda", generator=g), torch.randn(N, D, device="cuda", generator=g)
    first = None
    for before in (3.0, float("nan"), -1e30, 0.0):
        dW = torch.full((P * D + D + 4,), before, device="cuda")
        PC.pkg().capi.dense_backward_weights(P, D, N, 0.5, x, err, dW)
        assert bool((dW[P * D + D:] == before).all()) or before != before and bool(dW[P * D + D:].isnan().all())
        dW = dW[:P * D + D]
        assert first is None or torch.equal(first, dW)
        first = dW
    want, size = err.double().t() @ x.double(), err.double().abs().t() @ x.double().abs()
    assert bool(((first[:P * D].view(D, P) - want).abs() <= (N + 2) * 2.0 ** -24 * size).all())
    assert bool(((first[P * D:] - 0.5 * err.double().sum(0)).abs() <= (N + 2) * 2.0 ** -24 * 0.5 * err.double().abs().sum(0)).all())


# one, two and four cells per thread of the bias and peephole sums, groups of cells that leave threads idle, one time step (no recurrent
# gradient), chunks of 16 and 64 patterns, large and small tiles, inputs of odd length
@pytest.mark.parametrize("P,L,bidir,lengths", [
    (30, 256, True, [40, 33, 7]), (17, 7, False, [19, 4]), (33, 300, False, [120, 90, 61, 120]), (512, 512, True, [260] * 16),
    (20, 12, True, [1, 1, 1]), (16, 130, True, [9]), (70, 1040, True, [30, 8]), (8, 2, True, [5, 3]),
])
def test_recurrent_weight_gradients_are_the_same_in_every_call(P, L, bidir, lengths):
    """All four sections of a recurrent layer's weight gradient against 64-bit sums of the layer's own states, the same bits whatever
    the updates held before."""
    import torch
    print("recurrent weight gradients", P, L, bidir, lengths, flush=True)
    S, T = len(lengths), max(lengths)
    N, H, dirs, bias = S * T, L // (2 if bidir else 1), 2 if bidir else 1, 0.75
    W, x, outerr = PC.lstm_inputs(P, L, bidir, S, T, lengths, 7)
    layer = PC.pkg().capi.Lstm(P, L, bidir, S, T, bias)
    Wd, xd, err = PC.dev(W), PC.dev(x), PC.dev(outerr)
    layer.load_sequences(PC.dev(PC.make_pat_types(lengths, T)), T, min(lengths))
    out, dW = torch.zeros(L * N, device="cuda"), torch.zeros(len(W), device="cuda")
    layer.forward(Wd, xd, out)
    layer.backward_errors(Wd, err, None)
    first = None
    for before in (3.0, float("nan"), 0.0):
        dW.fill_(before)
        layer.backward_weights(xd, dW)
        assert first is None or torch.equal(first, dW)
        first = dW.clone()
    layer.check()
    X = xd.view(N, P).double()
    want, size = torch.zeros(len(W), device="cuda").double(), torch.zeros(len(W), device="cuda").double()
    rec, peep = 4 * P * L + 4 * L, 4 * P * L + 4 * L + 4 * L * H

    def put(at, a, b):
        want[at:at + a.shape[1] * b.shape[1]] = (a.t() @ b).reshape(-1)
        size[at:at + a.shape[1] * b.shape[1]] = (a.abs().t() @ b.abs()).reshape(-1)

    for d in range(dirs):
        delta = [layer.state(d, k).view(N, H).double() for k in ("dni", "dig", "dfg", "dog")]
        h, c = layer.state(d, "h").view(N, H).double(), layer.state(d, "c").view(N, H).double()
        now, earlier = (slice(0, N - S), slice(S, N)) if d else (slice(S, N), slice(0, N - S))
        for g in range(4):
            put(g * P * L + d * P * H, delta[g], X)
            put(4 * P * L + g * L + d * H, delta[g], torch.full((N, 1), bias, device="cuda").double())
            put(rec + g * L * H + d * H * H, delta[g][now], h[earlier])
        for k, (a, b) in enumerate(((delta[1][now], c[earlier]), (delta[2][now], c[earlier]), (delta[3], c))):
            want[peep + k * L + d * H:peep + k * L + d * H + H] = (a * b).sum(0)
            size[peep + k * L + d * H:peep + k * L + d * H + H] = (a * b).abs().sum(0)
    layer.close()
    assert bool(((first - want).abs() <= (N + 2) * 2.0 ** -24 * size).all())


@pytest.mark.parametrize("reserved", [True, False])
def test_weight_gradient_under_capture(reserved):
    """A captured product uses the stream's scratch where its owner has reserved one, and allocates none where not."""
    import torch
    P, D, N = 1024, 1028, 1300
    capi = PC.pkg().capi
    g = torch.Generator(device="cuda").manual_seed(5)
    x, err, dW = torch.randn(N, P, device="cuda", generator=g), torch.randn(N, D, device="cuda", generator=g), torch.zeros(P * D + D, device="cuda")
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    if reserved:
        capi.gemm_reserve(stream)
    held = capi.lib().cnt_gemm_scratch_buffers()
    capi.dense_backward_weights(P, D, 8, 0.5, x, err, dW)  # (the code is loaded outside the capture)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
        capi.dense_backward_weights(P, D, N, 0.5, x, err, dW, stream=stream)
    assert capi.lib().cnt_gemm_scratch_buffers() == held
    want, size = err.double().t() @ x.double(), err.double().abs().t() @ x.double().abs()
    for _ in range(3):
        dW.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert bool(((dW[:P * D].view(D, P) - want).abs() <= (N + 2) * 2.0 ** -24 * size).all())
        assert bool(((dW[P * D:] - 0.5 * err.double().sum(0)).abs() <= (N + 2) * 2.0 ** -24 * 0.5 * err.double().abs().sum(0)).all())
    del graph
    capi.gemm_release(stream)


@pytest.mark.parametrize("reserved", [True, False])
def test_recurrent_weight_gradients_under_capture(reserved):
    """The same on a stream with and without scratch: replays give what an eager call gives, the latter through atomic additions."""
    import torch
    P, L, lengths = 33, 260, [90, 71, 90]
    S, T = len(lengths), max(lengths)
    W, x, outerr = PC.lstm_inputs(P, L, True, S, T, lengths, 9)
    capi = PC.pkg().capi
    layer = capi.Lstm(P, L, True, S, T)
    Wd, xd, err = PC.dev(W), PC.dev(x), PC.dev(outerr)
    out, dW = torch.zeros(L * S * T, device="cuda"), torch.zeros(len(W), device="cuda")
    layer.load_sequences(PC.dev(PC.make_pat_types(lengths, T)), T, min(lengths))
    layer.forward(Wd, xd, out)
    layer.backward_errors(Wd, err, None)
    layer.backward_weights(xd, dW)
    torch.cuda.synchronize()
    want, stream, graph = dW.clone(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    if reserved:
        capi.gemm_reserve(stream)
    held = capi.lib().cnt_gemm_scratch_buffers()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
        layer.backward_weights(xd, dW, stream=stream)
    assert capi.lib().cnt_gemm_scratch_buffers() == held
    for _ in range(3):
        dW.fill_(7.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(dW, want) if reserved else PC.relerr(dW.cpu().numpy(), want.cpu().numpy()) < 1e-6
    del graph
    capi.gemm_release(stream)
    layer.close()


@pytest.mark.parametrize("m,n,k,tA,tB", [(70, 66, 37, True, False), (3100, 3076, 516, False, False)])
def test_matrix_product_of_infinite_huge_and_missing_values(m, n, k, tA, tB):
    """Values that have no finite bf16 parts give what fp32 arithmetic gives."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(5)
    A, B = torch.randn(m * k, device="cuda", generator=g), torch.randn(n * k, device="cuda", generator=g)
    row = (lambda i, q: i * k + q) if tA else (lambda i, q: q * m + i)
    A[row(3, 5)], A[row(9, 0)], A[row(20, k - 1)] = float("inf"), float("nan"), -float("inf")
    A[row(40, 2)] = 3.402823e38                          # rounds to an infinite bf16 value
    A[row(50, 7)], A[row(50, 8)] = float("inf"), -float("inf")
    B64 = B.view(n, k)
    B64[:, 2] = 0.25                                     # keeps the huge row finite
    B64[11, 5] = 0.0                                     # infinity times zero
    C, A64, B64 = _product(m, n, k, tA, tB, A, B)
    want = torch.zeros_like(C)
    for q in range(k):                                   # term by term: a library product may treat infinities its own way
        want += A64[:, q:q + 1] * B64[q:q + 1, :]
    assert torch.equal(C.isnan(), want.isnan())
    assert torch.equal(C.isposinf(), want.isposinf()) and torch.equal(C.isneginf(), want.isneginf())
    finite = want.isfinite()
    scale = (k + 2) * 2.0 ** -24 * (torch.nan_to_num(A64, 0.0, 0.0, 0.0).abs() @ torch.nan_to_num(B64).abs())
    assert bool(((C - want).abs() <= scale)[finite].all())


# every orientation, row of tiles and vector width; k a multiple of the staged depth, one more, and one tile only
@pytest.mark.parametrize("m,n,k,tA,tB", [(33, 64, 32, True, False), (64, 31, 65, False, True), (130, 96, 96, False, False),
                                         (61, 67, 7, True, False), (3077, 3101, 513, False, True), (3100, 3076, 544, True, False)])
def test_matrix_product_next_to_infinite_and_missing_values(m, n, k, tA, tB):
    """The sums around one that is not finite are formed again with it: they keep the bound of fp32 sums, whichever the
    operands' orientation, and so do those of the rows and columns at the edges."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    A, B = torch.randn(m * k, device="cuda", generator=g), torch.randn(n * k, device="cuda", generator=g)
    (A.view(m, k) if tA else A.view(k, m).t())[m - 1, k - 1] = float("nan")
    (B.view(k, n) if tB else B.view(n, k).t())[0, n - 1] = float("inf")
    C, A64, B64 = _product(m, n, k, tA, tB, A, B)
    assert bool(C[m - 1].isnan().all()) and bool((~C[:m - 1, n - 1].isfinite()).all())
    A64, B64 = torch.nan_to_num(A64, 0.0), torch.nan_to_num(B64, posinf=0.0)
    bound = (k + 2) * 2.0 ** -24 * (A64.abs() @ B64.abs())
    assert bool(((C - A64 @ B64).abs() <= bound)[:m - 1, :n - 1].all())


@pytest.mark.parametrize("everywhere,times", [(True, 4), (False, 20)])
def test_products_full_of_missing_values_stay_in_the_range_of_others(everywhere, times):
    """A pass of a network that has diverged is full of NaN; it takes about as long as another, and some times as long, not
    a hundred, where each sum meets its only NaN at the end (1.0 and 7 measured)."""
    import torch
    m, n, k = 1024, 6000, 1024
    A, B = torch.randn(m * k, device="cuda"), torch.randn(n * k, device="cuda")
    C = torch.empty(m * n, device="cuda")

    def best():
        spans = []
        for _ in range(4):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            PC.pkg().capi.matrix_product(C, m, n, k, A, True, B, False, False)
            end.record()
            torch.cuda.synchronize()
            spans.append(begin.elapsed_time(end))
        return min(spans)

    usual = best()
    A.view(m, k)[:, 0 if everywhere else k - 1:] = float("nan")
    missing = best()
    print("usual %.3f ms, NaN %.3f ms" % (usual, missing), flush=True)
    assert bool(C.isnan().all()) and missing < times * usual


def test_lstm_with_a_huge_input_and_much_padding():
    """The product over the listed slots of a fraction (much padding, enough slots) with a value that has no finite parts."""
    assert PC.run_lstm_case(60, 64, True, [260, 100] * 4, seed=6, huge=True) < TOL


@pytest.mark.parametrize("ea,eb", [(-108, 0), (-118, 40), (-126, 40), (-140, 60), (30, -126), (-66, -66), (-115, 110), (95, 0), (110, -20),
                                   (50, 46), (50, 50)])
@pytest.mark.parametrize("m,n,k,tA,tB", [(130, 66, 300, True, False), (67, 129, 65, False, True)])
def test_matrix_product_over_the_range_of_fp32(m, n, k, tA, tB, ea, eb):
    """Operands whose parts would fall below the smallest bf16 value, subnormal ones, and sums around the limit above which
    they are formed again: the bound of fp32 sums holds, plus half of the smallest fp32 value for the rounding of a subnormal
    result and as much for every term."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(k)
    A = (torch.randn(m * k, device="cuda", generator=g).double() * 2.0 ** ea).float()
    B = (torch.randn(n * k, device="cuda", generator=g).double() * 2.0 ** eb).float()
    C, A64, B64 = _product(m, n, k, tA, tB, A, B)
    bound = (k + 2) * 2.0 ** -24 * (A64.abs() @ B64.abs()) + (k + 1) * 2.0 ** -150
    assert bool(((C - A64 @ B64).abs() <= bound).all())


# both sides of the lines at which a dense layer's weight gradient changes its tile: 64 large tiles, 768 slots per split of k
@pytest.mark.parametrize("P,D,N", [(1000, 1021, 6143), (1000, 1021, 6144), (896, 1024, 7100), (1700, 2048, 1600)])
def test_wide_weight_gradient_on_both_tiles(P, D, N):
    import torch
    g = torch.Generator(device="cuda").manual_seed(N)
    x, err = torch.randn(N, P, device="cuda", generator=g), torch.randn(N, D, device="cuda", generator=g)
    dW = torch.full((P * D + D,), 3.0, device="cuda")
    PC.pkg().capi.dense_backward_weights(P, D, N, 1.0, x, err, dW)
    want, size = err.double().t() @ x.double(), err.double().abs().t() @ x.double().abs()
    assert bool(((dW[:P * D].view(D, P) - want).abs() <= (N + 2) * 2.0 ** -24 * size).all())
    assert bool(((dW[P * D:] - err.double().sum(0)).abs() <= (N + 2) * 2.0 ** -24 * err.double().abs().sum(0)).all())


@pytest.mark.parametrize("static", [False, True])
@pytest.mark.parametrize("P,D,N,bias", [(64, 128, 3000, 0.5), (30, 61, 997, 1.0), (256, 132, 2049, 0.25)])
def test_bias_gradient_of_infinite_huge_and_missing_errors(P, D, N, bias, static):
    """The bias gradients that a weight gradient's launch sums along are fp32 sums of the errors as they are: an infinite
    error gives an infinite sum, one that rounds to an infinite bf16 value a finite one.  Bound of the finite sums: N terms,
    each rounded once per addition, and the product with the bias value."""
    import torch
    capi = PC.pkg().capi
    g = torch.Generator(device="cuda").manual_seed(P + D)
    x, err = torch.randn(N, P, device="cuda", generator=g), torch.randn(N, D, device="cuda", generator=g)
    err[N - 1, 1] = 3.402823e38
    err[3, 2], err[N // 2, 2] = -3.4e38, 3.4e38
    err[0, 5], err[7, D - 1] = float("inf"), -float("inf")
    err[9, 8], err[10, 8] = float("inf"), -float("inf")
    err[N // 3, 11] = float("nan")
    dW = torch.full((P * D + D,), 3.0, device="cuda")
    (capi.dense_backward_weights_static if static else capi.dense_backward_weights)(P, D, N, bias, x, err, dW)
    got, want = dW[P * D:].double(), bias * err.double().sum(0)
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isposinf(), want.isposinf()) and torch.equal(got.isneginf(), want.isneginf())
    finite = want.isfinite()
    assert int((~finite).sum()) == 4
    bound = (N + 2) * 2.0 ** -24 * bias * err.double().abs().sum(0)
    assert bool(((got - want).abs() <= bound)[finite].all())
