"""GPU parity (through the C ABI) of the mixture-density layer: flat softmax unit and untied-variance
mixture unit, forward parameters, negative log-likelihood and gradients; 1e-4 L2-normalised per tensor,
zero patterns (padding frames, the reference's index collision) exact."""
import numpy as np
import pytest

import parity_cases as PC

pytestmark = pytest.mark.gpu
TOL = 1e-4


@pytest.mark.parametrize("lengths,M,D,extra", [
    ([5, 5, 5], 4, 6, 0),
    ([6, 3, 6], 2, 2, 0),          # Lp=10: padding frames collide with valid mixture-weight slots
    ([9, 4, 7, 9], 3, 5, 7),       # unit does not start at column 0, leading columns stay zero
    ([40, 25, 33, 40, 12, 40, 40, 31, 40, 20], 16, 60, 0),  # benchmark config 3 geometry, shortened
    ([600, 431, 377, 512, 300, 598, 465, 349, 553, 420], 16, 60, 0),  # benchmark config 3 at full size
    ([12, 7, 12], 8, 12, 4),       # every size a multiple of four behind four leading columns: the 16-byte path
    ([12, 7, 12], 8, 12, 2),       # the same unit two columns further on: not aligned, scalar path
])
@pytest.mark.parametrize("one_call", [False, True])
def test_mixture_unit(lengths, M, D, extra, one_call):
    # one_call: error and gradient through cnt_mdn_error_backward (one pass over the parameters for the units of at most
    # sixteen components whose data is 16-byte aligned, the two kernels in turn for the others)
    print("mdn mixture case", lengths, M, D, extra, one_call, flush=True)
    assert PC.run_mdn_mixture_case(lengths, M, D, extra, seed=M + D, one_call=one_call) < TOL


@pytest.mark.parametrize("M,D,one_call", [(3, 4, False), (3, 4, True), (4, 8, True)])
def test_mixture_unit_variance_floor_and_short_fraction(M, D, one_call):
    print("mdn floor case", M, D, one_call, flush=True)
    assert PC.run_mdn_mixture_case([7, 5], M, D, 0, seed=3, var_floor=0.8, maxT=12, one_call=one_call) < TOL


@pytest.mark.parametrize("lengths,K,extra", [([6, 6], 10, 0), ([9, 5, 7], 257, 3), ([30, 17], 1024, 0)])
def test_softmax_unit(lengths, K, extra):
    print("mdn softmax case", lengths, K, extra, flush=True)
    assert PC.run_softmax_case(lengths, K, extra, seed=K) < TOL


# a frame in registers: one quad, every lane's last quad, one more or less than a lane holds, the largest (1024) and the
# first size past it; four leading columns move the unit's first column, two take it off 16 bytes
@pytest.mark.parametrize("lengths,K,extra", [([3, 1], 4, 0), ([5, 2, 4], 252, 4), ([9, 9], 256, 0), ([6, 2], 260, 4), ([7], 512, 2),
                                             ([4, 3], 516, 0), ([5, 1], 1020, 4), ([2, 2], 1028, 0)])
def test_softmax_unit_sizes_in_registers(lengths, K, extra):
    print("mdn softmax sizes", lengths, K, extra, flush=True)
    assert PC.run_softmax_case(lengths, K, extra, seed=K) < TOL


def test_unsupported_units_are_rejected():
    capi = PC.pkg().capi
    with pytest.raises(RuntimeError):
        capi.Mdn(10, 2, 2, 4, [1, 0, 10, 0, 2, 0])      # sigmoid unit
    with pytest.raises(RuntimeError):
        capi.Mdn(10, 2, 2, 4, [1, 0, 10, 0, 2, 2], tie_variance=True)
    with pytest.raises(RuntimeError):
        capi.Mdn(10, 2, 2, 4, [2, 0, 10, 0, 2, 2])      # length does not match the unit count


@pytest.mark.parametrize("lengths,K,extra,continuous,with_softmax", [
    ([9, 5, 9], 7, 0, False, False), ([12, 12], 3, 4, True, False), ([20, 11, 20, 3], 16, 2, False, True),
    ([6], 1, 0, True, False),
])
def test_sigmoid_unit(lengths, K, extra, continuous, with_softmax):
    print("mdn sigmoid case", lengths, K, extra, continuous, with_softmax, flush=True)
    assert PC.run_sigmoid_case(lengths, K, extra, continuous, seed=K + extra, with_softmax=with_softmax) < TOL


@pytest.mark.parametrize("kind,lengths", [("softmax", [1]), ("softmax", [16000, 15000]), ("mixture", [16000, 15000]),
                                          ("mixture_odd", [1500, 1200, 40]), ("sigmoid", [9000, 8000]), ("both", [600, 411])])
def test_error_is_the_sum_over_frames_whatever_their_order(kind, lengths):
    """The error of a call against the 64-bit sum of what the frames contribute, formed from the unit's own buffers, and the
    same bits in every call.  Bounds: a mixture frame's log-sum is stored, so only the result is rounded (2^-24); -log of a
    probability is good to 2 units in its last place (2^-22 of the sum, whose terms have one sign), plus that rounding."""
    import torch

    print("mdn error sums", kind, lengths, flush=True)
    capi = PC.pkg().capi
    S, T = len(lengths), max(lengths)
    N = S * T
    pat = PC.make_pat_types(lengths, T)
    valid = pat != 0
    rng = np.random.default_rng(N)
    K, M, D = 60, {"mixture": 4, "mixture_odd": 3}.get(kind, 0), 8
    config, Lp, Lt = {"softmax": ([1, 0, K, 0, 1, -1], K, 1), "sigmoid": ([1, 0, K, 0, K, 0], K, K),
                      "both": ([2, 0, K, 0, 1, -1, K, K + 5, 1, 6, 0], K + 5, 6)}.get(
                          kind, ([1, 0, M * (1 + 2 * D), 0, D, M], M * (1 + 2 * D), D))
    x = rng.standard_normal((N, Lp)).astype(np.float32)
    tgt = rng.standard_normal((N, Lt)).astype(np.float32)
    if kind in ("softmax", "both"):
        tgt[:, 0] = rng.integers(0, K, size=N)
    layer = capi.Mdn(Lp, Lt, S, T, config)
    pd, xd, td = PC.dev(pat), PC.dev(x.reshape(-1)), PC.dev(tgt.reshape(-1))
    layer.load_sequences(pd, T)
    layer.forward(xd)
    results = torch.zeros(12, device="cuda")
    errors = torch.zeros(N * Lp, device="cuda")
    for i in range(12):
        if i % 4 == 3:
            layer.error_backward(td, results[i:i + 1], errors)
        else:
            layer.calculate_error(td, results[i:i + 1])
    torch.cuda.synchronize()
    got = results.cpu().numpy()
    want, bound = 0.0, 0.0
    if kind in ("softmax", "both"):
        p = layer.unit_buffer(0, 0).cpu().numpy().reshape(N, K)[np.arange(N), tgt[:, 0].astype(np.int64)].astype(np.float64)
        want += -np.log(p[valid]).sum()
        bound += want * 2.0 ** -22
    if kind in ("sigmoid", "both"):
        k = Lt - (kind == "both")
        p = layer.unit_buffer(int(kind == "both"), 0).cpu().numpy().reshape(N, k)
        b = np.where(tgt[:, Lt - k:] > 0, p, np.float32(1) - p).astype(np.float64)
        mean = -np.log(b[valid]).sum() / valid.sum()
        want += mean
        bound += mean * 2.0 ** -22
    if M:
        want = -layer.unit_buffer(0, 1).cpu().numpy()[N * M:][valid].astype(np.float64).sum()
    layer.close()
    assert len(set(got.tobytes()[4 * i:4 * i + 4] for i in range(12))) == 1, got
    assert abs(float(got[0]) - want) <= bound + abs(want) * 2.0 ** -24
