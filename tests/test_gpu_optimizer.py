"""GPU parity tests (through the C ABI) for the weight update kernels against the CPU oracle.
Every operation is a separately rounded fp32 / fp64 operation in both, so the bar is bit-exact; the one
tolerance is 1 ulp on the quotients that involve a square root (written below)."""
import numpy as np
import pytest

import oracle_lib as O
import parity_cases as PC

pytestmark = pytest.mark.gpu


def _setup(n, seed, with_mask):
    rng = np.random.default_rng(seed)
    w = rng.standard_normal(n).astype(np.float32)
    grads = [(rng.standard_normal(n) * 2).astype(np.float32) for _ in range(4)]
    grads[1][5 % n] = np.nan
    grads[2][7 % n] = np.inf
    mask = None
    if with_mask:
        mask = np.ones(n, np.float32)
        mask[::5] = 0.0
    return w, grads, mask


def _ulp_close(a, b, ulps):
    a = np.asarray(a, np.float32); b = np.asarray(b, np.float32)
    ia = a.view(np.int32).astype(np.int64); ib = b.view(np.int32).astype(np.int64)
    return bool(np.all((np.abs(ia - ib) <= ulps) | (a == b)))


@pytest.mark.parametrize("option,momentum,with_mask,n", [
    (0, 0.9, False, 100003), (0, 0.0, True, 777), (2, 0.5, False, 4096), (1, 0.0, False, 100003),
    (1, 0.9, True, 5000), (3, 0.3, False, 1234), (5, 0.0, False, 100003), (5, 0.9, True, 6001), (4, 0.9, False, 64),
    (5, 0.0, False, 1),
])
def test_three_calls_and_fused_step_match_oracle(option, momentum, with_mask, n):
    import torch

    print("optimizer case", option, momentum, with_mask, n, flush=True)
    capi = PC.pkg().capi
    w0, grads, mask = _setup(n, 11 + option, with_mask)
    nstat = 2 * n if option == 5 else n
    init = 0.0 if option == 5 else 1e-6
    lr, frac = 3e-3, 41.0
    # oracle
    w = w0.copy(); deltas = np.zeros(n, np.float32); stats = np.full(nstat, init, np.float32)
    cur = np.zeros(n, np.float32)
    b1 = b2 = 1.0
    # device, three calls and fused
    dev = lambda a: torch.from_numpy(a.copy()).cuda()
    dmask = dev(mask) if mask is not None else None
    A = {"w": dev(w0), "deltas": torch.zeros(n, device="cuda"), "stats": torch.full((nstat,), init, device="cuda"),
         "cur": torch.zeros(n, device="cuda")}
    B = {k: v.clone() for k, v in A.items()}
    for i, g in enumerate(grads):
        add = (i == 3)  # exercise the accumulating form once
        b1 = O.opt_next_beta_accum(b1, 1); b2 = O.opt_next_beta_accum(b2, 2)
        assert capi.opt_next_beta_accum(b1 / np.float32(1), 1) == O.opt_next_beta_accum(b1, 1)
        O.opt_accumulate(g, cur, add)
        O.opt_adjust_gradient(option, cur, stats, mask, frac, b1, b2)
        O.opt_update_weights(w, cur, deltas, mask, lr, momentum)
        dg = dev(g)
        capi.opt_accumulate(dg, A["cur"], add)
        capi.opt_adjust_gradient(option, A["cur"], A["stats"], dmask, frac, b1, b2)
        capi.opt_update_weights(A["w"], A["cur"], A["deltas"], dmask, lr, momentum)
        if not add:
            capi.opt_step(option, B["w"], dg, B["cur"], B["stats"], B["deltas"], dmask, frac, b1, b2, lr, momentum)
        else:
            capi.opt_accumulate(dg, B["cur"], True)
            capi.opt_adjust_gradient(option, B["cur"], B["stats"], dmask, frac, b1, b2)
            capi.opt_update_weights(B["w"], B["cur"], B["deltas"], dmask, lr, momentum)
    torch.cuda.synchronize()
    for name, ref in (("w", w), ("deltas", deltas), ("stats", stats), ("cur", cur)):
        got_a, got_b = A[name].cpu().numpy(), B[name].cpu().numpy()
        assert np.array_equal(got_a, got_b), name  # fused == three calls, bit for bit
        # sqrt-quotients may differ in the last place between host and device libraries: 2 ulp; all else exact
        ulps = 2 if option in (1, 5) else 0
        ok = _ulp_close(got_a, ref, ulps) or np.allclose(got_a, ref, rtol=3e-7, atol=1e-9)
        if not ok:
            bad = np.flatnonzero(got_a != ref)
            print(name, "mismatches", bad.size, "first", bad[:5], got_a[bad[:5]], ref[bad[:5]],
                  "max abs", np.nanmax(np.abs(got_a - ref)), flush=True)
        assert ok, name
    assert not np.any(np.isnan(A["w"].cpu().numpy()))


def test_negative_learning_rate_skips_update_and_bad_arguments():
    import torch

    capi = PC.pkg().capi
    w = torch.ones(16, device="cuda"); g = torch.ones(16, device="cuda"); d = torch.zeros(16, device="cuda")
    capi.opt_update_weights(w, g, d, None, -1.0, 0.9)
    torch.cuda.synchronize()
    assert torch.all(w == 1) and torch.all(d == 0)
    with pytest.raises(RuntimeError):
        capi.opt_adjust_gradient(5, g, None, None, 1.0, 0.9, 0.999)   # Adam without a statistics buffer
    with pytest.raises(RuntimeError):
        capi.opt_adjust_gradient(9, g, d, None, 1.0)


@pytest.mark.parametrize("option,with_mask,add", [(0, False, False), (1, True, True), (2, False, True), (3, True, False), (5, True, False), (5, False, True)])
@pytest.mark.parametrize("n", [1, 5, 1023, 2 ** 21 - 2, 2 ** 21 + 1, 2 ** 21 + 4, 2 ** 21 + 1027])
def test_a_weight_is_updated_the_same_wherever_it_stands(option, with_mask, add, n):
    # A few weights go one per thread, more than 2^21 in fours and the last ones by themselves: every array begins at another place behind
    # an aligned address, and the result is bit for bit that of the same weights, a part at a time, one by one; nothing beside an array changes.
    import torch

    capi = PC.pkg().capi
    rng = np.random.default_rng(n)
    per = {"w": 1, "g": 1, "cur": 1, "stats": 2 if option == 5 else 1, "deltas": 1, "mask": 1}
    host = {k: np.abs(rng.standard_normal(n * p)).astype(np.float32) for k, p in per.items()}
    host["mask"] = np.where(rng.random(n) < 0.3, 0.0, 1.0).astype(np.float32)
    host["g"][n // 2] = np.nan
    results = []
    for shifted in (False, True):
        whole = {}
        view = {}
        for at, (k, p) in enumerate(per.items()):
            skip = 1 + at % 3 if shifted else 0
            whole[k] = torch.full((skip + n * p + 8,), 7.0, device="cuda")
            whole[k][skip:skip + n * p] = torch.from_numpy(host[k]).cuda()
            view[k] = whole[k][skip:skip + n * p]
        for part in range(1 if shifted else 3):
            cut = n if shifted else (n + 2) // 3
            sub = {k: v[part * cut * per[k]:(part + 1) * cut * per[k]] for k, v in view.items()}
            if sub["w"].numel() == 0: continue
            args = (option, sub["cur"], sub["stats"], sub["mask"] if with_mask else None, 41.0, 0.9, 0.999)
            if add:  # the three calls, the first of them accumulating; else the one that does all
                capi.opt_accumulate(sub["g"], sub["cur"], True)
                capi.opt_adjust_gradient(*args)
                capi.opt_update_weights(sub["w"], sub["cur"], sub["deltas"], args[3], 3e-3, 0.9)
            else:
                capi.opt_step(option, sub["w"], sub["g"], sub["cur"], sub["stats"], sub["deltas"], args[3], 41.0, 0.9, 0.999, 3e-3, 0.9)
        torch.cuda.synchronize()
        if shifted:
            for k, p in per.items():
                skip = whole[k].numel() - n * p - 8
                assert torch.all(whole[k][:skip] == 7.0) and torch.all(whole[k][skip + n * p:] == 7.0), k
        results.append({k: view[k][:n * p].cpu().numpy().view(np.int32) for k, p in per.items()})
    for k in per:
        assert np.array_equal(results[0][k], results[1][k]), k
