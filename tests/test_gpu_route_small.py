"""Routing and the EMA update of small batches (one block) against the oracle,
at the sizes where the kernel is taken and left, with ties, NaN and infinite
logits, thresholds outside (0, 1], and undersized capacities."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

INDEX = ("counts", "expert_offsets", "token_offsets", "sorted_token", "token_slot")


def _batch(T, E, seed):
    rng = np.random.default_rng([T, E, seed])
    lg = rng.standard_normal((T, E)).astype(np.float32)
    if T > 4:
        lg[rng.integers(0, T, 1 + T // 9), rng.integers(0, E, 1 + T // 9)] = np.nan
        lg[rng.integers(0, T, 2), rng.integers(0, E, 2)] = [np.inf, -np.inf]
        lg[T // 2] = lg[T // 2 - 1]                       # equal tokens
        lg[T // 3] = np.nan                               # a token without any score
        lg[T // 4] = -3.0                                 # ties in the fallback
    thr = rng.uniform(0.4, 0.9, E).astype(np.float32)
    if E > 3:
        thr[:4] = [0.0, 1.5, np.nan, 0.9999999]
    return lg, thr


@pytest.mark.parametrize("T,E", [(1, 1), (1, 256), (15, 8), (17, 64), (16, 65), (63, 256), (64, 256), (127, 129),
                                 (128, 127), (128, 128), (252, 65), (253, 65), (256, 63), (256, 64), (255, 8),
                                 (256, 1), (257, 8), (64, 300), (32, 128), (33, 128), (64, 112), (64, 113), (65, 112),
                                 (128, 96), (128, 97), (129, 80), (129, 81)])
def test_small_routing_and_update_equal_the_oracle(et, orc, dev, T, E):
    print(f"small route T={T} E={E}", flush=True)
    for seed in (0, 1):
        lg, thr = _batch(T, E, seed)
        want = orc.route(lg, thr)
        L = torch.from_numpy(lg).to(dev)
        S = want.num_slots
        for cap in (None, S + 5, max(1, S - 3), 0):
            plan = et.route(L, torch.from_numpy(thr).to(dev), slot_capacity=cap)
            for f in INDEX + ("slot_gate",):
                a, b = getattr(plan, f).cpu().numpy(), getattr(want, f)
                n = len(b) if f in INDEX[:3] else min(S, len(a))
                assert np.array_equal(a[:n].view(np.uint32), b[:n].view(np.uint32)), (f, cap)
        for k in sorted({1, min(3, E), E}):
            th = torch.from_numpy(thr).to(dev)
            stat = torch.empty(E, device=dev)
            plan = et.route_update(L, th, k, 0.9, stat=stat)
            new, st = orc.threshold_update(lg, thr, k, 0.9)
            assert np.array_equal(th.cpu().numpy().view(np.uint32), new.view(np.uint32)), k
            assert np.array_equal(stat.cpu().numpy().view(np.uint32), st.view(np.uint32)), k
            assert np.array_equal(plan.token_slot.cpu().numpy(), want.token_slot[:S])
            assert np.array_equal(plan.sorted_token.cpu().numpy(), want.sorted_token[:S])
