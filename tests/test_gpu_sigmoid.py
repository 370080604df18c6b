"""The device sigmoid (hardware reciprocal with one residual correction) against
the oracle's (IEEE division) on patterns from the whole range of binary32: every
257th bit pattern's neighbourhood, all exponents, both signs, specials."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_sigmoid_equals_oracle_over_the_range(et, orc, dev):
    bits = np.concatenate([np.arange(0, 1 << 32, 1021, dtype=np.uint64),
                           np.arange(0x3e000000, 0x42b00000, 97, dtype=np.uint64),          # |l| in [1/8, 88]
                           np.arange(0xbe000000, 0xc2b00000, 97, dtype=np.uint64),
                           np.arange(0x42adff00, 0x42ae0100, dtype=np.uint64),               # around 87
                           np.arange(0xc2adff00, 0xc2ae0100, dtype=np.uint64)]).astype(np.uint32)
    l = bits.view(np.float32)
    l = l[~np.isnan(l)]                                # a NaN score is routed by the fallback
    print(f"sigmoid: {l.size} inputs", flush=True)
    plan = et.route(torch.from_numpy(l.reshape(-1, 1)).to(dev), torch.full((1,), -1.0, device=dev))
    want = orc.sigmoid(l)
    assert plan.num_slots == l.size
    assert np.array_equal(plan.slot_gate.cpu().numpy().view(np.uint32), want.view(np.uint32))
