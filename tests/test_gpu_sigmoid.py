"""The device sigmoid (hardware reciprocal with one residual correction): all 2^32
binary32 inputs against the form that divides by the operator, on the GPU
(tests/gpu_checks/sigmoid_check.hip); and, through a routing call, against the
oracle's (IEEE division on the host) on a sample of 5.8 million patterns: every
1021st of the whole range, every 97th with |l| in [1/8, 88] and all around 87."""
import ctypes
import os

import numpy as np
import pytest
import torch

from conftest import ROOT

HELPER = os.path.join(ROOT, "tests", "gpu_checks", "libsigmoidcheck.so")


def _helper():
    # (torch is imported, so the helper binds to its HIP runtime)
    if not os.path.exists(HELPER):
        raise RuntimeError(f"{HELPER} is not built; run __graft_entry__.build()")
    L = ctypes.CDLL(HELPER)
    L.sigmoid_check.restype = ctypes.c_int
    L.sigmoid_check.argtypes = [ctypes.POINTER(ctypes.c_ulonglong), ctypes.POINTER(ctypes.c_uint)]
    return L


def test_helper_is_built_and_exports_the_check():
    assert hasattr(_helper(), "sigmoid_check")


@pytest.mark.gpu
def test_sigmoid_equals_the_dividing_form_on_all_inputs(dev):
    torch.cuda.synchronize()
    print("sigmoid: all 2^32 inputs", flush=True)
    mis, first = ctypes.c_ulonglong(7), ctypes.c_uint(0)
    assert _helper().sigmoid_check(ctypes.byref(mis), ctypes.byref(first)) == 0
    assert mis.value == 0, f"{mis.value} inputs differ, first {first.value:#010x}"
    assert first.value == 0xFFFFFFFF


@pytest.mark.gpu
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
