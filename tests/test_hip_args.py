"""The binding's argument handling: what it takes as a device pointer or an
activation type, and what it refuses."""
import numpy as np
import pytest

from cima_amd import gguf, hip

torch = pytest.importorskip("torch")


def test_ptr_takes_pointers_and_refuses_host_data():
    assert hip._ptr(None) is None and hip._ptr(0) is None and hip._ptr(4096) == 4096
    with pytest.raises(hip.EngineError):
        hip._ptr(torch.zeros(4))
    for bad in (np.zeros(4), "x", 1.5):
        with pytest.raises(TypeError):
            hip._ptr(bad)


def test_act_of_takes_f32_and_f16_only():
    assert hip._act_of(torch.zeros(1)) == gguf.DT_F32
    assert hip._act_of(torch.zeros(1, dtype=torch.float16)) == gguf.DT_F16
    for t in (torch.bfloat16, torch.float64, torch.int32):
        with pytest.raises(hip.EngineError):
            hip._act_of(torch.zeros(1, dtype=t))
