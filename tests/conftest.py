import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
for p in (ROOT, ROOT / "bonsai.cpp_amd"):
    if str(p) not in sys.path:
        sys.path.insert(0, str(p))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU")


@pytest.fixture(scope="session")
def oracle():
    from oracle import b1_oracle
    b1_oracle.lib()  # builds oracle/_build/libb1oracle.so if it is missing
    return b1_oracle


KINDS = {"plain": (0, 0), "gate_residual": (1, 0), "swiglu": (2, 0), "packed": (3, 0), "packed_gelu": (3, 1),
         "packed_swiglu": (3, 2)}


@pytest.fixture(scope="session")
def gemm_plan():
    """gemm_plan(m, k, n, epilogue="plain", split=0): the name of the kernel a
    packed GEMM of that shape runs on 256 CUs (no device needed)."""
    import ctypes

    import bonsai_b1
    lib = bonsai_b1.load()

    def plan(m, k, n, epilogue="plain", split=0):
        kind, act = KINDS[epilogue]
        name = ctypes.create_string_buffer(32)
        lib.b1_gemm_plan(m, k, n, 256, kind, act, split, name, ctypes.c_size_t(len(name)))
        return name.value.decode()

    return plan


@pytest.fixture(scope="session")
def fused_plan():
    """fused_plan(m, k, n): the tile of the GEMM that converts fp32 activations
    itself, on 256 CUs."""
    import ctypes

    import bonsai_b1
    lib = bonsai_b1.load()

    def plan(m, k, n):
        name = ctypes.create_string_buffer(32)
        lib.b1_fused_plan(m, k, n, 256, name, ctypes.c_size_t(len(name)))
        return name.value.decode()

    return plan


@pytest.fixture(scope="session")
def exact_plan():
    """exact_plan(m, n): the rows an EXACT work-group takes on 256 CUs."""
    import bonsai_b1
    lib = bonsai_b1.load()
    return lambda m, n: lib.b1_exact_plan(m, n, 256)


@pytest.fixture(scope="session")
def unpack():
    """unpack(raw, n, k): float64 [n, k] of packed B1_0 weights on the GPU."""
    import torch

    def weights(raw, n, k):
        blocks = raw.reshape(n, k // 32, 6)
        scale = blocks[:, :, :2].contiguous().view(torch.float16).double()
        bits = torch.arange(8, device=raw.device, dtype=torch.uint8)
        sign = 2.0 * ((blocks[:, :, 2:].unsqueeze(-1) >> bits) & 1).double() - 1.0
        return (sign.reshape(n, k // 32, 32) * scale).reshape(n, k)

    return weights
