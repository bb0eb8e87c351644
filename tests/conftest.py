import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "rapid-h3_amd")):
    if p not in sys.path:
        sys.path.insert(0, p)

GOLDEN = os.path.join(ROOT, "tests", "golden")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP kernels through librh3)")


@pytest.fixture(scope="session")
def dev():
    """cuda:0 for GPU tests. Skips only when no GPU is visible; with a GPU, a missing librh3 fails."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU visible")
    from rapid_h3 import _native
    _native.lib()
    return torch.device("cuda:0")


@pytest.fixture(scope="session")
def golden():
    def load(name):
        with np.load(os.path.join(GOLDEN, name + ".npz"), allow_pickle=False) as f:
            return {k: f[k] for k in f.files}
    return load


def to_dev(a, device, dtype=None):
    """numpy (bf16 bits as uint16, e4m3 bits as uint8 when dtype says so) -> device tensor."""
    import torch
    a = np.ascontiguousarray(a)
    if a.dtype == np.uint16:
        return torch.from_numpy(a.view(np.int16)).to(device).view(torch.bfloat16)
    if dtype == "fp8":
        return torch.from_numpy(a).to(device).view(torch.float8_e4m3fn)
    return torch.from_numpy(a).to(device)


def to_np(t):
    """device tensor -> numpy (bf16 as uint16 bits, fp8 as uint8 bits)."""
    import torch
    t = t.detach().cpu()
    if t.dtype == torch.bfloat16:
        return t.view(torch.int16).numpy().view(np.uint16)
    if t.dtype == torch.float8_e4m3fn:
        return t.view(torch.uint8).numpy()
    return t.numpy()


def attention_plan(sq, sk, h, raw=False, tail=True, cus=0, q=None, out=None):
    """How the per-block attention runs a call (rh3_attention_plan): queries per workgroup, 1 where the main kernel
    quantizes the queries, workgroups run as two key halves, 1 where the pre-pass is two launches. raw: the one call
    without RMSNorm + RoPE, its out clear of q; or q and out as (address, token stride, head stride). cus 0: the
    device's."""
    import ctypes
    from rapid_h3 import _native as nat
    p = (ctypes.c_int64 * 4)()
    if raw:
        q, out = (1 << 40, h * 128, 128), (1 << 50, h * 128, 128)
    nat.call("rh3_attention_plan", *(q or (None, 0, 0)), *(out or (None, 0, 0)), sq, sk, h, int(tail), cus, p)
    return tuple(p)


def gemm_plan(m, n, k, cus=0):
    """How a GEMM runs a call (rh3_gemm_plan): tile rows and columns, rows before them on 256 x 256 tiles, the form of
    those (GEMM_*)."""
    import ctypes
    from rapid_h3 import _native as nat
    p = (ctypes.c_int64 * 4)()
    nat.call("rh3_gemm_plan", m, n, k, cus, p)
    return tuple(p)


GEMM_SMALL, GEMM_SINGLE, GEMM_SHARES, GEMM_COUNTED = range(4)   # no 256 x 256 tiles; a workgroup each; per CU: shares, counters


def on_256_cus():
    """The forms that the tests' shapes are chosen for are those of 256 CUs."""
    import torch
    return torch.cuda.get_device_properties(0).multi_processor_count == 256
