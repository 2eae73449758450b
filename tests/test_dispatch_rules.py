"""Which calls the kernels' dispatch lets through, without a GPU."""
import types

import pytest
import torch

from jax_llm_examples_amd.ops.hip import HipOps


def tensor(rows, cols, device="cuda:0", dtype=torch.float32):
    """What the rule looks at of a matrix on a GPU."""
    return types.SimpleNamespace(dtype=dtype, shape=(rows, cols), dim=lambda: 2, is_cuda=device.startswith("cuda"),
                                 device=torch.device(device), is_contiguous=lambda: True, data_ptr=lambda: 4096)


def rule(h, w, act=-1):
    ops = types.SimpleNamespace(gemm_f32_rows=lambda *a: "rows", gemm_f32_split=lambda *a: "split", _compute_units=256, _device_index=0,
                                split_ranges=HipOps.split_ranges)
    return HipOps._dense_float32(ops, h, w, act)


def test_dense_float32_products_by_size():
    assert rule(tensor(1, 64), tensor(32, 64)) == "rows"
    assert rule(tensor(512, 4096), tensor(4096, 4096)) == "split"
    assert rule(tensor(512, 4096, dtype=torch.bfloat16), tensor(4096, 4096)) is None
    assert rule(tensor(1, 64), tensor(32, 60)) is None  # (the library's product refuses it)


@pytest.mark.parametrize("rows", [1, 512])
@pytest.mark.parametrize("a, b", [("cuda:0", "cuda:1"), ("cuda:1", "cuda:0"), ("cuda:0", "cpu"), ("cpu", "cuda:0"),
                                  ("cuda:1", "cuda:1")])
def test_matrices_elsewhere_are_left_to_the_library(rows, a, b):
    assert rule(tensor(rows, 4096, a), tensor(4096, 4096, b)) is None


def test_leave_for_shared_memory_is_asked_for_on_the_device_of_the_launch():
    """What a kernel may use of a compute unit's shared memory is an attribute of a device: a process with two must not
    remember the first one's.  (One place asks for it, and no launcher keeps an answer.)"""
    import glob
    import os
    from jax_llm_examples_amd.ops import build
    asks = []
    for path in glob.glob(os.path.join(build.CSRC, "*.h*")):
        with open(path) as f:
            for line in f:
                if "hipFuncSetAttribute" in line:
                    asks.append(os.path.basename(path))
                kept = line.strip().startswith("static ") and ("allowed" in line or "hipError_t" in line)
                assert not kept, (path, line)
    assert asks == ["common.h"]
