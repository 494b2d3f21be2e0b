"""The single-read (cooperative) per-tensor FP8 save at scale groups past its
32 MiB minimum: an odd group count (the last group has no partner buffer) of
two pages per workgroup, and several small pages per workgroup."""

from __future__ import annotations

import pytest
import torch

import test_gpu_kernels as kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,geom", [
    pytest.param(torch.bfloat16, dict(L=3, pool=530, n=513, bs=16, H=8, D=128), id="bf16-3groups"),
    pytest.param(torch.float16, dict(L=1, pool=4200, n=4100, bs=16, H=2, D=64), id="fp16-cpt1"),
])
def test_single_read_large_groups(dtype, geom):
    kernels._assert_single_read(geom)
    kernels.test_fp8_tensor_single_read_bitexact(dtype, geom)
