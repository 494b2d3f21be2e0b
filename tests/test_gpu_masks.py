"""Additive masks of the lowest and highest finite values (what padding is
usually masked with) on every dense attention kernel, against float64
attention: such a value never turns into an infinity, so a row masked with it
everywhere is the mean of its tokens and no NaN."""

from __future__ import annotations

import pytest
import torch

from test_gpu_prefill import _ref

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _mask(Tq, T, low):
    """One pattern per row, repeated: no mask, all low, the second half low,
    -inf over the first half and low over the rest, low but for one token,
    the highest value at one token."""
    m = torch.zeros(Tq, T)
    for i in range(Tq):
        k = i % 6
        if k == 1:
            m[i] = low
        elif k == 2:
            m[i, T // 2:] = low
        elif k == 3:
            m[i, :T // 2] = float("-inf")
            m[i, T // 2:] = low
        elif k == 4:
            m[i] = low
            m[i, T - 1] = 0.0
        elif k == 5:
            m[i, T // 3] = -low
    return m.to(DEV)


@pytest.mark.parametrize("kv,dtype,Hq,Hkv,Tq,T,D", [
    ("dense", torch.float32, 2, 1, 6, 70, 80),       # single pass
    ("dense", torch.bfloat16, 2, 2, 6, 300, 96),
    ("dense", torch.float32, 4, 1, 6, 1100, 128),    # one row per wave, split and merged
    ("int4_sym", torch.float32, 4, 2, 6, 500, 64),
    ("dense", torch.bfloat16, 4, 4, 3, 2000, 64),    # three rows: below the row tiles
    ("dense", torch.bfloat16, 8, 8, 6, 3000, 128),   # row tiles, one wave, many splits
    ("dense", torch.float16, 8, 2, 30, 200, 128),    # four waves, few splits
    ("int4_sym", torch.float16, 4, 2, 30, 333, 128),
    ("dense", torch.bfloat16, 2, 1, 18, 65, 256),
])
@pytest.mark.parametrize("low", [torch.finfo(torch.float32).min, torch.finfo(torch.bfloat16).min])
def test_lowest_finite_mask(kv, dtype, Hq, Hkv, Tq, T, D, low):
    from korith_vllm_ext.codecs import get_codec
    from korith_vllm_ext.kernels import dense_attention
    from korith_vllm_ext.kernels.dispatch import int4_sym_attention

    g = torch.Generator().manual_seed(T + D)
    q, k, v = (torch.randn(2, h, n, D, generator=g).to(dtype).to(DEV)
               for h, n in ((Hq, Tq), (Hkv, T), (Hkv, T)))
    mask = _mask(Tq, T, low)
    if kv == "dense":
        out = dense_attention(q, k, v, 0.2, mask, torch.float32)
    else:
        codec = get_codec("int4_sym")
        kc, vc = codec.compress(k), codec.compress(v)
        k, v = codec.decompress_to(kc, dtype), codec.decompress_to(vc, dtype)
        out = int4_sym_attention(q, kc, vc, 0.2, mask, torch.float32)
    # fp32 sums of D products and T weights, as in the tests of the row tiles
    assert float((out.double() - _ref(q, k, v, 0.2, mask)).abs().max()) <= 1e-4
