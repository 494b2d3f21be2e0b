"""Save and restore of small pages (a few KV heads), which share workgroups:
every format at geometries on both sides of the kernels' page sizes, with page
counts that leave the last workgroup partly filled, against the oracle."""

from __future__ import annotations

import pytest
import torch

from helpers import bits
from oracle import codecs as oc

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")

GEOMS = [  # heads, head_dim, pages
    (1, 32, 5), (1, 64, 3), (1, 128, 9), (2, 64, 1), (2, 128, 7), (3, 64, 6), (4, 64, 5),
    (4, 128, 6), (5, 128, 2), (8, 128, 3), (16, 64, 2),
]


def _oracle(fmt, x, dtype):
    """The oracle's restored values of one layer's pages [2, n, 16, H, D]."""
    if fmt == "fp8_e4m3":
        return oc.fp8_tensor_decompress(*oc.fp8_tensor_compress(x), dtype)
    if fmt == "fp8_e4m3_ph":
        return oc.fp8_ph_decompress(*oc.fp8_ph_compress(x), dtype)
    if fmt == "int4_sym":
        return oc.int4_channel_decompress(*oc.int4_channel_compress(x), tuple(x.shape), dtype)
    if fmt == "int4_sym_block":
        codes, scales, meta = oc.int4_block_compress(x)
        return oc.int4_block_decompress(codes, scales, tuple(x.shape), meta, dtype)
    return oc.int4_asym_dequant_f32(*oc.int4_asym_quantize(x)).to(dtype)


@pytest.mark.parametrize("fmt", ["fp8_e4m3", "fp8_e4m3_ph", "int4_sym", "int4_sym_block",
                                 "int4_asym_g32"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_small_pages_match_oracle(fmt, dtype):
    from korith_vllm_ext import _paged

    for H, D, n in GEOMS:
        g = torch.Generator().manual_seed(H * 1000 + D + n)
        L, pool = 3, n + 4
        x = torch.randn(L, 2, pool, 16, H, D, generator=g)
        x[..., 3] *= 20
        x = x.to(dtype)
        src = torch.randperm(pool, generator=g)[:n].to(torch.int32)
        dst = torch.randperm(pool, generator=g)[:n].to(torch.int32)
        lay = _paged.BlobLayout(fmt, 2, n, 16, H, D)
        blobs = torch.zeros(L, (lay.total_bytes + 15) // 16 * 16, dtype=torch.uint8, device=DEV)
        bases = [blobs[l].data_ptr() for l in range(L)]
        cache, target = x.to(DEV), torch.full_like(x, -7.25, device=DEV)
        # one block id out of the pool: skipped on both ways, and flagged
        err = torch.zeros(1, dtype=torch.int32, device=DEV)
        _paged.quant_gather(lay, _paged.cache_view(list(cache)), src, bases, 2)
        bad = dst.clone()
        bad[n // 2] = pool
        _paged.dequant_scatter(lay, bases, 2, _paged.cache_view(list(target)), bad, err_flag=err)
        assert int(err) == 1
        want = torch.full_like(x, -7.25)
        for l in range(L):
            y = _oracle(fmt, x[l][:, src.long()].contiguous(), dtype)
            keep = [i for i in range(n) if i != n // 2]
            want[l][:, dst[keep].long()] = y.reshape(2, n, 16, H, D)[:, keep]
        assert (bits(target) == bits(want)).all(), (fmt, dtype, H, D, n)
