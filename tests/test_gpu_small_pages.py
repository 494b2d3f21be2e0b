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

# the asymmetric format also takes head_dims that are no power of two
ASYM_GEOMS = [(1, 96, 5), (2, 96, 3), (3, 96, 2)]
# pages enough for the block save's wave per page (4096 in the three layers) and
# for the per-tensor and per-channel formats' maxima over several pages at a time
MANY_GEOMS = [(1, 32, 701), (3, 64, 690), (2, 128, 690)]


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
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_small_pages_match_oracle(fmt, dtype):
    from korith_vllm_ext import _paged

    for H, D, n in GEOMS + (ASYM_GEOMS if fmt == "int4_asym_g32" else
                            MANY_GEOMS if fmt != "fp8_e4m3_ph" else []):
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
        # one block id out of the pool: skipped, and flagged
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


@pytest.mark.parametrize("fmt", ["fp8_e4m3", "fp8_e4m3_ph", "int4_sym", "int4_sym_block",
                                 "int4_asym_g32"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_small_page_save_skips_a_bad_id(fmt, dtype):
    """A source block id out of the pool is flagged, leaves its page's codes and
    params as they were, and the pages that share its workgroup get the bytes
    they get without it (a page of zeros in its place: no scale changes)."""
    from korith_vllm_ext import _paged

    for H, D, n in GEOMS + MANY_GEOMS[:2]:
        g = torch.Generator().manual_seed(H * 1000 + D + n)
        L, pool = 3, n + 4
        x = torch.randn(L, 2, pool, 16, H, D, generator=g).to(dtype)
        src = torch.randperm(pool, generator=g)[:n].to(torch.int32)
        bad = n // 2
        x[:, :, int(src[bad])] = 0
        cache = _paged.cache_view(list(x.to(DEV)))
        lay = _paged.BlobLayout(fmt, 2, n, 16, H, D)
        wrong = src.clone()
        wrong[bad] = pool
        blobs = [torch.full((L, (lay.total_bytes + 15) // 16 * 16), 0xA5, dtype=torch.uint8,
                            device=DEV) for _ in range(2)]
        err = torch.zeros(1, dtype=torch.int32, device=DEV)
        for ids, b in ((src, blobs[0]), (wrong, blobs[1])):
            _paged.quant_gather(lay, cache, ids, [b[l].data_ptr() for l in range(L)], 2,
                                err_flag=err)
            assert int(err) == (0 if ids is src else 1)
        want, got = blobs
        code = lay.code_bytes_per_page
        for p in range(2):
            at = lay.code_offset(p) + bad * code
            want[:, at:at + code] = 0xA5
            if not lay.shared_params:
                each = lay.plane_param_bytes // n
                at = lay.param_offset(p) + bad * each
                want[:, at:at + each] = 0xA5
        assert torch.equal(got, want), (fmt, dtype, H, D, n)
