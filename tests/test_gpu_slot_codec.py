"""Codec launches over token slots (amf_int4_quant_gather_slots and the
*_dequant_scatter_slots forms): the bytes and rows of gathering first and
scattering last, at the edges of pages and of the kernels' page sizes."""

from __future__ import annotations

import pytest
import torch

from helpers import bits

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _case(L, H, D, bs, T, dtype, seed, pad=0):
    """Cache layers [2, nb, bs, H, D] (pages `pad` rows apart), unordered slots
    and the gathered rows [L, 2, T, H, D]."""
    g = torch.Generator().manual_seed(seed)
    nb = -(-T // bs) + 3
    store = torch.randn(L, 2, nb, bs + pad, H, D, generator=g).to(dtype).to(DEV)
    store[..., 1] *= 20
    cache = [store[l][:, :, :bs] for l in range(L)]
    slots = torch.randperm(nb * bs, generator=g)[:T]
    rows = torch.stack([c.reshape(2, nb * bs, H, D)[:, slots.to(DEV)] for c in cache])
    return cache, slots, rows


# (heads, dim, tokens): pages of 256, 257..., up to 16384 chunks of 8 elements
# (the register kernel's launches and its largest page), past it, and ragged
# last pages
@pytest.mark.parametrize("H,D,T,dtype", [
    (1, 64, 31, torch.bfloat16), (1, 64, 129, torch.float16), (3, 128, 128, torch.bfloat16),
    (2, 64, 257, torch.bfloat16), (3, 64, 300, torch.float16), (5, 128, 130, torch.bfloat16),
    (8, 128, 400, torch.bfloat16), (8, 128, 256, torch.float16), (9, 128, 200, torch.bfloat16),
    (2, 128, 200, torch.float32),
])
def test_block_save_from_slots(H, D, T, dtype):
    from korith_vllm_ext.compressed_vram_pool import CompressedVRAMPool

    cache, slots, rows = _case(2, H, D, 16, T, dtype, H * 100 + T, pad=H % 2)
    pool = CompressedVRAMPool(2, 16 << 20, default_format="int4_sym_block")
    assert pool.put_from_slots("a", cache, slots) and pool.put_from_raw("b", rows)
    a, b = pool.get("a"), pool.get("b")
    assert a.layout == b.layout and a.num_tokens == b.num_tokens == T
    for x, y in zip(a.blobs, b.blobs):
        n = x.meta["_layout"].data_bytes  # every code, those of the padding too
        assert torch.equal(x.meta["_blob"][:n], y.meta["_blob"][:n])
        assert torch.equal(x.scales, y.scales)


@pytest.mark.parametrize("fmt", ["fp8_e4m3", "fp8_e4m3_ph", "int4_sym", "int4_sym_block"])
@pytest.mark.parametrize("H,D,T,n,dtype", [
    (2, 64, 96, 96, torch.bfloat16), (8, 128, 259, 200, torch.float16),
    (1, 128, 33, 17, torch.bfloat16), (3, 64, 130, 130, torch.float32),
    (8, 128, 1, 1, torch.bfloat16),
])
def test_restore_to_slots(fmt, H, D, T, n, dtype):
    from korith_vllm_ext.compressed_vram_pool import CompressedVRAMPool

    _, _, rows = _case(2, H, D, 16, T, dtype, T + n)
    cache, slots, _ = _case(2, H, D, 8, T, dtype, T, pad=1)
    pool = CompressedVRAMPool(2, 16 << 20, default_format=fmt)
    assert pool.put_from_raw("x", rows)
    dense = pool.restore_to_tensor("x", dtype)
    before = [c.clone() for c in cache]
    assert pool.restore_to_slots("x", cache, slots[:n]) == T
    for l in range(2):
        want = before[l]
        flat = want.reshape(2, -1, H, D).clone()
        flat[:, slots[:n].to(DEV)] = dense[l][:, :n]
        got = cache[l].reshape(2, -1, H, D)
        assert (bits(got) == bits(flat)).all() if dtype != torch.float32 else torch.equal(got, flat)


def test_slots_outside_the_pool_are_skipped():
    """The kernels' own check: rows outside are neither read nor written, and
    flagged; a save takes them as zeros."""
    import amf_hip

    H, D, bs, T, nb = 2, 64, 16, 40, 6
    cache = torch.randn(1, 2, nb, bs, H, D, device=DEV).to(torch.bfloat16)
    slots = torch.randperm(nb * bs)[:T]
    bad = slots.clone()
    bad[[3, 39]] = torch.tensor([-1, nb * bs])
    tab = torch.tensor([cache[0, p].data_ptr() for p in range(2)]).to(DEV)
    codes = torch.zeros(2, T * H * D // 2, dtype=torch.uint8, device=DEV)
    params = torch.zeros(2, 16, dtype=torch.uint8, device=DEV)
    ctab = torch.tensor([codes[p].data_ptr() for p in range(2)]).to(DEV)
    ptab = torch.tensor([params[p].data_ptr() for p in range(2)]).to(DEV)
    err = torch.zeros(1, dtype=torch.int32, device=DEV)
    ds = bad.to(DEV)
    args = (bs * H * D * 2, bs, amf_hip.DTYPE_BF16, ds.data_ptr(), nb * bs)
    amf_hip.call("amf_int4_quant_gather_slots", amf_hip.FMT_INT4_SYM_BLOCK, tab.data_ptr(), *args,
                 ctab.data_ptr(), ptab.data_ptr(), 2, T, T, H, D, err.data_ptr(),
                 amf_hip.stream_handle(DEV))
    assert int(err) == 1
    assert (codes.view(2, T, -1)[:, [3, 39]] == 0x88).all()
    out = torch.zeros_like(cache)
    otab = torch.tensor([out[0, p].data_ptr() for p in range(2)]).to(DEV)
    err.zero_()
    amf_hip.call("amf_int4_dequant_scatter_slots", amf_hip.FMT_INT4_SYM_BLOCK, ctab.data_ptr(),
                 ptab.data_ptr(), otab.data_ptr(), *args, 2, T, T, H, D, err.data_ptr(),
                 amf_hip.stream_handle(DEV))
    assert int(err) == 1
    good = torch.ones(T, dtype=torch.bool)
    good[[3, 39]] = False
    rows = out.view(2, nb * bs, H, D)
    written = rows.abs().sum((0, 2, 3)) != 0
    assert set(written.nonzero().flatten().tolist()) <= set(slots[good].tolist())
    src = cache.view(2, nb * bs, H, D)[:, slots[good].to(DEV)].float()
    s = params.view(torch.float16)[:, :1].float().view(2, 1, 1, 1)
    got = rows[:, slots[good].to(DEV)].float()
    assert float(((got - src).abs() / s).max()) <= 0.52  # half a step, and bf16 rounding
