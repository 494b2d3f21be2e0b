"""Paged INT4 decode at part counts on both sides of the merge's steps: pairs
of one part, up to and past the parts that one wave loads at once, past the
four-wave merge's first load and its first 64 (m, l) words, with empty and
one-token sequences beside long ones."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import attention as oatt
from oracle import codecs as oc
from oracle import gen

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


@pytest.mark.parametrize("Hkv,R,ctx", [
    (1, 8, [8100]),                  # hundreds of parts: past 64 parts a wave pass
    (1, 1, [2049]),                  # 65 parts
    (2, 4, [1000, 0, 1, 40]),        # 32 parts, none, one token, two
    (8, 2, [530, 32, 33]),           # 17 parts
    (8, 4, [500] * 12 + [90] * 20),  # few parts each: one wave per row
    (1, 4, [20000] + [17] * 3),      # one long sequence among short ones
])
def test_merge_part_counts(Hkv, R, ctx):
    from korith_vllm_ext.codecs import get_codec
    from korith_vllm_ext.int4_decode_attention import int4_decode_attention

    print(f"decode merge case Hkv={Hkv} R={R} ctx={ctx[:4]}", flush=True)
    g = torch.Generator().manual_seed(Hkv * 100 + R + len(ctx))
    S, D = len(ctx), 128
    pages = [(c + 15) // 16 for c in ctx]
    q = torch.randn(S, Hkv * R, D, generator=g).to(torch.bfloat16)
    kv = gen.kv_values((2, sum(pages) + 1, 16, Hkv, D), D, g, True)
    perm = torch.randperm(sum(pages), generator=g).to(torch.int32)
    bt = torch.zeros(S, max(pages), dtype=torch.int32)
    at = 0
    for s, n in enumerate(pages):
        bt[s, :n] = perm[at:at + n]
        at += n
    cl = torch.tensor(ctx, dtype=torch.int32)
    pool = get_codec("int4_asym_g32").compress(kv.to(DEV))
    out = int4_decode_attention(q.to(DEV), pool, block_tables=bt.to(DEV),
                                context_lens=cl.to(DEV), out_dtype=torch.float32).cpu().numpy()
    kv32 = oc.int4_asym_dequant_f32(*oc.int4_asym_quantize(kv))
    ref = oatt.paged_decode_f64(q.float().numpy(), kv32[0].numpy(), kv32[1].numpy(), bt.numpy(),
                                cl.numpy())
    # the decode's stated bounds: fp16 PV weights within 0.015 of the output
    assert np.abs(out - ref).max() <= 2e-2
    assert np.abs(out - ref).sum() / max(np.abs(ref).sum(), 1e-30) <= 1e-2


@pytest.mark.parametrize("Hkv,R,ctx", [
    (1, 4, [2000]),         # 63 parts, four waves a row
    (8, 4, [500] * 32),     # 12 parts or fewer, one wave a row
])
def test_infinite_last_part(Hkv, R, ctx):
    """A V group whose zero point is -inf in fp16, in the last token's page,
    makes its 32 dims -inf and nothing NaN: the merge reads the last part again
    in the place of parts that do not exist."""
    from korith_vllm_ext.codecs import get_codec
    from korith_vllm_ext.int4_decode_attention import int4_decode_attention

    print(f"infinite part case Hkv={Hkv} R={R} ctx={ctx[:4]}", flush=True)
    g = torch.Generator().manual_seed(7)
    S, D = len(ctx), 128
    pages = [(c + 15) // 16 for c in ctx]
    q = torch.randn(S, Hkv * R, D, generator=g).to(torch.bfloat16)
    kv = gen.kv_values((2, sum(pages), 16, Hkv, D), D, g, True)
    kv *= 0.25  # no score far below another: every weight positive
    bt = torch.zeros(S, max(pages), dtype=torch.int32)
    at = 0
    for s, n in enumerate(pages):
        bt[s, :n] = torch.arange(at, at + n, dtype=torch.int32)
        at += n
        kv[1, at - 1, (ctx[s] - 1) % 16, :, 40] = -70000.0  # dims 32 .. 63
    cl = torch.tensor(ctx, dtype=torch.int32)
    pool = get_codec("int4_asym_g32").compress(kv.to(DEV))
    out = int4_decode_attention(q.to(DEV), pool, block_tables=bt.to(DEV),
                                context_lens=cl.to(DEV), out_dtype=torch.float32).cpu().numpy()
    kv32 = oc.int4_asym_dequant_f32(*oc.int4_asym_quantize(kv))
    ref = oatt.paged_decode_f64(q.float().numpy(), kv32[0].numpy(), kv32[1].numpy(), bt.numpy(),
                                cl.numpy())
    inf = np.isneginf(ref)
    assert inf[:, :, 32:64].all() and np.isfinite(ref[~inf]).all()
    assert np.isneginf(out[inf]).all()
    assert np.abs(out[~inf] - ref[~inf]).max() <= 2e-2
