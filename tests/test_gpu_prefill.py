"""Attention of many query rows (q_len > 1, bf16 / fp16) on the MFMA tiles of
amf_prefill.hip, against float64 attention, at the edges of its row tiles, its
token tiles and its splits."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _ref(q, k, v, scale, mask):
    """float64 attention on the GPU (contiguous operands), GQA by repetition."""
    r = q.shape[1] // k.shape[1]
    k, v = (t.double().repeat_interleave(r, 1).contiguous() for t in (k, v))
    s = torch.matmul(q.double(), k.transpose(-1, -2).contiguous()) * scale
    if mask is not None:
        s = s + mask.double()
    return torch.matmul(torch.softmax(s, -1), v)


def _mask(kind, B, Hq, Tq, T, g):
    if kind is None:
        return None
    if kind == "causal":
        m = torch.zeros(Tq, T)
        for i in range(Tq):
            m[i, max(0, T - Tq + i + 1):] = float("-inf")
        return m.to(DEV)
    if kind == "heads":  # one per (batch, head, row), with holes
        m = torch.randn(B, Hq, Tq, T, generator=g)
        m[torch.rand(m.shape, generator=g) < 0.3] = float("-inf")
        m[..., 0] = 0.5
        return m.to(DEV)
    # every other column of a wider tensor: a token stride of 2
    return torch.randn(Tq, 2 * T, generator=g).to(DEV)[:, ::2]


@pytest.mark.parametrize("dtype,B,Hq,Hkv,Tq,T,D,kind", [
    (torch.bfloat16, 1, 8, 2, 2, 33, 128, None),        # 8 rows, one token past a tile
    (torch.float16, 2, 8, 1, 4, 64, 64, "causal"),      # 32 rows: the one-wave workgroup, full
    (torch.bfloat16, 1, 11, 1, 3, 129, 128, "heads"),   # 33 rows: past it; odd group
    (torch.float16, 1, 4, 4, 129, 131, 128, "causal"),  # 129 rows: a second tile of one row
    (torch.bfloat16, 2, 14, 2, 37, 300, 64, "causal"),  # group of 7
    (torch.bfloat16, 1, 16, 2, 40, 1000, 256, "causal"),
    (torch.float16, 1, 4, 2, 16, 515, 256, "strided"),
    (torch.float16, 1, 8, 2, 7, 515, 256, "strided"),   # a group of 4: tiles at any size
    (torch.bfloat16, 1, 2, 2, 16, 2049, 256, "causal"),  # past the pairs that 256 dims take
    (torch.float16, 2, 2, 1, 70, 1000, 256, "causal"),
    (torch.bfloat16, 3, 8, 8, 9, 4099, 128, "causal"),  # 9 rows, many splits, ragged end
    (torch.bfloat16, 1, 32, 8, 64, 2048, 128, "strided"),
    (torch.float16, 1, 6, 3, 50, 1, 128, None),         # a single token
])
def test_many_rows_match_f64(dtype, B, Hq, Hkv, Tq, T, D, kind):
    from korith_vllm_ext.kernels import dense_attention

    print(f"many-row case {dtype} B={B} Hq={Hq}/{Hkv} Tq={Tq} T={T} D={D} {kind}", flush=True)
    g = torch.Generator().manual_seed(1000 * Tq + T)
    q = torch.randn(B, Hq, Tq, D, generator=g).to(dtype).to(DEV)
    k = (torch.randn(B, Hkv, T, D, generator=g) * 2).to(dtype).to(DEV)
    v = torch.randn(B, Hkv, T, D, generator=g).to(dtype).to(DEV)
    mask = _mask(kind, B, Hq, Tq, T, g)
    ref = _ref(q, k, v, 0.11, mask)
    out = dense_attention(q, k, v, 0.11, mask, torch.float32)
    # fp32 sums of at most D products (scores) and T weights: 2e-5 of the
    # largest |v| (5) covers their rounding
    assert float((out.double() - ref).abs().max()) <= 1e-4
    # a 16-bit output is the fp32 one rounded once
    assert torch.equal(dense_attention(q, k, v, 0.11, mask), out.to(dtype))


@pytest.mark.parametrize("D,Tq,T", [(64, 24, 200), (128, 70, 333), (256, 12, 97)])
def test_many_rows_int4_sym_equals_restored(D, Tq, T):
    """Masked int4_sym K/V give the result of attention over the restored K/V
    bit for bit: the same tiles on the same rounded values."""
    from korith_vllm_ext.codecs import get_codec
    from korith_vllm_ext.int4_decode_attention import int4_decode_attention
    from korith_vllm_ext.kernels import dense_attention

    g = torch.Generator().manual_seed(D + Tq)
    codec = get_codec("int4_sym")
    for dtype in (torch.bfloat16, torch.float16):
        q = torch.randn(2, 8, Tq, D, generator=g).to(dtype).to(DEV)
        kc, vc = (codec.compress(torch.randn(2, 2, T, D, generator=g).to(dtype).to(DEV))
                  for _ in range(2))
        mask = _mask("causal", 2, 8, Tq, T, g)
        got = int4_decode_attention(q, kc, vc, mask=mask)
        want = dense_attention(q, codec.decompress_to(kc, dtype), codec.decompress_to(vc, dtype),
                               None, mask)
        assert torch.equal(got, want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_many_rows_non_finite(dtype):
    """Rows without a visible token are NaN, -inf tokens weigh nothing, and
    inf / NaN in K or V reach the rows that float64 attention shows them in."""
    from korith_vllm_ext.kernels import dense_attention

    g = torch.Generator().manual_seed(3)
    B, H, Tq, T, D = 1, 4, 20, 150, 128
    q, k, v = (torch.randn(B, H, n, D, generator=g).to(dtype).to(DEV)
               for n in (Tq, T, T))
    mask = torch.zeros(Tq, T, device=DEV)
    mask[3] = float("-inf")
    mask[5] = torch.finfo(torch.float32).min
    mask[7, 10:] = float("-inf")
    k[0, 1, 40] = float("inf")
    k[0, 2, 70] = float("nan")
    v[0, 3, 149, 5] = float("inf")
    out = dense_attention(q, k, v, None, mask, torch.float32)
    out, ref = out.double(), _ref(q, k, v, D ** -0.5, mask)
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    assert torch.equal(torch.isinf(out), torch.isinf(ref)) and torch.isinf(ref).any()
    ok = torch.isfinite(ref)
    assert float((out[ok] - ref[ok]).abs().max()) <= 1e-4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hq,Tq,T,D", [(2, 12, 77, 64), (4, 20, 200, 128), (1, 40, 130, 128),
                                       (4, 8, 90, 256), (4, 33, 97, 256)])
def test_many_rows_small_weights(dtype, Hq, Tq, T, D):
    """The softmax weights keep their 32 bits however small they are: one token
    of zeros holds the row's largest weight, so the output is what the weights
    of 2^-20 to 2^-59 give the others."""
    from korith_vllm_ext.kernels import dense_attention

    g = torch.Generator().manual_seed(Tq)
    q = torch.zeros(1, Hq, Tq, D, dtype=dtype, device=DEV)
    k = torch.zeros(1, 1, T, D, dtype=dtype, device=DEV)
    v = (torch.rand(1, 1, T, D, generator=g) + 0.5).to(dtype).to(DEV)
    v[:, :, 3] = 0
    # a row's tokens all weigh about 2^-(20 + row)
    mask = -0.6931471805599453 * (20.0 + torch.arange(Tq)[:, None] + torch.rand(Tq, T, generator=g))
    mask[:, 3] = 0.0
    mask = mask.to(DEV)
    out = dense_attention(q, k, v, None, mask, torch.float32).double()
    ref = _ref(q, k, v, D ** -0.5, mask)
    # 2^x at |x| < 61: its rounded argument puts the weights off by at most
    # 61 ln(2) 2^-23, 5e-6, and the sums of 200 positive terms by less
    assert float(((out - ref).abs() / ref).max()) <= 2e-5
