"""The work that users of this package have it do, as cases to be timed.

A case is one call (or a save and the load that answers it) through a public
entry point, on the KV geometries of this repository's configurations and
benchmark:

  save, restore   the C ABI through amf_hip: quantize-and-gather the pages of
                  a block table into blobs, dequantize-and-scatter them back,
                  every layer in one launch; the caller keeps address tables,
                  block ids and workspace, as a serving engine does
  pool            CompressedVRAMPool.restore_to_vllm: a pool hit, host work
                  and all
  slots           put_from_slots, then restore_to_slots into other slots: what
                  the connector does with a request's token slots
  codec           Codec.compress and decompress_to on a dense tensor
  decode          int4_decode_attention over the paged INT4 pool
  attend          int4_decode_attention(q, k, v): dense or int4_sym K/V, one
                  query row (decode) or many (chunked prefill, causal mask)
"""

import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "axropus-deploy_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import amf_hip  # noqa: E402
from korith_vllm_ext.codecs import get_codec  # noqa: E402
from korith_vllm_ext.compressed_vram_pool import CompressedVRAMPool  # noqa: E402
from korith_vllm_ext.int4_decode_attention import int4_decode_attention  # noqa: E402

BS = 16  # tokens of a vLLM page
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
FORMATS = {
    "fp8_e4m3": amf_hip.FMT_FP8_E4M3,
    "fp8_e4m3_ph": amf_hip.FMT_FP8_E4M3_PH,
    "int4_sym_block": amf_hip.FMT_INT4_SYM_BLOCK,
    "int4_sym": amf_hip.FMT_INT4_SYM,
    "int4_asym_g32": amf_hip.FMT_INT4_ASYM_G32,
}
# layers, KV heads of one rank, head_dim: Qwen2-0.5B; Llama-3-8B whole, in 4
# and in 8 tensor-parallel ranks; Llama-3-70B whole and in 8 ranks
MODELS = [(24, 2, 64), (32, 8, 128), (32, 2, 128), (32, 1, 128), (80, 8, 128), (80, 1, 128)]
# query heads, KV heads, head_dim of one attention layer
HEADS = [(32, 8, 128), (64, 8, 128), (8, 1, 128), (8, 2, 128), (8, 8, 128), (8, 2, 64)]


def listed():
    return [
        # the shortest prefix the connector keeps (64 tokens) hit in the pool:
        # nothing but latency
        {"name": "pool_hit_64_tokens", "kind": "pool", "fmt": "fp8_e4m3_ph", "layers": 24,
         "heads": 2, "dim": 64, "pages": 4, "dtype": "bf16"},
        # one decode step of two sequences with short contexts: latency again
        {"name": "decode_2_short", "kind": "decode", "seqs": 2, "q_heads": 32, "kv_heads": 8,
         "ctx_lo": 700, "ctx_hi": 1500, "dtype": "bf16"},
        # decode step of a busy server, contexts mixed
        {"name": "decode_32_mixed", "kind": "decode", "seqs": 32, "q_heads": 32, "kv_heads": 8,
         "ctx_lo": 1024, "ctx_hi": 32768, "dtype": "bf16"},
        # decode step of the 70B model over long contexts (8 query heads a KV head)
        {"name": "decode_8_long_gqa8", "kind": "decode", "seqs": 8, "q_heads": 64, "kv_heads": 8,
         "ctx_lo": 60000, "ctx_hi": 70000, "dtype": "bf16"},
        # an 8K-token prefix restored, 8B model on one GPU
        {"name": "restore_fp8_ph_8b", "kind": "restore", "fmt": "fp8_e4m3_ph", "layers": 32,
         "heads": 8, "dim": 128, "pages": 512, "dtype": "bf16"},
        # a long prefix saved on one of 8 tensor-parallel ranks of the 70B
        # model: pages of one KV head
        {"name": "save_fp8_ph_70b_tp8", "kind": "save", "fmt": "fp8_e4m3_ph", "layers": 80,
         "heads": 1, "dim": 128, "pages": 500, "dtype": "bf16"},
        # the decode pool's format: saved on a rank of 4, restored on a rank of 8
        {"name": "save_int4_asym_8b_tp4", "kind": "save", "fmt": "int4_asym_g32", "layers": 32,
         "heads": 2, "dim": 128, "pages": 1000, "dtype": "bf16"},
        {"name": "restore_int4_asym_70b_tp8", "kind": "restore", "fmt": "int4_asym_g32",
         "layers": 80, "heads": 1, "dim": 128, "pages": 777, "dtype": "bf16"},
        # the pool's default format (128-token blocks) under vLLM's 16-token
        # pages, a prompt that ends inside a block
        {"name": "slots_int4_block_8b", "kind": "slots", "fmt": "int4_sym_block", "layers": 32,
         "heads": 8, "dim": 128, "tokens": 4016, "dtype": "bf16"},
        # one layer's K and V of an 8K-token prompt through the codec itself
        {"name": "codec_int4_block_layer", "kind": "codec", "fmt": "int4_sym_block", "lead": 2,
         "tokens": 8192, "heads": 8, "dim": 128, "dtype": "bf16"},
        # positional decode over int4_sym K/V
        {"name": "attend_int4_decode", "kind": "attend", "kv": "int4_sym", "batch": 4,
         "q_heads": 32, "kv_heads": 8, "dim": 128, "q_len": 1, "kv_len": 8000,
         "dtype": "bf16"},
        # a 512-token chunk of a prompt against the 4K tokens so far
        {"name": "attend_chunk_causal", "kind": "attend", "kv": "dense", "batch": 1,
         "q_heads": 32, "kv_heads": 8, "dim": 128, "q_len": 512, "kv_len": 4096,
         "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["save", "restore", "pool", "slots", "codec", "decode", "decode", "attend",
                       "attend"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    fmt = rng.choice(sorted(FORMATS))
    L, H, D = rng.choice(MODELS)
    most = 400_000_000 // (L * 2 * BS * H * D)  # pages of the largest cases
    if kind in ("save", "restore"):
        return {"kind": kind, "fmt": rng.choice([fmt, fmt, fmt, fmt, "raw"]), "layers": L,
                "heads": H, "dim": D, "pages": _log_int(rng, 4, min(2048, most)),
                "dtype": dtype}
    if kind == "pool":
        return {"kind": kind, "fmt": fmt, "layers": L, "heads": H, "dim": D,
                "pages": _log_int(rng, 4, min(512, most)), "dtype": dtype}
    if kind == "slots":
        # whole vLLM pages, as the connector's aligned prefixes are, or any length
        t = _log_int(rng, 64, 16 * min(320, most // 2))
        return {"kind": kind, "fmt": fmt, "layers": L, "heads": H, "dim": D,
                "tokens": rng.choice([t // 16 * 16, t]), "dtype": dtype}
    if kind == "codec":
        # [2, tokens, heads, dim] of a layer, or [batch, heads, tokens, dim]
        t = _log_int(rng, 16, 16384)
        if rng.random() < 0.5:
            return {"kind": kind, "fmt": fmt, "lead": 2, "tokens": t, "heads": H, "dim": D,
                    "dtype": dtype}
        return {"kind": kind, "fmt": rng.choice(["int4_sym", "int4_sym_block", "fp8_e4m3"]),
                "lead": rng.choice([1, 2, 3, 4]), "tokens": H, "heads": min(t, 4096), "dim": D,
                "dtype": dtype}
    if kind == "decode":
        hq, hkv, _ = rng.choice([h for h in HEADS if h[2] == 128])
        seqs = _log_int(rng, 1, 64)
        hi = _log_int(rng, 16, min(65536, 500_000 * 8 // (seqs * hkv)))
        return {"kind": kind, "seqs": seqs, "q_heads": hq, "kv_heads": hkv,
                "ctx_lo": rng.randint(1, hi), "ctx_hi": hi, "dtype": dtype}
    hq, hkv, D = rng.choice(HEADS)
    batch = rng.choice([1, 1, 2, 4, 7])
    q_len = rng.choice([1, 1, _log_int(rng, 2, 16), _log_int(rng, 17, 512)])
    most = 32 * 512 * 4096 // (batch * hq * q_len)
    kv_len = max(q_len, _log_int(rng, 64, max(64, min(16384, most))))
    if q_len > kv_len // 2 and batch * hq * q_len * kv_len > 32 * 512 * 4096:
        batch = 1
    return {"kind": "attend", "kv": rng.choice(["dense", "int4_sym"]), "batch": batch,
            "q_heads": hq, "kv_heads": hkv, "dim": D, "q_len": q_len, "kv_len": kv_len,
            "dtype": dtype}


# ----------------------------------------------------------------- inputs --


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))


def _values(g, shape, dtype):
    """N(0, 1) with x20 on one in fifty channels, as KV activations have."""
    x = torch.randn(*shape, generator=g, device="cuda", dtype=dtype)
    k = max(1, round(0.02 * shape[-1]))
    x[..., torch.randperm(shape[-1], generator=g, device="cuda")[:k]] *= 20.0
    return x


def _table(g, pool, n):
    return torch.randperm(pool, generator=g, device="cuda")[:n].to(torch.int32)


def _pool_pages(pages):
    return pages + pages // 2 + 3


def _cache(g, case, pages, fill):
    """One vLLM cache as [layers, 2, pool, 16, heads, dim]."""
    shape = (case["layers"], 2, pages, BS, case["heads"], case["dim"])
    if fill:
        return _values(g, shape, DTYPES[case["dtype"]])
    return torch.zeros(shape, dtype=DTYPES[case["dtype"]], device="cuda")


def _plane_table(t, per_layer=2):
    """Device addresses of t[l, kv] (or of t[l] for both of a layer's planes)."""
    addrs = [(t[l, kv] if per_layer == 2 else t[l]).data_ptr()
             for l in range(t.shape[0]) for kv in range(2)]
    return torch.tensor(addrs, dtype=torch.int64).cuda()


def _blob(case, n):
    """Codes [layers, 2, bytes] and params (uint8) of n pages, zeroed, with
    their plane tables."""
    L, H, D, fmt = case["layers"], case["heads"], case["dim"], case["fmt"]
    elems = n * BS * H * D
    per = {"raw": 2 * elems, "fp8_e4m3": elems, "fp8_e4m3_ph": elems}.get(fmt, elems // 2)
    codes = torch.zeros(L, 2, per, dtype=torch.uint8, device="cuda")
    pbytes = {"fp8_e4m3_ph": n * H * 4, "int4_sym_block": n * 2,
              "int4_asym_g32": n * H * BS * (D // 32) * 4, "fp8_e4m3": 16,
              "int4_sym": D * 2}.get(fmt, 16)
    shared = fmt in ("fp8_e4m3", "int4_sym")
    pad = -(-pbytes // 16) * 16
    params = torch.zeros((L, pad) if shared else (L, 2, pad), dtype=torch.uint8, device="cuda")
    return {"codes": codes, "params": params, "codes_tab": _plane_table(codes),
            "params_tab": _plane_table(params, 1 if shared else 2)}


def _save(case, cache, cache_tab, ids, blob, ws):
    L, _, pool, _, H, D = cache.shape
    n, stride = ids.numel(), BS * H * D * cache.element_size()
    stream = amf_hip.stream_handle(cache.device)
    if case["fmt"] == "raw":
        amf_hip.call("amf_kv_gather_pages", cache_tab.data_ptr(), stride, ids.data_ptr(), pool,
                     blob["codes_tab"].data_ptr(), stride, 2 * L, n, stride, None, stream)
        return
    fn = "amf_fp8_quant_gather" if case["fmt"].startswith("fp8") else "amf_int4_quant_gather"
    amf_hip.call(fn, FORMATS[case["fmt"]], cache_tab.data_ptr(), stride,
                 amf_hip.dtype_tag(cache.dtype), ids.data_ptr(), pool,
                 blob["codes_tab"].data_ptr(), blob["params_tab"].data_ptr(), 2 * L, 2, n, BS, H,
                 D, ws.data_ptr(), ws.numel(), None, stream)


def _restore(case, blob, cache, cache_tab, ids):
    L, _, pool, _, H, D = cache.shape
    n, stride = ids.numel(), BS * H * D * cache.element_size()
    stream = amf_hip.stream_handle(cache.device)
    if case["fmt"] == "raw":
        amf_hip.call("amf_kv_scatter_pages", blob["codes_tab"].data_ptr(), stride,
                     cache_tab.data_ptr(), stride, ids.data_ptr(), pool, 2 * L, n, stride, None,
                     stream)
        return
    fn = "amf_fp8_dequant_scatter" if case["fmt"].startswith("fp8") else "amf_int4_dequant_scatter"
    amf_hip.call(fn, FORMATS[case["fmt"]], blob["codes_tab"].data_ptr(),
                 blob["params_tab"].data_ptr(), cache_tab.data_ptr(), stride,
                 amf_hip.dtype_tag(cache.dtype), ids.data_ptr(), pool, 2 * L, n, BS, H, D, None,
                 stream)


def _workspace(case):
    if case["fmt"] == "raw":
        return None
    n = amf_hip.quant_workspace_bytes(FORMATS[case["fmt"]], 2 * case["layers"], 2, case["dim"])
    return torch.empty(max(16, n), dtype=torch.uint8, device="cuda")


def _contexts(g, case):
    span = case["ctx_hi"] - case["ctx_lo"] + 1
    return torch.randint(0, span, (case["seqs"],), generator=g, device="cuda",
                         dtype=torch.int32) + case["ctx_lo"]


def _slots(g, pool, tokens):
    """Slots of a request's tokens: pages anywhere in the pool, in order
    inside a page; on the host, as the scheduler hands them over."""
    pages = _table(g, pool, -(-tokens // BS)).long().cpu()
    return (pages[:, None] * BS + torch.arange(BS)).reshape(-1)[:tokens].contiguous()


def _pool_for(case, tokens):
    raw = 2 * tokens * case["heads"] * case["dim"]
    return CompressedVRAMPool(case["layers"], (2 * raw // (1 << 20) + 2) << 20, 1 << 17,
                              default_format=case["fmt"])


def _source(case, seed):
    """The values that a page case starts from: (cache, ids, ids of the target)."""
    g = _gen(seed)
    n = case["pages"]
    pool = _pool_pages(n)
    return _cache(g, case, pool, True), _table(g, pool, n), _table(g, pool, n)


def _slot_source(case, seed):
    g = _gen(seed)
    pool = _pool_pages(-(-case["tokens"] // BS))
    return (_cache(g, case, pool, True), _slots(g, pool, case["tokens"]),
            _slots(g, pool, case["tokens"]), pool)


def _decode_source(case, seed):
    """q, context lengths, block table and the KV values of the page pool."""
    g = _gen(seed)
    dt = DTYPES[case["dtype"]]
    ctx = _contexts(g, case)
    pages = [-(-int(c) // BS) for c in ctx.tolist()]
    perm = torch.randperm(sum(pages), generator=g, device="cuda").to(torch.int32)
    table = torch.zeros(case["seqs"], max(pages), dtype=torch.int32, device="cuda")
    at = 0
    for s, n in enumerate(pages):
        table[s, :n] = perm[at:at + n]
        at += n
    q = torch.randn(case["seqs"], case["q_heads"], 128, generator=g, device="cuda").to(dt)
    kv = _values(g, (2, sum(pages), BS, case["kv_heads"], 128), dt)
    return q, ctx, table, kv


def _attend_source(case, seed):
    g = _gen(seed)
    dt = DTYPES[case["dtype"]]
    B, D, Tq, T = case["batch"], case["dim"], case["q_len"], case["kv_len"]
    q = torch.randn(B, case["q_heads"], Tq, D, generator=g, device="cuda").to(dt)
    k = _values(g, (B, case["kv_heads"], T, D), dt)
    v = _values(g, (B, case["kv_heads"], T, D), dt)
    mask = None
    if Tq > 1:  # row i sees the tokens up to its own, the last Tq being the chunk
        mask = torch.zeros(Tq, T, device="cuda")
        mask.masked_fill_(torch.arange(T, device="cuda")[None, :] >
                          torch.arange(T - Tq, T, device="cuda")[:, None], float("-inf"))
    return q, k, v, mask


def _codec_source(case, seed):
    shape = (case["lead"], case["tokens"], case["heads"], case["dim"])
    return _values(_gen(seed), shape, DTYPES[case["dtype"]])


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind in ("save", "restore"):
        cache, src, dst = _source(case, seed)
        blob, ws = _blob(case, case["pages"]), _workspace(case)
        tab = _plane_table(cache)
        if kind == "restore":  # saved earlier; the pages go elsewhere
            _save(case, cache, tab, src, blob, ws)
            cache, src = torch.zeros_like(cache), dst
            tab = _plane_table(cache)
        st.update(cache=cache, tab=tab, ids=src, blob=blob, ws=ws)
    elif kind == "pool":
        cache, src, dst = _source(case, seed)
        pool = _pool_for(case, case["pages"] * BS)
        if not pool.put_from_vllm("prefix", list(cache), src.tolist(), case["pages"] * BS):
            raise RuntimeError("the pool took no entry")
        target = torch.zeros_like(cache)
        st.update(pool=pool, target=target, layers=list(target), table=dst.tolist())
    elif kind == "slots":
        cache, src, dst, _ = _slot_source(case, seed)
        target = torch.zeros_like(cache)
        st.update(pool=_pool_for(case, case["tokens"] + 128), cache=cache, target=target,
                  src_layers=list(cache), dst_layers=list(target), src=src, dst=dst)
    elif kind == "codec":
        st.update(codec=get_codec(case["fmt"]), x=_codec_source(case, seed))
    elif kind == "decode":
        q, ctx, table, kv = _decode_source(case, seed)
        st.update(q=q, ctx=ctx, table=table, kv=get_codec("int4_asym_g32").compress(kv))
    else:
        q, k, v, mask = _attend_source(case, seed)
        if case["kv"] == "int4_sym":
            codec = get_codec("int4_sym")
            k, v = codec.compress(k), codec.compress(v)
        st.update(q=q, k=k, v=v, mask=mask)
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "save":
        _save(case, st["cache"], st["tab"], st["ids"], st["blob"], st["ws"])
        return st["blob"]["codes"], st["blob"]["params"]
    if kind == "restore":
        _restore(case, st["blob"], st["cache"], st["tab"], st["ids"])
        return st["cache"]
    if kind == "pool":
        st["pool"].restore_to_vllm("prefix", st["layers"], st["table"])
        return st["target"]
    if kind == "slots":
        st["pool"].put_from_slots("prefix", st["src_layers"], st["src"])
        st["pool"].restore_to_slots("prefix", st["dst_layers"], st["dst"])
        return st["target"]
    if kind == "codec":
        c = st["codec"].compress(st["x"])
        y = st["codec"].decompress_to(c, st["x"].dtype)
        return c.data.view(torch.uint8), c.scales, y
    if kind == "decode":
        return int4_decode_attention(st["q"], st["kv"], block_tables=st["table"],
                                     context_lens=st["ctx"])
    return int4_decode_attention(st["q"], st["k"], st["v"], mask=st["mask"])


# ------------------------------------------------------------------- work --


def _code_bytes(fmt, elems, H, D, pages, layers):
    """Codes and params of `elems` elements in `pages` pages of all planes."""
    if fmt == "raw":
        return 2 * elems
    if fmt == "fp8_e4m3":
        return elems + 16 * layers
    if fmt == "fp8_e4m3_ph":
        return elems + 4 * pages * H
    if fmt == "int4_sym_block":
        return elems // 2 + 2 * pages
    if fmt == "int4_sym":
        return elems // 2 + 2 * D * layers
    return elems // 2 + elems // 8


def work(case):
    kind = case["kind"]
    if kind in ("save", "restore", "pool"):
        L, H, D, n = case["layers"], case["heads"], case["dim"], case["pages"]
        elems = L * 2 * n * BS * H * D
        return {"bytes": 2 * elems + _code_bytes(case["fmt"], elems, H, D, 2 * L * n, L),
                "flops": 0}
    if kind == "slots":
        L, H, D, T = case["layers"], case["heads"], case["dim"], case["tokens"]
        elems = L * 2 * T * H * D
        return {"bytes": 2 * (2 * elems + _code_bytes(case["fmt"], elems, H, D,
                                                      2 * L * -(-T // BS), L)), "flops": 0}
    if kind == "codec":
        H, D = case["heads"], case["dim"]
        elems = case["lead"] * case["tokens"] * H * D
        pages = case["lead"] * -(-case["tokens"] // BS)
        return {"bytes": 2 * (2 * elems + _code_bytes(case["fmt"], elems, H, D, pages, 1)),
                "flops": 0}
    if kind == "decode":
        tokens = case["seqs"] * (case["ctx_lo"] + case["ctx_hi"]) / 2
        # per token and KV head: 64 code and 16 param bytes, K and V
        return {"bytes": tokens * case["kv_heads"] * 160 + case["seqs"] * case["q_heads"] * 512,
                "flops": tokens * case["q_heads"] * 128 * 4}
    B, Hq, Hkv, D = case["batch"], case["q_heads"], case["kv_heads"], case["dim"]
    Tq, T = case["q_len"], case["kv_len"]
    row = D // 2 if case["kv"] == "int4_sym" else 2 * D
    seen = Tq * T - Tq * (Tq - 1) // 2  # (query, token) pairs under the causal mask
    return {"bytes": 2 * B * Hkv * T * row + 4 * B * Hq * Tq * D + (4 * Tq * T if Tq > 1 else 0),
            "flops": 4 * B * Hq * seen * D}


def tolerance(case):
    """Codecs and copies are exact to the bit.  Attention answers in 16 bits:
    its distance from 64 bits is the rounding of the output (bf16: 1.7e-3,
    fp16: 2e-4), the decode's bounded fp16 weights (3e-4) and, for int4_sym
    K/V under a mask or at head_dim 64, the rounding of the restored K and V
    (fp16: 1.2e-3); four times what is seen."""
    if case["kind"] in ("decode", "attend"):
        if case["dtype"] == "bf16":
            return {"rel": 8e-3}
        return {"rel": 5e-3 if case.get("kv") == "int4_sym" else 1.5e-3}
    return "exact"


# ---------------------------------------------------------------- 64 bits --


def _over(x, n):
    """x / n, divided (a plain number would be multiplied by its reciprocal)."""
    return x / torch.full_like(x, n)


def _quantized(x, fmt, dims):
    """x as the format holds it, in 64 bits: one scale over the axes `dims`
    (asymmetric: over 32 neighbours of the last axis)."""
    x32 = x.float()
    if fmt == "raw":
        return x.double()
    if fmt == "int4_asym_g32":
        y = x32.reshape(*x.shape[:-1], -1, 32)
        mn = y.amin(-1, keepdim=True)
        s = _over((y.amax(-1, keepdim=True) - mn).clamp_min(1e-8), 15.0)
        c = ((y - mn) / s).round_().clamp_(0, 15)
        return (c.double() * s.half().double() + mn.half().double()).reshape(x.shape)
    amax = x32.abs().amax(dims, keepdim=True)
    if fmt.startswith("fp8"):
        floor = 1e-8 if fmt == "fp8_e4m3_ph" else float(torch.tensor(1e-8, dtype=x.dtype))
        s = _over(amax.clamp_min(floor), 448.0)
        c = (x32 / s.clamp_min(1e-12)).clamp_(-448, 448).to(torch.float8_e4m3fn)
        return c.float().double() * s.double()
    s = _over(amax.clamp_min(1e-8), 7.0)
    return (x32 / s).round_().clamp_(-8, 7).double() * s.half().double()


# axes of [.., pages, tokens, heads, dim] that share a scale
_PAGE_DIMS = {"fp8_e4m3_ph": (-3, -1), "int4_sym_block": (-3, -2, -1)}


def _layer64(x, fmt):
    """[2, pages, 16, heads, dim] of a layer as the format holds it."""
    if fmt == "fp8_e4m3":
        return _quantized(x, fmt, (0, 1, 2, 3, 4))
    if fmt == "int4_sym":
        return _quantized(x, fmt, (0, 1, 2, 3))
    return _quantized(x, fmt, _PAGE_DIMS.get(fmt))


def _tokens64(x, fmt):
    """[2, tokens, heads, dim] of a layer cut as dense entries are: blocks of
    128 tokens (int4_sym_block) or of 16, the last one filled with zeros."""
    P, T, H, D = x.shape
    block = (T if T <= 128 else 128) if fmt == "int4_sym_block" else BS
    pad = -T % block
    if pad:
        x = torch.cat([x, torch.zeros(P, pad, H, D, dtype=x.dtype, device=x.device)], 1)
    return _layer64(x.reshape(P, -1, block, H, D), fmt).reshape(P, -1, H, D)[:, :T]


def _attend64(q, k, v, mask):
    """q [heads, rows, dim] over k, v [tokens, dim] of one KV head, in 64 bits."""
    s = torch.matmul(q.double(), k.t().contiguous()) / math.sqrt(q.shape[-1])
    if mask is not None:
        s = s + mask.double()
    return torch.matmul(torch.softmax(s, -1), v.contiguous())


def exact(case, seed):
    kind, fmt = case["kind"], case.get("fmt")
    if kind == "save":
        return None  # codes
    if kind in ("restore", "pool"):
        cache, src, dst = _source(case, seed)
        out = torch.zeros(cache.shape, dtype=torch.float64, device="cuda")
        for l in range(cache.shape[0]):
            out[l][:, dst.long()] = _layer64(cache[l][:, src.long()], fmt)
        return out
    if kind == "slots":
        cache, src, dst, pool = _slot_source(case, seed)
        L, _, _, _, H, D = cache.shape
        rows = cache.view(L, 2, pool * BS, H, D)
        out = torch.zeros(rows.shape, dtype=torch.float64, device="cuda")
        for l in range(L):
            out[l][:, dst.cuda()] = _tokens64(rows[l][:, src.cuda()], fmt)
        return out.view(cache.shape)
    if kind == "codec":
        x = _codec_source(case, seed)
        if fmt == "fp8_e4m3":
            y = _quantized(x, fmt, (0, 1, 2, 3))
        elif fmt == "int4_sym":
            y = _quantized(x, fmt, (0, 1, 2))
        else:
            y = _tokens64(x, fmt)
        return None, None, y
    if kind == "decode":
        q, ctx, table, kv = _decode_source(case, seed)
        out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
        R = case["q_heads"] // case["kv_heads"]
        for s, c in enumerate(ctx.tolist()):
            ids = table[s, :-(-c // BS)].long()
            k, v = (_quantized(kv[i][ids], "int4_asym_g32", None).flatten(0, 1)[:c]
                    for i in range(2))
            for h in range(case["kv_heads"]):
                out[s, h * R:(h + 1) * R] = _attend64(q[s, h * R:(h + 1) * R], k[:, h], v[:, h],
                                                      None)
        return out
    q, k, v, mask = _attend_source(case, seed)
    if case["kv"] == "int4_sym":
        k, v = (_quantized(t, "int4_sym", (0, 1, 2)) for t in (k, v))
    else:
        k, v = k.double(), v.double()
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    R = case["q_heads"] // case["kv_heads"]
    for b in range(case["batch"]):
        for h in range(case["q_heads"]):
            out[b, h] = _attend64(q[b, h], k[b, h // R], v[b, h // R], mask)
    return out
